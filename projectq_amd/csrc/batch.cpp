// Batched circuits (see batch.hpp).
#include <cstdlib>
#include "batch.hpp"

#include <algorithm>
#include <complex>
#include <cstring>
#include <limits>
#include <memory>

namespace qs {

namespace {

template <class T>
T *to_device(const std::vector<T> &v) {
  if (v.empty()) return nullptr;
  T *d = nullptr;
  QS_HIP(hipMalloc(&d, v.size() * sizeof(T)));
  QS_HIP(hipMemcpy(d, v.data(), v.size() * sizeof(T), hipMemcpyHostToDevice));
  return d;
}

std::vector<BatchShape> candidate_shapes(bool c64) {
  if (c64)
    return {{12, 4, 5, false}, {11, 4, 5, false}, {10, 4, 4, false}, {12, 5, 5, false},
            {10, 5, 5, false}, {12, 4, 4, true}, {11, 4, 4, true}, {10, 4, 4, true}, {12, 4, 5, true}};
  return {{12, 4, 4, false}, {11, 4, 4, false}, {10, 4, 4, false}, {12, 4, 4, true}};
}

}  // namespace

Batch::Batch(bool c64, std::vector<BatchCircuit> circuits, bool autotune) : c64_(c64), circ_(std::move(circuits)) {
  if (circ_.empty()) throw ValueError("batch: no circuits");
  for (auto &c : circ_) {
    if (c.n < 1 || c.n > 30) throw ValueError("batch: circuits hold 1..30 qubits");
    for (auto &g : c.gates) {
      if (g.tpos.empty() || g.tpos.size() > 5) throw ValueError("batch: gates act on 1..5 qubits");
      for (uint32_t p : g.tpos)
        if (p >= c.n) throw ValueError("batch: gate target outside its circuit");
      if (g.cmask >> c.n) throw ValueError("batch: control outside its circuit");
    }
    for (auto &t : c.terms)
      if ((t.x | t.z) >> c.n) throw ValueError("batch: Pauli string outside its circuit");
  }
  std::vector<BatchShape> shapes = candidate_shapes(c64_);
  long forced = -1;  // PROJECTQ_AMD_BATCH_SHAPE=k: candidate k only, no timing (tests)
  if (const char *env = std::getenv("PROJECTQ_AMD_BATCH_SHAPE")) {
    forced = std::strtol(env, nullptr, 10);
    if (forced < 0 || forced >= (long)shapes.size())
      throw ValueError("PROJECTQ_AMD_BATCH_SHAPE: no such candidate shape");
  }
  try {  // a constructor that throws runs no destructor: free what was made so far
    dev::prepare_tile_kernels();
    QS_HIP(hipStreamCreateWithFlags(&stream_, hipStreamNonBlocking));
    QS_HIP(hipEventCreate(&ev0_));
    QS_HIP(hipEventCreate(&ev1_));
    QS_HIP(hipHostMalloc((void **)&h_energies_, circ_.size() * sizeof(double), hipHostMallocDefault));
    if (forced >= 0 || !autotune) {
      build(shapes[forced >= 0 ? (size_t)forced : 0]);
      return;
    }
    // autotuner: time every candidate shape on this batch (graph launches), keep the fastest.  Within 2% the
    // later one: the relabelling shapes with L = 4 and L = 5 take the same time to 0.5% on many batches, and the shape, so
    // the rounding of the energies, should not hang on the noise of a run.
    std::vector<double> e(circ_.size()), ms(shapes.size(), 0.0);
    for (size_t k = 0; k < shapes.size(); ++k) {
      build(shapes[k]);
      run(true, e.data());  // warm-up
      for (int r = 0; r < 3; ++r) ms[k] += run(true, e.data());
    }
    const double limit = 1.02 * *std::min_element(ms.begin(), ms.end());
    size_t best = shapes.size() - 1;
    while (ms[best] > limit) --best;
    build(shapes[best]);
  } catch (...) {
    destroy();
    throw;
  }
}

Batch::~Batch() { destroy(); }

void Batch::destroy() {
  release();
  if (ev0_) (void)hipEventDestroy(ev0_);
  if (ev1_) (void)hipEventDestroy(ev1_);
  if (h_energies_) (void)hipHostFree(h_energies_);
  if (stream_) (void)hipStreamDestroy(stream_);
  ev0_ = ev1_ = nullptr;
  h_energies_ = nullptr;
  stream_ = nullptr;
}

void Batch::release() {
  if (stream_) (void)hipStreamSynchronize(stream_);
  if (exec_) (void)hipGraphExecDestroy(exec_);
  if (graph_) (void)hipGraphDestroy(graph_);
  exec_ = nullptr;
  graph_ = nullptr;
  for (auto p : d_jobs_) (void)hipFree(p);
  for (auto p : d_block_job_) (void)hipFree(p);
  d_jobs_.clear();
  d_block_job_.clear();
  launch_jobs_.clear();
  launch_blocks_.clear();
  launch_tmax_.clear();
  void *bufs[] = {psi_, d_state_off_, d_stages_, d_rops_, d_tops_, d_mats_, d_epass_, d_eblock_, d_egroup_, d_estring_, d_eslot_, d_partials_, d_energies_};
  for (void *b : bufs) (void)hipFree(b);
  psi_ = d_state_off_ = nullptr;
  d_stages_ = d_rops_ = d_tops_ = d_mats_ = nullptr;
  d_epass_ = nullptr;
  d_eblock_ = nullptr;
  d_egroup_ = nullptr;
  d_estring_ = nullptr;
  d_eslot_ = nullptr;
  energy_launches_.clear();
  d_partials_ = d_energies_ = nullptr;
}

void Batch::build(const BatchShape &shape) {
  release();
  shape_ = shape;
  // ---- plan every circuit; collect programs and per-pass jobs
  std::vector<dev::TileStage> stages;
  std::vector<dev::RegOp> rops;
  std::vector<dev::TileOp> tops;
  std::vector<std::complex<double>> mats;
  std::vector<uint64_t> state_off(circ_.size());
  std::vector<std::vector<dev::BatchJob>> jobs;  // by pass index
  std::vector<std::vector<size_t>> job_circuit;  // circuit of every job, by pass index
  std::vector<std::vector<uint32_t>> final_pos(circ_.size());  // label -> position after the passes
  total_amps_ = 0;
  for (size_t c = 0; c < circ_.size(); ++c) {
    const BatchCircuit &bc = circ_[c];
    state_off[c] = total_amps_;
    total_amps_ += uint64_t(1) << bc.n;
    std::vector<PGate> gates;
    for (const PGate &g : bc.gates)
      if (!(g.tmask() & g.cmask)) gates.push_back(g);
    gates = merge_single_qubit_runs(gates);
    const unsigned t = std::min(bc.n, shape.tmax);
    TileShape ts{bc.n, t, shape.lmin};
    std::vector<PPass> passes = schedule_tiles(gates, ts, nullptr, 256, 16.0, shape.relabel);
    std::vector<uint32_t> &phys = final_pos[c];
    std::vector<uint32_t> label(bc.n);
    phys.resize(bc.n);
    for (uint32_t q = 0; q < bc.n; ++q) phys[q] = label[q] = q;
    for (size_t p = 0; p < passes.size(); ++p) {
      TileProgram prog;
      build_tile_pass(gates, passes[p], t, shape.rb, c64_, prog);
      for (const auto &sw : prog.swaps) {
        const uint32_t a = label[sw.first], b = label[sw.second];
        std::swap(label[sw.first], label[sw.second]);
        phys[a] = sw.second;
        phys[b] = sw.first;
      }
      if (prog.stages.empty()) continue;
      dev::BatchJob job{};
      job.state_off = state_off[c];
      job.stage_off = (uint32_t)stages.size();
      job.rop_off = (uint32_t)rops.size();
      job.top_off = (uint32_t)tops.size();
      job.mat_off = (uint32_t)mats.size();
      job.P = prog.P;
      stages.insert(stages.end(), prog.stages.begin(), prog.stages.end());
      rops.insert(rops.end(), prog.rops.begin(), prog.rops.end());
      tops.insert(tops.end(), prog.tops.begin(), prog.tops.end());
      mats.insert(mats.end(), prog.mats.begin(), prog.mats.end());
      if (jobs.size() <= p) {
        jobs.resize(p + 1);
        job_circuit.resize(p + 1);
      }
      jobs[p].push_back(job);
      job_circuit[p].push_back(c);
    }
  }
  // ---- launches: pass p of every circuit that has one
  for (size_t p = 0; p < jobs.size(); ++p) {
    auto &js = jobs[p];
    if (js.empty()) continue;
    uint32_t blocks = 0, tmax = 0;
    std::vector<uint32_t> block_job;
    for (size_t j = 0; j < js.size(); ++j) {
      js[j].first_block = blocks;
      const uint64_t tiles = (uint64_t(1) << circ_[job_circuit[p][j]].n) >> js[j].P.t;
      if (blocks + tiles > (uint64_t)std::numeric_limits<int32_t>::max()) throw ValueError("batch: too many tiles in one launch");
      for (uint64_t b = 0; b < tiles; ++b) block_job.push_back((uint32_t)j);
      blocks += (uint32_t)tiles;
      tmax = std::max(tmax, js[j].P.t);
    }
    d_jobs_.push_back(to_device(js));
    d_block_job_.push_back(to_device(block_job));
    launch_jobs_.push_back(js);
    launch_blocks_.push_back(blocks);
    launch_tmax_.push_back(tmax);
  }
  // ---- energies: every circuit's strings in plans of up to 128, every pass of a plan over its tiles
  std::vector<dev::BatchEnergyPass> epass;
  std::vector<EnergyGroup> egroup;
  std::vector<EnergyString> estring;
  std::vector<uint32_t> eslot;
  constexpr int kXcds = 8;
  constexpr uint64_t kBatchWorkgroups = 8;  // per circuit at least: 100 strings in one workgroup take 40 us
  constexpr uint32_t kSmallest = 8, kSizes = 5;  // tiles of 2^8 .. 2^12 amplitudes
  constexpr size_t kOwnLaunch = 1024;            // workgroups, four per CU
  // Workgroup w runs on XCD w mod 8.  Every circuit goes whole to one XCD (largest first, to the
  // least loaded), so the later passes over its state hit that XCD's L2; the XCDs' workgroup lists are
  // interleaved and padded with idle workgroups to equal length.
  std::vector<std::vector<dev::BatchEnergyBlock>> per_xcd[kSizes];
  for (auto &v : per_xcd) v.resize(kXcds);
  std::vector<size_t> order(circ_.size());
  std::vector<int> xcd_of(circ_.size());
  for (size_t c = 0; c < order.size(); ++c) order[c] = c;
  std::stable_sort(order.begin(), order.end(), [&](size_t a, size_t b) { return circ_[a].n > circ_[b].n; });
  std::vector<uint64_t> load(kXcds, 0);
  for (size_t c : order) {
    const int x = (int)(std::min_element(load.begin(), load.end()) - load.begin());
    load[x] += (uint64_t(1) << circ_[c].n) * std::max<size_t>(circ_[c].terms.size(), 1);
    xcd_of[c] = x;
  }
  auto plan = std::make_unique<EnergyPlan>();
  std::vector<EnergyTerm> terms;
  std::vector<std::vector<dev::BatchEnergyBlock>> of_circuit(circ_.size());
  std::vector<uint32_t> tile_bits(circ_.size(), kSmallest);
  for (size_t c = 0; c < circ_.size(); ++c) {
    eslot.push_back(eslot.empty() ? 0u : eslot.back());
    terms.clear();
    for (const dev::PauliTerm &t0 : circ_[c].terms) {
      // the strings act on the circuit's final layout (relabelling moves qubits); Hermitian, so the
      // coefficient with its phase is real, or imaginary for an odd number of Y
      EnergyTerm t{0, 0, 1.0, t0.c_re};
      for (uint32_t q = 0; q < circ_[c].n; ++q) {
        t.x |= ((t0.x >> q) & 1u) << final_pos[c][q];
        t.z |= ((t0.z >> q) & 1u) << final_pos[c][q];
      }
      if (__builtin_popcountll(t.x & t.z) & 1) {
        t.omega = std::complex<double>(0.0, 1.0);
        t.c = t0.c_im;
      }
      terms.push_back(t);
    }
    uint32_t slot = eslot.back();
    for (size_t t0 = 0; t0 < terms.size(); t0 += kEnergyMaxStrings) {
      const int m = (int)std::min<size_t>(kEnergyMaxStrings, terms.size() - t0);
      plan_energy(terms.data() + t0, m, circ_[c].n, c64_, kBatchWorkgroups, *plan);
      tile_bits[c] = plan->t;
      const uint32_t tiles = circ_[c].n > plan->t ? 1u << (circ_[c].n - plan->t) : 1u;
      for (uint32_t p = 0; p < plan->n_passes; ++p) {
        dev::BatchEnergyPass bp{state_off[c], uint64_t(1) << circ_[c].n, plan->L, plan->h, plan->passes[p]};
        bp.pass.first_group += (uint32_t)egroup.size();
        const uint32_t each = std::max(1u, tiles / 1024);
        for (uint32_t k = 0; k < tiles; k += each)
          of_circuit[c].push_back(dev::BatchEnergyBlock{(uint32_t)epass.size(), k, std::min(each, tiles - k), slot++});
        epass.push_back(bp);
      }
      for (uint32_t g = 0; g < plan->n_groups; ++g) {
        EnergyGroup eg = plan->groups[g];
        eg.next += (uint32_t)estring.size();
        egroup.push_back(eg);
      }
      estring.insert(estring.end(), plan->strings, plan->strings + plan->n_strings);
    }
    eslot.back() = slot;
  }
  eslot.insert(eslot.begin(), 0u);
  egroup.push_back(EnergyGroup{});  // kernels load one group ahead
  for (size_t c : order) {
    auto &list = per_xcd[tile_bits[c] - kSmallest][xcd_of[c]];
    list.insert(list.end(), of_circuit[c].begin(), of_circuit[c].end());
  }
  std::vector<dev::BatchEnergyBlock> eblock;
  auto launch = [&](uint32_t t, const std::vector<std::vector<dev::BatchEnergyBlock>> &lists) {
    size_t longest = 0;
    for (auto &v : lists) longest = std::max(longest, v.size());
    if (longest == 0) return;
    energy_launches_.push_back({t, (uint32_t)eblock.size(), (uint32_t)(longest * kXcds)});
    for (size_t k = 0; k < longest; ++k)
      for (int x = 0; x < kXcds; ++x) eblock.push_back(k < lists[x].size() ? lists[x][k] : dev::BatchEnergyBlock{dev::kNoPass, 0, 0, 0});
  };
  // the largest first; sizes that do not fill the chip go together
  std::vector<uint32_t> small;
  for (uint32_t s = kSizes; s-- > 0;) {
    size_t count = 0;
    for (auto &v : per_xcd[s]) count += v.size();
    if (count >= kOwnLaunch) launch(kSmallest + s, per_xcd[s]);
    else if (count > 0) small.push_back(s);
  }
  if (small.size() == 1) {
    launch(kSmallest + small[0], per_xcd[small[0]]);
  } else {
    std::vector<std::vector<dev::BatchEnergyBlock>> mixed(kXcds);
    for (uint32_t s : small)
      for (int x = 0; x < kXcds; ++x) mixed[x].insert(mixed[x].end(), per_xcd[s][x].begin(), per_xcd[s][x].end());
    launch(dev::kMixedTiles, mixed);
  }
  // ---- device buffers
  const size_t ab = c64_ ? 8 : 16;
  QS_HIP(hipMalloc(&psi_, total_amps_ * ab));
  d_state_off_ = to_device(state_off);
  d_stages_ = to_device(stages);
  d_rops_ = to_device(rops);
  two_qubit_ops_ = false;
  for (const dev::RegOp &op : rops) {
    const uint32_t kind = (op.code >> 8) & 15u;
    two_qubit_ops_ = two_qubit_ops_ || kind == dev::kOp2General || kind == dev::kOp2Diag;
  }
  d_tops_ = to_device(tops);
  if (c64_) {
    std::vector<float2> m(mats.size());
    for (size_t i = 0; i < m.size(); ++i) m[i] = make_float2((float)mats[i].real(), (float)mats[i].imag());
    d_mats_ = to_device(m);
  } else {
    std::vector<double2> m(mats.size());
    for (size_t i = 0; i < m.size(); ++i) m[i] = make_double2(mats[i].real(), mats[i].imag());
    d_mats_ = to_device(m);
  }
  d_epass_ = to_device(epass);
  d_eblock_ = to_device(eblock);
  d_egroup_ = to_device(egroup);
  d_estring_ = to_device(estring);
  d_eslot_ = to_device(eslot);
  QS_HIP(hipMalloc(&d_partials_, std::max<size_t>(eslot.back(), 1) * sizeof(double)));
  QS_HIP(hipMalloc(&d_energies_, circ_.size() * sizeof(double)));
  // ---- capture one run into a graph
  QS_HIP(hipStreamBeginCapture(stream_, hipStreamCaptureModeThreadLocal));
  try {
    enqueue();
  } catch (...) {
    hipGraph_t g = nullptr;
    (void)hipStreamEndCapture(stream_, &g);
    if (g) (void)hipGraphDestroy(g);
    throw;
  }
  QS_HIP(hipStreamEndCapture(stream_, &graph_));
  QS_HIP(hipGraphInstantiate(&exec_, graph_, nullptr, nullptr, 0));
}

void Batch::enqueue() {
  auto go = [&](auto tag) {
    using R = decltype(tag);
    amp_t<R> *psi = (amp_t<R> *)psi_;
    dev::batch_init<R>(psi, total_amps_, d_state_off_, (int)circ_.size(), stream_);
    for (size_t l = 0; l < launch_jobs_.size(); ++l)
      dev::batch_tile_pass<R>(psi, d_jobs_[l], d_block_job_[l], launch_blocks_[l], launch_tmax_[l], (int)shape_.rb,
                              (const dev::TileStage *)d_stages_, (const dev::RegOp *)d_rops_,
                              (const dev::TileOp *)d_tops_, (const amp_t<R> *)d_mats_, two_qubit_ops_, stream_);
    for (const EnergyLaunch &l : energy_launches_)
      dev::batch_energy<R>(psi, l.t, d_epass_, d_eblock_ + l.first_block, l.n_blocks, d_egroup_, d_estring_, d_partials_,
                           stream_);
  };
  if (c64_) go(float{});
  else go(double{});
  dev::batch_energy_finish(d_eslot_, (int)circ_.size(), d_partials_, d_energies_, stream_);
}

double Batch::run(bool graph, double *energies) {
  QS_HIP(hipEventRecord(ev0_, stream_));
  if (graph) QS_HIP(hipGraphLaunch(exec_, stream_));
  else enqueue();
  QS_HIP(hipEventRecord(ev1_, stream_));
  QS_HIP(hipMemcpyAsync(h_energies_, d_energies_, circ_.size() * sizeof(double), hipMemcpyDeviceToHost, stream_));
  QS_HIP(hipStreamSynchronize(stream_));
  float ms = 0.f;
  QS_HIP(hipEventElapsedTime(&ms, ev0_, ev1_));
  std::memcpy(energies, h_energies_, circ_.size() * sizeof(double));
  return ms;
}

}  // namespace qs
