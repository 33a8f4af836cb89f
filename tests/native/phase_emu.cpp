// Test-only CPU run of tile passes with phase ops: the product planner (planner.cpp) on a gate list, and
// the passes replayed with the kernel's rules for stages, register ops and pending factors.
#include <cstring>
#include <string>

#include "planner.hpp"

using cplx = std::complex<double>;

namespace {

struct Fail {
  std::string what;
};
void check(bool ok, const char *what) {
  if (!ok) throw Fail{what};
}

// op on the 16 amplitudes of one thread; `active`: its controls outside the register bits hold
void register_op(std::vector<cplx> &v, const qs::dev::RegOp &op, const cplx *m, bool active) {
  const uint32_t kind = (op.code >> 8) & 15u, b0 = op.code & 15u, cb = op.code >> 12;
  check(kind < qs::dev::kOpPhases, "a factor outside a group");
  check(kind != qs::dev::kOp2General && kind != qs::dev::kOp2Diag, "2-qubit op beside phases");
  if (!active) return;
  const uint32_t rc = cb ? 1u << (cb - 1) : 0u;
  for (uint32_t i = 0; i < 16; ++i) {
    if ((i & rc) != rc || ((i >> b0) & 1)) continue;
    cplx &a = v[i], &b = v[i | 1u << b0];
    const cplx x = a, y = b;
    a = m[0] * x + m[1] * y;
    b = m[2] * x + m[3] * y;
  }
}

void replay(cplx *psi, unsigned n, const qs::TileProgram &prog) {
  const qs::dev::TilePass &P = prog.P;
  const uint32_t size = 1u << P.t, seg = (1u << P.L) - 1;
  std::vector<cplx> tile(size);
  for (uint64_t k = 0; k < uint64_t(1) << (n - P.t); ++k) {
    uint64_t base = k << P.L;
    for (uint32_t b = 0; b < P.h; ++b)
      base = ((base >> P.hpos[b]) << (P.hpos[b] + 1)) | (base & ((uint64_t(1) << P.hpos[b]) - 1));
    auto at = [&](uint32_t l) {
      uint64_t i = base | (l & seg);
      for (uint32_t b = 0; b < P.h; ++b) i |= uint64_t((l >> (P.L + b)) & 1u) << P.hpos[b];
      return i;
    };
    for (uint32_t l = 0; l < size; ++l) tile[l] = psi[at(l)];
    for (const auto &st : prog.stages) {
      if (st.kind == qs::dev::kStageLds) {
        const auto &op = prog.tops[st.begin];
        uint32_t tm = 0;
        for (uint32_t j = 0; j < (1u << op.k); ++j) tm |= op.off[j];
        if ((base & op.gcmask) != op.gcmask) continue;
        for (uint32_t l = 0; l < size; ++l) {
          if ((l & tm) || (l & op.lcmask) != op.lcmask) continue;
          std::vector<cplx> x(size_t(1) << op.k), y(x.size());
          for (size_t j = 0; j < x.size(); ++j) x[j] = tile[l | op.off[j]];
          for (size_t r = 0; r < x.size(); ++r)
            for (size_t c = 0; c < x.size(); ++c) y[r] += prog.mats[op.mat + r * x.size() + c] * x[c];
          for (size_t j = 0; j < x.size(); ++j) tile[l | op.off[j]] = y[j];
        }
        continue;
      }
      uint32_t rm = 0;
      for (int b = 0; b < 4; ++b) rm |= 1u << st.fixed[b];
      for (uint32_t lb = 0; lb < size; ++lb) {
        if (lb & rm) continue;
        std::vector<cplx> v(16);
        auto reg = [&](uint32_t i) {
          uint32_t l = lb;
          for (int b = 0; b < 4; ++b) l |= ((i >> b) & 1u) << st.fixed[b];
          return l;
        };
        for (uint32_t i = 0; i < 16; ++i) v[i] = tile[reg(i)];
        auto active = [&](const qs::dev::RegOp &op) {
          check((op.lcmask & rm) == 0, "op");
          return (base & op.gcmask) == op.gcmask && (lb & op.lcmask) == op.lcmask;
        };
        for (uint32_t o = st.begin; o < st.end; ++o) {
          const auto &op = prog.rops[o];
          if (((op.code >> 8) & 15u) != qs::dev::kOpPhases) {
            check(op.mat + 4 <= prog.mats.size(), "op");
            register_op(v, op, prog.mats.data() + op.mat, active(op));
            continue;
          }
          check(op.code >> 12 == 0 && ((op.code >> 4) & 15u) == 0 && op.rcmask > 0 && o + op.rcmask < st.end &&
                    op.mat + op.rcmask <= prog.mats.size(),
                "phase encoding");
          cplx f = 1.0;
          for (uint32_t i = 0; i < op.rcmask; ++i) {
            const auto &term = prog.rops[o + 1 + i];
            check(term.code == qs::dev::kOpPhaseTerm << 8, "phase term");
            if (active(term)) f *= prog.mats[op.mat + i];
          }
          for (uint32_t i = 0; i < 16; ++i)
            if ((i & op.code & 15u) == (op.code & 15u)) v[i] *= f;
          o += op.rcmask;
        }
        for (uint32_t i = 0; i < 16; ++i) tile[reg(i)] = v[i];
      }
    }
    for (uint32_t l = 0; l < size; ++l) {
      uint32_t src = 0;
      for (uint32_t b = 0; b < P.t; ++b) src |= ((l >> b) & 1u) << P.sperm[b];
      psi[at(l)] = tile[src];
    }
  }
}

thread_local std::string message;

}  // namespace

// Gates as (targets, control mask, matrix) lists; psi: 2^n complex128, in place, in the reference layout.
// phases = 0 plans the same gates without phase ops.  Returns the number of passes (-1: error).
extern "C" int phase_run(unsigned n, unsigned t, unsigned lmin, int relabel, int phases, int n_gates, const uint32_t *k,
                         const uint32_t *tpos, const uint64_t *cmask, const double *mats, double *psi, int *n_phase_ops) {
  try {
    std::vector<qs::PGate> gates;
    for (int i = 0; i < n_gates; ++i) {
      qs::PGate g;
      for (uint32_t l = 0; l < k[i]; ++l) g.tpos.push_back(*tpos++);
      for (size_t e = 0; e < (size_t(1) << (2 * k[i])); ++e, mats += 2) g.m.push_back(cplx(mats[0], mats[1]));
      g.cmask = cmask[i];
      gates.push_back(std::move(g));
    }
    gates = qs::merge_single_qubit_runs(qs::cnot_to_cz(gates));
    if (phases) gates = qs::diagonals_to_phases(gates);
    const auto passes = qs::schedule_tiles(gates, qs::TileShape{n, t, lmin}, qs::slot_chooser(qs::kSlotEarliest), 256, 16.0,
                                           relabel != 0);
    std::vector<cplx> state((cplx *)psi, (cplx *)psi + (size_t(1) << n));
    std::vector<uint32_t> phys(n);
    for (uint32_t q = 0; q < n; ++q) phys[q] = q;
    *n_phase_ops = 0;
    std::vector<int> seen(gates.size(), 0);
    for (const auto &ps : passes) {
      qs::TileProgram prog;
      qs::build_tile_pass(gates, ps, t, 4, false, prog);
      for (const auto &op : prog.rops) *n_phase_ops += ((op.code >> 8) & 15u) == qs::dev::kOpPhases;
      for (int g : ps.gates) seen[g]++;
      replay(state.data(), n, prog);
      for (const auto &s : prog.swaps)
        for (uint32_t &p : phys) p = p == s.first ? s.second : p == s.second ? s.first : p;
    }
    for (int s : seen) check(s == 1, "a gate was left out or taken twice");
    for (uint64_t i = 0; i < (uint64_t(1) << n); ++i) {
      uint64_t from = 0;
      for (uint32_t q = 0; q < n; ++q) from |= ((i >> q) & 1u) << phys[q];
      ((cplx *)psi)[i] = state[from];
    }
    return (int)passes.size();
  } catch (const Fail &f) {
    message = f.what;
  } catch (const std::exception &e) {
    message = e.what();
  }
  return -1;
}
extern "C" const char *phase_error() { return message.c_str(); }
