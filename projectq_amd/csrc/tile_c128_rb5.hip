// Plain and batched tile passes: complex128 states, 5 register bits.
#include "tile_plain.hpp"

namespace qs {
namespace dev {

QS_INSTANTIATE_TILE(double, 5)

}  // namespace dev
}  // namespace qs
