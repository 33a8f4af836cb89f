// Plain and batched tile passes: complex128 states, 4 register bits.
#include "tile_plain.hpp"

namespace qs {
namespace dev {

QS_INSTANTIATE_TILE(double, 4)

}  // namespace dev
}  // namespace qs
