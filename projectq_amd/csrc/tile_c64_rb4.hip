// Plain and batched tile passes: complex64 states, 4 register bits.
#include "tile_plain.hpp"

namespace qs {
namespace dev {

QS_INSTANTIATE_TILE(float, 4)

}  // namespace dev
}  // namespace qs
