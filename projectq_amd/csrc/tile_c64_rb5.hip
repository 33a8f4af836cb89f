// Plain and batched tile passes: complex64 states, 5 register bits.
#include "tile_plain.hpp"

namespace qs {
namespace dev {

QS_INSTANTIATE_TILE(float, 5)

}  // namespace dev
}  // namespace qs
