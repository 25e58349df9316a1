// Dense q8 linears on the register tiles.
#include "reg_tiles_impl.hpp"

namespace sx::rt::detail {
hipError_t dense_q8(const Params &p, int act, int out_act, hipStream_t stream) { return dense<8>(p, act, out_act, stream); }
}  // namespace sx::rt::detail
