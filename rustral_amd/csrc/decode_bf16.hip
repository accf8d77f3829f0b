// decode_bf16.hip -- the decode kernels over bf16 pools (v_mfma_f32_16x16x32_bf16
// and _16x16x16_bf16).
#include "decode_stream.hpp"

namespace rkv {

Launch decode_bf16(int D, int G, int P, bool append) {
  return pick_d<uint16_t, RKV_BF16>(D, G, P, append);
}

}  // namespace rkv
