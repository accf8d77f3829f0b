// decode_fp8.hip -- the decode kernels over fp8 pools (v_mfma_f32_16x16x32_bf16).
#include "decode_stream.hpp"

namespace rkv {

Launch decode_fp8(int D, int G, int P, bool append) {
  return pick_d<uint8_t, RKV_FP8>(D, G, P, append);
}

}  // namespace rkv
