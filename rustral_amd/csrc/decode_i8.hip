// decode_i8.hip -- the decode kernels over int8 pools (v_mfma_i32_16x16x64_i8 and
// _16x16x32_i8; bf16 ones at 8 query heads per KV head).
#include "decode_stream.hpp"

namespace rkv {

Launch decode_i8(int D, int G, int P, bool append) {
  return pick_d<uint8_t, RKV_I8>(D, G, P, append);
}

}  // namespace rkv
