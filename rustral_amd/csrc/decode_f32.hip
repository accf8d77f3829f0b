// decode_f32.hip -- the decode kernels over fp32 pools.
#include "decode_stream.hpp"

namespace rkv {

Launch decode_f32(int D, int G, int P, bool append) {
  return pick_d<float, RKV_F32>(D, G, P, append);
}

}  // namespace rkv
