// The int8 ring tiles: per-token x per-channel scales, and g128 with one weight-scale row per channel.
#include "gemm_ring.h"

namespace hn {

int launch_ring_int8(GemmArgs& a, bool g128, int epilogue, int out_dtype, hipStream_t st, bool* taken) {
  return g128 ? launch_ring<HN_KIND_INT8, true, false>(a, epilogue, out_dtype, st, taken)
              : launch_ring<HN_KIND_INT8, false, false>(a, epilogue, out_dtype, st, taken);
}

}  // namespace hn
