// The fp8 ring tiles: 128 x 128 block weight scales.
#include "gemm_ring.h"

namespace hn {

int launch_ring_fp8(GemmArgs& a, int epilogue, int out_dtype, hipStream_t st, bool* taken) {
  return launch_ring<HN_KIND_FP8, true, true>(a, epilogue, out_dtype, st, taken);
}

}  // namespace hn
