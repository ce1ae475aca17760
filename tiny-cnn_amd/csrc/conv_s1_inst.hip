// conv_s1_inst.hip — the stride-1 convolution kernel of conv_s1_body.h, compiled four times,
// -DTDH_S1_PART=0..3: 3x3 and 5x5 windows, each with 16-byte and with scalar loads.
#include "conv_s1_body.h"

namespace tdh {

namespace {

template <int R, int S, int TC, int TM, int TN, bool VEC>
__global__ void __launch_bounds__(256, 2) conv_s1_kernel(const ConvS1Args a) {
  extern __shared__ __align__(16) float smem[];
  conv_s1_workgroup<R, S, TC, TM, TN, VEC>(a, smem, blockIdx.x, blockIdx.y, blockIdx.z);
}

template <int R, int S, int TC, int TM, int TN, bool VEC>
int launch_s1_inst(const S1Plan &p) {
  auto kernel = conv_s1_kernel<R, S, TC, TM, TN, VEC>;
  if (p.lds_bytes > 64 * 1024) {
    // raised once per kernel instance and size: the default dynamic LDS limit is 64 KiB
    static size_t raised = 0;
    if (p.lds_bytes > raised) {
      TDH_HIP(hipFuncSetAttribute(reinterpret_cast<const void *>(kernel),
                                  hipFuncAttributeMaxDynamicSharedMemorySize,
                                  static_cast<int>(p.lds_bytes)));
      raised = p.lds_bytes;
    }
  }
  TDH_LAUNCH(kernel, p.grid, dim3(256), p.lds_bytes, ctx().stream, p.args);
  TDH_LAUNCH_CHECK();
  return TDH_OK;
}

template <int R, int S, int TC, bool VEC>
int launch_s1_tc(const S1Plan &p) {
  switch (p.tm * 10 + p.tn) {
    case 22: return launch_s1_inst<R, S, TC, 2, 2, VEC>(p);
    case 21: return launch_s1_inst<R, S, TC, 2, 1, VEC>(p);
    case 14: return launch_s1_inst<R, S, TC, 1, 4, VEC>(p);
    case 12: return launch_s1_inst<R, S, TC, 1, 2, VEC>(p);
    default: return launch_s1_inst<R, S, TC, 1, 1, VEC>(p);
  }
}

template <int R, int S, bool VEC>
int launch_s1_rs(const S1Plan &p) {
  switch (p.tc) {
    case 64: return launch_s1_tc<R, S, 64, VEC>(p);
    case 32: return launch_s1_tc<R, S, 32, VEC>(p);
    case 16: return launch_s1_tc<R, S, 16, VEC>(p);
    default: return launch_s1_tc<R, S, 8, VEC>(p);
  }
}

}  // namespace

#if TDH_S1_PART == 0
int s1_launch_3x3_vec(const S1Plan &p) { return launch_s1_rs<3, 3, true>(p); }
#elif TDH_S1_PART == 1
int s1_launch_3x3_scalar(const S1Plan &p) { return launch_s1_rs<3, 3, false>(p); }
#elif TDH_S1_PART == 2
int s1_launch_5x5_vec(const S1Plan &p) { return launch_s1_rs<5, 5, true>(p); }
#elif TDH_S1_PART == 3
int s1_launch_5x5_scalar(const S1Plan &p) { return launch_s1_rs<5, 5, false>(p); }
#else
#error "TDH_S1_PART must be 0..3"
#endif

}  // namespace tdh
