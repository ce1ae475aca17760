// conv_x3_inst.hip — the three-part stride-1 convolution kernel of conv_x3_body.h, compiled eight
// times, -DTDH_X3_PART=0..7: windows of 1, 3, 5 and 7, with 16-byte and scalar loads.
#include "conv_x3_body.h"

namespace tdh {

namespace {

// POOL: a 2x2 max-pool in rows of 32, in an instance of its own: its code behind the products made the others, which pool
// nothing, up to 3 % slower (dX, us without / with: 32x32, 16 -> 16 channels, 3x3, 256 images 19.8 / 20.4; 40x40, 32 <- 64, 128 images 80.5 / 82.0).
// (In the fp32 kernel the same gained nothing: 0.998 to 1.022 over 150 drawn layers.)
template <int R, int S, int TC, int TM, int TN, bool VEC, bool POOL>
__global__ void __launch_bounds__(256, 2) conv_x3_kernel(const ConvS1Args a) {
  conv_x3_workgroup<R, S, TC, TM, TN, VEC, false, POOL>(a, blockIdx.x, blockIdx.y, blockIdx.z);
}

template <int R, int S, int TC, int TM, int TN, bool VEC, bool POOL = false>
int launch_x3_inst(const S1Plan &p) {
  if constexpr (TC == 32 && TN == 2 && !POOL) {
    if (p.args.pool_out) return launch_x3_inst<R, S, TC, TM, TN, VEC, true>(p);
  }
  auto kernel = conv_x3_kernel<R, S, TC, TM, TN, VEC, POOL>;
  if (p.lds_bytes > 64 * 1024) {
    static size_t raised = 0;
    if (p.lds_bytes > raised) {
      TDH_HIP(hipFuncSetAttribute(reinterpret_cast<const void *>(kernel), hipFuncAttributeMaxDynamicSharedMemorySize,
                                  static_cast<int>(p.lds_bytes)));
      raised = p.lds_bytes;
    }
  }
  TDH_LAUNCH(kernel, p.grid, dim3(256), p.lds_bytes, ctx().stream, p.args);
  TDH_LAUNCH_CHECK();
  return TDH_OK;
}

template <int R, int S, int TC, bool VEC>
int launch_x3_tc(const S1Plan &p) {
  switch (p.tm * 10 + p.tn) {
    case 22: return launch_x3_inst<R, S, TC, 2, 2, VEC>(p);
    case 21: return launch_x3_inst<R, S, TC, 2, 1, VEC>(p);
    default: return launch_x3_inst<R, S, TC, 1, 2, VEC>(p);
  }
}

template <int R, int S, bool VEC>
int launch_x3_rs(const S1Plan &p) {
  switch (p.tc) {
    case 64: return launch_x3_tc<R, S, 64, VEC>(p);
    case 32: return launch_x3_tc<R, S, 32, VEC>(p);
    case 16: return launch_x3_tc<R, S, 16, VEC>(p);
    default: return launch_x3_tc<R, S, 8, VEC>(p);
  }
}

}  // namespace

#define X3_JOIN_(a, b, c, d) a##b##c##d
#define X3_JOIN(a, b, c, d) X3_JOIN_(a, b, c, d)
#if TDH_X3_PART < 2
#define X3_WINDOW 1
#elif TDH_X3_PART < 4
#define X3_WINDOW 3
#elif TDH_X3_PART < 6
#define X3_WINDOW 5
#else
#define X3_WINDOW 7
#endif
#if TDH_X3_PART % 2 == 0
int X3_JOIN(x3_launch_, X3_WINDOW, _, vec)(const S1Plan &p) { return launch_x3_rs<X3_WINDOW, X3_WINDOW, true>(p); }
#else
int X3_JOIN(x3_launch_, X3_WINDOW, _, scalar)(const S1Plan &p) { return launch_x3_rs<X3_WINDOW, X3_WINDOW, false>(p); }
#endif

}  // namespace tdh
