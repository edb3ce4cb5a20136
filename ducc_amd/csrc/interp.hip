// interp.hip -- instantiation and launch of the type-2 interpolation kernels
// and of the kernel-derivative interpolation used for coordinate gradients.
#include "spread_impl.h"

namespace dmx {

namespace {
constexpr unsigned INTERP_MAX_BLOCKS = 8192;

// 3-D: 512 threads instead of 256 share a region.
// * 16^3 tiles (on request): always, once the region exceeds a third of the
//   LDS (W = 4, 6 in FP32: 3-4 % and 11-19 % faster; W = 5 in FP64: 15-27 %).
// * 8^3 tiles: only where one region alone fits a CU, which then has eight
//   waves instead of four: FP64 gradients with W = 10 to 13.  96x100x108
//   modes, 256 -> 512 threads: W = 11 and 12 gain at any density (1e6
//   clustered points 2.69 -> 2.11 ms, 1e6 uniform 5.41 -> 5.12, 6e6 uniform
//   10.3 -> 7.2); W = 10 and 13 gain at 250 points a tile (6.62 -> 5.57 and
//   16.0 -> 12.1 ms) and lose at 40 (3.59 -> 3.96 and 8.31 -> 8.60).  Where
//   two regions fit, one workgroup of 512 threads takes the registers of
//   two: W = 8 values 0.57 -> 0.65 ms, gradients of W = 8 and 9 1.50 -> 2.37
//   and 1.83 -> 3.07 ms.
// * 4^3 tiles (W >= 14) have too few points for them (5 % slower).
bool wide_workgroup(const SpreadArgs &a, size_t sh) {
  if (a.g.ndim != 3 || sh <= LDS_MAX_BYTES / 3) return false;
  if (a.g.log2tile != 3) return a.g.log2tile > 3;
  if (sh <= LDS_MAX_BYTES / 2 || a.g.W < 10) return false;
  if (a.g.W == 11 || a.g.W == 12) return true;
  // a hundred points a tile: subproblems beyond one per tile
  const size_t nt = (size_t)a.g.ntiles[0] * a.g.ntiles[1] * a.g.ntiles[2];
  return a.nsub_max > nt + nt * 100 / MAXSUB;
}

template <typename T, int NDIM, int W, int MODE>
void go(const SpreadArgs &a, void *out, int out_f64, hipStream_t s) {
  unsigned nb = (unsigned)std::min<size_t>(a.nsub_max, INTERP_MAX_BLOCKS);
  if (nb == 0) return;
  // 3-D FP64 values with W >= 9 in LDS are launch_interp_wave's
  constexpr bool wave = NDIM == 3 && sizeof(T) == 8 && MODE == 0 && W >= 9;
  if (a.use_lds) {
    if constexpr (wave) {
      throw Error("internal: region of a wide kernel beyond LDS");
    } else {
      size_t cells = interp_inner_pad(a.lds_side);
      for (int d = 1; d < NDIM; ++d) cells *= a.lds_side;
      size_t sh = 2 * cells * sizeof(T);
      if constexpr (NDIM == 3) {
        if (wide_workgroup(a, sh)) {
          allow_big_lds(k_interp<T, NDIM, W, true, MODE, 512>, sh);
          hipLaunchKernelGGL((k_interp<T, NDIM, W, true, MODE, 512>),
                             dim3(nb), dim3(512), sh, s, a, out, out_f64);
          DMX_HIP(hipGetLastError());
          return;
        }
      }
      allow_big_lds(k_interp<T, NDIM, W, true, MODE>, sh);
      hipLaunchKernelGGL((k_interp<T, NDIM, W, true, MODE>), dim3(nb),
                         dim3(256), sh, s, a, out, out_f64);
    }
  } else {
    if constexpr (NDIM == 3)
      hipLaunchKernelGGL((k_interp<T, NDIM, W, false, MODE>), dim3(nb),
                         dim3(256), 0, s, a, out, out_f64);
    else
      throw Error("internal: no-LDS interpolation only for 3D");
  }
  DMX_HIP(hipGetLastError());
}

template <typename T, int NDIM, int MODE>
void by_w(const SpreadArgs &a, void *out, int f64, hipStream_t s) {
  switch (a.g.W) {
    case 4: return go<T, NDIM, 4, MODE>(a, out, f64, s);
    case 5: return go<T, NDIM, 5, MODE>(a, out, f64, s);
    case 6: return go<T, NDIM, 6, MODE>(a, out, f64, s);
    case 7: return go<T, NDIM, 7, MODE>(a, out, f64, s);
    case 8: return go<T, NDIM, 8, MODE>(a, out, f64, s);
    default: break;
  }
  if constexpr (sizeof(T) == 8) {
    switch (a.g.W) {
      case 9: return go<T, NDIM, 9, MODE>(a, out, f64, s);
      case 10: return go<T, NDIM, 10, MODE>(a, out, f64, s);
      case 11: return go<T, NDIM, 11, MODE>(a, out, f64, s);
      case 12: return go<T, NDIM, 12, MODE>(a, out, f64, s);
      case 13: return go<T, NDIM, 13, MODE>(a, out, f64, s);
      case 14: return go<T, NDIM, 14, MODE>(a, out, f64, s);
      case 15: return go<T, NDIM, 15, MODE>(a, out, f64, s);
      case 16: return go<T, NDIM, 16, MODE>(a, out, f64, s);
      default: break;
    }
  }
  throw Error("requested support out of range");
}

template <int MODE>
void dispatch(bool fp64, const SpreadArgs &a, void *out, int f64,
              hipStream_t s) {
  switch (a.g.ndim) {
    case 1:
      return fp64 ? by_w<double, 1, MODE>(a, out, f64, s)
                  : by_w<float, 1, MODE>(a, out, f64, s);
    case 2:
      return fp64 ? by_w<double, 2, MODE>(a, out, f64, s)
                  : by_w<float, 2, MODE>(a, out, f64, s);
    case 3:
      return fp64 ? by_w<double, 3, MODE>(a, out, f64, s)
                  : by_w<float, 3, MODE>(a, out, f64, s);
  }
  throw Error("transform must be 1D/2D/3D");
}
}  // namespace

void launch_interp(bool fp64, const SpreadArgs &a, void *out, int out_f64,
                   hipStream_t s) {
  if (fp64 && launch_interp_wave(a, out, out_f64, s)) return;
  dispatch<0>(fp64, a, out, out_f64, s);
}

void launch_interp_grad(bool fp64, const SpreadArgs &a, void *out,
                        int out_f64, hipStream_t s) {
  dispatch<1>(fp64, a, out, out_f64, s);
}

}  // namespace dmx
