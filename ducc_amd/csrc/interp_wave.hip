// interp_wave.hip -- type-2 interpolation in 3-D with wide FP64 kernels
// (W >= 9): one wave per point instead of one lane per point.
//
// The region of a tile, (tile + W - 1)^3 complex doubles, takes 60-155 KB of
// LDS, so one or two workgroups fit a CU, and W^3 16-byte reads a point make
// LDS the bound.  With one lane per point (k_interp) the lanes read random
// cells (two-way conflicts and more on average), the three weight vectors
// take 6 W registers, which caps the waves in flight, and 1e6 clustered
// points at W = 11 took 1400 us, 1050 us with 512 threads (5 times the
// 270 us of the reads alone).  Here the 64 lanes of a wave own the taps
// (c1, c2) of the W x W plane and walk c0: a read of 64 lanes takes whole
// rows of W neighbouring cells, the row stride is W modulo 16 so that
// consecutive lanes stay on consecutive banks over row ends, each lane
// evaluates one of the 3 W weights (its polynomial stays in registers), and
// 1024 threads fit.  W = 11, 96x100x108 modes, 1e6 points: 713 us (810 us
// with a branch around the last lanes' reads; then also: row stride 19, W
// modulo 8, 845 us, and a subproblem split over two or four workgroups, each
// staging the region, 907 and 1050 us).  Against one lane per point, whole
// calls of uniform points on that grid: W = 9 697 -> 537 us (2e4 points), 2.56
// -> 2.58 ms (6e6); W = 12 1.68 -> 0.65 and 8.9 -> 4.4 ms; W = 15 3.0 -> 0.8
// and 18.0 -> 7.3 ms; W = 16 3.6 -> 0.9 and 28.5 -> 10.5 ms.
#include "spread_impl.h"

namespace dmx {

namespace {

constexpr int WT = 1024;  // threads

// the other lanes' v by a DPP pattern, zero where the pattern has no source
template <int CTRL, int ROWS>
__device__ __forceinline__ double dpp(double v) {
  const int lo = __builtin_amdgcn_update_dpp(0, __double2loint(v), CTRL, ROWS,
                                             0xf, true);
  const int hi = __builtin_amdgcn_update_dpp(0, __double2hiint(v), CTRL, ROWS,
                                             0xf, true);
  return __hiloint2double(hi, lo);
}
// the sum over the wave, in lane 63
__device__ __forceinline__ double wave_sum63(double v) {
  v += dpp<0xB1, 0xf>(v);   // lanes 1 apart
  v += dpp<0x4E, 0xf>(v);   // 2 apart
  v += dpp<0x141, 0xf>(v);  // mirrored halves of 8
  v += dpp<0x140, 0xf>(v);  // mirrored rows of 16: every lane has its row
  v += dpp<0x142, 0xa>(v);  // lane 15 of a row to the next: rows 1 and 3
  v += dpp<0x143, 0xc>(v);  // lane 31 to rows 2 and 3
  return v;
}

__device__ __forceinline__ double lane_value(double v, int lane) {
  return __hiloint2double(
      __builtin_amdgcn_readlane(__double2hiint(v), lane),
      __builtin_amdgcn_readlane(__double2loint(v), lane));
}

// points of a round: kernel arguments (then the result), offsets, index
struct WavePoint {
  double x[3];
  uint32_t o, j;
};

template <int W>
__global__ __launch_bounds__(WT) void k_interp_wave(SpreadArgs a, void *out,
                                                    int out_f64, int SP,
                                                    int chunk) {
  constexpr int NS = (W * W + 63) / 64;  // lane sets of the W x W plane
  constexpr int DP = W + 3 + (W & 1), NE = (DP + 1) / 2, NH = (W + 1) / 2;
  // Lanes past the plane read its last tap and drop the sum: a branch around
  // each of their reads, unrolled W times, spilled 40 to 142 registers a lane
  // at W = 12 to 15.  At W = 14 and 15 that leaves 12 to 15, and the walk with
  // the branch in a loop that is not unrolled is as fast or faster.
  constexpr bool MASK = W == 14 || W == 15;
  constexpr int UN = MASK ? 1 : W;
  extern __shared__ unsigned char smem_raw[];
  const int S = a.lds_side, tile = 1 << a.g.log2tile;
  const int ncell = S * S * SP, plane = S * SP;
  double2 *buf = (double2 *)smem_raw;
  WavePoint *pt = (WavePoint *)(buf + ncell);
  const double2 *grid = (const double2 *)a.grid;
  const int n0 = a.g.nover[0], n1 = a.g.nover[1], n2 = a.g.nover[2];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  // this lane's taps and weight polynomial (axis lane / W, piece lane % W)
  int off[NS], s1[NS], s2[NS];
#pragma unroll
  for (int s = 0; s < NS; ++s) {
    const int q = min(64 * s + lane, W * W - 1);
    off[s] = (q / W) * SP + q % W;
    s1[s] = W + q / W;
    s2[s] = 2 * W + q % W;
  }
  const bool last_in = 64 * (NS - 1) + lane < W * W;
  const int ax = min(lane / W, 2), piece = lane % W;
  const bool mirror = piece >= NH;
  double cf[2 * NE];
  {
    const double *c = (const double *)a.coef;
    const int i = mirror ? W - 1 - piece : piece;
#pragma unroll
    for (int s = 0; s < 2 * NE; ++s) cf[s] = c[s * NH + i];
  }
  const RegionWalk<3> walk0(tid, WT, S, SP);
  const uint32_t total = *a.nsub_total;
  for (uint32_t sidx = blockIdx.x; sidx < total; sidx += gridDim.x) {
    const Sub sb = a.subs[sidx];
    int b0[3];
    tile_origin(a.g, sb.tile, b0);
    {
      // region staging (the cells past S of a row are never read)
      constexpr int STG = 4;
      RegionWalk<3> rw = walk0;
      for (int cb = 0; cb < ncell; cb += STG * WT) {
        double2 v[STG];
#pragma unroll
        for (int k = 0; k < STG; ++k) {
          const bool in = cb + k * WT + tid < ncell;
          const size_t gi = region_grid_index(rw, b0, n0, n1, n2);
          v[k] = grid[in ? gi : 0];
          rw.next();
        }
#pragma unroll
        for (int k = 0; k < STG; ++k) {
          const int c = cb + k * WT + tid;
          if (c < ncell) buf[c] = v[k];
        }
      }
    }
    for (uint32_t c0 = sb.start; c0 < sb.end; c0 += (uint32_t)chunk) {
      const int nc = (int)min((uint32_t)chunk, sb.end - c0);
      if (tid < nc) {
        const uint32_t p = c0 + tid;
        WavePoint w;
        uint32_t o[3];
        if (a.rec) {
          const int L = a.g.log2tile;
          const uint32_t wd = a.recs.word[p];
          w.j = a.recs.j[p];
#pragma unroll
          for (int d = 0; d < 3; ++d) {
            o[d] = (wd >> (d * L)) & ((1u << L) - 1u);
            w.x[d] = ((const double *)a.recs.x[d])[p];
          }
        } else {
          w.j = a.idx[p];
          double x[3];
          load_point(a.g, a.coords, a.coords_sorted ? (size_t)p : (size_t)w.j,
                     3, x);
#pragma unroll
          for (int d = 0; d < 3; ++d) {
            double frac;
            int od = fold_axis(a.g, d, x[d], frac) - b0[d];
            w.x[d] = (double)(W - 1) - 2.0 * frac;
            if (od < 0 || od >= tile) {
              if (a.offcheck) atomicAdd(a.offcheck, 1u);
              od = od < 0 ? 0 : tile - 1;
            }
            o[d] = (uint32_t)od;
          }
        }
        w.o = (o[0] * (uint32_t)S + o[1]) * (uint32_t)SP + o[2];
        pt[tid] = w;
      }
      __syncthreads();  // the region and the points are in LDS
      for (int i = wave; i < nc; i += WT / 64) {
        const double x = pt[i].x[ax], x2 = x * x;
        const int base = __builtin_amdgcn_readfirstlane((int)pt[i].o);
        double od = cf[0], ev = cf[1];
#pragma unroll
        for (int s = 1; s < NE; ++s) {
          od = od * x2 + cf[2 * s];
          ev = ev * x2 + cf[2 * s + 1];
        }
        const double w = mirror ? ev - x * od : ev + x * od;
        double re[NS], im[NS];
#pragma unroll
        for (int s = 0; s < NS; ++s) re[s] = im[s] = 0.0;
        const double2 *b = buf + base;
#pragma unroll UN
        for (int c = 0; c < W; ++c) {
          const double w0 = lane_value(w, c);
#pragma unroll
          for (int s = 0; s < NS; ++s) {
            if (!MASK || s < NS - 1 || last_in) {
              const double2 g = b[c * plane + off[s]];
              re[s] += w0 * g.x;
              im[s] += w0 * g.y;
            }
          }
        }
        double tr = 0.0, ti = 0.0;
#pragma unroll
        for (int s = 0; s < NS; ++s) {
          const double w12 = __shfl(w, s1[s]) * __shfl(w, s2[s]);
          if (s < NS - 1 || last_in) {
            tr += re[s] * w12;
            ti += im[s] * w12;
          }
        }
        tr = wave_sum63(tr);
        ti = wave_sum63(ti);
        if (lane == 63) {
          pt[i].x[0] = tr;
          pt[i].x[1] = ti;
        }
      }
      __syncthreads();
      if (tid < nc)
        store_value<double>(out, pt[tid].j, out_f64, pt[tid].x[0],
                            pt[tid].x[1]);
      // (a thread overwrites only its own point and, after the barrier
      // above, cells nobody reads any more)
    }
  }
}

template <int W>
void go(const SpreadArgs &a, void *out, int out_f64, int SP, int chunk,
        size_t sh, hipStream_t s) {
  allow_big_lds(k_interp_wave<W>, sh);
  const unsigned nb = (unsigned)std::min<size_t>(a.nsub_max, 8192);
  hipLaunchKernelGGL((k_interp_wave<W>), dim3(nb), dim3(WT), sh, s, a, out,
                     out_f64, SP, chunk);
  DMX_HIP(hipGetLastError());
}

}  // namespace

bool launch_interp_wave(const SpreadArgs &a, void *out, int out_f64,
                        hipStream_t s) {
  if (a.g.ndim != 3 || !a.use_lds || a.g.W < 9 || a.g.W > 16) return false;
  // row stride: consecutive taps over a row's end on consecutive banks (16
  // cells; 8 where that leaves no room)
  const int S = a.lds_side;
  auto bytes = [&](int SP) { return (size_t)S * S * SP * sizeof(double2); };
  auto stride = [&](int m) {
    int SP = S;
    while ((SP - a.g.W) % m != 0) ++SP;
    return SP;
  };
  const size_t least = 64 * sizeof(WavePoint);
  int SP = stride(16);
  if (bytes(SP) + least > LDS_MAX_BYTES) SP = stride(8);
  if (bytes(SP) + least > LDS_MAX_BYTES) SP = S;
  const size_t cells = bytes(SP);
  if (cells + least > LDS_MAX_BYTES) return false;
  const int chunk = (int)std::min<size_t>(
      MAXSUB, (LDS_MAX_BYTES - cells) / sizeof(WavePoint) / 64 * 64);
  if (a.nsub_max == 0) return true;
  const size_t sh = cells + (size_t)chunk * sizeof(WavePoint);
  switch (a.g.W) {
    case 9: go<9>(a, out, out_f64, SP, chunk, sh, s); break;
    case 10: go<10>(a, out, out_f64, SP, chunk, sh, s); break;
    case 11: go<11>(a, out, out_f64, SP, chunk, sh, s); break;
    case 12: go<12>(a, out, out_f64, SP, chunk, sh, s); break;
    case 13: go<13>(a, out, out_f64, SP, chunk, sh, s); break;
    case 14: go<14>(a, out, out_f64, SP, chunk, sh, s); break;
    case 15: go<15>(a, out, out_f64, SP, chunk, sh, s); break;
    default: go<16>(a, out, out_f64, SP, chunk, sh, s); break;
  }
  return true;
}

}  // namespace dmx
