// fft.h -- launch descriptor of the Stockham FFT over a line set.
#pragma once
#include <cstdint>
#include <vector>

#include "dmx.h"

namespace dmx {

#define FFT_THREADS 256
#define FFT_MAXEL32 8192  // 64 KiB of complex float per workgroup
#define FFT_MAXEL64 4096  // 64 KiB of complex double per workgroup
#define FFT_MAXPASS 24
#define FFT_MIN_GROUPS 512  // workgroups that small line sets aim at
// butterflies per thread and pass for workgroups of at most MAXEL elements;
// of the wide composite radices only as many as MAXEL fills (the host uses
// them for workgroups that this covers)
constexpr int fft_km(int maxel, int R) {
  const int d = R * FFT_THREADS;
  if (R == 12 || R == 14 || R == 15) return maxel >= d ? maxel / d : 1;
  return (maxel + d - 1) / d;
}

// Constants of one Stockham pass, computed on the host: radix, butterflies
// per line (L/R), sub-transform length before the pass (Ns), twiddle stride
// L/(Ns*R), and float reciprocals for the division-free index math.
struct FftPass {
  int radix, nbf, ns, twstep;
  float inv_nbf, inv_ns;
};
// Lines along one axis of a row-major array.  Line (u, v) starts at
// U(u)*st_u + V(v)*st_v, element k at + k*st_ax, where the virtual indices
// map to actual ones through at most two ranges:
// U(u) = u < un1 ? ua1 + u : ua2 + (u - un1)   (same for V).
struct FftLaunch {
  void *data;       // result (and input, in place)
  const void *src;  // input at the same positions (null: data)
  double scale = 1.0;  // the input's factor
  const void *tw;  // exp(-2 pi i m / L), m < L, compute type
  int L, npass, sign;
  FftPass pass[FFT_MAXPASS];
  int64_t st_ax, st_u, st_v;
  int nu, nv;
  int un1, ua1, ua2, vn1, va1, va2;
  // elements kn1 <= k < ka2 are read as zero (the input is known to vanish
  // there)
  int kprune, kn1, ka2;
  // elements sn1 <= k < sa2 of the result are not stored (no later pass
  // reads them)
  int sprune, sn1, sa2;
};

// Crop + deconvolution of type 1 fused into the last column pass of a 2-D
// transform: the retained mode at grid (row, column) goes to the uniform
// array (strides ust0, ust1 in elements; complex128 if u_f64), times the
// FP64 correction factors cf0[|n0/2 - i0|] * cf1[|n1/2 - i1|]
// (comp_indices, nufft.h:142-151).
struct FftCrop {
  void *uni;
  const double *cf0, *cf1;
  int64_t ust0, ust1;
  int n0, N0, n1, N1;
  int fft_order, u_f64;
};

// One launch of k_fft: nv lines b (virtual -> actual through a range, as
// above) for every u (blockIdx.y) and outer index (blockIdx.z).  Element e
// of a line is read at src + z*st_o + u*in_u + b*in_b + e*in_e and has the
// natural index u*nin_u + b*nin_b + e*nin_e (zero in the k range); result k goes to dst
// with the out_ / nout_ numbers (not stored in the s range), times w_L^(k * u) (twiddle 1) or
// w_L^(k * b) (twiddle 2), or through the crop.
struct FftArgs {
  const void *src;
  void *dst;
  const void *tw;       // twiddles of length Ls
  const void *tw_full;  // twiddles of length L (twiddle)
  double scale = 1.0;   // factor of the input
  int Ls, LP, Bl, npass;
  FftPass pass[FFT_MAXPASS];
  int nv, vn1, va1, va2;
  int un1, ua1, ua2;
  int on1, oa1, oa2;
  int64_t in_b, in_e, in_u, out_b, out_k, out_u, st_o;
  int nin_b, nin_e, nin_u, nout_b, nout_k, nout_u;
  int kn1, kspan, sn1, sspan;  // pruned: [kn1, kn1 + kspan), ...
  int twiddle, tw_lds;
  // butterflies dealt with the line index running fastest (lines side by
  // side in memory) in the first, middle and last passes
  int bf_in, bf_mid, bf_out;
  int crop;
  FftCrop cr;
};

// FFT of length L = L1*L2 along a strided axis, as two coalesced passes:
// A: length-L1 FFTs over rows n1*L2+n2, times w_L^{n2 k1}, in place (or,
// with `a_dst`, from p.data into a_dst at the same positions);
// B: length-L2 FFTs over rows k1*L2+n2 of A's output, written to row
// k1 + L1*k2 of dst, i.e. in natural order (dst may be p.data when a_dst is
// given: the result then replaces the input; with `crop`, pass B writes the
// retained modes to the uniform array instead, see FftCrop).  Returns false
// when L has no split worth using.
bool fft_columns_2pass(const FftLaunch &p, int L1, void *dst, bool fp64,
                       const void *tw_L1, const void *tw_L2,
                       const void *tw_L, hipStream_t s,
                       void *a_dst = nullptr, const FftCrop *crop = nullptr);
// a divisor of L near sqrt(L) with both factors <= 128 (0: none)
int fft_split(int L);

// The same over contiguous lines (st_ax == 1) too long for LDS, or too few
// to fill the chip one workgroup a line; natural order in and out, pass A in
// place (or into a_dst), dst must not be pass A's output.
bool fft_long_2pass(const FftLaunch &p, int L1, void *dst, bool fp64,
                    const void *tw_L1, const void *tw_L2, const void *tw_L,
                    hipStream_t s, void *a_dst = nullptr);
// the divisor of L that fft_long_2pass takes (0: none)
int fft_split_long(int L, bool fp64);

void fft_twiddles(int L, bool fp64, std::vector<unsigned char> &out);
// the same table computed on the device into dst (L complex values of the
// compute type), for callers that make no host-to-device copies
void launch_fft_twiddles(void *dst, int L, bool fp64, hipStream_t s);
// Runs the FFT over every line of the set (in place).  `scratch` must be as
// large as the array when L exceeds the LDS capacity.
void fft_lineset(const FftLaunch &p, bool fp64, void *scratch, hipStream_t s);

}  // namespace dmx
