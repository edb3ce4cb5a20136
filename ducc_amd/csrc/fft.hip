// fft.hip -- hand-written mixed-radix Stockham c2c FFT over the oversampled
// grid (role of c2c / general_nd / cfftp passes, fft.h:848-850,
// fftnd_impl.h:593-, fft1d_impl.h:194-825).  Unnormalised; forward means
// exponent -1.  Grid sizes are 2*(2,3,5,7,11-smooth).
//
// A "line set" is every line along one axis of a row-major 3-D view
// (1-D and 2-D grids get leading unit axes); the two other axes index the
// lines and each may be restricted to the kept bands [0,(n+1)/2) and
// [N-n/2, N), which is the reference's pruned FFT (nufft.h:1287-1298,
// 1345-1356, 1749-1781, 1815-1851).
//
// LDS kernel (k_fft): a workgroup transforms Bl lines.  The first Stockham
// pass reads global memory (coalesced: along the line where it is
// contiguous, across Bl neighbouring lines otherwise), the last one writes
// it, and between them the lines live in LDS with register staging (one
// buffer: read all inputs -> barrier -> write all outputs).  Lines too long
// for LDS, and long columns, take two such passes over a factorization
// L = L1 * L2; what has no such split takes one global-memory Stockham pass
// per radix (out of place).
//
// What bounds it: latency of the dependent sweeps (load, exchanges, store)
// and the vector ALU; so the passes are as few as the radices allow
// (composite radices 6, 9, 10, 12, 14, 15, 16 in registers).
#include <algorithm>
#include <cmath>
#include <vector>

#include "dmx.h"
#include "fft_impl.h"

namespace dmx {

namespace {

// One out-of-place radix-R pass in global memory over all lines of the set.
template <typename T, int R>
__global__ __launch_bounds__(256) void k_fft_global_pass(FftLaunch p,
                                                         const void *src_,
                                                         void *dst_, int Ns) {
  using C = typename V2<T>::t;
  const C *src = (const C *)src_;
  C *dst = (C *)dst_;
  const C *tw = (const C *)p.tw;
  const int L = p.L;
  const int nbf = L / R;
  const int64_t q = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  const int64_t nl = (int64_t)p.nu * p.nv;
  if (q >= nl * nbf) return;
  const int64_t line = q / nbf;
  const int jj = (int)(q - line * nbf);
  const int u = (int)(line / p.nv), v = (int)(line - (int64_t)u * p.nv);
  const int64_t base = map_range(u, p.un1, p.ua1, p.ua2) * p.st_u +
                       map_range(v, p.vn1, p.va1, p.va2) * p.st_v;
  C x[R];
#pragma unroll
  for (int r = 0; r < R; ++r) {
    x[r] = src[base + (int64_t)(jj + r * nbf) * p.st_ax];
    x[r].x *= (T)p.scale;
    x[r].y *= (T)p.scale;
  }
  if (R > 1) {
    const int kk = jj % Ns;
    const int twstep = L / (Ns * R);
    if (Ns > 1) {
#pragma unroll
      for (int r = 1; r < R; ++r) {
        C w = tw[(int64_t)r * kk * twstep];
        if (p.sign > 0) w.y = -w.y;
        x[r] = cmul(x[r], w);
      }
    }
    dft<T, R>(x, p.sign);
    const int ob = (jj / Ns) * Ns * R + kk;
#pragma unroll
    for (int r = 0; r < R; ++r)
      dst[base + (int64_t)(ob + r * Ns) * p.st_ax] = x[r];
  } else {
    dst[base + (int64_t)jj * p.st_ax] = x[0];
  }
}

}  // namespace

namespace {
// Radices of the passes of a line of length L: the fewest passes (each is a
// sweep over LDS and two barriers), then the smallest radices.  allow: bit
// R set for each usable radix.  In LDS odd radices come first: the first pass
// writes its results R elements apart, free of bank conflicts for odd R.  In
// global memory the even ones do, so that the early passes write whole
// aligned segments (2000376 = 8 7^3 3^6 in FP64: the call's ten passes 284 ->
// 261 us).
constexpr uint32_t GLOBAL_RADICES =
    1u << 11 | 1u << 8 | 1u << 7 | 1u << 5 | 1u << 4 | 1u << 3 | 1u << 2;
constexpr int RADICES[14] = {16, 15, 14, 12, 11, 10, 9, 8, 7, 6, 5, 4, 3, 2};
void search_radices(int L, int from, int n, int sum, uint32_t allow,
                    int *cur, int *best, int &nbest, int &sbest) {
  if (L == 1) {
    if (n < nbest || (n == nbest && sum < sbest)) {
      nbest = n;
      sbest = sum;
      std::copy(cur, cur + n, best);
    }
    return;
  }
  if (n >= nbest || n >= FFT_MAXPASS) return;
  for (int i = from; i < 14; ++i) {
    const int R = RADICES[i];
    if (L % R || !((allow >> R) & 1)) continue;
    // even with R in every remaining pass: too many passes
    int64_t reach = 1;
    for (int k = n; k < nbest; ++k) reach = std::min<int64_t>(reach * R, L);
    if (reach < L) break;
    cur[n] = R;
    search_radices(L / R, i, n + 1, sum + R, allow, cur, best, nbest, sbest);
  }
}

int plan_passes(int L, uint32_t allow, FftPass *pass, bool lds = true) {
  int cur[FFT_MAXPASS], f[FFT_MAXPASS], n = FFT_MAXPASS + 1, sum = 0;
  search_radices(L, 0, 0, 0, allow, cur, f, n, sum);
  DMX_ASSERT(n <= FFT_MAXPASS, "FFT length is not 2,3,5,7,11-smooth");
  std::stable_sort(f, f + n, [lds](int a, int b) {
    const bool oa = a & 1, ob = b & 1;
    if (oa != ob) return lds ? oa : ob;
    return lds || !oa ? a > b : a < b;
  });
  int Ns = 1;
  for (int i = 0; i < n; ++i) {
    FftPass &q = pass[i];
    q.radix = f[i];
    q.nbf = L / f[i];
    q.ns = Ns;
    q.twstep = L / (Ns * f[i]);
    q.inv_nbf = 1.0f / (float)q.nbf;
    q.inv_ns = 1.0f / (float)Ns;
    Ns *= f[i];
  }
  return n;
}

// usable radices of a workgroup with nel elements in the MAXEL variant
uint32_t radices_for(int maxel, int nel) {
  uint32_t m = 0;
  for (int R : RADICES)
    if ((int64_t)fft_km(maxel, R) * R * FFT_THREADS >= nel) m |= 1u << R;
  return m;
}

void launch_fft(FftArgs &a, bool fp64, int sign, unsigned ny, unsigned nz,
                hipStream_t s) {
  const int full = fp64 ? FFT_MAXEL64 : FFT_MAXEL32;
  const int nel = a.Bl * a.Ls;
  const bool half = nel <= full / 2;
  a.LP = a.Bl > 1 ? a.Ls | 1 : a.Ls;
  a.npass = plan_passes(a.Ls, radices_for(half ? full / 2 : full, nel),
                        a.pass);
  const size_t sh = ((size_t)a.Bl * a.LP + (a.tw_lds ? a.Ls : 0)) *
                    (fp64 ? 16 : 8);
  const dim3 grid((unsigned)((a.nv + a.Bl - 1) / a.Bl), ny, nz);
  DMX_ASSERT(ny <= 65535 && nz <= 65535, "FFT line set too large");
  if (fp64) {
    if (half) launch_k_fft<double, FFT_MAXEL64 / 2>(a, sign, grid, sh, s);
    else launch_k_fft<double, FFT_MAXEL64>(a, sign, grid, sh, s);
  } else {
    if (half) launch_k_fft<float, FFT_MAXEL32 / 2>(a, sign, grid, sh, s);
    else launch_k_fft<float, FFT_MAXEL32>(a, sign, grid, sh, s);
  }
}
}  // namespace

void fft_twiddles(int L, bool fp64, std::vector<unsigned char> &out) {
  // exp(-2 pi i m / L), m = 0..L-1, computed in double
  const double pi = 3.141592653589793238462643383279502884197;
  size_t esz = fp64 ? 16 : 8;
  out.resize((size_t)L * esz);
  for (int m = 0; m < L; ++m) {
    // reduce the angle to the first octant-symmetric form for accuracy
    double c, s;
    long mm = m;
    // use sincospi-like evaluation on 2m/L in [0,2)
    double x = 2.0 * (double)mm / (double)L;
    if (x > 1.0) x -= 2.0;  // (-1, 1]
    c = std::cos(pi * x);
    s = -std::sin(pi * x);
    if (4 * (long)m == (long)L) { c = 0; s = -1; }
    if (2 * (long)m == (long)L) { c = -1; s = 0; }
    if (4 * (long)m == 3 * (long)L) { c = 0; s = 1; }
    if (fp64) {
      double *p = (double *)out.data() + 2 * (size_t)m;
      p[0] = c; p[1] = s;
    } else {
      float *p = (float *)out.data() + 2 * (size_t)m;
      p[0] = (float)c; p[1] = (float)s;
    }
  }
}

namespace {
__global__ void k_twiddles(void *out, int L, int fp64) {
  const int m = blockIdx.x * blockDim.x + threadIdx.x;
  if (m >= L) return;
  double x = 2.0 * (double)m / (double)L;
  if (x > 1.0) x -= 2.0;  // (-1, 1]
  double sn, c;
  sincospi(x, &sn, &c);
  double s = -sn;
  if (4 * (long)m == (long)L) { c = 0; s = -1; }
  if (2 * (long)m == (long)L) { c = -1; s = 0; }
  if (4 * (long)m == 3 * (long)L) { c = 0; s = 1; }
  if (fp64)
    ((double2 *)out)[m] = make_double2(c, s);
  else
    ((float2 *)out)[m] = make_float2((float)c, (float)s);
}
}  // namespace

void launch_fft_twiddles(void *dst, int L, bool fp64, hipStream_t s) {
  if (L <= 0) return;
  hipLaunchKernelGGL(k_twiddles, dim3((L + 255) / 256), dim3(256), 0, s, dst,
                     L, fp64 ? 1 : 0);
  DMX_HIP(hipGetLastError());
}

int fft_split(int L) {
  int best = 0;
  for (int d = 2; d * d <= L; ++d)
    if (L % d == 0 && L / d <= 128) best = d;
  return best;
}

bool fft_columns_2pass(const FftLaunch &p, int L1, void *dst, bool fp64,
                       const void *tw_L1, const void *tw_L2,
                       const void *tw_L, hipStream_t s, void *a_dst,
                       const FftCrop *crop) {
  const int L = p.L, L2 = L / L1;
  if (L1 < 2 || L2 < 2 || L1 * L2 != L || p.st_v != 1) return false;
  const int maxel = fp64 ? FFT_MAXEL64 : FFT_MAXEL32;
  // columns per workgroup: at least 32 (coalesced row segments), within
  // half the LDS budget when that allows 32 (more workgroups per CU)
  const int Lm = std::max(L1, L2);
  int Bl = (maxel / 2 - Lm) / (Lm + 1);
  if (Bl < 32) Bl = (maxel - Lm) / (Lm + 1);
  Bl = std::min(Bl, fp64 ? 32 : 64);
  if (Bl > (fp64 ? 8 : 16)) Bl -= Bl % (fp64 ? 8 : 16);  // whole cache lines
  Bl = std::max(1, std::min(Bl, p.nv));
  FftArgs c{};
  c.Bl = Bl;
  c.nv = p.nv;
  c.vn1 = p.vn1; c.va1 = p.va1; c.va2 = p.va2;
  c.on1 = p.un1; c.oa1 = p.ua1; c.oa2 = p.ua2;
  c.st_o = p.st_u;
  c.in_b = c.out_b = 1;
  c.tw_full = tw_L;
  c.tw_lds = 1;
  c.bf_in = c.bf_mid = c.bf_out = 1;
  const int64_t rs = p.st_ax;
  // pass A: length L1 over rows n1*L2+n2, twiddled (in place unless a_dst)
  void *amid = a_dst ? a_dst : p.data;
  c.src = p.src ? p.src : p.data;
  c.scale = p.scale;
  c.dst = amid;
  c.Ls = L1;
  c.tw = tw_L1;
  c.twiddle = 1;
  // pass A reads natural order: known-zero input rows as asked
  c.kn1 = p.kn1;
  c.kspan = p.kprune ? p.ka2 - p.kn1 : 0;
  c.nin_u = 1; c.nin_e = L2;
  c.in_u = rs; c.in_e = L2 * rs; c.out_u = rs; c.out_k = L2 * rs;
  c.un1 = L2;
  launch_fft(c, fp64, p.sign, (unsigned)L2, (unsigned)p.nu, s);
  // pass B: length L2 over rows k1*L2+n2, to row k1 + L1*k2 of dst
  c.src = amid;
  c.scale = 1.0;
  c.dst = dst;
  c.Ls = L2;
  c.tw = tw_L2;
  c.twiddle = 0;
  c.in_u = L2 * rs; c.in_e = rs; c.out_u = rs; c.out_k = L1 * rs;
  c.nout_u = 1; c.nout_k = L1;
  c.un1 = L1;
  c.kspan = 0;
  if (crop) {
    c.crop = 1;
    c.cr = *crop;
  }
  // pass B writes natural order: prune as asked
  c.sn1 = p.sn1;
  c.sspan = p.sprune ? p.sa2 - p.sn1 : 0;
  launch_fft(c, fp64, p.sign, (unsigned)L1, (unsigned)p.nu, s);
  return true;
}

int fft_split_long(int L, bool fp64) {
  // both factors with at least four lines of LDS
  const int most = (fp64 ? FFT_MAXEL64 : FFT_MAXEL32) / 4;
  int best = 0;
  for (int d = 2; d * d <= L; ++d)
    if (L % d == 0 && L / d <= most) best = d;
  return best;
}

// Contiguous lines as two passes over the L1 x L2 view of each line
// (element n1 * L2 + n2): A transforms the columns, neighbouring n2 side by
// side, B the rows, whose results k1 + L1 * k2 lie side by side for
// neighbouring k1; both passes read and write runs of neighbours.  The
// general alternative is one trip through memory per radix.  A launch's
// second and third index hold 65535 lines each: a larger set takes several
// pairs of launches.
bool fft_long_2pass(const FftLaunch &p, int L1, void *dst, bool fp64,
                    const void *tw_L1, const void *tw_L2, const void *tw_L,
                    hipStream_t s, void *a_dst) {
  const int L = p.L, L2 = L / L1;
  if (L1 < 2 || L1 * L2 != L || p.st_ax != 1) return false;
  const int maxel = fp64 ? FFT_MAXEL64 : FFT_MAXEL32, seg = fp64 ? 8 : 16;
  auto lines = [&](int Ls, int n) {
    int Bl = std::min(maxel / Ls, std::max(seg, maxel / 2 / Ls));
    const int64_t few = (int64_t)n * p.nu * p.nv / (FFT_MIN_GROUPS / 2);
    Bl = (int)std::min<int64_t>(Bl, std::max<int64_t>(seg / 4, few));
    return std::max(1, std::min(Bl, n));
  };
  void *amid = a_dst ? a_dst : p.data;
  constexpr int MOST = 65535;
  // lines (u0 + i, v0 + j) of the set, i < nu, j < nv
  auto part = [&](int u0, int nu, int v0, int nv) {
    FftArgs c{};
    c.un1 = p.un1 - u0; c.ua1 = p.ua1 + u0; c.ua2 = p.ua2;
    c.on1 = p.vn1 - v0; c.oa1 = p.va1 + v0; c.oa2 = p.va2;
    c.st_o = p.st_v;
    c.in_u = c.out_u = p.st_u;
    c.tw_full = tw_L;
    c.bf_in = c.bf_mid = c.bf_out = 1;
    c.src = p.src ? p.src : p.data;
    c.scale = p.scale;
    c.dst = amid;
    c.Ls = L1;
    c.tw = tw_L1;
    c.twiddle = 2;
    c.nv = c.vn1 = L2;
    c.Bl = lines(L1, L2);
    c.in_b = c.out_b = 1;
    c.in_e = c.out_k = L2;
    c.kn1 = p.kn1; c.kspan = p.kprune ? p.ka2 - p.kn1 : 0;
    c.nin_b = 1; c.nin_e = L2;
    launch_fft(c, fp64, p.sign, (unsigned)nu, (unsigned)nv, s);
    c.src = amid;
    c.scale = 1.0;
    c.dst = dst;
    c.Ls = L2;
    c.tw = tw_L2;
    c.twiddle = 0;
    c.nv = c.vn1 = L1;
    c.Bl = lines(L2, L1);
    c.in_b = L2;
    c.in_e = 1;
    c.out_b = 1;
    c.out_k = L1;
    c.kspan = 0;
    c.nout_b = 1; c.nout_k = L1;
    c.sn1 = p.sn1; c.sspan = p.sprune ? p.sa2 - p.sn1 : 0;
    c.bf_in = 0;
    launch_fft(c, fp64, p.sign, (unsigned)nu, (unsigned)nv, s);
  };
  for (int u0 = 0; u0 < p.nu; u0 += MOST)
    for (int v0 = 0; v0 < p.nv; v0 += MOST)
      part(u0, std::min(MOST, p.nu - u0), v0, std::min(MOST, p.nv - v0));
  return true;
}

void fft_lineset(const FftLaunch &base, bool fp64, void *scratch,
                 hipStream_t s) {
  FftLaunch p = base;
  if (p.nu <= 0 || p.nv <= 0 || p.L <= 1) return;
  const int maxel = fp64 ? FFT_MAXEL64 : FFT_MAXEL32;
  if (p.L <= maxel) {
    // lines per workgroup: contiguous ones within half the LDS budget, so
    // that several workgroups per CU overlap their loads with the passes of
    // the others; strided ones at least a 128-byte line of neighbours.  A
    // small set is spread over more workgroups, down to one contiguous line
    // or half a cache line of strided ones.
    const int seg = fp64 ? 8 : 16;
    int Bl = std::max(1, (maxel / 2) / p.L);
    if (p.st_ax != 1 && Bl < seg) Bl = std::max(Bl, std::min(seg, maxel / p.L));
    const int64_t lines = (int64_t)p.nu * p.nv;
    const int64_t few = std::max<int64_t>(p.st_ax == 1 ? 1 : seg / 2,
                                          lines / FFT_MIN_GROUPS);
    Bl = (int)std::min<int64_t>(Bl, few);
    Bl = std::max(1, std::min(Bl, p.nv));
    FftArgs c{};
    c.src = p.src ? p.src : p.data;
    c.scale = p.scale;
    c.dst = p.data;
    c.tw = p.tw;
    c.Ls = p.L;
    c.Bl = Bl;
    c.nv = p.nv;
    c.vn1 = p.vn1; c.va1 = p.va1; c.va2 = p.va2;
    c.un1 = p.un1; c.ua1 = p.ua1; c.ua2 = p.ua2;
    c.on1 = 1;
    c.in_b = c.out_b = p.st_v;
    c.in_e = c.out_k = p.st_ax;
    c.in_u = c.out_u = p.st_u;
    c.nin_e = c.nout_k = 1;
    c.kn1 = p.kn1; c.kspan = p.kprune ? p.ka2 - p.kn1 : 0;
    c.sn1 = p.sn1; c.sspan = p.sprune ? p.sa2 - p.sn1 : 0;
    c.bf_in = c.bf_mid = c.bf_out = p.st_ax != 1;
    launch_fft(c, fp64, p.sign, (unsigned)p.nu, 1, s);
    return;
  }
  p.npass = plan_passes(p.L, GLOBAL_RADICES, p.pass, false);
  // long lines: global Stockham passes, ping-pong between data and scratch
  DMX_ASSERT(scratch != nullptr, "internal: FFT scratch missing");
  const void *src = p.src ? p.src : p.data;
  void *dst = scratch;
  int Ns = 1;
  auto run = [&](int R) {
    int64_t nthr = (int64_t)p.nu * p.nv * (p.L / R);
    unsigned nb = (unsigned)((nthr + 255) / 256);
#define DMX_GP(TT, RR) \
  hipLaunchKernelGGL((k_fft_global_pass<TT, RR>), dim3(nb), dim3(256), 0, s, p, src, dst, Ns)
    if (fp64) {
      switch (R) {
        case 1: DMX_GP(double, 1); break; case 2: DMX_GP(double, 2); break;
        case 3: DMX_GP(double, 3); break; case 4: DMX_GP(double, 4); break;
        case 8: DMX_GP(double, 8); break;
        case 5: DMX_GP(double, 5); break; case 7: DMX_GP(double, 7); break;
        case 11: DMX_GP(double, 11); break;
      }
    } else {
      switch (R) {
        case 1: DMX_GP(float, 1); break; case 2: DMX_GP(float, 2); break;
        case 3: DMX_GP(float, 3); break; case 4: DMX_GP(float, 4); break;
        case 8: DMX_GP(float, 8); break;
        case 5: DMX_GP(float, 5); break; case 7: DMX_GP(float, 7); break;
        case 11: DMX_GP(float, 11); break;
      }
    }
#undef DMX_GP
    DMX_HIP(hipGetLastError());
    src = dst;
    dst = dst == p.data ? scratch : p.data;
    p.scale = 1.0;
  };
  // out of place: start so that the last pass writes the data array
  if (src != p.data && p.npass % 2 == 1) dst = p.data;
  for (int i = 0; i < p.npass; ++i) {
    run(p.pass[i].radix);
    Ns *= p.pass[i].radix;
  }
  if (src != p.data) {
    // odd number of passes: copy back with an identity pass
    Ns = 1;
    run(1);
  }
}

}  // namespace dmx
