// fft_impl.h -- the FFT kernel over a line set staged in LDS (k_fft) and its
// in-register butterflies; instantiated once per compute type and workgroup
// size (fft_f32.hip, fft_f32_half.hip, fft_f64.hip, fft_f64_half.hip, so
// that they compile side by side), described in fft.hip.
#pragma once
#include <cmath>

#include "dmx.h"
#include "fft.h"

namespace dmx {

namespace {

template <typename T> struct V2;
template <> struct V2<float> { using t = float2; };
template <> struct V2<double> { using t = double2; };

template <typename C> __device__ __forceinline__ C cmul(C a, C b) {
  C r;
  r.x = a.x * b.x - a.y * b.y;
  r.y = a.x * b.y + a.y * b.x;
  return r;
}
template <typename C> __device__ __forceinline__ C cadd(C a, C b) {
  C r; r.x = a.x + b.x; r.y = a.y + b.y; return r;
}
template <typename C> __device__ __forceinline__ C csub(C a, C b) {
  C r; r.x = a.x - b.x; r.y = a.y - b.y; return r;
}
// multiply by sign*i
template <typename C> __device__ __forceinline__ C cmuli(C a, int sign) {
  C r;
  if (sign < 0) { r.x = a.y; r.y = -a.x; }
  else { r.x = -a.y; r.y = a.x; }
  return r;
}

// cos/sin(2 pi k / R) for the odd radices
template <int R> struct Tw;
template <> struct Tw<3> {
  static constexpr double c[2] = {-0.5, -0.5};
  static constexpr double s[2] = {0.86602540378443864676, -0.86602540378443864676};
};
template <> struct Tw<5> {
  static constexpr double c[4] = {0.30901699437494742410, -0.80901699437494742410,
                                  -0.80901699437494742410, 0.30901699437494742410};
  static constexpr double s[4] = {0.95105651629515357212, 0.58778525229247312917,
                                  -0.58778525229247312917, -0.95105651629515357212};
};
template <> struct Tw<7> {
  static constexpr double c[6] = {0.62348980185873353053, -0.22252093395631440429,
                                  -0.90096886790241912624, -0.90096886790241912624,
                                  -0.22252093395631440429, 0.62348980185873353053};
  static constexpr double s[6] = {0.78183148246802980871, 0.97492791218182360702,
                                  0.43388373911755812048, -0.43388373911755812048,
                                  -0.97492791218182360702, -0.78183148246802980871};
};
template <> struct Tw<11> {
  static constexpr double c[10] = {
      0.84125353283118116886, 0.41541501300188642553, -0.14231483827328514044,
      -0.65486073394528506406, -0.95949297361449738989, -0.95949297361449738989,
      -0.65486073394528506406, -0.14231483827328514044, 0.41541501300188642553,
      0.84125353283118116886};
  static constexpr double s[10] = {
      0.54064081745559758211, 0.90963199535451837141, 0.98982144188093273238,
      0.75574957435425828377, 0.28173255684142969771, -0.28173255684142969771,
      -0.75574957435425828377, -0.98982144188093273238, -0.90963199535451837141,
      -0.54064081745559758211};
};

// a turned by an angle of tan(angle / 2) = t and sin(angle) = s: three
// shears, each a fused multiply-add that rounds once
template <typename T, typename C>
__device__ __forceinline__ C shear3(C a, T t, T s) {
  a.x -= t * a.y;
  a.y += s * a.x;
  a.x -= t * a.y;
  return a;
}

// a * exp(sign 2 pi i m / R), the inner twiddles of R = 9 and 16: a small
// turn by shears, then quarter turns; 45 degrees as in radix 8.  Full complex
// products rounded twice as often and, in single precision, took a cosine of
// 22.5 degrees that is off by half a unit: rows of 4096 came out at 1.22e-7
// (1.19e-7 with radix 8 and a pass more), with the turns at 1.15e-7; rows of
// 729 at 1.30e-7 (1.29e-7 with radix 3), with the turns at 1.25e-7.  Times
// of 2-D and 3-D calls are the same; a 1-D call of two latency-bound passes
// (u2nu, 100003 modes) went 80.6 -> 81.4 us.
template <typename T, int R, typename C>
__device__ __forceinline__ C turn(C a, int m, int sign) {
  const T sg = (T)sign;
  if constexpr (R == 16) {
    const T h = (T)0.70710678118654752440;
    const T t = sg * (T)0.19891236737965800691,  // tan(pi/16)
        s = sg * (T)0.38268343236508977173;      // sin(pi/8)
    C r;
    switch (m) {
      case 1: return shear3<T>(a, t, s);
      case 2:
        r.x = (a.x - sg * a.y) * h;
        r.y = (a.y + sg * a.x) * h;
        return r;
      case 3: return cmuli(shear3<T>(a, -t, -s), sign);
      case 4: return cmuli(a, sign);
      case 6:
        r.x = (-a.x - sg * a.y) * h;
        r.y = (-a.y + sg * a.x) * h;
        return r;
      case 9:
        r = shear3<T>(a, t, s);
        r.x = -r.x;
        r.y = -r.y;
        return r;
      default: return a;  // 0
    }
  } else {
    static_assert(R == 9, "turns of 40 degrees");
    C r;
    switch (m) {
      case 1:  // 40 degrees: tan 20, sin 40
        return shear3<T>(a, sg * (T)0.36397023426620236135,
                         sg * (T)0.64278760968653932632);
      case 2:  // 90 - 10
        return cmuli(shear3<T>(a, -sg * (T)0.08748866352592400522,
                               -sg * (T)0.17364817766693034885),
                     sign);
      case 4:  // 180 - 20
        r = shear3<T>(a, -sg * (T)0.17632698070846497347,
                      -sg * (T)0.34202014332566873304);
        r.x = -r.x;
        r.y = -r.y;
        return r;
      default: return a;  // 0
    }
  }
}

// the two factors of a composite radix (0: none)
constexpr int radix_a(int R) {
  return R == 6 ? 2 : R == 9 ? 3 : R == 10 ? 2 : R == 12 ? 4 : R == 14 ? 2
       : R == 15 ? 3 : R == 16 ? 4 : 0;
}

// in-register DFT of length R, exponent sign*2*pi*i*r*k/R
template <typename T, int R, typename C>
__device__ __forceinline__ void dft(C *v, int sign) {
  if constexpr (R == 1) {
    (void)v; (void)sign;
  } else if constexpr (R == 2) {
    C a = v[0], b = v[1];
    v[0] = cadd(a, b);
    v[1] = csub(a, b);
  } else if constexpr (R == 4) {
    C a0 = cadd(v[0], v[2]), a1 = csub(v[0], v[2]);
    C a2 = cadd(v[1], v[3]), a3 = cmuli(csub(v[1], v[3]), sign);
    v[0] = cadd(a0, a2);
    v[2] = csub(a0, a2);
    v[1] = cadd(a1, a3);
    v[3] = csub(a1, a3);
  } else if constexpr (R == 8) {
    // two length-4 DFTs (even / odd inputs), odd outputs times W^k with
    // W = exp(sign 2 pi i / 8), then the length-2 combination
    C e[4] = {v[0], v[2], v[4], v[6]}, o[4] = {v[1], v[3], v[5], v[7]};
    dft<T, 4>(e, sign);
    dft<T, 4>(o, sign);
    const T h = (T)0.70710678118654752440;
    const T sg = (T)sign;
    C w1, w3;
    w1.x = (o[1].x - sg * o[1].y) * h;  // (1 + sign i) / sqrt 2
    w1.y = (o[1].y + sg * o[1].x) * h;
    w3.x = (-o[3].x - sg * o[3].y) * h;  // (-1 + sign i) / sqrt 2
    w3.y = (-o[3].y + sg * o[3].x) * h;
    const C w2 = cmuli(o[2], sign);
    v[0] = cadd(e[0], o[0]);
    v[4] = csub(e[0], o[0]);
    v[1] = cadd(e[1], w1);
    v[5] = csub(e[1], w1);
    v[2] = cadd(e[2], w2);
    v[6] = csub(e[2], w2);
    v[3] = cadd(e[3], w3);
    v[7] = csub(e[3], w3);
  } else if constexpr (R == 6 || R == 10 || R == 12 || R == 14 || R == 15) {
    // coprime factors (Good-Thomas): inputs (B n1 + A n2) mod R, outputs at
    // the k with k = k1 mod A and k = k2 mod B; no inner twiddles
    constexpr int A = radix_a(R), B = R / A;
    C y[B][A];
#pragma unroll
    for (int n2 = 0; n2 < B; ++n2) {
      C t[A];
#pragma unroll
      for (int n1 = 0; n1 < A; ++n1) t[n1] = v[(B * n1 + A * n2) % R];
      dft<T, A>(t, sign);
#pragma unroll
      for (int n1 = 0; n1 < A; ++n1) y[n2][n1] = t[n1];
    }
#pragma unroll
    for (int k1 = 0; k1 < A; ++k1) {
      C t[B];
#pragma unroll
      for (int n2 = 0; n2 < B; ++n2) t[n2] = y[n2][k1];
      dft<T, B>(t, sign);
#pragma unroll
      for (int k = k1; k < R; k += A) v[k] = t[k % B];
    }
  } else if constexpr (R == 9 || R == 16) {
    // Cooley-Tukey A x A, inputs A n1 + n2, outputs k1 + A k2
    constexpr int A = radix_a(R);
    C y[A][A];
#pragma unroll
    for (int n2 = 0; n2 < A; ++n2) {
      C t[A];
#pragma unroll
      for (int n1 = 0; n1 < A; ++n1) t[n1] = v[A * n1 + n2];
      dft<T, A>(t, sign);
#pragma unroll
      for (int k1 = 0; k1 < A; ++k1)
        y[n2][k1] = turn<T, R>(t[k1], n2 * k1, sign);
    }
#pragma unroll
    for (int k1 = 0; k1 < A; ++k1) {
      C t[A];
#pragma unroll
      for (int n2 = 0; n2 < A; ++n2) t[n2] = y[n2][k1];
      dft<T, A>(t, sign);
#pragma unroll
      for (int k2 = 0; k2 < A; ++k2) v[k1 + A * k2] = t[k2];
    }
  } else {
    // odd R: pair r with R-r
    constexpr int H = (R - 1) / 2;
    C sp[H], sm[H];
#pragma unroll
    for (int r = 1; r <= H; ++r) {
      sp[r - 1] = cadd(v[r], v[R - r]);
      sm[r - 1] = csub(v[r], v[R - r]);
    }
    C y0 = v[0];
#pragma unroll
    for (int r = 0; r < H; ++r) y0 = cadd(y0, sp[r]);
    C out[R];
    out[0] = y0;
#pragma unroll
    for (int k = 1; k <= H; ++k) {
      C a = v[0], b;
      b.x = T(0);
      b.y = T(0);
#pragma unroll
      for (int r = 1; r <= H; ++r) {
        const int m = (r * k) % R;  // m in 1..R-1
        const T cc = (T)Tw<R>::c[m - 1], ss = (T)Tw<R>::s[m - 1];
        a.x += sp[r - 1].x * cc;
        a.y += sp[r - 1].y * cc;
        b.x += sm[r - 1].x * ss;
        b.y += sm[r - 1].y * ss;
      }
      C ib = cmuli(b, sign);
      out[k] = cadd(a, ib);
      out[R - k] = csub(a, ib);
    }
#pragma unroll
    for (int k = 0; k < R; ++k) v[k] = out[k];
  }
}

// Quotient and remainder of x / d for 0 <= x < 2^22 and 0 < d, from a
// float reciprocal and one correction step: the estimate is within one of
// the true quotient because x * inv carries a relative error below 2^-22.
// Integer division compiles to a long VALU sequence, which dominated the
// butterflies before.
__device__ __forceinline__ int fdivq(int x, int d, float inv, int &r) {
  int q = (int)((float)x * inv);
  r = x - q * d;
  if (r < 0) {
    --q;
    r += d;
  } else if (r >= d) {
    ++q;
    r -= d;
  }
  return q;
}

__device__ __forceinline__ int64_t map_range(int v, int n1, int a1, int a2) {
  return v < n1 ? (int64_t)(a1 + v) : (int64_t)(a2 + (v - n1));
}

// The lines of one workgroup: nl lines of length Ls staged in LDS with
// stride LP, and where their elements sit in global memory.
template <typename T, int SIGN>
struct LineSet {
  using C = typename V2<T>::t;
  C *buf;
  const C *tw;
  int nl, v0, u;
  float inv_nl;
  int64_t ibase, obase;  // element offsets of this (u, outer)
  int nin0, nout0;       // natural indices of this u's first element

  __device__ __forceinline__ int line(const FftArgs &p, int b) const {
    return (int)map_range(v0 + b, p.vn1, p.va1, p.va2);
  }
  // butterfly q of a pass with nbf butterflies a line -> line b, index jj
  __device__ __forceinline__ int split(int q, const FftPass &ps, bool bfast,
                                       int &b) const {
    if (nl == 1) {
      b = 0;
      return q;
    }
    int x, y;
    if (bfast) {
      x = fdivq(q, nl, inv_nl, y);
      b = y;
      return x;
    }
    b = fdivq(q, ps.nbf, ps.inv_nbf, y);
    return y;
  }
};

// Where a line's results go: element offset (of the uniform array with the
// crop), natural index, and the line's factor in the crop and the twiddles.
struct OutLine {
  int64_t o0;
  int nat0, tq;
  double cf;
};

__device__ __forceinline__ OutLine out_line(const FftArgs &p, int64_t obase,
                                            int nout0, int line, int u,
                                            int v) {
  OutLine l;
  l.o0 = obase + (int64_t)line * p.out_b;
  l.nat0 = nout0 + line * p.nout_b;
  l.tq = p.twiddle == 1 ? u : v;
  l.cf = 1.0;
  if (p.crop) {
    // grid column -> mode index, correction factor and offset
    const FftCrop &q = p.cr;
    const int h1 = q.n1 / 2;
    const int i1 = line < q.n1 - h1 ? line + h1 : line - (q.N1 - h1);
    int u1 = q.fft_order ? i1 + q.n1 - h1 : i1;
    if (u1 >= q.n1) u1 -= q.n1;
    l.o0 = (int64_t)u1 * q.ust1;
    l.cf = q.cf1[h1 > i1 ? h1 - i1 : i1 - h1];
  }
  return l;
}

// Results k0, k0 + dk, ... (R of them) of a line to global memory: through
// the crop, times the pass A twiddles, or as they are; the pruned range is
// left out.  One uniform branch selects the loop, so that no store waits for
// another element's arguments.
template <typename T, int R, int SIGN>
__device__ __forceinline__ void store_line(const FftArgs &p, const OutLine &l,
                                           int k0, int dk,
                                           const typename V2<T>::t *v) {
  using C = typename V2<T>::t;
  const int nat0 = l.nat0 + k0 * p.nout_k, dn = dk * p.nout_k;
  if (p.crop) {
    // retained rows and columns only reach here
    const FftCrop &q = p.cr;
    const int h0 = q.n0 / 2;
#pragma unroll
    for (int r = 0; r < R; ++r) {
      const int nat = nat0 + r * dn;
      if ((unsigned)(nat - p.sn1) < (unsigned)p.sspan) continue;
      const int i0 = nat < q.n0 - h0 ? nat + h0 : nat - (q.N0 - h0);
      int u0 = q.fft_order ? i0 + q.n0 - h0 : i0;
      if (u0 >= q.n0) u0 -= q.n0;
      const T fct = (T)(q.cf0[h0 > i0 ? h0 - i0 : i0 - h0] * l.cf);
      const int64_t ui = l.o0 + (int64_t)u0 * q.ust0;
      if (q.u_f64)
        ((double2 *)q.uni)[ui] =
            make_double2((double)(v[r].x * fct), (double)(v[r].y * fct));
      else
        ((float2 *)q.uni)[ui] =
            make_float2((float)(v[r].x * fct), (float)(v[r].y * fct));
    }
    return;
  }
  C *out = (C *)p.dst + (l.o0 + (int64_t)k0 * p.out_k);
  const int64_t step = (int64_t)dk * p.out_k;
  if (p.twiddle) {
    // k * (u or line) < L1 * L2 = L; pass A writes no pruned range
    const C *tw = (const C *)p.tw_full + (int64_t)k0 * l.tq;
    const int dt = dk * l.tq;
    C w[R];
#pragma unroll
    for (int r = 0; r < R; ++r) w[r] = tw[r * dt];
#pragma unroll
    for (int r = 0; r < R; ++r) {
      if (SIGN > 0) w[r].y = -w[r].y;
      out[r * step] = cmul(v[r], w[r]);
    }
  } else if (p.sspan) {
#pragma unroll
    for (int r = 0; r < R; ++r)
      if (!((unsigned)(nat0 + r * dn - p.sn1) < (unsigned)p.sspan))
        out[r * step] = v[r];
  } else {
#pragma unroll
    for (int r = 0; r < R; ++r) out[r * step] = v[r];
  }
}

// One radix-R Stockham pass over the workgroup's lines, the transform sign
// known at compile time.  The first pass (IN_G) reads its butterflies'
// elements jj + r * nbf from global memory, the last one (OUT_G) writes its
// results there, the others go through LDS; so a line set costs one LDS
// sweep less at each end.  All inputs of a lane's KM butterflies are read
// (and twiddled) before the barrier that frees the buffer.  A lane past the
// last butterfly loads the last one's elements (unconditional loads, all in
// flight at once) and writes nothing; an element known to be zero is not
// fetched, its load repeats the butterfly's first element.
template <typename T, int R, int KM, int SIGN, bool IN_G, bool OUT_G>
__device__ __forceinline__ void fft_pass(const FftArgs &p,
                                         const LineSet<T, SIGN> &s,
                                         const FftPass &ps, bool bfast) {
  using C = typename V2<T>::t;
  const int nbf = ps.nbf, Ns = ps.ns, total = nbf * s.nl;
  C v[KM][R];
  int ob[KM], lb[KM];
#pragma unroll
  for (int k = 0; k < KM; ++k) {
    const int q = (int)threadIdx.x + k * FFT_THREADS;
    // (a wave wholly past the end loads nothing)
    if (IN_G ? (q & ~63) < total : q < total) {
      int b;
      const int jj = s.split(IN_G ? min(q, total - 1) : q, ps, bfast, b);
      lb[k] = b;
      if constexpr (IN_G) {
        const C *src = (const C *)p.src;
        const int line = s.line(p, b);
        const int64_t a0 = s.ibase + (int64_t)line * p.in_b +
                           (int64_t)jj * p.in_e,
                      da = (int64_t)nbf * p.in_e;
        if (p.kspan) {
          const int n0 = s.nin0 + line * p.nin_b + jj * p.nin_e - p.kn1,
                    dn = nbf * p.nin_e;
#pragma unroll
          for (int r = 0; r < R; ++r) {
            const bool zero = (unsigned)(n0 + r * dn) < (unsigned)p.kspan;
            C x = src[a0 + (zero ? 0 : r * da)];
            v[k][r].x = zero ? T(0) : x.x;
            v[k][r].y = zero ? T(0) : x.y;
          }
        } else {
#pragma unroll
          for (int r = 0; r < R; ++r) v[k][r] = src[a0 + r * da];
        }
        if (p.scale != 1.0) {
          const T f = (T)p.scale;
#pragma unroll
          for (int r = 0; r < R; ++r) {
            v[k][r].x *= f;
            v[k][r].y *= f;
          }
        }
        ob[k] = jj * R;  // Ns == 1
      } else {
        const C *in = s.buf + b * p.LP + jj;
#pragma unroll
        for (int r = 0; r < R; ++r) v[k][r] = in[r * nbf];
        int kk = jj, jq = 0;  // the last pass has Ns == nbf
        if (!OUT_G) jq = fdivq(jj, Ns, ps.inv_ns, kk);
        const int t1 = kk * ps.twstep;
#pragma unroll
        for (int r = 1; r < R; ++r) {
          C w = s.tw[r * t1];
          if (SIGN > 0) w.y = -w.y;
          v[k][r] = cmul(v[k][r], w);
        }
        ob[k] = jq * Ns * R + kk;
      }
    }
  }
  if (!IN_G && !OUT_G) __syncthreads();
#pragma unroll
  for (int k = 0; k < KM; ++k) {
    const int q = (int)threadIdx.x + k * FFT_THREADS;
    if (q < total) {
      dft<T, R>(v[k], SIGN);
      if constexpr (OUT_G) {
        const OutLine l = out_line(p, s.obase, s.nout0, s.line(p, lb[k]), s.u,
                                   s.v0 + lb[k]);
        store_line<T, R, SIGN>(p, l, ob[k], Ns, v[k]);
      } else {
        C *out = s.buf + lb[k] * p.LP + ob[k];
#pragma unroll
        for (int r = 0; r < R; ++r) out[r * Ns] = v[k][r];
      }
    }
  }
  if (!OUT_G) __syncthreads();
}

template <typename T, int MAXEL, int SIGN, bool IN_G, bool OUT_G>
__device__ __forceinline__ void fft_pass_radix(const FftArgs &p,
                                               const LineSet<T, SIGN> &s,
                                               const FftPass &ps,
                                               bool bfast) {
#define DMX_PASS(R)                                                        \
  case R:                                                                  \
    fft_pass<T, R, fft_km(MAXEL, R), SIGN, IN_G, OUT_G>(p, s, ps, bfast);  \
    break
  switch (ps.radix) {
    DMX_PASS(16); DMX_PASS(15); DMX_PASS(14); DMX_PASS(12); DMX_PASS(11);
    DMX_PASS(10); DMX_PASS(9); DMX_PASS(8); DMX_PASS(7); DMX_PASS(6);
    DMX_PASS(5); DMX_PASS(4); DMX_PASS(3); DMX_PASS(2);
    default: break;
  }
#undef DMX_PASS
}

// MAXEL: the most elements (lines x length) the launch puts in one
// workgroup; it sizes the register staging of the passes, and the half-size
// variant leaves room for more workgroups per CU.  Waves a SIMD: the full-size
// variants hold twice the staging and two or three of their workgroups fit a
// CU, so they get the registers of three waves (at 5 and 4 waves, as the
// half-size ones, they spilled 500 registers a lane in FP32 and 150 in FP64:
// c2c of 3000^2 in FP64 232 -> 205 us, rows of a 3024^2 FP64 grid 99 -> 82).
template <typename T, int MAXEL, int SIGN>
__global__ __launch_bounds__(FFT_THREADS) __attribute__((
    amdgpu_waves_per_eu(
    sizeof(T) * MAXEL <= 16384 ? (sizeof(T) == 4 ? 5 : 4) : 3))) void
k_fft(FftArgs p) {
  using C = typename V2<T>::t;
  extern __shared__ unsigned char smem_raw[];
  const int v0 = (int)blockIdx.x * p.Bl, nl = min(p.Bl, p.nv - v0);
  C *buf = (C *)smem_raw;
  const C *tw = (const C *)p.tw;
  if (p.tw_lds) {
    // the twiddles sit behind the lines in LDS (read after a barrier: the
    // first pass uses none)
    C *t = buf + (size_t)p.Bl * p.LP;
    for (int i = threadIdx.x; i < p.Ls; i += FFT_THREADS) t[i] = tw[i];
    tw = t;
  }
  const int u = (int)map_range(blockIdx.y, p.un1, p.ua1, p.ua2);
  const int64_t z = map_range(blockIdx.z, p.on1, p.oa1, p.oa2);
  const LineSet<T, SIGN> s{buf, tw, nl, v0, u, 1.0f / (float)nl,
                     z * p.st_o + u * p.in_u, z * p.st_o + u * p.out_u,
                     u * p.nin_u, u * p.nout_u};
  const int np = p.npass;
  if (np == 1) {
    fft_pass_radix<T, MAXEL, SIGN, true, true>(p, s, p.pass[0], p.bf_in);
    return;
  }
  fft_pass_radix<T, MAXEL, SIGN, true, false>(p, s, p.pass[0], p.bf_in);
  for (int i = 1; i < np - 1; ++i)
    fft_pass_radix<T, MAXEL, SIGN, false, false>(p, s, p.pass[i], p.bf_mid);
  fft_pass_radix<T, MAXEL, SIGN, false, true>(p, s, p.pass[np - 1], p.bf_out);
}

}  // namespace

// launches the kernel of one compute type and workgroup size (the odd line
// stride takes full-size workgroups of even lines up to 128 bytes past the
// default 64 KiB: 16 lines of 512, 8 of 1024, ...)
template <typename T, int MAXEL>
void launch_k_fft(const FftArgs &a, int sign, dim3 grid, size_t lds,
                  hipStream_t s);

#define DMX_INSTANTIATE_FFT(T, MAXEL)                                       \
  namespace dmx {                                                           \
  template <>                                                               \
  void launch_k_fft<T, MAXEL>(const FftArgs &a, int sign, dim3 grid,        \
                              size_t lds, hipStream_t s) {                  \
    if (sign < 0) {                                                         \
      allow_big_lds(k_fft<T, MAXEL, -1>, lds);                              \
      hipLaunchKernelGGL((k_fft<T, MAXEL, -1>), grid, dim3(FFT_THREADS),    \
                         lds, s, a);                                        \
    } else {                                                                \
      allow_big_lds(k_fft<T, MAXEL, 1>, lds);                               \
      hipLaunchKernelGGL((k_fft<T, MAXEL, 1>), grid, dim3(FFT_THREADS),     \
                         lds, s, a);                                        \
    }                                                                       \
    DMX_HIP(hipGetLastError());                                             \
  }                                                                         \
  }

}  // namespace dmx
