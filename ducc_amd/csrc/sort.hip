// sort.hip -- folding points into tiles and the stable counting sort of the
// index build (role of nufft.h:892-907, 1364-1381, 1862-1892 and
// bucket_sort.h:170-354).  The order produced is the stable ascending order
// of the tile keys: ties keep input order, which is the unique permutation a
// stable sort gives and the one ducc0's bucket_sort2 returns.
//
// Layout: keys / indices are uint32 arrays of M in HBM.  The sort is an LSD
// radix sort with 8-bit digits: per pass one histogram kernel (one LDS
// histogram per 4096-key block), one exclusive scan of the digit-major
// block table, and one scatter kernel that ranks equal digits inside a
// wavefront with ballots (stable) and across the block's four wavefronts in
// wave order, so every pass is stable; the ranked block is staged in LDS and
// written out in digit runs.
#include "radix.h"

namespace dmx {

namespace {
using namespace radix;

// Tile key per point (nufft.h:1364-1381 role); one 4096-point block per
// workgroup, so that the first sort pass's per-block digit histogram comes
// out of the same sweep.  Each lane loads a batch of FB points before it
// folds them, so the loads of a batch are in flight together.
constexpr int FB = 16;
template <int NDIM>
__global__ __launch_bounds__(RT) void k_fold_keys(Geo g, const void *coords,
                                                  size_t M, uint32_t *keys,
                                                  uint32_t *hist0,
                                                  int nblocks) {
  __shared__ uint32_t h[RB];
  const int tid = threadIdx.x;
  if (hist0) h[tid] = 0;
  __syncthreads();
  const size_t base = (size_t)blockIdx.x * RTILE;
  for (int i0 = 0; i0 < RITEMS; i0 += FB) {
    double x[FB][NDIM];
#pragma unroll
    for (int q = 0; q < FB; ++q) {
      const size_t j = base + (size_t)(i0 + q) * RT + tid;
      if (j < M) load_point(g, coords, j, NDIM, x[q]);
    }
#pragma unroll
    for (int q = 0; q < FB; ++q) {
      const size_t j = base + (size_t)(i0 + q) * RT + tid;
      if (j >= M) continue;
      uint32_t t[NDIM];
#pragma unroll
      for (int d = 0; d < NDIM; ++d) {
        double fr;
        const int c0 = fold_axis(g, d, x[q][d], fr);
        t[d] = (uint32_t)((c0 + g.nsafe) >> g.log2tile);
      }
      uint32_t key = t[0];
#pragma unroll
      for (int d = 1; d < NDIM; ++d) key = key * (uint32_t)g.ntiles[d] + t[d];
      if (keys) keys[j] = key;
      if (hist0) atomicAdd(&h[key & 0xFFu], 1u);
    }
  }
  if (hist0) {
    __syncthreads();
    hist0[(size_t)tid * nblocks + blockIdx.x] = h[tid];
  }
}

__global__ __launch_bounds__(RT) void k_radix_hist(const uint32_t *keys,
                                                   size_t M, int shift,
                                                   uint32_t *hist,
                                                   int nblocks) {
  __shared__ uint32_t h[RB];
  h[threadIdx.x] = 0;
  __syncthreads();
  size_t base = (size_t)blockIdx.x * RTILE;
  // all of a lane's key loads in flight before its LDS atomics
  uint32_t kv[RITEMS];
#pragma unroll
  for (int i = 0; i < RITEMS; ++i) {
    size_t j = base + (size_t)i * RT + threadIdx.x;
    kv[i] = j < M ? keys[j] : 0u;
  }
#pragma unroll
  for (int i = 0; i < RITEMS; ++i) {
    size_t j = base + (size_t)i * RT + threadIdx.x;
    if (j < M) atomicAdd(&h[(kv[i] >> shift) & 0xFFu], 1u);
  }
  __syncthreads();
  hist[(size_t)threadIdx.x * nblocks + blockIdx.x] = h[threadIdx.x];
}

// Stable scatter of one 4096-key block, staged through LDS so that the
// global writes go out in digit runs (consecutive lanes -> consecutive
// addresses):
//  (1) wave w ranks its 1024 keys [w*1024, (w+1)*1024) in order, 64 at a
//      time: ballot peers give the rank inside the 64, a per-wave per-digit
//      counter in LDS (touched only by the group leader) the rank before;
//  (2) one prefix over (digit, wave) gives each key its position in the
//      block's locally sorted order, and each digit its global base;
//  (3) keys, then indices, are written to LDS in local order and read back
//      by position, so lane t of round i stores element i*256+t of the
//      sorted block at global base[digit] + (position - local start).
__global__ __launch_bounds__(RT) void k_radix_scatter(
    const uint32_t *keys_in, const uint32_t *idx_in, size_t M, int shift,
    const uint32_t *offs, const uint32_t *offs_chunk, int nblocks,
    uint32_t *keys_out, uint32_t *idx_out, uint32_t *tb_start_c,
    uint32_t *tb_end) {
  __shared__ RankShared rs;
  __shared__ uint32_t stage[RTILE];
  const int tid = threadIdx.x, wave = tid >> 6;
  const unsigned lane = lane_id();
  const size_t blk0 = (size_t)blockIdx.x * RTILE;
  const size_t c0 = blk0 + (size_t)wave * (RTILE / NW);
  uint32_t key[RITEMS], ival[RITEMS], dig[RITEMS];
  bool valid[RITEMS];
#pragma unroll
  for (int r = 0; r < RITEMS; ++r) {
    const size_t j = c0 + (size_t)r * 64 + lane;
    valid[r] = j < M;
    key[r] = valid[r] ? keys_in[j] : 0xFFFFFFFFu;
  }
  // this block's global base of digit tid (chunk scan + scanned chunk
  // sums), and the indices that travel with the keys: loaded now, so that
  // their latency overlaps the ranking
  const size_t og = (size_t)tid * nblocks + blockIdx.x;
  const uint32_t gofs = offs[og] + offs_chunk[og / STILE];
#pragma unroll
  for (int r = 0; r < RITEMS; ++r) {
    const size_t j = c0 + (size_t)r * 64 + lane;
    ival[r] = idx_in ? (valid[r] ? idx_in[j] : 0u) : (uint32_t)j;
    dig[r] = (key[r] >> shift) & 0xFFu;
  }
  uint32_t lpos[RITEMS];
  rank_block(dig, valid, lpos, rs, gofs);
  const uint32_t *gbase = rs.gbase;
  const int nvalid = (int)min((size_t)RTILE, M - blk0);
#pragma unroll
  for (int r = 0; r < RITEMS; ++r)
    if (valid[r]) stage[lpos[r]] = key[r];
  __syncthreads();
  uint32_t gpos[RITEMS];
#pragma unroll
  for (int i = 0; i < RITEMS; ++i) {
    const int q = i * RT + tid;
    gpos[i] = 0;
    if (q < nvalid) {
      const uint32_t k = stage[q];
      gpos[i] = gbase[(k >> shift) & 0xFFu] + (uint32_t)q;
      if (keys_out) keys_out[gpos[i]] = k;
      if (tb_end) {
        // final pass: equal keys are contiguous here and globally, so the
        // block's first / last element of a key bound the tile's range
        // (start kept complemented, so both arrays start at zero)
        if (q == 0 || stage[q - 1] != k) atomicMax(&tb_start_c[k], ~gpos[i]);
        if (q == nvalid - 1 || stage[q + 1] != k)
          atomicMax(&tb_end[k], gpos[i] + 1);
      }
    }
  }
  __syncthreads();
#pragma unroll
  for (int r = 0; r < RITEMS; ++r) {
    const size_t j = c0 + (size_t)r * 64 + lane;
    if (j < M) stage[lpos[r]] = ival[r];
  }
  __syncthreads();
#pragma unroll
  for (int i = 0; i < RITEMS; ++i) {
    const int q = i * RT + tid;
    if (q < nvalid) idx_out[gpos[i]] = stage[q];
  }
}

__global__ __launch_bounds__(ST) void k_scan_blocks(const uint32_t *in,
                                                    uint32_t *out, size_t n,
                                                    uint32_t *bsum) {
  __shared__ uint32_t sh[ST];
  size_t base = (size_t)blockIdx.x * STILE + (size_t)threadIdx.x * SITEMS;
  uint32_t v[SITEMS], s = 0;
#pragma unroll
  for (int i = 0; i < SITEMS; ++i) {
    v[i] = (base + i < n) ? in[base + i] : 0u;
    s += v[i];
  }
  uint32_t tot;
  uint32_t ex = block_exclusive_scan(s, sh, tot);
#pragma unroll
  for (int i = 0; i < SITEMS; ++i) {
    if (base + i < n) out[base + i] = ex;
    ex += v[i];
  }
  if (threadIdx.x == 0) bsum[blockIdx.x] = tot;
}

// one workgroup scans the whole array (in may equal out); used for the
// block sums of the multi-block scan and for short arrays in one launch
__global__ __launch_bounds__(ST) void k_scan_single(const uint32_t *in,
                                                    uint32_t *out, size_t n,
                                                    uint32_t *total) {
  __shared__ uint32_t sh[ST];
  uint32_t carry = 0;
  for (size_t c = 0; c < n; c += STILE) {
    size_t base = c + (size_t)threadIdx.x * SITEMS;
    uint32_t v[SITEMS], s = 0;
#pragma unroll
    for (int i = 0; i < SITEMS; ++i) {
      v[i] = (base + i < n) ? in[base + i] : 0u;
      s += v[i];
    }
    uint32_t tot;
    uint32_t ex = block_exclusive_scan(s, sh, tot) + carry;
#pragma unroll
    for (int i = 0; i < SITEMS; ++i) {
      if (base + i < n) out[base + i] = ex;
      ex += v[i];
    }
    carry += tot;
  }
  if (threadIdx.x == 0 && total) *total = carry;
}

__global__ __launch_bounds__(ST) void k_scan_add(uint32_t *out, size_t n,
                                                 const uint32_t *bsum) {
  size_t base = (size_t)blockIdx.x * STILE;
  uint32_t a = bsum[blockIdx.x];
  for (int i = threadIdx.x; i < STILE; i += ST)
    if (base + i < n) out[base + i] += a;
}

// ------------------------------------------------------------ subproblems
// tile [start, end) from the sort's final pass (start stored complemented;
// empty tiles have end 0), points per tile and subproblems per tile (runs
// of at most MAXSUB points)
__global__ void k_counts_nsub(uint32_t *tstart, const uint32_t *tend,
                              size_t ntiles, uint32_t *counts,
                              uint32_t *nsub) {
  size_t t = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= ntiles) return;
  const uint32_t e = tend[t];
  const uint32_t st = e ? ~tstart[t] : 0u;
  tstart[t] = st;
  const uint32_t c = e - st;
  counts[t] = c;
  nsub[t] = (c + MAXSUB - 1) / MAXSUB;
}

__global__ void k_fill_subs(const uint32_t *counts, const uint32_t *tstart,
                            const uint32_t *nsub, const uint32_t *sstart,
                            size_t ntiles, Sub *subs) {
  size_t t = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= ntiles) return;
  uint32_t n = nsub[t], s0 = sstart[t], ts = tstart[t], te = ts + counts[t];
  for (uint32_t s = 0; s < n; ++s) {
    Sub sb;
    sb.tile = (uint32_t)t;
    sb.start = ts + s * MAXSUB;
    sb.end = min(te, sb.start + (uint32_t)MAXSUB);
    sb.rank = s;
    subs[s0 + s] = sb;
  }
}

// The three steps above in one workgroup, for tile tables of at most 4096
// tiles (one launch instead of four; longer tables take the launches above,
// which measured faster from about 10^4 tiles on): per 4096-tile chunk, start / count / subproblem
// count of each tile, a block prefix of the subproblem counts (with the
// carry of the chunks before) and the subproblems themselves.  The scan
// wants TS_ITEMS consecutive tiles per lane, global memory wants
// consecutive tiles per wave: the chunk's tables pass through LDS (one pad
// word per TS_ITEMS entries keeps both access patterns free of bank
// conflicts), so every global load and store of the tables is coalesced.
constexpr int TS_ITEMS = 16;
constexpr int TS_CH = ST * TS_ITEMS, TS_CHP = TS_CH + TS_CH / TS_ITEMS;
__device__ __forceinline__ int ts_slot(int q) { return q + q / TS_ITEMS; }
__global__ __launch_bounds__(ST) void k_tile_subs_one(
    uint32_t *tstart, const uint32_t *tend, size_t ntiles, uint32_t *counts,
    uint32_t *nsub, uint32_t *sstart, Sub *subs, uint32_t *nsub_total) {
  __shared__ uint32_t sh[ST];
  __shared__ uint32_t la[TS_CHP], lb[TS_CHP];
  const int tid = threadIdx.x;
  uint32_t carry = 0;
  for (size_t c = 0; c < ntiles; c += TS_CH) {
    const int nc = (int)min((size_t)TS_CH, ntiles - c);
    // coalesced loads, all in flight (clamped indices past the chunk's end
    // read its last tile; those entries are never used)
    uint32_t ev[TS_ITEMS], sv[TS_ITEMS];
#pragma unroll
    for (int k = 0; k < TS_ITEMS; ++k) {
      if (k * ST >= nc) {
        ev[k] = sv[k] = 0;
        continue;
      }
      const size_t t = c + (size_t)min(k * ST + tid, nc - 1);
      ev[k] = tend[t];
      sv[k] = tstart[t];
    }
    __syncthreads();  // the previous chunk's LDS readers are done
#pragma unroll
    for (int k = 0; k < TS_ITEMS; ++k) {
      la[ts_slot(k * ST + tid)] = ev[k];
      lb[ts_slot(k * ST + tid)] = sv[k];
    }
    __syncthreads();
    const int q0 = tid * TS_ITEMS;
    uint32_t st[TS_ITEMS], cn[TS_ITEMS], ns[TS_ITEMS], sum = 0;
#pragma unroll
    for (int k = 0; k < TS_ITEMS; ++k) {
      st[k] = cn[k] = ns[k] = 0;
      if (q0 + k < nc) {
        const uint32_t e = la[ts_slot(q0 + k)];
        st[k] = e ? ~lb[ts_slot(q0 + k)] : 0u;
        cn[k] = e - st[k];
        ns[k] = (cn[k] + MAXSUB - 1) / MAXSUB;
        sum += ns[k];
      }
    }
    uint32_t tot;
    const uint32_t ex0 = block_exclusive_scan(sum, sh, tot) + carry;
    uint32_t ex = ex0;
#pragma unroll
    for (int k = 0; k < TS_ITEMS; ++k) {
      if (q0 + k >= nc) continue;
      for (uint32_t q = 0; q < ns[k]; ++q) {
        Sub sb;
        sb.tile = (uint32_t)(c + q0 + k);
        sb.start = st[k] + q * MAXSUB;
        sb.end = min(st[k] + cn[k], sb.start + (uint32_t)MAXSUB);
        sb.rank = q;
        subs[ex + q] = sb;
      }
      ex += ns[k];
    }
    // starts and counts, then subproblem counts and first subproblems,
    // back through LDS to coalesced stores
    __syncthreads();  // all lanes have read la / lb
#pragma unroll
    for (int k = 0; k < TS_ITEMS; ++k) {
      la[ts_slot(q0 + k)] = st[k];
      lb[ts_slot(q0 + k)] = cn[k];
    }
    __syncthreads();
#pragma unroll
    for (int k = 0; k < TS_ITEMS; ++k) {
      const int q = k * ST + tid;
      if (q < nc) {
        tstart[c + q] = la[ts_slot(q)];
        counts[c + q] = lb[ts_slot(q)];
      }
    }
    __syncthreads();
    ex = ex0;
#pragma unroll
    for (int k = 0; k < TS_ITEMS; ++k) {
      la[ts_slot(q0 + k)] = ns[k];
      lb[ts_slot(q0 + k)] = ex;
      ex += ns[k];
    }
    __syncthreads();
#pragma unroll
    for (int k = 0; k < TS_ITEMS; ++k) {
      const int q = k * ST + tid;
      if (q < nc) {
        nsub[c + q] = la[ts_slot(q)];
        sstart[c + q] = lb[ts_slot(q)];
      }
    }
    carry += tot;
  }
  if (tid == 0) *nsub_total = carry;
}

// ------------------------------------------------- one workgroup, one launch
// Index build of at most SMALL_M points in at most SMALL_TILES tiles: fold,
// stable LSD sort, tile table and subproblems by one workgroup of 1024
// threads in LDS.  Such a request is a chain of launch latencies: six
// launches of 2-9 us each took 27 us for 2000 points, this one 9 us.
constexpr int SMALL_T = 1024, SMALL_I = 4, SMALL_M = SMALL_T * SMALL_I,
              SMALL_TILES = 4096, SMALL_W = SMALL_T / 64;

// exclusive prefix over 1024 threads
__device__ __forceinline__ uint32_t scan1024(uint32_t v, uint32_t *sh,
                                             uint32_t &total) {
  const int t = threadIdx.x, lane = t & 63, w = t >> 6;
  uint32_t x = v;
#pragma unroll
  for (int o = 1; o < 64; o <<= 1) {
    const uint32_t y = __shfl_up(x, (unsigned)o);
    if (lane >= o) x += y;
  }
  if (lane == 63) sh[w] = x;
  __syncthreads();
  uint32_t before = 0, tot = 0;
#pragma unroll
  for (int i = 0; i < SMALL_W; ++i) {
    const uint32_t s = sh[i];
    before += i < w ? s : 0u;
    tot += s;
  }
  total = tot;
  __syncthreads();
  return before + x - v;
}

// lanes of the wave with the same value of the low `bits` bits
__device__ __forceinline__ unsigned long long peers_of(uint32_t d, bool valid,
                                                       int bits) {
  unsigned long long peers = __ballot(valid);
  for (int b = 0; b < bits; ++b) {
    const bool bit = (d >> b) & 1;
    const unsigned long long bal = __ballot(bit);
    peers &= bit ? bal : ~bal;
  }
  return peers;
}

template <int NDIM>
__device__ __forceinline__ uint32_t tile_key(const Geo &g, const double *x) {
  uint32_t key = 0;
#pragma unroll
  for (int d = 0; d < NDIM; ++d) {
    double fr;
    const int c0 = fold_axis(g, d, x[d], fr);
    const uint32_t t = (uint32_t)((c0 + g.nsafe) >> g.log2tile);
    key = d == 0 ? t : key * (uint32_t)g.ntiles[d] + t;
  }
  return key;
}

template <int NDIM>
__global__ __launch_bounds__(SMALL_T) void k_index_small(
    Geo g, const void *coords, int M, int keybits, int ntiles,
    uint32_t *idx_out, uint32_t *counts, uint32_t *tstart, uint32_t *nsub,
    uint32_t *sstart, Sub *subs, uint32_t *nsub_total) {
  __shared__ uint32_t skey[SMALL_M];
  __shared__ uint16_t sidx[SMALL_M];
  __shared__ union {
    uint32_t cnt[SMALL_W][256];  // digits of a wave's items (sort)
    struct {
      uint32_t st[SMALL_TILES], en[SMALL_TILES];  // tile ranges (after it)
    } t;
  } u;
  __shared__ uint32_t sh[SMALL_W];
  const int tid = threadIdx.x, wave = tid >> 6;
  const unsigned lane = lane_id();
  const unsigned long long below_mask =
      lane ? (~0ull >> (64 - lane)) : 0ull;
  // item r of lane l of wave w is number w*256 + r*64 + l
  const int q0 = wave * (64 * SMALL_I) + (int)lane;
  uint32_t key[SMALL_I], id[SMALL_I];
  bool valid[SMALL_I];
  {
    double x[SMALL_I][NDIM];
#pragma unroll
    for (int r = 0; r < SMALL_I; ++r) {
      id[r] = (uint32_t)(q0 + r * 64);
      valid[r] = (int)id[r] < M;
      if (valid[r]) load_point(g, coords, (size_t)id[r], NDIM, x[r]);
    }
#pragma unroll
    for (int r = 0; r < SMALL_I; ++r)
      key[r] = valid[r] ? tile_key<NDIM>(g, x[r]) : 0u;
  }
  for (int shift = 0; shift < keybits; shift += 8) {
    const int bits = min(8, keybits - shift);
    for (int c = tid; c < SMALL_W * 256; c += SMALL_T) u.cnt[0][c] = 0;
    __syncthreads();
    uint32_t rank[SMALL_I], dig[SMALL_I];
#pragma unroll
    for (int r = 0; r < SMALL_I; ++r) {
      dig[r] = (key[r] >> shift) & 0xFFu;
      const unsigned long long peers = peers_of(dig[r], valid[r], bits);
      const unsigned long long below = peers & below_mask;
      const uint32_t old = u.cnt[wave][dig[r]];
      __builtin_amdgcn_wave_barrier();
      if (valid[r] && below == 0)
        u.cnt[wave][dig[r]] = old + (uint32_t)__popcll(peers);
      __builtin_amdgcn_wave_barrier();
      rank[r] = old + (uint32_t)__popcll(below);
    }
    __syncthreads();
    // digit tid: its items in the waves before, its start in the block
    uint32_t run = 0, tot;
    if (tid < 256) {
#pragma unroll
      for (int w = 0; w < SMALL_W; ++w) {
        const uint32_t c = u.cnt[w][tid];
        u.cnt[w][tid] = run;
        run += c;
      }
    }
    const uint32_t start = scan1024(run, sh, tot);
    if (tid < 256) {
#pragma unroll
      for (int w = 0; w < SMALL_W; ++w) u.cnt[w][tid] += start;
    }
    __syncthreads();
#pragma unroll
    for (int r = 0; r < SMALL_I; ++r) {
      if (!valid[r]) continue;
      const uint32_t p = u.cnt[wave][dig[r]] + rank[r];
      skey[p] = key[r];
      sidx[p] = (uint16_t)id[r];
    }
    __syncthreads();
#pragma unroll
    for (int r = 0; r < SMALL_I; ++r) {
      const int q = q0 + r * 64;
      if (!valid[r]) continue;  // positions and items end at M alike
      key[r] = skey[q];
      id[r] = sidx[q];
    }
  }
  for (int c = tid; c < SMALL_TILES; c += SMALL_T) u.t.st[c] = u.t.en[c] = 0;
  __syncthreads();
#pragma unroll
  for (int r = 0; r < SMALL_I; ++r) {
    const int q = q0 + r * 64;
    if (!valid[r]) continue;
    idx_out[q] = id[r];
    if (q == 0 || skey[q - 1] != key[r]) u.t.st[key[r]] = (uint32_t)q;
    if (q == M - 1 || skey[q + 1] != key[r]) u.t.en[key[r]] = (uint32_t)q + 1;
  }
  __syncthreads();
  // four consecutive tiles per thread
  constexpr int TI = SMALL_TILES / SMALL_T;
  uint32_t ns[TI], sum = 0, tot;
#pragma unroll
  for (int k = 0; k < TI; ++k) {
    const int t = tid * TI + k;
    ns[k] = (u.t.en[t] - u.t.st[t] + MAXSUB - 1) / MAXSUB;
    sum += ns[k];
  }
  uint32_t ex = scan1024(sum, sh, tot);
#pragma unroll
  for (int k = 0; k < TI; ++k) {
    const int t = tid * TI + k;
    if (t >= ntiles) break;
    const uint32_t a = u.t.st[t], e = u.t.en[t];
    tstart[t] = a;
    counts[t] = e - a;
    nsub[t] = ns[k];
    sstart[t] = ex;
    for (uint32_t q = 0; q < ns[k]; ++q) {
      Sub sb;
      sb.tile = (uint32_t)t;
      sb.start = a + q * MAXSUB;
      sb.end = min(e, sb.start + (uint32_t)MAXSUB);
      sb.rank = q;
      subs[ex + q] = sb;
    }
    ex += ns[k];
  }
  if (tid == 0) *nsub_total = tot;
}

// ------------------------------------------------ one pass, whole keys
// Index build in one stable counting pass whose digit is the whole tile key
// (at most WIDE_TILES tiles): fold + histogram, chunk scans, the scan of the
// chunk sums with the tile table (a tile's start is its first table entry)
// and subproblems, scatter: four launches and one trip of the points where
// the 8-bit passes take ten launches and two.  1e6 points in 364 tiles:
// 62 -> 39 us; 1e5 points in 289 tiles: 60 -> 21 us; 2e6 points in 1600
// tiles: 87 -> 61 us.
constexpr int WIDE_TILES = 4096;

template <int NDIM, int ITEMS>
__global__ __launch_bounds__(RT) void k_fold_wide(Geo g, const void *coords,
                                                  size_t M, uint32_t *keys,
                                                  uint32_t *hist, int nbins,
                                                  int nblocks) {
  extern __shared__ uint32_t h[];
  const int tid = threadIdx.x;
  for (int c = tid; c < nbins; c += RT) h[c] = 0;
  __syncthreads();
  const size_t base = (size_t)blockIdx.x * (RT * ITEMS) + tid;
  double x[ITEMS][NDIM];
#pragma unroll
  for (int q = 0; q < ITEMS; ++q) {
    const size_t j = base + (size_t)q * RT;
    if (j < M) load_point(g, coords, j, NDIM, x[q]);
  }
#pragma unroll
  for (int q = 0; q < ITEMS; ++q) {
    const size_t j = base + (size_t)q * RT;
    if (j >= M) continue;
    const uint32_t key = tile_key<NDIM>(g, x[q]);
    keys[j] = key;
    atomicAdd(&h[key], 1u);
  }
  __syncthreads();
  for (int c = tid; c < nbins; c += RT)
    hist[(size_t)c * nblocks + blockIdx.x] = h[c];
}

// The scan of the table's chunk sums, the tile table and the subproblems, by
// one workgroup: tile t starts at the table's entry t * nblocks.
constexpr int WIDE_CHUNKS = 4096;
__global__ __launch_bounds__(1024) void k_tiles_wide(
    const uint32_t *offs, uint32_t *bsum, int nch, size_t M, int ntiles,
    int nblocks, uint32_t *counts, uint32_t *tstart, uint32_t *nsub,
    uint32_t *sstart, Sub *subs, uint32_t *nsub_total) {
  __shared__ uint32_t sb_[WIDE_CHUNKS], sh[SMALL_W];
  const int tid = threadIdx.x;
  uint32_t carry = 0, tot;
  for (int c = 0; c < nch; c += 1024) {
    const int i = c + tid;
    const uint32_t v = i < nch ? bsum[i] : 0u;
    const uint32_t x = scan1024(v, sh, tot) + carry;
    if (i < nch) sb_[i] = bsum[i] = x;
    carry += tot;
  }
  __syncthreads();
  carry = 0;
  for (int c = 0; c < ntiles; c += 1024) {
    const int t = c + tid;
    uint32_t a = 0, e = 0;
    if (t < ntiles) {
      const size_t o0 = (size_t)t * nblocks, o1 = o0 + nblocks;
      a = offs[o0] + sb_[o0 / STILE];
      e = t + 1 < ntiles ? offs[o1] + sb_[o1 / STILE] : (uint32_t)M;
      if (a == e) a = e = 0;  // an empty tile
    }
    const uint32_t ns = (e - a + MAXSUB - 1) / MAXSUB;
    const uint32_t ex = scan1024(ns, sh, tot) + carry;
    carry += tot;
    if (t < ntiles) {
      tstart[t] = a;
      counts[t] = e - a;
      nsub[t] = ns;
      sstart[t] = ex;
      for (uint32_t q = 0; q < ns; ++q) {
        Sub sb;
        sb.tile = (uint32_t)t;
        sb.start = a + q * MAXSUB;
        sb.end = min(e, sb.start + (uint32_t)MAXSUB);
        sb.rank = q;
        subs[ex + q] = sb;
      }
    }
  }
  if (tid == 0) *nsub_total = carry;
}

// Subproblems of every tile's positions [start[t * nk + k0], start[t * nk +
// k1]) in an order sorted by (tile, second key < nk), for several key ranges
// at once: one workgroup a range, four consecutive tiles per thread and
// round (a range takes 14 us of latencies, so they run side by side).
__global__ __launch_bounds__(1024) void k_tiles_range(
    const uint32_t *start, size_t ntiles, uint32_t nk, KeyRanges ranges,
    uint32_t *nsub, uint32_t *sstart, Sub *subs, size_t list,
    uint32_t *nsub_total) {
  __shared__ uint32_t sh[SMALL_W];
  const uint32_t k0 = ranges.r[blockIdx.x].k0, k1 = ranges.r[blockIdx.x].k1;
  nsub += blockIdx.x * ntiles;
  sstart += blockIdx.x * ntiles;
  subs += blockIdx.x * list;
  nsub_total += blockIdx.x;
  constexpr int TI = 4;
  uint32_t carry = 0, tot;
  for (size_t c = 0; c < ntiles; c += 1024 * TI) {
    const size_t t0 = c + (size_t)threadIdx.x * TI;
    uint32_t a[TI], e[TI], sum = 0;
#pragma unroll
    for (int k = 0; k < TI; ++k) {
      a[k] = e[k] = 0;
      if (t0 + k < ntiles) {
        a[k] = start[(t0 + k) * nk + k0];
        e[k] = start[(t0 + k) * nk + k1];
      }
    }
#pragma unroll
    for (int k = 0; k < TI; ++k) sum += (e[k] - a[k] + MAXSUB - 1) / MAXSUB;
    uint32_t ex = scan1024(sum, sh, tot) + carry;
    carry += tot;
#pragma unroll
    for (int k = 0; k < TI; ++k) {
      const uint32_t ns = (e[k] - a[k] + MAXSUB - 1) / MAXSUB;
      if (t0 + k < ntiles) {
        nsub[t0 + k] = ns;
        sstart[t0 + k] = ex;
      }
      for (uint32_t q = 0; q < ns; ++q) {
        Sub sb;
        sb.tile = (uint32_t)(t0 + k);
        sb.start = a[k] + q * MAXSUB;
        sb.end = min(e[k], sb.start + (uint32_t)MAXSUB);
        sb.rank = q;
        subs[ex++] = sb;
      }
    }
  }
  if (threadIdx.x == 0) *nsub_total = carry;
}

// Scatter of the indices of one block: ranks as in k_radix_scatter (wave
// ballots, per-wave digit counters).  Blocks of 4096 points (ITEMS 16) stage
// the indices in tile order in LDS, so that a tile's run in the block goes
// out as one piece: what bounds the scatter is the number of separate stores
// (2e6 points in 1600 tiles, runs of 2.6: 28 us, 36 us without staging).
// Blocks of 1024 points have runs of about one and store directly.
template <int ITEMS>
__global__ __launch_bounds__(RT) void k_scatter_wide(
    const uint32_t *keys, size_t M, int keybits, int nbins,
    const uint32_t *offs, const uint32_t *offs_chunk, int nblocks,
    uint32_t *idx_out) {
  constexpr bool STAGE = ITEMS == 16;
  extern __shared__ uint32_t lds[];
  uint32_t *sh = lds;                               // [RT] (scan)
  uint32_t *gofs = lds + RT;                        // [nbins]
  uint32_t *sidx = gofs + nbins;                    // [RT * ITEMS] (STAGE)
  uint16_t *cnt = (uint16_t *)(sidx + (STAGE ? RT * ITEMS : 0));  // [NW][nbins]
  uint16_t *skey = cnt + (size_t)NW * nbins;        // [RT * ITEMS] (STAGE)
  const int tid = threadIdx.x, wave = tid >> 6;
  const unsigned lane = lane_id();
  const unsigned long long below_mask =
      lane ? (~0ull >> (64 - lane)) : 0ull;
  const size_t blk0 = (size_t)blockIdx.x * (RT * ITEMS);
  const size_t c0 = blk0 + (size_t)wave * (64 * ITEMS) + lane;
  uint32_t key[ITEMS], rank[ITEMS];
#pragma unroll
  for (int r = 0; r < ITEMS; ++r) {
    const size_t j = c0 + (size_t)r * 64;
    key[r] = j < M ? keys[j] : 0u;
  }
  for (int c = tid; c < nbins; c += RT) {
    const size_t og = (size_t)c * nblocks + blockIdx.x;
    gofs[c] = offs[og] + offs_chunk[og / STILE];
  }
  for (int c = tid; c < NW * nbins; c += RT) cnt[c] = 0;
  __syncthreads();
  uint16_t *mine = cnt + (size_t)wave * nbins;
#pragma unroll
  for (int r = 0; r < ITEMS; ++r) {
    const bool valid = c0 + (size_t)r * 64 < M;
    const unsigned long long peers = peers_of(key[r], valid, keybits);
    const unsigned long long below = peers & below_mask;
    const uint32_t old = mine[key[r]];
    __builtin_amdgcn_wave_barrier();
    if (valid && below == 0)
      mine[key[r]] = (uint16_t)(old + (uint32_t)__popcll(peers));
    __builtin_amdgcn_wave_barrier();
    rank[r] = old + (uint32_t)__popcll(below);
  }
  __syncthreads();
  // per tile: the waves' prefixes (and, staged, its start in the block)
  if constexpr (STAGE) {
    const int per = (nbins + RT - 1) / RT, d0 = tid * per,
              d1 = min(d0 + per, nbins);
    uint32_t sum = 0, tot;
    for (int c = d0; c < d1; ++c)
#pragma unroll
      for (int w = 0; w < NW; ++w) sum += cnt[w * nbins + c];
    uint32_t run = block_exclusive_scan(sum, sh, tot);
    for (int c = d0; c < d1; ++c) {
      gofs[c] -= run;
#pragma unroll
      for (int w = 0; w < NW; ++w) {
        const uint32_t n = cnt[w * nbins + c];
        cnt[w * nbins + c] = (uint16_t)run;
        run += n;
      }
    }
  } else {
    for (int c = tid; c < nbins; c += RT) {
      uint32_t run = 0;
#pragma unroll
      for (int w = 0; w < NW; ++w) {
        const uint32_t n = cnt[w * nbins + c];
        cnt[w * nbins + c] = (uint16_t)run;
        run += n;
      }
    }
  }
  __syncthreads();
#pragma unroll
  for (int r = 0; r < ITEMS; ++r) {
    const size_t j = c0 + (size_t)r * 64;
    if (j >= M) continue;
    const uint32_t p = mine[key[r]] + rank[r];
    if constexpr (STAGE) {
      sidx[p] = (uint32_t)j;
      skey[p] = (uint16_t)key[r];
    } else {
      idx_out[gofs[key[r]] + p] = (uint32_t)j;
    }
  }
  if constexpr (STAGE) {
    __syncthreads();
    const int n = (int)min((size_t)(RT * ITEMS), M - blk0);
#pragma unroll
    for (int i = 0; i < ITEMS; ++i) {
      const int q = i * RT + tid;
      if (q < n) idx_out[gofs[skey[q]] + (uint32_t)q] = sidx[q];
    }
  }
}

template <typename T>
__global__ void k_gather_coords(const T *c, int ndim, const uint32_t *idx,
                                size_t M, T *out) {
  size_t j = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (j >= M) return;
  size_t s = idx[j];
  for (int d = 0; d < ndim; ++d) out[j * ndim + d] = c[s * ndim + d];
}

__global__ void k_zero16(uint4 *p, size_t n16) {
  size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  size_t stride = (size_t)gridDim.x * blockDim.x;
  for (; i < n16; i += stride) p[i] = make_uint4(0, 0, 0, 0);
}
__global__ void k_zero1(unsigned char *p, size_t n) {
  size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) p[i] = 0;
}

inline unsigned nblk(size_t n, unsigned t) { return (unsigned)((n + t - 1) / t); }
}  // namespace

void launch_fold_keys(const Geo &g, const void *coords, size_t M,
                      uint32_t *keys, uint32_t *hist0, hipStream_t s) {
  if (!M) return;
  const size_t nblocks = (M + RTILE - 1) / RTILE;
  const dim3 grid((unsigned)nblocks), block(RT);
  if (g.ndim == 1)
    hipLaunchKernelGGL(k_fold_keys<1>, grid, block, 0, s, g, coords, M, keys,
                       hist0, (int)nblocks);
  else if (g.ndim == 2)
    hipLaunchKernelGGL(k_fold_keys<2>, grid, block, 0, s, g, coords, M, keys,
                       hist0, (int)nblocks);
  else
    hipLaunchKernelGGL(k_fold_keys<3>, grid, block, 0, s, g, coords, M, keys,
                       hist0, (int)nblocks);
  DMX_HIP(hipGetLastError());
}

size_t scan_workspace(size_t n) {
  size_t nb = (n + STILE - 1) / STILE;
  return (nb + 64) * sizeof(uint32_t);
}

void exclusive_scan_u32(const uint32_t *in, uint32_t *out, size_t n,
                        uint32_t *total, void *work, hipStream_t s) {
  if (!n) return;
  size_t nb = (n + STILE - 1) / STILE;
  // one workgroup walks the chunks one after another (a load latency each):
  // only for one or two chunks; longer arrays take the three-launch scan
  if (nb <= 2) {
    hipLaunchKernelGGL(k_scan_single, dim3(1), dim3(ST), 0, s, in, out, n,
                       total);
    DMX_HIP(hipGetLastError());
    return;
  }
  uint32_t *bsum = (uint32_t *)work;
  hipLaunchKernelGGL(k_scan_blocks, dim3((unsigned)nb), dim3(ST), 0, s, in,
                     out, n, bsum);
  hipLaunchKernelGGL(k_scan_single, dim3(1), dim3(ST), 0, s,
                     (const uint32_t *)bsum, bsum, nb, total);
  hipLaunchKernelGGL(k_scan_add, dim3((unsigned)nb), dim3(ST), 0, s, out, n,
                     (const uint32_t *)bsum);
  DMX_HIP(hipGetLastError());
}

size_t radix_sort_workspace(size_t M) {
  size_t nblocks = (M + RTILE - 1) / RTILE;
  size_t hist = (size_t)RB * nblocks;
  return 4 * M * sizeof(uint32_t) + 2 * hist * sizeof(uint32_t) +
         scan_workspace(hist) + 256;
}

uint32_t *radix_sort_hist0(void *work, size_t M) {
  return (uint32_t *)work + 4 * M;
}

void radix_sort_pairs(const uint32_t *keys_in, size_t M, int keybits,
                      uint32_t *idx_out, uint32_t *keys_out, void *work,
                      size_t work_bytes, hipStream_t s, bool hist0_ready,
                      uint32_t *tb_start_c, uint32_t *tb_end) {
  if (!M) return;
  DMX_ASSERT(work_bytes >= radix_sort_workspace(M), "sort workspace too small");
  size_t nblocks = (M + RTILE - 1) / RTILE;
  size_t hist_n = (size_t)RB * nblocks;
  uint32_t *kbuf[2] = {(uint32_t *)work, (uint32_t *)work + M};
  uint32_t *ibuf[2] = {(uint32_t *)work + 2 * M, (uint32_t *)work + 3 * M};
  uint32_t *hist = (uint32_t *)work + 4 * M;
  uint32_t *offs = hist + hist_n;
  void *sw = offs + hist_n;
  int npass = keybits <= 0 ? 1 : (keybits + 7) / 8;
  const uint32_t *kin = keys_in;
  const uint32_t *iin = nullptr;  // identity permutation on the first pass
  for (int p = 0; p < npass; ++p) {
    bool last = p == npass - 1;
    uint32_t *kout = last ? keys_out : kbuf[p & 1];
    uint32_t *iout = last ? idx_out : ibuf[p & 1];
    uint32_t *bsum = (uint32_t *)sw;
    radix_pass_offsets(kin, M, 8 * p, hist, p == 0 && hist0_ready, offs,
                       bsum, s);
    hipLaunchKernelGGL(k_radix_scatter, dim3((unsigned)nblocks), dim3(RT), 0,
                       s, kin, iin, M, 8 * p, (const uint32_t *)offs,
                       (const uint32_t *)bsum,
                       (int)nblocks, kout, iout, last ? tb_start_c : nullptr,
                       last ? tb_end : nullptr);
    DMX_HIP(hipGetLastError());
    kin = kout;
    iin = iout;
  }
}

void radix_pass_offsets(const uint32_t *keys, size_t M, int shift,
                        uint32_t *hist, bool hist_ready, uint32_t *offs,
                        uint32_t *bsum, hipStream_t s) {
  const size_t nblocks = (M + RTILE - 1) / RTILE;
  const size_t hist_n = (size_t)RB * nblocks;
  if (!hist_ready)
    hipLaunchKernelGGL(k_radix_hist, dim3((unsigned)nblocks), dim3(RT), 0, s,
                       keys, M, shift, hist, (int)nblocks);
  // digit-major offsets: per-chunk scans and the scan of the chunk sums;
  // the scatter adds the two
  const size_t nch = (hist_n + STILE - 1) / STILE;
  hipLaunchKernelGGL(k_scan_blocks, dim3((unsigned)nch), dim3(ST), 0, s,
                     (const uint32_t *)hist, offs, hist_n, bsum);
  hipLaunchKernelGGL(k_scan_single, dim3(1), dim3(ST), 0, s,
                     (const uint32_t *)bsum, bsum, nch, nullptr);
  DMX_HIP(hipGetLastError());
}

void launch_tile_subs(size_t ntiles, uint32_t *counts, uint32_t *tstart,
                      const uint32_t *tend, uint32_t *nsub,
                      uint32_t *sub_start, Sub *subs, uint32_t *nsub_total,
                      void *scanwork, hipStream_t s) {
  DMX_ASSERT(ntiles > 0, "internal: no tiles");
  if (ntiles <= (size_t)ST * TS_ITEMS) {
    hipLaunchKernelGGL(k_tile_subs_one, dim3(1), dim3(ST), 0, s,
                       tstart, tend, ntiles, counts, nsub, sub_start, subs,
                       nsub_total);
    DMX_HIP(hipGetLastError());
    return;
  }
  hipLaunchKernelGGL(k_counts_nsub, dim3(nblk(ntiles, 256)), dim3(256), 0, s,
                     tstart, tend, ntiles, counts, nsub);
  exclusive_scan_u32(nsub, sub_start, ntiles, nsub_total, scanwork, s);
  hipLaunchKernelGGL(k_fill_subs, dim3(nblk(ntiles, 256)), dim3(256), 0, s,
                     counts, tstart, (const uint32_t *)nsub,
                     (const uint32_t *)sub_start, ntiles, subs);
  DMX_HIP(hipGetLastError());
}

// Whether one launch or one counting pass over whole keys builds the index.
// The pass's table has tiles x blocks entries and each of its blocks clears
// and scans a counter per tile and wave, while the runs it writes get
// shorter; the 8-bit passes do not depend on the tiles.  Measured where the
// two meet (uniform points, whole calls): 7e6 points in 1700 tiles, 1.5e6 in
// 2800, 6e5 in 3950, which is M * tiles^3 = 3.5e16 throughout (400^2 modes,
// 784 tiles, still gain at 1e7 points: 593 -> 531 us; 950^2, 3969 tiles, 3e6
// points would take 279 instead of 225, 7e5 in 1-D, 1e7 points in 2740
// tiles, 648 instead of 554).
bool index_one_pass(size_t M, size_t ntiles) {
  if (ntiles > (size_t)WIDE_TILES) return false;
  const double t = (double)ntiles;
  return M <= (size_t)SMALL_M || (double)M * t * t * t <= 3.5e16;
}

bool launch_index(const Geo &g, const void *coords, size_t M, int keybits,
                  size_t ntiles, uint32_t *idx, uint32_t *keys, void *work,
                  uint32_t *counts, uint32_t *tstart, uint32_t *nsub,
                  uint32_t *sub_start, Sub *subs, uint32_t *nsub_total,
                  hipStream_t s) {
  if (!M || !index_one_pass(M, ntiles)) return false;
#define DMX_BYDIM(KERNEL, ...)                              \
  switch (g.ndim) {                                         \
    case 1: KERNEL(1, __VA_ARGS__); break;                  \
    case 2: KERNEL(2, __VA_ARGS__); break;                  \
    default: KERNEL(3, __VA_ARGS__); break;                 \
  }
  if (M <= (size_t)SMALL_M) {
#define DMX_SMALL(D, _)                                                      \
  hipLaunchKernelGGL(k_index_small<D>, dim3(1), dim3(SMALL_T), 0, s, g,      \
                     coords, (int)M, keybits, (int)ntiles, idx, counts,      \
                     tstart, nsub, sub_start, subs, nsub_total)
    DMX_BYDIM(DMX_SMALL, 0)
#undef DMX_SMALL
    DMX_HIP(hipGetLastError());
    return true;
  }
  // blocks of 1024 points fill the chip up to about 5e5 points; the table
  // (histogram and offsets, tiles x blocks) has to fit the workspace of the
  // 8-bit passes, which this sort needs none of otherwise
  const size_t room = radix_sort_workspace(M) / sizeof(uint32_t);
  auto fits = [&](size_t items) {
    const size_t nb = (M + RT * items - 1) / (RT * items);
    const size_t tab = ntiles * nb;
    return (tab + STILE - 1) / STILE <= (size_t)WIDE_CHUNKS &&
           2 * tab + tab / STILE + 64 <= room;
  };
  const bool four = M <= ((size_t)1 << 19) && fits(4);
  if (!four && !fits(16)) return false;
  const size_t items = four ? 4 : 16;
  const size_t nb = (M + RT * items - 1) / (RT * items), tab = ntiles * nb;
  uint32_t *hist = (uint32_t *)work, *offs = hist + tab, *bsum = offs + tab;
  const size_t nch = (tab + STILE - 1) / STILE;
  const dim3 grid((unsigned)nb), block(RT);
  const size_t lh = ntiles * 4, ls = RT * 4 + ntiles * (4 + 2 * NW);
#define DMX_FOLD(D, I)                                                       \
  hipLaunchKernelGGL((k_fold_wide<D, I>), grid, block, lh, s, g, coords, M,  \
                     keys, hist, (int)ntiles, (int)nb)
  if (four) {
    DMX_BYDIM(DMX_FOLD, 4)
  } else {
    DMX_BYDIM(DMX_FOLD, 16)
  }
#undef DMX_FOLD
#undef DMX_BYDIM
  hipLaunchKernelGGL(k_scan_blocks, dim3((unsigned)nch), dim3(ST), 0, s,
                     (const uint32_t *)hist, offs, tab, bsum);
  hipLaunchKernelGGL(k_tiles_wide, dim3(1), dim3(1024), 0, s,
                     (const uint32_t *)offs, bsum, (int)nch, M, (int)ntiles,
                     (int)nb, counts, tstart, nsub, sub_start, subs,
                     nsub_total);
  if (four)
    hipLaunchKernelGGL(k_scatter_wide<4>, grid, block, ls, s,
                       (const uint32_t *)keys, M, keybits, (int)ntiles,
                       (const uint32_t *)offs, (const uint32_t *)bsum,
                       (int)nb, idx);
  else {
    const size_t lst = ls + (size_t)RT * 16 * (4 + 2);  // the staged block
    allow_big_lds(k_scatter_wide<16>, lst);
    hipLaunchKernelGGL(k_scatter_wide<16>, grid, block, lst, s,
                       (const uint32_t *)keys, M, keybits, (int)ntiles,
                       (const uint32_t *)offs, (const uint32_t *)bsum,
                       (int)nb, idx);
  }
  DMX_HIP(hipGetLastError());
  return true;
}

void launch_tiles_range(const uint32_t *start, size_t ntiles, uint32_t nk,
                        const KeyRanges &ranges, size_t nranges,
                        uint32_t *nsub, uint32_t *sub_start, Sub *subs,
                        size_t list, uint32_t *nsub_total, hipStream_t s) {
  DMX_ASSERT(nranges <= (size_t)KEY_RANGES, "internal: too many key ranges");
  hipLaunchKernelGGL(k_tiles_range, dim3((unsigned)nranges), dim3(1024), 0, s,
                     start, ntiles, nk, ranges, nsub, sub_start, subs, list,
                     nsub_total);
  DMX_HIP(hipGetLastError());
}

void launch_gather_coords(const void *coords, int coord_f32, int ndim,
                          const uint32_t *idx, size_t M, void *out,
                          hipStream_t s) {
  if (!M) return;
  if (coord_f32)
    hipLaunchKernelGGL(k_gather_coords<float>, dim3(nblk(M, 256)), dim3(256),
                       0, s, (const float *)coords, ndim, idx, M,
                       (float *)out);
  else
    hipLaunchKernelGGL(k_gather_coords<double>, dim3(nblk(M, 256)), dim3(256),
                       0, s, (const double *)coords, ndim, idx, M,
                       (double *)out);
  DMX_HIP(hipGetLastError());
}

void launch_zero(void *p, size_t bytes, hipStream_t s) {
  if (!bytes) return;
  size_t n16 = bytes / 16, rest = bytes - n16 * 16;
  if (n16) {
    unsigned nb = (unsigned)std::min<size_t>((n16 + 255) / 256, 8192);
    hipLaunchKernelGGL(k_zero16, dim3(nb), dim3(256), 0, s, (uint4 *)p, n16);
  }
  if (rest)
    hipLaunchKernelGGL(k_zero1, dim3(1), dim3(256), 0, s,
                       (unsigned char *)p + n16 * 16, rest);
  DMX_HIP(hipGetLastError());
}

}  // namespace dmx
