// sf_cull.hip -- device preparation of spatial sort and culling (gfx950).
//
// For a slice whose largest distance edge is small against its extent, the binary32 records are
// put in Morton (Z-curve) order of their key-space coordinates (flat: x; sphere: the unit
// vector), so that a group of consecutive records is spatially compact, and only pairs of groups
// whose bounding boxes are not farther apart than the largest edge are evaluated.  This file
// computes, on the device and in the caller's stream:
//   cull_coords   key-space coordinates per point and a bounding box per workgroup
//   cull_reduce   the slice's bounding box, its largest coordinate magnitude, a non-finite flag
//   cull_keys     Morton keys (8 or 10 bits per axis of the bounding box)
//   sort_*        stable radix sort of the keys, carrying point indices: the record order
//   cull_groups   the bounding box of every group of kGroup consecutive records
//   cull_units    the work units: a wave's 64 rows and one or two column groups within reach
//                 (launch_cull_count: their number alone, for wide row blocks)
// The host reads back the slice box and the number of units (kCullInfo words).
#include <hip/hip_runtime.h>

#include "sf_internal.h"
#include "sfmath.h"

namespace sfk {

namespace {

constexpr int kCullBlock = 256;

// key-space coordinates of point i (x is point-major, W values per point)
__device__ void cull_point(const double *x, int64_t i, int W, int D, int geom, double c[3]) {
  if (geom == 0) {
    for (int k = 0; k < 3; ++k) c[k] = k < D ? x[(size_t)W * i + k] : 0.0;
    return;
  }
  double so, co, sa, ca;
  if (geom == 1) {
    sf_sincosd(x[2 * i], &so, &co);
    sf_sincosd(x[2 * i + 1], &sa, &ca);
  } else {
    sf_sincos(x[2 * i], &so, &co);
    sf_sincos(x[2 * i + 1], &sa, &ca);
  }
  c[0] = ca * co;
  c[1] = ca * so;
  c[2] = sa;
}

// per workgroup: lo[3], hi[3], non-finite count, largest |coordinate| (8 doubles)
__global__ void __launch_bounds__(kCullBlock) cull_coords(const double *x, int64_t N, int W, int D,
                                                          int geom, double *kc, double *part) {
  __shared__ double red[8][kCullBlock];
  double lo[3] = {INFINITY, INFINITY, INFINITY}, hi[3] = {-INFINITY, -INFINITY, -INFINITY};
  double bad = 0.0, cmax = 0.0;
  const int64_t i = (int64_t)blockIdx.x * kCullBlock + threadIdx.x;
  if (i < N) {
    double c[3];
    cull_point(x, i, W, D, geom, c);
    for (int k = 0; k < 3; ++k) {
      kc[3 * i + k] = c[k];
      if (!(fabs(c[k]) < INFINITY)) bad = 1.0;
      lo[k] = c[k];
      hi[k] = c[k];
      cmax = fmax(cmax, fabs(c[k]));
    }
  }
  const int t = threadIdx.x;
  for (int k = 0; k < 3; ++k) {
    red[k][t] = lo[k];
    red[3 + k][t] = hi[k];
  }
  red[6][t] = bad;
  red[7][t] = cmax;
  __syncthreads();
  for (int w = kCullBlock / 2; w > 0; w >>= 1) {
    if (t < w) {
      for (int k = 0; k < 3; ++k) {
        red[k][t] = fmin(red[k][t], red[k][t + w]);
        red[3 + k][t] = fmax(red[3 + k][t], red[3 + k][t + w]);
      }
      red[6][t] += red[6][t + w];
      red[7][t] = fmax(red[7][t], red[7][t + w]);
    }
    __syncthreads();
  }
  if (t < 8) part[(size_t)blockIdx.x * 8 + t] = red[t][0];
}

// one workgroup: combine nblk partial boxes into glob (same 8-double layout)
__global__ void __launch_bounds__(kCullBlock) cull_reduce(const double *part, int nblk, double *glob) {
  static_assert(kCullInfo <= kCullBlock, "");
  __shared__ double red[8][kCullBlock];
  const int t = threadIdx.x;
  double v[8] = {INFINITY, INFINITY, INFINITY, -INFINITY, -INFINITY, -INFINITY, 0.0, 0.0};
  for (int b = t; b < nblk; b += kCullBlock) {
    const double *p = part + (size_t)b * 8;
    for (int k = 0; k < 3; ++k) {
      v[k] = fmin(v[k], p[k]);
      v[3 + k] = fmax(v[3 + k], p[3 + k]);
    }
    v[6] += p[6];
    v[7] = fmax(v[7], p[7]);
  }
  for (int k = 0; k < 8; ++k) red[k][t] = v[k];
  __syncthreads();
  for (int w = kCullBlock / 2; w > 0; w >>= 1) {
    if (t < w) {
      for (int k = 0; k < 3; ++k) {
        red[k][t] = fmin(red[k][t], red[k][t + w]);
        red[3 + k][t] = fmax(red[3 + k][t], red[3 + k][t + w]);
      }
      red[6][t] += red[6][t + w];
      red[7][t] = fmax(red[7][t], red[7][t + w]);
    }
    __syncthreads();
  }
  if (t < 8) glob[t] = red[t][0];
  if (t >= 8 && t < kCullInfo) ((unsigned long long *)glob)[t] = 0ull;  // the unit counters
}

__device__ uint32_t spread10(uint32_t v) {
  v &= 1023u;
  v = (v | (v << 16)) & 0x030000FFu;
  v = (v | (v << 8)) & 0x0300F00Fu;
  v = (v | (v << 4)) & 0x030C30C3u;
  v = (v | (v << 2)) & 0x09249249u;
  return v;
}

__global__ void __launch_bounds__(kCullBlock) cull_keys(const double *kc, int64_t N, const double *glob,
                                                        int bits, uint32_t *key) {
  const int64_t i = (int64_t)blockIdx.x * kCullBlock + threadIdx.x;
  if (i >= N) return;
  uint32_t q[3];
  for (int k = 0; k < 3; ++k) {
    const double w = glob[3 + k] - glob[k];
    const double t = w > 0 ? (kc[3 * i + k] - glob[k]) / w : 0.0;
    // a non-finite coordinate (the host then refuses culling) still gets an in-range key
    const double n = (double)(1 << bits);
    q[k] = (uint32_t)fmin(n - 1.0, fmax(0.0, floor(t * n)));
  }
  key[i] = spread10(q[0]) | (spread10(q[1]) << 1) | (spread10(q[2]) << 2);
}

// Stable radix sort of 24- or 30-bit keys in two passes of 12 bits or three of 10, each a count per
// workgroup, a scan over the workgroups and a scatter.  A workgroup takes `per` keys in a row (a
// multiple of kSortTile; 256 workgroups at most), tile after tile; a wave a quarter of each.  What
// bounds it at the sizes in use is launches: N = 262144 took 18 of a merge sort's (about 170 us of a
// 747 us call), six of these take 60.
constexpr int kSortRounds = 8;                          // keys per lane and tile
constexpr int kSortTile = kCullBlock * kSortRounds;
template <int BITS>
__global__ void __launch_bounds__(kCullBlock) sort_count(const uint32_t *key, int64_t N, int64_t per, int shift,
                                                         uint32_t *hist) {
  constexpr int R = 1 << BITS;
  __shared__ uint32_t h[R];
  for (int d = threadIdx.x; d < R; d += kCullBlock) h[d] = 0u;
  __syncthreads();
  const int64_t k0 = (int64_t)blockIdx.x * per, k1 = k0 + per < N ? k0 + per : N;
  for (int64_t k = k0 + threadIdx.x; k < k1; k += kCullBlock) atomicAdd(&h[(key[k] >> shift) & (R - 1)], 1u);
  __syncthreads();
  for (int d = threadIdx.x; d < R; d += kCullBlock) hist[(size_t)blockIdx.x * R + d] = h[d];
}

// per digit: counts of the workgroups to their exclusive sums, and the total (one thread per digit;
// 16 loads in flight, since the sums are a chain)
template <int BITS>
__global__ void __launch_bounds__(64) sort_scan(uint32_t *hist, int nblk, uint32_t *total) {
  constexpr int R = 1 << BITS, U = 16;
  const int d = (int)blockIdx.x * 64 + (int)threadIdx.x;
  uint32_t run = 0u;
  for (int b = 0; b < nblk; b += U) {
    uint32_t v[U];
#pragma unroll
    for (int k = 0; k < U; ++k) v[k] = b + k < nblk ? hist[(size_t)(b + k) * R + d] : 0u;
#pragma unroll
    for (int k = 0; k < U; ++k) {
      if (b + k < nblk) hist[(size_t)(b + k) * R + d] = run;
      run += v[k];
    }
  }
  total[d] = run;
}

// keys (and indices; null: the identity) of the workgroup to their places; key_out null on the last pass
template <int BITS>
__global__ void __launch_bounds__(kCullBlock) sort_scatter(const uint32_t *key, const int32_t *idx, int64_t N,
                                                           int64_t per, int shift, const uint32_t *hist,
                                                           const uint32_t *total, uint32_t *key_out,
                                                           int32_t *idx_out) {
  constexpr int R = 1 << BITS, W = kCullBlock / 64, Q = R / kCullBlock;
  __shared__ uint32_t base[R];          // next place of each digit
  __shared__ unsigned short wc[W][R];   // counts per wave of a tile, then what precedes the wave's
  __shared__ uint32_t wsum[W];
  const int t = threadIdx.x, w = t >> 6, lane = t & 63;
  {  // exclusive scan of the totals: thread t has the digits from t Q on
    uint32_t v[Q], sum = 0u;
#pragma unroll
    for (int q = 0; q < Q; ++q) {
      v[q] = total[t * Q + q];
      sum += v[q];
    }
    uint32_t inc = sum;
    for (int o = 1; o < 64; o <<= 1) {
      const uint32_t a = __shfl_up(inc, o);
      if (lane >= o) inc += a;
    }
    if (lane == 63) wsum[w] = inc;
    __syncthreads();
    uint32_t run = inc - sum;
    for (int k = 0; k < w; ++k) run += wsum[k];
#pragma unroll
    for (int q = 0; q < Q; ++q) {
      base[t * Q + q] = run + hist[(size_t)blockIdx.x * R + t * Q + q];
      run += v[q];
    }
  }
  const int64_t k0 = (int64_t)blockIdx.x * per, k1 = k0 + per < N ? k0 + per : N;
  for (int64_t kt = k0; kt < k1; kt += kSortTile) {
    for (int d = t; d < W * R; d += kCullBlock) (&wc[0][0])[d] = 0;
    __syncthreads();
    uint32_t kk[kSortRounds], rank[kSortRounds];
    const int64_t kw = kt + w * (64 * kSortRounds) + lane;
#pragma unroll
    for (int r = 0; r < kSortRounds; ++r) kk[r] = kw + 64 * r < k1 ? key[kw + 64 * r] : 0u;
#pragma unroll
    for (int r = 0; r < kSortRounds; ++r) {
      const bool ok = kw + 64 * r < k1;
      const uint32_t d = (kk[r] >> shift) & (R - 1);
      unsigned long long peers = __ballot(ok);  // lanes with the same digit
#pragma unroll
      for (int b = 0; b < BITS; ++b) {
        const unsigned long long one = __ballot((d >> b) & 1u);
        peers &= (d >> b) & 1u ? one : ~one;
      }
      const unsigned before = (unsigned)__popcll(peers & ((1ull << lane) - 1ull));
      const unsigned have = wc[w][d];
      rank[r] = have + before;
      // the first of the lanes adds them all; LDS operations of a wave complete in order
      if (ok && before == 0u) wc[w][d] = (unsigned short)(have + (unsigned)__popcll(peers));
      __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
      __builtin_amdgcn_wave_barrier();
    }
    __syncthreads();
    unsigned all[Q];
#pragma unroll
    for (int q = 0; q < Q; ++q) {
      const int d = t + q * kCullBlock;
      unsigned run = 0u;
      for (int k = 0; k < W; ++k) {
        const unsigned c = wc[k][d];
        wc[k][d] = (unsigned short)run;
        run += c;
      }
      all[q] = run;
    }
    __syncthreads();
#pragma unroll
    for (int r = 0; r < kSortRounds; ++r) {
      const int64_t k = kw + 64 * r;
      if (k < k1) {
        const uint32_t d = (kk[r] >> shift) & (R - 1);
        const uint32_t pos = base[d] + wc[w][d] + rank[r];
        if (key_out) key_out[pos] = kk[r];
        idx_out[pos] = idx ? idx[k] : (int32_t)k;
      }
    }
    __syncthreads();
#pragma unroll
    for (int q = 0; q < Q; ++q) base[t + q * kCullBlock] += all[q];
  }
}

// boxes (lo[3], hi[3]) of groups of 32 consecutive records, rounded outwards to binary32: two
// groups per wave
__global__ void __launch_bounds__(kCullBlock) cull_groups(const double *kc, const int32_t *perm, int64_t N,
                                                          float *gbox) {
  const int64_t k = (int64_t)blockIdx.x * kCullBlock + threadIdx.x;
  const int64_t i = perm[k < N ? k : N - 1];
  float lo[3], hi[3];
  for (int c = 0; c < 3; ++c) {
    const double v = kc[3 * i + c];
    lo[c] = __double2float_rd(v);
    hi[c] = __double2float_ru(v);
  }
  for (int o = 16; o > 0; o >>= 1)
    for (int c = 0; c < 3; ++c) {
      lo[c] = fminf(lo[c], __shfl_xor(lo[c], o));
      hi[c] = fmaxf(hi[c], __shfl_xor(hi[c], o));
    }
  if ((threadIdx.x & 31) == 0 && k < N)
    for (int c = 0; c < 3; ++c) {
      gbox[6 * (k / 32) + c] = lo[c];
      gbox[6 * (k / 32) + 3 + c] = hi[c];
    }
}

// Work units of a slice: row block rb (64 K records) with the pair of column groups (64 records) at
// j0, as far as their boxes are in reach and some column lies above some row.  The K waves of a row block
// take its rows K apart (unit k: rows rb 64 K + k + K lane).  One wave per row
// block and kUnitSpan runs of 64 groups, one group per lane.  The boxes are rounded outwards to
// binary32 and the limit carries a margin, so no counted pair is lost.  WRITE false: their number is
// added to *count and the squared limit goes to *lim (both in the slice's info); true: they are
// written to units (cap of them at most), where *count is the next free one.
// Latency bounds it: 30 and 40 us at N = 262144 (4096 row blocks, 8192 groups, 18e6 tests); spans of 4
// runs, with four times the reservations on one counter, made the whole call 4 % slower.
constexpr int kUnitSpan = 16;
template <bool WRITE>
__global__ void __launch_bounds__(kCullBlock) cull_units(const float *gbox, int64_t N, const double *info,
                                                         double reach, int K, int slice, Item *units,
                                                         unsigned long long cap, unsigned long long *count,
                                                         double *lim) {
  constexpr int W = kCullBlock / 64;
  __shared__ unsigned long long masks[W][kUnitSpan];
  __shared__ unsigned tot[W];
  __shared__ unsigned long long base;
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  // a pair of boxes farther apart than this holds no counted pair: relative 1e-6 plus the rounding of
  // coordinates of the slice's magnitude, and the rounding of three binary32 squares and their sum
  const double l = reach * (1.0 + 1e-6) + 1e-13 * fmax(1.0, info[7]);
  const float lim2 = __double2float_ru(l * l * (1.0 + 1e-5) + 1e-30);
  if (!WRITE && lim && blockIdx.x == 0 && blockIdx.y == 0 && threadIdx.x == 0) *lim = l;
  const int64_t rb = (int64_t)blockIdx.x * W + w;
  const int64_t last = (N - 1) / kGroup;
  unsigned mine = 0;
  const int64_t g0 = 2 * K * rb;  // first group of the row block
  if (rb * 64 * K < N) {
    float lo[3], hi[3];
    {
      const int64_t ga = g0 + (lane & (2 * K - 1));
      const float *a = gbox + 6 * (ga < last ? ga : last);
      for (int k = 0; k < 3; ++k) {
        lo[k] = a[k];
        hi[k] = a[3 + k];
      }
    }
    for (int o = K; o > 0; o >>= 1)
      for (int k = 0; k < 3; ++k) {
        lo[k] = fminf(lo[k], __shfl_xor(lo[k], o));
        hi[k] = fmaxf(hi[k], __shfl_xor(hi[k], o));
      }
#pragma unroll 4  // (loads of several runs in flight)
    for (int t = 0; t < kUnitSpan; ++t) {
      const int64_t g = ((int64_t)blockIdx.y * kUnitSpan + t) * 64 + lane;
      unsigned long long m = 0ull;
      if ((g | 63) >= g0 && (g & ~63ll) <= last) {  // (the same for the whole wave)
        const float *b = gbox + 6 * (g < last ? g : last);
        float d2 = 0.f;
        for (int k = 0; k < 3; ++k) {
          const float gap = fmaxf(0.f, fmaxf(b[k] - hi[k], lo[k] - b[3 + k]));
          d2 = __builtin_fmaf(gap, gap, d2);
        }
        m = __ballot(g <= last && g >= g0 && d2 <= lim2);
      }
      if (lane == 0) masks[w][t] = m;
      mine += (unsigned)K * (unsigned)__popcll((m | (m >> 1)) & 0x5555555555555555ull);
    }
  } else if (lane < kUnitSpan) {
    masks[w][lane] = 0ull;
  }
  if (lane == 0) tot[w] = mine;
  __syncthreads();
  if (threadIdx.x == 0) {
    unsigned n = 0;
    for (int k = 0; k < W; ++k) n += tot[k];
    base = n ? atomicAdd(count, (unsigned long long)n) : 0ull;
  }
  if constexpr (WRITE) {
    __syncthreads();
    unsigned long long o = base;
    for (int k = 0; k < w; ++k) o += tot[k];
    for (int t = 0; t < kUnitSpan; ++t) {
      const unsigned long long m = masks[w][t];
      const unsigned long long pairs = (m | (m >> 1)) & 0x5555555555555555ull;
      if ((pairs >> lane) & 1ull) {
        const unsigned long long k = o + (unsigned)K * (unsigned)__popcll(pairs & ((1ull << lane) - 1ull));
        const int64_t g = ((int64_t)blockIdx.y * kUnitSpan + t) * 64 + lane;
        const int64_t j0 = (g + ((m >> lane) & 1ull ? 0 : 1)) * kGroup;
        const int64_t j1 = (g + ((m >> lane) & 2ull ? 2 : 1)) * kGroup;
        for (int r = 0; r < K; ++r)
          if (k + r < cap)
            units[k + r] = Item{slice, (int32_t)(rb * 64 * K + r) | (K > 1 ? kWideUnit : 0), (int32_t)j0,
                                (int32_t)(j1 < N ? j1 : N)};
      }
      o += (unsigned)K * (unsigned)__popcll(pairs);
    }
  }
}

dim3 unit_grid(int64_t N, int K) {
  const int64_t rows = (N + 64 * K - 1) / (64 * K), groups = (N + kGroup - 1) / kGroup;
  return dim3((unsigned)((rows + kCullBlock / 64 - 1) / (kCullBlock / 64)),
              (unsigned)((groups + 64 * kUnitSpan - 1) / (64 * kUnitSpan)));
}

struct CullWs {
  double *kc, *part;
  uint32_t *key_a, *key_b, *hist, *total;
  int32_t *idx;
  size_t total_bytes;
};

size_t align256(size_t b) { return (b + 255) & ~(size_t)255; }

// keys per workgroup of the sort, and its workgroups
int64_t sort_per(int64_t N) {
  const int64_t tiles = (N + kSortTile - 1) / kSortTile;
  return (tiles + 255) / 256 * kSortTile;
}
int sort_blocks(int64_t N) { return (int)((N + sort_per(N) - 1) / sort_per(N)); }

// carves the workspace at base (sizes only when base is null)
void cull_ws_layout(int64_t N, char *base, CullWs &w) {
  const int64_t nblk = (N + kCullBlock - 1) / kCullBlock;
  size_t o = 0;
  auto at = [&](size_t bytes) {
    void *q = base ? (void *)(base + o) : nullptr;
    o += align256(bytes);
    return q;
  };
  w.kc = (double *)at(sizeof(double) * 3 * N);
  w.part = (double *)at(sizeof(double) * 8 * nblk);
  w.key_a = (uint32_t *)at(sizeof(uint32_t) * N);
  w.key_b = (uint32_t *)at(sizeof(uint32_t) * N);
  w.idx = (int32_t *)at(sizeof(int32_t) * N);
  w.hist = (uint32_t *)at(sizeof(uint32_t) * 4096 * (size_t)sort_blocks(N));
  w.total = (uint32_t *)at(sizeof(uint32_t) * 4096);
  w.total_bytes = o;
}

// one pass on the BITS digits from shift on
template <int BITS>
hipError_t sort_pass(const CullWs &w, int64_t N, int shift, const uint32_t *key, const int32_t *idx, uint32_t *key_out,
                     int32_t *idx_out, hipStream_t st) {
  const int nb = sort_blocks(N);
  const int64_t per = sort_per(N);
  hipLaunchKernelGGL(sort_count<BITS>, dim3(nb), dim3(kCullBlock), 0, st, key, N, per, shift, w.hist);
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) return e;
  hipLaunchKernelGGL(sort_scan<BITS>, dim3((1 << BITS) / 64), dim3(64), 0, st, w.hist, nb, w.total);
  if ((e = hipGetLastError()) != hipSuccess) return e;
  hipLaunchKernelGGL(sort_scatter<BITS>, dim3(nb), dim3(kCullBlock), 0, st, key, idx, N, per, shift,
                     (const uint32_t *)w.hist, (const uint32_t *)w.total, key_out, idx_out);
  return hipGetLastError();
}

}  // namespace

size_t cull_workspace_bytes(int64_t N) {
  CullWs w;
  cull_ws_layout(N, nullptr, w);
  return w.total_bytes;
}

// x: the slice's positions (device, point-major, W per point); geom 0 flat, 1 sphere in degrees,
// 2 sphere in radians; bits: of the Morton key per axis, 8 or 10.  Writes the record order to perm (N
// entries), to gbox one box per kGroup records (6 floats each), and to info (kCullInfo words) the slice
// box (8 doubles: lo[3], hi[3], non-finite count, largest |coordinate|), the number of work units of row
// blocks of 64 within `reach` (an unsigned 64-bit integer), the distance beyond which they were left out,
// and zeros for launch_cull_units and launch_cull_count.  ws: cull_workspace_bytes(N) bytes of device memory.
hipError_t launch_cull(const double *x, int64_t N, int W, int D, int geom, double reach, int bits, void *ws,
                       int32_t *perm, double *info, float *gbox, hipStream_t st) {
  static_assert(kGroup == 32, "cull_groups reduces over half waves, cull_units takes two groups to 64 rows");
  if (N < 1 || N > kWideUnit || (bits != 8 && bits != 10)) return hipErrorInvalidValue;
  CullWs w;
  cull_ws_layout(N, (char *)ws, w);
  const int nblk = (int)((N + kCullBlock - 1) / kCullBlock);
  hipError_t e;
  hipLaunchKernelGGL(cull_coords, dim3(nblk), dim3(kCullBlock), 0, st, x, N, W, D, geom, w.kc, w.part);
  if ((e = hipGetLastError()) != hipSuccess) return e;
  hipLaunchKernelGGL(cull_reduce, dim3(1), dim3(kCullBlock), 0, st, (const double *)w.part, nblk, info);
  if ((e = hipGetLastError()) != hipSuccess) return e;
  hipLaunchKernelGGL(cull_keys, dim3(nblk), dim3(kCullBlock), 0, st, (const double *)w.kc, N,
                     (const double *)info, bits, w.key_a);
  if ((e = hipGetLastError()) != hipSuccess) return e;
  if (bits == 8) {
    e = sort_pass<12>(w, N, 0, w.key_a, nullptr, w.key_b, w.idx, st);
    if (e == hipSuccess) e = sort_pass<12>(w, N, 12, w.key_b, w.idx, nullptr, perm, st);
  } else {
    e = sort_pass<10>(w, N, 0, w.key_a, nullptr, w.key_b, perm, st);
    if (e == hipSuccess) e = sort_pass<10>(w, N, 10, w.key_b, perm, w.key_a, w.idx, st);
    if (e == hipSuccess) e = sort_pass<10>(w, N, 20, w.key_a, w.idx, nullptr, perm, st);
  }
  if (e != hipSuccess) return e;
  hipLaunchKernelGGL(cull_groups, dim3(nblk), dim3(kCullBlock), 0, st, (const double *)w.kc,
                     (const int32_t *)perm, N, gbox);
  if ((e = hipGetLastError()) != hipSuccess) return e;
  hipLaunchKernelGGL(cull_units<false>, unit_grid(N, 1), dim3(kCullBlock), 0, st, (const float *)gbox, N,
                     (const double *)info, reach, 1, 0, (Item *)nullptr, 0ull, (unsigned long long *)(info + 8),
                     info + 9);
  return hipGetLastError();
}

// Counts the work units of row blocks of 64 K records (K: kWideRows) into info word 11.
hipError_t launch_cull_count(const float *gbox, int64_t N, double *info, double reach, int K, hipStream_t st) {
  static_assert(kWideRows > 1 && kWideRows <= 32 && (kWideRows & (kWideRows - 1)) == 0, "a wave reduces 2 K boxes");
  hipLaunchKernelGGL(cull_units<false>, unit_grid(N, K), dim3(kCullBlock), 0, st, gbox, N, (const double *)info, reach,
                     K, 0, (Item *)nullptr, 0ull, (unsigned long long *)(info + 11), (double *)nullptr);
  return hipGetLastError();
}

// Writes the slice's n work units (their number and the slice's info from launch_cull, or
// launch_cull_count) to units.
hipError_t launch_cull_units(const float *gbox, int64_t N, double *info, double reach, int K, int slice, Item *units,
                             int64_t n, hipStream_t st) {
  hipLaunchKernelGGL(cull_units<true>, unit_grid(N, K), dim3(kCullBlock), 0, st, gbox, N, (const double *)info, reach,
                     K, slice, units, (unsigned long long)n, (unsigned long long *)(info + 10), (double *)nullptr);
  return hipGetLastError();
}

}  // namespace sfk
