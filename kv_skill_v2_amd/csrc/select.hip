// Slot top-k selection read (D8, xenc/topk_read.py): the reader's query at a selection layer
// picks the k library slots whose selection keys score highest, and the read then runs over
// those k slots only, with one softmax.
//
//   select_scores_kernel  s[b, i] = pool_h <q[b, h], K[i, h / G]>  (pool = max or mean over the
//                         query heads, GQA group G = n_q / n_kv), -inf on invalid slots
//                         (xenc/topk_read.py:205-226)
//   topk_rows_kernel      the k largest s[b, :] per row, in descending order, ties to the lower
//                         index (xenc/topk_read.py:237-240; torch.topk leaves ties unspecified)
//   gather_pages_kernel   the selected slot rows copied, in selection order, into a compact page
//                         per selection set, zero-padded; the existing decode and MFMA read
//                         kernels then read that one-chunk library with route weight 1, which is
//                         the read of the selected set (xenc/topk_read.py:383-414)
#include <algorithm>

#include "xenc_common.h"

namespace xenc {
namespace {

typedef unsigned int u32x4 __attribute__((ext_vector_type(4)));

// ------------------------------------------------------------------------------------------
// Scores: one wave per (slot, query row); lanes run over hd for each kv head.  A workgroup of
// 4 waves takes 4 consecutive slots for one query row.  The keys dominate the traffic
// (n_kv * hd * 4 bytes per slot per query row); query rows are few (the batch at one position).
__global__ __launch_bounds__(256) void select_scores_kernel(
    const float* __restrict__ q, int n_q, int n_kv, int hd, const float* __restrict__ keys, int S,
    const unsigned char* __restrict__ valid, int pool_mean, float* __restrict__ scores, long long ld_s) {
  const int b = blockIdx.y;
  const int lane = threadIdx.x & (kWave - 1);
  const int i = blockIdx.x * 4 + threadIdx.x / kWave;
  if (i >= S) return;  // wave-uniform
  const int G = n_q / n_kv;
  float best = -INFINITY, sum = 0.f;
  for (int h = 0; h < n_q; ++h) {
    const float* qh = q + ((long long)b * n_q + h) * hd;
    const float* kh = keys + ((long long)i * n_kv + h / G) * hd;
    float p = 0.f;
    for (int e = lane; e < hd; e += kWave) p = fmaf(qh[e], kh[e], p);
    p = wave_sum(p);
    best = fmaxf(best, p);
    sum += p;
  }
  if (lane == 0) {
    const bool ok = valid == nullptr || valid[i] != 0;
    scores[(long long)b * ld_s + i] = ok ? (pool_mean ? sum / (float)n_q : best) : -INFINITY;
  }
}

// The same scores, bit for bit, for hd = HD in {64, 128, 256} and at most 8 query heads per kv head: a
// wave takes NS = 16 / GP slots at a time (GP: the heads padded to a power of two), so that the 16
// (head, slot) dots of a kv head share one reduction and a query value is read from LDS once per
// NS slots.  Bound by the keys' read: 8192 slots x 4 x 256 fp32 (33.5 MB), 16 heads: 22.6 us with a
// wave per slot and a full reduction per head, 8.8 us here.
//
// Lane l owns columns l, l + 64, ... as above.  The reduction adds the same pairs as wave_sum (lanes
// at distance 1, 2, 4, 8, then the 16-lane rows), but halves the values at each of the first four
// steps: lane l ends with the total of value v(l % 16), v the 4 bits of l % 16 reversed; value g * NS
// + s is head g of slot s, so the heads of a slot are the lanes that differ in their low bits.
template <int MASK>
__device__ __forceinline__ float lane_xor(float x) {
  if constexpr (MASK == 1) return dpp_f<0xB1>(x);                    // quad_perm [1,0,3,2]
  else if constexpr (MASK == 2) return dpp_f<0x4E>(x);               // quad_perm [2,3,0,1]
  else if constexpr (MASK == 4) return dpp_f<0x141>(dpp_f<0x1B>(x));  // i ^ 3, then i ^ 7
  else return dpp_f<0x140>(dpp_f<0x141>(x));                          // i ^ 7, then i ^ 15
}

template <int MASK, int CNT>
__device__ __forceinline__ void scatter16(float (&v)[16], int lane) {
  constexpr int H = CNT / 2;
  const bool hi = (lane & MASK) != 0;
#pragma unroll
  for (int i = 0; i < H; ++i) {
    const float keep = hi ? v[i + H] : v[i];
    v[i] = keep + lane_xor<MASK>(hi ? v[i] : v[i + H]);
  }
  if constexpr (MASK < 8) scatter16<2 * MASK, H>(v, lane);
}

template <int HD, int GP>
__global__ __launch_bounds__(256) void select_scores_tile_kernel(
    const float* __restrict__ q, int n_q, int n_kv, const float* __restrict__ keys, int S,
    const unsigned char* __restrict__ valid, int pool_mean, float* __restrict__ scores, long long ld_s) {
  constexpr int NS = 16 / GP, E = HD / kWave;
  extern __shared__ float qs[];   // [n_q][HD]
  const int b = blockIdx.y, G = n_q / n_kv;
  const int lane = threadIdx.x & (kWave - 1), wv = threadIdx.x / kWave;
  for (int i = threadIdx.x; i < n_q * HD; i += 256) qs[i] = q[(long long)b * n_q * HD + i];
  const int i0 = (blockIdx.x * 4 + wv) * NS;
  const float* krow[NS];   // slots past the end: the last one (not written)
#pragma unroll
  for (int s = 0; s < NS; ++s) krow[s] = keys + (long long)min(i0 + s, S - 1) * n_kv * HD + lane;
  float k[2][NS][E];
  auto load = [&](int set, int j) {
    const int o = min(j, n_kv - 1) * HD;
#pragma unroll
    for (int s = 0; s < NS; ++s)
#pragma unroll
      for (int e = 0; e < E; ++e) k[set][s][e] = __builtin_nontemporal_load(krow[s] + o + e * kWave);
  };
  load(0, 0);
  load(1, 1);
  __syncthreads();
  if (i0 >= S) return;   // wave-uniform
  const int v = ((lane & 1) << 3) | ((lane & 2) << 1) | ((lane & 4) >> 1) | ((lane & 8) >> 3);
  const int g = v / NS, s_own = v % NS;
  float best = -INFINITY, sum = 0.f;
  auto head = [&](int set, int j) {
    float p[16];
#pragma unroll
    for (int gg = 0; gg < GP; ++gg) {
      const float* qh = qs + (j * G + min(gg, G - 1)) * HD + lane;
      float qv[E];
#pragma unroll
      for (int e = 0; e < E; ++e) qv[e] = qh[e * kWave];
#pragma unroll
      for (int s = 0; s < NS; ++s) {
        float a = 0.f;
#pragma unroll
        for (int e = 0; e < E; ++e) a = fmaf(qv[e], k[set][s][e], a);
        p[gg * NS + s] = a;
      }
    }
    load(set, j + 2);
    scatter16<1, 16>(p, lane);
    float t = p[0];
    {
      const unsigned u = __float_as_uint(t);
      const auto r = __builtin_amdgcn_permlane16_swap(u, u, false, false);
      t = __uint_as_float(r[0]) + __uint_as_float(r[1]);
    }
    {
      const unsigned u = __float_as_uint(t);
      const auto r = __builtin_amdgcn_permlane32_swap(u, u, false, false);
      t = __uint_as_float(r[0]) + __uint_as_float(r[1]);
    }
    if (g < G) best = fmaxf(best, t);
    if (pool_mean)
      for (int gg = 0; gg < G; ++gg) {   // in head order, as one wave per slot adds them
        const int w = gg * NS + s_own;
        sum += __shfl(t, ((w & 1) << 3) | ((w & 2) << 1) | ((w & 4) >> 1) | ((w & 8) >> 3));
      }
  };
  for (int j = 0; j < n_kv; j += 2) {
    head(0, j);
    if (j + 1 < n_kv) head(1, j + 1);
  }
  if constexpr (GP >= 2) best = fmaxf(best, lane_xor<1>(best));
  if constexpr (GP >= 4) best = fmaxf(best, lane_xor<2>(best));
  if constexpr (GP >= 8) best = fmaxf(best, lane_xor<4>(best));
  const int i = i0 + s_own;
  if (lane < 16 && g == 0 && i < S) {
    const bool ok = valid == nullptr || valid[i] != 0;
    scores[(long long)b * ld_s + i] = ok ? (pool_mean ? sum / (float)n_q : best) : -INFINITY;
  }
}

// ------------------------------------------------------------------------------------------
// Top-k per row by radix select on an order-preserving integer key of the fp32 score:
// key(x) = bits(x) | 0x80000000 for x >= 0, ~bits(x) for x < 0 (larger x -> larger key).
// Four 8-bit passes (most significant byte first) narrow the k-th largest key T; the winners
// are every key > T plus the first (lowest-index) keys == T up to k, gathered in index order by
// a workgroup scan; a bitonic sort of the winners by (key desc, index asc) gives the order.
constexpr int kTopkThreads = 1024;
constexpr int kTopkMax = 1024;

__device__ __forceinline__ unsigned int order_key(float x) {
  const unsigned int u = __float_as_uint(x);
  return (u & 0x80000000u) ? ~u : (u | 0x80000000u);
}

// Inclusive scan of one int per thread over the workgroup (16 waves): wave scan with shuffles,
// wave totals through LDS.  Returns the inclusive prefix; *total = the workgroup sum.
__device__ __forceinline__ int block_scan(int v, int* wsum, int* total) {
  const int lane = threadIdx.x & (kWave - 1), wv = threadIdx.x / kWave;
#pragma unroll
  for (int o = 1; o < kWave; o <<= 1) {
    const int t = __shfl_up(v, o, kWave);
    if (lane >= o) v += t;
  }
  if (lane == kWave - 1) wsum[wv] = v;
  __syncthreads();
  int off = 0, tot = 0;
  for (int w = 0; w < kTopkThreads / kWave; ++w) {
    off += w < wv ? wsum[w] : 0;
    tot += wsum[w];
  }
  __syncthreads();
  *total = tot;
  return v + off;
}

__global__ __launch_bounds__(kTopkThreads) void topk_rows_kernel(
    const float* __restrict__ scores, long long ld_s, int S, int k, int* __restrict__ idx,
    float* __restrict__ vals, long long ld_o) {
  __shared__ int hist[256];
  __shared__ int wsum[kTopkThreads / kWave];
  __shared__ unsigned int sel_key[kTopkMax];
  __shared__ int sel_idx[kTopkMax];
  __shared__ unsigned int prefix_s, mask_s;
  __shared__ int need_s;
  const int b = blockIdx.x;
  const float* row = scores + (long long)b * ld_s;
  const int tid = threadIdx.x;

  // Radix select of the k-th largest key.
  unsigned int prefix = 0, mask = 0;
  int need = k;  // how many of the keys matching `prefix` (under `mask`) still belong to the top k
  for (int shift = 24; shift >= 0; shift -= 8) {
    if (tid < 256) hist[tid] = 0;
    __syncthreads();
    for (int i = tid; i < S; i += kTopkThreads) {
      const unsigned int key = order_key(row[i]);
      if ((key & mask) == prefix) atomicAdd(&hist[(key >> shift) & 255], 1);
    }
    __syncthreads();
    if (tid == 0) {
      int acc = 0, bin = 255;
      for (; bin > 0; --bin) {
        if (acc + hist[bin] >= need) break;
        acc += hist[bin];
      }
      need_s = need - acc;
      prefix_s = prefix | ((unsigned int)bin << shift);
      mask_s = mask | (255u << shift);
    }
    __syncthreads();
    prefix = prefix_s;
    mask = mask_s;
    need = need_s;
  }
  const unsigned int T = prefix;  // the k-th largest key; `need` of the keys == T are taken

  // Winners in index order: keys > T, and keys == T while fewer than `need` were taken.
  int base_gt = 0, base_eq = 0;
  for (int i0 = 0; i0 < S; i0 += kTopkThreads) {
    const int i = i0 + tid;
    unsigned int key = 0;
    int gt = 0, eq = 0;
    if (i < S) {
      key = order_key(row[i]);
      gt = key > T;
      eq = key == T;
    }
    int tot_gt, tot_eq;
    const int pgt = block_scan(gt, wsum, &tot_gt) - gt;
    const int peq = block_scan(eq, wsum, &tot_eq) - eq;
    const int n_gt_total_before = base_gt + pgt;
    const int n_eq_before = base_eq + peq;
    // Output slot: all keys > T come first in index order, then the first `need` keys == T.
    if (gt) {
      const int pos = n_gt_total_before;
      sel_key[pos] = key;
      sel_idx[pos] = i;
    } else if (eq && n_eq_before < need) {
      const int pos = (k - need) + n_eq_before;
      sel_key[pos] = key;
      sel_idx[pos] = i;
    }
    base_gt += tot_gt;
    base_eq += tot_eq;
  }
  __syncthreads();

  // Bitonic sort of the k winners (padded to a power of two) by (key desc, index asc).
  int P = 1;
  while (P < k) P <<= 1;
  for (int i = k + tid; i < P; i += kTopkThreads) {
    sel_key[i] = 0;
    sel_idx[i] = 0x7fffffff;
  }
  __syncthreads();
  for (int size = 2; size <= P; size <<= 1) {
    for (int stride = size >> 1; stride > 0; stride >>= 1) {
      for (int i = tid; i < P; i += kTopkThreads) {
        const int j = i ^ stride;
        if (j > i) {
          const bool desc = (i & size) == 0;  // first half of each block sorts "best first"
          const unsigned int ka = sel_key[i], kb = sel_key[j];
          const int ia = sel_idx[i], ib = sel_idx[j];
          const bool a_first = ka > kb || (ka == kb && ia < ib);
          if (desc != a_first) {
            sel_key[i] = kb; sel_key[j] = ka;
            sel_idx[i] = ib; sel_idx[j] = ia;
          }
        }
      }
      __syncthreads();
    }
  }
  for (int j = tid; j < k; j += kTopkThreads) {
    const int i = sel_idx[j];
    idx[(long long)b * ld_o + j] = i;
    if (vals) vals[(long long)b * ld_o + j] = row[i];
  }
}

// The same result for rows of at most 1024 KPT <= 32768 scores, whose keys stay in registers (element
// c * 1024 + tid).  A threshold T is built two bits at a time from the top, the largest with at least k
// keys >= T, until exactly k are (ties at the edge: down to the k-th largest key); a step counts with
// ballots, 16 wave counts through LDS and one barrier.  The winners need no order of their own: up to 256 are ranked by counting the ones before
// them ((key, index) pairs are distinct), more go through the bitonic sort.  Bound by the chain of
// steps: 8192 scores, k = 64: 53 us with four histogram passes over memory (one thread walking each
// histogram, atomics on the few exponent bins) and 8 block scans, 18 us with one bit a step and no
// early end, 13 us here.
template <int KPT>
__global__ __launch_bounds__(kTopkThreads) void topk_rows_regs_kernel(
    const float* __restrict__ scores, long long ld_s, int S, int k, int* __restrict__ idx,
    float* __restrict__ vals, long long ld_o) {
  constexpr int kWaves = kTopkThreads / kWave, kRankMax = 256;
  __shared__ unsigned long long wcnt[2][kWaves];
  __shared__ int wsum[kWaves];
  __shared__ unsigned long long win[kTopkMax];   // key << 32 | ~index: larger = earlier
  __shared__ int rank[kRankMax];
  __shared__ int n_win;
  const int b = blockIdx.x, tid = threadIdx.x, lane = tid & (kWave - 1), wv = tid / kWave;
  const float* row = scores + (long long)b * ld_s;
  unsigned key[KPT];   // elements past S: 0, below every threshold counted
#pragma unroll
  for (int c = 0; c < KPT; ++c) {
    const int i = c * kTopkThreads + tid;
    const float x = row[min(i, S - 1)];
    key[c] = i < S ? order_key(x) : 0u;
  }
  if (tid == 0) n_win = 0;
  if (tid < kRankMax) rank[tid] = 0;
  // The keys >= T + j * unit of the row for j = 1, 2, 3, 21 bits each; every thread gets the counts.
  int parity = 0;
  auto count_ge = [&](unsigned T, unsigned unit) {
    unsigned long long n = 0;
#pragma unroll
    for (int c = 0; c < KPT; ++c) {
#pragma unroll
      for (int j = 1; j <= 3; ++j)
        n += (unsigned long long)__popcll(__ballot(key[c] >= T + j * unit)) << (21 * (j - 1));
      if (c % 4 == 3) __builtin_amdgcn_sched_barrier(0);   // (else every ballot's mask is kept at once)
    }
    if (lane == 0) wcnt[parity][wv] = n;
    __syncthreads();
    unsigned long long tot = 0;
#pragma unroll
    for (int w = 0; w < kWaves; ++w) tot += wcnt[parity][w];
    parity ^= 1;
    return tot;
  };
  unsigned T = 0;
  int n_ge = S;   // the keys >= T (a key of 0, the NaN with every bit set, among them)
  for (int bit = 30; bit >= 0 && n_ge != k; bit -= 2) {
    const unsigned long long n = count_ge(T, 1u << bit);
    const int n1 = (int)(n & 0x1fffff), n2 = (int)((n >> 21) & 0x1fffff), n3 = (int)(n >> 42);
    const int j = n3 >= k ? 3 : n2 >= k ? 2 : n1 >= k ? 1 : 0;
    T += (unsigned)j << bit;
    if (j) n_ge = j == 3 ? n3 : j == 2 ? n2 : n1;
  }
  // Winners: the k keys >= T when there are just k; else T is the k-th largest key itself, and they are
  // every key > T and the first elements (in index order) with key == T.
  const bool ties = n_ge != k;   // workgroup-uniform
  int need = 0;
  if (ties) need = k - (T == 0xffffffffu ? 0 : (int)(count_ge(T, 1) & 0x1fffff));
  int eq_before = 0;
#pragma unroll
  for (int c = 0; c < KPT; ++c) {
    const int i = c * kTopkThreads + tid;
    const bool gt = i < S && key[c] > T, eq = i < S && key[c] == T;
    bool take = gt || eq;   // (the index test leaves out the elements past S, whose key is 0)
    if (ties) {
      int tot;
      const int before = block_scan(eq ? 1 : 0, wsum, &tot) - (eq ? 1 : 0);
      take = gt || (eq && eq_before + before < need);
      eq_before += tot;
    }
    const unsigned long long m = __ballot(take);
    if (m) {   // wave-uniform
      int at = 0;
      if (lane == 0) at = atomicAdd(&n_win, __popcll(m));
      at = __builtin_amdgcn_readfirstlane(at);
      if (take) win[at + __popcll(m & ((1ull << lane) - 1))] = ((unsigned long long)key[c] << 32) | (unsigned)~i;
    }
  }
  __syncthreads();
  if (k <= kRankMax) {   // four threads per winner count the winners before it
    const int i = tid % kRankMax, part = tid / kRankMax;
    constexpr int kParts = kTopkThreads / kRankMax;
    if (i < k) {
      const unsigned long long mine = win[i];
      int r = 0;
      for (int j = part; j < k; j += kParts) r += win[j] > mine ? 1 : 0;
      atomicAdd(&rank[i], r);
    }
    __syncthreads();
    if (tid < k) {
      const int e = (int)~(unsigned)win[tid];
      idx[(long long)b * ld_o + rank[tid]] = e;
      if (vals) vals[(long long)b * ld_o + rank[tid]] = row[e];
    }
    return;
  }
  int P = 1;
  while (P < k) P <<= 1;
  for (int i = k + tid; i < P; i += kTopkThreads) win[i] = 0;   // after every winner
  __syncthreads();
  for (int size = 2; size <= P; size <<= 1)
    for (int stride = size >> 1; stride > 0; stride >>= 1) {
      if (tid < P) {
        const int j = tid ^ stride;
        if (j > tid) {
          const bool desc = (tid & size) == 0;
          const unsigned long long x = win[tid], y = win[j];
          if (desc != (x > y)) {
            win[tid] = y;
            win[j] = x;
          }
        }
      }
      __syncthreads();
    }
  if (tid < k) {
    const int e = (int)~(unsigned)win[tid];
    idx[(long long)b * ld_o + tid] = e;
    if (vals) vals[(long long)b * ld_o + tid] = row[e];
  }
}

// ------------------------------------------------------------------------------------------
// Gather: out[g, j] = slot row idx[g, j] of the flat library (flat index f -> chunk f / n_flat,
// slot f % n_flat; chunk c lives on page chunk_page[c]) for j < k, zero rows for k <= j < kpad.
// One workgroup per (set g, 4 output rows); 16-byte copies.  With meta the first workgroup of a set also
// writes what makes the sets libraries of one chunk: S[g] = 0 (routing over one chunk is w = 1) and
// meta = page table [G] (g) | valid slots [G] (k) | chunk offsets [G + 1] (g).
__global__ __launch_bounds__(256) void gather_pages_kernel(
    const _Float16* __restrict__ pages, int slots_per_page, long long page_stride, int d,
    const int* __restrict__ chunk_page, int n_chunks, int n_flat, const int* __restrict__ idx,
    long long ld_idx, int k, int kpad, _Float16* __restrict__ out, float* __restrict__ S_out,
    int* __restrict__ meta) {
  const int g = blockIdx.y;
  if (meta && blockIdx.x == 0) {
    for (int e = threadIdx.x; e < d; e += 256) S_out[(long long)g * d + e] = 0.f;
    if (threadIdx.x == 0) {
      const int G = gridDim.y;
      meta[g] = g;
      meta[G + g] = k;
      meta[2 * G + g] = g;
      if (g == G - 1) meta[3 * G] = G;
    }
  }
  const int j = blockIdx.x * 4 + threadIdx.x / kWave;
  if (j >= kpad) return;
  const int lane = threadIdx.x & (kWave - 1);
  _Float16* dst = out + ((long long)g * kpad + j) * d;
  const _Float16* src = nullptr;
  if (j < k) {
    const int f = idx[(long long)g * ld_idx + j];
    const int c = f / n_flat, n = f % n_flat;
    if (f >= 0 && c < n_chunks && n < slots_per_page)
      src = pages + (long long)chunk_page[c] * page_stride + (long long)n * d;
  }
  for (int e = lane * 8; e < d; e += kWave * 8) {
    u32x4 v = {0u, 0u, 0u, 0u};
    if (src) v = *reinterpret_cast<const u32x4*>(src + e);
    *reinterpret_cast<u32x4*>(dst + e) = v;
  }
}

}  // namespace
}  // namespace xenc

using namespace xenc;

extern "C" int xenc_select_scores(const float* q, int B, int n_q, int n_kv, int hd,
                                  const float* keys, int S, const unsigned char* valid, int pool_mean,
                                  float* scores, long long ld_s, void* stream) {
  if (B < 0 || n_q <= 0 || n_kv <= 0 || n_q % n_kv != 0 || hd <= 0 || S < 0 || ld_s < S ||
      B > 65535)
    return XENC_EINVAL;
  if (B == 0 || S == 0) return XENC_OK;
  if (!q || !keys || !scores) return XENC_ENULL;
  hipStream_t st = reinterpret_cast<hipStream_t>(stream);
  const int G = n_q / n_kv;
  const size_t lds = (size_t)n_q * hd * sizeof(float);
  if ((hd == 64 || hd == 128 || hd == 256) && G <= 8 && lds <= 64 * 1024) {
    const int GP = G <= 1 ? 1 : G <= 2 ? 2 : G <= 4 ? 4 : 8, per = 4 * 16 / GP;   // slots per workgroup
    auto launch = [&](auto kernel) {
      hipLaunchKernelGGL(kernel, dim3((S + per - 1) / per, B), dim3(256), lds, st, q, n_q, n_kv, keys, S, valid,
                         pool_mean, scores, ld_s);
    };
#define XENC_SEL(HD)                                        \
  switch (GP) {                                             \
    case 1: launch(select_scores_tile_kernel<HD, 1>); break; \
    case 2: launch(select_scores_tile_kernel<HD, 2>); break; \
    case 4: launch(select_scores_tile_kernel<HD, 4>); break; \
    default: launch(select_scores_tile_kernel<HD, 8>); break; \
  }
    if (hd == 64) XENC_SEL(64) else if (hd == 128) XENC_SEL(128) else XENC_SEL(256)
#undef XENC_SEL
    return check_launch();
  }
  hipLaunchKernelGGL(select_scores_kernel, dim3((S + 3) / 4, B), dim3(256), 0, st, q, n_q, n_kv, hd, keys, S, valid,
                     pool_mean, scores, ld_s);
  return check_launch();
}

extern "C" int xenc_topk_rows(const float* scores, long long ld_s, int B, int S, int k, int* idx,
                              float* vals, long long ld_o, void* stream) {
  if (B < 0 || S < 0 || k < 0 || k > S || k > kTopkMax || ld_s < S || ld_o < k) return XENC_EINVAL;
  if (B == 0 || k == 0) return XENC_OK;
  if (!scores || !idx) return XENC_ENULL;
  auto launch = [&](auto kernel) {
    hipLaunchKernelGGL(kernel, dim3(B), dim3(kTopkThreads), 0, reinterpret_cast<hipStream_t>(stream), scores, ld_s, S, k,
                       idx, vals, ld_o);
  };
  if (S <= 8 * kTopkThreads) launch(topk_rows_regs_kernel<8>);
  else if (S <= 32 * kTopkThreads) launch(topk_rows_regs_kernel<32>);
  else launch(topk_rows_kernel);   // more keys than the registers hold
  return check_launch();
}

extern "C" int xenc_gather_library(const void* pages, int slots_per_page, long long page_stride, int d,
                                   const int* chunk_page, int n_chunks, int n_flat, const int* idx,
                                   long long ld_idx, int G, int k, int kpad, void* out, float* S_out, int* meta,
                                   void* stream) {
  if (slots_per_page <= 0 || d <= 0 || d % 8 != 0 || page_stride < (long long)slots_per_page * d ||
      page_stride % 8 != 0 || n_chunks <= 0 || n_flat <= 0 || G < 0 || k < 0 || kpad < k ||
      ld_idx < k || G > 65535)
    return XENC_EINVAL;
  if (G == 0 || kpad == 0) return XENC_OK;
  if (!pages || !chunk_page || !out || (k > 0 && !idx) || !S_out != !meta) return XENC_ENULL;
  if (!aligned16(pages) || !aligned16(out)) return XENC_EALIGN;
  hipLaunchKernelGGL(gather_pages_kernel, dim3((kpad + 3) / 4, G), dim3(256), 0,
                     reinterpret_cast<hipStream_t>(stream), static_cast<const _Float16*>(pages),
                     slots_per_page, page_stride, d, chunk_page, n_chunks, n_flat, idx, ld_idx, k,
                     kpad, static_cast<_Float16*>(out), S_out, meta);
  return check_launch();
}

extern "C" int xenc_gather_pages(const void* pages, int slots_per_page, long long page_stride, int d,
                                 const int* chunk_page, int n_chunks, int n_flat, const int* idx,
                                 long long ld_idx, int G, int k, int kpad, void* out, void* stream) {
  return xenc_gather_library(pages, slots_per_page, page_stride, d, chunk_page, n_chunks, n_flat, idx, ld_idx, G, k,
                             kpad, out, nullptr, nullptr, stream);
}
