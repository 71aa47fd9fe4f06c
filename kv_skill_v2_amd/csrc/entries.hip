// The read of many query rows by ENTRIES: the (row, chunk) pairs that routing kept, grouped by
// chunk, instead of every row against every chunk of its library (csrc/prefill.hip).  Same math
// (forward, linear read, and their dQ backward; xenc/injector.py:236-265), same fp16 operands and
// fp32 accumulation, four steps:
//
//   entries_list      per chunk the entries e = row * kk + j (rank j) that routed to it, in row order
//   entries_scores    (chunk, 32 or 64 of its entries): S^T = K_c X^T over the whole chunk, the
//                     masked softmax (or linear read, or the backward's dS and gamma) per entry ->
//                     p [entry][slot] fp16
//   entries_readout   (chunk, the same entries, 256 dims): part[e] = w[row, c] * p[e] . K_c in fp32
//   entries_merge     out[row] = sum_j part[row * kk + j] in rank order (backward: plus the routing
//                     term sum_j dl_j S_{c_j})
//
// A pair with route weight exactly 0 contributes nothing to the read or to its gradient, so with
// top_k of C chunks kept this is top_k / C of the dense work.  Without lists the entries are all
// pairs (e = row * kk + c): the same kernels then serve launches with too few 128-row x chunk tiles
// to fill the GPU.  Tile i of chunk gc is workgroup (i, gc) of a grid sized for the most entries a
// chunk can have; the ones past the chunk's count exit (they come last in dispatch order).
#include <algorithm>
#include <climits>
#include <type_traits>

#include "xenc_common.h"

namespace xenc {
namespace {

typedef _Float16 half8_t __attribute__((ext_vector_type(8)));
typedef _Float16 half4_t __attribute__((ext_vector_type(4)));
typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef float f32x4 __attribute__((ext_vector_type(4)));

constexpr int BK = 64;   // d (or slot) columns per k step: four MFMA k16 steps
constexpr int kEntThreads = 512, kEntWaves = kEntThreads / kWave;

__device__ __forceinline__ f32x16 mfma32(const half8_t& a, const half8_t& b, const f32x16& c) {
  return __builtin_amdgcn_mfma_f32_32x32x16_f16(a, b, c, 0, 0, 0);
}

// LDS tiles of rows of 64 halves, chunk c of 16 bytes of row r at position c ^ sw(r): the 16-byte
// fragment reads of consecutive rows fall on disjoint banks.
__device__ __forceinline__ int sw(int r) { return (r ^ (r >> 3)) & 7; }

__device__ __forceinline__ int library_of(const int* __restrict__ ptr, int G, int b) {
  int lo = 0, hi = G - 1;
  while (lo < hi) {
    const int mid = (lo + hi + 1) >> 1;
    if (ptr[mid] <= b) lo = mid; else hi = mid - 1;
  }
  return lo;
}

struct EntryArgs {
  int G, Ctot, Cp, kk, ld_list, d, N;   // Cp: Ctot rounded up to the XCDs (a chunk's tiles share one)
  const int* row_ptr;
  const int* chunk_ptr;
  const int* list;      // [Ctot][ld_list] entries by chunk; NULL: every row of the chunk's library
  const int* count;     // [Ctot]
  const _Float16* pages;
  long long page_stride;
  const int* chunk_page;
  const int* chunk_nvalid;
  const float* w;
  long long ldw;
};

// The entries of tile `tile` of chunk gc: its library, local chunk index and entry count.
struct Tile {
  int c, rbeg, n;
  const int* list;
  __device__ __forceinline__ Tile(const EntryArgs& A, int gc) {
    const int g = library_of(A.chunk_ptr, A.G, gc);
    c = gc - A.chunk_ptr[g];
    rbeg = A.row_ptr[g];
    list = A.list ? A.list + (long long)gc * A.ld_list : nullptr;
    n = A.list ? A.count[gc] : A.row_ptr[g + 1] - rbeg;
  }
  __device__ __forceinline__ int entry(const EntryArgs& A, int i) const {
    return list ? list[i] : (rbeg + i) * A.kk + c;
  }
};

// ------------------------------------------------------------------------------------------
// One workgroup per chunk: a pass over its library's rows in order, kListThreads rows at a time;
// a row's rank j of this chunk (at most one) becomes entry row * kk + j, placed by a scan.
constexpr int kListThreads = 1024, kListWaves = kListThreads / kWave;
__global__ __launch_bounds__(kListThreads) void entries_list_kernel(const int* __restrict__ idx, int kk,
                                                                    const int* __restrict__ row_ptr,
                                                                    const int* __restrict__ chunk_ptr, int G,
                                                                    int ld_list, int* __restrict__ list,
                                                                    int* __restrict__ count) {
  __shared__ int wsum[2][kListWaves];
  const int gc = blockIdx.x;
  const int g = library_of(chunk_ptr, G, gc);
  const int c = gc - chunk_ptr[g];
  const int rbeg = row_ptr[g], rend = row_ptr[g + 1];
  const int lane = threadIdx.x & (kWave - 1), wv = threadIdx.x / kWave;
  int base = 0;
  for (int r0 = rbeg, it = 0; r0 < rend; r0 += kListThreads, ++it) {
    const int row = r0 + threadIdx.x;
    int e = -1;
    if (row < rend)
      for (int j = 0; j < kk; ++j)
        if (idx[(long long)row * kk + j] == c) e = row * kk + j;
    const unsigned long long hit = __ballot(e >= 0);
    if (lane == 0) wsum[it & 1][wv] = __popcll(hit);
    __syncthreads();
    int off = base, tot = 0;
#pragma unroll
    for (int v = 0; v < kListWaves; ++v) {
      off += v < wv ? wsum[it & 1][v] : 0;
      tot += wsum[it & 1][v];
    }
    if (e >= 0) list[(long long)gc * ld_list + off + __popcll(hit & ((1ull << lane) - 1))] = e;
    base += tot;
  }
  if (threadIdx.x == 0) count[gc] = base;
}

// ------------------------------------------------------------------------------------------
// Scores: 8 waves over one chunk x 32 NT entries.  SG wave groups of 64 slots (two MFMA rows of
// 32); with a page of N <= 256 slots the remaining KS = 8 / SG waves per group split the columns
// (k step it * KS + ks), summed through LDS at the end.  A wave's slot fragments come from the
// layout-A page copy, FD iterations ahead; the entries' query rows (gathered) are staged straight
// into LDS, SD ahead, one barrier an iteration.  MODE as in scores_kernel (csrc/prefill.hip).
// Bound by the chunk's page through one CU's L2 port (2 MB a workgroup at 512 x 2048 in 31 us, about
// 65 GB/s, with loads two or four iterations ahead alike).  So launches of few tiles split the slots
// too: workgroup (tile, block) takes 64 SG slots from 64 SG block on.  The softmax is then left to the
// readout (MODE 4): p = 2^(s - m) with m the block's max rounded up to a whole number, and stats
// [entry][block] = (m, sum of the block's p), so the blocks join by exact powers of two.
// 333 rows, top-4 of 16 chunks of 512 x 2048: 48 us (128-row tiles over all pairs), 31 us whole
// chunks, 16 us in 4 blocks.
template <int MODE, int SG, int NT>
__global__ __launch_bounds__(kEntThreads) void entries_scores_kernel(
    const EntryArgs A, const _Float16* __restrict__ X, float temp, _Float16* __restrict__ P,
    _Float16* __restrict__ dS, float* __restrict__ gamma, int blocks, float2* __restrict__ stats) {
  constexpr int KS = kEntWaves / SG, RT = 32 * NT;
  constexpr int FD = NT == 1 ? 4 : 2;          // iterations the slot fragments are loaded ahead
  constexpr int SD = KS <= 2 && NT == 1 ? 4 : 2, NST = SD + 1;   // iterations the rows are staged ahead; stages
  constexpr int kSub = RT * BK;                                // halves of one staged k step
  constexpr int kStageB = NST * KS * kSub * 2;                 // bytes
  constexpr int kRedB = (kEntWaves - SG) * 2 * NT * 16 * kWave * 4;
  __shared__ alignas(16) char lds[kStageB > kRedB ? kStageB : kRedB];
  __shared__ float red[SG][RT];
  __shared__ int ent[RT];
  const int gc = blockIdx.x % A.Cp, tb = (int)(blockIdx.x / A.Cp);
  const int blk = tb % blocks, i0 = tb / blocks * RT;
  if (gc >= A.Ctot) return;
  const Tile T(A, gc);
  if (i0 >= T.n) return;
  const int tid = threadIdx.x, lane = tid & 63;
  const int wv = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int sb = blk * SG * 64;   // first slot
  const int sg = wv % SG, ks = wv / SG;
  const int hl = lane >> 5, l32 = lane & 31;
  const int N = A.N, d = A.d, nk = d / BK;
  const int ne = min(T.n - i0, RT);   // live entries of the tile
  if (tid < RT) ent[tid] = T.entry(A, i0 + min(tid, ne - 1));
  __syncthreads();
  const int nv = min(A.chunk_nvalid[gc], N);
  const _Float16* Ka = A.pages + (long long)A.chunk_page[gc] * A.page_stride;

  // Staging: sub-tile j (k step it * KS + j) of RT rows x 8 chunks of 16 bytes; rows past the tile
  // re-read its last one (never stored).
  constexpr int kChunks = KS * RT * 8;                         // 16-byte chunks per iteration
  constexpr int NS = kChunks / kEntThreads > 0 ? kChunks / kEntThreads : 1;
  const bool stager = kChunks >= kEntThreads || tid < kChunks;   // wave-uniform
  const _Float16* src[NS];
  int sj[NS];
#pragma unroll
  for (int i = 0; i < NS; ++i) {
    const int id = (tid + kEntThreads * i) % kChunks, rid = id % (RT * 8), r = rid >> 3;
    sj[i] = id / (RT * 8);
    src[i] = X + (long long)(ent[r] / A.kk) * d + (((rid & 7) ^ sw(r)) << 3);
  }
  auto stage = [&](int it) {
    if (!stager) return;
#pragma unroll
    for (int i = 0; i < NS; ++i)
      stage_to_lds(lds + (it % NST) * (KS * kSub * 2) + (kEntThreads * i + 64 * wv) * 16,
                   src[i] + min(it * KS + sj[i], nk - 1) * BK);
  };
  // Slot fragments of the wave's two 32-slot groups (past the page: its last group; masked).
  const _Float16* abase[2];
#pragma unroll
  for (int mt = 0; mt < 2; ++mt)
    abase[mt] = Ka + (long long)min(sb / 32 + sg * 2 + mt, N / 32 - 1) * (d / 16) * 512 + lane * 8;
  half8_t fa[FD][4][2];   // [iteration % FD][k16 step][slot group]
  auto load_a = [&](int set, int q, int it) {
    const int k = min(it * KS + ks, nk - 1);
#pragma unroll
    for (int mt = 0; mt < 2; ++mt) fa[set][q][mt] = *reinterpret_cast<const half8_t*>(abase[mt] + (k * 4 + q) * 512);
  };
  f32x16 acc[2][NT];
#pragma unroll
  for (int mt = 0; mt < 2; ++mt)
#pragma unroll
    for (int nt = 0; nt < NT; ++nt) acc[mt][nt] = (f32x16){};

  const int iters = (nk + KS - 1) / KS;
#pragma unroll
  for (int j = 0; j < SD; ++j) stage(j);
#pragma unroll
  for (int set = 0; set < FD; ++set)
#pragma unroll
    for (int q = 0; q < 4; ++q) load_a(set, q, set);
  wait_vmem<0>();
  __syncthreads();
  auto step = [&](auto set_c, int it) {
    constexpr int set = decltype(set_c)::value;
    stage(it + SD);   // into the stage read in iteration it - 1, before the barrier that ended it
    __builtin_amdgcn_sched_barrier(0);
    const _Float16* xb = reinterpret_cast<const _Float16*>(lds + (it % NST) * (KS * kSub * 2)) + ks * kSub;
    const bool live = it * KS + ks < nk;   // wave-uniform
    half8_t fb[4][NT];
#pragma unroll
    for (int q = 0; q < 4; ++q)
#pragma unroll
      for (int nt = 0; nt < NT; ++nt) {
        const int r = nt * 32 + l32;
        fb[q][nt] = *reinterpret_cast<const half8_t*>(xb + r * BK + (((q * 2 + hl) ^ sw(r)) << 3));
      }
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      if (live) {
#pragma unroll
        for (int mt = 0; mt < 2; ++mt)
#pragma unroll
          for (int nt = 0; nt < NT; ++nt) acc[mt][nt] = mfma32(fa[set][q][mt], fb[q][nt], acc[mt][nt]);
      }
      load_a(set, q, it + FD);
      __builtin_amdgcn_sched_barrier(0);
    }
    // Stage it + 1 (issued SD - 1 iterations ago, before that iteration's 8 fragment loads) has
    // landed: at most those 8 and the later iterations' NS + 8 loads each are in flight.
    static_assert(8 + (SD - 1) * (NS + 8) < 64, "vmcnt range");
    wait_vmem<8 + (SD - 1) * (NS + 8)>();
    __syncthreads();
  };
  for (int it = 0; it < iters; it += FD) {
    step(std::integral_constant<int, 0>{}, it);
    if (it + 1 < iters) step(std::integral_constant<int, 1>{}, it + 1);
    if constexpr (FD == 4) {
      if (it + 2 < iters) step(std::integral_constant<int, 2>{}, it + 2);
      if (it + 3 < iters) step(std::integral_constant<int, 3>{}, it + 3);
    }
  }
  wait_vmem<0>();

  // The column parts of a slot group, summed in ks order by its first wave.
  if constexpr (KS > 1) {
    __syncthreads();
    f32x4* part = reinterpret_cast<f32x4*>(lds);
    if (ks > 0) {
#pragma unroll
      for (int mt = 0; mt < 2; ++mt)
#pragma unroll
        for (int nt = 0; nt < NT; ++nt)
#pragma unroll
          for (int q = 0; q < 4; ++q)
            part[((((ks - 1) * SG + sg) * 2 * NT + mt * NT + nt) * 4 + q) * kWave + lane] =
                f32x4{acc[mt][nt][4 * q], acc[mt][nt][4 * q + 1], acc[mt][nt][4 * q + 2], acc[mt][nt][4 * q + 3]};
    }
    __syncthreads();
    if (ks == 0) {
#pragma unroll 1
      for (int k = 1; k < KS; ++k)
#pragma unroll
        for (int mt = 0; mt < 2; ++mt)
#pragma unroll
          for (int nt = 0; nt < NT; ++nt)
#pragma unroll
            for (int q = 0; q < 4; ++q) {
              const f32x4 v = part[((((k - 1) * SG + sg) * 2 * NT + mt * NT + nt) * 4 + q) * kWave + lane];
#pragma unroll
              for (int e = 0; e < 4; ++e) acc[mt][nt][4 * q + e] += v[e];
            }
    }
  }
  const bool own = ks == 0;   // wave-uniform: the waves that hold the slots' scores
  // acc[mt][nt][r] = S^T[slot][entry]: slot = sb + 64 sg + 32 mt + 8 (r / 4) + 4 hl + r % 4, entry 32 nt + l32.
  auto slot_of = [&](int mt, int r) { return sb + sg * 64 + mt * 32 + (r >> 2) * 8 + hl * 4 + (r & 3); };
  auto each_quad = [&](int nt, auto f) {   // f(first slot, mt, quad) over the wave's quads of 4 slots
#pragma unroll
    for (int mt = 0; mt < 2; ++mt)
#pragma unroll
      for (int q = 0; q < 4; ++q)
        if (slot_of(mt, 4 * q) < N) f(slot_of(mt, 4 * q), mt, q);
  };

  if constexpr (MODE == 2) {
    if (!own) return;
    const float inv = 1.f / sqrtf((float)nv);
#pragma unroll
    for (int nt = 0; nt < NT; ++nt) {
      if (nt * 32 + l32 >= ne) continue;
      _Float16* p = P + (long long)ent[nt * 32 + l32] * N;
      each_quad(nt, [&](int s0, int mt, int q) {
        half4_t h;
#pragma unroll
        for (int e = 0; e < 4; ++e) h[e] = (_Float16)(s0 + e < nv ? acc[mt][nt][4 * q + e] * inv : 0.f);
        *reinterpret_cast<half4_t*>(p + s0) = h;
      });
    }
  } else if constexpr (MODE == 0 || MODE == 4) {
    float rmax[NT], rsum[NT];
#pragma unroll
    for (int nt = 0; nt < NT; ++nt) {
      float m = -INFINITY;
#pragma unroll
      for (int mt = 0; mt < 2; ++mt)
#pragma unroll
        for (int r = 0; r < 16; ++r) {
          const float v = slot_of(mt, r) < nv ? acc[mt][nt][r] * temp : -INFINITY;
          acc[mt][nt][r] = v;
          m = fmaxf(m, v);
        }
      m = fmaxf(m, swap_partner<32>(m, hl != 0));
      if (own && hl == 0) red[sg][nt * 32 + l32] = m;
    }
    __syncthreads();
#pragma unroll
    for (int nt = 0; nt < NT; ++nt) {
      float m = red[0][nt * 32 + l32];
#pragma unroll
      for (int v = 1; v < SG; ++v) m = fmaxf(m, red[v][nt * 32 + l32]);
      // Finite for a whole chunk (>= 1 valid slot); a block may have none: m = 0 keeps its p at 0.
      rmax[nt] = MODE == 0 ? m : sb < nv ? ceilf(m) : 0.f;
    }
    __syncthreads();
#pragma unroll
    for (int nt = 0; nt < NT; ++nt) {
      float s = 0.f;
#pragma unroll
      for (int mt = 0; mt < 2; ++mt)
#pragma unroll
        for (int r = 0; r < 16; ++r) {
          const float e = __builtin_amdgcn_exp2f(acc[mt][nt][r] - rmax[nt]);
          acc[mt][nt][r] = e;
          s += e;
        }
      s += swap_partner<32>(s, hl != 0);
      if (own && hl == 0) red[sg][nt * 32 + l32] = s;
    }
    __syncthreads();
    if (!own) return;
#pragma unroll
    for (int nt = 0; nt < NT; ++nt) {
      float s = 0.f;
#pragma unroll
      for (int v = 0; v < SG; ++v) s += red[v][nt * 32 + l32];
      rsum[nt] = MODE == 0 ? 1.f / s : 1.f;
      if (MODE == 4 && sg == 0 && hl == 0 && nt * 32 + l32 < ne)
        stats[(long long)ent[nt * 32 + l32] * blocks + blk] = make_float2(sb < nv ? rmax[nt] : -INFINITY, s);
    }
#pragma unroll
    for (int nt = 0; nt < NT; ++nt) {
      if (nt * 32 + l32 >= ne) continue;
      _Float16* p = P + (long long)ent[nt * 32 + l32] * N;
      each_quad(nt, [&](int s0, int mt, int q) {
        half4_t h;
#pragma unroll
        for (int e = 0; e < 4; ++e) h[e] = (_Float16)(acc[mt][nt][4 * q + e] * rsum[nt]);
        *reinterpret_cast<half4_t*>(p + s0) = h;
      });
    }
  } else {
    // ---- backward: gamma = sum_n p U, dS = temp * w * p * (U - gamma) (linear: w * U / sqrt(n))
#pragma unroll
    for (int nt = 0; nt < NT; ++nt) {
      const _Float16* p = P + (long long)ent[nt * 32 + l32] * N;   // (past the tile: its last entry's)
      float s = 0.f;
      if (own)
        each_quad(nt, [&](int s0, int mt, int q) {
          const half4_t h = *reinterpret_cast<const half4_t*>(p + s0);
#pragma unroll
          for (int e = 0; e < 4; ++e) s += (float)h[e] * acc[mt][nt][4 * q + e];
        });
      s += swap_partner<32>(s, hl != 0);
      if (own && hl == 0) red[sg][nt * 32 + l32] = s;
    }
    __syncthreads();
    if (!own) return;
#pragma unroll
    for (int nt = 0; nt < NT; ++nt) {
      if (nt * 32 + l32 >= ne) continue;
      float s = 0.f;
#pragma unroll
      for (int v = 0; v < SG; ++v) s += red[v][nt * 32 + l32];
      const int e_id = ent[nt * 32 + l32];
      if (sg == 0 && hl == 0) gamma[e_id] = s;
      const float coef = (MODE == 1 ? temp : 1.f / sqrtf((float)nv)) * A.w[(long long)(e_id / A.kk) * A.ldw + T.c];
      const _Float16* p = P + (long long)e_id * N;
      _Float16* o = dS + (long long)e_id * N;
      each_quad(nt, [&](int s0, int mt, int q) {
        const half4_t pv = *reinterpret_cast<const half4_t*>(p + s0);
        half4_t h;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const float u = acc[mt][nt][4 * q + e];
          h[e] = (_Float16)(MODE == 1 ? coef * (float)pv[e] * (u - s) : (s0 + e < nv ? coef * u : 0.f));
        }
        *reinterpret_cast<half4_t*>(o + s0) = h;
      });
    }
  }
}

// ------------------------------------------------------------------------------------------
// Readout: 4 waves over (chunk, 32 NT entries, dpw tiles of 256 dims); wave w owns dims 64 w .. + 63 of a
// tile (two MFMA columns of 32).  The entries' whole p rows (N slots) are staged into LDS at once,
// one barrier; the dims' fragments come from the layout-B page copy, two k steps ahead, across the
// dim tiles.  dpw: one while that leaves at most 2048 workgroups, then more, so that a large launch
// stages a row set once for several tiles.  out row e (ONE: row e /
// kk) = scale * p[e] . K_c, scale = w[row, c] when w is given, else 1.
// SPLIT: p in `blocks` blocks of `bspan` slots as MODE 4 left them: block b of an entry enters with the
// factor 2^(m_b - M) (a power of two: an exact fp16 factor, or below its range with the weight it
// stands for), and the entry's scale carries 1 / sum_b 2^(m_b - M) l_b.
constexpr int kMaxBlocks = 8;
template <int NT, bool ONE, bool SPLIT>
__global__ __launch_bounds__(256) void entries_readout_kernel(const EntryArgs A, const _Float16* __restrict__ P,
                                                              int dim_tiles, int dpw, float* __restrict__ out,
                                                              long long ldo, int blocks, int bspan,
                                                              const float2* __restrict__ stats) {
  constexpr int RT = 32 * NT;
  extern __shared__ __align__(16) _Float16 pl[];   // [N / 64][RT][64]
  __shared__ int ent[RT];
  __shared__ float scale[RT];
  __shared__ _Float16 fac[SPLIT ? RT : 1][kMaxBlocks];
  int b = blockIdx.x;
  const int gc = b % A.Cp;
  b /= A.Cp;
  const int dgs = (dim_tiles + dpw - 1) / dpw;
  const int dt0 = b % dgs * dpw, dtn = min(dpw, dim_tiles - dt0), i0 = b / dgs * RT;
  if (gc >= A.Ctot) return;
  const Tile T(A, gc);
  if (i0 >= T.n) return;
  const int tid = threadIdx.x, lane = tid & 63;
  const int wv = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int hl = lane >> 5, l32 = lane & 31;
  const int N = A.N, d = A.d, nkb = N / BK, steps = dtn * nkb;
  const int ne = min(T.n - i0, RT);
  const _Float16* Kb = A.pages + (long long)A.chunk_page[gc] * A.page_stride + lane * 8;
  half8_t fb[2][4][2];   // [step % 2][k16 step][dim group]
  // Step v: k step v % nkb of dim tile v / nkb (32-dim groups past d: the last one; not stored).
  auto load_b = [&](int set, int q, int v) {
    const int vc = min(v, steps - 1), dt = dt0 + vc / nkb, k = vc % nkb;
#pragma unroll
    for (int nt = 0; nt < 2; ++nt) {
      const int db = min(dt * 8 + wv * 2 + nt, d / 32 - 1);
      fb[set][q][nt] = *reinterpret_cast<const half8_t*>(Kb + ((long long)db * (N / 16) + k * 4 + q) * 512);
    }
  };
#pragma unroll
  for (int set = 0; set < 2; ++set)
#pragma unroll
    for (int q = 0; q < 4; ++q) load_b(set, q, set);
  if (tid < RT) {
    const int e = T.entry(A, i0 + min(tid, ne - 1));
    ent[tid] = e;
    float sc = A.w ? A.w[(long long)(e / A.kk) * A.ldw + T.c] : 1.f;
    if constexpr (SPLIT) {
      float2 st[kMaxBlocks];
#pragma unroll
      for (int j = 0; j < kMaxBlocks; ++j) st[j] = stats[(long long)e * blocks + min(j, blocks - 1)];
      float M = st[0].x, L = 0.f;
#pragma unroll
      for (int j = 1; j < kMaxBlocks; ++j) M = fmaxf(M, st[j].x);
#pragma unroll
      for (int j = 0; j < kMaxBlocks; ++j) {
        const float f = __builtin_amdgcn_exp2f(st[j].x - M);
        fac[tid][j] = (_Float16)f;
        if (j < blocks) L += f * st[j].y;
      }
      sc /= L;
    }
    scale[tid] = sc;
  }
  __syncthreads();
  for (int kb = 0; kb < nkb; ++kb)
#pragma unroll
    for (int i = 0; i < NT; ++i) {
      const int rid = tid + 256 * i, r = rid >> 3;
      stage_to_lds(pl + (kb * RT * BK + (256 * i + 64 * wv) * 8),
                   P + (long long)ent[r] * N + kb * BK + (((rid & 7) ^ sw(r)) << 3));
    }
  wait_vmem<0>();
  __syncthreads();
  f32x16 acc[NT][2];
#pragma unroll
  for (int mt = 0; mt < NT; ++mt)
#pragma unroll
    for (int nt = 0; nt < 2; ++nt) acc[mt][nt] = (f32x16){};
  auto step = [&](auto set_c, int v) {
    constexpr int set = decltype(set_c)::value;
    const int kb = v % nkb;
    half8_t a[4][NT];
#pragma unroll
    for (int q = 0; q < 4; ++q)
#pragma unroll
      for (int mt = 0; mt < NT; ++mt) {
        const int r = mt * 32 + l32;
        a[q][mt] = *reinterpret_cast<const half8_t*>(pl + kb * RT * BK + r * BK + (((q * 2 + hl) ^ sw(r)) << 3));
      }
    if constexpr (SPLIT) {
#pragma unroll
      for (int mt = 0; mt < NT; ++mt) {
        const _Float16 f = fac[mt * 32 + l32][kb * BK / bspan];
        const half8_t f8 = {f, f, f, f, f, f, f, f};
#pragma unroll
        for (int q = 0; q < 4; ++q) a[q][mt] = a[q][mt] * f8;
      }
    }
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int q = 0; q < 4; ++q) {
#pragma unroll
      for (int mt = 0; mt < NT; ++mt)
#pragma unroll
        for (int nt = 0; nt < 2; ++nt) acc[mt][nt] = mfma32(a[q][mt], fb[set][q][nt], acc[mt][nt]);
      load_b(set, q, v + 2);
      __builtin_amdgcn_sched_barrier(0);
    }
    if (kb + 1 < nkb) return;   // wave-uniform
    // The tile's last k step.  acc[mt][nt][r]: entry 32 mt + 8 (r / 4) + 4 hl + r % 4, dim 32 nt + l32.
    const int dd0 = (dt0 + v / nkb) * 256 + wv * 64 + l32;
#pragma unroll
    for (int mt = 0; mt < NT; ++mt)
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const int i = mt * 32 + (r >> 2) * 8 + hl * 4 + (r & 3);
        if (i >= ne) continue;
        float* o = out + (long long)(ONE ? ent[i] / A.kk : ent[i]) * ldo;
        const float f = scale[i];
#pragma unroll
        for (int nt = 0; nt < 2; ++nt)
          if (dd0 + nt * 32 < d) o[dd0 + nt * 32] = acc[mt][nt][r] * f;
      }
#pragma unroll
    for (int mt = 0; mt < NT; ++mt)
#pragma unroll
      for (int nt = 0; nt < 2; ++nt) acc[mt][nt] = (f32x16){};
  };
  for (int v = 0; v < steps; v += 2) {
    step(std::integral_constant<int, 0>{}, v);
    if (v + 1 < steps) step(std::integral_constant<int, 1>{}, v + 1);
  }
}

// ------------------------------------------------------------------------------------------
// out[row] = sum over the row's entries of part, in rank order (idx: entries with idx < 0 are empty;
// without idx rank j is chunk j of the row's library).  ROUTE (backward) adds the routing term
// sum_j dl_j S_{c_j}, dl_j = route_temp * w_j (dw_j - sum_i w_i dw_i), dw = gamma (+ dw_ext).
template <bool ROUTE>
__global__ __launch_bounds__(256) void entries_merge_kernel(
    const float* __restrict__ part, int kk, const int* __restrict__ idx, const int* __restrict__ row_ptr,
    const int* __restrict__ chunk_ptr, int G, int d, const float* __restrict__ w, long long ldw,
    const float* __restrict__ gamma, const float* __restrict__ dw_ext, long long lde, const float* __restrict__ S,
    float route_temp, float* __restrict__ out, long long ldo) {
  const int row = blockIdx.x;
  const int g = library_of(row_ptr, G, row);
  const int c0 = chunk_ptr[g], C = chunk_ptr[g + 1] - c0;
  auto chunk_of = [&](int j) { return idx ? idx[(long long)row * kk + j] : (j < C ? j : -1); };
  float sdot = 0.f;
  if constexpr (ROUTE) {
    for (int j = 0; j < kk; ++j) {   // uniform: every thread the same sum in the same order
      const int c = chunk_of(j);
      if (c < 0) continue;
      const float dw = gamma[(long long)row * kk + j] + (dw_ext ? dw_ext[(long long)row * lde + c] : 0.f);
      sdot += w[(long long)row * ldw + c] * dw;
    }
  }
  for (int e = threadIdx.x * 4; e < d; e += 256 * 4) {
    f32x4 o = {0.f, 0.f, 0.f, 0.f};
#pragma unroll 4
    for (int j = 0; j < kk; ++j) {
      const int c = chunk_of(j);
      if (c < 0) continue;
      o += *reinterpret_cast<const f32x4*>(part + ((long long)row * kk + j) * d + e);
      if constexpr (ROUTE) {
        const float wj = w[(long long)row * ldw + c];
        const float dw = gamma[(long long)row * kk + j] + (dw_ext ? dw_ext[(long long)row * lde + c] : 0.f);
        const float dl = route_temp * wj * (dw - sdot);
        const f32x4 s = *reinterpret_cast<const f32x4*>(S + (long long)(c0 + c) * d + e);
#pragma unroll
        for (int i = 0; i < 4; ++i) o[i] = fmaf(dl, s[i], o[i]);
      }
    }
    *reinterpret_cast<f32x4*>(out + (long long)row * ldo + e) = o;
  }
}

constexpr int kBlockSlots = 128;   // slots per block of a split page

int check_entries(int M, int kk, int G, int n_chunks, int max_rows, int d, int N, long long page_stride) {
  if (M < 0 || kk <= 0 || G <= 0 || n_chunks <= 0 || max_rows < 0 || max_rows > M) return XENC_EINVAL;
  if (d <= 0 || d % BK != 0 || N <= 0 || N > 512 || N % BK != 0) return XENC_EINVAL;
  if (page_stride < (long long)N * d || page_stride % 8 != 0) return XENC_EINVAL;
  if ((long long)M * kk > INT_MAX) return XENC_EINVAL;
  return XENC_OK;
}

EntryArgs entry_args(int G, int n_chunks, int kk, int max_rows, int d, int N, const int* row_ptr,
                     const int* chunk_ptr, const int* list, const int* count, const void* pages, long long page_stride,
                     const int* chunk_page, const int* chunk_nvalid, const float* w, long long ldw) {
  // (fewer chunks than XCDs: unpadded, so that the tiles of a chunk spread over several XCDs)
  const int cp = n_chunks < kXcds ? n_chunks : (n_chunks + kXcds - 1) / kXcds * kXcds;
  return EntryArgs{G, n_chunks, cp, kk, max_rows, d, N, row_ptr, chunk_ptr, list,
                   count, static_cast<const _Float16*>(pages), page_stride, chunk_page, chunk_nvalid, w, ldw};
}

}  // namespace
}  // namespace xenc

using namespace xenc;

extern "C" int xenc_entries_list(const int* idx, int M, int kk, const int* row_ptr, const int* chunk_ptr, int G,
                                 int n_chunks, int max_rows, int* list, int* count, void* stream) {
  if (M < 0 || kk <= 0 || G <= 0 || n_chunks <= 0 || max_rows < 0 || max_rows > M) return XENC_EINVAL;
  if ((long long)M * kk > INT_MAX) return XENC_EINVAL;
  if (!row_ptr || !chunk_ptr || !count || (M > 0 && (!idx || !list))) return XENC_ENULL;
  hipLaunchKernelGGL(entries_list_kernel, dim3(n_chunks), dim3(kListThreads), 0, reinterpret_cast<hipStream_t>(stream),
                     idx, kk, row_ptr, chunk_ptr, G, max_rows, list, count);
  return check_launch();
}

extern "C" int xenc_entries_scores(int mode, const void* x, int M, int d, int kk, const int* row_ptr,
                                   const int* chunk_ptr, int G, int n_chunks, int max_rows, const int* list,
                                   const int* count, int tile_rows, const void* pages_a, int slots_per_page,
                                   long long page_stride, const int* chunk_page, const int* chunk_nvalid, float temp,
                                   const float* w, long long ldw, void* p, void* ds, float* gamma, int blocks,
                                   float* stats, void* stream) {
  const int N = slots_per_page;
  if (mode < 0 || mode > 3 || (tile_rows != 32 && tile_rows != 64)) return XENC_EINVAL;
  if (int rc = check_entries(M, kk, G, n_chunks, max_rows, d, N, page_stride)) return rc;
  if (M == 0 || max_rows == 0) return XENC_OK;
  if (!x || !row_ptr || !chunk_ptr || !pages_a || !chunk_page || !chunk_nvalid || !p || !list != !count)
    return XENC_ENULL;
  const bool bwd = mode & 1;
  if (bwd && (!w || !ds || !gamma)) return XENC_ENULL;
  if (!aligned16(x) || !aligned16(pages_a) || !aligned16(p) || (bwd && !aligned16(ds))) return XENC_EALIGN;
  const EntryArgs A = entry_args(G, n_chunks, kk, max_rows, d, N, row_ptr, chunk_ptr, list, count, pages_a, page_stride,
                                 chunk_page, chunk_nvalid, w, ldw);
  // Slot blocks: 128 slots each (forward modes, 32-entry tiles).
  if (blocks != 1 && (bwd || tile_rows != 32 || blocks != (N + kBlockSlots - 1) / kBlockSlots)) return XENC_EINVAL;
  if (blocks != 1 && mode == 0 && !stats) return XENC_ENULL;
  const long long grid = (long long)A.Cp * blocks * ((max_rows + tile_rows - 1) / tile_rows);
  if (grid > INT_MAX) return XENC_EINVAL;
  hipStream_t st = reinterpret_cast<hipStream_t>(stream);
  auto launch = [&](auto kernel) {
    hipLaunchKernelGGL(kernel, dim3((unsigned)grid), dim3(kEntThreads), 0, st, A, static_cast<const _Float16*>(x),
                       mode == 0 ? temp * kLog2e : temp, static_cast<_Float16*>(p), static_cast<_Float16*>(ds), gamma,
                       blocks, reinterpret_cast<float2*>(stats));
  };
  if (blocks > 1) {
    if (mode == 0) launch(entries_scores_kernel<4, kBlockSlots / 64, 1>);
    else launch(entries_scores_kernel<2, kBlockSlots / 64, 1>);
    return check_launch();
  }
#define XENC_ENT_SG(MODE, NT)                                          \
  if (N > 256) launch(entries_scores_kernel<MODE, 8, NT>);             \
  else if (N > 128) launch(entries_scores_kernel<MODE, 4, NT>);        \
  else if (N > 64) launch(entries_scores_kernel<MODE, 2, NT>);         \
  else launch(entries_scores_kernel<MODE, 1, NT>);
#define XENC_ENT(MODE)                                                 \
  if (tile_rows == 64 && N > 128) {                                    \
    if (N > 256) launch(entries_scores_kernel<MODE, 8, 2>);            \
    else launch(entries_scores_kernel<MODE, 4, 2>);                    \
  } else if (tile_rows == 64) {                                        \
    return XENC_EINVAL;                                                \
  } else {                                                             \
    XENC_ENT_SG(MODE, 1)                                               \
  }
  switch (mode) {
    case 0: XENC_ENT(0) break;
    case 1: XENC_ENT(1) break;
    case 2: XENC_ENT(2) break;
    default: XENC_ENT(3) break;
  }
#undef XENC_ENT
#undef XENC_ENT_SG
  return check_launch();
}

extern "C" int xenc_entries_readout(const void* a, int M, int d, int kk, const int* row_ptr, const int* chunk_ptr, int G,
                                    int n_chunks, int max_rows, const int* list, const int* count, int tile_rows,
                                    const void* pages_b, int slots_per_page, long long page_stride,
                                    const int* chunk_page, const float* w, long long ldw, int by_row, int blocks,
                                    const float* stats, float* out, long long ldo, void* stream) {
  const int N = slots_per_page;
  if (tile_rows != 32 && tile_rows != 64) return XENC_EINVAL;
  if (int rc = check_entries(M, kk, G, n_chunks, max_rows, d, N, page_stride)) return rc;
  if (ldo < d || (by_row && kk != 1)) return XENC_EINVAL;
  if (blocks != 1 && (tile_rows != 32 || blocks != (N + kBlockSlots - 1) / kBlockSlots)) return XENC_EINVAL;
  if (M == 0 || max_rows == 0) return XENC_OK;
  if (!a || !row_ptr || !chunk_ptr || !pages_b || !chunk_page || !out || !list != !count) return XENC_ENULL;
  if (!aligned16(a) || !aligned16(pages_b)) return XENC_EALIGN;
  const EntryArgs A = entry_args(G, n_chunks, kk, max_rows, d, N, row_ptr, chunk_ptr, list, count, pages_b, page_stride,
                                 chunk_page, nullptr, w, ldw);
  // Workgroups that will have entries: M * kk of them (at most every row of every chunk).
  const int dim_tiles = (d + 255) / 256;
  const long long row_tiles = (max_rows + tile_rows - 1) / tile_rows;
  const long long tiles = std::min<long long>(((long long)M * kk + tile_rows - 1) / tile_rows + n_chunks / 2,
                                              row_tiles * n_chunks);
  int dpw = 1;
  while (dpw < dim_tiles && tiles * ((dim_tiles + dpw - 1) / dpw) > 2048) dpw *= 2;
  const long long grid = (long long)A.Cp * ((dim_tiles + dpw - 1) / dpw) * row_tiles;
  if (grid > INT_MAX) return XENC_EINVAL;
  const size_t lds = (size_t)tile_rows * N * 2;
  hipStream_t st = reinterpret_cast<hipStream_t>(stream);
  auto launch = [&](auto kernel) {
    hipLaunchKernelGGL(kernel, dim3((unsigned)grid), dim3(256), lds, st, A, static_cast<const _Float16*>(a), dim_tiles,
                       dpw, out, ldo, blocks, kBlockSlots, reinterpret_cast<const float2*>(stats));
  };
  if (tile_rows == 64) {
    if (by_row) launch(entries_readout_kernel<2, true, false>);
    else launch(entries_readout_kernel<2, false, false>);
  } else if (blocks > 1 && stats) {
    if (by_row) launch(entries_readout_kernel<1, true, true>);
    else launch(entries_readout_kernel<1, false, true>);
  } else {
    if (by_row) launch(entries_readout_kernel<1, true, false>);
    else launch(entries_readout_kernel<1, false, false>);
  }
  return check_launch();
}

extern "C" int xenc_entries_merge(const float* part, int M, int d, int kk, const int* idx, const int* row_ptr,
                                  const int* chunk_ptr, int G, const float* w, long long ldw, const float* gamma,
                                  const float* dw_ext, long long lde, const float* S, float route_temp, float* out,
                                  long long ldo, void* stream) {
  if (M < 0 || kk <= 0 || G <= 0 || d <= 0 || d % 4 != 0 || ldo < d || ldo % 4 != 0) return XENC_EINVAL;
  if (M == 0) return XENC_OK;
  if (!part || !row_ptr || !chunk_ptr || !out || (S && (!w || !gamma))) return XENC_ENULL;
  if (!aligned16(part) || !aligned16(out) || (S && !aligned16(S))) return XENC_EALIGN;
  hipStream_t st = reinterpret_cast<hipStream_t>(stream);
  auto launch = [&](auto kernel) {
    hipLaunchKernelGGL(kernel, dim3(M), dim3(256), 0, st, part, kk, idx, row_ptr, chunk_ptr, G, d, w, ldw, gamma,
                       dw_ext, lde, S, route_temp, out, ldo);
  };
  if (S) launch(entries_merge_kernel<true>);
  else launch(entries_merge_kernel<false>);
  return check_launch();
}
