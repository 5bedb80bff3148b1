// Routing (a1) and token permutation / segmentation (a2) for the MoE expert path.
//
// Routing: one 256-thread workgroup per token, selection by ranks under the
// total order (score desc, index asc), so the choice and its order equal a
// sequential scan's and take a fixed number of barriers: each expert's rank
// inside its group (grouped routing) or 32-expert chunk (softmax) prunes the
// candidates to K per group, group scores and group ranks pick the groups,
// and a candidate's rank among the survivors is its output slot.  Weights
// are formed by one thread in a fixed fp32 sequence (see xtu_expf).
//
// Segmentation: a stable counting sort of the flat (token, expert) pairs by
// bucket, in two launches (per-block counts; every block sums all blocks'
// counts and places its own pairs).  Ranks inside a block are exact: a wave
// finds the lanes sharing its bucket with ballots, waves are ordered through
// an LDS table of counts, and blocks through the summed counts.
#include <mutex>
#include <stdio.h>

#include <type_traits>

#include "route_tiny.hpp"
#include "xtu_common.hpp"

// Segmentation workspace of xtu_segment_noalloc: one statically allocated
// array per GPU (each device holds its own copy until the process ends).
// Host code must not use this name as an address: it is a host-side stand-in.
// The device address comes from hipGetSymbolAddress, once per device.
static constexpr size_t kNoAllocScratchBytes = 4u << 20;
static __device__ __align__(256) int32_t scratch[kNoAllocScratchBytes / sizeof(int32_t)];

namespace xtu {
namespace {

using tiny::SmallArgs;

constexpr int kWave = 64;

__device__ __forceinline__ bool better(float sa, int ia, float sb, int ib) {
  return (sa > sb) || (sa == sb && ia < ib);
}

constexpr int kMaxE = 1024;
constexpr int kMaxK = 16;
constexpr int kMaxGroups = 64;

// Routing scratch of one team in LDS, laid out from a base for E experts and
// nc = groups * K candidate slots (words): sc, ws [E]; csc, ce [ncp];
// g1, g2, gs, gsel [64]; sel_e, sel_ws, sel_sc [16]; sum.
__host__ __device__ constexpr int route_team_words(int E, int nc) {
  return 2 * E + 2 * ((nc + 3) & ~3) + 4 * kMaxGroups + 3 * kMaxK + 4;
}

struct RouteScratch {
  float *sc, *ws, *csc, *g1, *g2, *gs, *sel_ws, *sel_sc;
  int *ce, *gsel, *sel_e;
  __device__ RouteScratch(float* base, int E, int nc) {
    const int ncp = (nc + 3) & ~3;
    sc = base;
    ws = sc + E;
    csc = ws + E;
    ce = reinterpret_cast<int*>(csc + ncp);
    g1 = reinterpret_cast<float*>(ce + ncp);
    g2 = g1 + kMaxGroups;
    gs = g2 + kMaxGroups;
    gsel = reinterpret_cast<int*>(gs + kMaxGroups);
    sel_e = gsel + kMaxGroups;
    sel_ws = reinterpret_cast<float*>(sel_e + kMaxK);
    sel_sc = sel_ws + kMaxK;
  }
};

// Make this wave's LDS writes visible to its other lanes.
__device__ __forceinline__ void wave_sync() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// A team of TEAM threads routes one token: TEAM = 64 is one wave (synced as
// a wave), TEAM = 256 is a quarter of a 1024-thread workgroup whose four
// teams run in lockstep through workgroup barriers.
template <int TEAM>
__device__ __forceinline__ void team_sync() {
  if constexpr (TEAM == kWave) wave_sync();
  else __syncthreads();
}

// Number of (score, index) pairs in [j0, j1) that beat (v, e): 4-wide LDS
// reads, independent of each other, so the latencies overlap.
__device__ __forceinline__ int count_better(const float* sc, const int* idx, int j0, int j1,
                                            float v, int e) {
  int r = 0;
  int j = j0;
  if ((j0 & 3) == 0) {
#pragma unroll 4
    for (; j + 4 <= j1; j += 4) {
      const f32x4_t s4 = *reinterpret_cast<const f32x4_t*>(sc + j);
      if (idx) {
        const i32x4_t i4 = *reinterpret_cast<const i32x4_t*>(idx + j);
#pragma unroll
        for (int q = 0; q < 4; ++q) r += better(s4[q], i4[q], v, e) ? 1 : 0;
      } else {
#pragma unroll
        for (int q = 0; q < 4; ++q) r += better(s4[q], j + q, v, e) ? 1 : 0;
      }
    }
  }
  for (; j < j1; ++j) r += better(sc[j], idx ? idx[j] : j, v, e) ? 1 : 0;
  return r;
}

// Route one token with a team (thread `tid` of TEAM; `valid` false: no token,
// the team only keeps step with the barriers).  MODE 0: softmax top-k over
// the logits; MODE 1: DeepSeek-V3 grouped sigmoid.  Threads k < K write the
// k-th choice to ids_out[k] / wts_out[k] (and to the LDS copies if given).
template <int MODE, int TEAM>
__device__ void route_token(const float* __restrict__ l, const float* __restrict__ bias, int E,
                            int K, int n_group, int topk_group, float scale, int renorm,
                            const RouteScratch& s, int tid, bool valid, int32_t* ids_out,
                            float* wts_out, int* ids_lds = nullptr, float* wts_lds = nullptr) {
#pragma clang fp contract(off)
  const float NEG = -__builtin_inff();
  const int gsz = MODE == 1 ? E / n_group : 32;   // group, or pruning chunk
  const int ng = MODE == 1 ? n_group : (E + 31) / 32;
  const int nc = ng * K;
  const int ncp = (nc + 3) & ~3;
  if (valid) {
    for (int e = tid; e < E; e += TEAM) {
      const float x = l[e];
      if (MODE == 0) {
        s.sc[e] = x;
        s.ws[e] = x;
      } else {
        const float w = xtu_sigmoid(x);
        s.sc[e] = w + (bias ? bias[e] : 0.0f);
        s.ws[e] = w;
      }
    }
  }
  for (int c = tid; c < ncp; c += TEAM) {
    s.csc[c] = NEG;
    s.ce[c] = 0x7fffffff;
  }
  team_sync<TEAM>();
  // rank inside the group / chunk; the K best of each become candidates
  if (valid) {
    for (int e = tid; e < E; e += TEAM) {
      const int g = e / gsz, j0 = g * gsz;
      const float v = s.sc[e];
      const int r = count_better(s.sc, nullptr, j0, min(j0 + gsz, E), v, e);
      if (r < K) {
        s.csc[g * K + r] = v;
        s.ce[g * K + r] = e;
      }
      if (MODE == 1) {
        if (r == 0) s.g1[g] = v;
        if (r == 1) s.g2[g] = v;
      }
    }
  }
  team_sync<TEAM>();
  if (MODE == 1) {
    // group score = best + second best; keep the topk_group best groups
    if (tid < ng) s.gs[tid] = gsz >= 2 ? s.g1[tid] + s.g2[tid] : s.g1[tid];
    team_sync<TEAM>();
    if (tid < ng) s.gsel[tid] = count_better(s.gs, nullptr, 0, ng, s.gs[tid], tid) < topk_group;
    team_sync<TEAM>();
    for (int c = tid; c < nc; c += TEAM)   // drop the candidates of the other groups
      if (!s.gsel[c / K]) {
        s.csc[c] = NEG;
        s.ce[c] = 0x7fffffff;
      }
    team_sync<TEAM>();
  }
  // rank among the surviving candidates = output slot
  for (int c = tid; c < nc; c += TEAM) {
    const int e = s.ce[c];
    if (e == 0x7fffffff) continue;
    const float v = s.csc[c];
    const int r = count_better(s.csc, s.ce, 0, ncp, v, e);
    if (r < K) {
      s.sel_e[r] = e;
      s.sel_ws[r] = s.ws[e];
      s.sel_sc[r] = v;
    }
  }
  team_sync<TEAM>();
  // weights: lanes k < K of the team's first wave, sums in k order
  float wk = 0.f;
  if (tid < K) wk = s.sel_ws[tid];
  int id = 0;
  float w = 0.f;
  if (MODE == 0) {
    const float lmax = s.sel_sc[0];
    const float ev = tid < K ? xtu_expf(wk - lmax) : 0.f;   // e^(l_k - lmax)
    float sum = 0.0f;
    if (renorm) {
      for (int k = 0; k < K; ++k) sum = sum + __shfl(ev, k, kWave);
    } else {
      team_sync<TEAM>();   // sel_* read before ws is rewritten
      if (valid)
        for (int e = tid; e < E; e += TEAM) s.ws[e] = xtu_expf(s.sc[e] - lmax);
      team_sync<TEAM>();
      if (tid == 0)
        for (int e = 0; e < E; ++e) sum = sum + s.ws[e];
      sum = __shfl(sum, 0, kWave);
    }
    if (tid < K) {
      id = s.sel_e[tid];
      w = __fdiv_rn(ev, sum);
    }
  } else {
    float sum = 0.0f;
    for (int k = 0; k < K; ++k) sum = sum + __shfl(wk, k, kWave);
    if (tid < K) {
      id = s.sel_e[tid];
      w = renorm ? __fdiv_rn(wk, sum) * scale : wk * scale;
    }
  }
  if (valid && tid < K) {
    ids_out[tid] = id;
    wts_out[tid] = w;
    if (ids_lds) {
      ids_lds[tid] = id;
      wts_lds[tid] = w;
    }
  }
  team_sync<TEAM>();   // the scratch may be reused for the next token
}

// 1024 / TEAM teams per workgroup, one token each: four 256-thread teams, or
// sixteen one-wave teams for at most 64 experts (wave syncs, no workgroup
// barrier).
template <int MODE, int TEAM = 256>
__global__ __launch_bounds__(1024) void route_kernel(const float* __restrict__ logits,
                                                     const float* __restrict__ bias, int T, int E,
                                                     int K, int n_group, int topk_group,
                                                     float scale, int renorm,
                                                     int32_t* __restrict__ ids,
                                                     float* __restrict__ wts) {
  extern __shared__ float route_lds[];
  constexpr int kTeams = 1024 / TEAM;
  const int team = threadIdx.x / TEAM, tid = threadIdx.x % TEAM;
  const long t = (long)blockIdx.x * kTeams + team;
  const int nc = (MODE == 1 ? n_group : (E + 31) / 32) * K;
  const RouteScratch s(route_lds + team * route_team_words(E, nc), E, nc);
  route_token<MODE, TEAM>(logits + t * E, bias, E, K, n_group, topk_group, scale, renorm, s, tid,
                          t < T, ids + t * K, wts + t * K);
}

// The team router's launch: one-wave teams for E <= 64.
template <int MODE>
void launch_route_teams(const float* logits, const float* bias, int T, int E, int K, int n_group,
                        int topk_group, float scale, int renorm, int nc, int32_t* ids,
                        float* wts, hipStream_t stream) {
  const size_t words = route_team_words(E, nc) * sizeof(float);
  if (E <= kWave)
    route_kernel<MODE, kWave><<<(T + 15) / 16, 1024, 16 * words, stream>>>(
        logits, bias, T, E, K, n_group, topk_group, scale, renorm, ids, wts);
  else
    route_kernel<MODE, 256><<<(T + 3) / 4, 1024, 4 * words, stream>>>(
        logits, bias, T, E, K, n_group, topk_group, scale, renorm, ids, wts);
}

// Batches of any size on E = 128 / 256 / 512 (tiny::wave_epl): one wave routes one
// token with tiny::route_token_wave (no workgroup barrier), four tokens per
// workgroup.  Same ids, order and fp32 sequences as route_kernel, which took
// 23.0 us for T = 4096 over 128 experts (5.0 here).
template <int MODE, int EPL>
__global__ __launch_bounds__(256) void route_wave_kernel(const float* __restrict__ logits,
                                                         const float* __restrict__ bias, int T,
                                                         int K, int n_group, int topk_group,
                                                         float scale, int renorm,
                                                         int32_t* __restrict__ ids,
                                                         float* __restrict__ wts) {
  const int w = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
  const long t = (long)blockIdx.x * 4 + w;
  if (t >= T) return;   // whole wave
  tiny::route_token_wave<MODE, EPL>(logits + t * (kWave * EPL), bias, K, n_group, topk_group,
                                    scale, renorm, threadIdx.x % kWave, ids + t * K, wts + t * K,
                                    nullptr, nullptr);
}

template <int MODE>
void launch_route_wave(int epl, const float* logits, const float* bias, int T, int K,
                       int n_group, int topk_group, float scale, int renorm, int32_t* ids,
                       float* wts, hipStream_t stream) {
  const dim3 grid((unsigned)((T + 3) / 4));
  if (epl == 2)
    route_wave_kernel<MODE, 2><<<grid, 256, 0, stream>>>(logits, bias, T, K, n_group, topk_group,
                                                         scale, renorm, ids, wts);
  else if (epl == 4)
    route_wave_kernel<MODE, 4><<<grid, 256, 0, stream>>>(logits, bias, T, K, n_group, topk_group,
                                                         scale, renorm, ids, wts);
  else
    route_wave_kernel<MODE, 8><<<grid, 256, 0, stream>>>(logits, bias, T, K, n_group, topk_group,
                                                         scale, renorm, ids, wts);
}

// ----------------------------------------------------------------------------
// segmentation
// ----------------------------------------------------------------------------
// A workgroup ranks one pair per thread and round: a wave finds the lanes
// sharing its bucket with one ballot per bit of the bucket id and writes its
// per-bucket counts as one row of a 16-bit [wave][bucket] table in LDS; an
// exclusive prefix down the table's columns (two buckets per thread) orders
// the waves.  A pair's position is then bucket start + its wave's prefix +
// its rank in the wave: a fixed number of barriers per 1024 pairs, whatever
// the bucket count.
constexpr int kSegThreads = 1024;
constexpr int kSegWaves = kSegThreads / kWave;
// Blocks of a large batch: enough to spread the ranking over the chip, few
// enough that every block can sum all blocks' counts by itself (128 blocks x
// 514 buckets = 0.26 MB of L2 reads per block), which saves a scan launch.
constexpr int kSegMaxBlocks = 128;
// pairs per block of the workspace bound's first term (see
// xtu_segment_workspace_bytes)
constexpr int kSegBoundChunk = 4096;

struct SegArgs {
  const int32_t* ids;
  const float* wts;
  const int32_t* id_map;   // optional id translation applied before bucketing
  int T, K, E, NS, drop_zero, A, NB;
  int rounds;              // rounds of kSegThreads pairs per block
};

struct SegOut {
  int32_t *seg_start, *active, *n_active, *tile_expert, *tile_row0, *n_tiles, *expert_tile_start;
  int NB, bm, A;
};

// Buckets rounded up so that a table row is whole 16-byte pieces.
__host__ __device__ constexpr int seg_nbp(int NB) { return (NB + 7) & ~7; }

__device__ __forceinline__ int bucket_of(const SegArgs& a, int p, float* w_out, int* tok_out) {
  const int TK = a.T * a.K;
  if (p < TK) {
    int e = a.ids[p];
    if (a.id_map && e >= 0 && e < a.E) e = a.id_map[e];
    const float w = a.wts[p];
    *w_out = w;
    *tok_out = p / a.K;
    int b = (e < 0 || e >= a.E) ? (a.E + a.NS) : e;
    if (a.drop_zero && w == 0.0f) b = a.E + a.NS;
    return b;
  }
  const int q = p - TK;
  *w_out = 1.0f;
  *tok_out = q / a.NS;
  return a.E + q % a.NS;
}

// Inclusive prefix sum across the 64 lanes of a wave (DPP row shifts, then
// row broadcasts); lanes whose source is out of range add 0.
__device__ __forceinline__ int wave_incl_scan(int x) {
  x += __builtin_amdgcn_update_dpp(0, x, 0x111, 0xF, 0xF, false);   // row_shr:1
  x += __builtin_amdgcn_update_dpp(0, x, 0x112, 0xF, 0xF, false);   // row_shr:2
  x += __builtin_amdgcn_update_dpp(0, x, 0x114, 0xF, 0xF, false);   // row_shr:4
  x += __builtin_amdgcn_update_dpp(0, x, 0x118, 0xF, 0xF, false);   // row_shr:8
  x += __builtin_amdgcn_update_dpp(0, x, 0x142, 0xA, 0xF, false);   // row_bcast:15
  x += __builtin_amdgcn_update_dpp(0, x, 0x143, 0xC, 0xF, false);   // row_bcast:31
  return x;
}

// Rank of this lane among the wave's valid lanes with its bucket b (below
// 1 << nbits); `same` = those lanes.
__device__ __forceinline__ int wave_bucket_rank(int b, bool valid, int nbits,
                                                unsigned long long& same) {
  unsigned long long m = __ballot(valid);
  for (int bit = 0; bit < nbits; ++bit) {
    const bool on = (b >> bit) & 1;
    const unsigned long long b1 = __ballot(valid && on);
    m &= on ? b1 : ~b1;
  }
  same = m;
  return __builtin_amdgcn_mbcnt_hi((uint32_t)(m >> 32),
                                   __builtin_amdgcn_mbcnt_lo((uint32_t)m, 0u));
}

__device__ __forceinline__ void clear_counts(uint16_t* wc, int nbp, int nw) {
  for (int i = threadIdx.x; i < nw * nbp / 8; i += blockDim.x)
    reinterpret_cast<u32x4_t*>(wc)[i] = u32x4_t{0u, 0u, 0u, 0u};
}

// Buckets 2t and 2t + 1 of thread t: the nw waves' counts become exclusive
// prefixes in place; c0, c1 = the totals (at most 1024: 16-bit halves).
__device__ __forceinline__ void column_prefix(uint16_t* wc, int nbp, int nw, int t, int& c0,
                                              int& c1) {
  uint32_t* col = reinterpret_cast<uint32_t*>(wc) + t;
  uint32_t c[kSegWaves], run = 0u;
#pragma unroll
  for (int w = 0; w < kSegWaves; ++w) c[w] = w < nw ? col[w * (nbp / 2)] : 0u;
#pragma unroll
  for (int w = 0; w < kSegWaves; ++w) {
    if (w < nw) col[w * (nbp / 2)] = run;
    run += c[w];
  }
  c0 = (int)(run & 0xffffu);
  c1 = (int)(run >> 16);
}

// Bucket totals c0, c1 of thread t's buckets (2t, 2t + 1) -> their first
// rows; with `write`, seg_start, the list of non-empty expert buckets and the
// GEMM tile list (tiles of bm rows inside each non-trash bucket).  Called by
// the whole block (kSegThreads or fewer threads, at least NB / 2).
__device__ __forceinline__ void bucket_starts(const SegOut& o, int t, int c0, int c1, bool write,
                                              int (*wsum)[kSegWaves], int& s0, int& s1) {
  const int NB = o.NB, e0 = 2 * t;
  // the last bucket is the trash bucket
  const bool x0 = e0 < NB - 1, x1 = e0 + 1 < NB - 1;
  const int n0 = x0 ? (c0 + o.bm - 1) / o.bm : 0, n1 = x1 ? (c1 + o.bm - 1) / o.bm : 0;
  const int a0 = x0 && c0 > 0 ? 1 : 0, a1 = x1 && c1 > 0 ? 1 : 0;
  const int lane = t % kWave, wv = t / kWave, nwv = (int)blockDim.x / kWave;
  const int ir = wave_incl_scan(c0 + c1), ia = wave_incl_scan(a0 + a1),
            it = wave_incl_scan(n0 + n1);
  if (lane == kWave - 1) {
    wsum[0][wv] = ir;
    wsum[1][wv] = ia;
    wsum[2][wv] = it;
  }
  __syncthreads();
  int br = ir - c0 - c1, ba = ia - a0 - a1, bt = it - n0 - n1, na = 0, nt = 0;
#pragma unroll
  for (int q = 0; q < kSegWaves; ++q) {
    if (q < nwv) {
      const int r = wsum[0][q], c = wsum[1][q], n = wsum[2][q];
      if (q < wv) {
        br += r;
        ba += c;
        bt += n;
      }
      na += c;
      nt += n;
    }
  }
  s0 = br;
  s1 = br + c0;
  if (!write) return;
  if (e0 < NB) {
    o.seg_start[e0] = s0;
    o.expert_tile_start[e0] = bt;
  }
  if (e0 + 1 < NB) {
    o.seg_start[e0 + 1] = s1;
    o.expert_tile_start[e0 + 1] = bt + n0;
  }
  if (a0) o.active[ba] = e0;
  if (a1) o.active[ba + a0] = e0 + 1;
  for (int j = 0; j < n0; ++j) {
    o.tile_expert[bt + j] = e0;
    o.tile_row0[bt + j] = s0 + j * o.bm;
  }
  for (int j = 0; j < n1; ++j) {
    o.tile_expert[bt + n0 + j] = e0 + 1;
    o.tile_row0[bt + n0 + j] = s1 + j * o.bm;
  }
  if (t == 0) {
    o.seg_start[NB] = o.A;
    o.expert_tile_start[NB] = nt;
    o.n_active[0] = na;
    o.n_tiles[0] = nt;
  }
}

// Bucket counts of each block's pairs: bcnt[block][nbp].
__global__ __launch_bounds__(kSegThreads) void seg_count_kernel(SegArgs a,
                                                                int32_t* __restrict__ bcnt) {
  extern __shared__ int cnt[];
  const int nbp = seg_nbp(a.NB);
  for (int e = threadIdx.x; e < nbp; e += kSegThreads) cnt[e] = 0;
  __syncthreads();
  const int base = blockIdx.x * a.rounds * kSegThreads;
  for (int r = 0; r < a.rounds; ++r) {
    const int p = base + r * kSegThreads + threadIdx.x;
    if (p < a.A) {
      float w;
      int tok;
      atomicAdd(&cnt[bucket_of(a, p, &w, &tok)], 1);
    }
  }
  __syncthreads();
  for (int e = threadIdx.x; e < nbp; e += kSegThreads)
    bcnt[(size_t)blockIdx.x * nbp + e] = cnt[e];
}

// Every block sums all blocks' counts for itself (bucket totals and the part
// before this block; nblocks <= kSegMaxBlocks), scans the totals and places
// its own pairs; block 0 also writes the bucket starts and tile lists.
// Latency bound.
__global__ __launch_bounds__(kSegThreads) void seg_place_kernel(
    SegArgs a, SegOut o, const int32_t* __restrict__ bcnt, int nblocks,
    int32_t* __restrict__ sorted_pair, int32_t* __restrict__ sorted_tok,
    float* __restrict__ sorted_wts, int32_t* __restrict__ inv) {
  extern __shared__ __attribute__((aligned(16))) int place_lds[];
  __shared__ int wsum[3][kSegWaves];
  const int nbp = seg_nbp(a.NB), half = nbp / 2;
  int* base = place_lds;   // [nbp] pairs of earlier blocks, then this block's next rows
  uint16_t* wc = reinterpret_cast<uint16_t*>(place_lds + nbp);   // [waves][nbp]
  int* tot = place_lds + nbp;   // [nbp] bucket totals, before wc is used
  const int tid = threadIdx.x, wv = tid / kWave;
  const int p0 = blockIdx.x * a.rounds * kSegThreads;
  // this thread's first pair, in flight beside the counts
  float w = 0.f;
  int tok = 0;
  int b = p0 + tid < a.A ? bucket_of(a, p0 + tid, &w, &tok) : -1;
  for (int e = tid; e < 2 * nbp; e += kSegThreads) place_lds[e] = 0;
  __syncthreads();
  // thread groups of gs threads each take every ng-th block's counts
  const int gs = (half + kWave - 1) / kWave * kWave, ng = kSegThreads / gs;
  const int g = tid / gs, t = tid % gs;
  if (g < ng && t < half) {
    int t0 = 0, t1 = 0, b0 = 0, b1 = 0;
#pragma unroll 8
    for (int j = g; j < nblocks; j += ng) {
      const int2 c = reinterpret_cast<const int2*>(bcnt + (size_t)j * nbp)[t];
      t0 += c.x;
      t1 += c.y;
      if (j < (int)blockIdx.x) {
        b0 += c.x;
        b1 += c.y;
      }
    }
    atomicAdd(&tot[2 * t], t0);
    atomicAdd(&tot[2 * t + 1], t1);
    atomicAdd(&base[2 * t], b0);
    atomicAdd(&base[2 * t + 1], b1);
  }
  __syncthreads();
  int s0, s1;
  {
    const int c0 = tid < half ? tot[2 * tid] : 0, c1 = tid < half ? tot[2 * tid + 1] : 0;
    bucket_starts(o, tid, c0, c1, blockIdx.x == 0, wsum, s0, s1);   // one barrier inside
  }
  if (tid < half) {
    base[2 * tid] += s0;
    base[2 * tid + 1] += s1;
  }
  const int nbits = 32 - __builtin_clz(a.NB - 1);   // bits of the largest bucket id (NB >= 2)
  for (int r = 0; r < a.rounds; ++r) {
    const int p = p0 + r * kSegThreads + tid;
    if (p - tid >= a.A) break;   // whole block
    if (r > 0) b = p < a.A ? bucket_of(a, p, &w, &tok) : -1;
    const bool valid = b >= 0;
    unsigned long long same;
    const int rank = wave_bucket_rank(b, valid, nbits, same);
    clear_counts(wc, nbp, kSegWaves);
    __syncthreads();
    if (valid && rank == 0) wc[wv * nbp + b] = (uint16_t)__popcll(same);
    __syncthreads();
    int c0 = 0, c1 = 0;
    if (tid < half) column_prefix(wc, nbp, kSegWaves, tid, c0, c1);
    __syncthreads();
    if (valid) {
      const int pos = base[b] + wc[wv * nbp + b] + rank;
      sorted_pair[pos] = p;
      sorted_tok[pos] = tok;
      sorted_wts[pos] = w;
      inv[p] = pos;
    }
    if (r + 1 < a.rounds) {
      __syncthreads();
      if (tid < half) {
        base[2 * tid] += c0;
        base[2 * tid + 1] += c1;
      }
    }
  }
}

// ----------------------------------------------------------------------------
// Small batches (decode): routing and the whole segmentation in one
// workgroup.  A = T*K + T*NS <= 1024 pairs, NB <= 2048 buckets.  Same
// outputs, same order and same fp32 sequence as the multi-launch path.
// ----------------------------------------------------------------------------
constexpr int kSmallMaxA = 1024;
constexpr int kSmallMaxNB = 2048;
static_assert(kSmallMaxA <= kSegThreads && kSmallMaxNB <= 2 * kSegThreads,
              "one pair and two buckets per thread");

// Buckets of the ballot segmentation, at most: its ballots are one per bucket,
// the count table's one per bit.  Routing and segmentation in one launch,
// ballots against the table: 17 buckets grouped sigmoid T = 1 / 8 6.1 / 12.1 us
// against 6.4 / 13.0, given ids 256 pairs 3.66 / 3.71; 25 buckets 6.9 / 13.5
// against 6.6 / 13.7, 4.2 / 3.5; 61 buckets (softmax, K = 4) 8.6 / 15.5 against
// 6.4 / 12.7, 6.4 / 3.7.
constexpr int kFewNB = 18;

struct FewSmem {
  int wc[kFewNB][kSegWaves];   // pairs of bucket v in wave q
  int bstart[kFewNB];
};

// Few buckets: a stable counting sort of the A pairs (pair p in thread p) over
// NB <= kFewNB buckets.  Per wave, one ballot per bucket gives each pair its rank
// among the wave's pairs of its bucket and the wave's count; one wave scans
// the bucket totals.  Position = bucket start + the bucket's pairs in
// earlier waves + rank: the same stable order.  Two barriers fewer than the
// count table: tiny Mixtral's layer (256 pairs over 9 buckets) 40.5 us against
// 41.1.
__device__ __forceinline__ void segment_few_buckets(const SmallArgs& a, FewSmem& g, int b, float w,
                                                    int A, int TK, int NB) {
  const int NW = blockDim.x / kWave;
  const int tid = threadIdx.x, lane = tid % kWave, wv = tid / kWave;
  const int K = a.K, NS = a.NS;
  int rank = 0;
  for (int v = 0; v < NB; ++v) {
    const unsigned long long m = __ballot(b == v);
    if (lane == 0) g.wc[v][wv] = __popcll(m);
    if (b == v)
      rank = __builtin_amdgcn_mbcnt_hi((uint32_t)(m >> 32),
                                       __builtin_amdgcn_mbcnt_lo((uint32_t)m, 0u));
  }
  __syncthreads();
  if (wv == 0) {
    // lane v: bucket v's rows, its start; active entries and tile lists
    int c = 0;
    if (lane < NB)
      for (int q = 0; q < NW; ++q) c += g.wc[lane][q];
    const int start = wave_incl_scan(c) - c;
    const bool live = lane < NB - 1 && c > 0;
    const unsigned long long am = __ballot(live);
    const int ai = __builtin_amdgcn_mbcnt_hi((uint32_t)(am >> 32),
                                             __builtin_amdgcn_mbcnt_lo((uint32_t)am, 0u));
    const int nt = (lane < NB - 1) ? (c + a.bm - 1) / a.bm : 0;
    const int tinc = wave_incl_scan(nt);
    const int t0 = tinc - nt;
    if (lane < NB) {
      g.bstart[lane] = start;
      a.seg_start[lane] = start;
      a.expert_tile_start[lane] = t0;
    }
    if (live) {
      a.active[ai] = lane;
      for (int j = 0; j < nt; ++j) {
        a.tile_expert[t0 + j] = lane;
        a.tile_row0[t0 + j] = start + j * a.bm;
      }
    }
    if (lane == 0) {
      const int n_til = __builtin_amdgcn_readlane(tinc, 63);
      a.seg_start[NB] = A;
      a.expert_tile_start[NB] = n_til;
      a.n_active[0] = __popcll(am);
      a.n_tiles[0] = n_til;
    }
  }
  __syncthreads();
  if (tid < A) {
    int pos = g.bstart[b] + rank;
    for (int q = 0; q < wv; ++q) pos += g.wc[b][q];
    a.sorted_pair[pos] = tid;
    a.inv[tid] = pos;
    a.sorted_tok[pos] = tid < TK ? tid / K : (tid - TK) / NS;
    a.sorted_wts[pos] = w;
  }
}

// Softmax top-K of one token by one thread, for at most kLaneE experts and
// kLaneK choices: the selection scan in (score desc, index asc) order and
// the weights in the same fp32 sequence as route_token (e^(l_k - lmax), the
// sum over the K chosen in selection order, or over all E in index order
// without renormalisation; one correctly rounded division each).
constexpr int kLaneE = 32, kLaneK = 8;

__device__ __forceinline__ void route_token_lane(const float* __restrict__ l, int E, int K,
                                                 int renorm, int32_t* ids_out, float* wts_out,
                                                 int32_t* ids_lds, float* wts_lds) {
  float v[kLaneE];
#pragma unroll
  for (int e = 0; e < kLaneE; ++e) v[e] = e < E ? l[e] : 0.f;
  int sel[kLaneK];
  float sv[kLaneK];
  uint32_t used = 0u;
#pragma unroll
  for (int k = 0; k < kLaneK; ++k) {
    if (k < K) {
      int best = -1;
      float bv = 0.f;
#pragma unroll
      for (int e = 0; e < kLaneE; ++e) {
        if (e < E && !((used >> e) & 1u) && (best < 0 || better(v[e], e, bv, best))) {
          best = e;
          bv = v[e];
        }
      }
      sel[k] = best;
      sv[k] = bv;
      used |= 1u << best;
    }
  }
  const float lmax = sv[0];
  float ev[kLaneK];
  float sum = 0.0f;
#pragma unroll
  for (int k = 0; k < kLaneK; ++k) {
    if (k < K) {
      ev[k] = xtu_expf(sv[k] - lmax);
      sum = sum + ev[k];
    }
  }
  if (!renorm) {
    sum = 0.0f;
#pragma unroll
    for (int e = 0; e < kLaneE; ++e)
      if (e < E) sum = sum + xtu_expf(v[e] - lmax);
  }
#pragma unroll
  for (int k = 0; k < kLaneK; ++k) {
    if (k < K) {
      const float w = __fdiv_rn(ev[k], sum);
      ids_out[k] = sel[k];
      wts_out[k] = w;
      ids_lds[k] = sel[k];
      wts_lds[k] = w;
    }
  }
}

// How route_seg_small_kernel routes its tokens: 256-thread teams, softmax by
// one thread per token (at most kLaneE experts), or one wave per token with
// 2 / 4 / 8 experts per lane (E = 128 / 256 / 512).
enum SmallRoute : int { kTeams = 0, kLanes = 1, kWave2 = 2, kWave4 = 4, kWave8 = 8 };

// One workgroup of at least A threads and NB / 2 threads.  MODE 0: softmax
// routing, 1: grouped sigmoid routing, 2: ids/wts given.  Then the whole
// segmentation, one pair per thread (FEW: over at most kFewNB buckets).
// Latency bound (one workgroup): with the pairs ranked by ballots instead of
// each pair scanning the pairs before it, 1023 pairs over 514 buckets 36.0 ->
// 6.0 us; with one wave per token instead of four 256-thread teams in
// lockstep, T = 16 grouped sigmoid over 256 experts 35.5 -> 8.8 us (routing
// and segmentation).
template <int MODE, int RT, bool FEW>
__global__ __launch_bounds__(kSegThreads) void route_seg_small_kernel(SmallArgs a) {
  __shared__ int s_ids[kSmallMaxA];
  __shared__ float s_w[kSmallMaxA];
  __shared__ int s_start[kSmallMaxNB];
  __shared__ int wsum[3][kSegWaves];
  extern __shared__ __attribute__((aligned(16))) float small_lds[];
  const int tid = threadIdx.x, wv = tid / kWave;
  const int T = a.T, K = a.K, E = a.E, NS = a.NS;
  const int TK = T * K, A = TK + T * NS, NB = E + NS + 1, trash = E + NS;
  if constexpr (MODE < 2) {
    if constexpr (RT == kLanes) {
      for (int t = tid; t < T; t += blockDim.x)
        route_token_lane(a.logits + (long)t * E, E, K, a.renorm, a.ids + (long)t * K,
                         a.wts + (long)t * K, s_ids + t * K, s_w + t * K);
    } else if constexpr (RT == kTeams) {
      // blockDim / 256 teams of 256 threads route that many tokens at a time
      const int nteam = blockDim.x / 256, team = tid / 256, ttid = tid % 256;
      const int nc = (MODE == 1 ? a.n_group : (E + 31) / 32) * K;
      const RouteScratch s(small_lds + team * route_team_words(E, nc), E, nc);
      for (int t0 = 0; t0 < T; t0 += nteam) {
        const int t = t0 + team;
        const bool valid = t < T;
        route_token<MODE, 256>(a.logits + (long)t * E, a.bias, E, K, a.n_group, a.topk_group,
                               a.scale, a.renorm, s, ttid, valid, a.ids + (long)t * K,
                               a.wts + (long)t * K, s_ids + t * K, s_w + t * K);
      }
    } else {
      const int nw = blockDim.x / kWave;
      for (int t = wv; t < T; t += nw)
        tiny::route_token_wave<MODE, RT>(a.logits + (long)t * E, a.bias, K, a.n_group,
                                         a.topk_group, a.scale, a.renorm, tid % kWave,
                                         a.ids + (long)t * K, a.wts + (long)t * K,
                                         s_ids + t * K, s_w + t * K);
    }
    __syncthreads();   // the routing's scratch becomes the count table
  }
  uint16_t* wc = reinterpret_cast<uint16_t*>(small_lds);   // [waves holding pairs][nbp]
  const int nbp = seg_nbp(NB), half = nbp / 2, nw = (A + kWave - 1) / kWave;
  int b = -1;
  float w = 1.0f;
  if (tid < TK) {
    int e;
    if constexpr (MODE < 2) {
      e = s_ids[tid];
      w = s_w[tid];
    } else {
      e = a.ids[tid];
      w = a.wts[tid];
    }
    if (a.id_map && e >= 0 && e < E) e = a.id_map[e];
    b = (e < 0 || e >= E) ? trash : e;
    if (a.drop_zero && w == 0.0f) b = trash;
  } else if (tid < A) {
    b = E + (tid - TK) % NS;
  }
  if constexpr (FEW) {
    __shared__ FewSmem few;
    segment_few_buckets(a, few, b, w, A, TK, NB);
    return;
  }
  clear_counts(wc, nbp, nw);
  const bool valid = b >= 0;
  unsigned long long same;
  const int rank = wave_bucket_rank(b, valid, 32 - __builtin_clz(NB - 1), same);
  __syncthreads();
  if (valid && rank == 0) wc[wv * nbp + b] = (uint16_t)__popcll(same);
  __syncthreads();
  int c0 = 0, c1 = 0, s0, s1;
  if (tid < half) column_prefix(wc, nbp, nw, tid, c0, c1);
  const SegOut o{a.seg_start, a.active, a.n_active, a.tile_expert, a.tile_row0, a.n_tiles,
                 a.expert_tile_start, NB, a.bm, A};
  bucket_starts(o, tid, c0, c1, true, wsum, s0, s1);
  if (2 * tid < NB) s_start[2 * tid] = s0;
  if (2 * tid + 1 < NB) s_start[2 * tid + 1] = s1;
  __syncthreads();
  if (valid) {
    const int pos = s_start[b] + wc[wv * nbp + b] + rank;
    a.sorted_pair[pos] = tid;
    a.inv[tid] = pos;
    a.sorted_tok[pos] = tid < TK ? tid / K : (tid - TK) / NS;
    a.sorted_wts[pos] = w;
  }
}

// Tiny batches: the whole routing + segmentation in one workgroup
// (tiny::route_segment_block).
template <int MODE, int EPL>
__global__ __launch_bounds__(1024) void route_seg_tiny_kernel(SmallArgs a) {
  __shared__ __attribute__((aligned(16))) tiny::TinySmem g;
  tiny::route_segment_block<MODE, EPL>(a, g);
}

template <int MODE>
hipError_t launch_small(const SmallArgs& a, hipStream_t stream) {
  const int epl = tiny::tiny_epl(a, MODE);
  // one wave per token, and one thread per bucket start for the last pass
  const int nb_waves = (a.E + a.NS + 2 + kWave - 1) / kWave;
  int tiny_waves = a.T > 4 ? a.T : 4;
  if (tiny_waves < nb_waves) tiny_waves = nb_waves < 16 ? nb_waves : 16;
  const int tiny_threads = kWave * tiny_waves;
  if (epl != 0) {
    if constexpr (MODE == 2) {
      route_seg_tiny_kernel<2, 1><<<1, tiny_threads, 0, stream>>>(a);
    } else {
      if (epl == 2) route_seg_tiny_kernel<MODE, 2><<<1, tiny_threads, 0, stream>>>(a);
      else if (epl == 4) route_seg_tiny_kernel<MODE, 4><<<1, tiny_threads, 0, stream>>>(a);
      else route_seg_tiny_kernel<MODE, 8><<<1, tiny_threads, 0, stream>>>(a);
    }
    return hipSuccess;
  }
  const int A = a.T * a.K + a.T * a.NS, nbp = seg_nbp(a.E + a.NS + 1);
  // threads of the segmentation: one pair and two buckets each
  int threads = A > nbp / 2 ? A : nbp / 2;
  const size_t table = (size_t)((A + kWave - 1) / kWave) * nbp * sizeof(uint16_t);
  auto launch = [&](auto rt_tag, int route_threads, size_t route_lds) {
    if (threads < route_threads) threads = route_threads;
    threads = (threads + kWave - 1) / kWave * kWave;
    // team routing: whole teams only
    if (decltype(rt_tag)::value == kTeams && MODE < 2) threads = (threads + 255) / 256 * 256;
    const size_t teams = decltype(rt_tag)::value == kTeams && MODE < 2 ? threads / 256 : 1;
    const size_t lds = teams * route_lds > table ? teams * route_lds : table;
    constexpr int RT = decltype(rt_tag)::value;
    if constexpr (RT < kWave2) {   // the wave routers' E is past kFewNB
      if (a.E + a.NS + 1 <= kFewNB) {
        route_seg_small_kernel<MODE, RT, true><<<1, threads, lds, stream>>>(a);
        return;
      }
    }
    route_seg_small_kernel<MODE, RT, false><<<1, threads, lds, stream>>>(a);
  };
  using Lanes = std::integral_constant<int, kLanes>;
  using Teams = std::integral_constant<int, kTeams>;
  if constexpr (MODE == 2) {
    launch(Teams{}, kWave, 0);
  } else {
    const int wepl = tiny::wave_epl(MODE, a.E, a.n_group, a.renorm, a.logits, a.bias);
    if (MODE == 0 && a.E <= kLaneE && a.K <= kLaneK) {
      // few experts: one thread per token, no routing barriers
      launch(Lanes{}, kWave, 0);
    } else if (wepl != 0) {
      const int rt = kWave * (a.T < kSegWaves ? a.T : kSegWaves);
      if (wepl == 2) launch(std::integral_constant<int, kWave2>{}, rt, 0);
      else if (wepl == 4) launch(std::integral_constant<int, kWave4>{}, rt, 0);
      else launch(std::integral_constant<int, kWave8>{}, rt, 0);
    } else {
      const int nc = (MODE == 1 ? a.n_group : (a.E + 31) / 32) * a.K;
      // one team for at most two tokens: fewer waves in lockstep through the barriers
      launch(Teams{}, a.T <= 2 ? 256 : 1024, route_team_words(a.E, nc) * sizeof(float));
    }
  }
  return hipSuccess;
}


}  // namespace
}  // namespace xtu

using namespace xtu;

extern "C" {

hipError_t xtu_route_softmax_topk(const float* logits, int T, int E, int K, int renormalize,
                                  int32_t* topk_ids, float* topk_weights, hipStream_t stream) {
  XTU_CHECK_ARG(T >= 0 && E > 0 && E <= 1024 && K > 0 && K <= 16 && K <= E);
  XTU_CHECK_ARG(T == 0 || (logits && topk_ids && topk_weights));
  if (T == 0) return hipSuccess;
  (void)hipGetLastError();
  if (const int epl = tiny::wave_epl(0, E, 1, renormalize, logits, nullptr)) {
    launch_route_wave<0>(epl, logits, nullptr, T, K, 1, 1, 1.0f, renormalize, topk_ids,
                         topk_weights, stream);
    return hipPeekAtLastError();
  }
  launch_route_teams<0>(logits, nullptr, T, E, K, 1, 1, 1.0f, renormalize, ((E + 31) / 32) * K,
                       topk_ids, topk_weights, stream);
  return hipPeekAtLastError();
}

hipError_t xtu_route_grouped_sigmoid(const float* logits, const float* bias, int T, int E,
                                     int n_group, int topk_group, int K, float routed_scaling,
                                     int renormalize, int32_t* topk_ids, float* topk_weights,
                                     hipStream_t stream) {
  XTU_CHECK_ARG(T >= 0 && E > 0 && E <= 1024 && K > 0 && K <= 16);
  XTU_CHECK_ARG(n_group > 0 && n_group <= 64 && E % n_group == 0);
  XTU_CHECK_ARG(topk_group > 0 && topk_group <= n_group && K <= topk_group * (E / n_group));
  XTU_CHECK_ARG(T == 0 || (logits && topk_ids && topk_weights));
  if (T == 0) return hipSuccess;
  (void)hipGetLastError();
  if (const int epl = tiny::wave_epl(1, E, n_group, renormalize, logits, bias)) {
    launch_route_wave<1>(epl, logits, bias, T, K, n_group, topk_group, routed_scaling,
                         renormalize, topk_ids, topk_weights, stream);
    return hipPeekAtLastError();
  }
  launch_route_teams<1>(logits, bias, T, E, K, n_group, topk_group, routed_scaling, renormalize,
                       n_group * K, topk_ids, topk_weights, stream);
  return hipPeekAtLastError();
}

// The counts of the blocks (at most kSegMaxBlocks; the bound grows with T,
// so a workspace sized for more tokens holds fewer), and never less than one
// row of counts per kSegBoundChunk pairs: xtu_segment_noalloc refuses the
// shapes whose bound passes its static scratch.
size_t xtu_segment_workspace_bytes(int T, int K, int E, int n_shared) {
  const long A = (long)T * K + (long)T * n_shared;
  const long NB = E + n_shared + 1;
  const long bound = (A + kSegBoundChunk - 1) / kSegBoundChunk;
  long nblocks = (A + kSegThreads - 1) / kSegThreads;
  if (nblocks > kSegMaxBlocks) nblocks = kSegMaxBlocks;
  const size_t b0 = (size_t)((bound > 0 ? bound : 1) * NB * sizeof(int32_t));
  const size_t b1 = (size_t)((nblocks > 0 ? nblocks : 1) * seg_nbp((int)NB) * sizeof(int32_t));
  return b0 > b1 ? b0 : b1;
}

int xtu_segment_max_tiles(int T, int K, int E, int n_shared, int bm) {
  const long A = (long)T * K + (long)T * n_shared;
  const long nb = E + n_shared;
  return (int)(A / bm + (A < nb ? A : nb) + 1);
}

}  // extern "C"

namespace xtu {
namespace {

// The two segmentation launches over a caller-supplied workspace of
// xtu_segment_workspace_bytes() bytes (every word written by seg_count_kernel
// before seg_place_kernel reads it, so it needs no clearing).  Latency bound:
// 45k pairs over 514 buckets 15.7 us, 74k over 258 16.9 us, 1.9k 11.4 us
// (4.7 of it the counts); a histogram, a one-block scan and a scatter of
// 4096-pair blocks, 16 rounds of four barriers each, took 43.2, 46.6 and
// 23.3 us.
hipError_t segment_impl(const int32_t* topk_ids, const float* topk_weights,
                        const int32_t* id_map, int T, int K, int E, int n_shared, int drop_zero,
                        int bm, void* workspace, int32_t* sorted_pair, int32_t* sorted_tok,
                        float* sorted_wts, int32_t* inv, int32_t* seg_start, int32_t* active,
                        int32_t* n_active, int32_t* tile_expert, int32_t* tile_row0,
                        int32_t* n_tiles, int32_t* expert_tile_start, hipStream_t stream) {
  XTU_CHECK_ARG(T >= 0 && K >= 0 && E > 0 && n_shared >= 0 && bm > 0);
  const int NB = E + n_shared + 1;
  XTU_CHECK_ARG(NB <= 2048);
  const long A = (long)T * K + (long)T * n_shared;
  XTU_CHECK_ARG(A < (1l << 30));
  XTU_CHECK_ARG(workspace && seg_start && active && n_active && tile_expert && tile_row0 &&
                n_tiles && expert_tile_start);
  XTU_CHECK_ARG(A == 0 || (sorted_pair && sorted_tok && sorted_wts && inv));
  XTU_CHECK_ARG(T * K == 0 || (topk_ids && topk_weights));
  const int rounds = (int)((A + (long)kSegThreads * kSegMaxBlocks - 1) /
                           ((long)kSegThreads * kSegMaxBlocks));
  const long chunk = (long)(rounds > 0 ? rounds : 1) * kSegThreads;
  const int nblocks = (int)((A + chunk - 1) / chunk);
  const int nbp = seg_nbp(NB);
  SegArgs a{topk_ids, topk_weights, id_map, T, K, E, n_shared, drop_zero, (int)A, NB, rounds};
  SegOut o{seg_start, active, n_active, tile_expert, tile_row0, n_tiles, expert_tile_start, NB,
           bm, (int)A};
  int32_t* bcnt = (int32_t*)workspace;
  (void)hipGetLastError();
  if (nblocks > 0) seg_count_kernel<<<nblocks, kSegThreads, nbp * sizeof(int), stream>>>(a, bcnt);
  const size_t table = (size_t)kSegWaves * nbp * sizeof(uint16_t);   // >= the totals' nbp words
  seg_place_kernel<<<nblocks > 0 ? nblocks : 1, kSegThreads, nbp * sizeof(int) + table, stream>>>(
      a, o, bcnt, nblocks, sorted_pair, sorted_tok, sorted_wts, inv);
  return hipPeekAtLastError();
}

// Device address of `scratch` on the current device, looked up once per
// device (hipGetSymbolAddress with that device current) and kept.
constexpr int kMaxDevices = 64;
std::mutex g_scratch_mu;
void* g_scratch_ptr[kMaxDevices] = {};

hipError_t scratch_address(void** out) {
  int dev = -1;
  hipError_t e = hipGetDevice(&dev);
  if (e != hipSuccess) return e;
  if (dev < 0 || dev >= kMaxDevices) return hipErrorInvalidDevice;
  std::lock_guard<std::mutex> lk(g_scratch_mu);
  if (!g_scratch_ptr[dev]) {
    void* p = nullptr;
    e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
    if (e != hipSuccess) return e;
    g_scratch_ptr[dev] = p;
  }
  *out = g_scratch_ptr[dev];
  return hipSuccess;
}

}  // namespace
}  // namespace xtu

extern "C" {

hipError_t xtu_segment(const int32_t* topk_ids, const float* topk_weights,
                       const int32_t* id_map, int T, int K, int E, int n_shared, int drop_zero,
                       int bm, void* workspace, int32_t* sorted_pair, int32_t* sorted_tok,
                       float* sorted_wts, int32_t* inv, int32_t* seg_start, int32_t* active,
                       int32_t* n_active, int32_t* tile_expert, int32_t* tile_row0,
                       int32_t* n_tiles, int32_t* expert_tile_start, hipStream_t stream) {
  return segment_impl(topk_ids, topk_weights, id_map, T, K, E, n_shared, drop_zero, bm,
                      workspace, sorted_pair, sorted_tok, sorted_wts, inv, seg_start, active,
                      n_active, tile_expert, tile_row0, n_tiles, expert_tile_start, stream);
}

hipError_t xtu_segment_noalloc(const int32_t* topk_ids, const float* topk_weights,
                               const int32_t* id_map, int T, int K, int E, int n_shared,
                               int drop_zero, int bm, int32_t* sorted_pair, int32_t* sorted_tok,
                               float* sorted_wts, int32_t* inv, int32_t* seg_start,
                               int32_t* active, int32_t* n_active, int32_t* tile_expert,
                               int32_t* tile_row0, int32_t* n_tiles, int32_t* expert_tile_start,
                               hipStream_t stream) {
  XTU_CHECK_ARG(T >= 0 && K >= 0 && E > 0 && n_shared >= 0);
  const size_t need = xtu_segment_workspace_bytes(T, K, E, n_shared);
  if (need > kNoAllocScratchBytes) {
    fprintf(stderr,
            "xtu_segment_noalloc: T=%d K=%d E=%d n_shared=%d needs %zu bytes of workspace, more "
            "than the %zu-byte static scratch; use xtu_segment with a workspace\n",
            T, K, E, n_shared, need, kNoAllocScratchBytes);
    return hipErrorInvalidValue;
  }
  void* ws = nullptr;
  const hipError_t e = scratch_address(&ws);
  if (e != hipSuccess) return e;
  return segment_impl(topk_ids, topk_weights, id_map, T, K, E, n_shared, drop_zero, bm, ws,
                      sorted_pair, sorted_tok, sorted_wts, inv, seg_start, active, n_active,
                      tile_expert, tile_row0, n_tiles, expert_tile_start, stream);
}

int xtu_route_segment_small_max_pairs(void) { return kSmallMaxA; }

hipError_t xtu_route_segment_small(int mode, const float* logits, const float* bias,
                                   int32_t* topk_ids, float* topk_weights, int T, int E, int K,
                                   int n_group, int topk_group, float routed_scaling,
                                   int renormalize, const int32_t* id_map, int n_shared,
                                   int drop_zero, int bm, int32_t* sorted_pair,
                                   int32_t* sorted_tok, float* sorted_wts, int32_t* inv,
                                   int32_t* seg_start, int32_t* active, int32_t* n_active,
                                   int32_t* tile_expert, int32_t* tile_row0, int32_t* n_tiles,
                                   int32_t* expert_tile_start, hipStream_t stream) {
  XTU_CHECK_ARG(mode >= 0 && mode <= 2 && T >= 0 && E > 0 && E <= 1024 && K > 0 && K <= 16 &&
                K <= E && n_shared >= 0 && bm > 0);
  XTU_CHECK_ARG((long)T * K + (long)T * n_shared <= kSmallMaxA && E + n_shared + 1 <= kSmallMaxNB);
  if (mode == 1)
    XTU_CHECK_ARG(n_group > 0 && n_group <= 64 && E % n_group == 0 && topk_group > 0 &&
                  topk_group <= n_group && K <= topk_group * (E / n_group));
  XTU_CHECK_ARG(topk_ids && topk_weights && (mode == 2 || T == 0 || logits));
  XTU_CHECK_ARG(sorted_pair && sorted_tok && sorted_wts && inv && seg_start && active &&
                n_active && tile_expert && tile_row0 && n_tiles && expert_tile_start);
  if (mode < 2 && T == 0) mode = 2;   // nothing to route: segment the empty batch
  SmallArgs a{logits, bias, topk_ids, topk_weights, id_map, T, K, E, n_group, topk_group,
              renormalize, n_shared, drop_zero, bm, routed_scaling, sorted_pair, sorted_tok, inv,
              seg_start, active, n_active, sorted_wts, tile_expert, tile_row0, n_tiles,
              expert_tile_start};
  (void)hipGetLastError();
  hipError_t err;
  if (mode == 0) err = launch_small<0>(a, stream);
  else if (mode == 1) err = launch_small<1>(a, stream);
  else err = launch_small<2>(a, stream);
  return err != hipSuccess ? err : hipPeekAtLastError();
}

}  // extern "C"
