// Grouped expert GEMMs for batches that give an expert a handful of rows
// (mid-size decode batches up to prompts): the layer is a weight stream, as at
// decode, but an expert's rows no longer fit one MFMA tile.
//
// What bounds it: HBM, until an expert holds some tens of rows.  1 KiB of
// fp4 weights is four 16x16x32 MFMAs per 16-row tile and 16 conversions (48
// VALU operations more for NVFP4's scale multiply), against ~400 cycles of a
// SIMD's share of the memory rate, so a few row tiles hide behind the stream
// as long as enough weight bytes are in flight.  Hence:
//   * a workgroup of four waves takes one tile of one expert's rows and
//     4 x PW 16-row weight panels; each wave streams its own PW panels from
//     the P16 layout straight into registers, four super-blocks per panel
//     ahead (nontemporal, never through LDS), and re-issues a register set as
//     soon as it is consumed, so 4 x PW KiB per wave stay in flight over the
//     barriers of the row stage;
//   * the tile's rows go through a double-buffered LDS stage in K chunks of a
//     round (four super-blocks) or a part of one, one barrier per chunk; a
//     chunk's rows are loaded one chunk ahead, in front of that chunk's
//     weights, so the in-order wait for them does not wait for weights issued
//     later.  Rows past the tile read as zero without touching memory;
//   * the K loop is specialised on the number of 16-row tiles, and the last
//     round (nothing left to issue) is peeled, so every wait count is exact.
//
// Products are exact in every format (bf16 rows against e2m1 x scale, e4m3
// or bf16 weights in bf16, fp32 accumulation; FP8's block scale multiplies
// the fp32 sum of its 128 k).
//
// Measured (MI355X), gate/up + down of one layer against the kernels these
// batches took before (prefill tiles of 128 rows with a barrier and one
// super-block of weights in flight per step; one workgroup per 16 gate
// columns re-reading its rows at decode):
//   Qwen3-Next NVFP4 T = 93     290 -> 161 us
//   Qwen3-Next MXFP4 T = 300    252 -> 160
//   DeepSeek-V3 MXFP4 T = 209  1204 -> 965 (6.2 TB/s)
//   DeepSeek-V3 MXFP4 T = 16 gate/up 366 -> 233 (6.9 TB/s)
//   DeepSeek-V3 FP8 T = 32      1030 (7.0 TB/s)
//   128-expert FP8 T = 64       132 -> 91
//   Qwen3-Next NVFP4 T = 4096   637 -> 500 (with the branch-free scales)
//   Qwen3-Next int8 T = 1000    339 -> 230 (whole layer 367 -> 255)
// Past some tens of rows per expert the LDS reads of the rows, the
// dequantisation and the MFMAs share the time about evenly (NVFP4 T = 4096:
// LDS 40%, VALU 35%, MFMA 31% busy at two waves per SIMD); int8 is bound by
// the expansion's VALU work (68% busy at T = 1000).
#include <type_traits>

#include "weight_format.hpp"

namespace xtu {
namespace {

// MXFP4 weights against int8 rows (the ALIGN rule of int8.hip): the same P16
// planes as MXFP4, expanded in registers to w8' = 2 e2m1 << (b - emin), exact
// int32 sums.  Reading the codes instead of the expanded int8 planes halves
// the bytes of the stream.
constexpr int kMXI8 = 4;
constexpr int kI8Marked = 0xFF;   // emin of a row the fp32 fallback computes: int8 weights 0
template <int FMT>
struct SFmt : WFmt<FMT> {};
template <>
struct SFmt<kMXI8> : WFmt<kMXFP4> {};

constexpr int kBufFlags = 0x00020000;   // raw buffer resource, dword 3
constexpr int kNt = 2;                  // nontemporal
constexpr int kDead = (int)0x80000000;  // offset past every buffer range: reads as zero

struct StreamArgs {
  const uint8_t* a;           // gate/up: x [T][K]; down: act [A][K] (bf16, or int8 rows)
  const int32_t* sorted_tok;  // gate/up row gather
  const uint8_t* w;
  const uint8_t* s;
  const float* gs;
  const int32_t* seg_start;
  const int32_t* tile_expert;
  const int32_t* tile_row0;
  const int32_t* tile_lo;     // m-tile range [*tile_lo, *tile_hi) of the tile list
  const int32_t* tile_hi;
  const int32_t* slot_map;    // expert -> weight slot (null: identity)
  void* out;                  // gate/up: act bf16 [A][I]; down: y fp32 [A][H]
  int H, I, bm;
  uint32_t a_bytes;           // gate/up: bytes of x
  long w_estride, s_estride;
  float limit, alpha, beta;
  const int32_t* pair_of;     // down: null = y row per sorted position; else y row
                              // pair_of[position] (the flat pair index)
  const int32_t* crow;        // int8: exponent of each a row
  const uint8_t* emin;        // int8: smallest e8m0 byte of each weight row [slot][N]
};

constexpr int kNW = 4;   // waves per workgroup
constexpr int kPD = 4;   // super-blocks per round: weights in flight per panel

// LDS row stage of NR row tiles: chunks per round (so that the stage of more
// rows stays small enough for two to four workgroups per CU), k per chunk,
// and bytes of one buffer (rows padded by 16 bytes: the 16 rows a wave
// reads at once start in different banks).
template <int FMT, int NR>
constexpr int chunks() {
  if (FMT == kMXI8) return NR <= 2 ? 1 : NR <= 4 ? 2 : 4;
  constexpr bool fp4 = FMT == kMXFP4 || FMT == kNVFP4;
  return NR == 1 ? 1 : NR == 2 ? (fp4 ? 2 : 1) : (fp4 ? 4 : 2);
}
template <int FMT, int NR>
constexpr int chunk_k() { return kPD * SFmt<FMT>::kSB / chunks<FMT, NR>(); }
template <int FMT>
constexpr int elem_bytes() { return FMT == kMXI8 ? 1 : 2; }
template <int FMT, int NR>
constexpr int stage_bytes() { return NR * 16 * (chunk_k<FMT, NR>() * elem_bytes<FMT>() + 16); }
template <int FMT, int MAXNR>
constexpr int stage_max() {
  const int m1 = stage_bytes<FMT, 1>(), m2 = stage_bytes<FMT, 2>(), mm = stage_bytes<FMT, MAXNR>();
  const int m = MAXNR >= 2 && m2 > m1 ? m2 : m1;
  return mm > m ? mm : m;
}

// Raw scales of one panel for one round.
template <int FMT>
struct RoundScale {
  uint32_t v[FMT == kNVFP4 ? 2 : 1];
};

// Byte tables of w8' << d for the codes 0..7 (pos) and 8..15 (neg), d = b - emin
// (0..3 in an unmarked row: the shifted magnitudes stay in their bytes; the
// negatives' shifted-in carries are masked off).  A marked row's are zero.
struct I8Table {
  uint32_t plo, phi, nlo, nhi;
};

__device__ __forceinline__ I8Table i8_table(uint32_t b, int em) {
  const uint32_t d = ((b & 0xffu) - (uint32_t)em) & 3u;
  const uint32_t keep = em == kI8Marked ? 0u : 0x01010101u * ((0xffu << d) & 0xffu);
  I8Table t;
  t.plo = (0x03020100u << d) & keep;   // 0, 1, 2, 3
  t.phi = (0x0c080604u << d) & keep;   // 4, 6, 8, 12
  t.nlo = (0xfdfeff00u << d) & keep;
  t.nhi = (0xf4f8fafcu << d) & keep;
  return t;
}

// 16 codes (two dwords, low nibble first) -> 16 int8, each dword's even codes
// first: look the magnitude up in both tables and select by the sign bit.
__device__ __forceinline__ uint32_t i8_select(const I8Table& t, uint32_t idx, uint32_t sign) {
  const uint32_t pos = __builtin_amdgcn_perm(t.phi, t.plo, idx);
  const uint32_t neg = __builtin_amdgcn_perm(t.nhi, t.nlo, idx);
  const uint32_t m = (sign << 8) - sign;   // 0xff in the bytes of negative codes
  return (neg & m) | (pos & ~m);
}

__device__ __forceinline__ i32x4_t i8_expand(const I8Table& t, uint32_t w0, uint32_t w1) {
  return i32x4_t{(int)i8_select(t, w0 & 0x07070707u, (w0 >> 3) & 0x01010101u),
                 (int)i8_select(t, (w0 >> 4) & 0x07070707u, (w0 >> 7) & 0x01010101u),
                 (int)i8_select(t, w1 & 0x07070707u, (w1 >> 3) & 0x01010101u),
                 (int)i8_select(t, (w1 >> 4) & 0x07070707u, (w1 >> 7) & 0x01010101u)};
}

template <int FMT, bool GU, int PW, int MAXNR, int WPS>
__global__ __launch_bounds__(64 * kNW, WPS) void stream_gemm_kernel(StreamArgs a) {
  using F = SFmt<FMT>;
  constexpr bool I8 = FMT == kMXI8;
  constexpr int ES = elem_bytes<FMT>();    // bytes per A element
  constexpr int PD = kPD;
  constexpr int KR = PD * F::kSB;          // k per round
  constexpr int kGK = 16 / ES;             // k of a lane's A piece of one MFMA
  constexpr int kG = F::kCK / kGK;         // MFMA k groups per super-block
  constexpr int kThreads = 64 * kNW;
  constexpr int NS = FMT == kFP8 ? (GU ? 2 : 1) : PW;   // scale streams
  // epilogue: output columns of a wave, staged row pitch (16-bit units)
  constexpr int NC = GU ? PW / 2 * 16 : PW * 16;
  constexpr int kPitch = GU ? NC + 8 : (NC + 4) * 2;
  constexpr int kStage = 2 * stage_max<FMT, MAXNR>(), kEpi = kNW * 16 * kPitch * 2;
  __shared__ __attribute__((aligned(16))) uint8_t As[kStage > kEpi ? kStage : kEpi];

  // ---- work item
  const int nbn = GU ? a.I / (8 * kNW * PW) : a.H / (16 * kNW * PW);
  const int lo = a.tile_lo[0];
  const int total = (a.tile_hi[0] - lo) * nbn;
  const int per = (total + 7) / 8;
  const int idx = blockIdx.x / 8;
  if (idx >= per) return;
  const int item = (blockIdx.x % 8) * per + idx;
  if (item >= total) return;
  const int tile = lo + item / nbn, nb = item % nbn;
  const int e = a.tile_expert[tile];
  const int ws = a.slot_map ? a.slot_map[e] : e;
  const int row0 = a.tile_row0[tile];
  const int rows = min(a.bm, a.seg_start[e + 1] - row0);
  const int K = GU ? a.H : a.I;
  const int nsteps = K / F::kSB;
  const int nrounds = (nsteps + PD - 1) / PD;
  const int tid = threadIdx.x;
  const int wv = __builtin_amdgcn_readfirstlane(tid / 64);
  const int lane = tid % 64;
  const int q = lane / 16, r16 = lane % 16;

  // ---- this wave's panels: gate/up: [0, PW/2) gate rows, [PW/2, PW) the up
  // rows of the same columns; down: PW consecutive panels
  int pan[PW];
#pragma unroll
  for (int p = 0; p < PW; ++p) {
    if (GU) pan[p] = (p < PW / 2 ? 0 : a.I / 16) + (nb * kNW + wv) * (PW / 2) + p % (PW / 2);
    else pan[p] = (nb * kNW + wv) * PW + p;
  }
  const __amdgpu_buffer_rsrc_t rw = __builtin_amdgcn_make_buffer_rsrc(
      (void*)(a.w + (long)ws * a.w_estride), 0, (int)a.w_estride, kBufFlags);
  const __amdgpu_buffer_rsrc_t rs = __builtin_amdgcn_make_buffer_rsrc(
      (void*)(a.s ? a.s + (long)ws * a.s_estride : a.w), 0, (int)a.s_estride, kBufFlags);
  const int sgroups = (int)scale_groups(K, F::kUG);

  u32x4_t w[PD][PW];
  RoundScale<FMT> sc[NS], sn[NS];
  // weights of step s into register set j (a step past K reads nothing)
  auto issue = [&](int s, int j) {
    const int off = s < nsteps ? lane * 16 : kDead;
#pragma unroll
    for (int p = 0; p < PW; ++p)
      w[j][p] = __builtin_bit_cast(u32x4_t, __builtin_amdgcn_raw_buffer_load_b128(
                                                rw, off, (pan[p] * nsteps + s) * 1024, kNt));
  };
  // scales of round r
  auto issue_scales = [&](int r, RoundScale<FMT> (&d)[NS]) {
    if constexpr (F::kSBY > 0) {
      const int s0 = r * PD, g = s0 / F::kUG, ob = (s0 % F::kUG) * F::kSBY;
#pragma unroll
      for (int p = 0; p < PW; ++p) {
        const int so = (pan[p] * sgroups + g) * 1024 + ob;
        d[p].v[0] = __builtin_amdgcn_raw_buffer_load_b32(rs, lane * 16, so, 0);
        if constexpr (FMT == kNVFP4)
          d[p].v[1] = __builtin_amdgcn_raw_buffer_load_b32(rs, lane * 16 + 4, so, 0);
      }
    } else if constexpr (FMT == kFP8) {   // lane l: the scale of the round's 128-k block l
      const int kb = r * (KR / 128) + lane % (KR / 128);
#pragma unroll
      for (int h = 0; h < NS; ++h) {
        const int rb = pan[h * (PW / 2)] / 8;
        d[h].v[0] = __builtin_amdgcn_raw_buffer_load_b32(
            rs, kb < K / 128 ? (rb * (K / 128) + kb) * 4 : kDead, 0, 0);
      }
    }
  };
  int em[PW];   // int8: emin of the lane's weight row of each panel
#pragma unroll
  for (int p = 0; p < PW; ++p)
    em[p] = I8 ? a.emin[(long)ws * (GU ? 2 * a.I : a.H) + pan[p] * 16 + r16] : 0;
  issue_scales(0, sc);
#pragma unroll
  for (int j = 0; j < PD; ++j) issue(j, j);
  __builtin_amdgcn_sched_barrier(0);

  auto run = [&](auto nr_tag) {
    constexpr int NR = decltype(nr_tag)::value;
    constexpr int KC = chunk_k<FMT, NR>(), SUB = KR / KC, CS = PD / SUB;
    constexpr int kLD = KC * ES + 16;                         // row pitch in bytes
    constexpr int ppr = KC * ES / 16;                         // 16-byte pieces per row
    constexpr int kPieces = NR * 16 * ppr;
    constexpr int NP = (kPieces + kThreads - 1) / kThreads;   // pieces per thread
    // ---- A pieces of this thread: byte offset of (row, column) at k = 0
    const __amdgpu_buffer_rsrc_t ra =
        GU ? __builtin_amdgcn_make_buffer_rsrc((void*)a.a, 0, (int)a.a_bytes, kBufFlags)
           : __builtin_amdgcn_make_buffer_rsrc((void*)(a.a + (long)row0 * K * ES), 0,
                                               rows * K * ES, kBufFlags);
    int aoff[NP];
#pragma unroll
    for (int i = 0; i < NP; ++i) {
      const int c = i * kThreads + tid, r = c / ppr, col = c % ppr;
      const int src = GU ? a.sorted_tok[row0 + min(r, rows - 1)] : r;
      aoff[i] = r < rows ? src * K * ES + col * 16 : kDead;
    }
    u32x4_t ar[NP];
    // a chunk that runs past K (K is a multiple of 128) loads zeros there
    auto load_a = [&](int k0) {
#pragma unroll
      for (int i = 0; i < NP; ++i) {
        const int kp = k0 + ((i * kThreads + tid) % ppr) * (16 / ES);
        ar[i] = __builtin_bit_cast(u32x4_t, __builtin_amdgcn_raw_buffer_load_b128(
                                                ra, kp < K ? aoff[i] : kDead, k0 * ES, 0));
      }
    };
    auto store_a = [&](int buf) {
#pragma unroll
      for (int i = 0; i < NP; ++i) {
        const int c = i * kThreads + tid;
        u32x4_t v = ar[i];
        if constexpr (I8) {   // k order of the expanded codes: even k, then odd k, of each 8
          v = u32x4_t{__builtin_amdgcn_perm(ar[i][1], ar[i][0], 0x06040200u),
                      __builtin_amdgcn_perm(ar[i][1], ar[i][0], 0x07050301u),
                      __builtin_amdgcn_perm(ar[i][3], ar[i][2], 0x06040200u),
                      __builtin_amdgcn_perm(ar[i][3], ar[i][2], 0x07050301u)};
        }
        if (kPieces % kThreads == 0 || c < kPieces)
          *reinterpret_cast<u32x4_t*>(As + buf * stage_bytes<FMT, NR>() + (c / ppr) * kLD +
                                      (c % ppr) * 16) = v;
      }
    };

    using acc_t = std::conditional_t<I8, i32x4_t, f32x4_t>;
    acc_t acc[NR][PW];
    f32x4_t part[FMT == kFP8 ? NR : 1][FMT == kFP8 ? PW : 1];
#pragma unroll
    for (int m = 0; m < NR; ++m)
#pragma unroll
      for (int p = 0; p < PW; ++p) acc[m][p] = acc_t{0, 0, 0, 0};

    auto compute = [&](int j, const uint8_t* ab) {
      // ab: this lane's row r16, k = q * kCK of the step
      I8Table tab[I8 ? PW : 1];
      if constexpr (I8) {
#pragma unroll
        for (int p = 0; p < PW; ++p) tab[p] = i8_table(sc[p].v[0] >> (8 * j), em[p]);
      }
#pragma unroll
      for (int g = 0; g < kG; ++g) {
        if constexpr (I8) {
          i32x4_t bi[PW];
#pragma unroll
          for (int p = 0; p < PW; ++p)
            bi[p] = i8_expand(tab[p], w[j][p][2 * g], w[j][p][2 * g + 1]);
#pragma unroll
          for (int m = 0; m < NR; ++m) {
            const i32x4_t av = *reinterpret_cast<const i32x4_t*>(ab + m * 16 * kLD + 16 * g);
#pragma unroll
            for (int p = 0; p < PW; ++p)
              acc[m][p] = __builtin_amdgcn_mfma_i32_16x16x64_i8(av, bi[p], acc[m][p], 0, 0, 0);
          }
        } else {
          bf16x8_t bv[PW];
#pragma unroll
          for (int p = 0; p < PW; ++p) {
            uint32_t o[4];
            if constexpr (FMT == kMXFP4) {
              fp4x8_to_bf16(w[j][p][g], e8m0_to_f32(sc[p].v[0] >> (8 * j)), o);
              bv[p] = as_bf16x8(o[0], o[1], o[2], o[3]);
            } else if constexpr (FMT == kNVFP4) {
              const uint32_t raw = sc[p].v[j / 2] >> (16 * (j % 2) + (g < 2 ? 0 : 8));
              fp4x8_to_bf16_mul(w[j][p][g], e4m3_to_f32(raw & 0xffu), o);
              bv[p] = as_bf16x8(o[0], o[1], o[2], o[3]);
            } else if constexpr (FMT == kFP8) {
#pragma unroll
              for (int h = 0; h < 2; ++h) {
                const uint32_t d = w[j][p][2 * g + h];
                o[2 * h] = __builtin_bit_cast(
                    uint32_t, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(d, 1.0f, false));
                o[2 * h + 1] = __builtin_bit_cast(
                    uint32_t, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(d, 1.0f, true));
              }
              bv[p] = as_bf16x8(o[0], o[1], o[2], o[3]);
            } else {
              bv[p] = as_bf16x8(w[j][p]);
            }
          }
#pragma unroll
          for (int m = 0; m < NR; ++m) {
            const bf16x8_t av =
                as_bf16x8(*reinterpret_cast<const u32x4_t*>(ab + m * 16 * kLD + 16 * g));
#pragma unroll
            for (int p = 0; p < PW; ++p) {
              if constexpr (FMT == kFP8) {
                const f32x4_t c0 =
                    (j % 2 == 0 && g == 0) ? f32x4_t{0.f, 0.f, 0.f, 0.f} : part[m][p];
                part[m][p] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(av, bv[p], c0, 0, 0, 0);
              } else {
                acc[m][p] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(av, bv[p], acc[m][p], 0, 0, 0);
              }
            }
          }
        }
      }
      if constexpr (FMT == kFP8) {
        if (j % 2 == 1) {
#pragma unroll
          for (int p = 0; p < PW; ++p) {
            const float bs = __builtin_bit_cast(
                float, __builtin_amdgcn_readlane((int)sc[GU ? p / (PW / 2) : 0].v[0], j / 2));
#pragma unroll
            for (int m = 0; m < NR; ++m)
#pragma unroll
              for (int i = 0; i < 4; ++i)
                acc[m][p][i] = __builtin_fmaf(bs, part[m][p][i], acc[m][p][i]);
          }
        }
      }
    };

    const int afrag = r16 * kLD + q * F::kCK * ES;
    // one round; MORE: rows and weights of the next one are issued behind it
    auto round = [&](int r, auto more_tag) {
      constexpr bool MORE = decltype(more_tag)::value;
#pragma unroll
      for (int c = 0; c < SUB; ++c) {
        const int chunk = r * SUB + c;
        constexpr bool kTail = !MORE;
        const bool next = !kTail || c + 1 < SUB;   // compile-time per unrolled c
        if (next) load_a((chunk + 1) * KC);
        if (MORE && c == 0) issue_scales(r + 1, sn);
        __builtin_amdgcn_sched_barrier(0);
        const uint8_t* ab = As + (chunk & 1) * stage_bytes<FMT, NR>() + afrag;
#pragma unroll
        for (int jj = 0; jj < CS; ++jj) {
          const int j = c * CS + jj;
          if (MORE || r * PD + j < nsteps) compute(j, ab + jj * F::kSB * ES);
          if (MORE) {
            issue((r + 1) * PD + j, j);
            __builtin_amdgcn_sched_barrier(0);
          }
        }
        if (next) {
          store_a((chunk + 1) & 1);
          __syncthreads();
        }
      }
      if (MORE) {
#pragma unroll
        for (int h = 0; h < NS; ++h) sc[h] = sn[h];
      }
    };
    load_a(0);
    store_a(0);
    __syncthreads();
    for (int r = 0; r + 1 < nrounds; ++r) round(r, std::true_type{});
    round(nrounds - 1, std::false_type{});

    // NVFP4 second-level scales: [slot][2] (gate, up) for gate/up, [slot] for down
    float gsv = 1.0f, gsu = 1.0f;
    if constexpr (FMT == kNVFP4) {
      if (a.gs) {
        gsv = GU ? a.gs[2 * ws] : a.gs[ws];
        gsu = GU ? a.gs[2 * ws + 1] : gsv;
      }
    }
    // the 16x16 results (column lane % 16, rows 4 (lane / 16) + i) go through
    // the wave's own LDS region and leave as 16-byte row pieces
    __syncthreads();
    uint16_t* stage = reinterpret_cast<uint16_t*>(As) + wv * (16 * kPitch);
    // value of accumulator i of (m, p): int8 sums by their row and column powers of two
    int cr[4];
    auto row_exps = [&](int m) {
      if constexpr (I8) {
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const int r = min(m * 16 + 4 * q + i, rows - 1);
          cr[i] = a.crow[GU ? a.sorted_tok[row0 + r] : row0 + r];
        }
      }
    };
    auto value = [&](int m, int p, int i) {
      if constexpr (I8) return (float)acc[m][p][i] * ldexpf(1.0f, em[p] - 128 + cr[i]);
      else return acc[m][p][i];
    };
    const long col0 = (long)pan[0] * 16;
#pragma unroll
    for (int m = 0; m < NR; ++m) {
      if (m * 16 >= rows) break;
      row_exps(m);
      if constexpr (GU) {
        uint16_t* act = reinterpret_cast<uint16_t*>(a.out);
#pragma unroll
        for (int p = 0; p < PW / 2; ++p)
#pragma unroll
          for (int i = 0; i < 4; ++i) {
            const float g = value(m, p, i) * gsv, u = value(m, p + PW / 2, i) * gsu;
            stage[(4 * q + i) * kPitch + 16 * p + r16] =
                f32_to_bf16(silu_gate(g, u, a.limit, a.alpha, a.beta));
          }
        __builtin_amdgcn_wave_barrier();
        for (int j = lane; j < 16 * (NC / 8); j += 64) {
          const int rr = j / (NC / 8), c8 = j % (NC / 8);
          if (m * 16 + rr < rows)
            *reinterpret_cast<u32x4_t*>(act + (long)(row0 + m * 16 + rr) * a.I + col0 + 8 * c8) =
                *reinterpret_cast<const u32x4_t*>(stage + rr * kPitch + 8 * c8);
        }
        __builtin_amdgcn_wave_barrier();
      } else {
        float* fst = reinterpret_cast<float*>(stage);
        float* y = reinterpret_cast<float*>(a.out);
#pragma unroll
        for (int p = 0; p < PW; ++p)
#pragma unroll
          for (int i = 0; i < 4; ++i)
            fst[(4 * q + i) * (NC + 4) + 16 * p + r16] = value(m, p, i) * gsv;
        __builtin_amdgcn_wave_barrier();
        for (int j = lane; j < 16 * (NC / 4); j += 64) {
          const int rr = j / (NC / 4), c4 = j % (NC / 4);
          if (m * 16 + rr < rows) {
            const int pos = row0 + m * 16 + rr;
            const long yr = a.pair_of ? a.pair_of[pos] : pos;
            *reinterpret_cast<f32x4_t*>(y + yr * a.H + col0 + 4 * c4) =
                *reinterpret_cast<const f32x4_t*>(fst + rr * (NC + 4) + 4 * c4);
          }
        }
        __builtin_amdgcn_wave_barrier();
      }
    }
  };
  if constexpr (MAXNR == 8) {
    if (rows > 96) return run(std::integral_constant<int, 8>{});
    if (rows > 64) return run(std::integral_constant<int, 6>{});
  }
  if constexpr (MAXNR >= 4) {
    if (rows > 48) return run(std::integral_constant<int, 4>{});
    if (rows > 32) return run(std::integral_constant<int, 3>{});
    if (rows > 16) return run(std::integral_constant<int, 2>{});
  }
  run(std::integral_constant<int, 1>{});
}

template <int FMT, bool GU, int PW, int MAXNR, int WPS>
hipError_t launch_shape(const StreamArgs& a, int max_tiles, hipStream_t stream) {
  const long items = (long)max_tiles * (GU ? a.I / (8 * kNW * PW) : a.H / (16 * kNW * PW));
  const long grid = (items + 7) / 8 * 8;
  if (grid >= (1L << 31)) return hipErrorInvalidValue;
  stream_gemm_kernel<FMT, GU, PW, MAXNR, WPS><<<dim3((unsigned)grid), 64 * kNW, 0, stream>>>(a);
  return hipPeekAtLastError();
}

// Rows per tile at most: MXFP4 and FP8 batches with more rows per expert run
// on the scaled-MFMA kernels instead.
constexpr int max_bm(int fmt) { return fmt == kMXFP4 || fmt == kFP8 ? 64 : 128; }

// Work items (four-panel ones) from which BF16 takes four panels per wave.
constexpr long kWideItems = 512;

// Panels per wave, row tiles of the tallest tile and waves per SIMD the
// registers are sized for, by format and tile height.  Measured, gate/up +
// down: four panels (half the LDS reads per weight, two waves per SIMD) for
// MXFP4 past 16 rows per tile, DeepSeek-V3 T = 800 1213 against 1312 us, and
// for BF16 where the chip is full without the narrow items, 128 experts
// T = 600 200 against 218 us, T = 1200 228 against 236, but tiny Mixtral (8
// experts) T = 128 43 against 32; two for NVFP4, whose fp32 products are live
// besides (T = 512 238 against 283 us), and FP8 (its block sums: 128 experts
// T = 600 121 against 173).
template <int FMT, bool GU>
hipError_t launch_tiles(const StreamArgs& a, int max_tiles, hipStream_t stream) {
  if (a.bm <= 16) return launch_shape<FMT, GU, 2, 1, 4>(a, max_tiles, stream);
  if constexpr (FMT == kMXFP4) {
    return launch_shape<FMT, GU, 4, 4, 2>(a, max_tiles, stream);
  } else if constexpr (FMT == kFP8) {
    return launch_shape<FMT, GU, 2, 4, 3>(a, max_tiles, stream);
  } else if constexpr (FMT == kBF16) {
    if ((long)max_tiles * (GU ? a.I / (32 * kNW) : a.H / (64 * kNW)) >= kWideItems)
      return launch_shape<FMT, GU, 4, 8, 2>(a, max_tiles, stream);
    return launch_shape<FMT, GU, 2, 8, 2>(a, max_tiles, stream);
  } else {
    if (a.bm > 64) return launch_shape<FMT, GU, 2, 8, 2>(a, max_tiles, stream);
    return launch_shape<FMT, GU, 2, 4, 3>(a, max_tiles, stream);
  }
}

template <int FMT>
hipError_t launch_stream(bool gu, StreamArgs a, int max_tiles, hipStream_t stream) {
  using F = SFmt<FMT>;
  const long N = gu ? 2L * a.I : a.H, K = gu ? a.H : a.I;
  if (!a.w_estride) a.w_estride = F::w_bytes(N, K);
  if (!a.s_estride) a.s_estride = F::s_bytes(N, K);
  if (a.w_estride >= (1L << 31) || a.s_estride >= (1L << 31)) return hipErrorInvalidValue;
  return gu ? launch_tiles<FMT, true>(a, max_tiles, stream)
            : launch_tiles<FMT, false>(a, max_tiles, stream);
}

bool stream_args_ok(int fmt, int H, int I, int bm, int max_tiles, long w_estride,
                    long s_estride) {
  return fmt >= 0 && fmt <= kMXI8 && H > 0 && I > 0 && H % 256 == 0 && I % 128 == 0 && bm > 0 &&
         bm <= max_bm(fmt) && max_tiles >= 0 && max_tiles < (1 << 30) && w_estride >= 0 &&
         s_estride >= 0;
}

}  // namespace
}  // namespace xtu

using namespace xtu;

extern "C" {

int xtu_stream_max_tile_m(int fmt) { return fmt >= 0 && fmt <= 3 ? max_bm(fmt) : 0; }

hipError_t xtu_stream_gate_up(int fmt, const void* x, int T, const int32_t* sorted_tok, int H,
                              int I, const void* w13, const void* s13, const float* gs13,
                              long w_estride, long s_estride, const int32_t* slot_map,
                              const int32_t* seg_start, const int32_t* tile_expert,
                              const int32_t* tile_row0, const int32_t* tile_lo,
                              const int32_t* tile_hi, int bm, int max_tiles, void* act,
                              float limit, float alpha, float beta, hipStream_t stream) {
  XTU_CHECK_ARG(fmt <= kNVFP4 && stream_args_ok(fmt, H, I, bm, max_tiles, w_estride, s_estride));
  XTU_CHECK_ARG(T > 0 && (long)T * H * 2 < (1L << 31));   // 32-bit row offsets
  XTU_CHECK_ARG(x && sorted_tok && w13 && (fmt == kBF16 || s13) && seg_start && tile_expert &&
                tile_row0 && tile_lo && tile_hi && act);
  if (max_tiles == 0) return hipSuccess;
  (void)hipGetLastError();
  StreamArgs a{(const uint8_t*)x, sorted_tok, (const uint8_t*)w13, (const uint8_t*)s13, gs13,
               seg_start, tile_expert, tile_row0, tile_lo, tile_hi, slot_map, act, H, I, bm,
               (uint32_t)((long)T * H * 2), w_estride, s_estride, limit, alpha, beta, nullptr,
               nullptr, nullptr};
  switch (fmt) {
    case kMXFP4: return launch_stream<kMXFP4>(true, a, max_tiles, stream);
    case kNVFP4: return launch_stream<kNVFP4>(true, a, max_tiles, stream);
    case kFP8: return launch_stream<kFP8>(true, a, max_tiles, stream);
    default: return launch_stream<kBF16>(true, a, max_tiles, stream);
  }
}

hipError_t xtu_stream_down(int fmt, const void* act, int H, int I, const void* w2, const void* s2,
                           const float* gs2, long w_estride, long s_estride,
                           const int32_t* slot_map, const int32_t* seg_start,
                           const int32_t* tile_expert, const int32_t* tile_row0,
                           const int32_t* tile_lo, const int32_t* tile_hi, int bm, int max_tiles,
                           const int32_t* sorted_pair, float* y, hipStream_t stream) {
  XTU_CHECK_ARG(fmt <= kNVFP4 && stream_args_ok(fmt, H, I, bm, max_tiles, w_estride, s_estride));
  XTU_CHECK_ARG((long)bm * I * 2 < (1L << 31));
  XTU_CHECK_ARG(act && w2 && (fmt == kBF16 || s2) && seg_start && tile_expert && tile_row0 &&
                tile_lo && tile_hi && y);
  if (max_tiles == 0) return hipSuccess;
  (void)hipGetLastError();
  StreamArgs a{(const uint8_t*)act, nullptr, (const uint8_t*)w2, (const uint8_t*)s2, gs2,
               seg_start, tile_expert, tile_row0, tile_lo, tile_hi, slot_map, y, H, I, bm, 0u,
               w_estride, s_estride, 0.f, 1.f, 0.f, sorted_pair, nullptr, nullptr};
  switch (fmt) {
    case kMXFP4: return launch_stream<kMXFP4>(false, a, max_tiles, stream);
    case kNVFP4: return launch_stream<kNVFP4>(false, a, max_tiles, stream);
    case kFP8: return launch_stream<kFP8>(false, a, max_tiles, stream);
    default: return launch_stream<kBF16>(false, a, max_tiles, stream);
  }
}

hipError_t xtu_stream_i8_gate_up(const int8_t* a8, const int32_t* crow, int T,
                                 const int32_t* sorted_tok, int H, int I, const void* w13,
                                 const void* s13, const uint8_t* emin13, const int32_t* slot_map,
                                 const int32_t* seg_start, const int32_t* tile_expert,
                                 const int32_t* tile_row0, const int32_t* tile_lo,
                                 const int32_t* tile_hi, int bm, int max_tiles, void* act,
                                 float limit, float alpha, float beta, hipStream_t stream) {
  XTU_CHECK_ARG(stream_args_ok(kMXI8, H, I, bm, max_tiles, 0, 0));
  XTU_CHECK_ARG(T > 0 && (long)T * H < (1L << 31));   // 32-bit row offsets
  XTU_CHECK_ARG(a8 && crow && sorted_tok && w13 && s13 && emin13 && seg_start && tile_expert &&
                tile_row0 && tile_lo && tile_hi && act);
  if (max_tiles == 0) return hipSuccess;
  (void)hipGetLastError();
  StreamArgs a{(const uint8_t*)a8, sorted_tok, (const uint8_t*)w13, (const uint8_t*)s13, nullptr,
               seg_start, tile_expert, tile_row0, tile_lo, tile_hi, slot_map, act, H, I, bm,
               (uint32_t)((long)T * H), 0, 0, limit, alpha, beta, nullptr, crow, emin13};
  return launch_stream<kMXI8>(true, a, max_tiles, stream);
}

hipError_t xtu_stream_i8_down(const int8_t* a8, const int32_t* crow, int H, int I, const void* w2,
                              const void* s2, const uint8_t* emin2, const int32_t* slot_map,
                              const int32_t* seg_start, const int32_t* tile_expert,
                              const int32_t* tile_row0, const int32_t* tile_lo,
                              const int32_t* tile_hi, int bm, int max_tiles, float* y,
                              hipStream_t stream) {
  XTU_CHECK_ARG(stream_args_ok(kMXI8, H, I, bm, max_tiles, 0, 0));
  XTU_CHECK_ARG((long)bm * I < (1L << 31));
  XTU_CHECK_ARG(a8 && crow && w2 && s2 && emin2 && seg_start && tile_expert && tile_row0 &&
                tile_lo && tile_hi && y);
  if (max_tiles == 0) return hipSuccess;
  (void)hipGetLastError();
  StreamArgs a{(const uint8_t*)a8, nullptr, (const uint8_t*)w2, (const uint8_t*)s2, nullptr,
               seg_start, tile_expert, tile_row0, tile_lo, tile_hi, slot_map, y, H, I, bm, 0u,
               0, 0, 0.f, 1.f, 0.f, nullptr, crow, emin2};
  return launch_stream<kMXI8>(false, a, max_tiles, stream);
}

}  // extern "C"
