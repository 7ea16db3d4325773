// urb_tall.hip -- grouped expert GEMMs over tall tiles: up to 128 tokens of one expert at once.
//
// The grouped GEMM (urb_gemm.hip) takes 32-token tiles at three or four workgroups per CU, which
// streams a batch's weights well but decodes an expert's MX weights once per 32 tokens and reads a
// fragment of activations from LDS for every four MFMAs.  From about gemm_tile_rows' count of
// tokens per expert on, the matrix cores are what a batch needs, and this kernel feeds them:
//
//  * an expert's tokens are cut into ceil(count / 128) tiles of equal height (a multiple of 16;
//    gemm_tile_span), so no tile is left with a few tokens;
//  * each of four waves owns four 16-row panels (gate/up: two of each) and sweeps them through the
//    tile's 16-token blocks: 4 x up to 8 accumulator blocks, so one decoded weight operand feeds up
//    to eight MFMAs and one activation fragment four;
//  * weights stream from HBM or L2 into a register ring of 1 KiB slabs (one slab = 128, 64 or 32
//    columns for MXFP4, MXFP8, BF16), activations through LDS: the rows of K step s + 1 are loaded
//    and stored in two halves between the MFMAs of step s, so staging takes few registers and each
//    load has half a step (some 1000 cycles of MFMAs) to arrive;
//  * two workgroups per CU (256 registers per wave, 64 KiB of LDS each), which cover each other's
//    barriers and epilogues.
//
// Bound by the matrix cores and what their feeding leaves idle (4096 tokens, top-8 over 256 MXFP4
// experts of 7168 x 2048: gate/up 2,263 -> 1,814-1,880 us, 1.0-1.06 PFLOP/s, where a large BF16
// library product reaches 1.41; down 1,341 -> 1,300 us, 940 MB of f32 rows to write among it; 2000
// tokens over 160 MXFP8 experts of 6144 x 2048: gate/up 1,648 -> 930, down 964 -> 591).  Left to
// itself the compiler sinks the staging loads to their stores: 2,294 us for that gate/up without the
// scheduling fences.
//
// Rows that are not BF16-valued (f32 hidden states) are split into hi and lo BF16 halves, as in the
// grouped GEMM; the two halves take the two LDS buffers, so such a tile stages without overlap and
// the other workgroup of the CU fills the gaps.
#include "urb_gemm.hpp"

#include <algorithm>

namespace urb {

namespace {

constexpr int kTT = kTallTile;      // most tokens per tile
constexpr int kTB = kTT / 16;       // 16-token blocks per tile
constexpr int kTP = 4;              // panels per wave (gate/up: two of each)

// __builtin_amdgcn_sched_barrier masks: what may still cross.  Left alone, the scheduler sinks a
// step's loads to just before their use, which exposes their whole latency.
constexpr int kStaging = 0x106;  // VALU, SALU, LDS reads: loads, LDS stores and MFMAs stay in place

struct TallLds {
  u16 a[2][kTT * kALd];
  int rexp[kTT];  // the f16 down's row scales, the gate/up's row maxima
};

// 1 KiB slabs of one panel per K step (128 columns).
template <int FMT>
constexpr int slabs_per_step() { return FMT == kFmtMXFP4 ? 1 : FMT == kFmtMXFP8 ? 2 : 4; }

// MFMA operand of part `part` (of 4 / slabs_per_step) of a slab.
template <int FMT>
__device__ __forceinline__ bf16x8 slab_bf16(const uint4& q, float sc, int part) {
  if constexpr (FMT == kFmtBF16) {
    return __builtin_bit_cast(bf16x8, q);
  } else if constexpr (FMT == kFmtMXFP4) {
    const uint32_t w = part == 0 ? q.x : part == 1 ? q.y : part == 2 ? q.z : q.w;
    return pack8(__builtin_amdgcn_cvt_scalef32_pk_bf16_fp4(w, sc, 0),
                 __builtin_amdgcn_cvt_scalef32_pk_bf16_fp4(w, sc, 1),
                 __builtin_amdgcn_cvt_scalef32_pk_bf16_fp4(w, sc, 2),
                 __builtin_amdgcn_cvt_scalef32_pk_bf16_fp4(w, sc, 3));
  } else {
    const uint32_t w0 = part ? q.z : q.x, w1 = part ? q.w : q.y;
    return pack8(__builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(w0, sc, false),
                 __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(w0, sc, true),
                 __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(w1, sc, false),
                 __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(w1, sc, true));
  }
}
template <int FMT>
__device__ __forceinline__ f16x8 slab_f16(const uint4& q, float sc, int part) {
  uint32_t p[4];
  if constexpr (FMT == kFmtMXFP4) {
    const uint32_t w = part == 0 ? q.x : part == 1 ? q.y : part == 2 ? q.z : q.w;
    p[0] = __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_f16_fp4(w, sc, 0));
    p[1] = __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_f16_fp4(w, sc, 1));
    p[2] = __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_f16_fp4(w, sc, 2));
    p[3] = __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_f16_fp4(w, sc, 3));
  } else {
    const uint32_t w0 = part ? q.z : q.x, w1 = part ? q.w : q.y;
    p[0] = __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_f16_fp8(w0, sc, false));
    p[1] = __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_f16_fp8(w0, sc, true));
    p[2] = __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_f16_fp8(w1, sc, false));
    p[3] = __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_f16_fp8(w1, sc, true));
  }
  return __builtin_bit_cast(f16x8, make_uint4(p[0], p[1], p[2], p[3]));
}

template <int FMT, bool PAIR, int ROWS>
__global__ __launch_bounds__(256, 2) void tall_kernel(const ExpertMats* __restrict__ mats, Perm perm,
                                                      int max_tiles, int rows, int K,
                                                      const float* __restrict__ in,
                                                      float* __restrict__ out, Epi epi,
                                                      int* status) {
  static_assert(!(ROWS == kRowsF16 && (PAIR || FMT == kFmtBF16)), "f16 rows: MX down projections");
  constexpr bool F16 = ROWS == kRowsF16;
  constexpr int NP = PAIR ? 2 : 4;  // panels per wave and matrix
  constexpr int SL = slabs_per_step<FMT>(), PARTS = 4 / SL;
  constexpr bool MX = FMT != kFmtBF16;
  __shared__ __attribute__((aligned(16))) TallLds lds;

  const int groups = rows / (kNT * NP);
  int w, group;
  if (!gemm_place(blockIdx.x, min(perm.meta[1], max_tiles), groups, 1, &w, &group)) return;
  const int expert = perm.tiles[2 * w], m0 = perm.tiles[2 * w + 1];
  const int count = perm.counts[expert], row0 = perm.offsets[expert] + m0;
  const int mrows = min(gemm_tile_span(count, kTT), count - m0);
  const ExpertMats m = mats[expert];
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int ln = lane & 15, lq = lane >> 4;
  const int panel0 = (group * 4 + wave) * NP;
  const size_t pbytes = kPanelRows * panel_row_bytes<FMT>(K);
  const size_t pscales = (size_t)kPanelRows * (K / 32);
  // wavefront-uniform panel bases; the lane's unit is at 16 lane (data), lane (scales)
  const uint8_t* pd[kTP];
  const uint8_t* ps[kTP];
#pragma unroll
  for (int p = 0; p < kTP; ++p) {
    const int mat = PAIR ? p / NP : 2, q = p % NP;
    pd[p] = m.data[mat] + (panel0 + q) * pbytes;
    ps[p] = MX ? m.scales[mat] + (panel0 + q) * pscales : nullptr;
  }

  // ---- this thread's staging slots: rows am + 32 g.  A slot past the tile's last row stages the
  // tile's first row instead: its products land in accumulator rows the epilogue never stores.
  constexpr int RG = kTT / 32;
  const int am = threadIdx.x >> 3;
  uint32_t a_row[RG];
#pragma unroll
  for (int g = 0; g < RG; ++g) {
    const int p = row0 + (am + 32 * g < mrows ? am + 32 * g : 0);
    a_row[g] = (uint32_t)(PAIR ? perm.perm_token[p] : p);
  }
  const int steps = K / kKS;
  // F16: the row's largest exponent field over the gate/up panel groups (Epi::rowexp: one group
  // per K step), and its epilogue scale
  if constexpr (F16) {
#pragma unroll
    for (int g = 0; g < RG; ++g) {
      const int* ex = epi.rowexp + (size_t)a_row[g] * steps;
      int e = 0;
      for (int gg = 0; gg < steps; ++gg) e = max(e, ex[gg]);
      if ((threadIdx.x & 7) == 0) lds.rexp[am + 32 * g] = 141 - e;
    }
    __syncthreads();  // the row's other seven threads stage their chunks by it
  }

  f32x4 acc[PAIR ? 2 : 1][NP][kTB];
#pragma unroll
  for (int h = 0; h < (PAIR ? 2 : 1); ++h)
#pragma unroll
    for (int q = 0; q < NP; ++q)
#pragma unroll
      for (int i = 0; i < kTB; ++i) acc[h][q][i] = f32x4{0.f, 0.f, 0.f, 0.f};

  // NMB: 16-token blocks of the tile; SPLIT: f32 rows as hi + lo halves (else 16-bit rows)
  auto body = [&](auto nmb, auto split) {
    constexpr int NMB = decltype(nmb)::value;
    constexpr bool SPLIT = decltype(split)::value;
    constexpr int G = (NMB + 1) / 2;          // 32-row staging groups
    constexpr int G0 = (G + 1) / 2;           // of them staged in the step's first half
    const uint8_t* rows16 = F16 ? reinterpret_cast<const uint8_t*>(in)
                                : reinterpret_cast<const uint8_t*>(epi.xb);
    // Byte offsets this thread keeps: its staged rows (16-bit rows: at most 131072 of 12288 values),
    // its staging stores (chunks c and 8 + c of row am; row group g is 512 B on) and its fragment
    // reads (MFMA j; 16-token block mb is 256 B on).
    const int c8 = threadIdx.x & 7;
    uint32_t a_off[G];
#pragma unroll
    for (int g = 0; g < G; ++g) a_off[g] = a_row[g] * (uint32_t)(2 * K) + 16u * c8;
    const uint32_t so0 = 2u * a_chunk<kTT>(am, c8), so1 = 2u * a_chunk<kTT>(am, 8 + c8);
    uint32_t fo[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) fo[j] = 2u * a_chunk<kTT>(ln, frag_k<FMT>(j, lq) >> 3);
    uint8_t* const lds_a = reinterpret_cast<uint8_t*>(&lds.a[0][0]);
    constexpr uint32_t kBuf = sizeof(lds.a[0]);
    auto frag = [&](int j, uint32_t buf, int mb) {
      return *reinterpret_cast<const uint4*>(lds_a + (fo[j] + buf) + mb * 256u);
    };

    // Weights: two slabs of each panel and the step's E8M0 scales.  A slab's slot is refilled with the
    // slab two on as soon as its last part is used (BF16 and MXFP8); MXFP4, one slab per step, loads
    // the next one a step ahead and moves it.  Every load is issued, those past the last slab
    // re-reading it: the step is one basic block.
    uint4 slab[2][kTP];
    const int slabs = steps * SL;
    uint32_t sc[kTP], sc_next[kTP];
    const uint32_t doff = 16u * lane;
    auto fetch = [&](uint4* to, int u) {
#pragma unroll
      for (int p = 0; p < kTP; ++p) to[p] = ldg16(pd[p] + (doff + (uint32_t)u * 1024u));
    };
    auto fetch_scales = [&](uint32_t* to, int s) {
      if constexpr (MX) {
#pragma unroll
        for (int p = 0; p < kTP; ++p) to[p] = ldg_u8(ps[p] + ((uint32_t)lane + (uint32_t)s * 64u));
      }
    };

    auto load16 = [&](AStage16& a, int g, int s) {
      const uint8_t* p = rows16 + (a_off[g] + (uint32_t)s * (2u * kKS));
      a.v[0] = ldg16(p);
      a.v[1] = ldg16(p + kKS);
      if constexpr (F16) a.e = epi.rowexp[(size_t)a_row[g] * steps + s];
    };
    auto store16 = [&](AStage16& a, int g, uint32_t buf) {
      if constexpr (F16) scale_a16(a, 141 - lds.rexp[am + 32 * g]);
      *reinterpret_cast<uint4*>(lds_a + (so0 + buf) + g * 512u) = a.v[0];
      *reinterpret_cast<uint4*>(lds_a + (so1 + buf) + g * 512u) = a.v[1];
    };

    // MFMA j of the step, the rows in the LDS buffer at byte `buf` (SPLIT: hi halves in buffer 0, lo
    // halves in buffer 1)
    auto mma = [&](int j, uint32_t buf) {
      const int part = j % PARTS;
      if constexpr (F16) {
        f16x8 a[NMB];
#pragma unroll
        for (int mb = 0; mb < NMB; ++mb) a[mb] = __builtin_bit_cast(f16x8, frag(j, buf, mb));
#pragma unroll
        for (int q = 0; q < NP; ++q) {
          const f16x8 b = slab_f16<FMT>(slab[(j / PARTS) & 1][q], e8m0_to_f32(sc[q]), part);
#pragma unroll
          for (int mb = 0; mb < NMB; ++mb)
            acc[0][q][mb] = __builtin_amdgcn_mfma_f32_16x16x32_f16(a[mb], b, acc[0][q][mb], 0, 0, 0);
        }
      } else {
#pragma unroll
        for (int half = 0; half < (SPLIT ? 2 : 1); ++half) {
          bf16x8 a[NMB];
#pragma unroll
          for (int mb = 0; mb < NMB; ++mb)
            a[mb] = __builtin_bit_cast(bf16x8, frag(j, SPLIT ? half * kBuf : buf, mb));
#pragma unroll
          for (int p = 0; p < kTP; ++p) {
            const int h = PAIR ? p / NP : 0, q = p % NP;
            const bf16x8 b =
                slab_bf16<FMT>(slab[(j / PARTS) & 1][p], MX ? e8m0_to_f32(sc[p]) : 1.0f, part);
#pragma unroll
            for (int mb = 0; mb < NMB; ++mb)
              acc[h][q][mb] =
                  __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[mb], b, acc[h][q][mb], 0, 0, 0);
          }
        }
      }
    };

#pragma unroll
    for (int i = 0; i < (SL == 1 ? 1 : 2); ++i) fetch(slab[i], i);
    fetch_scales(sc, 0);
    uint32_t buf = 0;
    if constexpr (!SPLIT) {
#pragma unroll
      for (int g = 0; g < G; ++g) {
        AStage16 st;
        load16(st, g, 0);
        store16(st, g, 0);
      }
      __syncthreads();
    }
    // drained here, so that the wait counts inside the loop are those of its own loads
    __builtin_amdgcn_s_waitcnt(0x0f70);  // vmcnt(0)
    for (int s = 0; s < steps; ++s) {
      const int s1 = min(s + 1, steps - 1);
      if constexpr (SPLIT) {
        // both LDS buffers hold this step's halves
        if (s) __syncthreads();
#pragma unroll
        for (int g = 0; g < G; ++g) {
          AStage a;
          load_a(a, in + (size_t)a_row[g] * K, true, s * kKS);
          store_a<kTT>(a, lds.a[0], lds.a[1], am + 32 * g);
        }
        __syncthreads();
      }
      AStage16 st[G0];
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        if (j == 0) {
          if constexpr (!SPLIT) {
#pragma unroll
            for (int g = 0; g < G0; ++g) load16(st[g], g, s1);
          }
          if constexpr (FMT == kFmtMXFP4) fetch(slab[1], s1);
          fetch_scales(sc_next, s1);
        }
        if constexpr (!SPLIT) {
          if (j == 2) {
#pragma unroll
            for (int g = 0; g < G0; ++g) store16(st[g], g, buf ^ kBuf);
#pragma unroll
            for (int g = G0; g < G; ++g) load16(st[g - G0], g, s1);
          }
        }
        if (j == 0 || j == 2) __builtin_amdgcn_sched_barrier(kStaging);
        mma(j, buf);
        if (j == 1) __builtin_amdgcn_sched_barrier(F16 ? 0 : kStaging);
        if (j == 3) __builtin_amdgcn_sched_barrier(0);
        if constexpr (FMT != kFmtMXFP4) {
          if (j % PARTS == PARTS - 1)
            fetch(slab[(j / PARTS) & 1], min(s * SL + j / PARTS + 2, slabs - 1));
        }
      }
      if constexpr (FMT == kFmtMXFP4) {
#pragma unroll
        for (int p = 0; p < kTP; ++p) slab[0][p] = slab[1][p];
      }
#pragma unroll
      for (int p = 0; p < kTP; ++p) sc[p] = sc_next[p];
      if constexpr (!SPLIT) {
#pragma unroll
        for (int g = G0; g < G; ++g) store16(st[g - G0], g, buf ^ kBuf);
        __syncthreads();
        buf ^= kBuf;
      }
    }
  };
  auto run = [&](auto split) {
    if (mrows > 96) body(Int<8>{}, split);
    else if (mrows > 64) body(Int<6>{}, split);
    else if (mrows > 32) body(Int<4>{}, split);
    else body(Int<2>{}, split);
  };
  if constexpr (F16) {
    run(std::false_type{});
  } else {
    const bool bf16_rows = epi.no_lo || (epi.lo_word && *epi.lo_word != epi.lo_gen);
    if (bf16_rows && epi.xb) run(std::false_type{});
    else run(std::true_type{});
  }
  gemm_epilogue<FMT, PAIR, NP, kTB, F16>(acc[0], acc[PAIR ? 1 : 0], epi, row0, mrows, panel0, group, rows,
                                         lds.rexp, out, status);
}

template <int FMT, bool PAIR, int ROWS>
void launch_shape(const ExpertMats* mats, const Perm& perm, int max_tiles, int rows, int K,
                  const float* in, float* out, const Epi& epi, int* status, hipStream_t s) {
  const int groups = rows / (kNT * (PAIR ? 2 : 4));
  const int blocks = 8 * gemm_blocks_per_xcd(max_tiles, groups, 1);
  tall_kernel<FMT, PAIR, ROWS><<<dim3(blocks), 256, 0, s>>>(mats, perm, max_tiles, rows, K, in, out,
                                                            epi, status);
}

template <int FMT>
void launch(bool pair, const ExpertMats* mats, const Perm& perm, int max_tiles, int rows, int K,
            const float* in, float* out, const Epi& epi, int* status, hipStream_t s) {
  if (pair) {
    launch_shape<FMT, true, kRowsAny>(mats, perm, max_tiles, rows, K, in, out, epi, status, s);
    return;
  }
  if constexpr (FMT != kFmtBF16) {
    if (epi.rowexp) {
      launch_shape<FMT, false, kRowsF16>(mats, perm, max_tiles, rows, K, in, out, epi, status, s);
      return;
    }
  }
  launch_shape<FMT, false, kRowsAny>(mats, perm, max_tiles, rows, K, in, out, epi, status, s);
}

}  // namespace

void launch_tall(int fmt, bool pair, const ExpertMats* mats, const Perm& perm, int max_tiles,
                 int rows, int K, const float* in, float* out, const Epi& epi, int* status,
                 hipStream_t s) {
  if (fmt == kFmtBF16)
    launch<kFmtBF16>(pair, mats, perm, max_tiles, rows, K, in, out, epi, status, s);
  else if (fmt == kFmtMXFP4)
    launch<kFmtMXFP4>(pair, mats, perm, max_tiles, rows, K, in, out, epi, status, s);
  else
    launch<kFmtMXFP8>(pair, mats, perm, max_tiles, rows, K, in, out, epi, status, s);
}

}  // namespace urb
