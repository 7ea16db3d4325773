// urb_gemm.hpp -- what the grouped GEMM kernels (urb_gemm.hip, urb_tall.hip) share: the kinds of
// activation rows they are built for and the projection epilogues of a tile.
#pragma once

#include "urb_device.hpp"
#include "urb_kernels.hpp"
#include "urb_panel.hpp"
#include "urb_quant.hpp"

namespace urb {

// Which activation rows a kernel is built for: decided per launch or per call (kRowsAny: f32 rows
// split into BF16 halves, or their BF16 form where every value has one), the f16 rows of the MX
// down projections, or BF16 rows (Epi::xb with no_lo: the host knows).  A kernel built for one
// kind keeps the registers of the others' staging free.
enum { kRowsAny = 0, kRowsF16 = 1, kRowsBF16 = 2 };

// The epilogue of one tile of 16 MBMAX token rows (permuted rows row0 .. row0 + mrows - 1), called
// by the four waves of its workgroup: a wave holds NP 16-row panels from panel0 on (acc0: gate or
// down, acc1: up), the workgroup the 4 NP panels of panel group `group`.  `rexp` (LDS, 16 MBMAX):
// the f16 down's row scales on entry, scratch for the gate/up.
template <int FMT, bool PAIR, int NP, int MBMAX, bool F16>
__device__ __forceinline__ void gemm_epilogue(f32x4 (&acc0)[NP][MBMAX], f32x4 (&acc1)[NP][MBMAX],
                                              const Epi& epi, int row0, int mrows, int panel0,
                                              int group, int rows, int* rexp,
                                              float* __restrict__ out, int* status) {
  const int lane = threadIdx.x & 63, ln = lane & 15, lq = lane >> 4;
  // ---- epilogue: lane holds column `row` of panel q, rows 4*lq + i of each 16-row block
  bool bad = false;
  // MX-activation gate/up: the SwiGLU rows quantized in place.  A 32-column block is one wave's
  // two panels, a 128-column block the workgroup's eight, so the block maxima take 16-lane
  // shuffles and, for 128, one pass through LDS.  (A quantize launch of its own read the rows in
  // f32 and wrote them in f32 for the down projection to convert again: 9000 rows of 2048, 47 us
  // plus 2.5 times the down's activation bytes.)
  if constexpr (PAIR && FMT != kFmtBF16 && NP == 2) {
    if (epi.qblock) {
      float amax[MBMAX][4];
#pragma unroll
      for (int mb = 0; mb < MBMAX; ++mb)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const int mm = mb * 16 + 4 * lq + i;
          amax[mb][i] = 0.0f;
          if (mm >= mrows) continue;
          const float rw = epi.row_w ? epi.row_w[epi.row_slot[row0 + mm]] : 1.0f;
#pragma unroll
          for (int q = 0; q < NP; ++q) {
            float v = epi_gate_up(epi, acc0[q][mb][i], acc1[q][mb][i], bad);
            if (epi.qround) {
              float r;
              if (rne_bf16(epi.row_w ? v * rw : v, &r)) v = r;
              else bad = true;
            }
            if (!finite(v)) bad = true;
            acc0[q][mb][i] = v;
            amax[mb][i] = fmaxf(amax[mb][i], fabsf(v));
          }
        }
#pragma unroll
      for (int mb = 0; mb < MBMAX; ++mb)
#pragma unroll
        for (int i = 0; i < 4; ++i)
#pragma unroll
          for (int x = 1; x < 16; x <<= 1)
            amax[mb][i] = fmaxf(amax[mb][i], __shfl_xor(amax[mb][i], x));
      if (epi.qblock == 128) {
        // maxima of non-negative floats through their bits
        if (threadIdx.x < 16 * MBMAX) rexp[threadIdx.x] = 0;
        __syncthreads();
        if (ln == 0) {
#pragma unroll
          for (int mb = 0; mb < MBMAX; ++mb)
#pragma unroll
            for (int i = 0; i < 4; ++i)
              atomicMax(&rexp[mb * 16 + 4 * lq + i], (int)f2u(amax[mb][i]));
        }
        __syncthreads();
#pragma unroll
        for (int mb = 0; mb < MBMAX; ++mb)
#pragma unroll
          for (int i = 0; i < 4; ++i) amax[mb][i] = u2f((uint32_t)rexp[mb * 16 + 4 * lq + i]);
      }
      u16* out16 = reinterpret_cast<u16*>(out);
#pragma unroll
      for (int mb = 0; mb < MBMAX; ++mb)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const int mm = mb * 16 + 4 * lq + i;
          if (mm >= mrows) continue;
          const float scale = e4m3_scale(amax[mb][i]);
          u16* o = out16 + (size_t)(row0 + mm) * rows + panel0 * kPanelRows + ln;
#pragma unroll
          for (int q = 0; q < NP; ++q)
            o[q * kPanelRows] =
                e4m3_value_bf16(encode_e4m3(acc0[q][mb][i] / scale), scale);
        }
      if (bad) flag(status, kStatusNonFinite);
      return;
    }
  }
  // gate/up with rowexp (the input of an f16 down projection): the largest exponent field e of
  // each token row's activations in this panel group first, then the activations as f16 times
  // 2^(141 - e) (the group's largest |value| in [2^14, 2^15)); the down projection rescales
  // each group to its row's largest e as it stages the row
  const bool rowmax = PAIR && epi.rowexp != nullptr;
  int ex[MBMAX][4];
#pragma unroll
  for (int mb = 0; mb < MBMAX; ++mb)
#pragma unroll
    for (int i = 0; i < 4; ++i) ex[mb][i] = 0;
#pragma unroll
  for (int q = 0; q < NP; ++q) {
    const int row = (panel0 + q) * kPanelRows + ln;
#pragma unroll
    for (int mb = 0; mb < MBMAX; ++mb) {
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int mm = mb * 16 + 4 * lq + i;
        if (mm >= mrows) continue;
        const size_t p = (size_t)(row0 + mm);
        if constexpr (PAIR) {
          const float a = epi_gate_up(epi, acc0[q][mb][i], acc1[q][mb][i], bad);
          if (rowmax) {
            acc0[q][mb][i] = a;
            ex[mb][i] = max(ex[mb][i], (int)((__float_as_uint(a) >> 23) & 0xffu));
          } else if (FMT == kFmtBF16 && epi.out16) {
            reinterpret_cast<u16*>(out)[p * rows + row] = (u16)(f2u(a) >> 16);
          } else {
            out[p * rows + row] = a;
          }
        } else {
          const float v =
              F16 ? epi_down<FMT>(epi, ldexpf(acc0[q][mb][i], -rexp[mm] - epi.wshift), bad)
                  : epi_down<FMT>(epi, acc0[q][mb][i], bad);
          if (!F16 && epi.out16) reinterpret_cast<u16*>(out)[p * rows + row] = (u16)(f2u(v) >> 16);
          else if (epi.stream_out) __builtin_nontemporal_store(v, &out[p * rows + row]);
          else out[p * rows + row] = v;
        }
      }
    }
  }
  if (bad) flag(status, kStatusNonFinite);
  if (rowmax) {
    // over the 16 lanes of each k-quad (the rows ln), then the four waves through LDS
#pragma unroll
    for (int mb = 0; mb < MBMAX; ++mb)
#pragma unroll
      for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int x = 1; x < 16; x <<= 1) ex[mb][i] = max(ex[mb][i], __shfl_xor(ex[mb][i], x));
    if (threadIdx.x < 16 * MBMAX) rexp[threadIdx.x] = 0;
    __syncthreads();
    if (ln == 0) {
#pragma unroll
      for (int mb = 0; mb < MBMAX; ++mb)
#pragma unroll
        for (int i = 0; i < 4; ++i) atomicMax(&rexp[mb * 16 + 4 * lq + i], ex[mb][i]);
    }
    __syncthreads();
    u16* out16 = reinterpret_cast<u16*>(out);
#pragma unroll
    for (int q = 0; q < NP; ++q) {
      const int row = (panel0 + q) * kPanelRows + ln;
#pragma unroll
      for (int mb = 0; mb < MBMAX; ++mb)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const int mm = mb * 16 + 4 * lq + i;
          if (mm >= mrows) continue;
          const _Float16 h = (_Float16)ldexpf(acc0[q][mb][i], 141 - rexp[mm]);
          out16[(size_t)(row0 + mm) * rows + row] = __builtin_bit_cast(u16, h);
        }
    }
    if ((int)threadIdx.x < mrows)
      epi.rowexp[(size_t)(row0 + threadIdx.x) * epi.groups + group] = rexp[threadIdx.x];
  }
}

}  // namespace urb
