// Device pieces shared by the GEMM kernels: activation
// functions, split-K ranges, direct-to-LDS loads and the staged row epilogue.
#pragma once
#include <stdint.h>

#include <type_traits>
#include <utility>

#include "internal.h"

typedef float floatx16 __attribute__((ext_vector_type(16)));

namespace gs {
namespace {

constexpr int GROUP_M = 8;

// f(0), f(1), ... with the index as a constant.
template <class F, int... I>
__device__ __forceinline__ void const_for(std::integer_sequence<int, I...>, F&& f) {
  (f(std::integral_constant<int, I>()), ...);
}

// GELU, tanh form (src/nn/vit.cr:130-148): 0.5*v*(1 + tanh(u)) with
// u = c*(v + 0.044715*v^3), c = (float)sqrt(2/pi). Evaluated through the exact
// identity 0.5*(1 + tanh(u)) = 1/(1 + exp(-2u)) with the hardware exp2 and
// reciprocal (a few instructions instead of a library tanh in every epilogue
// element); the relative error is a few ulp, far inside the fp32 parity
// tolerance. Saturates to v for large u and to -0 for large negative u.
__device__ __forceinline__ float gelu_tanh(float v) {
  const float c = 0.7978845608028654f;
  const float u = c * (v + 0.044715f * v * v * v);
  const float e = __builtin_amdgcn_exp2f(-2.8853900817779268f * u);  // exp(-2u)
  return v * __builtin_amdgcn_rcpf(1.0f + e);
}

// q = n / d, r = n % d for 0 <= n < 2^22, d >= 1, from rd = 1/d in fp32: the
// product n*rd is within 0.5 of n/d in that range, so one correction step
// makes the quotient exact.
__device__ __forceinline__ int divmod_small(int n, int d, float rd, int& r) {
  int q = (int)((float)n * rd);
  r = n - q * d;
  if (r < 0) {
    --q;
    r += d;
  } else if (r >= d) {
    ++q;
    r -= d;
  }
  return q;
}

__device__ __forceinline__ fx4 relu4(fx4 v) {
  return mk4(fmaxf(v.x, 0.f), fmaxf(v.y, 0.f), fmaxf(v.z, 0.f),
                     fmaxf(v.w, 0.f));
}

// EPI_DUAL's second store of four consecutive columns at element offset off:
// the value, or with EPI_DUAL_RELU_H bf16(max(v, 0)) (C2 then holds bf16).
__device__ __forceinline__ void dual_store(const GemmArgs& p, int flags, int64_t off, fx4 v) {
  if (flags & EPI_DUAL_RELU_H) {
    typedef __bf16 bf16x4_t __attribute__((ext_vector_type(4)));
    const fx4 r = relu4(v);
    const bf16x4_t h = {(__bf16)r.x, (__bf16)r.y, (__bf16)r.z, (__bf16)r.w};
    *(bf16x4_t*)((__bf16*)p.C2 + off) = h;
  } else {
    *(fx4*)(p.C2 + off) = v;
  }
}

// Split-K range of workgroup row blockIdx.y: the K steps (of `unit` elements)
// are cut at floor(y * steps / S), so ranges differ by at most one step and S
// need not divide the step count (the host keeps every range non-empty).
__device__ __forceinline__ void split_range(int K, int S, int unit, int& kbeg, int& kend) {
  const int steps = K / unit, y = blockIdx.y;
  kbeg = (int)((int64_t)y * steps / S) * unit;
  kend = (int)((int64_t)(y + 1) * steps / S) * unit;
}

// LDS byte address of a __shared__ pointer.
__device__ __forceinline__ uint32_t lds_addr(const float* ptr) {
  return (uint32_t)(uintptr_t)(const __attribute__((address_space(3))) float*)ptr;
}
// One wave-wide global_load_lds_dwordx4: lane l's 16 bytes at gptr land at
// LDS byte lds + 16*l (lds is wave-uniform, passed through M0). Issued as
// inline asm so that the compiler does not track it as an LDS store: its
// wait insertion cannot tell the two LDS buffers apart and would otherwise
// wait for the in-flight prefetch before every LDS read. The kernel waits
// for these loads itself (s_waitcnt vmcnt).
__device__ __forceinline__ void lds_dma16(const float* gptr, uint32_t lds) {
  asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, off"
               :
               : "s"(lds), "v"(gptr)
               : "memory", "m0");
}

// The same from a wave-uniform base and a lane's 32-bit byte offset.
__device__ __forceinline__ void lds_dma16_off(const void* base, uint32_t off, uint32_t lds) {
  asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2"
               :
               : "s"(lds), "v"(off), "s"(base)
               : "memory", "m0");
}

constexpr int W2M = 256, W2N = 128, W2K = 32;

constexpr int W2_SS = 68;                    // epilogue stage row stride (floats)
constexpr int W2_SS1 = 36;                   // the same for one 32-column block

// GELU / ReLU of four values, as the flags say
__device__ __forceinline__ fx4 epi_act(fx4 v, int flags) {
  if (flags & EPI_GELU) v = mk4(gelu_tanh(v.x), gelu_tanh(v.y), gelu_tanh(v.z), gelu_tanh(v.w));
  if (flags & EPI_RELU) v = relu4(v);
  return v;
}

// Second half of the row epilogues: the wave's LDS stage (32 rows of 32 * NB
// columns, row stride W2_SS / W2_SS1) is read back in 16-byte row segments,
// residuals are added and the rows stored. ACT: bias, GELU and ReLU happen
// here too (the stage holds raw sums).
template <bool ACT, int NB>
__device__ __forceinline__ void epi_store(const GemmArgs& p, int flags, int row0, int col0,
                                          float* stage, int lane) {
  constexpr int SS = NB == 2 ? W2_SS : W2_SS1;  // stage row stride (floats)
  const int M = p.M, N = p.N;
  // the stage belongs to this wave: LDS accesses of one wave complete in
  // order, so a wave-level fence orders the writes above and the reads below
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
  // readback: LPR lanes per row (4 columns each), RPP rows per pass, UPH
  // passes per 16-row half
  constexpr int LPR = 8 * NB, RPP = 64 / LPR, UPH = 16 / RPP;
  typedef __bf16 bf16x4_t __attribute__((ext_vector_type(4)));
  const int rin = lane / LPR, c4 = (lane % LPR) * 4;
  const float* const sp = stage + rin * SS + c4;
  fx4 bv = {};
  if constexpr (ACT) {
    if (flags & EPI_BIAS) {
      const float* const b = p.bias + min(col0 + c4, N - 4);
      bv = mk4(b[0], b[1], b[2], b[3]);
    }
  }
  if (flags & EPI_SCATTER) {
    // sub-pixel scatter: column col = (i * sc_r + j) * sc_C + c; with sc_C and
    // sc_Cout multiples of 4 the lane's 4 columns are one pixel's channels
    // c .. c + 3, all kept or all dropped, 16 contiguous output bytes
    const int col = col0 + c4;
    const int sidx = col / p.sc_C, sc_c = col - sidx * p.sc_C;
    const int sc_i = sidx / p.sc_r, sc_j = sidx - sc_i * p.sc_r;
    const int hw = p.sc_gh * p.sc_gw;
#pragma unroll
    for (int u = 0; u < 2 * UPH; ++u) {
      const int row = row0 + RPP * u + rin;
      fx4 v = *(const fx4*)(sp + RPP * u * SS);
      if constexpr (ACT) {
        if (flags & EPI_BIAS) v = v + bv;
        v = epi_act(v, flags);
      }
      if (row < M && col < N && sc_c < p.sc_Cout) {
        const int img = row / hw;
        const int rem = row - img * hw;
        const int yy = rem / p.sc_gw, xx = rem - yy * p.sc_gw;
        const int64_t oy = (int64_t)img * p.sc_gh * p.sc_r + yy * p.sc_r + sc_i;
        const int64_t ox = (int64_t)xx * p.sc_r + sc_j;
        const int64_t si = (oy * p.sc_gw * p.sc_r + ox) * p.sc_Cout + sc_c;
        if (flags & EPI_BF16OUT) {
          const bf16x4_t h = {(__bf16)v.x, (__bf16)v.y, (__bf16)v.z, (__bf16)v.w};
          *(bf16x4_t*)((__bf16*)p.C + si) = h;
        } else {
          *(fx4*)(p.C + si) = v;
        }
      }
    }
  } else {
    const bool inside = row0 + 32 <= M && col0 + 32 * NB <= N;
    const int64_t cb = (int64_t)row0 * p.ldc + col0;  // the block's first element (uniform)
    const uint32_t co = (uint32_t)rin * (uint32_t)p.ldc + c4, cs = RPP * (uint32_t)p.ldc;
    // two halves of 16 rows, the residuals of a half read before its stores
#pragma unroll
    for (int hq = 0; hq < 2; ++hq) {
      fx4 v[UPH];
#pragma unroll
      for (int u = 0; u < UPH; ++u) v[u] = *(const fx4*)(sp + (16 * hq + RPP * u) * SS);
      if constexpr (ACT) {
        if (flags & EPI_BIAS) {
#pragma unroll
          for (int u = 0; u < UPH; ++u) v[u] = v[u] + bv;
        }
        if (flags & (EPI_GELU | EPI_RELU)) {
#pragma unroll
          for (int u = 0; u < UPH; ++u) v[u] = epi_act(v[u], flags);
        }
      }
      if (flags & (EPI_RES1 | EPI_RES2)) {
        // rows and columns outside the output read its last ones (not stored)
        const int colc = min(col0 + c4, N - 4);
        fx4 x[UPH];
        if (flags & EPI_RES1) {
#pragma unroll
          for (int u = 0; u < UPH; ++u) {
            const int row = min(row0 + 16 * hq + RPP * u + rin, M - 1);
            x[u] = *(const fx4*)(p.R1 + (int64_t)row * p.ldr1 + colc);
          }
#pragma unroll
          for (int u = 0; u < UPH; ++u) v[u] = v[u] + x[u];
        }
        if (flags & EPI_RES2) {
#pragma unroll
          for (int u = 0; u < UPH; ++u) {
            const int row = min(row0 + 16 * hq + RPP * u + rin, M - 1);
            x[u] = *(const fx4*)(p.R2 + (int64_t)row * p.ldr2 + colc);
          }
#pragma unroll
          for (int u = 0; u < UPH; ++u) v[u] = x[u] + v[u];
        }
      }
      if (flags & EPI_BF16OUT) {
        char* const c = (char*)p.C + 2 * cb;
#pragma unroll
        for (int u = 0; u < UPH; ++u) {
          const bf16x4_t h = {(__bf16)v[u].x, (__bf16)v[u].y, (__bf16)v[u].z, (__bf16)v[u].w};
          if (inside || (row0 + 16 * hq + RPP * u + rin < M && col0 + c4 < N))
            *(bf16x4_t*)(c + 2 * (co + (16 / RPP * hq + u) * cs)) = h;
        }
      } else if (inside) {
        char* const c = (char*)p.C + 4 * cb;
#pragma unroll
        for (int u = 0; u < UPH; ++u) *(fx4*)(c + 4 * (co + (16 / RPP * hq + u) * cs)) = v[u];
        if (flags & EPI_DUAL) {
#pragma unroll
          for (int u = 0; u < UPH; ++u)
            dual_store(p, flags, cb + (co + (16 / RPP * hq + u) * cs), v[u]);
        }
      } else {
#pragma unroll
        for (int u = 0; u < UPH; ++u)
          if (row0 + 16 * hq + RPP * u + rin < M && col0 + c4 < N) {
            const int64_t o = cb + (co + (16 / RPP * hq + u) * cs);
            *(fx4*)(p.C + o) = v[u];
            if (flags & EPI_DUAL) dual_store(p, flags, o, v[u]);
          }
      }
    }
  }
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// Epilogue of one 32 x 64 block row of a wave (q0: columns col0 .. +31, q1:
// col0 + 32 .. +63; NB = 1: one 32-column block, q1 unused): bias, RoPE, GELU /
// ReLU on the accumulators, then through the wave's LDS stage (32 rows of W2_SS
// floats) so that residuals are read and outputs written as 16-byte row segments
// (16 lanes per 64-column row). Same per-element operations and order as
// gemm_epilogue_t. The scatter form (ConvT / pixel shuffle) stores 4-column
// segments, each inside one output pixel: the host admits it only with
// sc_C % 4 == 0, sc_Cout % 4 == 0 and no residual, RoPE or dual store
// (row_epi_ok).
// It is issue-bound: a wave leaves its matrix cores idle for every instruction
// here. The uniform choices are therefore taken once per four rows (first phase)
// or per 16-row half (second phase), not per element, and a block inside the
// output stores without row checks through a scalar base and 32-bit lane offsets.
// With the choices per element, as before: bf16 linear 24576 x 4096 x 1024 with
// GELU and its operand conversions 300.5 -> 285.3 us, 8 pairs at 512x512 in bf16
// 34.03 -> 32.81 ms, one pair in fp32 20.56 -> 20.43 ms, bit-identical outputs.
template <bool ROPE, int NB = 2>
__device__ __forceinline__ void w2_epi_row(const GemmArgs& p, const floatx16& q0,
                                           const floatx16& q1, int row0, int col0, float* stage,
                                           int lane, int l32, int hl) {
  static_assert(NB == 1 || NB == 2, "one or two 32-column blocks");
  constexpr int SS = NB == 2 ? W2_SS : W2_SS1;  // stage row stride (floats)
  const int M = p.M, N = p.N;
  const int flags = ROPE ? p.flags & ~(EPI_RES1 | EPI_RES2) : p.flags & ~EPI_ROPE;
  // NB = 2: col0 is a multiple of 64, so q0 is the y-axis half and q1 the
  // x-axis half of one head's RoPE columns. NB = 1: col0 is a multiple of 32
  // and names the half
  const float bv0 = (flags & EPI_BIAS) ? p.bias[min(col0 + l32, N - 1)] : 0.f;
  const float bv1 =
      (NB == 2 && (flags & EPI_BIAS)) ? p.bias[min(col0 + 32 + l32, N - 1)] : 0.f;
  const bool rope = ROPE && col0 < p.rope_ncols;
  const bool xhalf = NB == 1 && (col0 & 32) != 0;
  const float rtok = ROPE ? 1.0f / (float)p.tok_per_img : 0.f;
  const float rgw = ROPE ? 1.0f / (float)p.grid_w : 0.f;
  // With the tokens per image and the grid width multiples of 4, the four
  // rows of a register group lie in one image and grid row: their position is
  // decoded once (the first row's, x + j for row j) and the y-axis cos / sin
  // are read once. Rows at or past M are not stored; their group decodes the
  // last group start below M.
  const bool grp4 = ROPE && ((p.tok_per_img | p.grid_w) & 3) == 0;
  float* const srow = stage + 4 * hl * SS + l32;
#pragma unroll
  for (int g = 0; g < 4; ++g) {  // rows row0 + 8 g + 4 hl + 0 .. 3
    float v0[4], v1[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      v0[j] = q0[4 * g + j];
      v1[j] = q1[4 * g + j];
    }
    if (flags & EPI_BIAS) {
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        v0[j] = v0[j] + bv0;
        v1[j] = v1[j] + bv1;
      }
    }
    if (rope) {
      // cos / sin of the four rows at frequency l32 % 16: y axis, x axis
      float cy[4], sy[4], cx[4], sx[4];
      if (grp4) {
        const int rg = min(row0 + 8 * g + 4 * hl, (M - 1) & ~3);
        int tok, tx;
        divmod_small(rg, p.tok_per_img, rtok, tok);
        const int ty = divmod_small(tok, p.grid_w, rgw, tx);
        const int iy = ty * 16 + (l32 & 15), ix = tx * 16 + (l32 & 15);
        cy[0] = p.rope_cos[iy];
        sy[0] = p.rope_sin[iy];
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          cy[j] = cy[0];
          sy[j] = sy[0];
          cx[j] = p.rope_cos[ix + 16 * j];
          sx[j] = p.rope_sin[ix + 16 * j];
        }
      } else {
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          const int row = min(row0 + 8 * g + 4 * hl + j, M - 1);
          int tok, tx;
          divmod_small(row, p.tok_per_img, rtok, tok);
          const int ty = divmod_small(tok, p.grid_w, rgw, tx);
          const int iy = ty * 16 + (l32 & 15), ix = tx * 16 + (l32 & 15);
          cy[j] = p.rope_cos[iy];
          sy[j] = p.rope_sin[iy];
          cx[j] = p.rope_cos[ix];
          sx[j] = p.rope_sin[ix];
        }
      }
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        if constexpr (NB == 2) {
          const float p0 = __shfl_xor(v0[j], 16), p1 = __shfl_xor(v1[j], 16);
          v0[j] = (l32 < 16) ? (v0[j] * cy[j] - p0 * sy[j]) : (v0[j] * cy[j] + p0 * sy[j]);
          v1[j] = (l32 < 16) ? (v1[j] * cx[j] - p1 * sx[j]) : (v1[j] * cx[j] + p1 * sx[j]);
        } else {
          const float c = xhalf ? cx[j] : cy[j], sn = xhalf ? sx[j] : sy[j];
          const float p0 = __shfl_xor(v0[j], 16);
          v0[j] = (l32 < 16) ? (v0[j] * c - p0 * sn) : (v0[j] * c + p0 * sn);
        }
      }
    }
    if (flags & EPI_GELU) {
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        v0[j] = gelu_tanh(v0[j]);
        if constexpr (NB == 2) v1[j] = gelu_tanh(v1[j]);
      }
    }
    if (flags & EPI_RELU) {
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        v0[j] = fmaxf(v0[j], 0.f);
        v1[j] = fmaxf(v1[j], 0.f);
      }
    }
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      srow[(8 * g + j) * SS] = v0[j];
      if constexpr (NB == 2) srow[(8 * g + j) * SS + 32] = v1[j];
    }
  }
  epi_store<false, NB>(p, flags, row0, col0, stage, lane);
}

// a * b + c in two roundings: the operation without a contraction into a multiply-add.
__device__ __forceinline__ float mul_add_sep(float a, float b, float c) {
#pragma clang fp contract(off)
  return a * b + c;
}

// Row epilogue for accumulators of the transposed product (the weight fragment
// as the MFMA's first operand): lane l32 holds row row0 + l32 and register
// 4 g + j of q0 (q1) its column col0 (+ 32) + 8 g + 4 hl + j, so the stage is
// written 16 bytes at a time (a quarter of w2_epi_row's LDS writes), the two
// elements a RoPE rotation joins lie in one lane, and a lane decodes one
// position per block row. Same per-element operations and order as w2_epi_row.
template <bool ROPE>
__device__ __forceinline__ void w2_epi_row_t(const GemmArgs& p, const floatx16& q0,
                                             const floatx16& q1, int row0, int col0, float* stage,
                                             int lane, int l32, int hl) {
  const int flags = ROPE ? p.flags & ~(EPI_RES1 | EPI_RES2) : p.flags & ~EPI_ROPE;
  float* const srow = stage + l32 * W2_SS + 4 * hl;
  if (ROPE && col0 < p.rope_ncols) {
    int tok, tx;
    divmod_small(min(row0 + l32, p.M - 1), p.tok_per_img, 1.0f / (float)p.tok_per_img, tok);
    const int ty = divmod_small(tok, p.grid_w, 1.0f / (float)p.grid_w, tx);
    // all table and bias reads of the block row at once, 16 bytes each (with one
    // scalar read per element: 16384 x 3072 x 1024 149 us instead of 110)
    typedef float fx4u __attribute__((ext_vector_type(4), aligned(4)));
    fx4u cy[2], sy[2], cx[2], sx[2], bv[8] = {};
#pragma unroll
    for (int g = 0; g < 2; ++g) {
      const int fy = ty * 16 + 8 * g + 4 * hl, fx = tx * 16 + 8 * g + 4 * hl;
      cy[g] = *(const fx4u*)(p.rope_cos + fy);
      sy[g] = *(const fx4u*)(p.rope_sin + fy);
      cx[g] = *(const fx4u*)(p.rope_cos + fx);
      sx[g] = *(const fx4u*)(p.rope_sin + fx);
    }
    if (flags & EPI_BIAS) {
#pragma unroll
      for (int g = 0; g < 8; ++g) bv[g] = *(const fx4u*)(p.bias + col0 + 8 * g + 4 * hl);
    }
    // registers 4 g + j and 4 (g + 2) + j: frequency 8 g + 4 hl + j of the
    // axis (q0: y, q1: x)
#pragma unroll
    for (int g = 0; g < 2; ++g) {
      float r[4][4];  // y low / high, x low / high half
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        float y0 = q0[4 * g + j], y1 = q0[4 * g + 8 + j];
        float x0 = q1[4 * g + j], x1 = q1[4 * g + 8 + j];
        if (flags & EPI_BIAS) {
          y0 = y0 + bv[g][j];
          y1 = y1 + bv[g + 2][j];
          x0 = x0 + bv[g + 4][j];
          x1 = x1 + bv[g + 6][j];
        }
        // the rounding of w2_epi_row (the sine product rounded, the cosine's in the
        // multiply-add), or with EPI_ROPE_SEP that of gemm_epilogue_t (both rounded)
        const float s0 = -(y1 * sy[g][j]), s1 = y0 * sy[g][j];
        const float s2 = -(x1 * sx[g][j]), s3 = x0 * sx[g][j];
        if (flags & EPI_ROPE_SEP) {
          r[0][j] = mul_add_sep(y0, cy[g][j], s0);
          r[1][j] = mul_add_sep(y1, cy[g][j], s1);
          r[2][j] = mul_add_sep(x0, cx[g][j], s2);
          r[3][j] = mul_add_sep(x1, cx[g][j], s3);
        } else {
          r[0][j] = __builtin_fmaf(y0, cy[g][j], s0);
          r[1][j] = __builtin_fmaf(y1, cy[g][j], s1);
          r[2][j] = __builtin_fmaf(x0, cx[g][j], s2);
          r[3][j] = __builtin_fmaf(x1, cx[g][j], s3);
        }
      }
#pragma unroll
      for (int h = 0; h < 4; ++h)
        *(fx4*)(srow + 8 * g + 16 * h) =
            epi_act(mk4(r[h][0], r[h][1], r[h][2], r[h][3]), flags);
    }
    epi_store<false, 2>(p, flags, row0, col0, stage, lane);
    return;
  }
#pragma unroll
  for (int g = 0; g < 4; ++g) {
    *(fx4*)(srow + 8 * g) = mk4(q0[4 * g], q0[4 * g + 1], q0[4 * g + 2], q0[4 * g + 3]);
    *(fx4*)(srow + 8 * g + 32) = mk4(q1[4 * g], q1[4 * g + 1], q1[4 * g + 2], q1[4 * g + 3]);
  }
  epi_store<true, 2>(p, flags, row0, col0, stage, lane);
}

// 64 zero bytes: the source of a padded conv tap's 16-byte loads
__device__ __attribute__((aligned(64))) float g_zero16[16] = {};

bool aligned16(const void* ptr) { return ((uintptr_t)ptr & 15) == 0; }

// The staged epilogue of the one-wave-per-SIMD kernels stores 4 columns per
// lane with vector accesses, at 32-bit byte offsets within a block of 32 rows
// (kRowEpiMaxLdc).
bool row_epi_ok(const GemmArgs& g) {
  if (g.flags & EPI_SCATTER)  // 4-column segments stay within one output pixel
    return g.sc_C % 4 == 0 && g.sc_Cout % 4 == 0 && g.N % 4 == 0 && aligned16(g.C) &&
           !(g.flags & (EPI_RES1 | EPI_RES2 | EPI_ROPE | EPI_DUAL));
  if (g.N % 4 || g.ldc % 4 || !aligned16(g.C)) return false;
  if (g.ldc > kRowEpiMaxLdc) return false;
  if ((g.flags & EPI_RES1) && (g.ldr1 % 4 || !aligned16(g.R1))) return false;
  if ((g.flags & EPI_RES2) && (g.ldr2 % 4 || !aligned16(g.R2))) return false;
  if ((g.flags & EPI_DUAL) && !aligned16(g.C2)) return false;
  return true;
}

}  // namespace
}  // namespace gs
