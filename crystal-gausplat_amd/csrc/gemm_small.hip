// Small linears of the op-level entry points: launches of at most kSmallMaxTiles
// 32 x 32 output tiles, whose time is launches, allocations and the latency of one
// workgroup's K loop.
//
// One workgroup per 32 x 32 tile, K cut over its NW waves: a wave reads its rows of
// x and W straight into MFMA fragments (16 bytes per lane and load, no LDS, several
// loads in flight), multiplies them in the call's arithmetic, and the waves' sums are
// added in wave order through LDS before the epilogue. So there is one launch and no
// scratch: no split-K reduce pass, no bf16 copies of the operands.
// M x K x N, before and after, a call in a stream of calls: fp32 256 x 512 x 256 24.1 ->
// 7.7 us, 32 x 1024 x 4096 24.4 -> 11.5, 512 x 1024 x 1024 25.2 -> 20.1; bf16 256 x 512 x 256
// 31.4 -> 6.8, bf16x6 23.6 -> 7.0. A fragment load touches 32 rows for 32 bytes each, so
// long K is bound by the cache's tag rate: 256 x 2048 x 512 23.2 -> 18-20 us, but K = 4096
// lost (27 -> 33), and more tiles or longer K stay on the LDS-staged kernels.
#include <type_traits>

#include "bf16_split.h"
#include "gemm_device.h"
#include "internal.h"

namespace gs {
namespace {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));

// 8 consecutive k of a row as bf16 (nearest even), or as the three terms of the
// bf16x6 products.
__device__ __forceinline__ bf16x8 to_bf16(const fx4& u, const fx4& v) {
  const u32x4 h = {cvt_pk_bf16(u.x, u.y), cvt_pk_bf16(u.z, u.w), cvt_pk_bf16(v.x, v.y),
                   cvt_pk_bf16(v.z, v.w)};
  return __builtin_bit_cast(bf16x8, h);
}
__device__ __forceinline__ void to_bf16x3(const fx4& u, const fx4& v, bf16x8 (&t)[3]) {
  const float x[8] = {u.x, u.y, u.z, u.w, v.x, v.y, v.z, v.w};
  u32x4 h, m, l;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    uint32_t a, b, c;
    split3_pk(x[2 * i], x[2 * i + 1], a, b, c);
    h[i] = a;
    m[i] = b;
    l[i] = c;
  }
  t[0] = __builtin_bit_cast(bf16x8, h);
  t[1] = __builtin_bit_cast(bf16x8, m);
  t[2] = __builtin_bit_cast(bf16x8, l);
}

constexpr int kSmallStride = 36;  // floats per row of a wave's sums in LDS

// PREC: 0 fp32 MFMA, 1 bf16, 2 bf16x6. A step is 16 of k: lane half h reads k
// 8h .. 8h + 7 of its row of x (A) and of W (B); the fp32 MFMA of step t takes
// k = t and 8 + t.
template <int NW, int PREC>
__global__ __launch_bounds__(64 * NW) void linear_small_kernel(GemmArgs p) {
  constexpr int U = 4;  // steps whose loads are in flight together
  __shared__ __attribute__((aligned(16))) float sums[NW][32 * kSmallStride];
  const int M = p.M, N = p.N;
  const int tiles_n = (N + 31) / 32;
  const int m0 = (int)(blockIdx.x / tiles_n) * 32, n0 = (int)(blockIdx.x % tiles_n) * 32;
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int l32 = lane & 31, hl = lane >> 5;
  const float* a = p.A + (int64_t)min(m0 + l32, M - 1) * p.lda + 8 * hl;
  const float* b = p.B + (int64_t)min(n0 + l32, N - 1) * p.ldb + 8 * hl;
  const int steps = p.K / 16;
  const int s0 = steps * wave / NW, s1 = steps * (wave + 1) / NW;
  floatx16 acc = {};
  // NS steps: all their loads first, then the products
  auto run = [&](int s, auto count) {
    constexpr int NS = decltype(count)::value;
    fx4 ra[NS][2], rb[NS][2];
#pragma unroll
    for (int u = 0; u < NS; ++u) {
      ra[u][0] = *(const fx4*)(a + 16 * (s + u));
      ra[u][1] = *(const fx4*)(a + 16 * (s + u) + 4);
      rb[u][0] = *(const fx4*)(b + 16 * (s + u));
      rb[u][1] = *(const fx4*)(b + 16 * (s + u) + 4);
    }
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int u = 0; u < NS; ++u) {
      if constexpr (PREC == 0) {
#pragma unroll
        for (int t = 0; t < 8; ++t)
          acc = __builtin_amdgcn_mfma_f32_32x32x2f32(ra[u][t >> 2][t & 3], rb[u][t >> 2][t & 3], acc,
                                                     0, 0, 0);
      } else if constexpr (PREC == 1) {
        acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(to_bf16(ra[u][0], ra[u][1]),
                                                      to_bf16(rb[u][0], rb[u][1]), acc, 0, 0, 0);
      } else {
        bf16x8 x[3], w[3];
        to_bf16x3(ra[u][0], ra[u][1], x);
        to_bf16x3(rb[u][0], rb[u][1], w);
        // smallest terms first
        acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(x[2], w[0], acc, 0, 0, 0);
        acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(x[0], w[2], acc, 0, 0, 0);
        acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(x[1], w[1], acc, 0, 0, 0);
        acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(x[1], w[0], acc, 0, 0, 0);
        acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(x[0], w[1], acc, 0, 0, 0);
        acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(x[0], w[0], acc, 0, 0, 0);
      }
    }
  };
  int s = s0;
  for (; s + U <= s1; s += U) run(s, std::integral_constant<int, U>());
  for (; s < s1; ++s) run(s, std::integral_constant<int, 1>());
#pragma unroll
  for (int r = 0; r < 16; ++r)
    sums[wave][(8 * (r >> 2) + 4 * hl + (r & 3)) * kSmallStride + l32] = acc[r];
  __syncthreads();
  // 256 threads: row tid / 8, columns 4 (tid % 8) .. + 3
  if (tid >= 256) return;
  const int row = m0 + (tid >> 3), col = n0 + 4 * (tid & 7);
  if (row >= M || col >= N) return;
  const int at = (tid >> 3) * kSmallStride + 4 * (tid & 7);
  fx4 v = *(const fx4*)&sums[0][at];
#pragma unroll
  for (int w = 1; w < NW; ++w) v = v + *(const fx4*)&sums[w][at];
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    if (col + i >= N) break;
    float x = v[i];
    if (p.flags & EPI_BIAS) x = x + p.bias[col + i];
    if (p.flags & EPI_GELU) x = gelu_tanh(x);
    if (p.flags & EPI_RELU) x = fmaxf(x, 0.f);
    if (p.flags & EPI_RES1) x = x + p.R1[(int64_t)row * p.ldr1 + col + i];
    p.C[(int64_t)row * p.ldc + col + i] = x;
  }
}

}  // namespace

bool linear_small_ok(int64_t M, int64_t N, int64_t K) {
  return ((M + 31) / 32) * ((N + 31) / 32) <= kSmallMaxTiles && K <= kSmallMaxK;
}

int launch_linear_small(const GemmArgs& a, int prec, hipStream_t s) {
  GS_REQUIRE(linear_small_ok(a.M, a.N, a.K) && a.M > 0 && a.N > 0 && a.K > 0 && a.K % 32 == 0 &&
                 a.lda >= a.K && a.ldb >= a.K && a.lda % 4 == 0 && a.ldb % 4 == 0 && a.ldc >= a.N &&
                 aligned16(a.A) && aligned16(a.B) && a.C && prec >= 0 && prec <= 2 &&
                 (!(a.flags & EPI_BIAS) || a.bias) && (!(a.flags & EPI_RES1) || a.R1) &&
                 !(a.flags & ~(EPI_BIAS | EPI_GELU | EPI_RELU | EPI_RES1)),
             "linear_small: bad arguments");
  const dim3 grid((unsigned)(((a.M + 31) / 32) * ((a.N + 31) / 32)));
  hipEvent_t ev = prof_start(s);
  // waves: at most eight steps of K each
#define GS_SMALL(NW, P) hipLaunchKernelGGL((linear_small_kernel<NW, P>), grid, dim3(64 * NW), 0, s, a)
#define GS_SMALL_NW(P)      \
  if (a.K <= 256)           \
    GS_SMALL(4, P);         \
  else if (a.K <= 1024)     \
    GS_SMALL(8, P);         \
  else                      \
    GS_SMALL(16, P);
  if (prec == 0) {
    GS_SMALL_NW(0)
  } else if (prec == 1) {
    GS_SMALL_NW(1)
  } else {
    GS_SMALL_NW(2)
  }
#undef GS_SMALL_NW
#undef GS_SMALL
  GS_CHECK_HIP(hipGetLastError());
  if (ev)
    prof_stop(s, ev, prec == 0 ? "linear_small_kernel" : prec == 1 ? "linear_small_kernel<bf16>" : "linear_small_x6_kernel",
              2.0 * a.M * (double)a.N * a.K, 4.0 * ((double)a.M * a.K + (double)a.N * a.K + (double)a.M * a.N));
  return 0;
}

}  // namespace gs
