// bf16-input / fp32-accumulate GEMMs and implicit convolutions whose A is bf16
// (plain rows or an NHWC image) and whose weights are NT bf16 rows.
#include <algorithm>
#include <utility>

#include "gemm_device.h"

namespace gs {
namespace {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));

// Workgroup tile BM x BN of WVM x WVN waves, each (BM / WVM) x (BN / WVN) in MFMA
// 32x32x16 blocks; KS-deep K steps streamed straight into one of NST LDS stages
// (global_load_lds_dwordx4).
//
// What keeps the matrix cores waiting bounds it: at 24576 x 4096 x 1024 they are
// busy 41 % of the time at 2.05 GHz, and waves wait 43-46 % of their cycles. So:
// - One barrier per K step. A wave passes it with the last fragments of step k in
//   registers, and with all its reads of that stage done: the stage is refilled
//   with step k + NST at once, and step k + 1's first fragments are read under the
//   MFMAs of step k's last ones. Inside a step the fragments of slice s + 1 are
//   read under the MFMAs of slice s.
// - 64-deep steps: half the barriers per MFMA of 32-deep ones, and a 128-byte line
//   of every row per step.
// - 256 x 256 tiles at eight waves of 128 x 64 for launches that fill the chip: a
//   third less LDS-bound traffic per MFMA than 256 x 128. They have the CU alone,
//   so nothing runs under their epilogue (5-12 us of a K = 1024 tile's 35-42);
//   128 x 128 (two workgroups per CU) and 64 x 128 (three) serve the rest.
// - The transposed product (weight fragment first), so that the epilogue finds four
//   consecutive columns in a lane (w2_epi_row_t).
// The K order of every output is that of one accumulator over ascending 16-deep
// slices, so all tiles give the same bits unless K is split.
// Against the 256 x 128 kernel with two barriers per 32-deep step and the
// register-staged 128 x 128 kernel (split in K for small launches) it replaces, us:
//   16384 x 1024, K = 4096, residual   183 -> 138 (996 TFLOP/s)
//   16384 x 3072, K = 1024             127 -> 113
//   24576 x 4096, K = 1024, GELU       255 -> 232
//   12288 x 6144, K = 7168            1198 -> 960 (1127 TFLOP/s)
//   2048 x 1024, K = 1024, residual   25.6 -> 26.3 (same split of K)
// A 256 x 256 tile of four waves (128 x 128 each, one per SIMD) took 351 us at
// 24576 x 4096 x 1024: nothing to run while its only wave waits.
// Raised wave priority around the MFMAs: 256 x 256 tiles 3-5 % slower.
//
// LDS rows are KS bf16. Chunk c (16 bytes) of row r sits at slot c ^ sw(r), sw over
// the rows of one 256-byte bank line, so 16 consecutive rows read at one chunk hit
// 16 distinct bank groups. Lane l (half h) feeds slice s with k = 16 s + 8 h .. + 7.
// CONV: a K step is KS channels of one tap (cCin % KS == 0), padded taps load from
// g_zero16. A split launch gives each blockIdx.y one K range and stores its raw
// partial for gemm_splitk_reduce.
template <int BM, int BN, int WVM, int WVN, int KS, int NST, int OCC, bool CONV>
__global__ __launch_bounds__(64 * WVM * WVN, OCC) void gemm_bf16_pipe_kernel(GemmBatch batch) {
  constexpr int NW = WVM * WVN, WTM = BM / WVM / 32, WTN = BN / WVN / 32, NS = KS / 16;
  constexpr int CH = KS / 8, RPI = 64 / CH;  // 16-byte chunks per row, rows per load
  constexpr int STAGE = (BM + BN) * KS;      // bf16 per LDS stage
  constexpr int LA = BM / RPI / NW, LB = BN / RPI / NW, LPS = LA + LB;  // loads per wave and step
  static_assert(WTM * WVM * 32 == BM && WTN * WVN * 32 == BN && WTN % 2 == 0, "wave tiles");
  static_assert(LA * RPI * NW == BM && LB * RPI * NW == BN, "loads per wave");
  static_assert(KS == 64 || KS == 32, "swizzles below");
  static_assert(NW * 32 * W2_SS * 4 <= NST * STAGE * 2, "epilogue stages fit the LDS stages");
  const GemmArgs& p = batch.g[blockIdx.z];
  const int M = p.M, N = p.N;
  const int tiles_m = (M + BM - 1) / BM, tiles_n = (N + BN - 1) / BN;
  int bid = blockIdx.x;
  if ((gridDim.x & 7) == 0) bid = (bid & 7) * (gridDim.x >> 3) + (bid >> 3);  // one XCD, one run
  if (bid >= tiles_m * tiles_n) return;
  const int per_group = GROUP_M * tiles_n;
  const int first_m = bid / per_group * GROUP_M;
  const int gsz = min(tiles_m - first_m, GROUP_M);
  const int m0 = (first_m + (bid % per_group) % gsz) * BM, n0 = (bid % per_group) / gsz * BN;
  int kbeg, kend;
  split_range(p.K, batch.ksplit, KS, kbeg, kend);
  __shared__ __attribute__((aligned(16))) __bf16 lds[NST * STAGE];

  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wm = wave / WVN, wn = wave % WVN, l32 = lane & 31, hl = lane >> 5;
  // loader: wave w, instruction i fills rows RPI (NW i + w) .. of A, then of B
  const int rin = lane / CH;
  auto sw = [](int r) { return KS == 64 ? (r >> 1) & 7 : (r >> 2) & 3; };
  constexpr auto la = std::make_integer_sequence<int, LA>();
  constexpr auto lb = std::make_integer_sequence<int, LB>();
  const __bf16* ag[LA];
  const __bf16* bg[LB];
  int ohs[LA], ows[LA];
  const_for(la, [&](auto i) {
    const int r = RPI * (NW * i + wave) + rin, chunk = (lane % CH) ^ sw(r);
    const int64_t m = min(m0 + r, M - 1);
    if constexpr (CONV) {
      const int hw = p.cHo * p.cWo;
      const int img = (int)(m / hw), rem = (int)(m - (int64_t)img * hw);
      const int oh = rem / p.cWo, ow = rem - oh * p.cWo;
      const int ih0 = oh * p.cs - p.cp;
      ows[i] = ow * p.cs - p.cp;
      ag[i] = (const __bf16*)p.A + (((int64_t)img * p.cH + ih0) * p.cW + ows[i]) * p.cCin + 8 * chunk;
      ohs[i] = m0 + r < M ? ih0 : -(1 << 20);  // rows past M: never in bounds
    } else {
      ag[i] = (const __bf16*)p.A + m * p.lda + 8 * chunk;
    }
  });
  const_for(lb, [&](auto i) {
    const int r = RPI * (NW * i + wave) + rin, chunk = (lane % CH) ^ sw(r);
    bg[i] = (const __bf16*)p.Bh + (int64_t)min(n0 + r, N - 1) * p.ldb + 8 * chunk;
  });
  const uint32_t lds0 = lds_addr((const float*)lds);
  // conv tap of the next step to issue (wave-uniform)
  int tkh = 0, tkw = 0, tic = 0;
  if constexpr (CONV) {
    const int tap = kbeg / p.cCin;
    tic = kbeg - tap * p.cCin;
    tkh = tap / p.ckw;
    tkw = tap - tkh * p.ckw;
  }
  auto issue = [&](int buf, int k0) {
    const uint32_t dst = lds0 + (buf * STAGE + RPI * wave * KS) * 2;
    if constexpr (CONV) {
      const int64_t toff = ((int64_t)tkh * p.cW + tkw) * p.cCin + tic;
      const_for(la, [&](auto i) {
        const bool ok = (unsigned)(ohs[i] + tkh) < (unsigned)p.cH &&
                        (unsigned)(ows[i] + tkw) < (unsigned)p.cW;
        lds_dma16(ok ? (const float*)(ag[i] + toff) : g_zero16, dst + RPI * NW * i * KS * 2);
      });
      tic += KS;
      if (tic == p.cCin) {
        tic = 0;
        if (++tkw == p.ckw) {
          tkw = 0;
          ++tkh;
        }
      }
    } else {
      const_for(la, [&](auto i) {
        lds_dma16((const float*)(ag[i] + k0), dst + RPI * NW * i * KS * 2);
      });
    }
    const_for(lb, [&](auto i) {
      lds_dma16((const float*)(bg[i] + k0), dst + (BM + RPI * NW * i) * KS * 2);
    });
  };

  constexpr auto wtm = std::make_integer_sequence<int, WTM>();
  constexpr auto wtn = std::make_integer_sequence<int, WTN>();
  floatx16 acc[WTM][WTN] = {};
  bf16x8 fa[2][WTM], fb[2][WTN];
  const int ra0 = (wm * 32 * WTM + l32) * KS, rb0 = (BM + wn * 32 * WTN + l32) * KS;
  auto read = [&](auto f, int buf, auto s) {
    const __bf16* st = lds + buf * STAGE;
    const int co = ((2 * s + hl) ^ sw(l32)) << 3;
    const_for(wtn, [&](auto j) { fb[f][j] = *(const bf16x8*)(st + rb0 + j * 32 * KS + co); });
    const_for(wtm, [&](auto i) { fa[f][i] = *(const bf16x8*)(st + ra0 + i * 32 * KS + co); });
  };
  const std::integral_constant<int, 0> zero;
  const int nk = (kend - kbeg) / KS;
  const_for(std::make_integer_sequence<int, NST>(), [&](auto i) {
    if (i < nk) issue(i, kbeg + i * KS);
  });
  // step 0 landed for every wave; later steps stay in flight where all were issued
  if (nk >= NST)
    asm volatile("s_waitcnt vmcnt(%0)\n\ts_barrier" ::"n"((NST - 1) * LPS) : "memory");
  else
    asm volatile("s_waitcnt vmcnt(0)\n\ts_barrier" ::: "memory");
  read(zero, 0, zero);
  int buf = 0;
  for (int k = 0; k < nk; ++k) {
    const_for(std::make_integer_sequence<int, NS>(), [&](auto s) {
      constexpr int cu = s & 1;
      const std::integral_constant<int, cu ^ 1> nx;
      if constexpr (s + 1 < NS) {
        read(nx, buf, std::integral_constant<int, s + 1>());
      } else if (k + 1 < nk) {
        // this wave's loads of step k + 1 have landed (those of the NST - 2 steps
        // after it may be in flight) and its reads of step k are done; past the
        // barrier that holds for all waves, and step k's stage is free
        if (k + NST <= nk)
          asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"((NST - 2) * LPS) : "memory");
        else
          asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory");
        const int nb = buf + 1 == NST ? 0 : buf + 1;
        read(nx, nb, zero);
        if (k + NST < nk) issue(buf, kbeg + (k + NST) * KS);
        buf = nb;
      }
      const_for(wtm, [&](auto i) {
        const_for(wtn, [&](auto j) {
          acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(fb[cu][j], fa[cu][i], acc[i][j], 0, 0, 0);
        });
      });
      __builtin_amdgcn_sched_barrier(0);
    });
  }
  const int mw = m0 + wm * 32 * WTM, nw = n0 + wn * 32 * WTN;
  if (batch.ksplit > 1) {
    float* part = p.part + (int64_t)blockIdx.y * M * N;
    const_for(wtm, [&](auto i) {
      const int row = mw + 32 * i + l32;
      const_for(wtn, [&](auto j) {
#pragma unroll
        for (int g = 0; g < 4; ++g) {
          const int col = nw + 32 * j + 8 * g + 4 * hl;
          const floatx16& c = acc[i][j];
          if (row < M && col < N)
            *(fx4*)(part + (int64_t)row * N + col) = mk4(c[4 * g], c[4 * g + 1], c[4 * g + 2], c[4 * g + 3]);
        }
      });
    });
    return;
  }
  // the epilogue stages overlay the LDS stages: every wave's last reads first
  asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
  float* stage = (float*)lds + wave * 32 * W2_SS;
  const_for(std::make_integer_sequence<int, WTM * WTN / 2>(), [&](auto ix) {
    constexpr int i = ix / (WTN / 2), j = 2 * (ix % (WTN / 2));
    if (p.flags & EPI_ROPE)
      w2_epi_row_t<true>(p, acc[i][j], acc[i][j + 1], mw + 32 * i, nw + 32 * j, stage, lane, l32, hl);
    else
      w2_epi_row_t<false>(p, acc[i][j], acc[i][j + 1], mw + 32 * i, nw + 32 * j, stage, lane, l32, hl);
  });
}

// Tiles, with the time (us) of 64 of K: lat of a workgroup alone on its CU, thr its
// share of a CU that several keep busy; epi per tile besides.
struct PipeTile {
  int bm, bn, threads;
  float lat, thr, epi;
};
constexpr PipeTile kPipeTiles[] = {{256, 256, 512, 1.8f, 1.8f, 7.0f},
                                   {128, 128, 256, 0.66f, 0.60f, 0.9f},
                                   {64, 128, 256, 0.45f, 0.36f, 0.7f}};
constexpr int kPipeNumTiles = 3;
constexpr int kCUs = 256;  // MI355X compute units

// 64-deep K steps, or 32-deep ones where a row (of a conv: a tap) is no multiple of 64
bool pipe_deep(const GemmBatch& b, bool conv) {
  for (int i = 0; i < b.ngroups; ++i)
    if ((conv ? b.g[i].cCin : b.g[i].K) % 64) return false;
  return true;
}

}  // namespace

bool bf16_pipe_eligible(const GemmBatch& b, int aload, bool a_relu) {
  if ((aload != A_PLAIN_H && aload != A_CONV_H) || a_relu) return false;
  for (int i = 0; i < b.ngroups; ++i) {
    const GemmArgs& g = b.g[i];
    if (g.K % 32 || (aload == A_CONV_H ? g.cCin % 32 : g.lda % 8) || !aligned16(g.A) || g.ldb % 8 ||
        !aligned16(g.Bh) || !row_epi_ok(g) || ((g.flags & EPI_ROPE) && g.rope_ncols % 64))
      return false;
  }
  return true;
}

// Tile of a launch whose K is cut into b.ksplit ranges: the tiles of a CU (between
// the mean and the busiest CU's) times their time.
int plan_bf16_pipe(const GemmBatch& b, int aload) {
  const int ks = pipe_deep(b, aload == A_CONV_H) ? 64 : 32, S = std::max(b.ksplit, 1);
  const double k64 = (b.g[0].K / ks + S - 1) / S * ks / 64.0;
  double best = 0.0;
  int tile = 0;
  for (int c = 0; c < kPipeNumTiles; ++c) {
    const PipeTile& t = kPipeTiles[c];
    int64_t tiles = 0;
    for (int i = 0; i < b.ngroups; ++i)
      tiles += (int64_t)((b.g[i].M + t.bm - 1) / t.bm) * ((b.g[i].N + t.bn - 1) / t.bn);
    const double mean = (double)tiles * S / kCUs, most = (double)((tiles * S + kCUs - 1) / kCUs);
    const double cost = std::max(t.epi + k64 * t.lat, 0.5 * (mean + most) * (t.epi + k64 * t.thr));
    if (c == 0 || cost < best) {
      best = cost;
      tile = c;
    }
  }
  return tile;
}

int launch_bf16_pipe(const GemmBatch& b, int aload, int tile, hipStream_t s) {
  GS_REQUIRE(bf16_pipe_eligible(b, aload, false) && tile >= 0 && tile < kPipeNumTiles && b.ksplit >= 1,
             "gemm: this launch cannot run on the streaming bf16 kernel");
  const bool conv = aload == A_CONV_H, deep = pipe_deep(b, conv);
  const PipeTile& t = kPipeTiles[tile];
  int n = 0;
  for (int i = 0; i < b.ngroups; ++i)
    n = std::max(n, ((b.g[i].M + t.bm - 1) / t.bm) * ((b.g[i].N + t.bn - 1) / t.bn));
  const dim3 grid(n, b.ksplit, b.ngroups), block(t.threads);
#define GS_PIPE(BM_, BN_, WM_, WN_, OCC_)                                                            \
  if (t.bm == BM_ && t.bn == BN_) {                                                                  \
    if (conv && deep)                                                                                \
      hipLaunchKernelGGL((gemm_bf16_pipe_kernel<BM_, BN_, WM_, WN_, 64, 2, OCC_, true>), grid, block, 0, s, b);  \
    else if (conv)                                                                                   \
      hipLaunchKernelGGL((gemm_bf16_pipe_kernel<BM_, BN_, WM_, WN_, 32, 3, OCC_, true>), grid, block, 0, s, b);  \
    else if (deep)                                                                                   \
      hipLaunchKernelGGL((gemm_bf16_pipe_kernel<BM_, BN_, WM_, WN_, 64, 2, OCC_, false>), grid, block, 0, s, b); \
    else                                                                                             \
      hipLaunchKernelGGL((gemm_bf16_pipe_kernel<BM_, BN_, WM_, WN_, 32, 3, OCC_, false>), grid, block, 0, s, b); \
  }
  GS_PIPE(256, 256, 2, 4, 2)
  GS_PIPE(128, 128, 2, 2, 2)
  GS_PIPE(64, 128, 2, 2, 3)
#undef GS_PIPE
  GS_CHECK_HIP(hipGetLastError());
  return 0;
}

}  // namespace gs
