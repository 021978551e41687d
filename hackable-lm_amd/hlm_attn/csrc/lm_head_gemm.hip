// dhidden of the LM head's fused linear + cross-entropy: C = G W, with G the
// chunk's logit gradients (M rows x K = vocabulary) and W the head's weight (K
// rows x N = hidden size), bf16 in, fp32 sums, bf16 out -- the product that
// hackable-lm's chunk loop forms as `grad_logits @ weight` (kernels.py:878-942).
//
// K is the vocabulary, so C has few 256 x 256 tiles (48 for 4096 rows of 768)
// and long sums; a product that gives each tile to one CU leaves most of the
// chip idle (the library's: 320 us at K = 32768, 640 TFLOP/s).  Here S
// workgroups share a tile, each summing a run of K, and a second kernel adds
// their fp32 partial tiles in a fixed order.  Both kernels over fresh chunks of
// G: 184-194 us, 1060-1120 TFLOP/s, 12 of them the sum (K = 50257: 450 -> 277-290;
// 904 rows: 265 -> 118); inside the loss 193 + 12 us, the matrix cores 53% busy,
// no bank conflicts, 390 MB read of 318.  What bounds the first kernel is its
// feed: 64 KB per CU and 64-deep step against 2048 cycles of products.
//
// G's rows should not be a multiple of 4 KB apart: the 256 rows of a tile
// then fall on few memory channels (220 us instead of 184).
#include <algorithm>

#include "attn_common.h"

namespace hlm {

struct DhiddenArgs {
  const bf16* g;  // M rows, stride ldg; columns K .. round_up(K, 64) - 1 hold zeros
  const bf16* w;  // K rows, stride ldw
  bf16* c;        // M rows, stride ldc
  float* part;    // S > 1: S partial tiles per tile of C
  int64_t ldg, ldw, ldc;
  int M, N, K;
  int mt, nt, S, per;  // tiles of C, runs of K, 64-wide steps per run
};

constexpr int kGemmTile = 256, kGemmStep = 64, kGemmThreads = 512;

// Offset of a transposed operand's first (second = 0) or last 4 of the 8
// rows 8 (l / 32) + e of a 16-row step of a cs tile, for its 32 columns 32 db.
template <int D>
__device__ __forceinline__ int cs_tr_natural(int db, int second, int lane) {
  const int g = lane >> 4, rr = (lane >> 2) & 3, c = lane & 3;
  const int row = 8 * (g >> 1) + rr + 4 * second;
  const int col = 32 * db + 16 * (g & 1) + 4 * c;
  return CS<D>::byte(row, col >> 3) + 8 * ((col >> 2) & 1);
}

// One workgroup (8 waves, 2 x 4) per tile and run; a wave owns 128 rows x 64
// columns of C, held transposed (lanes own rows of C, four consecutive columns
// per accumulator quad): 0.75 KB of operand reads per product instead of the 1
// KB of a 64 x 64 wave tile, and the slower transposed reads (W) are the
// smaller part.  Steps of 64 along K pass through LDS as a G tile (256 x 64,
// cs<64>) and a W tile (64 x 256 as two cs<128> panels), copied as whole rows
// by LDS DMA.  G, which comes from HBM, has three stages and W, which other
// workgroups have brought into L2, two: all of the CU's LDS.
__global__ __launch_bounds__(kGemmThreads, 2) void lm_head_dhidden_kernel(DhiddenArgs a) {
  constexpr int NW = 8, GB = kGemmTile * kGemmStep * 2, WB = GB;  // bytes of a G and a W tile
  constexpr int GS = 3, WS = 2;                                   // stages of each
  __shared__ __attribute__((aligned(1024))) char lds[GS * GB + WS * WB];
  // Tiles of one run and row tile are neighbours on one XCD (they share G).
  const int xcd = blockIdx.x & 7, slot = blockIdx.x >> 3;
  const int units = a.mt * a.S, upx = (units + 7) / 8;
  const int unit = xcd * upx + slot / a.nt, ntile = slot % a.nt;
  if (slot / a.nt >= upx || unit >= units) return;
  const int run = unit / a.mt, mtile = unit % a.mt;
  const int m0 = mtile * kGemmTile, n0 = ntile * kGemmTile;
  const int steps_all = (a.K + kGemmStep - 1) / kGemmStep;
  const int t0 = run * a.per, steps = min(a.per, steps_all - t0);

  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int l32 = lane & 31, h32 = lane >> 5;
  const int wm = wave >> 2, wn = wave & 3;
  const unsigned base = lds_addr(lds);

  // Copies: 4 chunks of G (8 rows x 128 bytes) and 4 of W (4 rows x 256 bytes)
  // per wave and step; rows past M or K, and steps past the run's end, read
  // as zeros.
  const char* gp = reinterpret_cast<const char*>(a.g + (int64_t)m0 * a.ldg + (int64_t)t0 * kGemmStep);
  const char* wp = reinterpret_cast<const char*>(a.w + (int64_t)t0 * kGemmStep * a.ldw + n0);
  const int ldg2 = (int)(a.ldg * 2), ldw2 = (int)(a.ldw * 2);
  const int gext = min(kGemmTile, a.M - m0) * ldg2 - t0 * (kGemmStep * 2);
  const int krows = a.K - t0 * kGemmStep;
  int gof[4], wof[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int j = wave + NW * i;
    gof[i] = CS<64>::dma_row(j, lane) * ldg2 + CS<64>::dma_col_bytes(j, lane);
    const int jw = j & 15;  // chunk within panel j / 16
    wof[i] = CS<128>::dma_row(jw, lane) * ldw2 + CS<128>::dma_col_bytes(jw, lane) + (j >> 4) * 256;
    asm volatile("" : "+v"(gof[i]), "+v"(wof[i]));
  }
  auto g_rsrc = [&](int t) __attribute__((always_inline)) {
    return bytes_rsrc(gp + (int64_t)t * (kGemmStep * 2), t < steps ? gext - t * (kGemmStep * 2) : 0);
  };
  auto w_rsrc = [&](int t) __attribute__((always_inline)) {
    const int rows = min(krows - t * kGemmStep, kGemmStep);
    return bytes_rsrc(wp + (int64_t)t * kGemmStep * ldw2, t < steps ? (rows - 1) * ldw2 + (a.N - n0) * 2 : 0);
  };
  const unsigned gdst = base + wave * 1024, wdst = base + GS * GB + wave * 1024;

  unsigned ga[4], wa[2][2];  // LDS addresses of this lane's operands in stage 0
#pragma unroll
  for (int s = 0; s < 4; ++s) ga[s] = base + wm * 128 * 128 + CS<64>::byte(l32, 2 * s + h32);
#pragma unroll
  for (int nb = 0; nb < 2; ++nb)
#pragma unroll
    for (int k = 0; k < 2; ++k)
      wa[nb][k] = base + GS * GB + (wn >> 1) * (WB / 2) + cs_tr_natural<128>(2 * (wn & 1) + nb, k, lane);

  f32x16 acc[4][2];
#pragma unroll
  for (int mb = 0; mb < 4; ++mb)
#pragma unroll
    for (int nb = 0; nb < 2; ++nb) acc[mb][nb] = zero16();

  // Before the loop, in the loop's order: all of steps 0 .. GS - 2 and the
  // first two W copies of step WS - 1 (= 1).
  static_assert(WS == 2 && GS == 3, "the order of the copies, and the counts of the waits");
  {
    const __amdgpu_buffer_rsrc_t r0 = w_rsrc(0), r1 = w_rsrc(1);
#pragma unroll
    for (int i = 0; i < 4; ++i) lds_dma_at<16>(r0, wdst + NW * i * 1024, wof[i]);
#pragma unroll
    for (int t = 0; t < GS - 1; ++t) {
      const __amdgpu_buffer_rsrc_t r = g_rsrc(t);
#pragma unroll
      for (int i = 0; i < 4; ++i) lds_dma_at<16>(r, gdst + t * GB + NW * i * 1024, gof[i]);
    }
#pragma unroll
    for (int i = 0; i < 2; ++i) lds_dma_at<16>(r1, wdst + WB + NW * i * 1024, wof[i]);
  }
  bf16x8 go[2][4], wo[2][2];  // operands of one 16-deep slice, two in turn
  // Read i of 8 of a slice: the four transposed halves of W, then G's four.
  auto read_one = [&](int buf, int s, int i, unsigned goff, unsigned woff) __attribute__((always_inline)) {
    if (i < 2)
      wo[buf][i] = cs_operand_tr<128>(woff, (int)wa[i][0], (int)wa[i][1], 16 * s);
    else
      go[buf][i - 2] = cs_operand<64>(goff, (int)ga[s], i - 2);
  };
  auto product = [&](int buf, int i) __attribute__((always_inline)) {
    acc[i >> 1][i & 1] = mfma32(wo[buf][i & 1], go[buf][i >> 1], acc[i >> 1][i & 1]);
  };
  __amdgpu_buffer_rsrc_t rw, rg;
  // One slice: the 8 products of `buf` with the 6 operand reads of the next
  // slice and two of the 8 copies between them, so that no wave stands at a
  // full copy queue (64 copies of 16 cycles per CU and step) with its
  // products unissued.
  auto slice = [&](int buf, int s_next, unsigned goff, unsigned woff, int c0, unsigned dst) __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      product(buf, i);
      if (i < 6) read_one(buf ^ 1, s_next, i, goff, woff);
      __builtin_amdgcn_sched_barrier(0);
      if (i == 0 || i == 4) {
        const int c = c0 + i / 4;
        if (c < 4)
          lds_dma_at<16>(rw, wdst + dst + NW * c * 1024, wof[c]);
        else
          lds_dma_at<16>(rg, gdst + dst + NW * (c - 4) * 1024, gof[c - 4]);
        __builtin_amdgcn_sched_barrier(0);
      }
    }
  };
  dma_barrier<(GS - 2) * 4 + 2>();
#pragma unroll
  for (int i = 0; i < 6; ++i) read_one(0, 0, i, 0, 0);
  unsigned gst = 0, wst = 0;  // stage offsets of step it
  // Step it's last slice runs after the barrier that step it + 1 needs, so its
  // products cover the latency of that step's first reads.
  rw = w_rsrc(WS - 1);
  rg = g_rsrc(GS - 1);
  for (int it = 0; it < steps; ++it) {
    const unsigned wprev = WB - wst, gprev = gst == 0 ? (GS - 1) * GB : gst - GB, gnext = gst == (GS - 1) * GB ? 0 : gst + GB;
    slice(0, 1, gst, wst, 2, wprev);  // W copies 2, 3
    slice(1, 2, gst, wst, 4, gprev);  // G copies
    slice(0, 3, gst, wst, 6, gprev);
    // All reads of step it are done and the copies of step it + 1 have landed
    // (G(it + 2) may be in flight); past the barrier that holds for every
    // wave, and step it's stages are free.
    dma_barrier<(GS - 2) * 4>();
    rw = w_rsrc(it + WS);
    rg = g_rsrc(it + GS);
    slice(1, 0, gnext, wprev, 0, wst);  // W copies 0, 1 of step it + WS
    gst = gnext;
    wst = wprev;
  }
  dma_barrier<0>();  // copies past the run's end still write the stages

  // Lane (l32, h32) holds C[32 mb + l32][32 nb + 8 i + 4 h32 + j] of the wave's
  // block in acc[mb][nb][4 i + j].
  if (a.S > 1) {
    f32x4* dst = reinterpret_cast<f32x4*>(a.part) +
                 ((int64_t)run * a.mt * a.nt + mtile * a.nt + ntile) * (kGemmTile * kGemmTile / 4) + wave * (32 * 64) + lane;
#pragma unroll
    for (int mb = 0; mb < 4; ++mb)
#pragma unroll
      for (int nb = 0; nb < 2; ++nb)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          f32x4 v;
#pragma unroll
          for (int j = 0; j < 4; ++j) v[j] = acc[mb][nb][4 * i + j];
          dst[((mb * 2 + nb) * 4 + i) * 64] = v;
        }
    return;
  }
#pragma unroll
  for (int mb = 0; mb < 4; ++mb)
#pragma unroll
    for (int nb = 0; nb < 2; ++nb)
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int r = m0 + wm * 128 + 32 * mb + l32, n = n0 + wn * 64 + 32 * nb + 8 * i + 4 * h32;
        bf16x4 v;
#pragma unroll
        for (int j = 0; j < 4; ++j) v[j] = (bf16)acc[mb][nb][4 * i + j];
        if (r < a.M && n < a.N) *reinterpret_cast<bf16x4*>(a.c + (int64_t)r * a.ldc + n) = v;
      }
}

// Adds a tile's S partial tiles in their order.  One thread per accumulator
// quad (four columns of one row).
__global__ __launch_bounds__(256) void lm_head_dhidden_sum_kernel(DhiddenArgs a) {
  constexpr int QUADS = kGemmTile * kGemmTile / 4;
  const int tile = blockIdx.x / (QUADS / 256), q = (blockIdx.x % (QUADS / 256)) * 256 + threadIdx.x;
  const int lane = q & 63, i = (q >> 6) & 3, nb = (q >> 8) & 1, mb = (q >> 9) & 3, wave = q >> 11;
  const int r = (tile / a.nt) * kGemmTile + (wave >> 2) * 128 + 32 * mb + (lane & 31);
  const int n = (tile % a.nt) * kGemmTile + (wave & 3) * 64 + 32 * nb + 8 * i + 4 * (lane >> 5);
  if (r >= a.M || n >= a.N) return;
  const f32x4* src = reinterpret_cast<const f32x4*>(a.part) + (int64_t)tile * QUADS + q;
  const int64_t stride = (int64_t)a.mt * a.nt * QUADS;
  f32x4 sum = src[0];
  for (int s = 1; s < a.S; ++s) sum += src[s * stride];
  bf16x4 v;
#pragma unroll
  for (int j = 0; j < 4; ++j) v[j] = (bf16)sum[j];
  *reinterpret_cast<bf16x4*>(a.c + (int64_t)r * a.ldc + n) = v;
}

// Runs of K per tile: as many as one workgroup per CU takes, of at least 8
// steps.
int lm_head_dhidden_runs(int M, int N, int K) {
  const int64_t tiles = (int64_t)((M + 255) / 256) * ((N + 255) / 256);
  const int steps = (K + kGemmStep - 1) / kGemmStep;
  const int S = (int)std::min<int64_t>(std::max<int64_t>(256 / std::max<int64_t>(tiles, 1), 1), std::max(steps / 8, 1));
  const int per = (steps + S - 1) / S;
  return (steps + per - 1) / per;  // every run has work
}

// Whether the kernels above beat a product that does not split K: few tiles
// whose runs can fill the CUs, and a K that is long against what a split pays
// before its first and after its last product (12 us with 100 columns, where
// the library takes 5).  Kernel times in us, this / the library's (585 sizes,
// rows x hidden x vocabulary):
//   taken    4096 x 768 x 32768 194 / 319, x 6000 53 / 79; 272 x 256 x 4000 18 / 20;
//            4096 x 512 x 4000 38 / 43; 3000 x 768 x 6000 64 / 63; 4096 x 2048 x 6000 101 / 106
//   refused  by K: 272 x 256 x 900 25 / 9, x 3000 19 / 16; 4096 x 1024 x 2000 39 / 30, x 4000 52 / 51;
//            3000 x 768 x 4000 51 / 41; 4096 x 2048 x 4000 78 / 73
//            by the CUs: 8192 x 768 x 32768 (96 tiles, 192 workgroups) 405 / 390; more than 128 tiles
// (5600 rows of 768 or 1024, 66 and 88 tiles, are refused too and would gain
// 25% at 32768.)
bool lm_head_dhidden_pays(int M, int N, int K) {
  const int64_t tiles = (int64_t)((M + 255) / 256) * ((N + 255) / 256);
  if (tiles > 128 || tiles * (256 / tiles) < 205) return false;
  return (K + kGemmStep - 1) / kGemmStep >= (tiles <= 32 ? 63 : 94);
}

hipError_t launch_lm_head_dhidden(const void* g, int64_t ldg, const void* w, int64_t ldw, void* c, int64_t ldc, float* part,
                                  int M, int N, int K, hipStream_t stream) {
  DhiddenArgs a;
  a.g = static_cast<const bf16*>(g);
  a.w = static_cast<const bf16*>(w);
  a.c = static_cast<bf16*>(c);
  a.part = part;
  a.ldg = ldg;
  a.ldw = ldw;
  a.ldc = ldc;
  a.M = M;
  a.N = N;
  a.K = K;
  a.mt = (M + 255) / 256;
  a.nt = (N + 255) / 256;
  a.S = lm_head_dhidden_runs(M, N, K);
  const int steps = (K + kGemmStep - 1) / kGemmStep;
  a.per = (steps + a.S - 1) / a.S;
  const int upx = (a.mt * a.S + 7) / 8;
  hipLaunchKernelGGL(lm_head_dhidden_kernel, dim3((unsigned)(8 * upx * a.nt)), dim3(kGemmThreads), 0, stream, a);
  const hipError_t err = hipGetLastError();
  if (err != hipSuccess || a.S == 1) return err;
  hipLaunchKernelGGL(lm_head_dhidden_sum_kernel, dim3((unsigned)(a.mt * a.nt * (kGemmTile * kGemmTile / 4 / 256))), dim3(256), 0,
                     stream, a);
  return hipGetLastError();
}

}  // namespace hlm
