// Proven products whose operands the direct-to-LDS kernels cannot load: K no multiple of 16, rows that start at any byte,
// row strides of 8 MiB and more.
//
// What bounds them: the loads. Byte by byte (16 loads a chunk), on tiles chosen for large products, 16 x 3001 x 1000 took
// 74 us, 300 x 777 x 513 147, 4000 x 1001 x 1003 309 and 16000 x 3001 x 2999 2780. A lane's 16 bytes at any alignment are
// one load instruction as well (row_chunk, gemm.h), through registers instead of direct to LDS: 7.3, 7.4, 17 and 269 us.
// PF stages of 128 K bytes are in flight, and each is written to LDS, with the swizzle of gemm.h, one stage before its
// use. Rows past the operand repeat its last row, whose results are not stored, so only a K tail needs a branch. The
// epilogue runs from registers, as in gemm_deep.hip.
#include "gemm.h"

namespace anvil {

template <int BM, int BN, int PF, int OSZ, bool MUL24>
__global__ __launch_bounds__(256, 2) void gemm_i8_any(GemmArgs g) {
  constexpr int BK = 128, CPR = BK / 16, KS = BK / 32;
  constexpr int WM = BM / 2, WN = BN / 2, TM = WM / 32, TN = WN / 32;
  constexpr int JA = BM * CPR / 256, JB = BN * CPR / 256;
  constexpr int STAGE = (BM + BN) * BK;
  __shared__ __attribute__((aligned(16))) int8_t smem[2 * STAGE];
  __shared__ int8_t lut_s[256];

  const int t = threadIdx.x, lane = t & 63;
  const int wave = __builtin_amdgcn_readfirstlane(t >> 6), wm = wave >> 1, wn = wave & 1;
  const int half = lane >> 5, l32 = lane & 31;
  const int ntiles = g.tiles_m * g.tiles_n;
  int pid = blockIdx.x;
  if ((ntiles & 7) == 0) pid = (pid & 7) * (ntiles >> 3) + (pid >> 3);   // consecutive tiles on one XCD
  const int in_group = GROUP_M * g.tiles_n;
  const int first_m = (pid / in_group) * GROUP_M;
  const int gsize = min(g.tiles_m - first_m, GROUP_M);
  const int m0 = (first_m + (pid % in_group) % gsize) * BM, n0 = ((pid % in_group) / gsize) * BN;
  if (g.causal == 1 && n0 > m0 + BM - 1) return;
  const int b0 = blockIdx.y / g.batch1, b1 = blockIdx.y % g.batch1;
  const int K = g.causal == 2 ? min(g.K, m0 + BM) : g.K;
  if (g.lut) lut_s[t ^ 128] = g.lut[t];                  // rotated: the entry of v at index v & 255

  const int lr = t / CPR, lc = t % CPR;                  // this thread's chunk: row lr + 32 j, K bytes 16 lc
  const int8_t *pa[JA], *pb[JB];
#pragma unroll
  for (int j = 0; j < JA; ++j)
    pa[j] = g.A + b0 * g.sa0 + b1 * g.sa1 + (long long)min(m0 + lr + 32 * j, g.M - 1) * g.lda;
#pragma unroll
  for (int j = 0; j < JB; ++j)
    pb[j] = g.B + b0 * g.sb0 + b1 * g.sb1 + (long long)min(n0 + bperm(lr) + 32 * j, g.N - 1) * g.ldb;
  v4i ra[PF][JA], rb[PF][JB];
  auto gload = [&](auto set_c, int k0) {
    constexpr int S = decltype(set_c)::value;
    const int k = k0 + 16 * lc;
    if (k0 + BK <= K) {
#pragma unroll
      for (int j = 0; j < JA; ++j) __builtin_memcpy(&ra[S][j], pa[j] + k, 16);
#pragma unroll
      for (int j = 0; j < JB; ++j) __builtin_memcpy(&rb[S][j], pb[j] + k, 16);
    } else {
#pragma unroll
      for (int j = 0; j < JA; ++j) ra[S][j] = row_chunk(pa[j], k, K);
#pragma unroll
      for (int j = 0; j < JB; ++j) rb[S][j] = row_chunk(pb[j], k, K);
    }
  };
  const int wr = lr * BK + swz<BK>(lr, lc) * 16;         // 32 rows on, the swizzle differs by 4 chunks
  auto lstore = [&](auto set_c, int buf) {
    constexpr int S = decltype(set_c)::value;
    int8_t* s = smem + buf * STAGE;
#pragma unroll
    for (int j = 0; j < JA; ++j) *reinterpret_cast<v4i*>(s + 32 * BK * j + (wr ^ 64 * (j & 1))) = ra[S][j];
#pragma unroll
    for (int j = 0; j < JB; ++j) *reinterpret_cast<v4i*>(s + BM * BK + 32 * BK * j + (wr ^ 64 * (j & 1))) = rb[S][j];
  };
  v16i acc[TN][TM];
#pragma unroll
  for (int i = 0; i < TN; ++i)
#pragma unroll
    for (int j = 0; j < TM; ++j) acc[i][j] = v16i{0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0};
  auto compute = [&](int buf) {
    const int8_t* s = smem + buf * STAGE;
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) {
      v4i af[TM], bf[TN];
      const int ch = ks * 2 + half;
#pragma unroll
      for (int j = 0; j < TM; ++j) {
        const int r = wm * WM + j * 32 + l32;
        af[j] = *reinterpret_cast<const v4i*>(s + r * BK + (swz<BK>(r, ch) << 4));
      }
#pragma unroll
      for (int i = 0; i < TN; ++i) {
        const int r = wn * WN + i * 32 + l32;
        bf[i] = *reinterpret_cast<const v4i*>(s + BM * BK + r * BK + (swz<BK>(r, ch) << 4));
      }
#pragma unroll
      for (int i = 0; i < TN; ++i)
#pragma unroll
        for (int j = 0; j < TM; ++j) acc[i][j] = __builtin_amdgcn_mfma_i32_32x32x32_i8(bf[i], af[j], acc[i][j], 0, 0, 0);
    }
  };

  const int nk = (K + BK - 1) / BK;
  static_for<PF>([&](auto s) {
    if (decltype(s)::value < nk) gload(s, decltype(s)::value * BK);
  });
  lstore(std::integral_constant<int, 0>{}, 0);
  __syncthreads();
  for (int kt0 = 0; kt0 < nk; kt0 += PF)
    static_for<PF>([&](auto u) {
      constexpr int U = decltype(u)::value;
      const int kt = kt0 + U;
      if (kt >= nk) return;
      if (kt + PF < nk) gload(u, (kt + PF) * BK);        // into the registers of stage kt, which is in LDS
      compute(kt & 1);
      if (kt + 1 < nk) lstore(std::integral_constant<int, (U + 1) % PF>{}, (kt + 1) & 1);
      __syncthreads();
    });

  char* Cb = reinterpret_cast<char*>(g.C) + (b0 * g.sc0 + b1 * g.sc1) * OSZ;
  const int mult = g.mult, rnd = g.rnd, shift = g.shift;
  const int mrow = m0 + wm * WM + l32, ncol = n0 + wn * WN + 16 * half;
  auto finish = [&](auto lut_c) {
    constexpr int LUT = decltype(lut_c)::value;
#pragma unroll
    for (int j = 0; j < TM; ++j)
#pragma unroll
      for (int i = 0; i < TN; ++i) {
        const int m = mrow + 32 * j, n = ncol + 32 * i;
        if (m >= g.M || n >= g.N) continue;
        int v[16];
        requant16<OSZ, MUL24, LUT>(acc[i][j], mult, rnd, shift, lut_s, v);
        char* cp = Cb + (m * g.ldc + n) * OSZ;
        if (n + 16 <= g.N) {                             // one store at any alignment
          if constexpr (OSZ == 1) {
            const v4i w = pack16(v);
            __builtin_memcpy(cp, &w, 16);
          } else {
            const v4i w0 = pack8h(v), w1 = pack8h(v + 8);
            __builtin_memcpy(cp, &w0, 16);
            __builtin_memcpy(cp + 16, &w1, 16);
          }
        } else {
          for (int e = 0; e < 16 && n + e < g.N; ++e) {
            if (OSZ == 1)
              cp[e] = (char)v[e];
            else
              reinterpret_cast<int16_t*>(cp)[e] = (int16_t)v[e];
          }
        }
      }
  };
  if (OSZ == 1 && g.lut)
    finish(std::integral_constant<int, OSZ == 1 ? 1 : 0>{});
  else
    finish(std::integral_constant<int, 0>{});
}

template <int BM, int BN, int PF>
static void launch_tiles(GemmArgs& g, int osz, bool mul24, int batch, hipStream_t s) {
  g.tiles_m = (g.M + BM - 1) / BM;
  g.tiles_n = (g.N + BN - 1) / BN;
  const dim3 grid(g.tiles_m * g.tiles_n, batch);
  auto go = [&](auto kernel) { ANVIL_LAUNCH(kernel, grid, dim3(256), 0, s, g); };
  if (osz == 1)
    mul24 ? go(gemm_i8_any<BM, BN, PF, 1, true>) : go(gemm_i8_any<BM, BN, PF, 1, false>);
  else
    mul24 ? go(gemm_i8_any<BM, BN, PF, 2, true>) : go(gemm_i8_any<BM, BN, PF, 2, false>);
}

// 64 x 64 tiles with three stages in flight where at most two of them come to a CU (as deep_tiles in gemm.hip: latency
// bounds the product) or one side is no longer than a tile, 128 x 128 tiles, which read the operands half as often,
// otherwise. Measured, 64 x 64 against 128 x 128: 16 x 3001 x 1000 7.3 and 11.4 us, 2048 x 1024 x 777 (two tiles a CU) 10.7
// and 13.1, 2048 x 1500 x 777 (three) 14.4 and 13.8, 4000 x 1001 x 1003 24 and 17, 16000 x 3001 x 2999 483 and 269.
// (A second stage in flight gains nothing on 128 x 128 tiles, 272 us; 256 x 128 tiles 325.)
void launch_any(GemmArgs& g, int osz, bool mul24, int batch, int num_cu, hipStream_t s) {
  const long long tiles = (long long)((g.M + 63) / 64) * ((g.N + 63) / 64) * batch;
  if (tiles <= 2ll * num_cu || g.M <= 64 || g.N <= 64)
    launch_tiles<64, 64, 3>(g, osz, mul24, batch, s);
  else
    launch_tiles<128, 128, 1>(g, osz, mul24, batch, s);
}

}  // namespace anvil
