// GEMM tiles for products that leave CUs idle: a one-sequence forward, a few rows against a wide weight, small blocks.
//
// What bounds them: not MFMAs and not bandwidth but the latency of the operand loads. After a kernel boundary the XCD's L2
// holds none of the operands, a load takes about a microsecond, and a K loop that keeps two stages of 64 K bytes in flight
// pays that latency once every two stages: 1024 x 768 x 3072 on 128 x 128 tiles took 15.6 us with its residual add,
// 1024 x 768 x 768 7.5 us. These kernels keep three stages of 128 K bytes in flight (NS = 4, two workgroups a CU), on 64 x
// 64 tiles, which spread the same product over four times the CUs: 9.3 and 5.0 us. (Eight stages, one workgroup a CU: 9.5
// and 5.6 us, so past three stages load latency is no longer all of it: with one workgroup a CU a stage is also a chain of
// fragment reads, four MFMAs on one accumulator, a wait and a barrier. 128 x 128 tiles with four stages: 16.4 and 8.8 us.)
// K up to 256 takes NS = 2: one stage in flight, issued before the stage in LDS is used, so that K's two stages arrive one
// after the other; what hides their latency is the four workgroups a CU that its LDS leaves room for.
//
// One workgroup of four waves (2 x 2) per BM x BN tile, direct-to-LDS loads as in fast_tile (gemm.hip), stage s in array
// s % NS. The waves walk the stages with one barrier a stage. Bt rows enter LDS in bperm order, so a lane's accumulators
// are 16 consecutive columns of its row and the epilogue runs from registers (one 16-byte store a tile, no staging).
// The LUT and an interior tile's residual load before the first stage, so their latency is the pipeline's own.
#include <algorithm>

#include "gemm.h"

namespace anvil {

template <int BM, int BN, int NS, int OSZ, bool MUL24, bool RES>
__device__ __forceinline__ void deep_tile(const GemmArgs& g, int pid, const int bz) {
  constexpr int BK = 128, CPR = BK / 16, KS = BK / 32;
  constexpr int WM = BM / 2, WN = BN / 2, TM = WM / 32, TN = WN / 32;
  static_assert(TM >= 1 && TN >= 1 && NS >= 2 && NS <= 4, "wave tile and stages");
  constexpr int JA = BM * CPR / 256, JB = BN * CPR / 256, G = JA + JB;   // a wave's loads per stage
  constexpr int STAGE = (BM + BN) * BK;
  __shared__ __attribute__((aligned(1024))) int8_t L0[STAGE], L1[STAGE];
  __shared__ __attribute__((aligned(1024))) int8_t L2[NS > 2 ? STAGE : 16], L3[NS > 3 ? STAGE : 16];
  __shared__ int8_t lut_s[256];
  // the array of stage u, chosen at compile time: the compiler then knows which loads fill what a fragment read reads
  auto arr = [&](auto u) -> int8_t* {
    constexpr int U = decltype(u)::value % NS;
    if constexpr (U == 0) return L0;
    else if constexpr (U == 1) return L1;
    else if constexpr (U == 2) return L2;
    else return L3;
  };

  const int t = threadIdx.x, lane = t & 63;
  const int wave = __builtin_amdgcn_readfirstlane(t >> 6), wm = wave >> 1, wn = wave & 1;
  const int half = lane >> 5, l32 = lane & 31;
  const int ntiles = g.tiles_m * g.tiles_n;
  if ((ntiles & 7) == 0) pid = (pid & 7) * (ntiles >> 3) + (pid >> 3);   // consecutive tiles on one XCD
  const int in_group = GROUP_M * g.tiles_n;
  const int first_m = (pid / in_group) * GROUP_M;
  const int gsize = min(g.tiles_m - first_m, GROUP_M);
  const int m0 = (first_m + (pid % in_group) % gsize) * BM, n0 = ((pid % in_group) / gsize) * BN;
  const int b0 = bz / g.batch1, b1 = bz % g.batch1;
  const int K = g.K;
  const __amdgpu_buffer_rsrc_t ra = uniform_rsrc(g.A + b0 * g.sa0 + b1 * g.sa1 + (long long)m0 * g.lda,
                                                 operand_bytes(min(g.M - m0, BM), g.lda, g.kba, K));
  const __amdgpu_buffer_rsrc_t rb = uniform_rsrc(g.B + b0 * g.sb0 + b1 * g.sb1 + (long long)n0 * g.ldb,
                                                 operand_bytes(min(g.N - n0, BN), g.ldb, g.kbb, K));
  const int mrow = m0 + wm * WM + l32, ncol = n0 + wn * WN + 16 * half;   // tile (i, j): row + 32 j, columns + 32 i

  // oldest loads: the LUT (out of range without one) and the residual
  const __amdgpu_buffer_rsrc_t rl = uniform_rsrc(g.lut ? g.lut : g.A, g.lut ? 256 : 0);
  const int8_t lv = (int8_t)__builtin_amdgcn_raw_buffer_load_b8(rl, (unsigned)t, 0, 0);
  const int8_t* Rb = g.R + b0 * g.sr0 + b1 * g.sr1;
  v4i rv[RES ? TM : 1][RES ? TN : 1];
  if constexpr (RES) {
    // the tile's rows through 32-bit offsets (the launch checks BM ldr): rows past M and a chunk past the last row's N
    // columns are out of range; no access when R's rows are not 16-byte aligned
    const __amdgpu_buffer_rsrc_t rr =
        uniform_rsrc(g.vec_res ? Rb + (long long)m0 * g.ldr + n0 : g.A,
                     g.vec_res ? (int)((min(g.M - m0, BM) - 1) * g.ldr + (min(g.N - n0, BN) & ~15)) : 0);
#pragma unroll
    for (int j = 0; j < TM; ++j)
#pragma unroll
      for (int i = 0; i < TN; ++i)
        rv[j][i] = __builtin_bit_cast(v4i, __builtin_amdgcn_raw_buffer_load_b128(
            rr, (unsigned)((mrow - m0 + 32 * j) * g.ldr + ncol - n0 + 32 * i), 0, 0));
  }

  unsigned offa[JA], offb[JB];
  int ka[JA], kb[JB];
#pragma unroll
  for (int j = 0; j < JA; ++j) {
    const int P = (wave + 4 * j) * 64 + lane, row = P / CPR, c = swz<BK>(row, P % CPR);
    offa[j] = (unsigned)(row * g.lda + (c >> 2) * g.kba + (c & 3) * 16);
    ka[j] = c * 16;
  }
#pragma unroll
  for (int j = 0; j < JB; ++j) {
    const int P = (wave + 4 * j) * 64 + lane, row = P / CPR, c = swz<BK>(row, P % CPR);
    offb[j] = (unsigned)(((row & ~31) | bperm(row & 31)) * g.ldb + (c >> 2) * g.kbb + (c & 3) * 16);
    kb[j] = c * 16;
  }
  // chunks past K load zeros; a stage past K is issued all the same (all zeros), which keeps the wait counts fixed
  auto issue = [&](int8_t* a, int k0) {
    const unsigned oa = (unsigned)((k0 >> 6) * g.kba), ob = (unsigned)((k0 >> 6) * g.kbb);
#pragma unroll
    for (int j = 0; j < JA; ++j) dma16(ra, a + (wave + 4 * j) * 1024, k0 + ka[j] < K ? offa[j] + oa : OOB);
#pragma unroll
    for (int j = 0; j < JB; ++j) dma16(rb, a + BM * BK + (wave + 4 * j) * 1024, k0 + kb[j] < K ? offb[j] + ob : OOB);
  };

  v16i acc[TN][TM];
#pragma unroll
  for (int i = 0; i < TN; ++i)
#pragma unroll
    for (int j = 0; j < TM; ++j) acc[i][j] = v16i{0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0};
  v4i af[2][TM], bf[2][TN];
  auto load_frags = [&](int set, const int8_t* a, int ks) {
    const int ch = ks * 2 + half;
#pragma unroll
    for (int j = 0; j < TM; ++j) {
      const int r = wm * WM + j * 32 + l32;
      af[set][j] = *reinterpret_cast<const v4i*>(a + r * BK + (swz<BK>(r, ch) << 4));
    }
#pragma unroll
    for (int i = 0; i < TN; ++i) {
      const int r = wn * WN + i * 32 + l32;
      bf[set][i] = *reinterpret_cast<const v4i*>(a + BM * BK + r * BK + (swz<BK>(r, ch) << 4));
    }
  };
  auto mm = [&](int set) {
#pragma unroll
    for (int i = 0; i < TN; ++i)
#pragma unroll
      for (int j = 0; j < TM; ++j)
        acc[i][j] = __builtin_amdgcn_mfma_i32_32x32x32_i8(bf[set][i], af[set][j], acc[i][j], 0, 0, 0);
  };
  const int nk = (K + BK - 1) / BK;
  // as fast_tile's: stage kt + NS - 1 loads into the array of stage kt - 1, and before its last k-step a wave waits for
  // its share of stage kt + 1 and meets the others
  auto step = [&](int kt, const int8_t* cur, int8_t* nxt, const int8_t* next) {
    issue(nxt, (kt + NS - 1) * BK);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int ks = 0; ks < KS - 1; ++ks) {
      load_frags((ks + 1) & 1, cur, ks + 1);
      __builtin_amdgcn_sched_barrier(0);
      mm(ks & 1);
      __builtin_amdgcn_sched_barrier(0);
    }
    wait_vm_lgkm0<(NS - 2) * G>();
    stage_barrier();
    load_frags(0, next, 0);
    __builtin_amdgcn_sched_barrier(0);
    mm((KS - 1) & 1);
  };
  static_for<NS - 1>([&](auto u) { issue(arr(u), decltype(u)::value * BK); });
  if (g.lut) lut_s[t ^ 128] = lv;                        // rotated: the entry of v at index v & 255
  wait_vm_lgkm0<(NS - 2) * G>();
  stage_barrier();
  load_frags(0, L0, 0);
  // each step is left to the common end on the last stage, so a step's predecessor is always the step before it and the
  // compiler's own counts of loads in flight stay exact
#define ANVIL_DEEP_STEP(u)                                                                                 \
  if constexpr (NS > u) {                                                                                  \
    step(kt, arr(std::integral_constant<int, u>{}), arr(std::integral_constant<int, u + NS - 1>{}),          \
         arr(std::integral_constant<int, u + 1>{}));                                                       \
    if (++kt == nk) break;                                                                                 \
  }
  for (int kt = 0;;) {
    ANVIL_DEEP_STEP(0) ANVIL_DEEP_STEP(1) ANVIL_DEEP_STEP(2) ANVIL_DEEP_STEP(3)
  }
#undef ANVIL_DEEP_STEP

  char* Cb = reinterpret_cast<char*>(g.C) + (b0 * g.sc0 + b1 * g.sc1) * OSZ;
  int8_t* Db = g.D + b0 * g.sd0 + b1 * g.sd1;
  const int mult = g.mult, rnd = g.rnd, shift = g.shift;
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
        const bool whole = n + 16 <= g.N;
        if constexpr (RES) {                             // D = clamp((R ma + y mb + rnd2) >> shift2), proven in int32
          const int8_t* rp = Rb + (long long)m * g.ldr + n;
          int8_t* dp = Db + (long long)m * g.ldd + n;
          if (whole && g.vec_res) {
            const v4i w = pack16(v);
            v4i ov;
            if (PackedAdd::applies(g.ma, g.mb)) {
              const PackedAdd add(g.ma, g.mb, g.rnd2, g.shift2);
#pragma unroll
              for (int q = 0; q < 4; ++q) ov[q] = (int)add((unsigned)rv[j][i][q], (unsigned)w[q]);
            } else {
              int o[16];
#pragma unroll
              for (int e = 0; e < 16; ++e) {
                const int r = (int)(int8_t)((unsigned)rv[j][i][e >> 2] >> (8 * (e & 3)));
                o[e] = min(max((r * g.ma + v[e] * g.mb + g.rnd2) >> g.shift2, -128), 127);
              }
              ov = pack16(o);
            }
            *reinterpret_cast<v4i*>(dp) = ov;
          } else {
            for (int e = 0; e < 16 && n + e < g.N; ++e)
              dp[e] = (int8_t)min(max((rp[e] * g.ma + v[e] * g.mb + g.rnd2) >> g.shift2, -128), 127);
          }
          if (!g.store_y) continue;
        }
        char* cp = Cb + cpos(g, m, n) * OSZ;
        if (whole) {                                     // one store at any alignment
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
  wait_vmcnt(0);                                         // the trailing zero loads land before the LDS is released
}

template <int BM, int BN, int NS, int OSZ, bool MUL24, bool RES>
__global__ __launch_bounds__(256) void gemm_i8_deep(GemmArgs g) {
  deep_tile<BM, BN, NS, OSZ, MUL24, RES>(g, blockIdx.x, blockIdx.y);
}

// up to GEMM_GROUP_MAX products in one launch, as gemm_i8_fast_group's
template <int BM, int BN, int NS, int OSZ, bool MUL24>
__global__ __launch_bounds__(256) void gemm_i8_deep_group(GemmGroupArgs a) {
  const int w = blockIdx.x;
  int i = 0;
#pragma unroll
  for (int j = 1; j < GEMM_GROUP_MAX; ++j) i += (j < a.n && w >= a.first[j]) ? 1 : 0;
  const GemmArgs& g = a.g[i];
  const int ntiles = g.tiles_m * g.tiles_n, local = w - a.first[i];
  const int bz = local / ntiles;
  if (bz >= g.nbatch) return;                            // padding up to the next member's multiple of 8
  deep_tile<BM, BN, NS, OSZ, MUL24, false>(g, local - bz * ntiles, bz);
}

template <int BM, int BN, int NS, bool MUL24>
static void launch_tiles(GemmArgs& g, int osz, int batch, hipStream_t s) {
  g.tiles_m = (g.M + BM - 1) / BM;
  g.tiles_n = (g.N + BN - 1) / BN;
  const dim3 grid(g.tiles_m * g.tiles_n, batch);
  if (osz == 2)
    ANVIL_LAUNCH((gemm_i8_deep<BM, BN, NS, 2, MUL24, false>), grid, dim3(256), 0, s, g);
  else if (g.res)
    ANVIL_LAUNCH((gemm_i8_deep<BM, BN, NS, 1, MUL24, true>), grid, dim3(256), 0, s, g);
  else
    ANVIL_LAUNCH((gemm_i8_deep<BM, BN, NS, 1, MUL24, false>), grid, dim3(256), 0, s, g);
}

template <int BM, int BN, int NS, bool MUL24>
static void launch_group(GemmArgs* gs, const int* batch, int n, int osz, hipStream_t s) {
  GemmGroupArgs a{};
  long long w = 0;
  for (int i = 0; i < n; ++i) {
    gs[i].tiles_m = (gs[i].M + BM - 1) / BM;
    gs[i].tiles_n = (gs[i].N + BN - 1) / BN;
    gs[i].nbatch = batch[i];
    a.g[i] = gs[i];
    a.first[i] = (int)w;
    w += ((long long)gs[i].tiles_m * gs[i].tiles_n * batch[i] + 7) / 8 * 8;   // few tiles: far below 2^31
  }
  a.first[n] = (int)w;
  a.n = n;
  if (osz == 1)
    ANVIL_LAUNCH((gemm_i8_deep_group<BM, BN, NS, 1, MUL24>), dim3((unsigned)w), dim3(256), 0, s, a);
  else
    ANVIL_LAUNCH((gemm_i8_deep_group<BM, BN, NS, 2, MUL24>), dim3((unsigned)w), dim3(256), 0, s, a);
}

void launch_deep(GemmArgs& g, int ns, int osz, bool mul24, int batch, hipStream_t s) {
  if (ns == 2)
    mul24 ? launch_tiles<64, 64, 2, true>(g, osz, batch, s) : launch_tiles<64, 64, 2, false>(g, osz, batch, s);
  else
    mul24 ? launch_tiles<64, 64, 4, true>(g, osz, batch, s) : launch_tiles<64, 64, 4, false>(g, osz, batch, s);
}

void launch_deep_group(GemmArgs* gs, const int* batch, int n, int ns, int osz, bool mul24, hipStream_t s) {
  if (ns == 2)
    mul24 ? launch_group<64, 64, 2, true>(gs, batch, n, osz, s) : launch_group<64, 64, 2, false>(gs, batch, n, osz, s);
  else
    mul24 ? launch_group<64, 64, 4, true>(gs, batch, n, osz, s) : launch_group<64, 64, 4, false>(gs, batch, n, osz, s);
}

}  // namespace anvil
