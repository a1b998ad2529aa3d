// Row programs: a run of row-wise graph ops (rmsnorm_int, qlinear, add_requant, lut, lut_mul) over the rows of one
// activation, evaluated in one launch. In a block of small width these are everything but attention: rmsnorm -> q, k, v,
// and y -> residual add -> rmsnorm -> MLP -> residual add -> the next block's rmsnorm -> q, k, v (or the logits).
//
// What bounds them: at small widths each op alone is a launch of 4 us or more whose time is its latency (dispatch, the
// first loads, a K loop of one or two steps, the stores) and a pass of the activations through memory; a row needs none
// of the other rows, so a wave can take its rows through all of the ops. What is left is mostly its epilogues: on
// the 32-wide frozen model's 262,144 rows of int16 the middle program (y .. mlp .. next q, k, v: 19 ops) takes 45 us, of
// which 50 MB in and out are 10 and its MFMA 2; whole model 242 -> 123 us, at 32 rows 57 -> 39.
//
// One wave takes 32 rows at a time, and every value of the program stays in LDS as chunks of 16 bytes a lane (int16: two):
// lane l's chunk c of a value holds columns 32 c + 16 (l / 32) .. + 15 of row l % 32. That is at once the layout of
//   - an operand fragment of v_mfma_i32_32x32x32_i8: lane l supplies row l % 32, K bytes 16 (l / 32) .. + 15 of K block c;
//   - a product's result: the weights' rows enter the MFMA in bperm order (common.h), which gives each lane 16
//     consecutive columns of its row;
//   - a direct-to-LDS load of the value's rows.
// So no op reads a chunk that another lane wrote: LDS serves as per-lane memory with a run-time index, at conflict-free
// 1 KiB accesses, and the kernel has no barrier after its constants are staged. The ops are read by scalar loads through
// the constant address space: as kernel arguments (a host page) or through a global pointer, which the kernel's own
// stores turn into vector loads, the middle program took 79 us instead of 51.
//
// The weights of all products of a program form one stream of 1 KiB fragments in the order the products use them
// ([column block of 32][K block] each), staged in LDS with the rsqrt tables, norm weights and int8 tables once per
// workgroup by direct-to-LDS loads, all in flight together (through registers, eight loads at a time, small batches of
// the frozen model took 46 us instead of 39). A transposed result (V^T, what the attention kernel reads) swaps the MFMA's
// operands: a lane then holds four consecutive rows of one column, one 4-byte store.
#include <algorithm>

#include "gemm.h"

namespace anvil {

struct RowArgs {
  const anvil_row_op* op;              // in device memory
  int nops, nblocks, seq, frags;       // seq: rows of one sequence (transposed results); frags: of the weight stream
  int rows;
  unsigned long long mseq;             // n / seq as (n mseq) >> (32 + kseq)
  int kseq;
  const int8_t* w;
  const int8_t* tables[ANVIL_ROW_TABLES_MAX];
  int ntables, slots, nloads;          // nloads: the LOADs, which come first
  // LDS: `slots` KiB of values a wave, the int8 tables, the rsqrt tables and weights of the norms (norm_bytes; NORM op i
  // finds its at byte offsets k and table), the weight stream
  int norm_bytes;
};

// the clamp bounds of a shift in the pre-shift domain, saturated to int32 (lo = -2^b, hi = 2^b - 1 after the shift)
__device__ __forceinline__ int pre_lo(int b, int s) { return s >= 31 - b ? INT32_MIN : -(1 << (b + s)); }
__device__ __forceinline__ int pre_hi(int b, int s) { return s >= 31 - b ? INT32_MAX : (1 << (b + s)) - 1; }

__device__ __forceinline__ int sbyte_of(const v4i& v, int e) { return (int)(int8_t)((unsigned)v[e >> 2] >> (8 * (e & 3))); }
__device__ __forceinline__ int shalf_of(const v4i& v, int e) { return (int)(int16_t)((unsigned)v[e >> 1] >> (16 * (e & 1))); }

// sext(half H of x) * m, |m| < 2^23, in one SDWA multiply
template <int H>
__device__ __forceinline__ int mul_half(unsigned x, int m) {
  int d;
  if constexpr (H == 0)
    asm("v_mul_i32_i24_sdwa %0, %1, sext(%2) dst_sel:DWORD dst_unused:UNUSED_PAD src0_sel:DWORD src1_sel:WORD_0"
        : "=v"(d) : "s"(m), "v"(x));
  else
    asm("v_mul_i32_i24_sdwa %0, %1, sext(%2) dst_sel:DWORD dst_unused:UNUSED_PAD src0_sel:DWORD src1_sel:WORD_1"
        : "=v"(d) : "s"(m), "v"(x));
  return d;
}
// sext(byte B of x) * m
template <int B>
__device__ __forceinline__ int mul_byte(unsigned x, int m) {
  int d;
  if constexpr (B == 0)
    asm("v_mul_i32_i24_sdwa %0, %1, sext(%2) dst_sel:DWORD dst_unused:UNUSED_PAD src0_sel:DWORD src1_sel:BYTE_0"
        : "=v"(d) : "v"(m), "v"(x));
  else if constexpr (B == 1)
    asm("v_mul_i32_i24_sdwa %0, %1, sext(%2) dst_sel:DWORD dst_unused:UNUSED_PAD src0_sel:DWORD src1_sel:BYTE_1"
        : "=v"(d) : "v"(m), "v"(x));
  else if constexpr (B == 2)
    asm("v_mul_i32_i24_sdwa %0, %1, sext(%2) dst_sel:DWORD dst_unused:UNUSED_PAD src0_sel:DWORD src1_sel:BYTE_2"
        : "=v"(d) : "v"(m), "v"(x));
  else
    asm("v_mul_i32_i24_sdwa %0, %1, sext(%2) dst_sel:DWORD dst_unused:UNUSED_PAD src0_sel:DWORD src1_sel:BYTE_3"
        : "=v"(d) : "v"(m), "v"(x));
  return d;
}
// x0 >> sh and x1 >> sh as the halves of one dword (clamped beforehand)
__device__ __forceinline__ unsigned sra_pack2(int x0, int x1, int sh) {
  unsigned d;
  asm("v_ashrrev_i32_sdwa %0, %1, %2 dst_sel:WORD_0 dst_unused:UNUSED_PAD src0_sel:DWORD src1_sel:DWORD"
      : "=v"(d) : "s"(sh), "v"(x0));
  asm("v_ashrrev_i32_sdwa %0, %1, %2 dst_sel:WORD_1 dst_unused:UNUSED_PRESERVE src0_sel:DWORD src1_sel:DWORD"
      : "+v"(d) : "s"(sh), "v"(x1));
  return d;
}
__device__ __forceinline__ v4i sra_pack16(const int* x, int sh) {       // 16 clamped values, shifted, as int8
  return v4i{(int)sra_pack4(x[0], x[1], x[2], x[3], sh), (int)sra_pack4(x[4], x[5], x[6], x[7], sh),
             (int)sra_pack4(x[8], x[9], x[10], x[11], sh), (int)sra_pack4(x[12], x[13], x[14], x[15], sh)};
}
__device__ __forceinline__ v4i sra_pack8h(const int* x, int sh) {       // 8 clamped values, shifted, as int16
  return v4i{(int)sra_pack2(x[0], x[1], sh), (int)sra_pack2(x[2], x[3], sh), (int)sra_pack2(x[4], x[5], sh),
             (int)sra_pack2(x[6], x[7], sh)};
}

typedef __attribute__((address_space(4))) anvil_row_op ConstOp;
__device__ __forceinline__ anvil_row_op read_op(const ConstOp* o) {
  anvil_row_op r;
  r.kind = o->kind, r.a = o->a, r.b = o->b, r.dst = o->dst, r.n = o->n, r.k = o->k, r.table = o->table, r.m24 = o->m24;
  r.wide = o->wide, r.wide_a = o->wide_a, r.wide_b = o->wide_b, r.trans = o->trans, r.mult = o->mult, r.mult2 = o->mult2;
  r.shift = o->shift, r.c = o->c, r.e = o->e, r.lut_len = o->lut_len, r.in = o->in, r.lut = o->lut, r.out = o->out;
  r.ld = o->ld, r.kb = o->kb;
  return r;
}

constexpr int ROW_WAVES = 8;           // waves a workgroup at most

__global__ __launch_bounds__(64 * ROW_WAVES, 4) void row_program(RowArgs p) {
  constexpr int R = 32, NB = 32;                        // rows a wave; columns of a chunk, K bytes of a block
  extern __shared__ __attribute__((aligned(1024))) int8_t smem[];
  const int lane = threadIdx.x & 63, row = lane % R, g16 = 16 * (lane / R);
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), waves = blockDim.x >> 6;
  int8_t* base = smem + 1024 * p.slots * wave;          // this wave's values
  int8_t* mine = base + 16 * lane;
  uint8_t* tab = reinterpret_cast<uint8_t*>(smem) + 1024 * p.slots * waves;
  int8_t* norm = reinterpret_cast<int8_t*>(tab) + 256 * ANVIL_ROW_TABLES_MAX;
  const int8_t* wst = norm + p.norm_bytes + 16 * lane;
  // the ops through the constant address space: scalar loads, which the kernel's own stores do not invalidate
  const ConstOp* ops = (const ConstOp*)(unsigned long long)p.op;
  // touch every cache line of the ops now: their scalar loads later hit, where each op's first use was a miss of its own
  {
    int touch = 0;
    for (int i = 0; i < p.nops; ++i) touch |= ops[i].kind | ops[i].lut_len;
    asm volatile("" ::"s"(touch));
  }
  // the int8 tables, rotated: the entry of v at index v & 255
  if (wave == 0)
    for (int i = 0; i < p.ntables; ++i)
      reinterpret_cast<unsigned*>(tab + 256 * i)[lane ^ 32] = reinterpret_cast<const unsigned*>(p.tables[i])[lane];
  // the norms' constants and the weights straight into LDS, all in flight together
  auto stage = [&](const void* src, int bytes, int8_t* dst) {
    const __amdgpu_buffer_rsrc_t rs = uniform_rsrc(src, bytes);
    for (int c = wave; 1024 * c < bytes; c += waves) dma16(rs, dst + 1024 * c, 1024 * c + 16 * lane);
  };
  for (int i = 0; i < p.nops; ++i) {
    if (ops[i].kind != ANVIL_ROW_NORM) continue;
    stage(ops[i].lut, 4 * ops[i].lut_len, norm + ops[i].k);
    stage(ops[i].in, ops[i].n, norm + ops[i].table);
  }
  stage(p.w, 1024 * p.frags, norm + p.norm_bytes);
  wait_vm_lgkm0<0>();
  __syncthreads();
  auto chunk = [&](int slot, int c) -> v4i& { return *reinterpret_cast<v4i*>(mine + 1024 * (slot + c)); };

  for (int blk = blockIdx.x * waves + wave; blk < p.nblocks; blk += gridDim.x * waves) {
    const int m0 = blk * R;
    const long long m = m0 + row;
    const bool live = m < p.rows;
    const int8_t* frag = wst;                           // the next weight fragment
    __builtin_amdgcn_s_waitcnt(0xC07F);                 // lgkmcnt(0): the last rows' LDS accesses, before loads land there
    // every LOAD's rows straight into LDS, all in flight together; columns past the width and rows past the end as zeros
    for (int o = 0; o < p.nloads; ++o) {
      const anvil_row_op op = read_op(ops + o);
      const int isz = op.wide ? 2 : 1;
      const unsigned lanes = (unsigned)(row * op.ld * isz + g16 * isz);
      for (int c = 0; c < (op.n + NB - 1) / NB; ++c) {
        const long long at = m0 * op.ld * isz + (op.wide ? 2ll * NB * c : (long long)(c >> 1) * op.kb + 32 * (c & 1));
        const __amdgpu_buffer_rsrc_t rs = uniform_rsrc((const int8_t*)op.in + at, (int)(R * op.ld * isz));
        const unsigned off = live && c * NB + g16 < op.n ? lanes : OOB;
        dma16(rs, base + 1024 * (op.dst + c * isz), off);
        if (op.wide) dma16(rs, base + 1024 * (op.dst + 2 * c + 1), off == OOB ? OOB : off + 16);
      }
    }
    wait_vm_lgkm0<0>();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    for (int o = p.nloads; o < p.nops; ++o) {
      const anvil_row_op op = read_op(ops + o);
      const int width = op.n;
      const int nch = (width + NB - 1) / NB;
      // a result chunk: columns col .. col + 15 of this lane's row, int8 or int16 (two halves)
      int8_t* orow = (int8_t*)op.out + m * op.ld * (op.wide ? 2 : 1) + (op.wide ? 2 * g16 : g16);
      const bool store = op.out != nullptr && live;
      auto block_off = [&](int c) { return (long long)(c >> 1) * op.kb + 32 * (c & 1); };
      auto put8 = [&](int c, v4i v) {
        chunk(op.dst, c) = v;
        if (store && c * NB + g16 < width) *reinterpret_cast<v4i*>(orow + block_off(c)) = v;
      };
      auto put16 = [&](int c, v4i lo, v4i hi) {
        chunk(op.dst, 2 * c) = lo;
        chunk(op.dst, 2 * c + 1) = hi;
        if (store && c * NB + g16 < width) {
          *reinterpret_cast<v4i*>(orow + 2 * NB * c) = lo;
          *reinterpret_cast<v4i*>(orow + 2 * NB * c + 16) = hi;
        }
      };
      switch (op.kind) {
        case ANVIL_ROW_NORM: {
          // rmsnorm_int (anvil/semantics.py:164-182), as the row kernels compute it: every lane of a row forms the
          // row's table index, multiplier, shift and bounds; |x w| and |lut M| below 2^23 (host-checked)
          int ss = 0;
          if (op.wide_a) {
            const int rc = op.c ? 1 << (op.c - 1) : 0;
            for (int c = 0; c < 2 * nch; ++c) {
              const v4i x = (c >> 1) * NB + g16 < width ? chunk(op.a, c) : v4i{0, 0, 0, 0};
#pragma unroll
              for (int q = 0; q < 4; ++q) {
                ss += (unsigned)(square_half<0>((unsigned)x[q]) + rc) >> op.c;
                ss += (unsigned)(square_half<1>((unsigned)x[q]) + rc) >> op.c;
              }
            }
          } else {
            for (int c = 0; c < nch; ++c) {
              const v4i x = c * NB + g16 < width ? chunk(op.a, c) : v4i{0, 0, 0, 0};
#pragma unroll
              for (int q = 0; q < 4; ++q) ss = __builtin_amdgcn_sdot4(x[q], x[q], ss, false);
            }
          }
          ss += __shfl_xor(ss, 32, 64);
          ss += op.e;
          const int k = rsqrt_shift(ss, op.lut_len, 32 - __builtin_clz((unsigned)op.lut_len));
          const int rm = reinterpret_cast<const int*>(norm + op.k)[ss >> (2 * k)] * op.mult;
          const int sh = op.shift + k;
          const int rnd = sh ? 1 << (sh - 1) : 0;
          const int lo = sh >= 24 ? INT32_MIN : -128 * (1 << sh), hi = sh >= 24 ? INT32_MAX : 128 * (1 << sh) - 1;
          for (int c = 0; c < nch; ++c) {
            const int col = c * NB + g16;
            const v4i w = col < width ? *reinterpret_cast<const v4i*>(norm + op.table + col) : v4i{0, 0, 0, 0};
            v4i h;
            if (op.wide_a) {
              const v4i x0 = chunk(op.a, 2 * c), x1 = chunk(op.a, 2 * c + 1);
#pragma unroll
              for (int q = 0; q < 4; ++q) {
                const unsigned xa = (unsigned)(q < 2 ? x0[2 * q] : x1[2 * q - 4]);
                const unsigned xb = (unsigned)(q < 2 ? x0[2 * q + 1] : x1[2 * q - 3]);
                const unsigned wd = (unsigned)w[q];
                const int y0 = med3i(mad_i24v(mul_half_byte<0, 0>(xa, wd), rm, rnd), lo, hi);
                const int y1 = med3i(mad_i24v(mul_half_byte<1, 1>(xa, wd), rm, rnd), lo, hi);
                const int y2 = med3i(mad_i24v(mul_half_byte<0, 2>(xb, wd), rm, rnd), lo, hi);
                const int y3 = med3i(mad_i24v(mul_half_byte<1, 3>(xb, wd), rm, rnd), lo, hi);
                h[q] = (int)sra_pack4v(y0, y1, y2, y3, sh);
              }
            } else {
              const v4i x = chunk(op.a, c);
#pragma unroll
              for (int q = 0; q < 4; ++q) {
                const unsigned xd = (unsigned)x[q], wd = (unsigned)w[q];
                const int y0 = med3i(mad_i24v(mul_sbytes<0>(xd, wd), rm, rnd), lo, hi);
                const int y1 = med3i(mad_i24v(mul_sbytes<1>(xd, wd), rm, rnd), lo, hi);
                const int y2 = med3i(mad_i24v(mul_sbytes<2>(xd, wd), rm, rnd), lo, hi);
                const int y3 = med3i(mad_i24v(mul_sbytes<3>(xd, wd), rm, rnd), lo, hi);
                h[q] = (int)sra_pack4v(y0, y1, y2, y3, sh);
              }
            }
            put8(c, h);
          }
          break;
        }
        case ANVIL_ROW_GEMM: {
          const int nk = op.k, mult = op.mult, rnd = op.shift ? 1 << (op.shift - 1) : 0, shift = op.shift;
          const bool m24 = op.m24, tr = op.trans;
          const int bits = op.wide ? 15 : 7;
          const int lo = pre_lo(bits, shift), hi = pre_hi(bits, shift);
          for (int nb = 0; nb < nch; ++nb) {
            v16i d = {0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0};
            for (int kb = 0; kb < nk; ++kb, frag += 1024) {
              const v4i x = chunk(op.a, kb), w = *reinterpret_cast<const v4i*>(frag);
              d = tr ? __builtin_amdgcn_mfma_i32_32x32x32_i8(x, w, d, 0, 0, 0)
                     : __builtin_amdgcn_mfma_i32_32x32x32_i8(w, x, d, 0, 0, 0);
            }
            int acc[16];
#pragma unroll
            for (int e = 0; e < 16; ++e) acc[e] = d[e];
            // clamped before the shift; proven: acc M + rnd inside int32
            if (m24) {
#pragma unroll
              for (int e = 0; e < 16; ++e) acc[e] = med3i(__mul24(acc[e], mult) + rnd, lo, hi);
            } else {
#pragma unroll
              for (int e = 0; e < 16; ++e) acc[e] = med3i(acc[e] * mult + rnd, lo, hi);
            }
            if (op.wide) {
              put16(nb, sra_pack8h(acc, shift), sra_pack8h(acc + 8, shift));
              continue;
            }
            v4i res = sra_pack16(acc, shift);
            if (op.table >= 0) {
              const uint8_t* t = tab + 256 * op.table;
#pragma unroll
              for (int e = 0; e < 16; ++e) acc[e] = t[(unsigned)res[e >> 2] >> (8 * (e & 3)) & 255];
              res = pack16(acc);
            }
            if (tr) {
              // four groups of four consecutive rows of one column: group q is rows 8 q + 4 (l / 32) .. of column
              // bperm(l % 32)
#pragma unroll
              for (int q = 0; q < 4; ++q) {
                const int n = nb * NB + bperm(lane & 31);
                const int mq = m0 + 8 * q + 4 * (lane >> 5);
                if (n >= width || mq >= p.rows) continue;
                int b = (int)(((unsigned long long)(unsigned)mq * p.mseq) >> (32 + p.kseq)), t = mq - b * p.seq;
                int8_t* d = (int8_t*)op.out + b * op.kb + (long long)n * op.ld + t;
                const unsigned v = (unsigned)res[q];
                if (p.seq % 4 == 0) {                  // sequences start at multiples of four rows: one aligned store
                  *reinterpret_cast<unsigned*>(d) = v;
                } else {
                  for (int e = 0; e < 4 && mq + e < p.rows; ++e) {
                    *d = (int8_t)(v >> (8 * e));
                    ++d;
                    if (++t == p.seq) t = 0, d += op.kb - p.seq;
                  }
                }
              }
            } else {
              put8(nb, res);
            }
          }
          break;
        }
        case ANVIL_ROW_ADD: {
          const int ma = op.mult, mb = op.mult2, rnd = op.shift ? 1 << (op.shift - 1) : 0, shift = op.shift;
          if (!op.wide_a && !op.wide_b && !op.wide && op.m24) {      // |ma|, |mb| below 2^24
            const PackedAdd add(ma, mb, rnd, shift);
            for (int c = 0; c < nch; ++c) {
              const v4i x = chunk(op.a, c), y = chunk(op.b, c);
              v4i v;
#pragma unroll
              for (int q = 0; q < 4; ++q) v[q] = (int)add((unsigned)x[q], (unsigned)y[q]);
              put8(c, v);
            }
            break;
          }
          const int bits = op.wide ? 15 : 7;
          const int lo = pre_lo(bits, shift), hi = pre_hi(bits, shift);
          if (op.wide_a && op.wide_b && op.wide && op.m24) {         // the wide stream: |ma|, |mb| below 2^23
            for (int c = 0; c < 2 * nch; ++c) {
              const v4i x = chunk(op.a, c), y = chunk(op.b, c);
              v4i v;
#pragma unroll
              for (int q = 0; q < 4; ++q) {
                const unsigned xd = (unsigned)x[q], yd = (unsigned)y[q];
                v[q] = (int)sra_pack2(med3i(mul_half<0>(xd, ma) + mul_half<0>(yd, mb) + rnd, lo, hi),
                                      med3i(mul_half<1>(xd, ma) + mul_half<1>(yd, mb) + rnd, lo, hi), shift);
              }
              chunk(op.dst, c) = v;
              if (store && (c >> 1) * NB + g16 < width)
                *reinterpret_cast<v4i*>(orow + 2 * NB * (c >> 1) + 16 * (c & 1)) = v;
            }
            break;
          }
          for (int c = 0; c < nch; ++c) {
            int x[16], y[16];
            if (op.wide_a) {
              const v4i x0 = chunk(op.a, 2 * c), x1 = chunk(op.a, 2 * c + 1);
#pragma unroll
              for (int e = 0; e < 16; ++e) x[e] = e < 8 ? shalf_of(x0, e) : shalf_of(x1, e - 8);
            } else {
              const v4i x0 = chunk(op.a, c);
#pragma unroll
              for (int e = 0; e < 16; ++e) x[e] = sbyte_of(x0, e);
            }
            if (op.wide_b) {
              const v4i y0 = chunk(op.b, 2 * c), y1 = chunk(op.b, 2 * c + 1);
#pragma unroll
              for (int e = 0; e < 16; ++e) y[e] = e < 8 ? shalf_of(y0, e) : shalf_of(y1, e - 8);
            } else {
              const v4i y0 = chunk(op.b, c);
#pragma unroll
              for (int e = 0; e < 16; ++e) y[e] = sbyte_of(y0, e);
            }
            // proven inside int32; with m24 both multipliers are below 2^23, and a 24-bit multiply's low 32 bits are exact
#pragma unroll
            for (int e = 0; e < 16; ++e) {
              const int s = op.m24 ? __mul24(x[e], ma) + __mul24(y[e], mb) + rnd : x[e] * ma + y[e] * mb + rnd;
              x[e] = med3i(s, lo, hi) >> shift;
            }
            if (op.wide)
              put16(c, pack8h(x), pack8h(x + 8));
            else
              put8(c, pack16(x));
          }
          break;
        }
        case ANVIL_ROW_LUT: {
          const uint8_t* t = tab + 256 * op.table;
          for (int c = 0; c < nch; ++c) {
            const v4i x = chunk(op.a, c);
            int v[16];
#pragma unroll
            for (int e = 0; e < 16; ++e) v[e] = t[(unsigned)x[e >> 2] >> (8 * (e & 3)) & 255];
            put8(c, pack16(v));
          }
          break;
        }
        default: {                                     // ANVIL_ROW_LUT_MUL: requant(table[x] y)
          const uint8_t* t = tab + 256 * op.table;
          const int mult = op.mult, rnd = op.shift ? 1 << (op.shift - 1) : 0, shift = op.shift;
          const int lo = pre_lo(7, shift), hi = pre_hi(7, shift);
          for (int c = 0; c < nch; ++c) {
            const v4i x = chunk(op.a, c), y = chunk(op.b, c);
            int v[16];
#pragma unroll
            for (int q = 0; q < 4; ++q) {
              const unsigned xd = (unsigned)x[q], yd = (unsigned)y[q];
              v[4 * q] = mul_byte<0>(yd, (int)(int8_t)t[xd & 255]);
              v[4 * q + 1] = mul_byte<1>(yd, (int)(int8_t)t[xd >> 8 & 255]);
              v[4 * q + 2] = mul_byte<2>(yd, (int)(int8_t)t[xd >> 16 & 255]);
              v[4 * q + 3] = mul_byte<3>(yd, (int)(int8_t)t[xd >> 24]);
            }
            if (op.m24) {                               // proven in int32
#pragma unroll
              for (int e = 0; e < 16; ++e) v[e] = med3i(__mul24(v[e], mult) + rnd, lo, hi);
            } else {
#pragma unroll
              for (int e = 0; e < 16; ++e) v[e] = med3i(v[e] * mult + rnd, lo, hi);
            }
            put8(c, sra_pack16(v, shift));
          }
          break;
        }
      }
    }
  }
}

}  // namespace anvil

using namespace anvil;

constexpr long long LDS_MAX = 160 * 1024;   // of a CU
constexpr long long STAGE_MAX = 96 * 1024;  // one wave's values and all constants of a program

// A checked program: its launch, and its ops in device memory.
struct anvil_row_prog {
  RowArgs args;
  int waves;
  unsigned grid, lds;
};

extern "C" int anvil_row_create(anvil_ctx* ctx, const anvil_row_op* ops, int nops, int64_t rows, int seq,
                                const int8_t* w, int64_t w_bytes, const int8_t* const* tables, int ntables,
                                anvil_row_prog** prog) {
  if (!prog) return set_error(ANVIL_E_VALUE, "anvil_row_create: null output pointer");
  *prog = nullptr;
  if (!ops || (ntables > 0 && !tables)) return set_error(ANVIL_E_VALUE, "anvil_row_create: null pointer");
  if (nops < 1 || nops > ANVIL_ROW_OPS_MAX)
    return set_error(ANVIL_E_VALUE, "anvil_row_create: %d ops outside [1, %d]", nops, ANVIL_ROW_OPS_MAX);
  if (ntables < 0 || ntables > ANVIL_ROW_TABLES_MAX)
    return set_error(ANVIL_E_VALUE, "anvil_row_create: %d tables outside [0, %d]", ntables, ANVIL_ROW_TABLES_MAX);
  if (rows < 1 || seq < 1 || rows % seq || rows >= (1ll << 31) - 32)
    return set_error(ANVIL_E_VALUE, "anvil_row_create: %lld rows in sequences of %d", (long long)rows, seq);
  auto al = [](const void* q, int n) { return ((uintptr_t)q % n) == 0; };
  const int nb = 32, tile = 32;
  RowArgs p{};
  std::vector<anvil_row_op> dev_ops(ops, ops + nops);
  long long blocks = 0;                                 // K blocks of the weight stream
  int top = 0;
  for (int i = 0; i < nops; ++i) {
    const anvil_row_op& o = ops[i];
    auto bad = [&](const char* what) { return set_error(ANVIL_E_VALUE, "anvil_row_create: op %d: %s", i, what); };
    if (o.kind < ANVIL_ROW_LOAD || o.kind > ANVIL_ROW_LUT_MUL) return bad("unknown kind");
    if (o.n < 16 || o.n % 16 || o.n > 4096) return bad("a width that is no multiple of 16 up to 4096");
    if (o.shift < 0 || o.shift > 31) return bad("shift outside [0, 31]");
    const int nch = (o.n + nb - 1) / nb;
    const bool gemm = o.kind == ANVIL_ROW_GEMM, trans = gemm && o.trans;
    auto slot = [&](int s, int chunks, bool wide) {     // a value's chunks inside the LDS budget
      const int end = s + chunks * (wide ? 2 : 1);
      top = std::max(top, end);
      return s >= 0 && end <= ANVIL_ROW_SLOTS_MAX;
    };
    if (!trans && !slot(o.dst, nch, o.wide)) return bad("result slot out of range");
    if (o.kind == ANVIL_ROW_LOAD && p.nloads++ != i) return bad("LOADs come first");
    if (o.kind != ANVIL_ROW_LOAD && !slot(o.a, gemm ? o.k : nch, o.wide_a)) return bad("operand slot out of range");
    if ((o.kind == ANVIL_ROW_ADD || o.kind == ANVIL_ROW_LUT_MUL) && !slot(o.b, nch, o.wide_b))
      return bad("operand slot out of range");
    const bool only8 = o.kind == ANVIL_ROW_LUT || o.kind == ANVIL_ROW_LUT_MUL;
    if ((only8 && (o.wide || o.wide_a || o.wide_b)) || (o.kind == ANVIL_ROW_NORM && o.wide) || (gemm && o.wide_a) ||
        (trans && o.wide))
      return bad("an int16 operand or result that this op does not take");
    if (gemm && (o.k < 1 || o.k > ANVIL_ROW_SLOTS_MAX)) return bad("K blocks outside the LDS budget");
    if (gemm) blocks += (long long)nch * o.k;
    if ((only8 && (o.table < 0 || o.table >= ntables)) || (gemm && (o.table >= ntables || (o.table >= 0 && o.wide))))
      return bad("table index out of range");
    if (o.m24 && gemm && (o.mult >= (1 << 23) || o.mult <= -(1 << 23))) return bad("m24 with |mult| >= 2^23");
    if (o.m24 && o.kind == ANVIL_ROW_LUT_MUL && (o.mult >= (1 << 23) || o.mult <= -(1 << 23)))
      return bad("m24 with |mult| >= 2^23");
    if (o.m24 && o.kind == ANVIL_ROW_ADD) {
      const int lim = o.wide || o.wide_a || o.wide_b ? 1 << 23 : 1 << 24;
      if (o.mult >= lim || o.mult <= -lim || o.mult2 >= lim || o.mult2 <= -lim) return bad("m24 multipliers");
    }
    if (o.kind == ANVIL_ROW_LOAD && (!o.in || !al(o.in, 16))) return bad("null or misaligned input");
    if (o.kind == ANVIL_ROW_NORM && (!o.in || !al(o.in, 16) || !o.lut || o.lut_len < 1 || o.lut_len > 4096 || o.lut_len % 4 || o.c < 0 ||
                                     o.c > 30 || o.e < 0))
      return bad("rmsnorm weights, table, square shift or start value");
    if (o.kind == ANVIL_ROW_NORM) {                     // where its constants are staged
      dev_ops[i].k = p.norm_bytes;
      dev_ops[i].table = p.norm_bytes + (4 * o.lut_len + 1023) / 1024 * 1024;
      p.norm_bytes = dev_ops[i].table + (o.n + 1023) / 1024 * 1024;
    }
    if (trans) {
      if (!o.out || !al(o.out, 4) || o.ld % 4 || o.kb % 4 || o.ld < seq || o.kb < 0)
        return bad("a transposed result needs rows of at least a sequence, 4-byte aligned");
    } else if (o.out || o.kind == ANVIL_ROW_LOAD) {
      const bool kblocked = !o.wide && o.kb != 64;
      if ((o.out && !al(o.out, 16)) || (o.ld * (o.wide ? 2 : 1)) % 16 || o.kb % 16 ||
          o.ld > (1 << 24) || (kblocked ? o.ld != 64 || o.kb < rows * 64 : o.ld < o.n))
        return bad("a row stride or block stride out of range");
    }
  }
  for (int i = 0; i < ntables; ++i) {
    if (!tables[i] || !al(tables[i], 4)) return set_error(ANVIL_E_VALUE, "anvil_row_create: table %d", i);
    p.tables[i] = tables[i];
  }
  if (blocks * 1024 != w_bytes || (blocks && (!w || !al(w, 16))))
    return set_error(ANVIL_E_VALUE, "anvil_row_create: a weight stream of %lld bytes for %lld K blocks",
                     (long long)w_bytes, blocks);
  if (int r = check_ctx(ctx)) return r;
  p.nops = nops;
  p.nblocks = (int)((rows + tile - 1) / tile);
  p.seq = seq;
  while ((1 << p.kseq) < seq) ++p.kseq;                 // m = ceil(2^(32+k) / seq), 2^k >= seq: exact below 2^32
  p.mseq = ((1ull << (32 + p.kseq)) + seq - 1) / seq;
  p.frags = (int)blocks;
  p.rows = (int)rows;
  p.w = w;
  p.ntables = ntables;
  p.slots = top;
  // The waves a workgroup that keep most waves resident (at most four a SIMD by registers; they share the constants),
  // fewer when the row blocks would not fill the CUs; as many workgroups as stay resident, each wave walking row blocks.
  const long long share = 256ll * ANVIL_ROW_TABLES_MAX + p.norm_bytes + w_bytes;
  if (share + 1024ll * top > STAGE_MAX)
    return set_error(ANVIL_E_VALUE, "anvil_row_create: %lld bytes of weights and tables beside %d KiB of values exceed "
                                    "%lld", share, top, STAGE_MAX);
  int waves = 1;
  long long per_cu = 0;
  for (int n = 1; n <= ROW_WAVES; ++n) {
    if (n > 1 && p.nblocks < (long long)n * ctx->num_cu) break;
    const long long fit = std::min<long long>(16 / n, LDS_MAX / (share + 1024ll * top * n));
    if (fit * n > per_cu * waves) waves = n, per_cu = fit;
  }
  const unsigned lds = (unsigned)(share + 1024ll * top * waves);
  const unsigned grid = (unsigned)std::min<long long>((p.nblocks + waves - 1) / waves, per_cu * ctx->num_cu);
  if (lds > 64 * 1024)
    ANVIL_HIP(hipFuncSetAttribute(reinterpret_cast<const void*>(row_program),
                                  hipFuncAttributeMaxDynamicSharedMemorySize, LDS_MAX));
  void* dev = nullptr;
  ANVIL_HIP(hipMalloc(&dev, sizeof(anvil_row_op) * nops));
  if (hipError_t e = hipMemcpy(dev, dev_ops.data(), sizeof(anvil_row_op) * nops, hipMemcpyHostToDevice); e != hipSuccess) {
    (void)hipFree(dev);
    return hip_fail(e, "hipMemcpy of a row program");
  }
  p.op = (const anvil_row_op*)dev;
  *prog = new anvil_row_prog{p, waves, grid, lds};
  return ANVIL_OK;
}

extern "C" int anvil_row_launch(anvil_ctx* ctx, anvil_row_prog* prog) {
  if (int r = check_ctx(ctx)) return r;
  if (!prog) return set_error(ANVIL_E_VALUE, "anvil_row_launch: null program");
  ANVIL_LAUNCH(row_program, dim3(prog->grid), dim3(64 * prog->waves), prog->lds, ctx->stream, prog->args);
  ANVIL_LAUNCHED();
  return ANVIL_OK;
}

extern "C" int anvil_row_destroy(anvil_ctx* ctx, anvil_row_prog* prog) {
  if (int r = check_ctx(ctx)) return r;
  if (!prog) return ANVIL_OK;
  ANVIL_HIP(hipStreamSynchronize(ctx->stream));
  ANVIL_HIP(hipFree(const_cast<anvil_row_op*>(prog->args.op)));
  delete prog;
  return ANVIL_OK;
}
