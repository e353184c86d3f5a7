// Absorbed MLA extend (chunked-prefill) attention over the packed INT2 cache.
//
// Reference behaviour: the packed pool's extend path of the patched SGLang
// (deployment/patches/rolaq_sglang.patch:208-235 builds q = [q_nope_out | q_pe]
// in the rotated frame and hands the chunk's own k = [k_nope | k_pe] and the
// pool to the MLA attention); prefix rows are the cache's rows (INT2 codes
// dequantized as (code - zero) * scale and rounded to bf16, the HF cache's
// stored form, mla_quant/cache.py:1030-1039), except the first P and the last
// W positions of the extended sequence, which are the BF16 window rows; the
// chunk's rows enter as the given BF16 keys; attention is causal.
//
// Layout of the work: two launches.
//   gather  every key row of the extended sequences -- [latent | rope], INT2
//           rows dequantized and rounded to bf16 once -- into the caller's
//           workspace as fp16 (the same numbers: a bf16 value is exact in fp16
//           between 2^-17 and 65504), sequence b at rows koff_b .. koff_b +
//           prefix_b + q_b - 1 (koff_b = sum over b' < b of prefix_b' + q_b');
//           HBM-bound, read once per call instead of once per query block.
//   attend  a block takes 128 consecutive (token, head) query rows of one
//           sequence (all heads share the keys: MQA), 32 per wave, and walks
//           its keys in tiles copied from the workspace into a ring of LDS
//           buffers. Per wave and 32 keys:
//   S^T[32 keys, 32 rows] = K . Q^T   on fp16 MFMA 32x32x16 (Q converted to fp16
//                                     once, held in registers: exact products);
//   the causal mask only on keys that reach past the block's first query position
//   softmax in the log2 domain against a per-row reference (the row's maximum
//   over its first keys + 8); scores that pass it by more than 15 move it to
//   their maximum + 8 and scale O and the row sum by the difference in place
//   (scale_acc32x8), so every probability fits fp16
//   O^T[D, 32 rows] += V^T . P^T      on fp16 MFMA 32x32x16, the keys of each
//                                     lane taken in the order the score MFMA left
//                                     them, P rounded to fp16 (relative error 2^-12).
// A sequence whose key rows do not fit the workspace (the caller's key_rows
// was short of the true sum) gets NaN outputs.
#include "rolaq_common.h"
#include "rolaq_args.h"

#include <type_traits>

namespace rolaq {

constexpr float kExtSlack = 15.0f;    // max exp2 argument: a probability stays <= 2^15 (fp16)
constexpr float kExtHeadroom = 8.0f;  // a reference sits this far above the maximum it was set from
constexpr float kExtNoRef = -1.0e30f;  // reference of a row that has seen no key yet (log2 units)

template <int D, int R>
struct ExtGeo {
  static constexpr int DR = D + R;
  static constexpr int RB = 2 * DR;                 // bytes per key row (workspace and LDS)
  static constexpr int CPR = RB / 16;               // 16-byte chunks per key row
  static constexpr int WAVES = 4;                   // one per SIMD: O and Q fill its 512 registers
  static constexpr int RW = 32;                     // query rows per wave
  static constexpr int BM = WAVES * RW;             // query rows per block
  static constexpr int KT = D == 256 ? 64 : 32;     // keys per step: one 36,864-byte tile at both widths
  static constexpr int KSQ = DR / 16;               // K-steps of the score MFMA
  static constexpr int ND = D / 32;                 // output column blocks
  static constexpr int TILE = KT * RB;
  static constexpr int NBUF = 4;                    // ring of tiles in LDS
  static constexpr int WROWS = KT / WAVES;          // key rows that one wave copies
  static constexpr int NDMA = WROWS * CPR / 64;     // its 16-byte-per-lane copies per tile
  static_assert(WROWS * CPR % 64 == 0 && NDMA == 9 && TILE == 36864, "tile copy");
};

// Swizzle of a key row in LDS: 16-byte chunk c of row r sits at chunk
// c ^ ext_sw(r) (only the low 3 / 2 bits change, so it stays in its row). A
// row is 72 (D = 512) or 36 chunks, 8 or 4 modulo the 16 chunks that the 64
// banks hold: with these bits the 16 rows of one column that a quarter wave of
// a score read touches, and the 4 rows x 64 bytes of half a wave of a
// transposed read, fall on 16 distinct chunk positions each.
template <int D>
__device__ __forceinline__ int ext_sw(int r) {
  return D == 512 ? ((r & 2) << 1) | ((r >> 1) & 2) | ((r >> 3) & 1) : (r >> 2) & 3;
}

// Up to four 1 KB copies of 16 bytes per lane into LDS, past the registers:
// copy j from base + off_j + 1024 j (off per lane) to lds + 1024 j + 16 lane
// (the instruction's offset counts on both sides). In assembly because the
// compiler, which tracks such copies, would wait for all of them before any
// LDS read that follows; the kernel waits by count instead (meet). Nothing is
// returned to a register.
__device__ __forceinline__ void copy_to_lds(uint64_t base, uint32_t o0, uint32_t lds) {
  asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2" ::"s"(lds), "v"(o0), "s"(base)
               : "memory", "m0");
}
__device__ __forceinline__ void copy_to_lds4(uint64_t base, uint32_t o0, uint32_t o1, uint32_t o2, uint32_t o3,
                                             uint32_t lds) {
  asm volatile(
      "s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %5\n\t"
      "global_load_lds_dwordx4 %2, %5 offset:1024\n\t"
      "global_load_lds_dwordx4 %3, %5 offset:2048\n\t"
      "global_load_lds_dwordx4 %4, %5 offset:3072" ::"s"(lds),
      "v"(o0), "v"(o1), "v"(o2), "v"(o3), "s"(base)
      : "memory", "m0");
}

__device__ __forceinline__ float max_over_halves(float v) {
  const auto h = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  return fmaxf(__uint_as_float(h[0]), __uint_as_float(h[1]));
}

__device__ __forceinline__ float add_over_halves(float v) {
  const auto h = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  return __uint_as_float(h[0]) + __uint_as_float(h[1]);
}

// Workspace row of key 0 of sequence b.
__device__ __forceinline__ int64_t key_offset(const ExtendArgs& a, int b) {
  int64_t off = 0;
  for (int i = 0; i < b; ++i) off += a.prefix_lens[i] + (a.qo_indptr[i + 1] - a.qo_indptr[i]);
  return off;
}

// Key rows of sequence blockIdx.x as fp16 (one thread per 16-byte chunk, rows
// strided over blockIdx.y): chunk rows from k_chunk, prefix rows from the BF16
// window (t < P or t >= L - W of the extended length L) or the INT2 row
// ((code - zero) * scale rounded to bf16), rope from rope_buf.
template <int D, int R>
__global__ __launch_bounds__(256) void extend_gather_kernel(ExtendArgs a) {
  constexpr int DR = D + R, CPR = DR / 8, NG = D / 128;
  const int b = blockIdx.x;
  const int64_t qo0 = a.qo_indptr[b];
  const int64_t Tq = a.qo_indptr[b + 1] - qo0;
  const int64_t prefix = a.prefix_lens[b];
  const int64_t L = prefix + Tq;
  const int64_t req = a.req_idx[b];
  const bool ring = req >= 0 && req < a.max_reqs;
  const int P = ring ? a.P : 0, W = ring ? a.W : 0;
  const int64_t koff = key_offset(a, b);
  const int64_t kv0 = a.kv_indptr[b];
  const int pmask = (1 << a.page_shift) - 1;
  const int64_t n = min(L, a.ws_rows - koff) * CPR;
  for (int64_t e = (int64_t)blockIdx.y * blockDim.x + threadIdx.x; e < n; e += (int64_t)gridDim.y * blockDim.x) {
    const int64_t t = e / CPR;
    const int c = (int)(e - t * CPR);
    u32x4 v;
    if (t >= prefix) {
      v = bf16x8_to_f16x8(gload<u32x4>(a.kc + (qo0 + t - prefix) * a.kc_st + 8 * c));
    } else {
      const int64_t slot = ((int64_t)a.kv_indices[kv0 + (t >> a.page_shift)] << a.page_shift) + (t & pmask);
      if (c >= D / 8) {
        v = bf16x8_to_f16x8(gload<u32x4>(a.rope + slot * R + 8 * (c - D / 8)));
      } else if (t < P || t >= L - W) {
        const int64_t inner = t < P ? t : P + (t - P) % (W > 0 ? W : 1);
        v = bf16x8_to_f16x8(gload<u32x4>(a.hp + (1 + req * (P + W) + inner) * D + 8 * c));
      } else {
        // elements 8c .. 8c + 7 sit in bytes 2c, 2c + 1 of the packed row
        const uint32_t bits = gload<uint16_t>(a.codes + slot * (D / 4) + 2 * c);
        const f32x2 sz = gload<f32x2>(a.params + slot * (2 * NG) + 2 * (c / 16));
        float f[8];
#pragma unroll
        for (int k = 0; k < 8; ++k) f[k] = (float((bits >> (2 * k)) & 3u) - sz.y) * sz.x;
        v = bf16x8_to_f16x8(
            u32x4{pack_bf16(f[0], f[1]), pack_bf16(f[2], f[3]), pack_bf16(f[4], f[5]), pack_bf16(f[6], f[7])});
      }
    }
    *reinterpret_cast<u32x4*>(a.ws + (koff + t) * DR + 8 * c) = v;
  }
}

// ---------------------------------------------------------------------------
// Attend. What bounds it: the matrix cores and their power. 16-row waves on
// 16x16x32 MFMA (the form before) read 1 KB of LDS per 16-cycle MFMA, all of
// the CU's 256 bytes per clock; 32 rows per wave on 32x32x16 need half of
// that. One wave per SIMD (O and Q fill its registers) issues an instruction
// every 4 to 5 cycles, so the instructions are counted (below), and all VALU
// work sits behind MFMAs, in whose shadow it is free: a 32x32x16 MFMA alone
// takes 14 to 15 ns, with six VALU operations behind it 16.
// Measured, before -> after: 4 x 2048 queries over 14336 keys, 40 heads, D =
// 256: 5.42 -> 4.47 ms (1.22 PFLOP/s, 3108 cycles per 64 keys and wave, of
// which 2176 are MFMAs, at 1.62 GHz: the clock falls with the matrix cores'
// power); six ragged chunks, 16 heads, D = 512: 1.04 -> 0.43 ms; 96 queries
// over 12345 keys: 0.89 -> 0.58 ms.
//
// A lane holds one query row (column la32 of the MFMAs): its scores, its
// reference, its sum and its outputs, so nothing crosses lanes but the two
// halves' maximum. The softmax of 32 keys runs behind the MFMAs of the
// previous keys' output (D = 512), and at D = 256, where registers allow a
// second S, behind those of the next keys' scores as well.
//
// Key tiles are copied from the workspace straight into the ring: while the
// MFMAs read tiles i - 1 (V), i and i + 1 (K), the copies of later tiles are in
// flight, each requested after the barrier that ends the use of its buffer and
// awaited by count at a later one.
// ---------------------------------------------------------------------------
template <int D, int R>
__global__ __launch_bounds__((64 * ExtGeo<D, R>::WAVES), 1) void extend_kernel(ExtendArgs a) {
  using G = ExtGeo<D, R>;
  constexpr int RB = G::RB, CPR = G::CPR, KT = G::KT, KSQ = G::KSQ, ND = G::ND, BM = G::BM, RW = G::RW;
  define_acc32_macros();
  extern __shared__ __attribute__((aligned(16))) uint8_t s_buf[];

  const int b = blockIdx.x;
  const int64_t qo0 = a.qo_indptr[b];
  const int64_t Tq = a.qo_indptr[b + 1] - qo0;
  // heavier blocks (later tokens) first
  const int64_t r0 = (int64_t)(gridDim.y - 1 - blockIdx.y) * BM;
  const int64_t nrows = Tq * a.H;
  if (r0 >= nrows) return;
  const int64_t prefix = a.prefix_lens[b];
  const int64_t L = prefix + Tq;
  const int64_t koff = key_offset(a, b);
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int g = lane >> 5, la32 = lane & 31;
  if (koff + L > a.ws_rows) {
    // the sequence's key rows did not fit the workspace: its outputs are NaN
    for (int64_t e = tid; e < (int64_t)BM * D; e += 64 * G::WAVES) {
      const int64_t r = r0 + e / D;
      if (r < nrows) a.out[(qo0 + r / a.H) * a.o_st + (r % a.H) * a.o_sh + e % D] = 0x7FC0;
    }
    return;
  }
  // last query token of the block -> keys 0 .. prefix + t_last
  const int64_t t_last = min(nrows - 1, r0 + BM - 1) / a.H;
  const int kend = (int)(prefix + t_last + 1);
  const int n = (kend + KT - 1) / KT;  // steps

  // ---- tile copies: this wave's rows of a tile, 16-byte chunk 64 j + lane ------
  const uint32_t lds0 = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) uint8_t*)s_buf;
  // byte offset of the chunk from kBias bytes before the wave's first row, less
  // the 1024 (j % 4) that the copy's own offset adds (kBias keeps the
  // unsigned offsets from wrapping, also when clamp_rows moves them to row 0)
  constexpr int kBias = 3 * 1024;
  uint32_t doff[G::NDMA];
#pragma unroll
  for (int j = 0; j < G::NDMA; ++j) {
    const int ci = 64 * j + lane, row = ci / CPR, pc = ci - row * CPR;
    doff[j] = kBias + row * RB + 16 * (pc ^ ext_sw<D>(G::WROWS * wave + row)) - 1024 * (j % 4);
  }
  const uint64_t keys_v = reinterpret_cast<uint64_t>(a.ws) + (uint64_t)koff * RB - kBias;
  const uint64_t keys = (uint64_t)(uint32_t)__builtin_amdgcn_readfirstlane((uint32_t)keys_v) |
                        (uint64_t)(uint32_t)__builtin_amdgcn_readfirstlane((uint32_t)(keys_v >> 32)) << 32;
  // Third p of the copies of tile i. Rows past the block's last key read that
  // key again: they are masked (clamp_rows(i) comes before the parts). In
  // place of tiles past the last one that one is copied again, to buffers that
  // nothing reads any more, so that every step issues the same copies.
  auto clamp_rows = [&](int i) {
    if (__builtin_expect(i == n - 1, 0)) {
      asm volatile("");  // a branch, taken once
      const int last = max(kend - 1 - KT * i - G::WROWS * wave, 0);
#pragma unroll
      for (int j = 0; j < G::NDMA; ++j) {
        const int row = (64 * j + lane) / CPR;
        doff[j] -= (row - min(row, last)) * RB;
      }
    }
  };
  auto copy_part = [&](int i, int p) {
    const int row0 = min(KT * min(i, n - 1) + G::WROWS * wave, kend - 1);
    const uint64_t src = keys + (uint64_t)row0 * RB;
    const uint32_t dst = lds0 + (i % G::NBUF) * G::TILE + G::WROWS * RB * wave + 4096 * p;
    if (p < 2)
      copy_to_lds4(src, doff[4 * p], doff[4 * p + 1], doff[4 * p + 2], doff[4 * p + 3], dst);
    else
      copy_to_lds(src, doff[8], dst);
  };
#pragma unroll
  for (int t = 0; t < 3; ++t) {
    clamp_rows(t);
#pragma unroll
    for (int p = 0; p < 3; ++p) copy_part(t, p);
  }

  // ---- query rows of this wave: Q^T fragments (fp16) and causal limits --------
  u32x4 qf[KSQ];
  int qp;  // causal limit of the lane's row (-1: no row)
  {
    const int64_t r = r0 + RW * wave + la32;
    const bool ok = r < nrows;
    const int64_t t = ok ? r / a.H : 0, h = ok ? r % a.H : 0;
    qp = ok ? (int)(prefix + t) : -1;
    const uint16_t* qr = a.q + (qo0 + t) * a.q_st + h * a.q_sh + 8 * g;
#pragma unroll
    for (int ks = 0; ks < KSQ; ++ks)
      qf[ks] = ok ? bf16x8_to_f16x8(gload<u32x4>(qr + 16 * ks)) : u32x4{0u, 0u, 0u, 0u};
  }
  const float c2 = a.sm_scale * kLog2e;
  const int qfirst = (int)(prefix + r0 / a.H);  // causal limit of the block's first row

  // ---- LDS read addresses: a few lane bases plus immediate offsets ------------
  // score operand of K-step ks: row la32 of the unit's 32 keys, chunk 2 ks + g
  constexpr int KB = D == 512 ? 4 : 2;   // K-steps per swizzled group of chunks
  uint32_t kbase[KB];
#pragma unroll
  for (int k = 0; k < KB; ++k) kbase[k] = la32 * RB + 16 * ((2 * k + g) ^ ext_sw<D>(la32));
  // transposed reads of V (ds_read_b64_tr_b16: within each 16-lane group, lane
  // 4s + e receives element e of the chunks addressed by lanes s, s + 4,
  // s + 8, s + 12): half h of MFMA m's 16 keys and column block nd: lane
  // addresses key 16 m + 8 h + 4 g + (la >> 2) at columns 32 nd + 16 ((lane >>
  // 4) & 1) + 4 (la & 3), and receives keys 16 m + 8 h + 4 g + 0..3 of column
  // 32 nd + la32: the order in which the score MFMA leaves a lane's keys
  constexpr int VB = D == 512 ? 2 : 1;   // column blocks per swizzled group
  uint32_t vbase[VB][2];
  {
    const int la = lane & 15, x = 2 * ((lane >> 4) & 1) + ((la & 3) >> 1);
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      const int row = 8 * h + 4 * g + (la >> 2);
#pragma unroll
      for (int v = 0; v < VB; ++v) vbase[v][h] = row * RB + 16 * ((4 * v + x) ^ ext_sw<D>(row)) + 8 * (la & 1);
    }
  }
  auto kread = [&](const uint8_t* kb, int ks) {
    return *reinterpret_cast<const u32x4*>(kb + kbase[ks % KB] + 32 * KB * (ks / KB));
  };
  auto vread = [&](const uint8_t* vb, int m, int nd) {
    typedef short s16x4 __attribute__((ext_vector_type(4)));
    typedef __attribute__((address_space(3))) s16x4 lds_s16x4;
    u32x2 v[2];
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      const uint8_t* p = vb + vbase[nd % VB][h] + 64 * VB * (nd / VB) + 16 * m * RB;
      v[h] = __builtin_bit_cast(u32x2, __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4*)(p)));
    }
    return u32x4{v[0].x, v[0].y, v[1].x, v[1].y};
  };

  f32x16 O[ND];  // O^T: columns d = 32 nd + 8 (j / 4) + 4 g + j % 4 of the lane's row
#pragma unroll
  for (int nd = 0; nd < ND; ++nd)
#pragma unroll
    for (int j = 0; j < 16; ++j) O[nd][j] = 0.f;
  float m_ref = kExtNoRef, l_run = 0.f;

  // The MFMAs of a 32-key unit, KSQ for its scores and 2 ND for an output,
  // run in pairs whose LDS operands are read kAhead pairs before and awaited
  // once per pair; the scheduling barriers keep the order in which it is
  // written. One wave issues an instruction every 4 to 5 cycles, so each
  // one counts (a wait before every MFMA, one M0 setting per copy and
  // per-copy row clamps cost 160 of 550 per 64 keys).
  constexpr int kAhead = 2, kRing = 2 * (kAhead + 1);
  constexpr int kAllK = KSQ, kAllV = 2 * ND;
  u32x4 kf[kRing], vf[kRing];
  // MFMA k of a unit's scores S^T (K rows kb of 32 keys). The accumulators are
  // VGPRs, written by MFMAs in assembly: left to the compiler, which gives
  // every MFMA of a kernel with AGPR accumulators an AGPR one, each score
  // would be copied before its softmax. The compiler does not see the
  // results' latency: between a unit's last score MFMA and the first use of
  // its scores there are output MFMAs, or settle().
  auto score_mfma = [&](f32x16& S, int k) {
    if (k == 0)
      asm volatile("v_mfma_f32_32x32x16_f16 %0, %1, %2, 0" : "=v"(S) : "v"(kf[0]), "v"(qf[0]));
    else
      asm volatile("v_mfma_f32_32x32x16_f16 %0, %1, %2, %0" : "+v"(S) : "v"(kf[k % kRing]), "v"(qf[k]));
  };
  auto settle = [&](f32x16& S) { asm volatile("s_nop 7\n\ts_nop 7\n\ts_nop 2" : "+v"(S)); };
  auto output_mfma = [&](const u32x4 (&P)[2], int k) {
    O[k % ND] = mfma32x32x16_f16(vf[k % kRing], P[k / ND], O[k % ND]);
  };
  // the operands of MFMAs k and k + 1
  auto kfetch = [&](const uint8_t* kb, int k) {
    kf[k % kRing] = kread(kb, k);
    kf[(k + 1) % kRing] = kread(kb, k + 1);
  };
  auto vfetch = [&](const uint8_t* vb, int k) {
    vf[k % kRing] = vread(vb, k / ND, k % ND);
    vf[(k + 1) % kRing] = vread(vb, (k + 1) / ND, (k + 1) % ND);
  };
  // LDS reads but the last n have returned (the lgkmcnt field; n <= 15)
  auto landed = [&](auto n) {
    __builtin_amdgcn_s_waitcnt(0xF | (0x3 << 14) | (0x7 << 4) | (decltype(n)::value << 8));
    __builtin_amdgcn_sched_barrier(0);
  };
  // Pairs of score MFMAs of a unit's rows at kb, the next pairs' reads ahead
  // of them (the last ones those of the output that follows, at vb); each
  // slot's other work is done by `slice`
  auto score_phase = [&](f32x16& S, const uint8_t* kb, const uint8_t* vb, auto slice) {
#pragma unroll
    for (int k = 0; k < kAllK; k += 2) {
      const int a2 = k + 2 * kAhead;
      if (a2 < kAllK)
        kfetch(kb, a2);
      else
        vfetch(vb, a2 - kAllK);
      __builtin_amdgcn_sched_barrier(0);
      // reads after this pair's: K pairs have two, V pairs four
      if (a2 < kAllK)
        landed(std::integral_constant<int, 4>{});
      else if (a2 == kAllK)
        landed(std::integral_constant<int, 6>{});
      else
        landed(std::integral_constant<int, 8>{});
#pragma unroll
      for (int q = 0; q < 2; ++q) {
        score_mfma(S, k + q);
        slice(k + q);
        __builtin_amdgcn_sched_barrier(0);
      }
    }
  };
  // Pairs of output MFMAs; the reads of the next unit's scores (kn) go out
  // ahead of the last ones. With `cross`, kn is another tile: it is awaited
  // where every V operand is in registers, and its first reads go out under
  // the remaining MFMAs.
  auto output_phase = [&](const u32x4 (&P)[2], const uint8_t* vb, const uint8_t* kn, bool cross, auto slice,
                          auto meet) {
#pragma unroll
    for (int k = 0; k < kAllV; k += 2) {
      const int a2 = k + 2 * kAhead;
      if (a2 == kAllV && cross) meet();
      if (a2 < kAllV)
        vfetch(vb, a2);
      else
        kfetch(kn, a2 - kAllV);
      __builtin_amdgcn_sched_barrier(0);
      if (a2 < kAllV)
        landed(std::integral_constant<int, 8>{});
      else if (a2 == kAllV)
        landed(std::integral_constant<int, 6>{});
      else
        landed(std::integral_constant<int, 4>{});
#pragma unroll
      for (int q = 0; q < 2; ++q) {
        output_mfma(P, k + q);
        slice(k + q);
        __builtin_amdgcn_sched_barrier(0);
      }
    }
  };
  // keys past a row's causal limit (only in units that reach past the block's
  // first row): -inf, so that a row without any key in the unit adds nothing
  auto mask = [&](f32x16& S, int key0) {
    if (__builtin_expect(key0 + 31 > qfirst, 0)) {
      asm volatile("");  // a branch, not selects in every unit
      const int lim = qp < 0 ? -1 : qp - key0 - 4 * g;
#pragma unroll
      for (int j = 0; j < 16; ++j) S[j] = 8 * (j / 4) + j % 4 <= lim ? S[j] : -__builtin_inff();
    }
  };
  // Softmax of a unit's S against the row's reference (log2 domain, the scale
  // inside the exp2's argument): a unit that passes the reference by more than
  // the slack moves it to the unit's maximum + 8; f scales what was summed
  // before. It runs in `slots` slices, one behind each of that many MFMAs: the
  // maximum in slices 1..4, the reference, then the probabilities of eight
  // pairs of keys, six operations each, spread over the remaining slices.
  float mx, f, mn, t0, t1;
  uint64_t need;
  auto softmax_slice = [&](const f32x16& S, u32x4 (&p)[2], int k, int slots) {
    constexpr int kFirst = 6, kOps = 48;
    if (k >= 1 && k <= 4) {
#pragma unroll
      for (int e = 4 * (k - 1); e < 4 * k; ++e) mx = e == 0 ? S[0] : fmaxf(mx, S[e]);
    }
    if (k == 5) {
      mx = max_over_halves(mx) * c2;
      const bool over = mx > m_ref + kExtSlack;
      mn = over ? mx + kExtHeadroom : m_ref;
      need = __builtin_amdgcn_ballot_w64(over);
      f = __builtin_amdgcn_exp2f(m_ref - mn);
      m_ref = mn;
      l_run *= f;
    }
    if (k >= kFirst) {
      const int span = slots - kFirst;
#pragma unroll
      for (int o = (k - kFirst) * kOps / span; o < (k + 1 - kFirst) * kOps / span; ++o) {
        const int e = o / 6, m = e / 4, d = e % 4;
        switch (o % 6) {
          case 0: t0 = fmaf(S[8 * m + 2 * d], c2, -mn); break;
          case 1: t1 = fmaf(S[8 * m + 2 * d + 1], c2, -mn); break;
          case 2: t0 = __builtin_amdgcn_exp2f(t0); break;
          case 3: t1 = __builtin_amdgcn_exp2f(t1); break;
          case 4:  // the sum of the fp16 probabilities the output MFMA uses, a pair behind
            if (e > 0) l_run = sum_f16x2_fma(p[(e - 1) / 4][(e - 1) % 4], l_run);
            break;
          default: {
            uint32_t pk = pack_f16(t0, t1);
            asm volatile("" : "+v"(pk));  // formed here, not where a later unit uses it
            p[m][d] = pk;
          }
        }
      }
      if (k == slots - 1) l_run = sum_f16x2_fma(p[1][3], l_run);
    }
  };
  auto rescale = [&]() {
#pragma unroll
    for (int nd = 0; nd < ND; nd += 8) scale_acc32x8(*reinterpret_cast<f32x16(*)[8]>(&O[nd]), f, need);
  };
  // this wave's copies of the next tile have landed (those of one more tile
  // may be in flight) and its LDS reads are done; then every wave's
  auto meet = [&]() {
    asm volatile("s_waitcnt vmcnt(9) lgkmcnt(0)" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
  };
  auto buf = [&](int i) { return (const uint8_t*)s_buf + (i % G::NBUF) * G::TILE; };

  asm volatile("s_waitcnt vmcnt(18)" ::: "memory");  // tile 0
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");

  auto nothing = [](int) {};
  if constexpr (D == 256) {
    // Units u of 32 keys, two per tile. During unit u the matrix cores run
    // S_{u+1} and O += V_{u-1} P_{u-1} while the VALU turns S_u into P_u.
    constexpr int kSlots = kAllK + kAllV;
    f32x16 S0, S1;
    u32x4 P0[2], P1[2] = {u32x4{0u, 0u, 0u, 0u}, u32x4{0u, 0u, 0u, 0u}};
#pragma unroll
    for (int k = 0; k < kAhead; ++k) kfetch(buf(0), 2 * k);
    score_phase(S0, buf(0), buf(0), nothing);
    settle(S0);
#pragma unroll
    for (int k = 0; k < kAhead; ++k) kfetch(buf(0) + 32 * RB, 2 * k);
    int t = 0;
    do {
      const uint8_t* const kb = buf(t);
      // the first pass has no output pending: zero probabilities on tile 0
      const uint8_t* const vb = buf(t > 0 ? t - 1 : 0) + 32 * RB;
      const uint8_t* const kn = buf(t + 1);
      // ---- unit 2t: S_{2t+1} from tile t, V_{2t-1} from tile t - 1 ----
      mask(S0, KT * t);
      __builtin_amdgcn_sched_barrier(0);
      score_phase(S1, kb + 32 * RB, vb, [&](int k) { softmax_slice(S0, P0, k, kSlots); });
      output_phase(P1, vb, kn, true, [&](int k) { softmax_slice(S0, P0, kAllK + k, kSlots); }, meet);
      rescale();
      // ---- unit 2t + 1: S_{2t+2} from tile t + 1 (after the last tile: not used), V_{2t} from tile t ----
      mask(S1, KT * t + 32);
      clamp_rows(t + 3);
      __builtin_amdgcn_sched_barrier(0);
      score_phase(S0, kn, kb, [&](int k) {
        softmax_slice(S1, P1, k, kSlots);
        if (k % 6 == 1) copy_part(t + 3, k / 6);
      });
      output_phase(P0, kb, kn + 32 * RB, false, [&](int k) { softmax_slice(S1, P1, kAllK + k, kSlots); }, meet);
      rescale();
    } while (++t < n);
    const uint8_t* const vb = buf(n - 1) + 32 * RB;
#pragma unroll
    for (int k = 0; k < kAhead; ++k) vfetch(vb, 2 * k);
    output_phase(P1, vb, vb, false, nothing, meet);
  } else {
    // One 32-key unit per tile, and no registers for a second S: during step
    // i the matrix cores run S_i, then O += V_{i-1} P_{i-1} while the VALU
    // turns S_i into P_i.
    f32x16 S;
    u32x4 P[2], pn[2];
#pragma unroll
    for (int k = 0; k < kAhead; ++k) kfetch(buf(0), 2 * k);
    score_phase(S, buf(0), buf(0), nothing);
    settle(S);
    mask(S, 0);
#pragma unroll
    for (int k = 0; k < kAllV; ++k) softmax_slice(S, P, k, kAllV);
    meet();
#pragma unroll
    for (int k = 0; k < kAhead; ++k) kfetch(buf(1), 2 * k);
    for (int i = 1; i <= n; ++i) {
      const uint8_t* const vb = buf(i - 1);
      if (i < n) {
        clamp_rows(i + 2);
        __builtin_amdgcn_sched_barrier(0);
        score_phase(S, buf(i), vb, [&](int k) {
          if (k % 12 == 1) copy_part(i + 2, k / 12);
        });
        settle(S);
        mask(S, KT * i);
      } else {
        // after the last step: its output alone
#pragma unroll
        for (int k = 0; k < kAhead; ++k) vfetch(vb, 2 * k);
#pragma unroll
        for (int j = 0; j < 16; ++j) S[j] = -__builtin_inff();
      }
      __builtin_amdgcn_sched_barrier(0);
      output_phase(P, vb, buf(i + 1), true, [&](int k) { softmax_slice(S, pn, k, kAllV); }, meet);
#pragma unroll
      for (int m = 0; m < 2; ++m) P[m] = pn[m];
      rescale();
    }
  }

  // no copy may outlive the block's LDS
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");

  // ---- normalise and store -----------------------------------------------------
  const float l = add_over_halves(l_run);
  const float inv = l > 0.f ? 1.0f / l : 0.f;
  const int64_t r = r0 + RW * wave + la32;
  const bool ok = r < nrows;
  uint16_t* const dst = a.out + (qo0 + (ok ? r / a.H : 0)) * a.o_st + (ok ? r % a.H : 0) * a.o_sh;
#pragma unroll
  for (int nd = 0; nd < ND; ++nd) {
    uint32_t w[4][2];  // columns 32 nd + 8 q + 4 g + (0..3)
#pragma unroll
    for (int q = 0; q < 4; ++q)
#pragma unroll
      for (int k = 0; k < 2; ++k) w[q][k] = pack_bf16(O[nd][4 * q + 2 * k] * inv, O[nd][4 * q + 2 * k + 1] * inv);
    if (a.o_vec) {
      // the halves' pieces joined to 8 consecutive columns per lane: columns
      // 32 nd + 16 p + 8 g + (0..7)
#pragma unroll
      for (int p = 0; p < 2; ++p) {
        const auto x = __builtin_amdgcn_permlane32_swap(w[2 * p][0], w[2 * p + 1][0], false, false);
        const auto y = __builtin_amdgcn_permlane32_swap(w[2 * p][1], w[2 * p + 1][1], false, false);
        if (ok) *reinterpret_cast<u32x4*>(dst + 32 * nd + 16 * p + 8 * g) = u32x4{x[0], y[0], x[1], y[1]};
      }
    } else if (ok) {
#pragma unroll
      for (int q = 0; q < 4; ++q)
#pragma unroll
        for (int k = 0; k < 2; ++k) {
          dst[32 * nd + 8 * q + 4 * g + 2 * k] = (uint16_t)w[q][k];
          dst[32 * nd + 8 * q + 4 * g + 2 * k + 1] = (uint16_t)(w[q][k] >> 16);
        }
    }
  }
}

}  // namespace rolaq

hipError_t rolaq_launch_extend(const rolaq::ExtendArgs& args, int D, int R, int max_q_len, hipStream_t stream) {
  using namespace rolaq;
  ExtendArgs a = args;
  // 16-byte output stores where the rows allow them
  a.o_vec = (reinterpret_cast<uintptr_t>(a.out) % 16) == 0 && a.o_st % 8 == 0 && a.o_sh % 8 == 0;
#define ROLAQ_EXT(DD, RR)                                                                               \
  if (D == DD && R == RR) {                                                                             \
    using G = ExtGeo<DD, RR>;                                                                           \
    const int64_t rows = (int64_t)max_q_len * a.H;                                                      \
    const dim3 grid((unsigned)a.B, (unsigned)((rows + G::BM - 1) / G::BM));                             \
    const int lds = G::NBUF * G::TILE;                                                                  \
    const hipError_t e = hipFuncSetAttribute((const void*)extend_kernel<DD, RR>,                        \
                                             hipFuncAttributeMaxDynamicSharedMemorySize, lds);          \
    if (e != hipSuccess) return e;                                                                      \
    hipLaunchKernelGGL((extend_gather_kernel<DD, RR>), dim3((unsigned)a.B, 64), dim3(256), 0, stream, a); \
    hipLaunchKernelGGL((extend_kernel<DD, RR>), grid, dim3(64 * G::WAVES), lds, stream, a);             \
    return hipGetLastError();                                                                           \
  }
  ROLAQ_EXT(256, 32)
  ROLAQ_EXT(512, 64)
#undef ROLAQ_EXT
  return hipErrorInvalidValue;
}
