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
// Layout of the work: two launches, or three where the keys are split.
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

#include <algorithm>
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

__device__ __forceinline__ int uniform(int v) { return __builtin_amdgcn_readfirstlane(v); }
__device__ __forceinline__ int64_t uniform(int64_t v) {
  return (int64_t)((uint64_t)(uint32_t)uniform((int)v) | (uint64_t)(uint32_t)uniform((int)(v >> 32)) << 32);
}

// ---------------------------------------------------------------------------
// Splitting the keys. Where the blocks of 128 query rows alone would leave
// CUs idle (a short chunk over a long prefix) or end unevenly (ragged
// batches), a block's keys are split over several work items, whose FP32
// partials and LSE go to scratch and are merged by a third launch. The plan
// needs the lengths, which only the device has: one block of the gather
// launch makes it, in the shadow of the others, and writes it to the scratch:
// the end of the caller's workspace past the key rows, when it is long enough
// (rolaq_extend_scratch_rows). Without it the blocks take whole sequences.
// Measured without -> with: 96 queries over 12345 keys, 16 heads, D = 512: 580
// -> 80 us (gather 10, attend 53, merge 14); six ragged chunks: 443 -> 424 us.
// ---------------------------------------------------------------------------
struct ExtItem {        // 64 bytes: all that a block of the attend launch starts from
  int64_t r0, nrows;    // first query row (token * H + head) in the sequence, the sequence's rows
  int64_t koff;         // workspace row of the sequence's key 0
  int32_t qo0, prefix;
  int32_t s0, s1;       // steps of KT keys (s0 == s1: nothing to do)
  int32_t slot;         // partial slot, or -1: the block writes the output
  int32_t pad[5];
};
struct ExtMerge {       // 32 bytes: a block of query rows and its partials
  int64_t r0, nrows;
  int32_t qo0, slot0, n, pad;  // n < 2: nothing to merge
};
struct ExtHead {
  int32_t items, merges;  // items < 0: no plan
  int32_t pad[62];
};
constexpr int kExtRows = 128;    // query rows per item
constexpr int kExtMinSteps = 4;  // least steps worth an item of its own

struct ExtScratch {
  ExtHead* head;
  ExtItem* items;
  ExtMerge* merges;
  float* lse;  // [slots, 128], log2 domain
  float* o;    // [slots, 128 * D], in the attend kernel's lane order
};
__host__ __device__ inline ExtScratch ext_scratch(uint8_t* base, int items, int slots) {
  ExtScratch x;
  x.head = reinterpret_cast<ExtHead*>(base);
  x.items = reinterpret_cast<ExtItem*>(base + sizeof(ExtHead));
  x.merges = reinterpret_cast<ExtMerge*>(x.items + items);
  x.lse = reinterpret_cast<float*>(x.merges + (slots + 1) / 2 * 2);
  x.o = x.lse + (int64_t)slots * kExtRows;
  return x;
}

// Sum over the wave, the same on every lane: DPP scans within rows of 16, the
// rows' totals broadcast (VALU only; as 64-bit shuffles this was 24 dependent
// LDS permutes on the way to every block's first load).
template <int CTRL, int ROWS>
__device__ __forceinline__ int64_t add_dpp(int64_t v) {
  const uint32_t lo = __builtin_amdgcn_update_dpp(0, (int)v, CTRL, ROWS, 0xF, false);
  const uint32_t hi = __builtin_amdgcn_update_dpp(0, (int)(v >> 32), CTRL, ROWS, 0xF, false);
  return v + (int64_t)((uint64_t)hi << 32 | lo);
}
__device__ __forceinline__ int64_t wave_scan64(int64_t v) {  // inclusive; lane 63 has the sum
  v = add_dpp<0x111, 0xF>(v);  // row_shr 1, 2, 4, 8: lane 15 of a row has its total
  v = add_dpp<0x112, 0xF>(v);
  v = add_dpp<0x114, 0xF>(v);
  v = add_dpp<0x118, 0xF>(v);
  v = add_dpp<0x142, 0xA>(v);  // lane 15 of rows 0 and 2 to rows 1 and 3
  return add_dpp<0x143, 0xC>(v);  // lane 31 to rows 2 and 3
}
__device__ __forceinline__ int64_t wave_sum64(int64_t v) {
  v = wave_scan64(v);
  const uint32_t lo = __builtin_amdgcn_readlane((int)v, 63), hi = __builtin_amdgcn_readlane((int)(v >> 32), 63);
  return (int64_t)((uint64_t)hi << 32 | lo);
}
// Workspace row of key 0 of sequence b and the key rows of all sequences
// (every lane of a wave takes part).
__device__ __forceinline__ void key_rows(const ExtendArgs& a, int b, int64_t* koff, int64_t* total) {
  int64_t before = 0, all = 0;
  for (int i = threadIdx.x & 63; i < a.B; i += 64) {
    const int64_t n = a.prefix_lens[i] + (a.qo_indptr[i + 1] - a.qo_indptr[i]);
    before += i < b ? n : 0;
    all += n;
  }
  *koff = wave_sum64(before);
  *total = wave_sum64(all);
}

// Whether the key rows end before the scratch. If they do not (the caller
// stated fewer than there are) the gather writes them over it, so nothing in it
// is read: every kernel asks this itself.
__device__ __forceinline__ bool scratch_is_free(const ExtendArgs& a) {
  int64_t koff, total;
  key_rows(a, 0, &koff, &total);
  return uniform(total) <= a.ws_rows - a.scratch_rows;
}

// The plan. Items are the 128-row blocks of every sequence, the keys of all
// blocks of one sequence cut at the same multiples of a chunk of at most KC
// steps. KC is the best of 32 candidates, one per lane -- multiples of a CU's
// equal share of all steps, fractions of the longest sequence, no cut -- by an
// estimate: steps per CU, plus an item's start and end, plus the partials'
// traffic. Longer chunks go first; a sequence's items are ordered so that the
// same chunk of its blocks lands on one XCD (blocks go to the 8 XCDs
// round-robin), whose L2 then serves its key rows. The block's latency is the
// gather's where there is little to gather, so every step is spread over
// lanes (a first version with one thread per sequence took 20 us), and its cost
// grows with the batch as the gather's does: lengths are read once per stage of
// kStage sequences, places come from scans (with every sequence counting those
// before it, 1000 chunks of 4 queries over 2500 keys took 2990 us, 2430 without
// a plan, now 2400; 4000 of one over 1200 keys 23900, 7700 and 7740).
template <int D, int R>
__device__ void extend_plan(const ExtendArgs& a) {
  constexpr int KT = D == 256 ? 64 : 32;
  constexpr int kCands = 32, kShares = 16, kStage = 512;
  __shared__ unsigned long long s_work, s_keys, s_n[kCands], s_slots[kCands];
  __shared__ int s_longest, s_mx[kCands];
  __shared__ int s_seq[kStage][2];  // blocks and steps of a stage's sequences
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const ExtScratch x = ext_scratch(a.scratch, a.max_items, a.max_slots);
  if (tid == 0) s_work = 0, s_keys = 0, s_longest = 0;
  if (tid < kCands) s_n[tid] = 0, s_slots[tid] = 0, s_mx[tid] = 0;
  __syncthreads();
  struct Shape {
    int64_t prefix, rows, keys;
    int blocks, steps;  // blocks of rows; steps of the last one
  };
  auto shape = [&](int b) {
    const int64_t q = a.qo_indptr[b + 1] - a.qo_indptr[b];
    Shape s;
    s.prefix = a.prefix_lens[b];
    s.keys = s.prefix + q;
    s.rows = q > 0 ? q * a.H : 0;
    s.blocks = (int)((s.rows + kExtRows - 1) / kExtRows);
    s.steps = s.blocks ? (int)((s.keys + KT - 1) / KT) : 0;
    return s;
  };
  // rows 0 .. r of a sequence see keys below this many steps
  auto steps_of = [&](const Shape& s, int64_t r) {
    r = min(r, s.rows - 1);
    const int64_t t = s.rows < (1ll << 31) ? (int64_t)((uint32_t)r / (uint32_t)a.H) : r / a.H;
    return (int)((s.prefix + t) / KT) + 1;
  };
  {
    int64_t work = 0, keys = 0;
    int longest = 0;
    for (int b = tid; b < a.B; b += blockDim.x) {
      const Shape s = shape(b);
      if (b < kStage) s_seq[b][0] = s.blocks, s_seq[b][1] = s.steps;
      keys += s.keys;
      if (s.blocks) work += (int64_t)s.blocks * (steps_of(s, kExtRows - 1) + s.steps) / 2;
      longest = max(longest, s.steps);
    }
    if (wave * 64 < a.B) {
      work = wave_sum64(work);
      keys = wave_sum64(keys);
      if (lane == 0) atomicAdd(&s_work, (unsigned long long)work), atomicAdd(&s_keys, (unsigned long long)keys);
      atomicMax(&s_longest, longest);
    }
  }
  __syncthreads();
  const int longest = s_longest;
  const float work = (float)s_work, share = work / a.cus;
  // candidate c's KC, and the chunks of a sequence for it: count, steps of each
  auto chunk_of = [&](int c) {
    const int kc = c < kShares ? (int)fminf(ceilf(share * __builtin_amdgcn_exp2f(0.2f * (c - 9))), 1.0e9f)
                               : (longest + (c - kShares + 1)) / (c - kShares + 2);
    return c == kCands - 1 ? (1 << 30) : max(kExtMinSteps, kc);
  };
  auto cut = [](int steps, int kc, int& n, int& len) {
    n = (int)(((uint32_t)steps + (uint32_t)kc - 1) / (uint32_t)kc);
    len = n > 1 ? (int)(((uint32_t)steps + (uint32_t)n - 1) / (uint32_t)n) : steps;
  };
  {
    const int c = tid % kCands, kc = chunk_of(c);
    unsigned long long n_all = 0, slots = 0;
    int mx = 0;
    for (int b0 = 0; b0 < a.B; b0 += kStage) {
      const int m = min(kStage, a.B - b0);
      if (b0 > 0) {
        __syncthreads();
        for (int i = tid; i < m; i += blockDim.x) {
          const Shape s = shape(b0 + i);
          s_seq[i][0] = s.blocks, s_seq[i][1] = s.steps;
        }
        __syncthreads();
      }
      for (int i = tid / kCands; i < m; i += blockDim.x / kCands) {
        const int blocks = s_seq[i][0];
        int n, len;
        cut(s_seq[i][1], kc, n, len);
        n_all += (unsigned long long)blocks * n;  // (a sequence without blocks has no steps: n = 0)
        if (n > 1) slots += (unsigned long long)blocks * n;
        mx = max(mx, len);
      }
    }
    if (tid / kCands < a.B) {
      atomicAdd(&s_n[c], n_all);
      atomicAdd(&s_slots[c], slots);
      atomicMax(&s_mx[c], mx);
    }
  }
  __syncthreads();
  if ((int64_t)s_keys > a.ws_rows - a.scratch_rows) return;  // key rows lie in the scratch: nothing is written there
  // chunks longer than the stated bound: the launch's blocks go without a plan
  if (s_n[kCands - 1] > (unsigned long long)a.max_items) {
    if (tid == 0) x.head->items = -1, x.head->merges = 0;
    return;
  }
  int pick, mx;
  {
    constexpr float kItem = 5.f;                       // an item's start and end, in steps
    constexpr float kSlot = D == 512 ? 0.065f : 0.033f;  // a partial written and merged
    const int c = lane % kCands;
    const unsigned long long n = s_n[c], sl = s_slots[c];
    const int m = s_mx[c];
    float t = n <= (unsigned long long)a.cus ? m + kItem : (work + n * kItem) / a.cus + 0.5f * m;
    t += kSlot * sl + (sl ? 4.f : 0.f);
    if (sl > (unsigned long long)a.max_slots || n > (unsigned long long)a.max_items) t = 3.0e38f;
    pick = c;
#pragma unroll
    for (int o = 16; o > 0; o >>= 1) {
      const float t2 = __shfl_xor(t, o);
      const int p2 = __shfl_xor(pick, o);
      if (t2 < t || (t2 == t && p2 > pick)) t = t2, pick = p2;
    }
    mx = s_mx[pick];
  }
  const int kc = chunk_of(pick);
  // A sequence's items start behind those of the sequences before it, the ones
  // with long chunks first; its partials, merges and key rows in batch order. A
  // wave, or a group of waves where there are fewer, takes the sequences of a
  // range 64 at a time, a lane each: scans give the places, and the 64 sequences'
  // items are written an item per lane, which finds its sequence in the scan.
  struct Places {
    int64_t early, late, marks, keys;  // items by class, merges << 32 | partials, key rows
  };
  struct Seq {
    Shape s;
    int n, len, items;
    bool late;
  };
  auto sequence = [&](int b) {
    Seq q{};
    if (b < a.B) {
      q.s = shape(b);
      cut(q.s.steps, kc, q.n, q.len);
      q.items = q.s.blocks * q.n;
      q.late = 4 * (int64_t)q.len < 3 * (int64_t)mx;
    }
    return q;
  };
  auto places = [](const Seq& q) {
    return Places{q.late ? 0 : q.items, q.late ? q.items : 0,
                  q.n > 1 ? (int64_t)q.s.blocks << 32 | q.items : 0, q.s.keys};
  };
  const int waves = blockDim.x / 64, chunks = (a.B + 63) / 64, groups = min(waves, chunks), per = waves / groups;
  const int group = min(wave / per, groups - 1), sub = wave - group * per;
  const int c0 = chunks * group / groups, c1 = chunks * (group + 1) / groups;
  __shared__ Places s_range[4];
  Places at{0, 0, 0, 0}, all{0, 0, 0, 0};
  {
    Places mine{0, 0, 0, 0};
    for (int c = c0; c < c1; ++c) {
      const Places p = places(sequence(64 * c + lane));
      mine.early += p.early, mine.late += p.late, mine.marks += p.marks, mine.keys += p.keys;
    }
    mine.early = wave_sum64(mine.early), mine.late = wave_sum64(mine.late);
    mine.marks = wave_sum64(mine.marks), mine.keys = wave_sum64(mine.keys);
    if (groups == 1) {
      all = mine;
    } else {
      if (lane == 0 && sub == 0) s_range[group] = mine;
      __syncthreads();
      for (int g = 0; g < groups; ++g) {
        const Places p = s_range[g];
        if (g < group) at.early += p.early, at.late += p.late, at.marks += p.marks, at.keys += p.keys;
        all.early += p.early, all.marks += p.marks;
      }
    }
  }
  if (tid == 0) x.head->items = (int)s_n[pick], x.head->merges = (int)(all.marks >> 32);
  if (sub >= per) return;  // (waves that divide into no group)
  at.late += all.early;
  for (int c = c0; c < c1; ++c) {
    const int b = 64 * c + lane;
    const Seq q = sequence(b);
    const Places mine = places(q);
    const Places incl{wave_scan64(mine.early), wave_scan64(mine.late), wave_scan64(mine.marks), wave_scan64(mine.keys)};
    const int upto = (int)(incl.early + incl.late);  // the items up to this sequence's last
    const int base = (int)(q.late ? at.late + incl.late : at.early + incl.early) - q.items;
    const int64_t marks = at.marks + incl.marks - mine.marks;
    const int slot0 = (int)(uint32_t)marks, merge0 = (int)(marks >> 32);
    const int64_t koff = at.keys + incl.keys - q.s.keys;
    const int qo0 = b < a.B ? a.qo_indptr[b] : 0;
    const int total = __shfl(upto, 63), live = min(64, a.B - 64 * c);
    const int top = live > 1 ? 1 << (31 - __clz(live - 1)) : 0;
    for (int j0 = 64 * sub; j0 < total; j0 += 64 * per) {
      const int jj = min(j0 + lane, total - 1);
      int l = 0;  // the sequences whose items all come before item jj
      for (int step = top; step > 0; step >>= 1)
        if (__shfl(upto, l + step - 1) <= jj) l += step;
      const int items = __shfl(q.items, l), j = jj - (__shfl(upto, l) - items);
      Shape s;
      s.prefix = __shfl(q.s.prefix, l), s.rows = __shfl(q.s.rows, l), s.blocks = __shfl(q.s.blocks, l);
      const int n = __shfl(q.n, l), len = __shfl(q.len, l), first = __shfl(base, l), slot = __shfl(slot0, l);
      const int merge = __shfl(merge0, l);
      // item j: chunks in groups of 8 (fewer at the end), blocks in turn within a group
      const int eight = j / (8 * s.blocks), width = min(8, n - 8 * eight), k = j - 8 * s.blocks * eight;
      const int chunk = 8 * eight + k % width, blk = s.blocks - 1 - k / width;  // later blocks first
      ExtItem it;
      it.r0 = (int64_t)blk * kExtRows;
      it.nrows = s.rows;
      it.koff = __shfl(koff, l);
      it.qo0 = __shfl(qo0, l);
      it.prefix = (int32_t)s.prefix;
      const int end = steps_of(s, it.r0 + kExtRows - 1);  // the block's own steps
      it.s0 = min(chunk * len, end);
      it.s1 = min((chunk + 1) * len, end);
      it.slot = end > len ? slot + blk * n + chunk : -1;
      if (j0 + lane < total) {
        x.items[first + j] = it;
        if (n > 1 && chunk == 0)
          x.merges[merge + blk] = ExtMerge{it.r0, s.rows, it.qo0, slot + blk * n, (end + len - 1) / len, 0};
      }
    }
    at.early += __shfl(incl.early, 63), at.late += __shfl(incl.late, 63);
    at.marks += __shfl(incl.marks, 63), at.keys += __shfl(incl.keys, 63);
  }
}

// Key rows of sequence blockIdx.x as fp16 (one thread per 16-byte chunk, rows
// strided over blockIdx.y): chunk rows from k_chunk, prefix rows from the BF16
// window (t < P or t >= L - W of the extended length L) or the INT2 row
// ((code - zero) * scale rounded to bf16), rope from rope_buf. With scratch,
// block (0, 0) makes the plan instead.
template <int D, int R>
__global__ __launch_bounds__(256) void extend_gather_kernel(ExtendArgs a) {
  constexpr int DR = D + R, CPR = DR / 8, NG = D / 128;
  int y = blockIdx.y, ny = gridDim.y;
  if (a.scratch) {
    if (y == 0) {
      if (blockIdx.x == 0) extend_plan<D, R>(a);
      return;
    }
    --y, --ny;
  }
  const int b = blockIdx.x;
  const int64_t qo0 = a.qo_indptr[b];
  const int64_t Tq = a.qo_indptr[b + 1] - qo0;
  const int64_t prefix = a.prefix_lens[b];
  const int64_t L = prefix + Tq;
  const int64_t req = a.req_idx[b];
  const bool ring = req >= 0 && req < a.max_reqs;
  const int P = ring ? a.P : 0, W = ring ? a.W : 0;
  int64_t koff, total;
  key_rows(a, b, &koff, &total);
  const int64_t kv0 = a.kv_indptr[b];
  const int pmask = (1 << a.page_shift) - 1;
  const int64_t n = min(L, a.ws_rows - koff) * CPR;
  for (int64_t e = (int64_t)y * blockDim.x + threadIdx.x; e < n; e += (int64_t)ny * blockDim.x) {
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
// 256: 5.42 -> 4.52 ms (1.21 PFLOP/s, 3108 cycles per 64 keys and wave, of
// which 2176 are MFMAs, at 1.62 GHz: the clock falls with the matrix cores'
// power); six ragged chunks, 16 heads, D = 512: 1.06 -> 0.44 ms; 96 queries
// over 12345 keys: 0.89 -> 0.58 ms (both with whole sequences per block).
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

  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int g = lane >> 5, la32 = lane & 31;

  // ---- the work item: from the plan, or block (sequence, rows) with all keys ---
  ExtScratch x{};
  ExtItem it;
  bool planned = a.scratch != nullptr;
  if (planned) {
    x = ext_scratch(a.scratch, a.max_items, a.max_slots);
    const int items = x.head->items;
    it = x.items[blockIdx.x];  // (within the array, whether planned or not)
    planned = scratch_is_free(a) && items >= 0;
    if (planned && ((int)blockIdx.x >= items || it.s0 >= it.s1)) return;
  }
  if (!planned) {
    // heavier blocks (later tokens) first
    const int b = blockIdx.x % a.B;
    const int y = a.row_blocks - 1 - (int)(blockIdx.x / a.B + blockIdx.y + gridDim.y * blockIdx.z);
    if (y < 0) return;
    it.qo0 = a.qo_indptr[b];
    const int64_t Tq = a.qo_indptr[b + 1] - it.qo0;
    it.r0 = (int64_t)y * BM;
    it.nrows = Tq * a.H;
    if (it.r0 >= it.nrows) return;
    it.prefix = (int)a.prefix_lens[b];
    int64_t total;
    key_rows(a, b, &it.koff, &total);
    if (it.koff + it.prefix + Tq > a.ws_rows) {
      // the sequence's key rows did not fit the workspace: its outputs are NaN
      for (int64_t e = tid; e < (int64_t)BM * D; e += 64 * G::WAVES) {
        const int64_t r = it.r0 + e / D;
        if (r < it.nrows) a.out[(it.qo0 + r / a.H) * a.o_st + (r % a.H) * a.o_sh + e % D] = 0x7FC0;
      }
      return;
    }
    it.s0 = 0;
    it.s1 = 1 << 30;
    it.slot = -1;
  }
  // (the same on every lane, kept in scalar registers)
  const int64_t r0 = uniform(it.r0), nrows = uniform(it.nrows), qo0 = uniform(it.qo0), prefix = uniform(it.prefix);
  const int s0 = uniform(it.s0), s1 = uniform(it.s1), slot = uniform(it.slot);
  // the block's first and last query token, within the sequence; keys are
  // counted from the item's first one on
  // (a 64-bit division is some 150 instructions of a start that is bound by them;
  // at D = 256 the loop came out 0.5 % slower with the 32-bit one beside it, 4 x 2048
  // queries over 14336 keys 4452 -> 4475 us, for 1 % of a call of 12 x 200)
  auto token_of = [&](int64_t row) {
    return D == 512 && nrows >> 31 == 0 ? (int64_t)((uint32_t)row / (uint32_t)a.H) : row / a.H;
  };
  const int64_t t_first = uniform(token_of(r0)), t_last = uniform(token_of(min(nrows - 1, r0 + BM - 1)));
  const int key0 = s0 * KT;
  const int64_t koff = uniform(it.koff) + key0;
  const int kend = (int)min(prefix + t_last + 1, (int64_t)s1 * KT) - key0;
  const int n = (kend + KT - 1) / KT;  // steps

  // ---- query rows of this wave ------------------------------------------------
  // the lane's row of the sequence (whether there is one), token and head
  struct Row {
    bool ok;
    int64_t t;
    int h;
  };
  auto row_of = [&](int lane32) {
    const int rest = (int)(r0 - t_first * a.H) + RW * wave + lane32;  // from the first token's head 0
    Row r{r0 + RW * wave + lane32 < nrows, t_first, 0};
    if (r.ok) r.t += rest / a.H, r.h = rest % a.H;
    return r;
  };
  // They are copied to LDS as whole rows (like a key tile, into ring buffers
  // without a tile yet) and read back as Q^T fragments: read from memory in
  // the fragments' layout each load would touch 32 rows, which took most of a
  // 20,000-cycle start.
  const uint32_t lds0 = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) uint8_t*)s_buf;
  constexpr int kQBuf = D == 512 ? 0 : 2;  // the last 128 rows' worth of buffers
  int qp;                                  // causal limit of the lane's row (-2^30: no row)
  {
    const Row r = row_of(la32);
    qp = r.ok ? (int)(prefix + r.t) - key0 : -(1 << 30);
    const int64_t mine = reinterpret_cast<int64_t>(a.q + (qo0 + r.t) * a.q_st + r.h * a.q_sh);
    // nine pieces are whole rows, 8 at D = 512 and 16 at D = 256, whose places
    // repeat in the next nine but for the swizzle's bit of row 8: the places are
    // worked out once (a start is bound by its instructions)
    constexpr int kTurn = 9, kTurnRows = kTurn * 64 / CPR;
    static_assert(kTurnRows * CPR == kTurn * 64 && RW % kTurnRows == 0, "whole rows per turn");
    const int lo = (int)mine, hi = (int)(mine >> 32);
#pragma unroll
    for (int j = 0; j < kTurn; ++j) {
      const int ci = 64 * j + lane, row = ci / CPR, pc = ci - row * CPR;
      const uint32_t off = 16 * (pc ^ ext_sw<D>(row));
#pragma unroll
      for (int k = 0; k < RW / kTurnRows; ++k) {
        const uint64_t base = (uint32_t)__builtin_amdgcn_ds_bpermute(4 * row + 4 * kTurnRows * k, lo) |
                              (uint64_t)(uint32_t)__builtin_amdgcn_ds_bpermute(4 * row + 4 * kTurnRows * k, hi) << 32;
        const uint64_t src = base + (off ^ (16 * ext_sw<D>(kTurnRows * k)));
        asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, off"
                     ::"s"(lds0 + kQBuf * G::TILE + RW * RB * wave + 1024 * (j + kTurn * k)), "v"(src)
                     : "memory", "m0");
      }
    }
  }
  const float c2 = a.sm_scale * kLog2e;
  const int qfirst = (int)(prefix + t_first) - key0;  // causal limit of the block's first row

  // ---- tile copies: this wave's rows of a tile, 16-byte chunk 64 j + lane ------
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
  const uint64_t keys = reinterpret_cast<uint64_t>(a.ws) + (uint64_t)koff * RB - kBias;
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
  auto first_tile = [&](int t) {
    clamp_rows(t);
#pragma unroll
    for (int p = 0; p < 3; ++p) copy_part(t, p);
  };
  if constexpr (kQBuf == 2) {
    first_tile(0);
    first_tile(1);
  }

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
  // ---- Q^T fragments (fp16), then the first tiles -----------------------------
  if constexpr (kQBuf == 2)
    asm volatile("s_waitcnt vmcnt(18)" ::: "memory");
  else
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  u32x4 qf[KSQ];
#pragma unroll
  for (int ks = 0; ks < KSQ; ++ks) qf[ks] = kread(s_buf + kQBuf * G::TILE + RW * RB * wave, ks);
#pragma unroll
  for (int ks = 0; ks < KSQ; ++ks) {
    qf[ks] = bf16x8_to_f16x8(qf[ks]) & keep_mask(qp >= -(1 << 29));
    asm volatile("" : "+v"(qf[ks])::"memory");
  }
  __builtin_amdgcn_s_barrier();  // every wave has its fragments: the buffers are free
  asm volatile("" ::: "memory");
  if constexpr (kQBuf == 0) {
    first_tile(0);
    first_tile(1);
  }
  first_tile(2);
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
  auto mask = [&](f32x16& S, int key) {
    if (__builtin_expect(key + 31 > qfirst, 0)) {
      asm volatile("");  // a branch, not selects in every unit
      const int lim = qp - key - 4 * g;
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
    // (at D = 512 the first half's probabilities take the place of those that
    // the first half of the output MFMAs has used)
    constexpr int kFirst = D == 512 ? 16 : 6, kOps = 48;
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
    u32x4 P[2];
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
      u32x4 pn[2];
      output_phase(P, vb, buf(i + 1), true, [&](int k) { softmax_slice(S, pn, k, kAllV); }, meet);
#pragma unroll
      for (int m = 0; m < 2; ++m) P[m] = pn[m];
      rescale();
    }
  }

  // no copy may outlive the block's LDS
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");

  // ---- normalise and store -----------------------------------------------------
  // the lane's place again: kept since the start, it would take registers
  // from the loop, and a spilled one's reload would wait for the stores
  int lane_now;
  asm volatile("v_mbcnt_lo_u32_b32 %0, -1, 0\n\tv_mbcnt_hi_u32_b32 %0, -1, %0" : "=v"(lane_now));
  const int ge = lane_now >> 5;
  const float l = add_over_halves(l_run);
  const float inv = l > 0.f ? 1.0f / l : 0.f;
  if (slot >= 0) {
    // a partial: FP32, 16 bytes per lane in the accumulators' order (whole
    // kilobytes per store), and the rows' LSE (log2 domain)
    f32x4* const po = reinterpret_cast<f32x4*>(x.o) + ((int64_t)slot * G::WAVES + wave) * ND * 4 * 64 + lane_now;
#pragma unroll
    for (int nd = 0; nd < ND; ++nd)
#pragma unroll
      for (int q = 0; q < 4; ++q)
        po[(4 * nd + q) * 64] = f32x4{O[nd][4 * q] * inv, O[nd][4 * q + 1] * inv, O[nd][4 * q + 2] * inv,
                                      O[nd][4 * q + 3] * inv};
    if (ge == 0)
      x.lse[(int64_t)slot * BM + RW * wave + lane_now] = l == 0.f ? kExtNoRef : m_ref + __log2f(l);
    return;
  }
  const Row r = row_of(lane_now & 31);
  const bool ok = r.ok;
  uint16_t* const dst = a.out + (qo0 + r.t) * a.o_st + r.h * a.o_sh + 4 * ge;
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
        if (ok) *reinterpret_cast<u32x4*>(dst + 32 * nd + 16 * p + 4 * ge) = u32x4{x[0], y[0], x[1], y[1]};
      }
    } else if (ok) {
#pragma unroll
      for (int q = 0; q < 4; ++q)
#pragma unroll
        for (int k = 0; k < 2; ++k) {
          dst[32 * nd + 8 * q + 2 * k] = (uint16_t)w[q][k];
          dst[32 * nd + 8 * q + 2 * k + 1] = (uint16_t)(w[q][k] >> 16);
        }
    }
  }
}

// ---------------------------------------------------------------------------
// Merge of a plan's partials: out = sum_c 2^(lse_c - M) O_c / sum_c 2^(lse_c - M)
// in FP32, to bf16. A thread takes four columns of a row; what it reads of a
// partial is 16 bytes of a whole kilobyte per wave.
// ---------------------------------------------------------------------------
template <int D, int R>
__global__ __launch_bounds__(256) void extend_merge_kernel(ExtendArgs a) {
  using G = ExtGeo<D, R>;
  constexpr int ND = G::ND, PARTS = D / 8;  // 256-thread parts of a block of rows
  const ExtScratch x = ext_scratch(a.scratch, a.max_items, a.max_slots);
  const int entries = (a.max_slots + 1) / 2;
  const bool free = scratch_is_free(a);
  for (int u = blockIdx.x; u < entries * PARTS; u += gridDim.x) {
    // (the entry is read with the count, not after it)
    const ExtMerge m = x.merges[u / PARTS];
    if (!free || u >= x.head->merges * PARTS) return;
    if (m.n < 2) continue;
    const int e = (u % PARTS) * 256 + threadIdx.x;
    const int lane = e & 63, q = (e >> 6) & 3, nd = (e >> 8) % ND, w = e / (256 * ND);
    const int row = G::RW * w + (lane & 31);
    if (m.r0 + row >= m.nrows) continue;
    const float* lse = x.lse + (int64_t)m.slot0 * G::BM + row;
    const f32x4* po = reinterpret_cast<const f32x4*>(x.o) + (int64_t)m.slot0 * G::BM * D / 4 + e;
    float M = kExtNoRef, den = 0.f;
    for (int c = 0; c < m.n; ++c) M = fmaxf(M, lse[(int64_t)c * G::BM]);
    f32x4 acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll 4
    for (int c = 0; c < m.n; ++c) {
      const float wt = __builtin_amdgcn_exp2f(lse[(int64_t)c * G::BM] - M);
      den += wt;
      acc += wt * po[(int64_t)c * G::BM * D / 4];
    }
    const float inv = 1.f / den;
    const int64_t t = (m.r0 + row) / a.H, h = (m.r0 + row) % a.H;
    uint16_t* dst = a.out + (m.qo0 + t) * a.o_st + h * a.o_sh + 32 * nd + 8 * q + 4 * (lane >> 5);
    const u32x2 v = {pack_bf16(acc[0] * inv, acc[1] * inv), pack_bf16(acc[2] * inv, acc[3] * inv)};
    if (a.o_vec) {
      *reinterpret_cast<u32x2*>(dst) = v;
    } else {
#pragma unroll
      for (int i = 0; i < 4; ++i) dst[i] = (uint16_t)(v[i / 2] >> (16 * (i % 2)));
    }
  }
}

}  // namespace rolaq

namespace {

struct ExtPlanSize {
  int row_blocks;  // blocks of query rows of the longest possible chunk
  int items, slots;
  int64_t rows;    // workspace rows of the scratch, 0: no plan
};

// What a plan may need at most, from what the host knows: the chunk lengths'
// bound and the sum of all key rows.
ExtPlanSize extend_plan_size(int B, int H, int D, int R, int max_q_len, int64_t key_rows, int num_cus) {
  using namespace rolaq;
  ExtPlanSize p{};
  const int64_t kt = D == 256 ? 64 : 32;
  const int64_t rb = ((int64_t)max_q_len * H + kExtRows - 1) / kExtRows;
  p.row_blocks = (int)rb;
  // A plan pays where some sequence has many steps: its block of the gather
  // launch, the merge launch and the partials take about as long as 12 steps
  // (one sequence of 250 keys: 36 us with a plan, 28 without; 2000 keys: 41
  // and 72). The longest one is taken to be no longer than twice the mean.
  // With a block for every CU anyway it can only shorten the end, by half of
  // that sequence's steps at most (5 x 550 queries over 80 keys, 20 heads: 57
  // us with a plan, 51 without). From 7/8 of the CUs on that holds as well: of 98
  // batches of 2 to 8 sequences with 224 to 255 blocks and 12 to 32 steps in the
  // mean, equal and ragged, 94 were slower with a plan, by up to 21 % (4 x 200
  // queries over 650 keys, 40 heads: 47.1 us, 39.2 without), and 4 faster, by 12 %
  // at most; of those with 177 to 208 blocks, ragged ones are up to 39 % faster.
  const int64_t longest = std::min(key_rows, 2 * ((key_rows + B - 1) / std::max(B, 1)));
  if (longest < (8 * rb * B < 7 * (int64_t)num_cus ? 24 : 64) * kt) return p;
  // Slots: at most two per CU (a plan of more would only add partials), and no
  // more than chunks of the least length make
  const int64_t chunks = ((key_rows + kt - 1) / kt + kExtMinSteps - 1) / kExtMinSteps;
  const int64_t slots = std::min<int64_t>(2 * (int64_t)num_cus, rb * B * chunks);
  if (slots < 2 || chunks < 2 || rb * B > (1 << 20)) return p;
  p.slots = (int)slots;
  p.items = (int)(rb * B + slots);
  const ExtScratch x = ext_scratch(nullptr, p.items, p.slots);
  const int64_t bytes = reinterpret_cast<intptr_t>(x.o) + (int64_t)p.slots * kExtRows * D * 4;
  p.rows = (bytes + 2 * (D + R) - 1) / (2 * (D + R));
  return p;
}

}  // namespace

int64_t rolaq_extend_plan_rows(int B, int H, int D, int R, int max_q_len, int64_t key_rows, int num_cus) {
  return extend_plan_size(B, H, D, R, max_q_len, key_rows, num_cus).rows;
}

hipError_t rolaq_launch_extend(const rolaq::ExtendArgs& args, int D, int R, int max_q_len, int64_t key_rows,
                               int num_cus, hipStream_t stream) {
  using namespace rolaq;
  ExtendArgs a = args;
  // 16-byte output stores where the rows allow them
  a.o_vec = (reinterpret_cast<uintptr_t>(a.out) % 16) == 0 && a.o_st % 8 == 0 && a.o_sh % 8 == 0;
  const ExtPlanSize p = extend_plan_size(a.B, a.H, D, R, max_q_len, key_rows, num_cus);
  a.row_blocks = p.row_blocks;
  a.cus = num_cus;
  // the attend launch: an item per block, or (sequence, row block), the latter
  // over two dimensions (in one, 2^24 blocks of 256 threads are too many to launch)
  const unsigned ny = (unsigned)std::min(std::max(p.row_blocks, 1), 65535);
  dim3 blocks((unsigned)a.B, ny, ((unsigned)p.row_blocks + ny - 1) / ny);
  if (p.rows > 0 && a.ws_rows - key_rows >= p.rows) {
    a.scratch = reinterpret_cast<uint8_t*>(a.ws + (a.ws_rows - p.rows) * (D + R));
    a.scratch_rows = p.rows;
    a.max_items = p.items;
    a.max_slots = p.slots;
    blocks = dim3((unsigned)p.items);
  }
  // gather: about 16 rows per block, 64 blocks per sequence at least (their
  // lengths may differ) and no more than 2048 in all; with few rows no more than
  // give every thread one chunk (a row is D / 8 + R / 8 chunks: at 16 rows a block
  // a thread had up to five of them one after another, 5 queries over 100 keys, D =
  // 512: 3.3 -> 5.5 us for the gather)
  const int64_t chunks = std::max<int64_t>(1, (key_rows * ((D + R) / 8) + 255) / 256);
  const int64_t gy = std::min<int64_t>({std::max<int64_t>(64, 2048 / a.B), chunks, std::max<int64_t>(64, (key_rows + 15) / 16)});
#define ROLAQ_EXT(DD, RR)                                                                               \
  if (D == DD && R == RR) {                                                                             \
    using G = ExtGeo<DD, RR>;                                                                           \
    static_assert(G::BM == kExtRows, "rows per item");                                                  \
    const int lds = G::NBUF * G::TILE;                                                                  \
    const hipError_t e = hipFuncSetAttribute((const void*)extend_kernel<DD, RR>,                        \
                                             hipFuncAttributeMaxDynamicSharedMemorySize, lds);          \
    if (e != hipSuccess) return e;                                                                      \
    hipLaunchKernelGGL((extend_gather_kernel<DD, RR>), dim3((unsigned)a.B, (unsigned)(gy + (a.scratch ? 1 : 0))), \
                       dim3(256), 0, stream, a);                                                        \
    hipLaunchKernelGGL((extend_kernel<DD, RR>), blocks, dim3(64 * G::WAVES), lds, stream, a);           \
    if (a.scratch)                                                                                      \
      hipLaunchKernelGGL((extend_merge_kernel<DD, RR>), dim3(16 * (unsigned)num_cus), dim3(256), 0, stream, a); \
    return hipGetLastError();                                                                           \
  }
  ROLAQ_EXT(256, 32)
  ROLAQ_EXT(512, 64)
#undef ROLAQ_EXT
  return hipErrorInvalidValue;
}
