// Causal chunked-prefill attention over an MLX-layout affine-quantized KV cache, on MFMA.
//
// Computes, per (sequence b, query head h, query row l), the quantity m5engine/attention.py:29-103
// evaluates for L > 1 (blocked online softmax over key blocks, :64-100, causal when the mask is a
// string, :55-58/:70-73):
//   out = softmax(scale * q K^T + mask) V,  K = sK * codesK + bK,  V = sV * codesV + bV
// with query l at position S_b - L + l, keys <= position when causal, keys > position - window
// when a sliding window is set.
//
// Design (head_dim D = 128, 96 or 64, 64-key tiles, a workgroup = 8 waves = 256 query rows, one per CU):
//  * A workgroup serves 256 consecutive rows of one (sequence, KV head) in position-major order
//    (row = position * rep + local head), so all rep query heads of a position share each K/V
//    tile and a causal boundary cuts only a few positions.
//  * The raw tiles (codes, scales, biases) stream into a 3-slot LDS ring by buffer->LDS DMA, two
//    steps ahead of their use, with no registers held in flight; rows past the sequence end read
//    as zero through the buffer range check (they are masked). Each 64-key tile is then
//    dequantized once per workgroup, LDS to LDS, into fp16 operands: K row-major, V transposed
//    (V^T[d][slot]) with its key slots permuted to match the score layout below. The fp16
//    operands are triple-buffered: tile t + 2 is dequantized while tile t is computed (the
//    quantized tile loop below says how the steps overlap).
//  * Per wave (32 rows = the columns of a 32x32 MFMA): S^T = K Q^T (v_mfma_f32_32x32x16_f16;
//    A = K rows from LDS, B = Q^T held in registers). In the MFMA result layout every lane holds
//    16 keys of one query column, so the row max / sum are lane-local plus one permlane swap, and
//    the probabilities converted to fp16 are already the B operand of O^T = V^T P^T: no shuffle.
//  * Q enters the MFMA exactly (times a per-row power of two that keeps it inside the fp16
//    range); the softmax scale in log2 units and that power are applied to the fp32 scores.
//  * A bf16 cache group beyond the fp16 range (its bias overflows on conversion) cannot be held by
//    the fp16 operands: the row blocks that read one return NaN rather than wrong finite values.
//  * Online softmax with threshold rescaling (a row's running maximum moves only when a tile's
//    maximum exceeds it by more than 2^6), fp32 accumulators.
//  * Long key ranges are split over several workgroups. Up to 4 splits of a row block are merged (log-sum-exp
//    over their (m, l, o) partials) by the last of them to finish, more by a launch of their own.
//  * An unquantized fp16/bf16 cache (BITS == 16, head_dim 128 or 64) takes a simpler loop: K operands
//    straight from the raw ring, only V^T staged, the MFMAs in the cache's type.

#pragma once

#include <math.h>

#include <type_traits>

#include "common.h"
#include "dma.h"
#include "launch.h"
#include "merge.h"
#include "prefill_plan.h"

namespace kvq {

constexpr int kPW = 8;        // waves per workgroup
// fp16 per K row in LDS: D + 8 (rows shift by 4 banks)
template <int D>
constexpr int kKS = D + 8;
constexpr int kVS = 72;       // fp16 per V^T row in LDS: 64 + 8
constexpr float kPSlack = 6.0f;
constexpr int kRawSlots = 3;

// The raw tile ring. A slot holds one 64-key tile as loaded: [K codes][V codes][sK, bK, sV, bV],
// code rows with their 16-byte chunks permuted by row (chunk c of row r at position pos(r, c)), each
// scale/bias array as 64 PC 4-byte cells: with an even number NG = D / G of scale groups per row,
// cell PC key + c holds groups 2c and 2c + 1 of the key (PC = NG / 2); with an odd number, cell
// NG key + g holds group g in its low half (PC = NG; the rows are then only 2-byte aligned).
// BITS == 16 is the unquantized cache: raw T rows, no scales or biases.
template <int BITS, int G = 64, int D = 128>
struct RawCfg {
  static constexpr bool DENSE = BITS == 16;
  static_assert(G == 32 || G == 64 || G == 128, "group sizes 32, 64, 128");
  static_assert(D == 128 || D == 64 || (D == 96 && G == 32 && !DENSE), "head_dim 128 or 64, or 96 for quantized caches");
  static_assert(G <= D && D % G == 0, "a group lies in one row");
  static constexpr int NG = D / G;                  // scale groups per key row
  static constexpr int ROWB = D * BITS / 8;         // code bytes per key row
  static constexpr int CPR = ROWB / 16;             // 16-byte chunks per row
  static constexpr int KB = kPT * ROWB;             // bytes of a K (or V) code tile
  static constexpr int CI = KB / 1024;              // DMA instructions per K (or V) code tile
  static constexpr bool CELL1 = NG % 2 == 1;        // one group per scale/bias cell
  static constexpr int PC = CELL1 ? NG : NG / 2;    // 4-byte cells per key in a scale/bias array
  static constexpr int SBB = DENSE ? 0 : 256 * PC;  // bytes of one scale/bias array
  static constexpr int SLOT = 2 * KB + 4 * SBB;
  // the waves that dequantize: V^T in waves [0, NSW), K in [NSW, 2 NSW) (256 threads each for
  // D = 128, 192 for D = 96, 128 for D = 64); the other waves only compute
  static constexpr int NSW = D / 32;
  // code DMA instructions per wave: when the 2 CI of a tile do not divide over the 8 waves (D = 96, or
  // 4-bit D = 64) the dequantizing waves issue them and the others none
  static constexpr int CODE_WAVES = (2 * CI) % kPW == 0 ? kPW : 2 * NSW;
  static constexpr int CPW = 2 * CI / CODE_WAVES;
  // The chunk swizzle of row r. Quantized tiles fold in r / 16: the V^T staging reads one dim
  // quad of 8 keys per lane, and keys 16 apart (the same key % CPR) would otherwise share LDS
  // banks (a 4-way conflict at 8 bits); this spreads them over the banks. Unquantized rows: the
  // operand reads take one chunk of 32 consecutive rows, of which those 512 / ROWB apart share banks;
  // r / 4 gives such rows of 128 bytes distinct chunks, r itself such rows of 256.
  static __device__ __forceinline__ constexpr int swz(int r) {
    return (!DENSE ? r ^ (r >> 4) : D == 64 ? r >> 2 : r) % CPR;
  }
  // Rows of 6 or 3 chunks (D = 96) rotate them by a multiple that depends on r / 16 instead: such rows
  // are 24 or 12 banks long, so keys 4 apart already differ and only keys 16 apart would meet (the
  // four rotations 0, 3, 5, 2 of 6 give the V^T staging's chunk pairs four starts).
  static constexpr bool ROT = (CPR & (CPR - 1)) != 0;
  static __device__ __forceinline__ constexpr int rot(int r) {
    return CPR == 6 ? (0x2530 >> (4 * ((r >> 4) & 3))) & 7 : ((r >> 4) & 3) % 3;
  }
  // position of chunk c in row r, and the chunk at position q
  static __device__ __forceinline__ constexpr int pos(int r, int c) {
    return ROT ? (c + rot(r)) % CPR : c ^ swz(r);
  }
  static __device__ __forceinline__ constexpr int chunk_at(int r, int q) {
    return ROT ? (q + CPR - rot(r)) % CPR : q ^ swz(r);
  }
  // 64-cell scale/bias DMA instructions: 4 PC of them fill the four arrays. Up to 8 they go one per
  // wave (with PC = 1 two waves fill the same cells); the 12 of D = 96 go two to each of the six
  // waves that load codes.
  static constexpr int SBW = DENSE ? 0 : 4 * PC <= kPW ? 1 : 4 * PC / CODE_WAVES;
  static constexpr bool SB_ALL = 4 * PC <= kPW;     // every wave issues them
  static constexpr int IPT = CPW + SBW;             // DMA instructions per tile of a wave that loads codes
  static constexpr int IPT_NOCODE = SB_ALL ? SBW : 0;  // ... and of one that does not
  static_assert(CPW * CODE_WAVES == 2 * CI, "code DMAs divide evenly over the waves that issue them");
  static_assert(CODE_WAVES >= 2 * NSW, "the dequantizing waves load codes");
  static_assert(DENSE || SB_ALL || SBW * CODE_WAVES == 4 * PC, "scale/bias DMAs divide evenly");
  // scale/bias DMA j of wave w: its array and which 64 cells of it
  static __device__ __forceinline__ constexpr int sb_array(int w, int j) { return SB_ALL ? w / 2 : (w * SBW + j) / PC; }
  static __device__ __forceinline__ constexpr int sb_part(int w, int j) {
    return SB_ALL ? (w % 2) % PC : (w * SBW + j) % PC;
  }
  // byte offset of group g of key `key` inside a scale/bias array
  static __host__ __device__ constexpr int sb_off(int key, int g) {
    return CELL1 ? 4 * (PC * key + g) : 4 * (PC * key + g / 2) + 2 * (g & 1);
  }
};

typedef _Float16 h4 __attribute__((ext_vector_type(4)));

struct PreParams {
  const uint16_t* q;
  int64_t q_sb, q_sh, q_sl;
  const uint8_t* kc;
  const uint8_t* vc;
  int64_t kc_sb, kc_sh, kc_ss;  // bytes
  int64_t vc_sb, vc_sh, vc_ss;  // bytes
  const uint16_t* ks;
  const uint16_t* kb;
  const uint16_t* vs;
  const uint16_t* vb;
  int64_t ksb_sb, ksb_sh, ksb_ss;  // elements
  int64_t vsb_sb, vsb_sh, vsb_ss;
  const int32_t* seq_lens;
  uint16_t* out;
  int64_t o_sb, o_sh, o_sl;
  float* part_o;
  float* part_ml;
  unsigned* counters;  // arrivals per unit, zero between launches
  int order, nbk, lo;  // how workgroups are numbered (prefill_wg)
  int Hq, Hkv, L, S, rep, nrows, rowblocks, nsplit, nunits;
  int chunk;           // keys per split (a multiple of 64); see split_keys
  int fused;           // 1: the last split of a row block merges; 0: prefill_combine_kernel does
  float scale_log2;
  int causal, window;
  // paged cache (PAGED kernels): rows of sequence b live in 64-row pages, page table[b][r / 64];
  // the codes/scales/biases batch strides above are then page strides
  const int32_t* table;
  int64_t table_stride;
  int num_pages;
  // the caches' range exponents (kvq_qtensor.range_exp), or null: the fp16 operands are staged
  // times 2^-E, and 2^E returns in the score scale (K) and the output (V)
  const int32_t* k_rexp;
  const int32_t* v_rexp;
  int out8;  // 1: output rows are only 8-byte aligned (unquantized head_dim 64)
  // general mask (kvq_mask; MASKED kernels), over the reference's grouped score layout, and what
  // mask_classes_kernel found in it: per row block (and KV head, if the mask has one: w_kv units of
  // row blocks apart) 2 words per 64 tiles, [any][mixed], bit i of word w being tile 64 w + i
  const void* mask;
  int mask_kind;
  int64_t m_sb, m_skv, m_srep, m_sl;
  const uint64_t* words;
  int nwords;  // words per bitmap
  int w_kv;    // 1: the bitmaps have a KV head axis
};

// The tiles of a row block that hold a visible key, under a general mask, and how the splits share
// them: `chunk` tiles of that list each.
struct MaskSplit {
  const uint64_t* any;    // [nwords], then the mixed bitmap
  int n, chunk, nsplit;
};
__device__ __forceinline__ uint64_t load_uniform_u64(const uint64_t* p, int i) {
  return ((const __attribute__((address_space(4))) uint64_t*)p)[i];
}
__device__ __forceinline__ uint64_t uniform64(uint64_t x) {
  return (uint64_t)(uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)x) |
         ((uint64_t)(uint32_t)__builtin_amdgcn_readfirstlane((int)(x >> 32)) << 32);
}
__device__ __forceinline__ MaskSplit split_masked(const PreParams& p, int b, int kvh, int rb) {
  MaskSplit m;
  m.any = p.words + (int64_t)((p.w_kv ? b * p.Hkv + kvh : b) * p.rowblocks + rb) * (2 * p.nwords);
  m.n = 0;
  for (int w = 0; w < p.nwords; ++w) m.n += __builtin_popcountll(load_uniform_u64(m.any, w));
  m.n = __builtin_amdgcn_readfirstlane(m.n);  // (wave-uniform, as everything the tile walk is made of)
  m.chunk = max(p.chunk / kPT, (m.n + p.nsplit - 1) / p.nsplit);
  m.nsplit = max((m.n + m.chunk - 1) / m.chunk, 1);
  return m;
}

// V^T slot of key `kk` (0..63) inside a tile: the 16 keys of PV k-step j = kk / 16 are stored so
// that slots 16j + 8h + i hold the keys the score layout gives lane half h at i.
__host__ __device__ constexpr int v_slot_key(int slot) {
  return 16 * (slot >> 4) + ((slot & 7) < 4 ? 4 * ((slot >> 3) & 1) + (slot & 7) : 8 + 4 * ((slot >> 3) & 1) + (slot & 7) - 4);
}
// The 8 keys of V^T slot chunk c8 are v_base_key(c8) + v_key_offset(i): a per-lane base plus
// compile-time offsets, so the staging addresses them with immediate offsets.
__host__ __device__ constexpr int v_base_key(int c8) { return 16 * (c8 >> 1) + 4 * (c8 & 1); }
__host__ __device__ constexpr int v_key_offset(int i) { return i < 4 ? i : i + 4; }
constexpr bool v_keys_split() {
  for (int c8 = 0; c8 < 8; ++c8)
    for (int i = 0; i < 8; ++i)
      if (v_slot_key(8 * c8 + i) != v_base_key(c8) + v_key_offset(i) || (v_base_key(c8) & 3) != 0 ||
          (v_key_offset(i) & 7) != (i & 3) || ((v_base_key(c8) + v_key_offset(i)) >> 4) != (v_base_key(c8) >> 4))
        return false;
  return true;
}
static_assert(v_keys_split(), "slot keys are a per-lane base (low two bits clear) plus i-dependent offsets below 16");


// This wave's share of a raw tile: CPW 1 KiB code loads (K instructions first, then V; none for
// waves from CODE_WAVES on) and SBW 64-cell scale/bias loads (array sb_array, cells from
// 64 sb_part; 4-byte cells, or 2-byte values into the low halves when a cell holds one group).
template <int BITS, int G = 64, int D = 128>
struct RawShare {
  using C = RawCfg<BITS, G, D>;
  static constexpr int SBN = C::SBW > 0 ? C::SBW : 1;
  __amdgpu_buffer_rsrc_t code_r[C::CPW], sb_r[SBN];
  uint32_t code_vo[C::CPW], code_lds[C::CPW], sb_vo[SBN], sb_lds[SBN];
  int64_t code_ss[C::CPW], sb_ss[SBN];  // bytes per key row
  bool code_on;                         // this wave issues code loads (wave-uniform)

  __device__ __forceinline__ void init(const PreParams& p, __amdgpu_buffer_rsrc_t kr, __amdgpu_buffer_rsrc_t vr,
                                       const __amdgpu_buffer_rsrc_t (&sr)[4], int wave, int lane) {
    code_on = wave < C::CODE_WAVES;
#pragma unroll
    for (int j = 0; j < C::CPW; ++j) {
      const int q = code_on ? wave * C::CPW + j : 0;
      const bool is_k = q < C::CI;
      const int i = is_k ? q : q - C::CI;
      // 16-byte cell 64 i + lane of the tile: chunk position cell % CPR of row cell / CPR
      const int r = C::ROT ? (64 * i + lane) / C::CPR : i * (64 / C::CPR) + lane / C::CPR;
      const int c = C::chunk_at(r, C::ROT ? (64 * i + lane) % C::CPR : lane % C::CPR);
      code_r[j] = is_k ? kr : vr;
      code_ss[j] = is_k ? p.kc_ss : p.vc_ss;
      code_vo[j] = (uint32_t)(r * code_ss[j] + 16 * c);
      code_lds[j] = (is_k ? 0 : C::KB) + 1024 * i;
    }
#pragma unroll
    for (int j = 0; j < SBN; ++j) {
      const int w = C::SB_ALL || code_on ? wave : 0;
      const int a = C::sb_array(w, j), part = C::sb_part(w, j);
      const int cell = 64 * part + lane;  // cell cell % PC of key cell / PC
      sb_r[j] = a == 0 ? sr[0] : a == 1 ? sr[1] : a == 2 ? sr[2] : sr[3];
      sb_ss[j] = C::DENSE ? 0 : 2 * (a < 2 ? p.ksb_ss : p.vsb_ss);
      sb_vo[j] = (uint32_t)((cell / C::PC) * sb_ss[j] + (C::CELL1 ? 2 : 4) * (cell % C::PC));
      sb_lds[j] = 2 * C::KB + C::SBB * a + 256 * part;
    }
  }
  // raw tile of keys [k0, k0 + 64) into the slot at LDS address `slot`
  __device__ __forceinline__ void issue(uint32_t slot, int k0) const {
    if (code_on) {
#pragma unroll
      for (int j = 0; j < C::CPW; ++j) dma_b128(code_r[j], slot + code_lds[j], code_vo[j], (uint32_t)(k0 * code_ss[j]));
    }
    if (C::SB_ALL || code_on) {
#pragma unroll
      for (int j = 0; j < C::SBW; ++j) dma_sb(sb_r[j], slot + sb_lds[j], sb_vo[j], (uint32_t)(k0 * sb_ss[j]));
    }
  }
  static __device__ __forceinline__ void dma_sb(__amdgpu_buffer_rsrc_t r, uint32_t lds, uint32_t vo, uint32_t so) {
    if constexpr (C::CELL1) {
      dma_b16(r, lds, vo, so);
    } else {
      dma_b32(r, lds, vo, so);
    }
  }

  // Paged cache: the wave's arrays at page 0 of this KV head, and their page strides (bytes).
  const uint8_t* code_base[C::CPW];
  const uint8_t* sb_base[SBN];
  int64_t code_ps[C::CPW], sb_ps[SBN];
  __device__ __forceinline__ void init_paged(const PreParams& p, int kvh, int wave) {
#pragma unroll
    for (int j = 0; j < C::CPW; ++j) {
      const bool is_k = (code_on ? wave * C::CPW + j : 0) < C::CI;
      code_base[j] = is_k ? p.kc + (int64_t)kvh * p.kc_sh : p.vc + (int64_t)kvh * p.vc_sh;
      code_ps[j] = is_k ? p.kc_sb : p.vc_sb;
    }
#pragma unroll
    for (int j = 0; j < SBN; ++j) {
      const int a = C::sb_array(C::SB_ALL || code_on ? wave : 0, j);
      const uint16_t* arr = a == 0 ? p.ks : a == 1 ? p.kb : a == 2 ? p.vs : p.vb;
      sb_base[j] = (const uint8_t*)(arr + (int64_t)kvh * (a < 2 ? p.ksb_sh : p.vsb_sh));
      sb_ps[j] = 2 * (a < 2 ? p.ksb_sb : p.vsb_sb);
    }
  }
  // raw tile of page `pg` (its first nv rows valid) into the slot at LDS address `slot`
  __device__ __forceinline__ void issue_paged(uint32_t slot, int pg, int nv) const {
    if (code_on) {
#pragma unroll
      for (int j = 0; j < C::CPW; ++j)
        dma_b128(make_rsrc(code_base[j] + (int64_t)pg * code_ps[j], (uint32_t)(nv * code_ss[j])), slot + code_lds[j],
                 code_vo[j], 0u);
    }
    if (C::SB_ALL || code_on) {
#pragma unroll
      for (int j = 0; j < C::SBW; ++j)
        dma_sb(make_rsrc(sb_base[j] + (int64_t)pg * sb_ps[j], (uint32_t)(nv * sb_ss[j])), slot + sb_lds[j], sb_vo[j],
               0u);
    }
  }
};

__device__ __forceinline__ _Float16 to_half(uint16_t r, F16) { return __builtin_bit_cast(_Float16, r); }
__device__ __forceinline__ _Float16 to_half(uint16_t r, BF16) { return (_Float16)__uint_as_float((uint32_t)r << 16); }
// A scale or bias as its fp16 operand value times m = 2^-E (the cache's range exponent, include/kvq.h):
// exact in fp32, rounded once. An fp16 cache never needs the factor (its values fit the operands).
__device__ __forceinline__ _Float16 to_half_scaled(uint16_t r, float, F16) { return __builtin_bit_cast(_Float16, r); }
__device__ __forceinline__ _Float16 to_half_scaled(uint16_t r, float m, BF16) {
  return (_Float16)(__uint_as_float((uint32_t)r << 16) * m);
}

// 1024 + c as fp16 for two codes: the code bytes selected by `sel` become the low mantissa bytes of
// 0x64xx (= 1024 + c exactly); subtracting 1024 and one packed FMA give c * s + b in fp16.
constexpr uint32_t kF16x1024 = 0x64646464u;
__device__ __forceinline__ uint32_t dequant_pair(uint32_t bytes, uint32_t sel, h2 s2, h2 b2) {
  h2 x = __builtin_bit_cast(h2, perm(kF16x1024, bytes, sel)) - h2{(_Float16)1024.0f, (_Float16)1024.0f};
  x = x * s2 + b2;
  return __builtin_bit_cast(uint32_t, x);
}

// The 8 codes of `n` (8-bit: two words; 4-bit: one word) dequantized to 4 fp16 pairs (dims 2m, 2m+1).
template <int BITS>
__device__ __forceinline__ void dequant8(const uint32_t* w, h2 s2, h2 b2, uint32_t* out) {
  if constexpr (BITS == 8) {
    out[0] = dequant_pair(w[0], 0x04010400u, s2, b2);
    out[1] = dequant_pair(w[0], 0x04030402u, s2, b2);
    out[2] = dequant_pair(w[1], 0x04010400u, s2, b2);
    out[3] = dequant_pair(w[1], 0x04030402u, s2, b2);
  } else {
    const uint32_t lo = w[0] & 0x0F0F0F0Fu, hi = (w[0] >> 4) & 0x0F0F0F0Fu;
    const uint32_t t0 = perm(hi, lo, 0x05010400u), t1 = perm(hi, lo, 0x07030602u);  // codes 0..3, 4..7 as bytes
    out[0] = dequant_pair(t0, 0x04010400u, s2, b2);
    out[1] = dequant_pair(t0, 0x04030402u, s2, b2);
    out[2] = dequant_pair(t1, 0x04010400u, s2, b2);
    out[3] = dequant_pair(t1, 0x04030402u, s2, b2);
  }
}

// Dequantize the raw tile at `raw` into the fp16 operands. Threads 0 .. 64 NSW - 1 (NSW = D / 32
// waves) build V^T: thread t takes the 8 keys of slot chunk t % 8 at dims [4 (t / 8), +4) and writes
// 4 V^T rows of 8 slots. The next 64 NSW threads build K: thread 64 NSW + u takes dims [32 q, +32)
// of key u % 64, q = u / 64. Threads beyond take no part.
//
// V^T, first part: the wave's lanes convert the scale and bias of the wave's group (dims
// [32 w, 32 w + 32) lie in one group) for the 64 keys (lane = key) into a per-wave table of fp16
// (scale, bias) pairs, which stage_v then reads for its 8 keys. Only this wave touches its table,
// and the LDS operations of one wave complete in program order, so a wave barrier (which keeps
// the compiler from moving the lanes' accesses across it) is all the ordering the reads need.
template <typename T, int BITS, int G, int D>
__device__ __forceinline__ void stage_v_table(const uint8_t* raw, uint32_t* sbt, int tid, bool& range_bad, float vmul) {
  using C = RawCfg<BITS, G, D>;
  const int key = tid & 63, g = (4 * (tid >> 3)) / G;
  const uint8_t* sbase = raw + 2 * C::KB + C::sb_off(key, g);
  const uint16_t sv = *(const uint16_t*)(sbase + 2 * C::SBB), bv = *(const uint16_t*)(sbase + 3 * C::SBB);
  const h2 sbp = {to_half_scaled(sv, vmul, T{}), to_half_scaled(bv, vmul, T{})};
  sbt[key] = __builtin_bit_cast(uint32_t, sbp);
  // a bf16 group beyond the fp16 range has a bias (its largest-magnitude element) that converts to
  // inf; the operands cannot hold it
  if constexpr (T::id == KVQ_DTYPE_BF16) range_bad |= __builtin_isinf((float)sbp[1]);
}

// V^T, second part (after stage_v_table of the same tile), in two halves: half H builds dims
// 4 d4 + 2H and + 2H + 1 (V^T rows 2H, 2H + 1 of the thread's four).
template <int BITS, int G, int D, int H>
__device__ __forceinline__ void stage_v(const uint8_t* raw, _Float16* vlds, const uint32_t* sbt, int tid) {
  using C = RawCfg<BITS, G, D>;
  const int c8 = tid & 7, d4 = tid >> 3;
  // key i of the chunk is kb + v_key_offset(i), and its swizzle swz(key) is
  // (((kb % CPR) | (i & 3)) ^ (kb >> 4)) % CPR: kb has its low two bits clear and kb % 16 is 0 or
  // 4, the offsets are i & 3 modulo 8 and below 12 (so key >> 4 == kb >> 4), CPR is a power of
  // two. Four code addresses per lane; everything else is an immediate offset
  const int kb = v_base_key(c8);
  const uint8_t* vr = raw + C::KB + kb * C::ROWB;
  uint32_t x[8];  // key i: the dim pair of this half
#pragma unroll
  for (int i = 0; i < 8; ++i) {
    const int ko = v_key_offset(i);
    const int sw = (((kb % C::CPR) | (i & 3)) ^ (kb >> 4)) % C::CPR;
    // (rotated rows depend on key >> 4 alone: one address per lane)
    auto at = [&](int c) { return C::ROT ? C::pos(kb, c) : c ^ sw; };
    uint32_t bytes;  // codes of dims 4 d4 .. 4 d4 + 3 as 4 bytes
    if constexpr (BITS == 8) {
      bytes = *(const uint32_t*)(vr + ko * C::ROWB + 16 * at(d4 >> 2) + 4 * (d4 & 3));
    } else {
      const uint32_t h = *(const uint16_t*)(vr + ko * C::ROWB + 16 * at(d4 >> 3) + 2 * (d4 & 7));
      bytes = perm((h >> 4) & 0x0F0Fu, h & 0x0F0Fu, 0x05010400u);
    }
    const h2 sbp = __builtin_bit_cast(h2, sbt[kb + ko]);
    const _Float16 sh = sbp[0], bh = sbp[1];
    x[i] = dequant_pair(bytes, H == 0 ? 0x04010400u : 0x04030402u, h2{sh, sh}, h2{bh, bh});
  }
#pragma unroll
  for (int e = 2 * H; e < 2 * H + 2; ++e) {
    const uint32_t sel = (e & 1) ? 0x07060302u : 0x05040100u;
    u4 v;
#pragma unroll
    for (int ip = 0; ip < 4; ++ip) v[ip] = perm(x[2 * ip + 1], x[2 * ip], sel);
    *(u4*)&vlds[(4 * d4 + e) * kVS + 8 * c8] = v;
  }
}

// K, in two halves: half H builds dims [32 q + 16 H, +16) of key u % 64.
template <typename T, int BITS, int G, int D, int H>
__device__ __forceinline__ void stage_k(const uint8_t* raw, _Float16* klds, int tid, bool& range_bad, float kmul) {
  using C = RawCfg<BITS, G, D>;
  const int u = tid - 64 * C::NSW;
  const int key = u & 63, q = u >> 6;
  const uint8_t* kr = raw + key * C::ROWB;
  uint32_t w[4];  // the half's 16 codes
  if constexpr (BITS == 8) {
    const u4 a = *(const u4*)(kr + 16 * C::pos(key, 2 * q + H));
#pragma unroll
    for (int i = 0; i < 4; ++i) w[i] = a[i];
  } else {
    const u2 a = *(const u2*)(kr + 16 * C::pos(key, q) + 8 * H);
    w[0] = a[0];
    w[1] = a[1];
  }
  const uint8_t* sbase = raw + 2 * C::KB + C::sb_off(key, (32 * q + 16 * H) / G);
  const _Float16 sh = to_half_scaled(*(const uint16_t*)sbase, kmul, T{});
  const _Float16 bh = to_half_scaled(*(const uint16_t*)(sbase + C::SBB), kmul, T{});
  if constexpr (T::id == KVQ_DTYPE_BF16) range_bad |= __builtin_isinf((float)bh);
#pragma unroll
  for (int c = 0; c < 2; ++c) {
    uint32_t x[4];
    dequant8<BITS>(&w[(BITS / 4) * c], h2{sh, sh}, h2{bh, bh}, x);
    *(u4*)&klds[key * kKS<D> + 32 * q + 16 * H + 8 * c] = u4{x[0], x[1], x[2], x[3]};
  }
}

// The whole tile, all threads.
template <typename T, int BITS, int G, int D>
__device__ __forceinline__ void stage_from_raw(const uint8_t* raw, _Float16* klds, _Float16* vlds, uint32_t* sbt,
                                               int tid, bool& range_bad, float kmul, float vmul) {
  constexpr int NST = 64 * RawCfg<BITS, G, D>::NSW;  // threads per operand
  if (tid < NST) {
    stage_v_table<T, BITS, G, D>(raw, sbt, tid, range_bad, vmul);
    __builtin_amdgcn_wave_barrier();
    stage_v<BITS, G, D, 0>(raw, vlds, sbt, tid);
    stage_v<BITS, G, D, 1>(raw, vlds, sbt, tid);
  } else if (tid < 2 * NST) {
    stage_k<T, BITS, G, D, 0>(raw, klds, tid, range_bad, kmul);
    stage_k<T, BITS, G, D, 1>(raw, klds, tid, range_bad, kmul);
  }
}

// Unquantized cache: build half of V^T from the raw V rows of a tile (phase 0: slots 0-31, phase
// 1: slots 32-63). Thread t (0 .. 2 D - 1; the others take no part) takes slot chunk c8 = 4 phase + t % 4
// and dims 2 (t / 4), 2 (t / 4) + 1: 8 keys x 2 dims read as 32-bit words, written as two 8-slot V^T
// rows.
template <int D>
__device__ __forceinline__ void stage_v_raw(const uint8_t* raw, _Float16* vlds, int t, int phase) {
  using C = RawCfg<16, 64, D>;
  if (D < 128 && t >= 2 * D) return;
  const int c8 = 4 * phase + (t & 3), d2 = t >> 2;
  const uint8_t* vr = raw + C::KB;
  uint32_t w[8];
#pragma unroll
  for (int i = 0; i < 8; ++i) {
    const int key = v_slot_key(8 * c8 + i);
    w[i] = *(const uint32_t*)(vr + key * C::ROWB + 16 * ((d2 >> 2) ^ C::swz(key)) + 4 * (d2 & 3));
  }
  u4 lo, hi;
#pragma unroll
  for (int a = 0; a < 4; ++a) {
    lo[a] = perm(w[2 * a + 1], w[2 * a], 0x05040100u);
    hi[a] = perm(w[2 * a + 1], w[2 * a], 0x07060302u);
  }
  *(u4*)&vlds[(2 * d2) * kVS + 8 * c8] = lo;
  *(u4*)&vlds[(2 * d2 + 1) * kVS + 8 * c8] = hi;
}

// Whether a split's partial rows are kept in fp32: for the calls that kernels with fp32 partials served before
// this one (head_dim 96 and general masks the decode kernel, unquantized head_dim 64 the head_dim-256
// kernel's form of that width). The others pack them to fp16, which their workspaces are sized for.
template <int BITS, int D, int MASKED>
constexpr bool kF32Partials = MASKED != 0 || D == 96 || (BITS == 16 && D == 64);

// MASKED: 0, or under a general mask: 1 boolean, 2 additive. The tile loop then walks the list of tiles
// with a visible key, and reads the mask beside those that are not visible as a whole.
template <typename T, int BITS, bool PAGED = false, int G = 64, int D = 128, int MASKED = 0>
__global__ __launch_bounds__(kPW * 64, 1) void prefill_attn_kernel(PreParams p) {
  static_assert(!(PAGED && MASKED), "general masks: contiguous caches");
  using RC = RawCfg<BITS, G, D>;
  constexpr bool DENSE = RC::DENSE;  // unquantized cache: K operands are read from the raw ring
  constexpr int KS = kKS<D>;
  constexpr int KSTEPS = D / 16;   // k-steps of S^T = K Q^T over the head dimension
  constexpr int NDB = D / 32;      // 32-dim blocks of O^T
  constexpr int QW = D / 16;       // 16-byte words of a lane's packed output row
  __shared__ __align__(16) _Float16 k_lds[DENSE ? 1 : 3][DENSE ? 8 : kPT * KS];
  __shared__ __align__(16) _Float16 v_lds[DENSE ? 2 : 3][D * kVS];
  __shared__ __align__(16) uint8_t raw[kRawSlots][RC::SLOT];
  __shared__ uint32_t sb_tab[DENSE ? 1 : kPW / 2][64];  // per V^T-building wave: (scale, bias) pairs
  // after the tile loop the table's storage holds per-wave flags (words 0-7) and the split arrival
  // count (word 8): the LDS budget has no room for more
  unsigned* const s_flags = &sb_tab[0][0];
  unsigned* const s_arrived = &sb_tab[0][8];
  bool range_bad = false;  // some tile this lane staged held a group beyond the fp16 range
  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int qc = lane & 31, hh = lane >> 5;

  const PreWg wg = prefill_wg(p, (int)blockIdx.x, (int)gridDim.x);
  const int rb = wg.rb, split = wg.split, bk = wg.bk;  // bk = b * Hkv + kvh
  const int b = bk / p.Hkv, kvh = bk % p.Hkv;
  const int unit = bk * p.rowblocks + rb;
  const int S_b = p.seq_lens ? min(max(load_uniform_i32(p.seq_lens, b), 0), p.S) : p.S;

  // ---- the workgroup's rows, their positions, and the key range they see
  const int fr0 = rb * kPRows;
  const int frl = min(fr0 + kPRows, p.nrows) - 1;
  KeySplit ks;
  MaskSplit ms;
  if constexpr (MASKED) {
    ms = split_masked(p, b, kvh, rb);
  } else {
    ks = split_keys(p, S_b, fr0, frl);
  }
  const int nsplit = MASKED ? ms.nsplit : ks.nsplit;
  if (split >= nsplit) return;
  const int pos_min = S_b - p.L + fr0 / p.rep, pos_max = S_b - p.L + frl / p.rep;
  // keys every row of the workgroup sees: tiles inside need no mask
  const int hi_all = p.causal ? min(S_b, pos_min + 1) : S_b;
  const int lo_all = p.window > 0 ? max(0, pos_max - p.window + 1) : 0;
  int k_begin = 0, ntile;  // tile starts stay 64-aligned
  if constexpr (MASKED) {
    ntile = __builtin_amdgcn_readfirstlane(max(min(ms.chunk, ms.n - split * ms.chunk), 0));
  } else {
    k_begin = ks.lo + split * ks.chunk;
    const int k_end = min(k_begin + ks.chunk, ks.hi);
    ntile = k_end > k_begin ? (k_end - k_begin + kPT - 1) / kPT : 0;
  }
  // under a mask: the walk over the listed tiles (the word in hand, its index, tiles left to hand out),
  // and the tiles handed out but not yet computed, in order (bit 31: mixed)
  uint64_t wk_any = 0, wk_mixed = 0;
  int wk_w = -1, wk_left = ntile, wk_last = 0;
  int tq[4] = {0, 0, 0, 0};
  auto next_tile = [&]() -> int {
    if (wk_left > 0) {
      while (wk_any == 0) {
        ++wk_w;
        wk_any = uniform64(load_uniform_u64(ms.any, wk_w));
        wk_mixed = uniform64(load_uniform_u64(ms.any, p.nwords + wk_w));
      }
      const int i = __builtin_ctzll(wk_any);
      wk_any &= wk_any - 1;
      --wk_left;
      wk_last = (64 * wk_w + i) | ((int)((wk_mixed >> i) & 1) << 31);
    }
    return __builtin_amdgcn_readfirstlane(wk_last);  // past the last tile it is handed out again
  };
  if constexpr (MASKED) {
    if (ntile > 0) {
      // skip the tiles of the splits before this one
      int skip = split * ms.chunk;
      for (;;) {
        ++wk_w;
        wk_any = uniform64(load_uniform_u64(ms.any, wk_w));
        const int c = __builtin_popcountll(wk_any);
        if (skip < c) break;
        skip -= c;
      }
      for (; skip > 0; --skip) wk_any &= wk_any - 1;
      wk_mixed = uniform64(load_uniform_u64(ms.any, p.nwords + wk_w));
    }
  }

  // ---- this lane's query row (MFMA column qc of this wave)
  const int fr = fr0 + wave * 32 + qc;
  const bool row_ok = fr < p.nrows;
  const int lq = row_ok ? fr / p.rep : 0;
  const int head = kvh * p.rep + (row_ok ? fr % p.rep : 0);
  const int pos = S_b - p.L + lq;
  const int lo_r = p.window > 0 ? max(0, pos - p.window + 1) : 0;
  const int hi_r = p.causal ? min(S_b, pos + 1) : S_b;

  // ---- the raw query slice (loaded before the tile stream; row and head are clamped, so every
  // lane's load is in bounds)
  u4 qraw[KSTEPS];
  {
    const uint16_t* qrow = p.q + (int64_t)b * p.q_sb + (int64_t)head * p.q_sh + (int64_t)lq * p.q_sl + 8 * hh;
#pragma unroll
    for (int j = 0; j < KSTEPS; ++j) qraw[j] = *(const u4*)(qrow + 16 * j);
  }

  // ---- raw tile stream: buffer resources over the S_b valid rows of this (sequence, KV head)
  // (the host checks S * row stride fits 32 bits); tiles past the last re-read the last one
  RawShare<BITS, G, D> share;
  {
    const __amdgpu_buffer_rsrc_t kr =
        make_rsrc(p.kc + (int64_t)b * p.kc_sb + (int64_t)kvh * p.kc_sh, (uint32_t)((int64_t)S_b * p.kc_ss));
    const __amdgpu_buffer_rsrc_t vr =
        make_rsrc(p.vc + (int64_t)b * p.vc_sb + (int64_t)kvh * p.vc_sh, (uint32_t)((int64_t)S_b * p.vc_ss));
    const int64_t ko = (int64_t)b * p.ksb_sb + (int64_t)kvh * p.ksb_sh;
    const int64_t vo = (int64_t)b * p.vsb_sb + (int64_t)kvh * p.vsb_sh;
    const uint32_t kn = (uint32_t)((int64_t)S_b * p.ksb_ss * 2), vn = (uint32_t)((int64_t)S_b * p.vsb_ss * 2);
    __amdgpu_buffer_rsrc_t sr[4] = {kr, kr, kr, kr};
    if constexpr (!DENSE) {
      sr[0] = make_rsrc(p.ks + ko, kn);
      sr[1] = make_rsrc(p.kb + ko, kn);
      sr[2] = make_rsrc(p.vs + vo, vn);
      sr[3] = make_rsrc(p.vb + vo, vn);
    }
    share.init(p, kr, vr, sr, wave, lane);
    if constexpr (PAGED) share.init_paged(p, kvh, wave);
  }
  const uint32_t raw_lds = lds_addr(&raw[0][0]);
  const int last = max(ntile - 1, 0);
  // paged cache: a tile (64 rows, 64-aligned) is one page; its page number is read one tile ahead
  // (a scalar load), clamped to the pool, and the tile's buffer resources span only that page's
  // valid rows, so rows past S_b still read as zero
  auto page_of = [&](int k0) -> int {
    const int pi = min(k0, max(S_b - 1, 0)) >> 6;
    return __builtin_amdgcn_readfirstlane(min(max(p.table[(int64_t)b * p.table_stride + pi], 0), p.num_pages - 1));
  };
  int pg_next = PAGED ? page_of(k_begin) : 0;
  auto issue_raw = [&](int i) {
    int k0 = k_begin + kPT * min(i, last);
    if constexpr (MASKED) {  // tiles are issued in order, each once: the queue holds those not computed yet
      const int e = next_tile();
      tq[min(i, DENSE ? 2 : 3)] = e;
      k0 = kPT * (e & 0x7fffffff);
    }
    const uint32_t slot = raw_lds + (i % kRawSlots) * RC::SLOT;
    if constexpr (PAGED) {
      const int pg = pg_next;
      pg_next = page_of(k_begin + kPT * min(i + 1, last));
      share.issue_paged(slot, pg, __builtin_amdgcn_readfirstlane(max(min(kPT, S_b - k0), 0)));
    } else {
      share.issue(slot, k0);
    }
  };
  // the first tiles of the ring (the tile loops below say how far ahead each runs)
  if (ntile > 0) {
#pragma unroll
    for (int j = 0; j < (DENSE ? 2 : kRawSlots); ++j) issue_raw(j);
  }

  // ---- range exponents of the K and V caches (0 for an unquantized cache, an fp16 cache -- whose
  // values always fit the fp16 operands -- or a null pointer) and the factors 2^-E the staging
  // applies to the scales and biases; 2^E_K returns in the score scale, 2^E_V in the output. Read
  // here, after the first tile loads are issued, so that waiting for the word delays no load. (The
  // factors are held in VGPRs: the tile loop has spare vector registers and no spare scalar ones.)
  float kmul = 1.0f, vmul = 1.0f, kback = 1.0f, vback = 1.0f;
  if constexpr (!DENSE && T::id == KVQ_DTYPE_BF16) {
    const int ek = p.k_rexp ? min(max(*p.k_rexp, 0), 127) : 0;
    const int ev = p.v_rexp ? min(max(*p.v_rexp, 0), 127) : 0;
    kmul = ldexpf(1.0f, -ek);
    vmul = ldexpf(1.0f, -ev);
    kback = ldexpf(1.0f, ek);
    vback = ldexpf(1.0f, ev);
    asm volatile("" : "+v"(kmul), "+v"(vmul), "+v"(kback), "+v"(vback));
  }

  // ---- Q^T operand: k-step j holds dims 16j + 8hh .. +7. Quantized cache: the query times 2^qe in
  // fp16 (exact: a power of two, with qe chosen so the row's largest element lands in [2^13, 2^14);
  // a bf16 query has 8 significant bits, so only elements below 2^-14 of the operand's scale lose
  // bits), and the scores are multiplied by inv2 = scale * log2(e) * 2^-qe in fp32. Folding the
  // softmax scale into the fp16 operand instead would round every query element. Unquantized
  // cache: the raw query (exact), the scores multiplied by scale*log2(e) in fp32.
  u4 qop[KSTEPS];
  float inv2;
  if constexpr (DENSE) {
#pragma unroll
    for (int j = 0; j < KSTEPS; ++j) qop[j] = row_ok ? qraw[j] : u4{0, 0, 0, 0};
    inv2 = p.scale_log2;
  } else {
    float qv[KSTEPS][8];
    float qmax = 0.0f;
#pragma unroll
    for (int j = 0; j < KSTEPS; ++j) {
      const u4 raw_q = row_ok ? qraw[j] : u4{0, 0, 0, 0};
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        qv[j][2 * i] = to_float((uint16_t)(raw_q[i] & 0xffffu), T{});
        qv[j][2 * i + 1] = to_float((uint16_t)(raw_q[i] >> 16), T{});
        qmax = fmaxf(qmax, fmaxf(fabsf(qv[j][2 * i]), fabsf(qv[j][2 * i + 1])));
      }
    }
    qmax = max_xor32(qmax);
    int e = 0;
    if (qmax > 0.0f) frexpf(qmax, &e);
    const int qe = 14 - e;  // |q| * 2^qe < 2^14
    const float qmul = ldexpf(1.0f, qe);
    inv2 = ldexpf(p.scale_log2, -qe) * kback;  // the K operands are staged times 2^-E_K
#pragma unroll
    for (int j = 0; j < KSTEPS; ++j)
#pragma unroll
      for (int i = 0; i < 4; ++i) qop[j][i] = pack_f16x2(qv[j][2 * i] * qmul, qv[j][2 * i + 1] * qmul);
  }
  // ---- under a mask the scores are brought to log2 units as they are masked (an additive mask is added
  // there), so the softmax that follows applies no scale of its own
  const float sinv = MASKED ? 1.0f : inv2;
  const uint8_t* mrow = nullptr;
  if constexpr (MASKED) {
    const int el = MASKED == 1 ? 1 : p.mask_kind == KVQ_MASK_F32 ? 4 : 2;
    mrow = (const uint8_t*)p.mask +
           el * ((int64_t)b * p.m_sb + (int64_t)kvh * p.m_skv + (int64_t)(head - kvh * p.rep) * p.m_srep + (int64_t)lq * p.m_sl);
  }
  // the 16 scores of the 32-key block from k (this lane's keys k + 8 c + 4 hh + e, its mask row mrow)
  auto general_mask = [&](f16v& acc, int k, bool mixed) {
    if (!mixed) {
#pragma unroll
      for (int i = 0; i < 16; ++i) acc[i] *= inv2;
      return;
    }
    const bool whole = k + 32 <= p.S;  // else the row of the mask ends inside the block
#pragma unroll
    for (int c = 0; c < 4; ++c) {
      const int t = k + 8 * c + 4 * hh;
      if constexpr (MASKED == 1) {
        uint32_t m = 0;
        if (whole) {
          __builtin_memcpy(&m, mrow + t, 4);
        } else {
#pragma unroll
          for (int e = 0; e < 4; ++e)
            if (t + e < p.S) m |= (uint32_t)mrow[t + e] << (8 * e);
        }
#pragma unroll
        for (int e = 0; e < 4; ++e)
          acc[4 * c + e] = (m >> (8 * e)) & 0xffu ? acc[4 * c + e] * inv2 : -INFINITY;
      } else {
        float a[4] = {-INFINITY, -INFINITY, -INFINITY, -INFINITY};
        if (p.mask_kind == KVQ_MASK_F32) {
          if (whole) {
            __builtin_memcpy(a, mrow + 4 * (int64_t)t, 16);
          } else {
#pragma unroll
            for (int e = 0; e < 4; ++e)
              if (t + e < p.S) a[e] = ((const float*)mrow)[t + e];
          }
        } else {
          uint16_t r[4] = {0, 0, 0, 0};
          if (whole) {
            __builtin_memcpy(r, mrow + 2 * (int64_t)t, 8);
          } else {
#pragma unroll
            for (int e = 0; e < 4; ++e)
              if (t + e < p.S) r[e] = ((const uint16_t*)mrow)[t + e];
          }
#pragma unroll
          for (int e = 0; e < 4; ++e)
            if (whole || t + e < p.S) a[e] = p.mask_kind == KVQ_MASK_BF16 ? to_float(r[e], BF16{}) : to_float(r[e], F16{});
        }
#pragma unroll
        for (int e = 0; e < 4; ++e) acc[4 * c + e] = fmaf(acc[4 * c + e], inv2, a[e] * 1.4426950408889634f);
        if (!whole) {  // keys past the end stay hidden whatever their score was
#pragma unroll
          for (int e = 0; e < 4; ++e)
            if (t + e >= p.S) acc[4 * c + e] = -INFINITY;
        }
      }
    }
  };
  // MFMA operand type: bf16 for an unquantized bf16 cache, else fp16
  using OT = typename std::conditional<DENSE && T::id == KVQ_DTYPE_BF16, BF16, F16>::type;

  float m_run = -INFINITY, l_run = 0.0f;
  f16v oacc[NDB];
#pragma unroll
  for (int db = 0; db < NDB; ++db) oacc[db] = f16v{};

  if constexpr (DENSE) {
    // ---- the pieces of a tile step
    // this lane's query sees keys k0 + 32kb + 8(i/4) + 4hh + i%4. Only tiles on a causal diagonal or
    // window edge need a mask (a branch the whole workgroup takes or skips); there, each element's
    // offset c = 32kb + 8(i/4) + i%4 is a constant compared with the lane's bounds
    auto mask_tile = [&](f16v (&acc)[2], int k0) {
      if constexpr (MASKED) {
        general_mask(acc[0], kPT * (tq[0] & 0x7fffffff), tq[0] < 0);
        general_mask(acc[1], kPT * (tq[0] & 0x7fffffff) + 32, tq[0] < 0);
        tq[0] = tq[1];
        tq[1] = tq[2];
        return;
      }
      const bool need_mask = !(k0 >= lo_all && k0 + kPT <= hi_all);
      if (__builtin_expect(need_mask, 0)) {
        const int lo = lo_r - k0 - 4 * hh, hi = hi_r - k0 - 4 * hh;
        if (lo <= 0) {  // no key of the tile is below the lane's window
#pragma unroll
          for (int kb = 0; kb < 2; ++kb)
#pragma unroll
            for (int i = 0; i < 16; ++i)
              if (32 * kb + 8 * (i >> 2) + (i & 3) >= hi) acc[kb][i] = -INFINITY;
        } else {
#pragma unroll
          for (int kb = 0; kb < 2; ++kb)
#pragma unroll
            for (int i = 0; i < 16; ++i) {
              const int c = 32 * kb + 8 * (i >> 2) + (i & 3);
              if (c < lo || c >= hi) acc[kb][i] = -INFINITY;
            }
        }
      }
    };
    // the tile's row maximum in log2 units; the running maximum moves (and the accumulators are
    // rescaled) only when it exceeds the running one by more than the slack
    auto update_max = [&](const f16v (&acc)[2]) {
      float tm = -INFINITY;
#pragma unroll
      for (int kb = 0; kb < 2; ++kb)
#pragma unroll
        for (int i = 0; i < 16; ++i) tm = fmaxf(tm, acc[kb][i]);
      tm = max_xor32(tm) * sinv;
      if (__builtin_amdgcn_ballot_w64(tm > m_run + kPSlack) != 0) {
        const float m_new = tm > m_run + kPSlack ? fmaxf(m_run, tm) : m_run;
        const float corr = m_new == m_run ? 1.0f : exp2_fast(m_run - m_new);
        l_run *= corr;
#pragma unroll
        for (int db = 0; db < NDB; ++db)
#pragma unroll
          for (int i = 0; i < 16; ++i) oacc[db][i] *= corr;
        m_run = m_new;
      }
    };
    // p = 2^(acc * inv2 - m): rounded to the operand type it is the B operand of O^T = V^T P^T; the
    // row sum is kept in fp32 (of the rounded values, so the output stays a convex combination of V
    // rows), in two chains
    auto probs = [&](const f16v (&acc)[2], u4 (&pop)[4]) {
      const float nm = m_run == -INFINITY ? 0.0f : -m_run;
      float lsum[2] = {0.0f, 0.0f};
#pragma unroll
      for (int j = 0; j < 4; ++j) {
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const float p0 = exp2_fast(fmaf(acc[j >> 1][8 * (j & 1) + 2 * e], sinv, nm));
          const float p1 = exp2_fast(fmaf(acc[j >> 1][8 * (j & 1) + 2 * e + 1], sinv, nm));
          pop[j][e] = pack2(p0, p1, OT{});
          lsum[e & 1] = add_pair(pop[j][e], lsum[e & 1], OT{});
        }
      }
      l_run += lsum[0] + lsum[1];
    };
    // O^T += V^T P^T: the 4 NDB V^T operands stream through a 4-deep register ring; the NDB dim blocks
    // alternate. vl = this lane's start in a V^T buffer.
    auto pv = [&](const _Float16* vl, const u4 (&pop)[4]) {
      auto vop = [&](int i) { return *(const u4*)(vl + (i % NDB) * 32 * kVS + 16 * (i / NDB)); };
      u4 ring[4] = {vop(0), vop(1), vop(2), vop(3)};
#pragma unroll
      for (int i = 0; i < 4 * NDB; ++i) {
        oacc[i % NDB] = mfma_32x32x16(ring[i & 3], pop[i / NDB], oacc[i % NDB], OT{});
        if (i + 4 < 4 * NDB) ring[i & 3] = vop(i + 4);
      }
    };

    // ---- unquantized cache: K operands are read from the raw ring while tile t is computed, so
    // tile t + 2 is issued into the slot of tile t - 1 and lands within the step (issued once the
    // step's QK MFMAs are, which measured 4-5% faster than at the step's start); V^T is built from
    // the raw rows into a double buffer, half by waves 4-7 before their MFMAs and half by waves 0-3
    // after theirs (the two waves that share a SIMD are in opposite phases)
    if (ntile > 0) {
      wait_vm<0>();
      __syncthreads();
      stage_v_raw<D>(raw[0], v_lds[0], tid & 255, tid >> 8);
      __syncthreads();
    }
    // this lane's K operand bytes within a raw slot: key row 32 (i & 1) + qc, 16-byte chunk
    // 2 (i >> 1) + hh at its swizzled position
    const int kswz = RC::swz(qc);
    for (int t = 0; t < ntile; ++t) {
      const int cur = t & 1;
      const int k0 = k_begin + kPT * t;
      if (t + 1 < ntile && wave >= kPW / 2) stage_v_raw<D>(raw[(t + 1) % kRawSlots], v_lds[cur ^ 1], tid - 256, 0);
      f16v sacc[2] = {f16v{}, f16v{}};
      {
        const uint8_t* kraw = raw[t % kRawSlots] + qc * RC::ROWB;
        auto kop = [&](int i) -> u4 {
          return *(const u4*)(kraw + (i & 1) * 32 * RC::ROWB + 16 * ((2 * (i >> 1) + hh) ^ kswz));
        };
        u4 ring[4] = {kop(0), kop(1), kop(2), kop(3)};
#pragma unroll
        for (int i = 0; i < 2 * KSTEPS; ++i) {
          sacc[i & 1] = mfma_32x32x16(ring[i & 3], qop[i >> 1], sacc[i & 1], OT{});
          if (i + 4 < 2 * KSTEPS) ring[i & 3] = kop(i + 4);
        }
      }
      if (t + 2 < ntile) issue_raw(t + 2);  // into the slot of tile t - 1 (read in the last step)
      mask_tile(sacc, k0);
      update_max(sacc);
      u4 pop[4];
      probs(sacc, pop);
      pv(&v_lds[cur][qc * kVS + 8 * hh], pop);
      if (t + 1 < ntile && wave < kPW / 2) stage_v_raw<D>(raw[(t + 1) % kRawSlots], v_lds[cur ^ 1], tid, 1);
      wait_vm<0>();  // tile t + 2 has landed
      __syncthreads();
    }
  } else if (ntile > 0) {
    // ---- quantized cache, software-pipelined over 32-key blocks. Step t (tile t) runs two halves;
    // half h takes the scores of block h of the tile, already computed, and
    //  * takes their row maximum (and the rare rescale) first, then issues the MFMAs of the next
    //    block's scores (block 1 of tile t, then block 0 of tile t + 1) and runs the exponentials
    //    while they execute (the maximum first measured about 1% faster than after two MFMAs), then
    //  * accumulates O += V P for the block while the dequantizing waves build half of tile t + 2
    //    (the V^T waves its V^T, the K waves its K),
    // so every wave always has MFMA work beside its VALU work, and two 16-register score blocks are
    // live rather than two tiles.
    //  * fp16 operands: tile j in k_lds[j % 3] and v_lds[j % 3] (step t reads K of tiles t and
    //    t + 1 and V of tile t, and writes tile t + 2);
    //  * raw ring: tile j in slot j % 3; step t reads tile t + 2 and issues tile t + 4 into the slot
    //    of tile t + 1 (dequantized in step t - 1), so every tile is loaded two steps ahead;
    //  * one barrier per step orders all of it.
    constexpr int KBUF = kPT * KS, VBUF = D * kVS;
    const _Float16* kl_lane = &k_lds[0][qc * KS + 8 * hh];  // this lane's K operands, V^T operands
    const _Float16* vl_lane = &v_lds[0][qc * kVS + 8 * hh];
    // S^T = K Q^T for the 32-key block whose K rows start at kl (this lane's offset included):
    // KSTEPS MFMAs over the head dimension, the K operands streamed through a 4-deep register ring
    // (deeper rings of 6 and 8, and an 8-deep V^T ring, measured slower); MFMAs [J0, J1) of them
    auto qk_ring = [&](u4 (&ring)[4], const _Float16* kl) {
#pragma unroll
      for (int j = 0; j < 4; ++j) ring[j] = *(const u4*)(kl + 16 * j);
    };
    auto qk_run = [&](auto j0, auto j1, f16v& acc, u4 (&ring)[4], const _Float16* kl) {
#pragma unroll
      for (int j = decltype(j0)::value; j < decltype(j1)::value; ++j) {
        acc = mfma_32x32x16(ring[j & 3], qop[j], j == 0 ? f16v{} : acc, OT{});
        if (j + 4 < KSTEPS) ring[j & 3] = *(const u4*)(kl + 16 * (j + 4));
      }
    };
    using J0 = std::integral_constant<int, 0>;
    using JE = std::integral_constant<int, KSTEPS>;
    // the block's keys [k, k + 32): mask (only on a causal diagonal or window edge), row maximum
    auto mask_blk = [&](f16v& acc, int k, int entry) {
      if constexpr (MASKED) {
        general_mask(acc, k, entry < 0);
        return;
      }
      if (__builtin_expect(!(k >= lo_all && k + 32 <= hi_all), 0)) {
        const int lo = lo_r - k - 4 * hh, hi = hi_r - k - 4 * hh;
#pragma unroll
        for (int i = 0; i < 16; ++i) {
          const int c = 8 * (i >> 2) + (i & 3);
          if (c < lo || c >= hi) acc[i] = -INFINITY;
        }
      }
    };
    auto max_blk = [&](const f16v& acc) {
      float tm = -INFINITY;
#pragma unroll
      for (int i = 0; i < 16; ++i) tm = fmaxf(tm, acc[i]);
      return max_xor32(tm) * sinv;
    };
    auto rescale = [&](float tm) {
      if (__builtin_amdgcn_ballot_w64(tm > m_run + kPSlack) != 0) {
        const float m_new = tm > m_run + kPSlack ? fmaxf(m_run, tm) : m_run;
        const float corr = m_new == m_run ? 1.0f : exp2_fast(m_run - m_new);
        l_run *= corr;
#pragma unroll
        for (int db = 0; db < NDB; ++db)
#pragma unroll
          for (int i = 0; i < 16; ++i) oacc[db][i] *= corr;
        m_run = m_new;
      }
    };
    // p = 2^(acc * inv2 - m) for the block's 32 keys: the B operands of its two PV k-steps
    auto probs_blk = [&](const f16v& acc, u4 (&pop)[2]) {
      const float nm = m_run == -INFINITY ? 0.0f : -m_run;
      float lsum[2] = {0.0f, 0.0f};
#pragma unroll
      for (int j = 0; j < 2; ++j)
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const float p0 = exp2_fast(fmaf(acc[8 * j + 2 * e], sinv, nm));
          const float p1 = exp2_fast(fmaf(acc[8 * j + 2 * e + 1], sinv, nm));
          pop[j][e] = pack2(p0, p1, OT{});
          lsum[e & 1] = add_pair(pop[j][e], lsum[e & 1], OT{});
        }
      l_run += lsum[0] + lsum[1];
    };
    // O^T += V^T P^T over block kb's two k-steps (V^T slots 32 kb .. 32 kb + 31): 2 NDB MFMAs, the
    // NDB dim blocks alternating, V^T operands through a 4-deep ring
    auto pv_blk = [&](const _Float16* vl, const u4 (&pop)[2], auto kb) {
      constexpr int KB = decltype(kb)::value;
      auto vop = [&](int i) { return *(const u4*)(vl + (i % NDB) * 32 * kVS + 16 * (2 * KB + i / NDB)); };
      u4 ring[4] = {vop(0), vop(1), vop(2), vop(3)};
#pragma unroll
      for (int i = 0; i < 2 * NDB; ++i) {
        oacc[i % NDB] = mfma_32x32x16(ring[i & 3], pop[i / NDB], oacc[i % NDB], OT{});
        if (i + 4 < 2 * NDB) ring[i & 3] = vop(i + 4);
      }
    };
    using B0 = std::integral_constant<int, 0>;
    using B1 = std::integral_constant<int, 1>;

    // The wave's role: 0 builds V^T (waves [0, NSW)), 1 builds K (waves [NSW, 2 NSW)), 2 only
    // computes (head_dim 64: waves from 2 NSW on). The loop is compiled once per role, so each copy
    // keeps only its own staging addresses live, and waits for its own number of loads per tile.
    static_assert(RC::CODE_WAVES == kPW || RC::CODE_WAVES == 2 * RC::NSW, "computing-only waves all load codes or none");
    f16v sX, sY;  // the scores of block 0 (entering a step: tile t's) and block 1 of a tile
    auto step = [&](auto role, auto qkn, auto stg, int t) {
      constexpr int ROLE = decltype(role)::value;
      constexpr bool QKN = decltype(qkn)::value, STG = decltype(stg)::value;
      constexpr int IPT = (ROLE < 2 || RC::CODE_WAVES == kPW) ? RC::IPT : RC::IPT_NOCODE;
      // the step's buffers, as element (byte, for the raw ring) offsets from each array's start
      const int k_t = opaque((t % 3) * KBUF), k_t1 = opaque(((t + 1) % 3) * KBUF);
      const int k_w = opaque(((t + 2) % 3) * KBUF);
      const int v_t = opaque((t % 3) * VBUF), v_w = opaque(((t + 2) % 3) * VBUF);
      const uint8_t* raw2 = &raw[0][0] + opaque(((t + 2) % kRawSlots) * RC::SLOT);
      if constexpr (STG && ROLE == 0) {
        stage_v_table<T, BITS, G, D>(raw2, sb_tab[wave & 3], tid, range_bad, vmul);
        __builtin_amdgcn_wave_barrier();
      }
      const int entry = MASKED ? tq[0] : 0;
      const int k0 = MASKED ? kPT * (entry & 0x7fffffff) : k_begin + kPT * t;
      if constexpr (MASKED) {
        tq[0] = tq[1];
        tq[1] = tq[2];
        tq[2] = tq[3];
      }
      const _Float16* vl = vl_lane + v_t;
      u4 ring[4];
      u4 pop[2];
      // half 0: softmax of block 0 beside S(block 1) = K(t) rows 32-63 Q^T
      {
        const _Float16* kl = kl_lane + k_t + 32 * KS;
        mask_blk(sX, k0, entry);
        const float tm = max_blk(sX);
        rescale(tm);
        qk_ring(ring, kl);
        qk_run(J0{}, JE{}, sY, ring, kl);
        probs_blk(sX, pop);
      }
      pv_blk(vl, pop, B0{});
      if constexpr (STG && ROLE == 0) stage_v<BITS, G, D, 0>(raw2, &v_lds[0][0] + v_w, sb_tab[wave & 3], tid);
      if constexpr (STG && ROLE == 1) stage_k<T, BITS, G, D, 0>(raw2, &k_lds[0][0] + k_w, tid, range_bad, kmul);
      // tile t + 4 into the slot of tile t + 1, issued between the halves (at the step's start
      // it delays the first half: about 2% slower on C3, as are the other positions tried)
      issue_raw(t + 4);
      // half 1: softmax of block 1 beside S(block 0 of tile t + 1) = K(t + 1) rows 0-31 Q^T
      {
        const _Float16* kl = kl_lane + k_t1;
        mask_blk(sY, k0 + 32, entry);
        const float tm = max_blk(sY);
        rescale(tm);
        if constexpr (QKN) {
          qk_ring(ring, kl);
          qk_run(J0{}, JE{}, sX, ring, kl);
        }
        probs_blk(sY, pop);
      }
      pv_blk(vl, pop, B1{});
      if constexpr (STG && ROLE == 0) stage_v<BITS, G, D, 1>(raw2, &v_lds[0][0] + v_w, sb_tab[wave & 3], tid);
      if constexpr (STG && ROLE == 1) stage_k<T, BITS, G, D, 1>(raw2, &k_lds[0][0] + k_w, tid, range_bad, kmul);
      wait_vm<IPT>();  // tile t + 3 has landed (tile t + 4 may be in flight)
      __syncthreads();
    };
    using Y = std::true_type;
    using N = std::false_type;

    auto run = [&](auto role) {
      constexpr int ROLE = decltype(role)::value;
      constexpr int IPT = (ROLE < 2 || RC::CODE_WAVES == kPW) ? RC::IPT : RC::IPT_NOCODE;
      // prologue: tiles 0 and 1 dequantized, S(tile 0, block 0) computed, tile 2 landed, tile 3 in
      // flight
      wait_vm<2 * IPT>();
      __syncthreads();
      stage_from_raw<T, BITS, G, D>(raw[0], k_lds[0], v_lds[0], sb_tab[wave & 3], tid, range_bad, kmul, vmul);
      wait_vm<IPT>();
      __syncthreads();
      issue_raw(3);  // into the slot of tile 0
      stage_from_raw<T, BITS, G, D>(raw[1], k_lds[1], v_lds[1], sb_tab[wave & 3], tid, range_bad, kmul, vmul);
      {
        u4 ring[4];
        qk_ring(ring, kl_lane);
        qk_run(J0{}, JE{}, sX, ring, kl_lane);
      }
      wait_vm<IPT>();
      __syncthreads();
      int t = 0;
      for (; t + 2 < ntile; ++t) step(role, Y{}, Y{}, t);
      if (t + 1 < ntile) step(role, Y{}, N{}, t++);
      step(role, N{}, N{}, t);
    };
    if (wave < RC::NSW) {
      run(std::integral_constant<int, 0>{});
    } else if constexpr (2 * RC::NSW == kPW) {
      run(std::integral_constant<int, 1>{});
    } else {
      if (wave < 2 * RC::NSW) {
        run(std::integral_constant<int, 1>{});
      } else {
        run(std::integral_constant<int, 2>{});
      }
    }
  }
  wait_vm<0>();  // no load into this workgroup's LDS outlives it
  if constexpr (!DENSE && T::id == KVQ_DTYPE_BF16) {
    // a group beyond the fp16 range poisons the workgroup's rows: NaN propagates through the split
    // merge (0 * NaN is NaN) to every output row of the row block. (The tables are free: the last
    // tile step staged nothing and ended with a barrier.)
    const bool wave_bad = __builtin_amdgcn_ballot_w64(range_bad) != 0;
    if (lane == 0) s_flags[wave] = wave_bad;
    __syncthreads();
    unsigned any_bad = 0;
#pragma unroll
    for (int w = 0; w < kPW; ++w) any_bad |= s_flags[w];
    if (any_bad) {
#pragma unroll
      for (int db = 0; db < NDB; ++db)
#pragma unroll
        for (int i = 0; i < 16; ++i) oacc[db][i] = __builtin_nanf("");
    }
  }

  // ---- epilogue: this lane holds O^T[d][row] for d = 32db + 8(i/4) + 4hh + i%4
  float l_tot = add_xor32(l_run);
  if (nsplit > 1) {
    // Key split: publish this split's partials, count the arrival, and let the unit's last split to
    // arrive merge them into its own registers.
    //  * A partial row is o / l in fp16, times 2^-e with e chosen per row so every stored value is
    //    below 2^14, and the row's record (m, l, 2^e). The merge scales row s by w_s l_s 2^e_s.
    //  * The merging split rounds its own partial through the same fp16 packing, so every split's
    //    term is formed from the same values whichever split merges: the result is
    //    bit-reproducible from call to call.
    //  * The packed row keeps the register image: lane `lane` of wave `wave` of split s holds words
    //    u (0 .. QW - 1) of 16 bytes at byte ((s * kPW + wave) * QW + u) * 1024 + 16 lane of the unit's o
    //    block; word u packs value groups 2u and 2u + 1 (group 4 db + c = oacc[db][4c .. 4c+3]).
    //    Record of row r at byte 16 (s * kPRows + r) of the unit's record block.
    //  * With fp32 partials (kF32Partials) a row is o itself in the cache's units, word u (0 .. 2 QW - 1) value
    //    group u, and its record (m, l), 8 bytes: the merge scales row s by w_s.
    constexpr bool F32P = kF32Partials<BITS, D, MASKED>;
    constexpr int NW = F32P ? 2 * QW : QW;       // 16-byte words of a lane's row
    constexpr uint32_t split_o = kPW * NW * 1024;
    const __amdgpu_buffer_rsrc_t ro =
        make_rsrc((const uint8_t*)p.part_o + (int64_t)unit * p.nsplit * split_o, (uint32_t)p.nsplit * split_o);
    constexpr uint32_t REC = F32P ? 8 : 16;  // bytes of a record
    const __amdgpu_buffer_rsrc_t rm = make_rsrc(p.part_ml + (int64_t)unit * p.nsplit * (kPRows * REC / 4),
                                                (uint32_t)p.nsplit * (kPRows * REC));
    const uint32_t lo = (uint32_t)wave * (NW * 1024) + 16 * lane;
    const uint32_t row_ml = REC * (wave * 32 + qc);
    auto load_rec = [&](int s) -> f4 {
      if constexpr (F32P) {
        const float2 r = load_agent_b64(rm, row_ml, s * (kPRows * REC));
        return f4{r.x, r.y, 1.0f, 0.0f};
      } else {
        return load_agent_b128(rm, row_ml, s * (kPRows * REC));
      }
    };
    f4 own[NW];
    float own_sc = 1.0f;
    if constexpr (F32P) {  // (the V operands were staged times 2^-E_V)
#pragma unroll
      for (int g = 0; g < NW; ++g)
#pragma unroll
        for (int i = 0; i < 4; ++i) own[g][i] = oacc[g >> 2][4 * (g & 3) + i] * vback;
    } else {
      const float inv_l = l_tot > 0.0f ? 1.0f / l_tot : 0.0f;
      float mx = 0.0f;
#pragma unroll
      for (int db = 0; db < NDB; ++db)
#pragma unroll
        for (int i = 0; i < 16; ++i) mx = fmaxf(mx, fabsf(oacc[db][i]));
      mx = max_xor32(mx) * inv_l;
      // mx * 2^-e lies in [2^13, 2^14): every row uses the full fp16 mantissa whatever its
      // magnitude (small rows would otherwise be stored as subnormals)
      int ex = 0;
      if (mx > 0.0f) frexpf(mx, &ex);
      const int e = mx > 0.0f ? min(max(ex - 14, -100), 100) : 0;
      own_sc = ldexpf(1.0f, e) * vback;  // the V operands were staged times 2^-E_V
      const float f = ldexpf(inv_l, -e);
#pragma unroll
      for (int u = 0; u < NW; ++u) {
        u4 x;
#pragma unroll
        for (int h = 0; h < 2; ++h) {
          const int g = 2 * u + h, db = g >> 2, c = g & 3;
          x[2 * h] = pack_f16x2(oacc[db][4 * c] * f, oacc[db][4 * c + 1] * f);
          x[2 * h + 1] = pack_f16x2(oacc[db][4 * c + 2] * f, oacc[db][4 * c + 3] * f);
        }
        own[u] = __builtin_bit_cast(f4, x);
      }
    }
#pragma unroll
    for (int u = 0; u < NW; ++u) store_agent_b128(ro, lo + u * 1024 + split * split_o, own[u]);
    if constexpr (F32P) {
      if (hh == 0) store_agent_b64(rm, row_ml + split * (kPRows * REC), make_float2(m_run, l_tot));
    } else {
      if (hh == 0) store_agent_b128(rm, row_ml + split * (kPRows * REC), f4{m_run, l_tot, own_sc, 0.0f});
    }
    if (!p.fused) return;
    // The stores are acknowledged (written through to the device's coherence point) before the
    // arrival is counted, so the last arrival sees every split's partials.
    __builtin_amdgcn_s_waitcnt(0);
    __syncthreads();
    if (tid == 0) *s_arrived = __hip_atomic_fetch_add(&p.counters[unit], 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    __syncthreads();
    if (*s_arrived != (unsigned)(nsplit - 1)) return;
    if (tid == 0) __hip_atomic_store(&p.counters[unit], 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);

    // M = max over the splits that saw a key; weights 2^(m_s - M)
    float M = l_tot > 0.0f ? m_run : -INFINITY;
    for (int s2 = 0; s2 < nsplit; ++s2) {
      if (s2 == split) continue;
      const f4 rec = load_rec(s2);
      if (rec[1] > 0.0f) M = fmaxf(M, rec[0]);
    }
    // the splits are summed in split order, each term one explicit fma
    f16v macc[NDB];
#pragma unroll
    for (int db = 0; db < NDB; ++db) macc[db] = f16v{};
    float l_acc = 0.0f;
    for (int s2 = 0; s2 < nsplit; ++s2) {
      f4 rec;
      f4 po[NW];
      if (s2 == split) {
        rec = f4{m_run, l_tot, own_sc, 0.0f};
#pragma unroll
        for (int u = 0; u < NW; ++u) po[u] = own[u];
      } else {
        rec = load_rec(s2);
#pragma unroll
        for (int u = 0; u < NW; ++u) po[u] = load_agent_b128(ro, lo + u * 1024, s2 * split_o);
      }
      const float w = (M == -INFINITY || rec[1] <= 0.0f) ? 0.0f : exp2_fast(rec[0] - M);
      l_acc = fmaf(w, rec[1], l_acc);
      const float F = F32P ? w : (w * rec[1]) * rec[2];
#pragma unroll
      for (int u = 0; u < NW; ++u) {
        if constexpr (F32P) {
#pragma unroll
          for (int k = 0; k < 4; ++k) macc[u >> 2][4 * (u & 3) + k] = fmaf(F, po[u][k], macc[u >> 2][4 * (u & 3) + k]);
        } else {
#pragma unroll
          for (int h = 0; h < 2; ++h) {
            const int g = 2 * u + h, db = g >> 2, c = g & 3;
            // halves are extracted with integer shifts: converting the elements of an h2 bit-cast
            // from a u4 element let the compiler (ROCm 7.2) fold all four words of a u4 into the
            // first one's register in v_fma_mix_f32
#pragma unroll
            for (int k = 0; k < 4; ++k) {
              const uint32_t w = __builtin_bit_cast(u4, po[u])[2 * h + (k >> 1)];
              const float x = (float)__builtin_bit_cast(_Float16, (uint16_t)((k & 1) ? w >> 16 : w & 0xffffu));
              macc[db][4 * c + k] = fmaf(F, x, macc[db][4 * c + k]);
            }
          }
        }
      }
    }
    l_tot = l_acc;
#pragma unroll
    for (int db = 0; db < NDB; ++db) oacc[db] = macc[db];
  }
  // ---- output. A lane holds 8-byte pieces of one row; stored directly, each store instruction
  // would write 8 bytes into each of 32 rows. Each wave instead stages its 32 rows in LDS (the
  // rings are free once every wave is past this barrier) and stores whole rows: 16 bytes a lane, so
  // an instruction writes 4 (D = 128) or 8 (D = 64) complete rows (D = 96: 5 1/3).
  // (after a split merge l_tot and oacc are in true units; else the V operands' 2^-ev returns here)
  const float inv = l_tot > 0.0f ? (1.0f / l_tot) * (nsplit > 1 ? 1.0f : vback) : 0.0f;
  constexpr int OP = D + 8;                 // fp16 per staged row: rows shift by 4 banks
  constexpr int WSB = 32 * OP * 2;          // staging bytes per wave
  constexpr int NRW = kRawSlots * RC::SLOT / WSB;           // waves staged in the raw ring
  constexpr int NVW = (DENSE ? 2 : 3) * D * kVS * 2 / WSB;  // ... and in the V^T ring
  static_assert(NRW + NVW >= kPW, "every wave's rows fit the raw and V^T rings");
  __syncthreads();
  uint16_t* const stage =
      (uint16_t*)(wave < NRW ? &raw[0][0] + wave * WSB : (uint8_t*)&v_lds[0][0] + (wave - NRW) * WSB);
#pragma unroll
  for (int db = 0; db < NDB; ++db)
#pragma unroll
    for (int c = 0; c < 4; ++c) {
      u2 w;
      w[0] = (uint32_t)from_float(oacc[db][4 * c] * inv, T{}) | ((uint32_t)from_float(oacc[db][4 * c + 1] * inv, T{}) << 16);
      w[1] = (uint32_t)from_float(oacc[db][4 * c + 2] * inv, T{}) | ((uint32_t)from_float(oacc[db][4 * c + 3] * inv, T{}) << 16);
      *(u2*)(stage + qc * OP + 32 * db + 8 * c + 4 * hh) = w;
    }
  // the output offset of this lane's row (lanes 0-31 own the wave's rows), read by the lanes that
  // store it
  const int64_t roff = (int64_t)b * p.o_sb + (int64_t)head * p.o_sh + (int64_t)lq * p.o_sl;
  const int roff_lo = (int)(uint32_t)roff, roff_hi = (int)(roff >> 32);
  __builtin_amdgcn_wave_barrier();  // the wave's LDS writes are issued before its reads (LDS keeps a wave's order)
  constexpr int CPR = D / 8;   // 16-byte chunks per row
#pragma unroll
  for (int it = 0; it < CPR / 2; ++it) {
    constexpr bool whole = 64 % CPR == 0;  // a store instruction covers whole rows
    const int r = whole ? it * (64 / CPR) + lane / CPR : (64 * it + lane) / CPR;
    const int cc = whole ? lane % CPR : (64 * it + lane) % CPR;
    const u4 v = *(const u4*)(stage + r * OP + 8 * cc);
    const int64_t ro = (int64_t)(((uint64_t)(uint32_t)__shfl(roff_hi, r) << 32) | (uint32_t)__shfl(roff_lo, r));
    if (fr0 + wave * 32 + r < p.nrows) {
      if (DENSE && D == 64 && p.out8) {  // rows that are only 8-byte aligned
        *(u2*)(p.out + ro + 8 * cc) = u2{v[0], v[1]};
        *(u2*)(p.out + ro + 8 * cc + 4) = u2{v[2], v[3]};
      } else {
        *(u4*)(p.out + ro + 8 * cc) = v;  // the host checks 16-byte aligned rows and strides
      }
    }
  }
}

// The split merge as a launch of its own, for row blocks cut into many splits: in the kernel above the
// last split loads the others one after another (about 0.9 us each at 128 dims). A workgroup takes one
// 16-byte word u of the packed rows of one wave (32 rows) of a row block; its 8 waves take the splits
// in turn, four in flight each, and wave 0 sums the eight partial merges. Row blocks that were not
// split have been written already. F32P: the partials are fp32 (kF32Partials), a word 4 values of a row rather than 8.
template <typename T, int D, bool F32P, bool MASKED = false>
__global__ __launch_bounds__(kPW * 64) void prefill_combine_kernel(PreParams p) {
  constexpr int QW = F32P ? D / 8 : D / 16;  // words per row
  constexpr int NV = F32P ? 4 : 8;           // values per word
  constexpr int NREC = F32P ? 2 : 4;         // floats per record
  constexpr int split_o = kPW * QW * 1024;
  __shared__ float s_m[kPW][64], s_l[kPW][64];
  __shared__ __align__(16) float s_o[kPW][64][NV];
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int u = blockIdx.x % QW, w = (blockIdx.x / QW) % kPW, unit = blockIdx.x / (QW * kPW);
  const int rb = unit % p.rowblocks, bk = unit / p.rowblocks;
  const int b = bk / p.Hkv, kvh = bk % p.Hkv;
  const int S_b = p.seq_lens ? min(max(load_uniform_i32(p.seq_lens, b), 0), p.S) : p.S;
  const int fr0 = rb * kPRows, frl = min(fr0 + kPRows, p.nrows) - 1;
  struct {
    int nsplit;
  } ks;
  if constexpr (MASKED) {
    ks.nsplit = split_masked(p, b, kvh, rb).nsplit;
  } else {
    ks.nsplit = split_keys(p, S_b, fr0, frl).nsplit;
  }
  if (ks.nsplit == 1 || fr0 + 32 * w >= p.nrows) return;
  const uint8_t* po = (const uint8_t*)p.part_o + (int64_t)unit * p.nsplit * split_o + (w * QW + u) * 1024 + 16 * lane;
  const float* rec = p.part_ml + (int64_t)unit * p.nsplit * (kPRows * NREC) + (32 * w + (lane & 31)) * NREC;
  constexpr int CH = 4;
  float M = -INFINITY, l = 0.0f, acc[NV] = {};
  for (int s0 = wave; s0 < ks.nsplit; s0 += kPW * CH) {
    f4 r[CH];
    u4 v[CH];
#pragma unroll
    for (int i = 0; i < CH; ++i) {
      const int s = min(s0 + kPW * i, ks.nsplit - 1);  // past the last split it is re-read, and not counted
      if constexpr (F32P) {
        const float2 x = *(const float2*)(rec + s * (kPRows * NREC));
        r[i] = f4{x.x, x.y, 1.0f, 0.0f};
      } else {
        r[i] = *(const f4*)(rec + s * (kPRows * NREC));
      }
      v[i] = *(const u4*)(po + (int64_t)s * split_o);
    }
    float Mn = M;
#pragma unroll
    for (int i = 0; i < CH; ++i)
      if (s0 + kPW * i < ks.nsplit && r[i][1] > 0.0f) Mn = fmaxf(Mn, r[i][0]);
    const float corr = M == Mn ? 1.0f : exp2_fast(M - Mn);
    l *= corr;
#pragma unroll
    for (int e = 0; e < NV; ++e) acc[e] *= corr;
    M = Mn;
#pragma unroll
    for (int i = 0; i < CH; ++i) {
      if (s0 + kPW * i >= ks.nsplit) continue;
      // a row that saw no key in the split counts 0, but for NaN (a poisoned row block)
      const float ws = r[i][1] > 0.0f ? exp2_fast(r[i][0] - M) : 0.0f;
      l += ws * r[i][1];
      const float F = F32P ? ws : (ws * r[i][1]) * r[i][2];
#pragma unroll
      for (int e = 0; e < NV; ++e) {
        const uint32_t x = v[i][F32P ? e : e >> 1];
        acc[e] = fmaf(F, F32P ? __uint_as_float(x)
                              : (float)__builtin_bit_cast(_Float16, (uint16_t)((e & 1) ? x >> 16 : x & 0xffffu)), acc[e]);
      }
    }
  }
  s_m[wave][lane] = M;
  s_l[wave][lane] = l;
#pragma unroll
  for (int e = 0; e < NV; e += 4) *(f4*)&s_o[wave][lane][e] = f4{acc[e], acc[e + 1], acc[e + 2], acc[e + 3]};
  __syncthreads();
  const int row = fr0 + 32 * w + (lane & 31);
  if (wave != 0 || row >= p.nrows) return;
  M = -INFINITY;
#pragma unroll
  for (int k = 0; k < kPW; ++k) M = fmaxf(M, s_m[k][lane]);
  l = 0.0f;
  f4 o[NV / 4] = {};
#pragma unroll
  for (int k = 0; k < kPW; ++k) {
    const float f = s_m[k][lane] == -INFINITY ? (M == -INFINITY ? 1.0f : 0.0f) : exp2_fast(s_m[k][lane] - M);
    l += f * s_l[k][lane];
#pragma unroll
    for (int h = 0; h < NV / 4; ++h) o[h] += f * *(const f4*)&s_o[k][lane][4 * h];
  }
  const float inv = l > 0.0f ? 1.0f / l : 0.0f;
  // word u holds value groups NV / 4 u ..; group 4 db + c holds dims 32 db + 8 c + 4 hh .. + 3
  uint16_t* dst = p.out + (int64_t)b * p.o_sb + (int64_t)(kvh * p.rep + row % p.rep) * p.o_sh +
                  (int64_t)(row / p.rep) * p.o_sl + 4 * (lane >> 5);
#pragma unroll
  for (int h = 0; h < NV / 4; ++h) {
    const int g = NV / 4 * u + h;
    u2 x;
    x[0] = (uint32_t)from_float(o[h][0] * inv, T{}) | ((uint32_t)from_float(o[h][1] * inv, T{}) << 16);
    x[1] = (uint32_t)from_float(o[h][2] * inv, T{}) | ((uint32_t)from_float(o[h][3] * inv, T{}) << 16);
    *(u2*)(dst + 32 * (g >> 2) + 8 * (g & 3)) = x;
  }
}

// prefill_masked.hip: the MASKED launches and the kernel that classes the mask's tiles.
hipError_t launch_prefill_masked_t(const PreParams& p, int B, int dtype, int D, int bits, int G, hipStream_t stream);

}  // namespace kvq
