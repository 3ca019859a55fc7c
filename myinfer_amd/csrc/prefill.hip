// Host side of the prefill kernel (prefill_kernel.h): plan, workspace, launch.

#include <algorithm>

#include "prefill_kernel.h"

namespace kvq {

size_t prefill_workspace_bytes(int B, int Hq, int Hkv, int L, int D, int S, int window) {
  size_t n = 256;
  for (int causal : {0, 1}) {
    const PrePlan pl = prefill_plan(B, Hq, Hkv, L, S, window, causal);
    // (the size serves quantized and unquantized calls: at 64 dims the latter's partials are fp32, the larger)
    if (pl.nsplit > 1) n = std::max(n, prefill_layout(pl, D, D != 128).total);
  }
  return n;
}

template <typename T, int BITS, bool PAGED = false, int G = 64, int D = 128>
static hipError_t launch_prefill_t(const PreParams& p, hipStream_t stream) {
  hipLaunchKernelGGL((prefill_attn_kernel<T, BITS, PAGED, G, D>), dim3(prefill_grid(p)), dim3(kPW * 64), 0, stream,
                     p);
  hipError_t e = hipGetLastError();
  if (e != hipSuccess || p.nsplit == 1 || p.fused) return e;
  constexpr bool f32 = kF32Partials<BITS, D, 0>;
  hipLaunchKernelGGL((prefill_combine_kernel<T, D, f32>), dim3(p.nunits * kPW * (D / (f32 ? 8 : 16))), dim3(kPW * 64), 0,
                     stream, p);
  return hipGetLastError();
}

// The quantized instantiation for (dtype, D in {64, 128}, bits in {4, 8}, G in {32, 64, 128}, G <= D) or
// (dtype, D = 96, bits, G = 32).
template <bool PAGED>
static hipError_t launch_prefill_quant(const PreParams& p, int dtype, int D, int bits, int G, hipStream_t stream) {
  auto by_g = [&](auto t, auto d, auto b) -> hipError_t {
    using TT = decltype(t);
    constexpr int DD = decltype(d)::value;
    constexpr int BB = decltype(b)::value;
    if (G == 32) return launch_prefill_t<TT, BB, PAGED, 32, DD>(p, stream);
    if constexpr (DD == 96) {
      return hipErrorInvalidValue;
    } else {
      if constexpr (DD >= 128) {
        if (G == 128) return launch_prefill_t<TT, BB, PAGED, 128, DD>(p, stream);
      }
      return launch_prefill_t<TT, BB, PAGED, 64, DD>(p, stream);
    }
  };
  auto by_d = [&](auto t, auto b) -> hipError_t {
    if (D == 96) return by_g(t, std::integral_constant<int, 96>{}, b);
    return D == 64 ? by_g(t, std::integral_constant<int, 64>{}, b) : by_g(t, std::integral_constant<int, 128>{}, b);
  };
  auto by_b = [&](auto t) -> hipError_t {
    return bits == 8 ? by_d(t, std::integral_constant<int, 8>{}) : by_d(t, std::integral_constant<int, 4>{});
  };
  return dtype == KVQ_DTYPE_BF16 ? by_b(BF16{}) : by_b(F16{});
}

// Everything but the K/V operands.
static PreParams prefill_params(const kvq_rows* q, const int32_t* seq_lens, const kvq_rows* out, int Hq, int Hkv, int L, int D,
                                int S, float scale, int causal, int window, void* workspace, const PrePlan& pl,
                                bool f32_partials) {
  PreParams p{};
  p.q = (const uint16_t*)q->data;
  p.q_sb = q->stride_b;
  p.q_sh = q->stride_h;
  p.q_sl = q->stride_l;
  p.seq_lens = seq_lens;
  p.out = (uint16_t*)out->data;
  p.o_sb = out->stride_b;
  p.o_sh = out->stride_h;
  p.o_sl = out->stride_l;
  const PreLayout lay = prefill_layout(pl, D, f32_partials);
  p.counters = (unsigned*)workspace;
  p.part_o = (float*)((char*)workspace + lay.o);
  p.part_ml = (float*)((char*)workspace + lay.ml);
  p.Hq = Hq;
  p.Hkv = Hkv;
  p.L = L;
  p.S = S;
  p.rep = Hq / Hkv;
  p.nrows = p.rep * L;
  p.rowblocks = pl.rowblocks;
  p.nsplit = pl.nsplit;
  p.chunk = pl.chunk;
  p.order = pl.order;
  p.nbk = pl.nbk;
  p.lo = pl.lo;
  p.fused = pl.nsplit <= kPFusedMaxSplit;
  p.nunits = pl.nunits;
  p.scale_log2 = scale * 1.4426950408889634f;
  p.causal = causal;
  p.window = window;
  return p;
}

static void quant_operands(PreParams& p, const kvq_qtensor* k, const kvq_qtensor* v) {
  p.kc = (const uint8_t*)k->codes;
  p.vc = (const uint8_t*)v->codes;
  p.kc_sb = k->codes_stride_b * 4;
  p.kc_sh = k->codes_stride_h * 4;
  p.kc_ss = k->codes_stride_s * 4;
  p.vc_sb = v->codes_stride_b * 4;
  p.vc_sh = v->codes_stride_h * 4;
  p.vc_ss = v->codes_stride_s * 4;
  p.ks = (const uint16_t*)k->scales;
  p.kb = (const uint16_t*)k->biases;
  p.vs = (const uint16_t*)v->scales;
  p.vb = (const uint16_t*)v->biases;
  p.ksb_sb = k->sb_stride_b;
  p.ksb_sh = k->sb_stride_h;
  p.ksb_ss = k->sb_stride_s;
  p.vsb_sb = v->sb_stride_b;
  p.vsb_sh = v->sb_stride_h;
  p.vsb_ss = v->sb_stride_s;
  p.k_rexp = k->range_exp;
  p.v_rexp = v->range_exp;
}

static void dense_operands(PreParams& p, const kvq_rows* k, const kvq_rows* v) {
  p.kc = (const uint8_t*)k->data;
  p.vc = (const uint8_t*)v->data;
  p.kc_sb = k->stride_b * 2;
  p.kc_sh = k->stride_h * 2;
  p.kc_ss = k->stride_l * 2;
  p.vc_sb = v->stride_b * 2;
  p.vc_sh = v->stride_h * 2;
  p.vc_ss = v->stride_l * 2;
}

hipError_t launch_prefill(const kvq_rows* q, const kvq_qtensor* k, const kvq_qtensor* v, const int32_t* seq_lens,
                          const kvq_rows* out, int B, int Hq, int Hkv, int L, int D, int S, int bits, int G, int dtype,
                          float scale, int causal, int window, void* workspace, hipStream_t stream) {
  const PrePlan pl = prefill_plan(B, Hq, Hkv, L, S, window, causal);
  PreParams p = prefill_params(q, seq_lens, out, Hq, Hkv, L, D, S, scale, causal, window, workspace, pl,
                               D == 96);
  quant_operands(p, k, v);
  return launch_prefill_quant<false>(p, dtype, D, bits, G, stream);
}

hipError_t launch_prefill_paged(const kvq_rows* q, const kvq_qtensor* k, const kvq_qtensor* v, int num_pages,
                                const int32_t* table, int64_t table_stride, const int32_t* seq_lens, const kvq_rows* out,
                                int B, int Hq, int Hkv, int L, int D, int S, int bits, int G, int dtype, float scale,
                                int causal, int window, void* workspace, hipStream_t stream) {
  const PrePlan pl = prefill_plan(B, Hq, Hkv, L, S, window, causal);
  PreParams p = prefill_params(q, seq_lens, out, Hq, Hkv, L, D, S, scale, causal, window, workspace, pl,
                               D == 96);
  quant_operands(p, k, v);  // (batch strides are page strides)
  p.table = table;
  p.table_stride = table_stride;
  p.num_pages = num_pages;
  return launch_prefill_quant<true>(p, dtype, D, bits, G, stream);
}

hipError_t launch_prefill_dense(const kvq_rows* q, const kvq_rows* k, const kvq_rows* v, const int32_t* seq_lens,
                                const kvq_rows* out, int B, int Hq, int Hkv, int L, int D, int S, int dtype,
                                float scale, int causal, int window, void* workspace, hipStream_t stream) {
  const PrePlan pl = prefill_plan(B, Hq, Hkv, L, S, window, causal);
  PreParams p = prefill_params(q, seq_lens, out, Hq, Hkv, L, D, S, scale, causal, window, workspace, pl, D == 64);
  dense_operands(p, k, v);
  p.out8 = ((uintptr_t)out->data % 16 || (out->stride_b | out->stride_h | out->stride_l) % 8) ? 1 : 0;
  const bool bf = dtype == KVQ_DTYPE_BF16;
  if (D == 64)
    return bf ? launch_prefill_t<BF16, 16, false, 64, 64>(p, stream) : launch_prefill_t<F16, 16, false, 64, 64>(p, stream);
  return bf ? launch_prefill_t<BF16, 16>(p, stream) : launch_prefill_t<F16, 16>(p, stream);
}

// ---- general masks (prefill_masked.hip)

// The plan of a masked call within `bytes` of workspace: [arrival counters][the splits' partials, if any]
// [tile bitmaps]. False when the bitmaps alone do not fit.
struct MaskedPlan {
  PrePlan pl;
  size_t words;  // offset of the bitmaps
  int nwords;
};
static bool plan_masked(int B, int Hq, int Hkv, int L, int D, int S, const kvq_mask* mask, size_t bytes, MaskedPlan* m) {
  PrePlan pl = prefill_plan(B, Hq, Hkv, L, S, 0, 0);
  pl.order = kMasked;  // most masks are causal and then some: the row blocks of the last positions first
  m->nwords = ((S + kPT - 1) / kPT + 63) / 64;
  const size_t need = (size_t)B * (mask->stride_kvh ? Hkv : 1) * pl.rowblocks * m->nwords * 16;
  for (;; set_splits(&pl, pl.nsplit - 1)) {
    m->words = pl.nsplit > 1 ? (prefill_layout(pl, D, true).total + 255) / 256 * 256 : kCounterBytes;
    if (m->words + need <= bytes) break;
    if (pl.nsplit == 1) return false;
  }
  m->pl = pl;
  return true;
}

// A masked decode call's time grows with its passes over all keys, visible or not: about 60 us per 10^6
// passes x units x keys. This kernel's calls start at 20 us (classes, tiles, a merge) and skip what no
// row sees. Left-padded prompts, decode against prefill in us: 2 x 4 KV heads of 8 query heads, 128
// tokens (262 000) 15 / 20, 256 (524 000) 37 / 24; 4 x 8 KV heads of 4, 64 rows over 600 keys (614 000)
// 32 / 33, 1000 tokens 536 / 63; 16 KV heads of 64 dims, 256 tokens (262 000) 18 / 23, 500 (10^6) 41 / 21.
bool prefill_masked_rows(int B, int Hq, int Hkv, int L, int D, int S) {
  if (D != 64 && D != 96 && D != 128) return false;
  const int64_t rows = (int64_t)(Hq / Hkv) * L;
  const int per = D == 96 ? 4 : 1024 / D;  // rows of a decode pass at the usual groups
  return rows >= 128 && (rows + per - 1) / per * B * Hkv * S >= 400000;
}

size_t prefill_masked_bytes(int B, int Hq, int Hkv, int L, int D, int S) {
  if (!prefill_masked_rows(B, Hq, Hkv, L, D, S)) return 0;
  const PrePlan pl = prefill_plan(B, Hq, Hkv, L, S, 0, 0);
  const size_t words = (size_t)B * Hkv * pl.rowblocks * (((S + kPT - 1) / kPT + 63) / 64) * 16;
  return (pl.nsplit > 1 ? (prefill_layout(pl, D, true).total + 255) / 256 * 256 : kCounterBytes) + words;
}

bool prefill_masked_fits(int B, int Hq, int Hkv, int L, int D, int S, const kvq_mask* mask, size_t bytes) {
  MaskedPlan m;
  return plan_masked(B, Hq, Hkv, L, D, S, mask, bytes, &m);
}

hipError_t launch_prefill_masked(const kvq_rows* q, const kvq_qtensor* k, const kvq_qtensor* v, const kvq_rows* kd,
                                 const kvq_rows* vd, const kvq_rows* out, int B, int Hq, int Hkv, int L, int D, int S,
                                 int bits, int G, int dtype, float scale, const kvq_mask* mask, void* workspace,
                                 size_t workspace_bytes, hipStream_t stream) {
  MaskedPlan m;
  if (!plan_masked(B, Hq, Hkv, L, D, S, mask, workspace_bytes, &m)) return hipErrorInvalidValue;
  PreParams p = prefill_params(q, nullptr, out, Hq, Hkv, L, D, S, scale, 0, 0, workspace, m.pl, true);
  if (bits == 16) {
    dense_operands(p, kd, vd);
  } else {
    quant_operands(p, k, v);
  }
  p.out8 = ((uintptr_t)out->data % 16 || (out->stride_b | out->stride_h | out->stride_l) % 8) ? 1 : 0;
  p.mask = mask->data;
  p.mask_kind = mask->kind;
  p.m_sb = mask->stride_b;
  p.m_skv = mask->stride_kvh;
  p.m_srep = mask->stride_rep;
  p.m_sl = mask->stride_l;
  p.words = (const uint64_t*)((const char*)workspace + m.words);
  p.nwords = m.nwords;
  p.w_kv = mask->stride_kvh != 0;
  return launch_prefill_masked_t(p, B, dtype, D, bits, G, stream);
}

}  // namespace kvq
