// Host side of the decode kernel (decode_kernel.h): plan, workspace, launch.

#include <stdlib.h>

#include <algorithm>

#include "decode_kernel.h"

namespace kvq {

struct DecPlan {
  int R, rowblocks, chunk, nsplit, span, nunits, nw, nslot, fused;
};

struct DecTune {
  int nw, nslot, target_wgs, fused;
};

// The in-kernel split merge (the last split of a unit merges) costs an arrival counter and a
// round trip per split partial in one workgroup; the combine launch costs a kernel boundary. With
// few splits the in-kernel merge is faster (3-4 splits: C5 window layer 12.5 against 13.3 us, C2 at
// batch 8 and C5's global layer about 1% faster), with many it is slower (17 splits: C1 12.6 against
// 11.4 us; 32: C2 at batch 1 24.2 against 21.7 us).
constexpr int kFusedMaxSplit = kFewSplits;

// Launch-shape defaults; KVQ_DECODE_TUNE="waves,slots,workgroups[,fused]" overrides them (read
// once per process; fused 0 or 1 forces the split merge's form, omitted leaves it to the plan).
// 8-wave workgroups take 2 ring slots (the ring of 3 would not fit in LDS).
static DecTune decode_tune() {
  static DecTune t = [] {
    DecTune d{4, 2, 256, -1};
    if (const char* e = getenv("KVQ_DECODE_TUNE")) {
      int a = 0, b = 0, c = 0, f = -1;
      if (sscanf(e, "%d,%d,%d,%d", &a, &b, &c, &f) >= 3 && (a == 4 || (a == 8 && b == 2)) && b >= 2 && b <= 4 && c >= 1)
        d = {a, b, c, f < 0 ? -1 : f != 0};
    }
    return d;
  }();
  return t;
}

DecPlan decode_plan(int B, int Hq, int Hkv, int L, int D, int S, int window, int bits, int G) {
  DecPlan pl;
  const DecTune tune = decode_tune();
  const bool dense = bits == 16;
  if (dense) G = 64;  // the unquantized kernels keep the column layout of group 64
  const bool tuned = D == 128 && !dense && G == 64;  // the launch shapes built for other than 4 waves x 2 slots
  pl.nw = tuned ? tune.nw : 4;
  pl.nslot = tuned ? tune.nslot : 2;
  pl.R = 16 / (D / G);
  const int nrows = (Hq / Hkv) * L;
  pl.rowblocks = (nrows + pl.R - 1) / pl.R;
  pl.span = window > 0 ? std::min(S, window + L - 1 + kTile - 1) : S;  // the window, from a tile boundary
  const int tiles_seq = (pl.span + kTile - 1) / kTile;
  pl.nunits = B * Hkv * pl.rowblocks;
  // as many splits as the target holds whole: a unit count that does not divide 256 would otherwise leave a
  // few workgroups to run after the others. With the count rounded up instead, 32768 8-bit keys of 24, 40
  // and 72 units took 53.0, 88.7 and 151.9 us; so 41.6, 64.3 and 111.8. Past 128 units none is split: 144 and
  // 240 took 306 and 463 us, so 245 and 371 (5000 keys: 54.7 and 79.2, so 41.6 and 60.5). Where it costs the workgroups no
  // length (or little, and row blocks share keys) the count also makes the grid a multiple of the XCDs,
  // which keeps a unit's splits, and the row blocks of a key range, on one
  auto tiles_of = [&](int n) {
    const int t = (tiles_seq + n - 1) / n;
    return std::max(pl.nw, (t + pl.nw - 1) / pl.nw * pl.nw);
  };
  const int ns = std::max(1, std::min<int>(tune.target_wgs / pl.nunits, kMaxSplit));
  const int whole = std::max(1, kXcds / (pl.nunits & -pl.nunits));  // (kXcds is a power of two)
  int tpw = tiles_of(ns);
  if (ns > whole && 8 * tiles_of(ns - ns % whole) <= (pl.rowblocks > 1 ? 9 : 8) * tpw) tpw = tiles_of(ns - ns % whole);
  pl.chunk = tpw * kTile;
  pl.nsplit = (pl.span + pl.chunk - 1) / pl.chunk;
  const bool fused = tune.fused < 0 ? pl.nsplit <= kFusedMaxSplit : tune.fused != 0;
  // (with 16 query rows of 128 dims a thread owns two float4s of a partial; the in-kernel merge
  // then handles at most kFewSplits splits)
  const bool few_only = pl.R * D / 4 > 4 * 64;
  pl.fused = fused && pl.nunits <= kMaxCountedUnits && (!few_only || pl.nsplit <= kFewSplits);
  return pl;
}

// Workspace: [split counters (the shared block), zero between calls][(m, l) per row and split]
// [o per row and split]
struct DecLayout {
  size_t counters, ml, o, total;
};
static DecLayout decode_layout(const DecPlan& pl, int D) {
  auto up = [](size_t x) { return (x + 255) / 256 * 256; };
  DecLayout l;
  const size_t prow = (size_t)pl.nunits * pl.R * pl.nsplit;
  l.counters = 0;
  l.ml = kCounterBytes;
  l.o = l.ml + up(prow * sizeof(float2));
  l.total = l.o + up(prow * D * sizeof(float));
  return l;
}

int decode_kernel_dim(int D) { return D <= 64 ? 64 : D <= 128 ? 128 : 256; }

size_t decode_workspace_bytes(int B, int Hq, int Hkv, int L, int D, int S, int window, int bits, int G) {
  const int Dk = decode_kernel_dim(D);
  const DecPlan pl = decode_plan(B, Hq, Hkv, L, Dk, S, window, bits, G);
  return decode_layout(pl, Dk).total;
}

// Whether kernel width D with scale group G serves narrower rows: head dims that run at width D
// (decode_kernel_dim) and are multiples of G, i.e. 32 dims at width 64 (G 32), 96 at 128 (G 32) and
// 192 at 256 (G 64); unquantized rows (G stands at 64) of any multiple of 8 at width 64 or 128.
template <int D, int BITS, int G>
constexpr bool narrow_rows() {
  if constexpr (BITS == 16) return D <= 128;
  const int lo = D == 64 ? 0 : D / 2;  // the widths below D end here
  return (lo / G + 1) * G < D;
}

template <typename T, int D, int BITS, int NW, int NSLOT, bool PAGED = false, int G = 64>
static hipError_t launch_decode_t(const DecParams& p, hipStream_t stream) {
  if (p.dv != D) {
    // rows narrower than the kernel (decode_kernel_dim): the default launch shape, plain, paged or
    // masked
    if constexpr (NW == 4 && NSLOT == 2 && narrow_rows<D, BITS, G>()) {
      if (p.mask_kind != 0) {
        if constexpr (!PAGED) {
          hipLaunchKernelGGL((decode_attn_kernel<T, D, BITS, NW, NSLOT, PAGED, G, true, true>),
                             dim3(p.nunits * p.nsplit), dim3(NW * 64), 0, stream, p);
        } else {
          return hipErrorInvalidValue;
        }
      } else {
        hipLaunchKernelGGL((decode_attn_kernel<T, D, BITS, NW, NSLOT, PAGED, G, false, true>), dim3(p.nunits * p.nsplit),
                           dim3(NW * 64), 0, stream, p);
      }
    } else {
      return hipErrorInvalidValue;
    }
  } else if (p.mask_kind != 0) {
    if constexpr (NW == 4 && NSLOT == 2 && !PAGED) {
      hipLaunchKernelGGL((decode_attn_kernel<T, D, BITS, NW, NSLOT, PAGED, G, true>), dim3(p.nunits * p.nsplit),
                         dim3(NW * 64), 0, stream, p);
    } else {
      return hipErrorInvalidValue;  // masked calls always take the default launch shape
    }
  } else {
    hipLaunchKernelGGL((decode_attn_kernel<T, D, BITS, NW, NSLOT, PAGED, G>), dim3(p.nunits * p.nsplit), dim3(NW * 64),
                       0, stream, p);
  }
  hipError_t e = hipGetLastError();
  if (e != hipSuccess || p.nsplit == 1 || p.fused) return e;
  return launch_combine<T, D>(merge_params(p, DecCfg<D, BITS, G>::R), p.nunits / (p.Hkv * p.rowblocks), stream,
                              p.dv);
}

template <typename T, int D, int BITS, int G = 64>
static hipError_t launch_decode_shape(const DecParams& p, const DecPlan& pl, hipStream_t stream) {
  if (p.mask_kind != 0 || p.dv != D) return launch_decode_t<T, D, BITS, 4, 2, false, G>(p, stream);
  if constexpr (BITS == 16) {
    return launch_decode_t<T, D, BITS, 4, 2>(p, stream);  // a 3-slot ring of raw rows does not fit
  } else if constexpr (G != 64) {
    return launch_decode_t<T, D, BITS, 4, 2, false, G>(p, stream);
  } else if constexpr (D == 128) {
    if (pl.nw == 8) return launch_decode_t<T, D, BITS, 8, 2>(p, stream);
    if (pl.nslot == 2) return launch_decode_t<T, D, BITS, 4, 2>(p, stream);
    if (pl.nslot == 3) return launch_decode_t<T, D, BITS, 4, 3>(p, stream);
    return launch_decode_t<T, D, BITS, 4, 4>(p, stream);
  } else {
    return launch_decode_t<T, D, BITS, 4, 2>(p, stream);
  }
}

// Everything but the K/V operands.
static DecParams decode_params(const kvq_rows* q, const int32_t* seq_lens, const kvq_rows* out, int Hq, int Hkv,
                               int L, int D, int S, float scale, int causal, int window, void* workspace,
                               const DecPlan& pl) {
  const DecLayout lay = decode_layout(pl, D);
  DecParams p{};
  p.q = (const uint16_t*)q->data;
  p.q_sb = q->stride_b;
  p.q_sh = q->stride_h;
  p.q_sl = q->stride_l;
  p.seq_lens = seq_lens;
  p.out = (uint16_t*)out->data;
  p.o_sb = out->stride_b;
  p.o_sh = out->stride_h;
  p.o_sl = out->stride_l;
  p.counters = (unsigned*)((char*)workspace + lay.counters);
  p.part_ml = (float*)((char*)workspace + lay.ml);
  p.part_o = (float*)((char*)workspace + lay.o);
  p.Hq = Hq;
  p.Hkv = Hkv;
  p.L = L;
  p.S = S;
  p.rep = Hq / Hkv;
  p.nrows = p.rep * L;
  p.rowblocks = pl.rowblocks;
  p.nsplit = pl.nsplit;
  p.chunk = pl.chunk;
  p.nunits = pl.nunits;
  p.xcd_remap = ((int64_t)pl.nunits * pl.nsplit) % kXcds == 0;
  p.fused = pl.fused;
  p.scale_log2 = scale * 1.4426950408889634f;
  p.causal = causal;
  p.window = window;
  p.dv = D;
  p.d_nsplit = make_div31((uint32_t)pl.nsplit);
  p.d_rowblocks = make_div31((uint32_t)pl.rowblocks);
  p.d_hkv = make_div31((uint32_t)Hkv);
  p.d_l = make_div31((uint32_t)L);
  return p;
}

// Calls past one decode pass's rows (two for the groups whose passes are shorter than 8) take the MULTI
// kernels: they are the ones that prefill kernels serve where the rows are more or the keys many.
static bool multi_rows(int nrows, int R) { return nrows > std::max(R, 8); }

static void set_mask(DecParams& p, const kvq_mask* mask) {
  if (!mask) return;
  p.mask = mask->data;
  p.mask_kind = mask->kind;
  p.m_sb = mask->stride_b;
  p.m_skv = mask->stride_kvh;
  p.m_srep = mask->stride_rep;
  p.m_sl = mask->stride_l;
}

hipError_t launch_decode(const kvq_rows* q, const kvq_qtensor* k, const kvq_qtensor* v, const int32_t* seq_lens,
                         const kvq_rows* out, int B, int Hq, int Hkv, int L, int D, int S, int bits, int G, int dtype,
                         float scale, int causal, int window, void* workspace, hipStream_t stream, const kvq_mask* mask) {
  const int Dk = decode_kernel_dim(D);
  const DecPlan pl = decode_plan(B, Hq, Hkv, L, Dk, S, window, bits, G);
  DecParams p = decode_params(q, seq_lens, out, Hq, Hkv, L, Dk, S, scale, causal, window, workspace, pl);
  p.dv = D;
  set_mask(p, mask);
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
  if (!mask && D == Dk && multi_rows(p.nrows, pl.R)) return launch_decode_multi(p, dtype, Dk, bits, G, false, stream);
  return dispatch_quant(dtype, Dk, bits, G, [&](auto t, auto d, auto b, auto g) {
    return launch_decode_shape<decltype(t), decltype(d)::value, decltype(b)::value, decltype(g)::value>(p, pl, stream);
  });
}

hipError_t launch_decode_paged(const kvq_rows* q, const kvq_qtensor* k, const kvq_qtensor* v, int num_pages,
                               const int32_t* table, int64_t table_stride, const int32_t* seq_lens, const kvq_rows* out,
                               int B, int Hq, int Hkv, int L, int D, int S, int bits, int G, int dtype, float scale,
                               int causal, int window, void* workspace, hipStream_t stream) {
  const int Dk = decode_kernel_dim(D);
  const DecPlan pl = decode_plan(B, Hq, Hkv, L, Dk, S, window, bits, G);
  DecParams p = decode_params(q, seq_lens, out, Hq, Hkv, L, Dk, S, scale, causal, window, workspace, pl);
  p.dv = D;
  p.kc = (const uint8_t*)k->codes;
  p.vc = (const uint8_t*)v->codes;
  p.kc_sb = k->codes_stride_b * 4;  // page strides
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
  p.table = table;
  p.table_stride = table_stride;
  p.num_pages = num_pages;
  if (D == Dk && multi_rows(p.nrows, pl.R)) return launch_decode_multi(p, dtype, Dk, bits, G, true, stream);
  return dispatch_quant(dtype, Dk, bits, G, [&](auto t, auto d, auto b, auto g) {
    return launch_decode_t<decltype(t), decltype(d)::value, decltype(b)::value, 4, 2, true, decltype(g)::value>(p, stream);
  });
}

hipError_t launch_decode_dense(const kvq_rows* q, const kvq_rows* k, const kvq_rows* v, const int32_t* seq_lens,
                               const kvq_rows* out, int B, int Hq, int Hkv, int L, int D, int S, int dtype, float scale,
                               int causal, int window, void* workspace, hipStream_t stream, const kvq_mask* mask) {
  const int Dk = decode_kernel_dim(D);
  const DecPlan pl = decode_plan(B, Hq, Hkv, L, Dk, S, window, 16, 64);
  DecParams p = decode_params(q, seq_lens, out, Hq, Hkv, L, Dk, S, scale, causal, window, workspace, pl);
  p.dv = D;
  set_mask(p, mask);
  p.kc = (const uint8_t*)k->data;
  p.vc = (const uint8_t*)v->data;
  p.kc_sb = k->stride_b * 2;
  p.kc_sh = k->stride_h * 2;
  p.kc_ss = k->stride_l * 2;
  p.vc_sb = v->stride_b * 2;
  p.vc_sh = v->stride_h * 2;
  p.vc_ss = v->stride_l * 2;
  const bool bf = dtype == KVQ_DTYPE_BF16;
  if (Dk == 256) return hipErrorInvalidValue;  // unquantized rows past 128 dims run through the head_dim-256 kernel
  if (Dk == 128) return bf ? launch_decode_shape<BF16, 128, 16>(p, pl, stream) : launch_decode_shape<F16, 128, 16>(p, pl, stream);
  return bf ? launch_decode_shape<BF16, 64, 16>(p, pl, stream) : launch_decode_shape<F16, 64, 16>(p, pl, stream);
}

}  // namespace kvq
