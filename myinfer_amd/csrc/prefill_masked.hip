// The prefill kernel under a general mask (boolean masks with no causal / window / right-padding
// structure -- left-padded batches above all --, per-head masks and additive masks;
// m5engine/attention.py:55-56, :76-80). Such calls ran on the decode kernel, 8 rows a pass over all keys:
// 42 TFLOP/s of visible pairs for four left-padded 1023-token prompts.
//
// A first launch classes the mask per row block of 256 query rows and tile of 64 keys: no key visible to
// any row (the tile is skipped: a causal prompt's upper half, the padding), all keys visible to all
// rows (computed without reading the mask again), or mixed (the mask is read beside the tile). It reads
// the mask once per row block that shares it, 64 bytes a row and wave.

#include <type_traits>

#include "prefill_kernel.h"

namespace kvq {

// 16 waves, one tile each; the workgroups of a row block cover 64 nwords tiles, so that every bit of the
// bitmaps is written.
constexpr int kClassWaves = 16;
template <int EL>  // bytes of a mask element
__global__ __launch_bounds__(kClassWaves * 64) void mask_classes_kernel(PreParams p, uint16_t* words, int nkv) {
  __shared__ unsigned s_any, s_mixed;
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int groups = 4 * p.nwords;  // 16-tile groups of a row block
  const int g = blockIdx.x % groups, u = blockIdx.x / groups;
  const int rb = u % p.rowblocks, bkv = u / p.rowblocks;
  const int b = bkv / nkv, kvh = bkv % nkv;
  if (threadIdx.x == 0) s_any = s_mixed = 0;
  __syncthreads();
  const int fr0 = rb * kPRows, frl = min(fr0 + kPRows, p.nrows) - 1;
  bool any = false, all = true;
  // the block's distinct mask rows: positions, or (position, head) pairs when the heads' masks differ
  const bool heads = p.m_srep != 0;
  const int i0 = heads ? fr0 : fr0 / p.rep, i1 = heads ? frl : frl / p.rep;
  auto row_at = [&](int r) -> int64_t {
    return heads ? (int64_t)(r / p.rep) * p.m_sl + (int64_t)(r % p.rep) * p.m_srep : (int64_t)r * p.m_sl;
  };
  const uint8_t* base = (const uint8_t*)p.mask + EL * ((int64_t)b * p.m_sb + (int64_t)kvh * p.m_skv);
  const int k0 = (g * kClassWaves + wave) * kPT;
  bool in;  // the lane's keys exist
  if constexpr (EL == 1) {
    // a row's 64 bytes by 16 lanes, 4 rows at a time (rows start at any byte)
    constexpr int CH = 16;
    const int key = k0 + 4 * (lane & 15), sub = lane >> 4;
    in = key + 4 <= p.S;
    if (k0 < p.S) {
      for (int i = i0; i <= i1; i += 4 * CH) {
        uint32_t x[CH];
#pragma unroll
        for (int c = 0; c < CH; ++c) {
          const uint8_t* q = base + row_at(min(i + 4 * c + sub, i1)) + key;
          if (in) {
            __builtin_memcpy(&x[c], q, 4);
          } else {  // past the row's end counts as hidden
            x[c] = 0;
#pragma unroll
            for (int e = 0; e < 4; ++e)
              if (key + e < p.S) x[c] |= (uint32_t)q[e] << (8 * e);
          }
        }
#pragma unroll
        for (int c = 0; c < CH; ++c) {
          any |= x[c] != 0;
          all &= ((x[c] - 0x01010101u) & ~x[c] & 0x80808080u) == 0;  // no byte is 0
        }
      }
    }
    in = key < p.S;
  } else {
    constexpr int CH = 16;
    const int key = k0 + lane;
    in = key < p.S;
    for (int i = i0; i <= i1; i += CH) {
      uint32_t x[CH];
#pragma unroll
      for (int c = 0; c < CH; ++c) {
        const uint8_t* q = base + EL * (row_at(min(i + c, i1)) + (in ? key : 0));
        x[c] = EL == 2 ? *(const uint16_t*)q : *(const uint32_t*)q;
      }
#pragma unroll
      for (int c = 0; c < CH; ++c) {
        // hidden: the value in log2 units is -inf (as the lowest value of fp32 and bf16 times log2 e is in fp32;
        // fp16's is -94502, a finite addend, whose tiles are computed)
        const float a = EL == 4 ? __uint_as_float(x[c])
                                : p.mask_kind == KVQ_MASK_BF16 ? to_float((uint16_t)x[c], BF16{}) : to_float((uint16_t)x[c], F16{});
        any |= !(a * 1.4426950408889634f == -INFINITY);
        all &= a == 0.0f;
      }
    }
  }
  const bool some = __builtin_amdgcn_ballot_w64(in && any) != 0;
  const bool full = __builtin_amdgcn_ballot_w64(in && all) == ~0ull;
  if (lane == 0 && some) {
    atomicOr(&s_any, 1u << wave);
    if (!full) atomicOr(&s_mixed, 1u << wave);
  }
  __syncthreads();
  if (threadIdx.x == 0) {
    uint16_t* w = words + (int64_t)u * (8 * p.nwords) + g;  // [any: 4 nwords][mixed: 4 nwords]
    w[0] = (uint16_t)s_any;
    w[4 * p.nwords] = (uint16_t)s_mixed;
  }
}

template <typename T, int BITS, int G, int D>
static hipError_t launch_t(const PreParams& p, hipStream_t stream) {
  const dim3 grid(prefill_grid(p)), block(kPW * 64);
  if (p.mask_kind == KVQ_MASK_BOOL) {
    hipLaunchKernelGGL((prefill_attn_kernel<T, BITS, false, G, D, 1>), grid, block, 0, stream, p);
  } else if constexpr (BITS == 16) {
    hipLaunchKernelGGL((prefill_attn_kernel<T, BITS, false, G, D, 2>), grid, block, 0, stream, p);
  } else {
    return hipErrorInvalidValue;  // additive masks: unquantized caches only
  }
  hipError_t e = hipGetLastError();
  if (e != hipSuccess || p.nsplit == 1 || p.fused) return e;
  hipLaunchKernelGGL((prefill_combine_kernel<T, D, true, true>), dim3(p.nunits * kPW * (D / 8)), block, 0, stream, p);
  return hipGetLastError();
}

hipError_t launch_prefill_masked_t(const PreParams& p, int B, int dtype, int D, int bits, int G, hipStream_t stream) {
  const int nkv = p.w_kv ? p.Hkv : 1;
  const dim3 grid((unsigned)(B * nkv * p.rowblocks) * 4u * (unsigned)p.nwords), block(kClassWaves * 64);
  uint16_t* words = (uint16_t*)p.words;
  if (p.mask_kind == KVQ_MASK_BOOL) {
    hipLaunchKernelGGL(mask_classes_kernel<1>, grid, block, 0, stream, p, words, nkv);
  } else if (p.mask_kind == KVQ_MASK_F32) {
    hipLaunchKernelGGL(mask_classes_kernel<4>, grid, block, 0, stream, p, words, nkv);
  } else {
    hipLaunchKernelGGL(mask_classes_kernel<2>, grid, block, 0, stream, p, words, nkv);
  }
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) return e;
  auto go = [&](auto t) -> hipError_t {
    using TT = decltype(t);
    if (bits == 16) return D == 64 ? launch_t<TT, 16, 64, 64>(p, stream) : launch_t<TT, 16, 64, 128>(p, stream);
    auto by_g = [&](auto b) -> hipError_t {
      constexpr int BB = decltype(b)::value;
      if (D == 96) return launch_t<TT, BB, 32, 96>(p, stream);
      if (D == 64) return G == 32 ? launch_t<TT, BB, 32, 64>(p, stream) : launch_t<TT, BB, 64, 64>(p, stream);
      return G == 32 ? launch_t<TT, BB, 32, 128>(p, stream)
                     : G == 64 ? launch_t<TT, BB, 64, 128>(p, stream) : launch_t<TT, BB, 128, 128>(p, stream);
    };
    return bits == 8 ? by_g(std::integral_constant<int, 8>{}) : by_g(std::integral_constant<int, 4>{});
  };
  return dtype == KVQ_DTYPE_BF16 ? go(BF16{}) : go(F16{});
}

}  // namespace kvq
