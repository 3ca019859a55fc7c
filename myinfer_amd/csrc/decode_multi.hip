// The decode kernel over several passes' query rows (speculative verification, short chunks and prompts:
// some query positions times the heads of a GQA group). Each row block is a unit of its own whose
// keys are read again, from L2 where the blocks run side by side: 64 rows of 4 KV heads over 8192
// 8-bit keys take 14.4 us against 18.4 on the prefill kernel, whose workgroups compute 256 rows
// whether they are there or not and take a launch to merge 32 splits. (Several row groups computed in one workgroup
// over one reading of the keys measured the same or slower up to 40 rows: 16.6 against 17.5 us at
// 40, 19.7 against 13.0 at 24; the groups' work is not hidden behind a 2-slot ring.)

#include "decode_kernel.h"

namespace kvq {

template <typename T, int D, int BITS, int G, bool PAGED>
static hipError_t launch_multi_t(const DecParams& p, hipStream_t stream) {
  hipLaunchKernelGGL((decode_attn_kernel<T, D, BITS, 4, 2, PAGED, G, false, false, true>), dim3(p.nunits * p.nsplit),
                     dim3(256), 0, stream, p);
  hipError_t e = hipGetLastError();
  if (e != hipSuccess || p.nsplit == 1 || p.fused) return e;
  return launch_combine<T, D>(merge_params(p, DecCfg<D, BITS, G>::R), p.nunits / (p.Hkv * p.rowblocks), stream);
}

hipError_t launch_decode_multi(const DecParams& p, int dtype, int D, int bits, int G, bool paged, hipStream_t stream) {
  return dispatch_quant(dtype, D, bits, G, [&](auto t, auto d, auto b, auto g) -> hipError_t {
    using T = decltype(t);
    constexpr int DD = decltype(d)::value, BB = decltype(b)::value, GG = decltype(g)::value;
    return paged ? launch_multi_t<T, DD, BB, GG, true>(p, stream) : launch_multi_t<T, DD, BB, GG, false>(p, stream);
  });
}

}  // namespace kvq
