// recurrent_gla forward for bf16 inputs at head dimension 128, two waves per 16-step sub-block (the block form and the
// formulas: gla_recurrent_stream.hip).  With one wave per sub-block the workgroup of a (batch, head) pair has one wave
// per SIMD, whose 412 registers leave no room for a second, and every latency of that wave is idle time of the SIMD.
// Here wave W < NB takes sub-block W and the first half of the key features, wave W >= NB sub-block 2 NB - 1 - W and the
// second half.  Waves W and W + NB share a SIMD, and a sub-block I multiplies with I earlier ones, so every SIMD
// carries the same number of score blocks.
//
// Everything that is elementwise in the key features halves per wave.  Scores and the state's term are sums over the key
// features and enter `out` linearly, so a wave forms
//     sum_{j<=t} A'_tj v_j + (q_t e^{L_t})'^T S_in
// with the sums taken over its own features, for ALL value features, and the two waves of a sub-block exchange half of
// that sum, 16 rows of 64 value features each, once per block through LDS: no exchange of score blocks, no tile of rescaled
// queries, and no more barriers than one wave per sub-block takes.
#include "gla_subblock.hpp"
#include "gla_recurrent_stream.hpp"

namespace gla {

// The kernel and its form for the second pass of head dimension 256 (as a shared function inlined into both it spilled: 677 against
// 665 us a training step of B4 T4096 H16).
namespace two_waves {
#define GLA_FWD2_NAME recurrent_stream_fwd_kernel
#define GLA_FWD2_SECOND false
#include "gla_recurrent_stream_fwd2.inc"
#undef GLA_FWD2_NAME
#undef GLA_FWD2_SECOND
#define GLA_FWD2_NAME recurrent_stream_second_kernel
#define GLA_FWD2_SECOND true
#include "gla_recurrent_stream_fwd2.inc"
#undef GLA_FWD2_NAME
#undef GLA_FWD2_SECOND
}  // namespace two_waves

template <typename TO, bool SECOND>
static int launch_fwd2(hipStream_t st, int B, Segments sg, int H, int reverse, int hdt, const void *h0, const float *g,
                       const void *v, const void *k, const void *q, void *hT, void *out, const float *out1)
{
    typedef __bf16 T;
    constexpr int C = 64, D = 128, LS = TileGeom<T, D>::kStride;
    const size_t lds = (size_t)(3 * C + 2 * D) * LS * sizeof(T) + (size_t)(C / 16) * D * sizeof(float) +
                       (size_t)(C / 8) * (D / 32) * 64 * sizeof(f32x4);
    auto kern = SECOND ? two_waves::recurrent_stream_second_kernel<TO, C, D> : two_waves::recurrent_stream_fwd_kernel<TO, C, D>;
    static LdsGrant grant;
    if (int e = allow_lds(grant, (const void *)kern, lds)) return e;
    dim3 grid(H, sg.S, B), block(C * 8);
    hipLaunchKernelGGL(kern, grid, block, lds, st, h0, g, (const T *)v, (const T *)k, (const T *)q, hT, (TO *)out, sg, H,
                       reverse, hdt, out1);
    return launch_status();
}

template <typename TO>
int launch_recurrent_stream_fwd2(hipStream_t st, int B, Segments sg, int H, int reverse, int hdt, const void *h0,
                                 const float *g, const void *v, const void *k, const void *q, void *hT, void *out,
                                 const float *out1)
{
    return out1 ? launch_fwd2<TO, true>(st, B, sg, H, reverse, hdt, h0, g, v, k, q, hT, out, out1)
                : launch_fwd2<TO, false>(st, B, sg, H, reverse, hdt, h0, g, v, k, q, hT, out, nullptr);
}
template int launch_recurrent_stream_fwd2<__bf16>(hipStream_t, int, Segments, int, int, int, const void *, const float *,
                                                  const void *, const void *, const void *, void *, void *, const float *);
template int launch_recurrent_stream_fwd2<float>(hipStream_t, int, Segments, int, int, int, const void *, const float *,
                                                 const void *, const void *, const void *, void *, void *, const float *);

}  // namespace gla
