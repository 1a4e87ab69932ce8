// recurrent_gla forward in fp32 vector arithmetic: S_t = exp(g_t) S_{t-1} + k_t v_t^T, o_t = S_t^T q_t (gla.py:35-37)
// step by step, for every element type, head dimension and length.  It is what a decode step (T = 1) runs, and every
// case without matrix-core kernels (fp32 data, head dimensions 16 and 32).
//
// At T = 1 the state is all there is: D x D values read and written for 5 D of everything else.  The state's value
// columns are independent, so a workgroup takes 32 of them with all key rows: whole 128-byte lines of an fp32 state, 16 KB
// per workgroup at D = 128, and D / 32 workgroups per (batch, head) pair.  One step at B*H = 1024, D = 128, fp32 states
// (134 MB): 87 us on the matrix-core kernel, which works through a block of 64 steps whatever T is, 23 us here =
// 5.8 TB/s (with LDS for 8 steps held at T = 1 as well: 25.7 us); one sequence of 16 heads 20 -> 5 us.
// Over many steps it is bound by the vector instructions and, with few workgroups, by the chain of a step: four columns
// per thread and the sum over the rows left to LDS once per 8 steps; the next 8 steps' inputs are requested before the
// current ones are worked through.  B*H = 256, T = 2048, D = 128, fp32: 1.87 ms for the kernel this replaced (one
// workgroup per pair, 16 columns per wave, the sum over 16 lanes formed every step), 0.98 ms here; D = 64
// 0.76 -> 0.59 ms, D = 32 0.61 -> 0.54 ms.
#include "gla_common.hpp"
#include "gla_recurrent_stream.hpp"

namespace gla {

// The workgroup's share: D key rows x W value columns per workgroup; a thread owns RPT neighbouring rows of 4 neighbouring columns.
template <int D> struct StepsGeom {
    static constexpr int W = D < 32 ? D : 32, CL = W / 4;
    static constexpr int NT = D * CL < 256 ? D * CL : 256;       // threads
    static constexpr int RPT = D * CL / NT, NP = NT / 16;         // NP: partial sums per output, one per 16 lanes
    static constexpr int kStepFloats = 3 * D + W + NP * W;       // LDS per step of a batch
    static_assert(NT % 64 == 0 && RPT * NT == D * CL, "whole waves, the same number of rows for every thread");
};

constexpr int kStepsBatch = 8;           // steps whose inputs and partial outputs are in LDS at once

template <typename T, typename TO, int D>
__global__ __launch_bounds__(StepsGeom<D>::NT) void recurrent_steps_kernel(
    const void *__restrict__ h0, const float *__restrict__ g, const T *__restrict__ v, const T *__restrict__ k,
    const T *__restrict__ q, void *hT, TO *__restrict__ out, Segments sg, int H, int reverse, int hdt)
{
    typedef StepsGeom<D> G;
    constexpr int W = G::W, CL = G::CL, NT = G::NT, RPT = G::RPT, NP = G::NP, TB = kStepsBatch;
    constexpr int kItems = (TB * D / 4 + NT - 1) / NT;           // groups of 4 features a thread brings in per batch
    extern __shared__ __align__(16) float smem[];
    const int tid = threadIdx.x, cl = tid % CL, rg = tid / CL;
    const SegmentRows seg(sg, blockIdx.z, blockIdx.y);
    const int T_len = seg.len;
    const int h = blockIdx.x / (D / W), slab = blockIdx.x % (D / W);
    const int64_t bh = (int64_t)seg.index * H + h;
    const int64_t ho = (bh * D + rg * RPT) * D + slab * W + 4 * cl;
    const int64_t seq = (seg.row0 * H + h) * D, rowstride = (int64_t)H * D;
    const int tb = T_len < TB ? T_len : TB;                      // the launcher's LDS holds this many steps
    float *sf = smem, *sk = sf + tb * D, *sq = sk + tb * D;      // [tb][D] e^g, key, query
    float *sv = sq + tb * D, *part = sv + tb * W;                // [tb][W] value; [tb][NP][W] partial outputs

    float S[RPT][4];
#pragma unroll
    for (int i = 0; i < RPT; ++i) {
#pragma unroll
        for (int j = 0; j < 4; ++j) S[i][j] = 0.f;
        if (h0) load_hidden<4>(h0, hdt, ho + (int64_t)i * D, S[i]);
    }

    auto row = [&](int step) { return seq + (int64_t)(reverse ? T_len - 1 - step : step) * rowstride; };
    float gN[kItems][4], kN[kItems][4], qN[kItems][4], vN[4];
    auto fetch = [&](int t0) {
        const int nb = T_len - t0 < TB ? T_len - t0 : TB;
#pragma unroll
        for (int u = 0; u < kItems; ++u) {
            const int i = tid + u * NT;
            if (i < nb * (D / 4)) {
                const int64_t o = row(t0 + i / (D / 4)) + i % (D / 4) * 4;
                load_vec<float, 4>(g + o, gN[u]);
                load_vec<T, 4>(k + o, kN[u]);
                load_vec<T, 4>(q + o, qN[u]);
            }
        }
        if (tid < nb * CL) load_vec<T, 4>(v + row(t0 + tid / CL) + slab * W + tid % CL * 4, vN);
    };
    static_assert(TB * CL <= NT, "one group of 4 value features per thread and batch");
    fetch(0);
    for (int t0 = 0; t0 < T_len; t0 += TB) {
        const int nb = T_len - t0 < TB ? T_len - t0 : TB;
#pragma unroll
        for (int u = 0; u < kItems; ++u) {
            const int i = tid + u * NT;
            if (i < nb * (D / 4)) {
                float x[4];
#pragma unroll
                for (int e = 0; e < 4; ++e) x[e] = fast_exp2(gN[u][e] * kLog2e);
                store_vec<float, 4>(sf + 4 * i, x);
                store_vec<float, 4>(sk + 4 * i, kN[u]);
                store_vec<float, 4>(sq + 4 * i, qN[u]);
            }
        }
        if (tid < nb * CL) store_vec<float, 4>(sv + 4 * tid, vN);
        lds_barrier();
        if (t0 + TB < T_len) fetch(t0 + TB);                     // on its way while this batch is worked through
        for (int s = 0; s < nb; ++s) {
            float vv[4], f[RPT], kk[RPT], qq[RPT], o[4] = {0.f, 0.f, 0.f, 0.f};
            load_vec<float, 4>(sv + s * W + 4 * cl, vv);
            load_vec<float, RPT>(sf + s * D + rg * RPT, f);
            load_vec<float, RPT>(sk + s * D + rg * RPT, kk);
            load_vec<float, RPT>(sq + s * D + rg * RPT, qq);
#pragma unroll
            for (int i = 0; i < RPT; ++i)
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    S[i][j] = f[i] * S[i][j] + kk[i] * vv[j];
                    o[j] += qq[i] * S[i][j];
                }
            // sum over the row groups of 16 lanes (4 lanes apart at D = 16 only, 8 apart); the rest goes through LDS
            // once per batch (a sum over the whole wave here took four more cross-lane trips per step)
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                if (CL == 4) o[j] += dpp_f32<0x124>(o[j]);       // row_ror:4
                o[j] += dpp_f32<0x128>(o[j]);                    // row_ror:8
            }
            if ((tid & 15) < CL) store_vec<float, 4>(part + (s * NP + (tid >> 4)) * W + 4 * cl, o);
        }
        lds_barrier();
        if (tid < nb * CL) {
            const int s = tid / CL, col = tid % CL * 4;
            float o[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int m = 0; m < NP; ++m) {
                float x[4];
                load_vec<float, 4>(part + (s * NP + m) * W + col, x);
#pragma unroll
                for (int j = 0; j < 4; ++j) o[j] += x[j];
            }
            store_vec<TO, 4>(out + row(t0 + s) + slab * W + col, o);
        }
    }
#pragma unroll
    for (int i = 0; i < RPT; ++i) store_hidden<4>(hT, hdt, ho + (int64_t)i * D, S[i]);
}

template <typename T, typename TO>
int launch_recurrent_steps(hipStream_t st, int B, Segments sg, int H, int D, int reverse, int hdt, const void *h0,
                           const float *g, const void *v, const void *k, const void *q, void *hT, void *out)
{
    const size_t tb = sg.L < kStepsBatch ? sg.L : kStepsBatch;
#define GLA_STEPS_CASE(D_)                                                                                          \
    case D_:                                                                                                        \
        hipLaunchKernelGGL((recurrent_steps_kernel<T, TO, D_>), dim3(H * (D_ / StepsGeom<D_>::W), sg.S, B),               \
                           dim3(StepsGeom<D_>::NT), tb * StepsGeom<D_>::kStepFloats * sizeof(float), st, h0, g, (const T *)v, (const T *)k, (const T *)q, hT,     \
                           (TO *)out, sg, H, reverse, hdt);                                                      \
        break
    switch (D) {
    GLA_STEPS_CASE(16);
    GLA_STEPS_CASE(32);
    GLA_STEPS_CASE(64);
    GLA_STEPS_CASE(128);
    GLA_STEPS_CASE(256);
    default: return GLA_ERR_SHAPE;
    }
#undef GLA_STEPS_CASE
    return launch_status();
}

template int launch_recurrent_steps<__bf16, __bf16>(hipStream_t, int, Segments, int, int, int, int, const void *, const float *,
                                                    const void *, const void *, const void *, void *, void *);
template int launch_recurrent_steps<__bf16, float>(hipStream_t, int, Segments, int, int, int, int, const void *, const float *,
                                                   const void *, const void *, const void *, void *, void *);
template int launch_recurrent_steps<float, float>(hipStream_t, int, Segments, int, int, int, int, const void *, const float *,
                                                  const void *, const void *, const void *, void *, void *);

}  // namespace gla
