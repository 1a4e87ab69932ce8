// recurrent_gla backward for bf16 data (dout included) at head dimension 128, two waves per 16-step sub-block: the two sweeps
// of gla_recurrent_stream_bwd.hip (block form and formulas there; gla.py:271-360, 263), cut as in
// gla_recurrent_stream_fwd2.hip: wave W < NB takes sub-block W and the first half of the key features, wave W >= NB
// sub-block 2 NB - 1 - W and the second half, so that the two waves of a SIMD carry NB - 1 links of Horner chains between them.
// Gates, the rescaled tiles, dq, dk, q*dq and d(log_fgate) are handled on the wave's 64 key features, 32 at a time.
// Products that contract over the value features (dA = dO V^T, the states' terms of dq and dk) are formed by both waves, with
// operands from LDS tiles that both fill.
//
// B4 T4096 H16 D128 (256 workgroups of 1024 steps): sweep 1 225 -> 152 us, 650 MB at 4.3 TB/s, against 4.9 of a large copy.
// With one wave per sub-block it was one wave per SIMD with more than 400 registers.
#include "gla_recurrent_stream_bwd.hpp"
#include "gla_recurrent_stream.hpp"

namespace gla {

// ---------------------------------------------------------------------------------------------------
// sweep 1: dq and q*dq, the state S in accumulator registers
// ---------------------------------------------------------------------------------------------------
// WIDE: dq is a float array (head dimension 256 adds two such runs and rounds once, gla_split.hip)
template <int C, int D, bool WIDE>
__global__ __launch_bounds__(C * 8) void recurrent_stream_dq128_kernel(
    const void *__restrict__ h0, const float *__restrict__ g, const BT *__restrict__ v, const BT *__restrict__ k,
    const BT *__restrict__ q, const void *__restrict__ dhT, const BT *__restrict__ dout,
    std::conditional_t<WIDE, float, BT> *__restrict__ dq, float *__restrict__ qdq, Segments sg, int H, int reverse, int hdt)
{
    typedef BT T;
    typedef std::conditional_t<WIDE, float, BT> TG;
    constexpr int NB = C / 16, NW = 2 * NB, KS = D / 32, NT = D / 16;
    constexpr int DH = D / 2, KH = DH / 32;                          // a wave's key features, in slices of 32
    constexpr int RT = NT / NB, NTW = NT / 2;                        // its state tiles: RT value tiles x NTW key tiles
    static_assert(NT % NB == 0 && DH % 32 == 0, "the state tiles split evenly over the waves");
    constexpr int LS = TileGeom<T, D>::kStride;
    constexpr int XS = 32 + 16 / (int)sizeof(T);
    typedef FragTypes<T>::d8 D8;
    typedef FragTypes<T>::t4 T4;
    extern __shared__ __align__(16) unsigned char smem[];
    T *Vn = reinterpret_cast<T *>(smem);           // [C][LS]  value
    T *tO = Vn + C * LS;                           // [C][LS]  dout
    T *Kh = tO + C * LS;                           // [C][LS]  k * exp(tau_J - l_j), bf16 head
    T *Kl = Kh + C * LS;                           // [C][LS]  ... and remainder
    T *Sh = Kl + C * LS;                           // [D][LS]  state at the start of the block, [dk][dv], head
    T *Sl = Sh + D * LS;                           // [D][LS]  ... and remainder
    T *xs = Sl + D * LS;                           // [NW][2][16][XS] per-wave scratch (hard gates only)
    float *rtab = reinterpret_cast<float *>(xs + NW * 2 * 16 * XS);   // [NB][D] exp(tau_m)

    const int lane = threadIdx.x & 63;
    const int W = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int I = W < NB ? W : NW - 1 - W;         // the wave's sub-block
    const int fo = W < NB ? 0 : DH;                // ... and its first feature
    const int r = lane & 15, c = lane >> 4;
    const SegmentRows seg(sg, blockIdx.z, blockIdx.y);
    const int T_len = seg.len;
    const int h = blockIdx.x;
    const int64_t seq = (seg.row0 * H + h) * D;
    const int64_t rowstride = (int64_t)H * D;
    const int64_t bh = (int64_t)seg.index * H + h;
    const TrLane<T> L = make_tr_lane<T>(LS);
    const TrLane<T> Lx = make_tr_lane<T>(XS);
    const int ptl = plain_tr_lane<T>(LS);
    const int wrow = 16 * I * LS + L.nat;          // this lane's row of a tile, features 8c..8c+7
    T *xh = xs + (2 * W) * 16 * XS, *xl = xh + 16 * XS;
    const int N = (T_len + C - 1) / C;
    const int tv = RT * (W % NB), nt0 = NTW * (W / NB);

    // state: S[i][j][e] = state[dk = 16(nt0 + j) + r][dv = 16(tv + i) + 4c + e]
    f32x4 S[RT][NTW];
#pragma unroll
    for (int i = 0; i < RT; ++i)
#pragma unroll
        for (int j = 0; j < NTW; ++j) {
            float t4[4];
            load_hidden<4>(h0, hdt, bh * D * D + (int64_t)(16 * (nt0 + j) + r) * D + 16 * (tv + i) + 4 * c, t4);
            S[i][j] = f32x4{t4[0], t4[1], t4[2], t4[3]};
        }
    auto publish_state = [&]() {
#pragma unroll
        for (int i = 0; i < RT; ++i)
#pragma unroll
            for (int j = 0; j < NTW; ++j) {
                T4 hi, lo;
                split4<T>(S[i][j], hi, lo);
                const int off = (16 * (nt0 + j) + r) * LS + 16 * (tv + i) + 4 * c;
                *reinterpret_cast<T4 *>(Sh + off) = hi;
                *reinterpret_cast<T4 *>(Sl + off) = lo;
            }
    };
    publish_state();

    f32x8 gN[KH];
    D8 qN[KH], kN[KH], vN[KH], dN[KH];
    bool validN;
    int64_t rowN;
    // The rows of a block are requested in two pieces, see the loop (all before the state update 2 us more; keys and queries ahead of
    // the slices, or a block's results stored a block late, the same).
    auto fetch_g = [&](int n) {
        const int s = n * C + 16 * I + r;
        validN = s < T_len;
        const int sc = validN ? s : T_len - 1;
        rowN = seq + (int64_t)(reverse ? T_len - 1 - sc : sc) * rowstride + fo + 8 * c;
#pragma unroll
        for (int ks = 0; ks < KH; ++ks) gN[ks] = ld8(g + rowN + 32 * ks);
    };
    auto fetch_qk = [&]() {
#pragma unroll
        for (int ks = 0; ks < KH; ++ks) {
            qN[ks] = ld8(q + rowN + 32 * ks);
            kN[ks] = ld8(k + rowN + 32 * ks);
        }
    };
    auto fetch_vo = [&]() {
#pragma unroll
        for (int ks = 0; ks < KH; ++ks) {
            vN[ks] = ld8(v + rowN + 32 * ks);
            dN[ks] = ld8(dout + rowN + 32 * ks);
        }
    };
    fetch_g(0);
    fetch_qk();
    fetch_vo();

#pragma unroll 1
    for (int n = 0; n < N; ++n) {
        const bool valid = validN;
        const int64_t row = rowN;            // element offset of the lane's first 8 features of its row
        float p[8 * KH];                     // l_i
        D8 qf[KH], kf[KH];
        bool one_anchor[KH];
        if ((n + 1) * C > T_len && !valid) {   // only the last block can hold padded steps
            float z[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int ks = 0; ks < KH; ++ks) {
                gN[ks] = pack8<float>(z);
                qN[ks] = kN[ks] = vN[ks] = dN[ks] = pack8<T>(z);
            }
        }
#pragma unroll
        for (int ks = 0; ks < KH; ++ks) {
            float *pp = p + 8 * ks;
            float bq[8];
#pragma unroll
            for (int e = 0; e < 8; ++e) pp[e] = gN[ks].v[e] * kLog2e;
            qf[ks] = qN[ks];
            kf[ks] = kN[ks];
            unpack8(kf[ks], bq);
            st8(Vn + wrow + fo + 32 * ks, vN[ks]);
            st8(tO + wrow + fo + 32 * ks, dN[ks]);

            // gate prefix, totals through the wave's part of the table row, one anchor or not
            float *rt = rtab + I * D + fo + 32 * ks + 8 * c;
#pragma unroll
            for (int e = 0; e < 8; ++e) pp[e] = prefix_sum_rows(pp[e]);
            if (r == 15) st8(rt, pack8<float>(pp));
            asm volatile("" ::: "memory");
            const f32x8 tau = ld8(rt);
            float span = 0.f, sv[8], rw[8];
#pragma unroll
            for (int e = 0; e < 8; ++e) {
                sv[e] = tau.v[e] - pp[e];
                span = fmaxf(span, fmaxf(fabsf(pp[e]), fabsf(sv[e])));
            }
            one_anchor[ks] = wave_all_below(span, kOneAnchorSpan);
            if (__builtin_expect(!one_anchor[ks], false)) {
                // hard gates: l_i and tau - l_i from the sibling hierarchy instead (a suffix sum of its own, not the
                // difference of two long prefix sums)
                float p8[8], s8[8];
#pragma unroll
                for (int e = 0; e < 8; ++e) {
                    p8[e] = gN[ks].v[e] * kLog2e;
                    s8[e] = 0.f;
                }
                hier_step<1>(p8, s8, (r & 1) != 0);
                hier_step<2>(p8, s8, (r & 2) != 0);
                hier_step<4>(p8, s8, (r & 4) != 0);
                hier_step<8>(p8, s8, (r & 8) != 0);
#pragma unroll
                for (int e = 0; e < 8; ++e) {
                    pp[e] = p8[e];
                    sv[e] = s8[e];
                }
            }
#pragma unroll
            for (int e = 0; e < 8; ++e) {
                bq[e] *= fast_exp2(sv[e]);               // tau - l_i <= 0 whatever the gates
                rw[e] = fast_exp2(pp[e] + sv[e]);
            }
            D8 kh, kl;
            split8<T>(bq, kh, kl);
            st8(Kh + wrow + fo + 32 * ks, kh);
            st8(Kl + wrow + fo + 32 * ks, kl);
            asm volatile("" ::: "memory");
            if (r == 0) st8(rt, pack8<float>(rw));
        }
        lds_barrier();                       // tiles of this block and the published state are in place
        if (__builtin_expect(!(one_anchor[0] && one_anchor[1]), false)) {
            // Hard gates: the own sub-block's part of dq from the dyadic levels, inputs fetched again.  It waits in the rows'
            // place in the q*dq array, and the call is made here, where next to nothing but the state is live: among the
            // products below what lives across it was spilled on the path without it (B4 T4096 H16 D128 201 against 150 us).
            f32x4 At = {0.f, 0.f, 0.f, 0.f}, An = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int k2 = 0; k2 < KS; ++k2) {
                const D8 o8 = ld8(tO + wrow + 32 * k2), v8 = ld8(Vn + wrow + 32 * k2);
                At = mma_d(v8, o8, At);
                An = mma_d(o8, v8, An);
            }
            float diag = 0.f;
#pragma unroll
            for (int e = 0; e < 4; ++e) diag += (4 * c + e == r) ? At[e] : 0.f;
            diag = reduce_over_cgroups(diag);
#pragma unroll 1
            for (int ks = 0; ks < KH; ++ks) {
                const HardSliceDq hs = hard_slice_dq<XS, false>(
                    g + row + 32 * ks, q + row + 32 * ks, k + row + 32 * ks, valid ? 1.f : 0.f, diag, At, An, (LdsBT)xh,
                    (LdsBT)xl, Lx.nat, Lx.k4, (LdsF32) nullptr, (LdsBT) nullptr, (LdsBT) nullptr);
                if (valid) st8(qdq + row + 32 * ks, pack8<float>(hs.dq8));
            }
        }
        const bool more = n + 1 < N;
        if (more) fetch_g(n + 1);
        __builtin_amdgcn_sched_barrier(0);

        // dA = dO V^T contracts over all value features.  dAt[e] = dA[i = r][j = 4c+e] of the own sub-block;
        // dA^T of the pairs with the earlier sub-blocks, [j][i] = v_j . do_i.
        D8 dof[KS];
        T4 dah[NB], dal[NB], lowTh, lowTl;
        f32x4 dAt = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int k2 = 0; k2 < KS; ++k2) {
            dof[k2] = ld8(tO + wrow + 32 * k2);
            dAt = mma_d(ld8(Vn + wrow + 32 * k2), dof[k2], dAt);
        }
#pragma unroll
        for (int J = 0; J < NB - 1; ++J) {
            f32x4 da = {0.f, 0.f, 0.f, 0.f};
            if (J < I) {
#pragma unroll
                for (int k2 = 0; k2 < KS; ++k2) da = mma_d(ld8(Vn + L.nat + 16 * J * LS + 32 * k2), dof[k2], da);
            }
            split4<T>(da, dah[J], dal[J]);
        }
        float dd = 0.f;
        {
            f32x4 low;                       // dA^T below the diagonal
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                dd += (4 * c + e == r) ? dAt[e] : 0.f;
                low[e] = (4 * c + e < r) ? dAt[e] : 0.f;
            }
            dd = reduce_over_cgroups(dd);
            split4<T>(low, lowTh, lowTl);
        }
        __builtin_amdgcn_sched_barrier(0);

#pragma unroll
        for (int ks = 0; ks < KH; ++ks) {
            const int f = fo + 32 * ks;
            // the state term of the slice, then the earlier sub-blocks in ascending order
            f32x4 acc[2] = {{0.f, 0.f, 0.f, 0.f}, {0.f, 0.f, 0.f, 0.f}};
#pragma unroll
            for (int k2 = 0; k2 < KS; ++k2)
#pragma unroll
                for (int tt = 0; tt < 2; ++tt) {
                    acc[tt] = mma_d(ld8(Sl + L.own + (f + 4 * tt) * LS + 32 * k2), dof[k2], acc[tt]);
                    acc[tt] = mma_d(ld8(Sh + L.own + (f + 4 * tt) * LS + 32 * k2), dof[k2], acc[tt]);
                }
#pragma unroll
            for (int J = 0; J < NB - 1; ++J) {
                if (J < I) {
                    const f32x8 rr = ld8(rtab + J * D + f + 8 * c);
#pragma unroll
                    for (int tt = 0; tt < 2; ++tt) {
#pragma unroll
                        for (int e = 0; e < 4; ++e) acc[tt][e] *= rr.v[4 * tt + e];
                        const int at = L.k4 + f + 4 * tt + 16 * J * LS;
                        acc[tt] = mma_t_split(lds_tr4(Kh + at, LS), lds_tr4(Kl + at, LS), dah[J], dal[J], acc[tt]);
                    }
                }
            }
            // the own sub-block
            float dqo[8];                        // its part of dq (already scaled)
            f32x4 gq[2] = {{0.f, 0.f, 0.f, 0.f}, {0.f, 0.f, 0.f, 0.f}};
            if (__builtin_expect(one_anchor[ks], true)) {
#pragma unroll
                for (int tt = 0; tt < 2; ++tt) {
                    const int at = L.k4 + f + 4 * tt + 16 * I * LS;
                    gq[tt] = mma_t_split(lds_tr4(Kh + at, LS), lds_tr4(Kl + at, LS), lowTh, lowTl, gq[tt]);
                }
                unpack8(kf[ks], dqo);
#pragma unroll
                for (int e = 0; e < 8; ++e) dqo[e] *= dd;                    // diagonal term (gla.py:1181-1185)
            } else {
                const f32x8 t = ld8(refetch(qdq) + row + 32 * ks);
#pragma unroll
                for (int e = 0; e < 8; ++e) dqo[e] = valid ? t.v[e] : 0.f;
            }
            const f32x8 rw = ld8(rtab + I * D + f + 8 * c);
            float o[8], a[8];
            unpack8(qf[ks], a);
            f32x8 prod;
#pragma unroll
            for (int e = 0; e < 8; ++e) {
                const float el = fast_exp2(p[8 * ks + e]);
                const float es = one_anchor[ks] ? el * __builtin_amdgcn_rcpf(rw.v[e]) : 0.f;   // e^{-s} = e^{l} / e^{tau}
                o[e] = el * acc[e >> 2][e & 3] + es * gq[e >> 2][e & 3] + dqo[e];
                prod.v[e] = a[e] * o[e];
            }
            if (valid) {
                st8(dq + row + 32 * ks, pack8<TG>(o));
                st8(qdq + row + 32 * ks, prod);
            }
        }
        __builtin_amdgcn_sched_barrier(0);
        if (more) {
            fetch_qk();
            fetch_vo();
        }
        __builtin_amdgcn_sched_barrier(0);

        // ---- state update: S <- S e^{tau_J} + V_J^T (k e^{tau_J - l})_J over the sub-blocks in order ------
#pragma unroll
        for (int J = 0; J < NB; ++J) {
            T4 va[RT];
#pragma unroll
            for (int i = 0; i < RT; ++i) va[i] = lds_tr4(Vn + ptl + 16 * J * LS + 16 * (tv + i), LS);
#pragma unroll
            for (int j = 0; j < NTW; ++j) {
                const float rr = rtab[J * D + 16 * (nt0 + j) + r];
                const T4 kl = lds_tr4(Kl + ptl + 16 * J * LS + 16 * (nt0 + j), LS);
                const T4 kh = lds_tr4(Kh + ptl + 16 * J * LS + 16 * (nt0 + j), LS);
#pragma unroll
                for (int i = 0; i < RT; ++i) {
                    S[i][j] *= rr;
                    S[i][j] = mma_t2(va[i], va[i], kl, kh, S[i][j]);
                }
            }
        }
        lds_barrier();                       // every wave is done with the tiles and the old state
        publish_state();
    }

    // The last term of gla.py:263, sum_v dhT * hT per key feature, from the state this sweep ends with (just
    // published as bf16 head + remainder), is added to q*dq of the LAST step: see recurrent_stream_dq2_kernel.
    __syncthreads();           // the published state and every q*dq row are in place
    {
        constexpr int LPF = C * 8 / D, PART = D / LPF;                   // lanes per key feature, values of a lane
        static_assert(LPF == 4 && PART % 8 == 0, "a quad of lanes shares a key feature");
        const int d = threadIdx.x / LPF, part = threadIdx.x % LPF;
        float acc = 0.f;
#pragma unroll
        for (int i = 0; i < PART; i += 8) {
            float dv8[8], sh[8], sl[8];
            load_hidden<8>(dhT, hdt, bh * D * D + (int64_t)d * D + part * PART + i, dv8);
            unpack8(ld8(Sh + d * LS + part * PART + i), sh);
            unpack8(ld8(Sl + d * LS + part * PART + i), sl);
#pragma unroll
            for (int e = 0; e < 8; ++e) acc += dv8[e] * (sh[e] + sl[e]);
        }
        acc += dpp_f32<kDppQuadXor1>(acc);
        acc += dpp_f32<kDppQuadXor2>(acc);
        if (part == 0) {
            float *lp = qdq + seq + (int64_t)(reverse ? 0 : T_len - 1) * rowstride + d;
            *lp += acc;
        }
    }
}

template <int C, int D, bool WIDE>
static int launch_dq128(hipStream_t st, int B, Segments sg, int H, int reverse, int hdt, const void *h0, const float *g,
                        const void *v, const void *k, const void *q, const void *dhT, const void *dout, void *dq,
                        float *qdq)
{
    typedef BT T;
    constexpr int LS = TileGeom<T, D>::kStride;
    constexpr int XS = 32 + 16 / (int)sizeof(T);
    const size_t lds = ((size_t)(4 * C + 2 * D) * LS + (size_t)(C / 8) * 2 * 16 * XS) * sizeof(T) +
                       (size_t)(C / 16) * D * sizeof(float);
    auto kern = recurrent_stream_dq128_kernel<C, D, WIDE>;
    static LdsGrant grant;
    if (int e = allow_lds(grant, (const void *)kern, lds)) return e;
    dim3 grid(H, sg.S, B), block(C * 8);
    hipLaunchKernelGGL(kern, grid, block, lds, st, h0, g, (const T *)v, (const T *)k, (const T *)q, dhT, (const T *)dout,
                       (std::conditional_t<WIDE, float, T> *)dq, qdq, sg, H, reverse, hdt);
    return launch_status();
}

int launch_recurrent_stream_dq128(hipStream_t st, int B, Segments sg, int H, int reverse, int hdt, const void *h0,
                                  const float *g, const void *v, const void *k, const void *q, const void *dhT,
                                  const void *dout, void *dq, float *qdq, int wide)
{
    return wide ? launch_dq128<64, 128, true>(st, B, sg, H, reverse, hdt, h0, g, v, k, q, dhT, dout, dq, qdq)
                : launch_dq128<64, 128, false>(st, B, sg, H, reverse, hdt, h0, g, v, k, q, dhT, dout, dq, qdq);
}

}  // namespace gla
