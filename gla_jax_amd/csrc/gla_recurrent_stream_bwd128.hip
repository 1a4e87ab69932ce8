// recurrent_gla backward for bf16 data (dout included) at head dimension 128, two waves per 16-step sub-block: the two sweeps
// of gla_recurrent_stream_bwd.hip (block form and formulas there; gla.py:271-360, 263), cut as in
// gla_recurrent_stream_fwd2.hip: wave W < NB takes sub-block W and the first half of the key features, wave W >= NB
// sub-block 2 NB - 1 - W and the second half, so that the two waves of a SIMD carry NB - 1 links of Horner chains between them.
// Gates, the rescaled tiles, dq, dk, q*dq and d(log_fgate) are handled on the wave's 64 key features, 32 at a time.
// Products that contract over the value features (dA = dO V^T, the states' terms of dq and dk) are formed by both waves, with
// operands from LDS tiles that both fill.
//
// B4 T4096 H16 D128 (256 workgroups of 1024 steps): sweep 1 225 -> 152 us, 652 MB by counter (its rows are 604) at 4.3 TB/s, against
// 4.9 of a large copy; sweep 2 320 -> 244 us, 984 MB by counter at 4.1 TB/s: its rows and states are 839, the rest the value rows that
// both waves read and spilled registers, about ten a lane and block.  With one wave per sub-block it was one wave per SIMD with more than
// 400 registers.
// What sweep 2 waits for is the sum of its parts: a 64-step block is 32 000 cycles, of them (counted) 12 000 of vector arithmetic, 6 000
// of matrix instructions and 9 000 of LDS traffic per SIMD or CU, which two waves between two barriers overlap little.
#include "gla_recurrent_stream_bwd.hpp"
#include "gla_recurrent_stream.hpp"

namespace gla {

// ---------------------------------------------------------------------------------------------------
// sweep 1: dq and q*dq, the state S in accumulator registers
// ---------------------------------------------------------------------------------------------------
// WIDE: the passes of head dimension 256 (gla_split.hip).  1: dq is a float array; 2: the value-side rows of the other half, and
// dq1, what the first pass left, is added before the one rounding.
template <int C, int D, int WIDE>
__global__ __launch_bounds__(C * 8) void recurrent_stream_dq128_kernel(
    const void *__restrict__ h0, const float *__restrict__ g, const BT *__restrict__ v, const BT *__restrict__ k,
    const BT *__restrict__ q, const void *__restrict__ dhT, const BT *__restrict__ dout,
    std::conditional_t<WIDE == 1, float, BT> *__restrict__ dq, float *__restrict__ qdq,
    Segments sg, int H, int reverse, int hdt, const float *__restrict__ dq1)
{
    typedef BT T;
    typedef std::conditional_t<WIDE == 1, float, BT> TG;
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
    if constexpr (WIDE == 2) {
        const int other = ((h ^ 1) - h) * D;
        v += other;
        dout += other;
    }
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
            if constexpr (WIDE == 2) {
                const f32x8 t = ld8(dq1 + row + 32 * ks);
#pragma unroll
                for (int e = 0; e < 8; ++e) o[e] += t.v[e];
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

template <int C, int D, int WIDE>
static int launch_dq128(hipStream_t st, int B, Segments sg, int H, int reverse, int hdt, const void *h0, const float *g,
                        const void *v, const void *k, const void *q, const void *dhT, const void *dout, void *dq,
                        float *qdq, const float *dq1)
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
                       (std::conditional_t<WIDE == 1, float, T> *)dq, qdq, sg, H, reverse, hdt, dq1);
    return launch_status();
}

int launch_recurrent_stream_dq128(hipStream_t st, int B, Segments sg, int H, int reverse, int hdt, const void *h0,
                                  const float *g, const void *v, const void *k, const void *q, const void *dhT,
                                  const void *dout, void *dq, float *qdq, int wide, const float *dq1)
{
    auto run = wide == 2 ? launch_dq128<64, 128, 2> : wide ? launch_dq128<64, 128, 1> : launch_dq128<64, 128, 0>;
    return run(st, B, sg, H, reverse, hdt, h0, g, v, k, q, dhT, dout, dq, qdq, dq1);
}

// ---------------------------------------------------------------------------------------------------
// sweep 2: dk, dv, dh0 and d(log_fgate), dS in accumulator registers.
// The scores A = Q~ K~^T and the state's term of dv are sums over the key features and enter dv linearly: each wave forms them
// on its own 64 key features, for all value features, and hands the half that the other wave stores to it through LDS, once
// per block.  So K~ never leaves the wave's registers, and a block has two barriers.  Both waves of a sub-block read its value
// rows from memory (the second time from cache), which no other wave needs.
// ---------------------------------------------------------------------------------------------------
template <int C, int D, int WIDE>
__global__ __launch_bounds__(C * 8) void recurrent_stream_rev128_kernel(
    const float *__restrict__ g, const BT *__restrict__ v, const BT *__restrict__ k, const BT *__restrict__ q,
    const void *__restrict__ dhT, const BT *__restrict__ dout, void *__restrict__ dh0, float *__restrict__ dg,
    std::conditional_t<WIDE == 1, float, BT> *__restrict__ dv, std::conditional_t<WIDE == 1, float, BT> *__restrict__ dk,
    Segments sg, int H, int reverse, int hdt, const float *__restrict__ dv1, const float *__restrict__ dk1, float *__restrict__ dg1)
{
    typedef BT T;
    typedef std::conditional_t<WIDE == 1, float, BT> TG;
    constexpr int NB = C / 16, NW = 2 * NB, KS = D / 32, NT = D / 16;
    constexpr int DH = D / 2, KH = DH / 32;                          // a wave's features, in slices of 32
    constexpr int RT = NT / NB, NTW = NT / 2;                        // its state tiles: RT key tiles x NTW value tiles
    static_assert(NT % NB == 0 && KH == 2, "the state tiles split evenly over the waves");
    constexpr int LS = TileGeom<T, D>::kStride;
    constexpr int XS = 32 + 16 / (int)sizeof(T);
    typedef FragTypes<T>::d8 D8;
    typedef FragTypes<T>::t4 T4;
    extern __shared__ __align__(16) unsigned char smem[];
    T *tO = reinterpret_cast<T *>(smem);           // [C][LS]  dout
    T *Qh = tO + C * LS;                           // [C][LS]  q * exp(l_i), bf16 head
    T *Ql = Qh + C * LS;                           // [C][LS]  ... and remainder
    T *DTh = Ql + C * LS;                          // [D][LS]  dS' as [dv][dk], head
    T *DTl = DTh + D * LS;                         // [D][LS]  ... and remainder
    f32x4 *xch = reinterpret_cast<f32x4 *>(DTl + D * LS);            // [NW][2 KH][64] the other wave's half of dv
    static_assert(2 * 16 * XS * sizeof(T) <= 2 * KH * 64 * sizeof(f32x4), "the levels' scratch lies in the wave's part of xch");
    float *rtab = reinterpret_cast<float *>(xch + NW * 2 * KH * 64); // [NB][D] exp(tau_m)
    float *dltab = rtab + NB * D;                  // [NB][D] sub-block sums of q*dq - k*dk
    float *runtab = dltab + NB * D;                // [2][D]  sum over the later blocks, double-buffered

    const int lane = threadIdx.x & 63;
    const int W = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int J0 = W < NB ? W : NW - 1 - W;        // the wave's sub-block
    const int fo = W < NB ? 0 : DH;                // ... and its first feature
    const int PW = NW - 1 - W;                     // the wave with the other half of the sub-block
    const int r = lane & 15, c = lane >> 4;
    const SegmentRows seg(sg, blockIdx.z, blockIdx.y);
    const int T_len = seg.len;
    const int h = blockIdx.x;
    const int64_t seq = (seg.row0 * H + h) * D;
    const int64_t rowstride = (int64_t)H * D;
    if constexpr (WIDE == 2) {           // (see sweep 1; the gates' gradient is added to dg1, `dg` holds sweep 1's q*dq of this pass)
        const int other = ((h ^ 1) - h) * D;
        v += other;
        dout += other;
        dv += other;
        dv1 += other;
    }
    const int64_t bh = (int64_t)seg.index * H + h;
    TrLane<T> L = make_tr_lane<T>(LS);
    const TrLane<T> Lx = make_tr_lane<T>(XS);
    int ptl = plain_tr_lane<T>(LS);
    int c8 = 8 * c, slot = lane;
    // this wave's part of xch: written by it, dv's half read by wave PW
    auto mine = [&](int i) -> f32x4 & { return xch[(W * 2 * KH + i) * 64 + slot]; };
    auto theirs = [&](int i) -> const f32x4 & { return xch[(PW * 2 * KH + i) * 64 + slot]; };
    T *xh = reinterpret_cast<T *>(xch + W * 2 * KH * 64), *xl = xh + 16 * XS;   // (hard gates only)
    const int N = (T_len + C - 1) / C;
    const int tk = RT * (W % NB), nt0 = NTW * (W / NB);

    int pub = r * LS + 4 * c;
    // dS: DS[i][j][e] = dS[dk = 16(tk + i) + 4c + e][dv = 16(nt0 + j) + r]; memory is read and written by rows
    f32x4 DS[RT][NTW];
    auto hidden_at = [&](int i, int j) {
        return bh * D * D + (int64_t)(16 * (tk + i) + 4 * c + (r & 3)) * D + 16 * (nt0 + j) + (r & ~3);
    };
#pragma unroll
    for (int i = 0; i < RT; ++i)
#pragma unroll
        for (int j = 0; j < NTW; ++j) {
            float t4[4];
            load_hidden<4>(dhT, hdt, hidden_at(i, j), t4);
            quad_transpose(t4);
            DS[i][j] = f32x4{t4[0], t4[1], t4[2], t4[3]};
        }
    auto publish = [&]() {
#pragma unroll
        for (int i = 0; i < RT; ++i)
#pragma unroll
            for (int j = 0; j < NTW; ++j) {
                T4 hi, lo;
                split4<T>(DS[i][j], hi, lo);
                const int off = 16 * (nt0 + j) * LS + 16 * (tk + i) + pub;
                *reinterpret_cast<T4 *>(DTh + off) = hi;
                *reinterpret_cast<T4 *>(DTl + off) = lo;
            }
    };
    // the wave with the longer chains of the two on a SIMD goes first when both are ready
    if (J0 < NB / 2) __builtin_amdgcn_s_setprio(1);
    publish();
    for (int d = threadIdx.x; d < 2 * D; d += C * 8) runtab[d] = 0.f;

    f32x8 gN[KH];
    D8 qN[KH], kN[KH], dN[KH], vN[KS];
    bool validN;
    int64_t rowN;
    auto fetch_g = [&](int n) {
        const int s = n * C + 16 * J0 + r;
        validN = s < T_len;
        const int sc = validN ? s : T_len - 1;
        rowN = seq + (int64_t)(reverse ? T_len - 1 - sc : sc) * rowstride + fo + 8 * c;
#pragma unroll
        for (int ks = 0; ks < KH; ++ks) gN[ks] = ld8(g + rowN + 32 * ks);
    };
    auto fetch_rest = [&]() {
#pragma unroll
        for (int ks = 0; ks < KH; ++ks) {
            qN[ks] = ld8(q + rowN + 32 * ks);
            kN[ks] = ld8(k + rowN + 32 * ks);
            dN[ks] = ld8(dout + rowN + 32 * ks);
        }
#pragma unroll
        for (int k2 = 0; k2 < KS; ++k2) vN[k2] = ld8(v + rowN - fo + 32 * k2);
    };
    // (all rows but the gates' are requested behind dv: ahead of dk they cost 25 more spilled registers and 75 us)
    fetch_g(N - 1);
    fetch_rest();

#pragma unroll 1
    for (int n = N - 1; n >= 0; --n) {
        const bool valid = validN;
        const int64_t row = rowN;            // element offset of the lane's first 8 features of its row
        // The tiles take more than the 64 KB that an access's own offset reaches: addresses are formed where they are used.
        // Left to themselves they are all formed ahead of the loop and spilled, and a reload waits for every row requested before it
        // (475 us against 247).
        asm volatile("" : "+v"(L.nat), "+v"(L.own), "+v"(L.k4), "+v"(L.k8), "+v"(ptl), "+v"(c8), "+v"(slot), "+v"(pub));
        const int wrow = 16 * J0 * LS + L.nat;
        float kt[8 * KH], sc[8 * KH];        // k e^{tau - l_i}; what the chain of dk is scaled by at its end
        D8 qf[KH], kf[KH], vf[KS];
        f32x4 Aown = {0.f, 0.f, 0.f, 0.f};   // this half's share of the scores A[i = 4c+e][j = r] of the own sub-block
        bool one_anchor;
        {
            if ((n + 1) * C > T_len && !valid) {   // only the last block can hold padded steps
                float z[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
#pragma unroll
                for (int ks = 0; ks < KH; ++ks) {
                    gN[ks] = pack8<float>(z);
                    qN[ks] = kN[ks] = dN[ks] = pack8<T>(z);
                }
#pragma unroll
                for (int k2 = 0; k2 < KS; ++k2) vN[k2] = pack8<T>(z);
            }
#pragma unroll
            for (int k2 = 0; k2 < KS; ++k2) vf[k2] = vN[k2];
            float p[8 * KH], sv[8 * KH];     // l_i; tau - l_i
            float *rt = rtab + J0 * D + fo + c8;
#pragma unroll
            for (int ks = 0; ks < KH; ++ks) {
                qf[ks] = qN[ks];
                kf[ks] = kN[ks];
                st8(tO + wrow + fo + 32 * ks, dN[ks]);
#pragma unroll
                for (int e = 0; e < 8; ++e) p[8 * ks + e] = prefix_sum_rows(gN[ks].v[e] * kLog2e);
                if (r == 15) st8(rt + 32 * ks, pack8<float>(p + 8 * ks));
            }
            asm volatile("" ::: "memory");
            float span = 0.f;
#pragma unroll
            for (int ks = 0; ks < KH; ++ks) {
                const f32x8 tau = ld8(rt + 32 * ks);
#pragma unroll
                for (int e = 0; e < 8; ++e) {
                    const int i = 8 * ks + e;
                    sv[i] = tau.v[e] - p[i];
                    span = fmaxf(span, fmaxf(fabsf(p[i]), fabsf(sv[i])));
                }
            }
            one_anchor = wave_all_below(span, kOneAnchorSpan);
            if (__builtin_expect(!one_anchor, false)) {
                // hard gates: l_i and tau - l_i from the sibling hierarchy (see sweep 1)
#pragma unroll
                for (int ks = 0; ks < KH; ++ks) {
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
                        p[8 * ks + e] = p8[e];
                        sv[8 * ks + e] = s8[e];
                    }
                }
            }
            float dot = 0.f;
            f32x4 G = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int ks = 0; ks < KH; ++ks) {
                float a[8], bq[8], kd[8], rw[8];
                unpack8(qf[ks], a);
                unpack8(kf[ks], bq);
#pragma unroll
                for (int e = 0; e < 8; ++e) {
                    const int i = 8 * ks + e;
                    dot += a[e] * bq[e];
                    a[e] *= fast_exp2(p[i]);
                    const float es = fast_exp2(sv[i]);
                    kt[i] = bq[e] * es;
                    rw[e] = fast_exp2(p[i] + sv[i]);
                    // One anchor: e^{tau - l} = e^{tau} e^{-l}, so that the own sub-block is one more link of the chain of
                    // dk, and its scores are (q e^{l}) (k e^{-l}).  Hard gates: e^{-l} may not exist.
                    sc[i] = one_anchor ? fast_exp2(-p[i]) : es;
                    kd[e] = bq[e] * sc[i];
                }
                D8 h8, l8, kh, kl;
                split8<T>(a, h8, l8);
                split8<T>(kd, kh, kl);
                st8(Qh + wrow + fo + 32 * ks, h8);
                st8(Ql + wrow + fo + 32 * ks, l8);
                G = mma_d_split(h8, l8, kh, kl, G);       // (not used with hard gates)
                asm volatile("" ::: "memory");
                if (r == 0) st8(rt + 32 * ks, pack8<float>(rw));
            }
            dot = reduce_over_cgroups(dot);
#pragma unroll
            for (int e = 0; e < 4; ++e)      // A_ii = q_i.k_i (gla.py:983)
                Aown[e] = (4 * c + e > r) ? G[e] : ((4 * c + e == r) ? dot : 0.f);
        }
        lds_barrier();                       // tiles of this block and the published dS' are in place
        if (__builtin_expect(!one_anchor, false)) {
            // Hard gates: the own sub-block's part of dk and its scores from the dyadic levels, inputs fetched again, here
            // where little is live across the call (see sweep 1).  dk's part waits in the wave's part of xch.
            f32x4 At = {0.f, 0.f, 0.f, 0.f}, An = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int k2 = 0; k2 < KS; ++k2) {
                const D8 o8 = ld8(tO + wrow + 32 * k2);
                At = mma_d(vf[k2], o8, At);
                An = mma_d(o8, vf[k2], An);
            }
            float diag = 0.f;
#pragma unroll
            for (int e = 0; e < 4; ++e) diag += (4 * c + e == r) ? At[e] : 0.f;
            diag = reduce_over_cgroups(diag);
            const float live = valid ? 1.f : 0.f;
            const f32x4 z4 = {0.f, 0.f, 0.f, 0.f};
            const HardSliceRev h0s = hard_slice_rev<XS, false>(g + row, q + row, k + row, live, diag, At, An, z4, z4, z4, z4, 0.f,
                                                               (LdsBT)xh, (LdsBT)xl, Lx.nat, Lx.k4, (LdsF32) nullptr,
                                                               (LdsBT) nullptr, (LdsBT) nullptr);
            const HardSliceRev h1s = hard_slice_rev<XS, false>(g + row + 32, q + row + 32, k + row + 32, live, diag, At, An,
                                                               h0s.G[0], h0s.G[1], h0s.G[2], h0s.G[3], h0s.dot, (LdsBT)xh,
                                                               (LdsBT)xl, Lx.nat, Lx.k4, (LdsF32) nullptr, (LdsBT) nullptr,
                                                               (LdsBT) nullptr);
            asm volatile("" ::: "memory");
#pragma unroll
            for (int tt = 0; tt < 2; ++tt) {
                mine(tt) = f32x4{h0s.dk8[4 * tt], h0s.dk8[4 * tt + 1], h0s.dk8[4 * tt + 2], h0s.dk8[4 * tt + 3]};
                mine(2 + tt) = f32x4{h1s.dk8[4 * tt], h1s.dk8[4 * tt + 1], h1s.dk8[4 * tt + 2], h1s.dk8[4 * tt + 3]};
            }
            const float dot = reduce_over_cgroups(h1s.dot);
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const int o = 4 * c + e;
                float acc = (o == r) ? dot : 0.f;
#pragma unroll
                for (int l = 0; l < 4; ++l) {
                    const int h_ = 1 << l;
                    const bool ok = ((o ^ r) < 2 * h_) && (o & h_) && !(r & h_);
                    acc += ok ? h1s.G[l][e] : 0.f;
                }
                Aown[e] = acc;
            }
        }
        const bool more = n > 0;
        if (more) fetch_g(n - 1);
        f32x8 qdq[KH];                       // q*dq of the rows (sweep 1 left it in the d(log_fgate) buffer)
#pragma unroll
        for (int ks = 0; ks < KH; ++ks) qdq[ks] = ld8(dg + row + 32 * ks);
        __builtin_amdgcn_sched_barrier(0);

        // ---- dA = dO V^T of the own and the later sub-blocks, [i = 4c+e][j = r]; this half's share of the scores ----
        T4 Ach[NB], Acl[NB], dAh[NB], dAl[NB];           // [0]: the own sub-block; [I]: the later ones
        D8 Kth[KH], Ktl[KH];                 // k e^{Lend - L_j}
        float dd = 0.f;
        {
            f32x4 dAn = {0.f, 0.f, 0.f, 0.f}, low;
#pragma unroll
            for (int k2 = 0; k2 < KS; ++k2) dAn = mma_d(ld8(tO + wrow + 32 * k2), vf[k2], dAn);
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                dd += (4 * c + e == r) ? dAn[e] : 0.f;
                low[e] = (4 * c + e > r) ? dAn[e] : 0.f;
            }
            dd = reduce_over_cgroups(dd);
            split4<T>(low, dAh[0], dAl[0]);
            split4<T>(Aown, Ach[0], Acl[0]);
        }
#pragma unroll
        for (int I = 1; I < NB; ++I) {
            Ach[I] = pack4<T>(f32x4{0.f, 0.f, 0.f, 0.f});
            Acl[I] = dAh[I] = dAl[I] = Ach[I];
            if (I > J0) {
                f32x4 as = {0.f, 0.f, 0.f, 0.f}, da = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
                for (int k2 = 0; k2 < KS; ++k2) da = mma_d(ld8(tO + L.nat + 16 * I * LS + 32 * k2), vf[k2], da);
#pragma unroll
                for (int ks = 0; ks < KH; ++ks) {
                    const int at = L.nat + 16 * I * LS + fo + 32 * ks;
                    D8 kh, kl;
                    split8<T>(kt + 8 * ks, kh, kl);
                    as = mma_d_split(ld8(Qh + at), ld8(Ql + at), kh, kl, as);
                    const f32x8 rr = ld8(rtab + I * D + fo + 32 * ks + c8);
#pragma unroll
                    for (int e = 0; e < 8; ++e) kt[8 * ks + e] *= rr.v[e];
                }
                split4<T>(as, Ach[I], Acl[I]);
                split4<T>(da, dAh[I], dAl[I]);
            }
        }
#pragma unroll
        for (int ks = 0; ks < KH; ++ks) split8<T>(kt + 8 * ks, Kth[ks], Ktl[ks]);
        __builtin_amdgcn_sched_barrier(0);

        // -- dk of the wave's features: dS' v first, then the later sub-blocks in descending order, then the own one
#pragma unroll
        for (int ks = 0; ks < KH; ++ks) {
            const int f = fo + 32 * ks;
            f32x4 acc[2] = {{0.f, 0.f, 0.f, 0.f}, {0.f, 0.f, 0.f, 0.f}};
            // (dS' v)[dk][j] = sum_dv dS'[dk][dv] v_j[dv]: 32 dv rows per step, read transposed, 16 per read.  Read
            // (k2, half) holds dv = 32 k2 + 8 c + 4 half + m, which is what lane (j, c) holds of v_j.
#pragma unroll
            for (int k2 = 0; k2 < KS; ++k2)
#pragma unroll
                for (int tt = 0; tt < 2; ++tt) {
                    acc[tt] = mma_d(lds_tr4x2(DTl + L.k8 + 32 * k2 * LS + f + 4 * tt, 4 * LS), vf[k2], acc[tt]);
                    acc[tt] = mma_d(lds_tr4x2(DTh + L.k8 + 32 * k2 * LS + f + 4 * tt, 4 * LS), vf[k2], acc[tt]);
                }
            auto link = [&](int I, T4 ah, T4 al) {
                const f32x8 rr = ld8(rtab + I * D + f + c8);
#pragma unroll
                for (int tt = 0; tt < 2; ++tt) {
#pragma unroll
                    for (int e = 0; e < 4; ++e) acc[tt][e] *= rr.v[4 * tt + e];
                    const int at = L.k4 + f + 4 * tt + 16 * I * LS;
                    acc[tt] = mma_t_split(lds_tr4(Qh + at, LS), lds_tr4(Ql + at, LS), ah, al, acc[tt]);
                }
            };
#pragma unroll
            for (int I = NB - 1; I >= 1; --I)
                if (I > J0) link(I, dAh[I], dAl[I]);
            float o[8], a[8], kk[8];
            unpack8(kf[ks], kk);
            if (__builtin_expect(one_anchor, true)) {
                link(J0, dAh[0], dAl[0]);
                unpack8(qf[ks], a);
#pragma unroll
                for (int e = 0; e < 8; ++e) o[e] = dd * a[e];                // diagonal term (gla.py:1181-1185)
            } else {
#pragma unroll
                for (int tt = 0; tt < 2; ++tt) {
                    const f32x4 t = mine(2 * ks + tt);
#pragma unroll
                    for (int e = 0; e < 4; ++e) o[4 * tt + e] = t[e];
                }
            }
#pragma unroll
            for (int e = 0; e < 8; ++e) {
                o[e] += sc[8 * ks + e] * acc[e >> 2][e & 3];
                // q*dq - k*dk of the row, then its reverse running sum inside the sub-block
                qdq[ks].v[e] = suffix_sum_rows((valid ? qdq[ks].v[e] : 0.f) - kk[e] * o[e]);
            }
            if constexpr (WIDE == 2) {
                const f32x8 t = ld8(dk1 + row + 32 * ks);
#pragma unroll
                for (int e = 0; e < 8; ++e) o[e] += t.v[e];
            }
            if (valid) st8(dk + row + 32 * ks, pack8<TG>(o));
            if (r == 0) st8(dltab + J0 * D + f + c8, qdq[ks]);
        }
        __builtin_amdgcn_sched_barrier(0);

        // -- this half's share of dv, all value features: dS'^T K~ first, then the own and the later sub-blocks
        f32x4 own[2 * KH];
        auto dv_slice = [&](int f, f32x4 &x0, f32x4 &x1) {
            f32x4 acc[2] = {{0.f, 0.f, 0.f, 0.f}, {0.f, 0.f, 0.f, 0.f}};
#pragma unroll
            for (int k2 = 0; k2 < KH; ++k2)
#pragma unroll
                for (int tt = 0; tt < 2; ++tt) {
                    const int at = L.own + (f + 4 * tt) * LS + fo + 32 * k2;
                    acc[tt] = mma_d_split(ld8(DTh + at), ld8(DTl + at), Kth[k2], Ktl[k2], acc[tt]);
                }
#pragma unroll
            for (int I = 0; I < NB; ++I) {
                if (I >= J0) {
                    const T4 bh4 = I == J0 ? Ach[0] : Ach[I], bl4 = I == J0 ? Acl[0] : Acl[I];
#pragma unroll
                    for (int tt = 0; tt < 2; ++tt) {
                        const T4 oa = lds_tr4(tO + L.k4 + f + 4 * tt + 16 * I * LS, LS);
                        acc[tt] = mma_t2(oa, oa, bl4, bh4, acc[tt]);
                    }
                }
            }
            x0 = acc[0];
            x1 = acc[1];
        };
#pragma unroll
        for (int ks = 0; ks < KH; ++ks) {
            f32x4 x0, x1;
            dv_slice(DH - fo + 32 * ks, x0, x1);
            mine(2 * ks) = x0;
            mine(2 * ks + 1) = x1;
        }
#pragma unroll
        for (int ks = 0; ks < KH; ++ks) dv_slice(fo + 32 * ks, own[2 * ks], own[2 * ks + 1]);

        __builtin_amdgcn_sched_barrier(0);
        if (more) fetch_rest();
        __builtin_amdgcn_sched_barrier(0);
        // ---- dS <- dS r_I + (q e^{l})_I^T dO_I over the sub-blocks, last first ---------------------------
#pragma unroll
        for (int I = NB - 1; I >= 0; --I) {
            T4 ob[NTW];
#pragma unroll
            for (int j = 0; j < NTW; ++j) ob[j] = lds_tr4(tO + ptl + 16 * I * LS + 16 * (nt0 + j), LS);
#pragma unroll
            for (int i = 0; i < RT; ++i) {
                const f32x4 rr = *reinterpret_cast<const f32x4 *>(rtab + I * D + 16 * (tk + i) + c8 / 2);
                const T4 qah = lds_tr4(Qh + ptl + 16 * I * LS + 16 * (tk + i), LS);
                const T4 qal = lds_tr4(Ql + ptl + 16 * I * LS + 16 * (tk + i), LS);
#pragma unroll
                for (int j = 0; j < NTW; ++j) {
#pragma unroll
                    for (int e = 0; e < 4; ++e) DS[i][j][e] *= rr[e];
                    DS[i][j] = mma_t2(qah, qal, ob[j], ob[j], DS[i][j]);
                }
            }
        }
        lds_barrier();                       // sub-block sums and dv's halves complete; every wave is done with the tiles
#pragma unroll
        for (int ks = 0; ks < KH; ++ks) {
            const int f = fo + 32 * ks + c8;
            float o[8];
#pragma unroll
            for (int tt = 0; tt < 2; ++tt) {
                const f32x4 t = theirs(2 * ks + tt);
#pragma unroll
                for (int e = 0; e < 4; ++e) o[4 * tt + e] = own[2 * ks + tt][e] + t[e];
            }
            if constexpr (WIDE == 2) {
                const f32x8 t = ld8(dv1 + row + 32 * ks);
#pragma unroll
                for (int e = 0; e < 8; ++e) o[e] += t.v[e];
            }
            if (valid) st8(dv + row + 32 * ks, pack8<TG>(o));
            f32x8 tot = ld8(runtab + (n & 1) * D + f);
#pragma unroll
            for (int e = 0; e < 8; ++e) qdq[ks].v[e] += tot.v[e];
#pragma unroll
            for (int m = 0; m < NB; ++m) {
                const f32x8 t = ld8(dltab + m * D + f);
#pragma unroll
                for (int e = 0; e < 8; ++e) {
                    qdq[ks].v[e] += m > J0 ? t.v[e] : 0.f;
                    tot.v[e] += t.v[e];
                }
            }
            if (J0 == 0 && r == 0) st8(runtab + ((n & 1) ^ 1) * D + f, tot);
            if constexpr (WIDE == 2) {
                const f32x8 t = ld8(dg1 + row + 32 * ks);
#pragma unroll
                for (int e = 0; e < 8; ++e) qdq[ks].v[e] += t.v[e];
                if (valid) st8(dg1 + row + 32 * ks, qdq[ks]);
            } else if (valid) {
                st8(dg + row + 32 * ks, qdq[ks]);
            }
        }
        publish();
    }

#pragma unroll
    for (int i = 0; i < RT; ++i)
#pragma unroll
        for (int j = 0; j < NTW; ++j) {
            float t4[4] = {DS[i][j][0], DS[i][j][1], DS[i][j][2], DS[i][j][3]};
            quad_transpose(t4);
            store_hidden<4>(dh0, hdt, hidden_at(i, j), t4);
        }
}

template <int C, int D, int WIDE>
static int launch_rev128(hipStream_t st, int B, Segments sg, int H, int reverse, int hdt, const float *g, const void *v,
                         const void *k, const void *q, const void *dhT, const void *dout, void *dh0, float *dg, void *dv,
                         void *dk, const float *dv1, const float *dk1, float *dg1)
{
    typedef BT T;
    typedef std::conditional_t<WIDE == 1, float, T> TG;
    constexpr int LS = TileGeom<T, D>::kStride, NB = C / 16;
    const size_t lds = (size_t)(3 * C + 2 * D) * LS * sizeof(T) + (size_t)2 * NB * (D / 32) * 64 * sizeof(f32x4) +
                       (size_t)(2 * NB + 2) * D * sizeof(float);
    auto kern = recurrent_stream_rev128_kernel<C, D, WIDE>;
    static LdsGrant grant;
    if (int e = allow_lds(grant, (const void *)kern, lds)) return e;
    dim3 grid(H, sg.S, B), block(C * 8);
    hipLaunchKernelGGL(kern, grid, block, lds, st, g, (const T *)v, (const T *)k, (const T *)q, dhT, (const T *)dout, dh0, dg,
                       (TG *)dv, (TG *)dk, sg, H, reverse, hdt, dv1, dk1, dg1);
    return launch_status();
}

int launch_recurrent_stream_rev128(hipStream_t st, int B, Segments sg, int H, int reverse, int hdt, const float *g,
                                   const void *v, const void *k, const void *q, const void *dhT, const void *dout, void *dh0,
                                   float *dg, void *dv, void *dk, int wide, const float *dv1,
                                   const float *dk1, float *dg1)
{
    auto run = wide == 2 ? launch_rev128<64, 128, 2> : wide ? launch_rev128<64, 128, 1> : launch_rev128<64, 128, 0>;
    return run(st, B, sg, H, reverse, hdt, g, v, k, q, dhT, dout, dh0, dg, dv, dk, dv1, dk1, dg1);
}

}  // namespace gla
