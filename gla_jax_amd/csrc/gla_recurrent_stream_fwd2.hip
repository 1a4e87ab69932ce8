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

// SECOND: the second pass of head dimension 256 (gla_split.hip): head h takes the value rows of head h ^ 1, and `out1`, what the
// first pass left there in fp32, is added before the one rounding.
template <typename TO, int C, int D, bool SECOND>
__global__ __launch_bounds__(C * 8) void recurrent_stream_fwd2_kernel(
    const void *__restrict__ h0, const float *__restrict__ g, const __bf16 *__restrict__ v,
    const __bf16 *__restrict__ k, const __bf16 *__restrict__ q, void *__restrict__ hT,
    TO *__restrict__ out, Segments sg, int H, int reverse, int hdt, const float *__restrict__ out1)
{
    typedef __bf16 T;
    constexpr int NB = C / 16, NW = 2 * NB, KS = D / 32, NT = D / 16;
    constexpr int DH = D / 2, KH = DH / 32, NV = DH / 4;             // a wave's key features
    constexpr int RT = NT / NB, NTW = NT / 2;                        // its state tiles: RT value tiles x NTW key tiles
    static_assert(NT % NB == 0 && DH % 32 == 0, "the state tiles split evenly over the waves");
    constexpr int LS = TileGeom<T, D>::kStride;
    typedef typename FragTypes<T>::d8 D8;
    typedef typename FragTypes<T>::t4 T4;
    extern __shared__ __align__(16) unsigned char smem[];
    T *Vn = reinterpret_cast<T *>(smem);           // [C][LS]  value
    T *Kh = Vn + C * LS;                           // [C][LS]  k * exp(tau_J - l_j)
    T *Kl = Kh + C * LS;                           // [C][LS]  what the bf16 rounding of Kh leaves over
    T *St = Kl + C * LS;                           // [D][LS]  state at the start of the block, [dv][dk]: bf16 head
    T *Sl = St + D * LS;                           // [D][LS]  ... and the bf16 of what the head leaves over
    float *rtab = reinterpret_cast<float *>(Sl + D * LS);            // [NB][D] exp(tau_m)
    f32x4 *xch = reinterpret_cast<f32x4 *>(rtab + NB * D);           // [NW][KS][64] the other half's value features

    const int lane = threadIdx.x & 63;
    const int W = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int I = W < NB ? W : NW - 1 - W;         // the wave's sub-block
    const int half = W < NB ? 0 : 1, fo = half * DH;   // ... and its first key feature; it stores the same value features
    const int r = lane & 15, c = lane >> 4;
    const SegmentRows seg(sg, blockIdx.z, blockIdx.y);
    const int T_len = seg.len;
    const int h = blockIdx.x;
    const int64_t seq = (seg.row0 * H + h) * D;      // element offset of (b, t = 0, h)
    const int64_t rowstride = (int64_t)H * D;
    if constexpr (SECOND) {
        const int other = ((h ^ 1) - h) * D;
        v += other;
        out += other;
        out1 += other;
    }
    const int64_t bh = (int64_t)seg.index * H + h;
    const TrLane<T> L = make_tr_lane<T>(LS);
    const int ptl = plain_tr_lane<T>(LS);
    const int wrow = 16 * I * LS + L.nat + fo;     // this lane's row of a [token][feature] tile, its half
    const int N = (T_len + C - 1) / C;
    const int wv = RT * (W % NB), nt0 = NTW * (W / NB);

    // state: S[i][j][e] = state[dk = 16(nt0 + j) + 4c + e][dv = 16(wv + i) + r]; accessed in memory by quads of lanes that
    // exchange (see recurrent_stream_fwd_kernel)
    f32x4 S[RT][NTW];
    auto state_at = [&](int i, int nt) {
        return bh * D * D + (int64_t)(16 * (nt0 + nt) + 4 * c + (r & 3)) * D + 16 * (wv + i) + (r & 12);
    };
#pragma unroll
    for (int i = 0; i < RT; ++i)
#pragma unroll
        for (int nt = 0; nt < NTW; ++nt) {
            float t4[4];
            load_hidden<4>(h0, hdt, state_at(i, nt), t4);
            quad_transpose(t4);
            S[i][nt] = f32x4{t4[0], t4[1], t4[2], t4[3]};
        }
    auto publish_state = [&]() {
#pragma unroll
        for (int i = 0; i < RT; ++i)
#pragma unroll
            for (int nt = 0; nt < NTW; ++nt) {
                T4 hi, lo;
                split4<T>(S[i][nt], hi, lo);
                const int off = (16 * (wv + i) + r) * LS + 16 * (nt0 + nt) + 4 * c;
                *reinterpret_cast<T4 *>(St + off) = hi;
                *reinterpret_cast<T4 *>(Sl + off) = lo;
            }
    };
    publish_state();

    // inputs of the wave's half of its 16 steps of a block, one block ahead
    f32x8 gN[KH];
    D8 qN[KH], kN[KH], vN[KH];
    bool validN;
    int64_t rowN;
    auto fetch = [&](int n) {
        const int s = n * C + 16 * I + r;                      // logical step
        validN = s < T_len;
        const int sc = validN ? s : T_len - 1;
        rowN = seq + (int64_t)(reverse ? T_len - 1 - sc : sc) * rowstride + fo;
#pragma unroll
        for (int ks = 0; ks < KH; ++ks) {
            gN[ks] = ld8(g + rowN + 32 * ks + 8 * c);
            kN[ks] = ld8(k + rowN + 32 * ks + 8 * c);
            qN[ks] = ld8(q + rowN + 32 * ks + 8 * c);
            vN[ks] = ld8(v + rowN + 32 * ks + 8 * c);
        }
    };
    fetch(0);

#pragma unroll 1
    for (int n = 0; n < N; ++n) {
        const bool valid = validN;
        const int64_t row = rowN;
        f32x4 accD = {0.f, 0.f, 0.f, 0.f};   // transposed scores of the own sub-block: [j = 4c+e][i = r]
        float qh[NV];                        // q * exp(l_i), walked down the earlier sub-blocks below
        {
            float p[NV];
            D8 qf[KH], kf[KH];
            if ((n + 1) * C > T_len && !valid) {   // only the last block can hold padded steps
                float z[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
#pragma unroll
                for (int ks = 0; ks < KH; ++ks) {
                    gN[ks] = pack8<float>(z);
                    qN[ks] = kN[ks] = vN[ks] = pack8<T>(z);
                }
            }
#pragma unroll
            for (int ks = 0; ks < KH; ++ks) {
#pragma unroll
                for (int e = 0; e < 8; ++e) p[8 * ks + e] = gN[ks].v[e] * kLog2e;
                qf[ks] = qN[ks];
                kf[ks] = kN[ks];
                st8(Vn + wrow + 32 * ks, vN[ks]);
            }
            subblock_forward<T, DH, true, false, true>(p, qf, kf, g + row, q + row, k + row, valid, rtab + I * D + fo, Kh + wrow, true,
                                          Kl + wrow, r, c, accD, qh);
        }
        lds_barrier();                       // tiles of this block and the published state are in place

        // ---- earlier sub-blocks J < I, walking the q side down; scores kept as packed MFMA operands ----
        // (operands and scores as bf16 head + remainder: the products keep 16 bits of mantissa)
        T4 sc[NB], sl[NB];
#pragma unroll
        for (int J = NB - 2; J >= 0; --J) {
            f32x4 a = {0.f, 0.f, 0.f, 0.f};
            if (J < I) {
#pragma unroll
                for (int ks = 0; ks < KH; ++ks) {
                    D8 qbh, qbl;
                    split8<T>(qh + 8 * ks, qbh, qbl);
                    const int at = L.nat + 16 * J * LS + fo + 32 * ks;
                    a = mma_d_split(ld8(Kh + at), ld8(Kl + at), qbh, qbl, a);
                    f32x8 rr = ld8(rtab + J * D + fo + 32 * ks + 8 * c);
#pragma unroll
                    for (int e = 0; e < 8; ++e) qh[8 * ks + e] *= rr.v[e];
                }
            }
            split4<T>(a, sc[J], sl[J]);
        }
        sc[NB - 1] = pack4<T>(f32x4{0.f, 0.f, 0.f, 0.f});
        sl[NB - 1] = sc[NB - 1];
        T4 scD, slD;
        split4<T>(accD, scD, slD);
        D8 qb[KH], ql[KH];                   // q * exp(L_i), operand of the state term: bf16 head and remainder
#pragma unroll
        for (int ks = 0; ks < KH; ++ks) split8<T>(qh + 8 * ks, qb[ks], ql[ks]);

        // ---- the wave's part of out^T[dv][i] in slices of 32 value features: state term, then the score blocks; the
        // partner's slices first
        auto slice = [&](int f, f32x4 (&acc)[2]) {
            acc[0] = acc[1] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int k2 = 0; k2 < KH; ++k2)
#pragma unroll
                for (int tt = 0; tt < 2; ++tt) {
                    const int at = L.own + (f + 4 * tt) * LS + fo + 32 * k2;
                    const D8 sh = ld8(St + at);
                    acc[tt] = mma_d(ld8(Sl + at), qb[k2], acc[tt]);
                    acc[tt] = mma_d(sh, ql[k2], acc[tt]);
                    acc[tt] = mma_d(sh, qb[k2], acc[tt]);
                }
#pragma unroll
            for (int J = 0; J < NB; ++J) {
                if (J <= I) {
                    const T4 b4 = J == I ? scD : sc[J], l4 = J == I ? slD : sl[J];
#pragma unroll
                    for (int tt = 0; tt < 2; ++tt) {
                        const T4 va = lds_tr4(Vn + L.k4 + f + 4 * tt + 16 * J * LS, LS);
                        acc[tt] = mma_t2(va, va, l4, b4, acc[tt]);
                    }
                }
            }
        };
#pragma unroll
        for (int ks = 0; ks < KH; ++ks) {
            f32x4 acc[2];
            slice(DH - fo + 32 * ks, acc);
#pragma unroll
            for (int tt = 0; tt < 2; ++tt) xch[(W * KS + 2 * ks + tt) * 64 + lane] = acc[tt];
        }
        f32x4 own[KH][2];
#pragma unroll
        for (int ks = 0; ks < KH; ++ks) slice(fo + 32 * ks, own[ks]);

        // The next block's rows are requested only here: the registers that receive them are not held through
        // the score and output phases above.
        if (n + 1 < N) fetch(n + 1);

        // ---- state update: S <- S e^{tau_J} + V_J^T (k e^{tau_J - l})_J over the sub-blocks in order ------
#pragma unroll
        for (int J = 0; J < NB; ++J) {
            T4 va[RT];
#pragma unroll
            for (int i = 0; i < RT; ++i) va[i] = lds_tr4(Vn + ptl + 16 * J * LS + 16 * (wv + i), LS);
#pragma unroll
            for (int nt = 0; nt < NTW; ++nt) {
                const f32x4 rr = *reinterpret_cast<const f32x4 *>(rtab + J * D + 16 * (nt0 + nt) + 4 * c);
                const T4 kl = lds_tr4(Kl + ptl + 16 * J * LS + 16 * (nt0 + nt), LS);
                const T4 kh = lds_tr4(Kh + ptl + 16 * J * LS + 16 * (nt0 + nt), LS);
#pragma unroll
                for (int i = 0; i < RT; ++i) {
                    S[i][nt] *= rr;
                    S[i][nt] = mma_t2(kl, kh, va[i], va[i], S[i][nt]);
                }
            }
        }
        lds_barrier();                       // the exchanged halves are in place; every wave is done with tiles and old state
#pragma unroll
        for (int ks = 0; ks < KH; ++ks) {
            float o[8];
#pragma unroll
            for (int tt = 0; tt < 2; ++tt) {
                const f32x4 other = xch[((NW - 1 - W) * KS + 2 * ks + tt) * 64 + lane];
#pragma unroll
                for (int e = 0; e < 4; ++e) o[4 * tt + e] = own[ks][tt][e] + other[e];
            }
            if constexpr (SECOND) {
                const f32x8 t = ld8(out1 + row + 32 * ks + 8 * c);
#pragma unroll
                for (int e = 0; e < 8; ++e) o[e] += t.v[e];
            }
            if (valid) st8(out + row + 32 * ks + 8 * c, pack8<TO>(o));
        }
        publish_state();
    }

#pragma unroll
    for (int i = 0; i < RT; ++i)
#pragma unroll
        for (int nt = 0; nt < NTW; ++nt) {
            float t4[4] = {S[i][nt][0], S[i][nt][1], S[i][nt][2], S[i][nt][3]};
            quad_transpose(t4);
            store_hidden<4>(hT, hdt, state_at(i, nt), t4);
        }
}

template <typename TO, bool SECOND>
static int launch_fwd2(hipStream_t st, int B, Segments sg, int H, int reverse, int hdt, const void *h0, const float *g,
                       const void *v, const void *k, const void *q, void *hT, void *out, const float *out1)
{
    typedef __bf16 T;
    constexpr int C = 64, D = 128, LS = TileGeom<T, D>::kStride;
    const size_t lds = (size_t)(3 * C + 2 * D) * LS * sizeof(T) + (size_t)(C / 16) * D * sizeof(float) +
                       (size_t)(C / 8) * (D / 32) * 64 * sizeof(f32x4);
    auto kern = recurrent_stream_fwd2_kernel<TO, C, D, SECOND>;
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
