// Launchers of the matrix-core recurrent_gla kernels (bf16 inputs, head dimension 64 or 128).  `hdt` is the
// gla_dtype of the state arrays (h0, hT, dhT, dh0).
#pragma once

#include "gla_common.hpp"

namespace gla {

// A launch covers every sequence of T rows as S segments of L rows, the last one shorter where they do not divide T
// (a whole sequence: S = 1, L = T).  The grid is (heads, segments, batch entries); state arrays are indexed by segment,
// [B][S][H][D][D].
struct Segments {
    int T, S, L;
};
struct SegmentRows {
    int64_t row0;      // the segment's first row in a [B,T,...] array
    int len;           // its rows
    int index;         // which of the B * S segments it is
    __device__ __forceinline__ SegmentRows(const Segments &sg, int b, int p)
    {
        const int left = sg.T - p * sg.L;
        row0 = (int64_t)b * sg.T + p * sg.L;
        len = left < sg.L ? left : sg.L;
        index = b * sg.S + p;
    }
};

// TO = element type of `out` (__bf16, or float for the recurrent_gla_naive flavour).
template <typename TO>
int launch_recurrent_stream_fwd(hipStream_t st, int B, Segments sg, int H, int D, int reverse, int hdt,
                                const void *h0, const float *g, const void *v, const void *k, const void *q,
                                void *hT, void *out);

// The same with two waves per sub-block (head dimension 128).  out1 given: the second pass of head dimension 256, head h takes
// the rows of head h ^ 1 of v, out and out1, and out1, the first pass's fp32 `out`, is added to `out`.
template <typename TO>
int launch_recurrent_stream_fwd2(hipStream_t st, int B, Segments sg, int H, int reverse, int hdt, const void *h0,
                                 const float *g, const void *v, const void *k, const void *q, void *hT, void *out,
                                 const float *out1 = nullptr);

// The forward in fp32 vector arithmetic (gla_recurrent_steps.hip): any element types and head dimension.
// h0 may be null: the states start from zeros.
template <typename T, typename TO>
int launch_recurrent_steps(hipStream_t st, int B, Segments sg, int H, int D, int reverse, int hdt, const void *h0,
                           const float *g, const void *v, const void *k, const void *q, void *hT, void *out);

// The forward without its outputs: hidden_final alone (what a segment contributes to the state that leaves it).
// h0 may be null: the state starts from zeros.  g_shift = +1 or -1: every step takes the gate of the next (previous)
// row of the array instead of its own (the recurrence of the state's cotangent, where the decay between two steps
// belongs to the later one); the first step of a sequence, whose gate scales the initial state, may get any row's.
// gate_sums (may be null; not with g_shift): [B][H][D] floats, the sum of every segment's gates.
// other_half != 0: head h takes the rows of head h ^ 1 of v (the second pass of head dimension 256).
int launch_recurrent_stream_state(hipStream_t st, int B, Segments sg, int H, int D, int reverse, int hdt, const void *h0,
                                 const float *g, const void *v, const void *k, const void *q, void *hT,
                                 int g_shift = 0, float *gate_sums = nullptr, int other_half = 0);

// Sweep 1 of the backward: dq, and q*dq in fp32 into `qdq` (the last step's carries sum_v dhT * (final state)
// on top).  dout_f32 != 0: `dout` is float (the recurrent_gla_naive flavour), else bf16.  wide != 0 (head dimension
// 128 only): `dq` is a float array, for the two passes that make up head dimension 256.
int launch_recurrent_stream_dq(hipStream_t st, int B, Segments sg, int H, int D, int reverse, int hdt, int dout_f32,
                               const void *h0, const float *g, const void *v, const void *k, const void *q,
                               const void *dhT, const void *dout, void *dq, float *qdq, int wide = 0);

// The same sweep with two waves per sub-block (head dimension 64).
int launch_recurrent_stream_dq2(hipStream_t st, int B, Segments sg, int H, int D, int reverse, int hdt, int dout_f32,
                                const void *h0, const float *g, const void *v, const void *k, const void *q,
                                const void *dhT, const void *dout, void *dq, float *qdq);

// The same sweep with two waves per sub-block (head dimension 128, `dout` in bf16).  wide = 2: the second pass of head dimension
// 256, head h takes the rows of head h ^ 1 of v and dout, and dq1, the first pass's float dq, is added to dq (in bf16; `qdq`
// is the second pass's own).
int launch_recurrent_stream_dq128(hipStream_t st, int B, Segments sg, int H, int reverse, int hdt, const void *h0,
                                  const float *g, const void *v, const void *k, const void *q, const void *dhT,
                                  const void *dout, void *dq, float *qdq, int wide, const float *dq1 = nullptr);

// Sweep 2: dk, dv, dh0 and dlog_fgate (`dg` holds sweep 1's q*dq on entry).  wide != 0 (head dimension 128 only):
// `dv` and `dk` are float arrays.
int launch_recurrent_stream_rev(hipStream_t st, int B, Segments sg, int H, int D, int reverse, int hdt, int dout_f32,
                                const float *g, const void *v, const void *k, const void *q, const void *dhT,
                                const void *dout, void *dh0, float *dg, void *dv, void *dk, int wide = 0);

// The same sweep with two waves per sub-block (head dimension 128, `dout` in bf16).  wide = 2 as above, with dv, dv1, dk, dk1; the
// gates' gradient is added to what dg1 holds.
int launch_recurrent_stream_rev128(hipStream_t st, int B, Segments sg, int H, int reverse, int hdt, const float *g,
                                   const void *v, const void *k, const void *q, const void *dhT, const void *dout, void *dh0,
                                   float *dg, void *dv, void *dk, int wide, const float *dv1 = nullptr,
                                   const float *dk1 = nullptr, float *dg1 = nullptr);

// The same sweep with two waves per sub-block (head dimension 64).
int launch_recurrent_stream_rev2(hipStream_t st, int B, Segments sg, int H, int D, int reverse, int hdt, int dout_f32,
                                 const float *g, const void *v, const void *k, const void *q, const void *dhT,
                                 const void *dout, void *dh0, float *dg, void *dv, void *dk);

}  // namespace gla
