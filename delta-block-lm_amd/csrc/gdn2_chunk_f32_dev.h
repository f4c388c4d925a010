// Device helpers of the f32 chunk kernels (gdn2_chunk_f32.hip, channel-wise
// gates, and gdn2_chunk_fs.hip, scalar gates): MFMA operand layouts, input reads
// and the per-chunk arrays.
//
// A 16-token chunk is one MFMA tile, and no product is transposed through LDS
// where an operand layout can be read instead.  With lane l = 16 g + n:
//   frag  x[token n][16 tau + 4 g + r]   (one 16-byte read)
//         A operand of x Y^T and B operand of Y x^T, reduction over channels
//   col   x[token 4 g + q][16 tau + n]
//         B operand of M x and A operand of x^T Y, reduction over tokens
//   acc   rows 4 g + i, column n (the accumulator); register i is also an A or B
//         operand whose reduction slice is {4 g + i}, so products chain in
//         registers, and a [token][channel] accumulator has the layout of a col
// A tile-packed state (a 16-byte piece per lane) is a B operand as it is loaded.
#pragma once

#include "gdn2_chunk_f32.h"
#include "gdn2_mfma.h"

namespace gdn2 {

namespace {

constexpr int C = FC_C;

template <int CTRL>
__device__ __forceinline__ float fc_dpp(float x) {
    return __builtin_bit_cast(
        float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, x), CTRL, 0xF, 0xF, false));
}
// Sum over the 16 lanes n of a lane group, in all of them.
__device__ __forceinline__ float fc_row_sum(float x) {
    x += fc_dpp<0xB1>(x);
    x += fc_dpp<0x4E>(x);
    x += fc_dpp<0x141>(x);
    return x + fc_dpp<0x140>(x);
}
// Sum over the four lane groups g, in all of them.
__device__ __forceinline__ float fc_group_sum(float x) {
    x += __shfl_xor(x, 16);
    return x + __shfl_xor(x, 32);
}
__device__ __forceinline__ float fc_lane(float x, int i) {
    return __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, x), i));
}
__device__ __forceinline__ f32x4 fc_mma(float a, float b, f32x4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
}
// a (frag or acc registers) times b, one 16-step reduction slice.
__device__ __forceinline__ f32x4 fc_mma4(const f32x4 &a, const f32x4 &b, f32x4 c) {
#pragma unroll
    for (int r = 0; r < 4; ++r) c = fc_mma(a[r], b[r], c);
    return c;
}
__device__ __forceinline__ f32x4 fc_rows(float x, int g) {  // rows 4 g + i of a per-token value (lane n: token n)
    return f32x4{__shfl(x, 4 * g), __shfl(x, 4 * g + 1), __shfl(x, 4 * g + 2), __shfl(x, 4 * g + 3)};
}
__device__ __forceinline__ f32x4 fc_keep(f32x4 x, bool on) { return on ? x : zero4(); }
__device__ __forceinline__ f32x4 fc_keep4(f32x4 x, const f32x4 &on) {
#pragma unroll
    for (int i = 0; i < 4; ++i) x[i] = on[i] != 0.f ? x[i] : 0.f;
    return x;
}
__device__ __forceinline__ f32x4 fc_g4(const float *p) { return *reinterpret_cast<const fc_u4 *>(p); }

// Reads of one chunk of a [token][channel] input, unmasked.  VEC (fc_vec_view on
// every input of the call): unit channel stride, a width of whole 16-channel
// tiles, aligned 4-channel pieces and byte offsets within a chunk that fit 32
// bits, so a read is one load from a uniform base; rows past the sequence read
// its last row.  Otherwise any element strides and widths, zero past either.
template <bool BF, bool VEC>
struct FcSrc {
    static constexpr int ES = BF ? 2 : 4;
    View v;
    const char *base;
    uint32_t fo, s1;
    int b, h, t0, T, W, last;
    __device__ __forceinline__ FcSrc(const View &view, int b_, int h_, int c, int T_, int W_)
        : v(view), b(b_), h(h_), t0(c * C), T(T_), W(W_) {
        const int l = lane_id();
        if (VEC) {
            base = static_cast<const char *>(v.data) + (b * v.s0 + t0 * v.s1 + h * v.s2) * ES;
            s1 = (uint32_t)v.s1 * ES;
            last = min(C - 1, T - 1 - t0);
            fo = (uint32_t)min(l & 15, last) * s1 + 4 * ES * (l >> 4);
        }
    }
    __device__ __forceinline__ float at(int t, int ch) const {
        if (t0 + t >= T || ch >= W) return 0.f;
        return BF ? ld4<bf16_t>(v, b, t0 + t, h, ch) : ld4<float>(v, b, t0 + t, h, ch);
    }
    __device__ __forceinline__ f32x4 frag(int tau) const {
        if (VEC) {
            const char *p = base + fo + 16 * ES * tau;
            if (BF) {
                const uint2 x = *reinterpret_cast<const uint2 *>(p);
                return f32x4{__uint_as_float(x.x << 16), __uint_as_float(x.x & 0xffff0000u),
                             __uint_as_float(x.y << 16), __uint_as_float(x.y & 0xffff0000u)};
            }
            return *reinterpret_cast<const f32x4 *>(p);
        }
        const int l = lane_id();
        f32x4 x;
#pragma unroll
        for (int r = 0; r < 4; ++r) x[r] = at(l & 15, 16 * tau + 4 * (l >> 4) + r);
        return x;
    }
    __device__ __forceinline__ f32x4 col(int tau) const {
        const int l = lane_id(), g = l >> 4, n = l & 15;
        f32x4 x;
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            if (VEC) {
                const char *p = base + ((uint32_t)min(4 * g + q, last) * s1 + n * ES) + 16 * ES * tau;
                x[q] = BF ? bf16_to_f32(*reinterpret_cast<const bf16_t *>(p)) : *reinterpret_cast<const float *>(p);
            } else {
                x[q] = at(4 * g + q, 16 * tau + n);
            }
        }
        return x;
    }
};

// A chunk's [token 4 g + i][16 tile + n] tile of a dense [B][T][H][W] output.
template <bool BF, bool VEC>
__device__ __forceinline__ void fc_put(void *dst, int bf16, const SeqArgs &s, int b, int h, int c, int W, int tile,
                                       const f32x4 &x) {
    const int l = lane_id(), g = l >> 4, ch = 16 * tile + (l & 15);
    const int64_t o0 = (((int64_t)b * s.T + c * C) * s.H + h) * W;
    const int left = s.T - c * C;
#pragma unroll
    for (int i = 0; i < 4; ++i)
        if (4 * g + i < left && (VEC || ch < W)) {
            if (VEC) {
                const uint32_t o = (uint32_t)(4 * g + i) * (uint32_t)(s.H * W) + ch;
                if (bf16) *reinterpret_cast<bf16_t *>(static_cast<char *>(dst) + o0 * 2 + o * 2u) = f32_to_bf16(x[i]);
                else *reinterpret_cast<float *>(static_cast<char *>(dst) + o0 * 4 + o * 4u) = x[i];
            } else {
                store_out(dst, bf16, o0 + (int64_t)(4 * g + i) * s.H * W + ch, x[i]);
            }
        }
}

// Token n's valid and reset flags (lane (g, n); the document limits in place of
// the masks when given).
__device__ __forceinline__ void fc_flags(const SeqArgs &s, int b, int c, bool &on, bool &rst) {
    const int tg = c * C + (lane_id() & 15);
    on = rst = false;
    if (tg < s.T) {
        if (s.doc) {
            const int st = static_cast<const int *>(s.doc_start.data)[b * s.doc_start.s0 + tg * s.doc_start.s1];
            const int en = static_cast<const int *>(s.doc_end.data)[b * s.doc_end.s0 + tg * s.doc_end.s1];
            on = en >= st;
            rst = on && st == tg;
        } else {
            on = ld4<float>(s.valid, b, tg, 0, 0) != 0.f;
            rst = on && ld4<float>(s.reset, b, tg, 0, 0) != 0.f;
        }
    }
}

// T = (I + A)^-1 for A strictly lower in acc layout; returns row n of T, columns
// 4 g + r (the A operand of T x, and one 16-byte piece of the row-major T).
// T (I + A) = I by rows: from the last column on, T_nq is final and leaves T_nj
// -= T_nq A_qj for j < q (entries above the diagonal stay zero).
__device__ __forceinline__ f32x4 fc_inverse(const f32x4 &A, int g, int n) {
    float x[C];
#pragma unroll
    for (int j = 0; j < C; ++j) x[j] = j == n ? 1.f : 0.f;
#pragma unroll
    for (int q = C - 1; q > 0; --q)
#pragma unroll
        for (int j = 0; j < q; ++j) x[j] -= x[q] * fc_lane(A[q & 3], 16 * (q >> 2) + j);
    f32x4 t;
#pragma unroll
    for (int r = 0; r < 4; ++r) t[r] = g == 0 ? x[r] : (g == 1 ? x[4 + r] : (g == 2 ? x[8 + r] : x[12 + r]));
    return t;
}

// The map's factors from T (fc_inverse): W' tile tau from the col tile b . e . k,
// U tile vt from the col tile w . v, and the 16 x 16 array tm.
__device__ __forceinline__ void fc_put_w(const FcArgs &a, int64_t ci, int KP, int tau, const f32x4 &t, const f32x4 &x,
                                         int g, int n) {
    const f32x4 w = fc_mma4(t, x, zero4());
    float *p = a.fw + ci * C * KP;
#pragma unroll
    for (int i = 0; i < 4; ++i) p[(4 * g + i) * KP + 16 * tau + n] = w[i];
}
__device__ __forceinline__ void fc_put_u(const FcArgs &a, int64_t ci, int VT, int vt, const f32x4 &t, const f32x4 &x) {
    *reinterpret_cast<fc_u4 *>(a.fu + (ci * VT + vt) * 256 + 4 * lane_id()) = fc_mma4(t, x, zero4());
}
__device__ __forceinline__ void fc_put_rows(float *p, const f32x4 &x, int g, int n) {  // acc -> [16][16]
#pragma unroll
    for (int i = 0; i < 4; ++i) p[(4 * g + i) * C + n] = x[i];
}
__device__ __forceinline__ f32x4 fc_get_rows(const float *p, int g, int n) {  // [16][16] -> acc
    return f32x4{p[(4 * g) * C + n], p[(4 * g + 1) * C + n], p[(4 * g + 2) * C + n], p[(4 * g + 3) * C + n]};
}
__device__ __forceinline__ f32x4 fc_get_col(const float *p, int KP, int tau, int g, int n) {  // [16][KP] -> col
    const float *x = p + 16 * tau + n;
    return f32x4{x[(4 * g) * KP], x[(4 * g + 1) * KP], x[(4 * g + 2) * KP], x[(4 * g + 3) * KP]};
}
// Key tile tau of a tile-packed state across the stored tiles of value tile vt:
// register i holds row 16 tau + n, column 16 vt + 4 g + i (four one-word loads
// that together read the tile's 1 KiB once).
__device__ __forceinline__ f32x4 fc_get_across(const float *st, int KT, int tau, int vt, int g, int n) {
    const float *p = st + (vt * KT + tau) * 256 + (n >> 2) * 64 + 16 * g + (n & 3);
    return f32x4{p[0], p[4], p[8], p[12]};
}

// Score adjoint coefficients of token n: cs = dscore |k| / |delta|, ck = dscore
// |delta| / |k| (zero at a zero edit or key).
__device__ void fc_score_adj(const FcArgs &a, int64_t ci, int b, int h, int c, int VT, bool on, float ksq, float &cs,
                             float &ck) {
    const SeqArgs &s = a.s;
    const int l = lane_id(), n = l & 15, tg = c * C + n;
    f32x4 d2 = zero4();
    for (int vt = 0; vt < VT; ++vt) {
        const f32x4 d = fc_g4(a.fu + (ci * VT + vt) * 256 + 4 * l);
        d2 += d * d;
    }
    float dsq = 0.f;  // token n's sum sits in group n / 4, register n % 4
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const float x = __shfl(fc_row_sum(d2[i]), 16 * (n >> 2));
        if ((n & 3) == i) dsq = x;
    }
    const float nk = sqrtf(ksq), nd = sqrtf(dsq);
    const float dsc = tg < s.T ? s.dscores[((int64_t)b * s.T + tg) * s.H + h] : 0.f;
    const bool ok = on && nk > 0.f && nd > 0.f;
    cs = ok ? dsc * nk / nd : 0.f;
    ck = ok ? dsc * nd / nk : 0.f;
}

inline void fc_mark(const hipEvent_t *ev, int i, hipStream_t stream) {
    if (ev) (void)hipEventRecord(ev[i], stream);
}

}  // namespace

// FC_DISPATCH(tiles, F, ...) calls F<KM, in_bf16, vec>(...) for the argument block
// a, with KM = 2, 4 or 8 tiles of 16 channels, the smallest that holds `tiles`.
#define FC_FORMS(KM, F, ...)                                                    \
    do {                                                                        \
        if (a.in_bf16 && a.vec) F<KM, true, true>(__VA_ARGS__);                 \
        else if (a.in_bf16) F<KM, true, false>(__VA_ARGS__);                    \
        else if (a.vec) F<KM, false, true>(__VA_ARGS__);                        \
        else F<KM, false, false>(__VA_ARGS__);                                  \
    } while (0)
#define FC_DISPATCH(tiles, F, ...)                                              \
    do {                                                                        \
        if ((tiles) <= 2) FC_FORMS(2, F, __VA_ARGS__);                          \
        else if ((tiles) <= 4) FC_FORMS(4, F, __VA_ARGS__);                     \
        else FC_FORMS(8, F, __VA_ARGS__);                                       \
    } while (0)

}  // namespace gdn2
