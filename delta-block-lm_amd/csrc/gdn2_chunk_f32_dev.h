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
// A packed tile (the col or acc registers as one 16-byte piece per lane, 1 KiB) is
// read back the same way in one load, or across (fc_across) as a frag in four.
#pragma once

#include "gdn2_chunk_f32.h"
#include "gdn2_mfma.h"

namespace gdn2 {

namespace {

constexpr int C = FC_C;

template <int CTRL>
__device__ __forceinline__ float fc_dpp(float x) {
    return __builtin_bit_cast(
        float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, x), CTRL, 0xF, 0xF, true));
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
// x[0] = the sum of x[0] .. x[N - 1] (N a power of two), pairwise: each 16-channel
// tile's product first and the tiles in a tree, as a chain of 64 or 128 f32 additions
// has twice the error.
template <int N>
__device__ __forceinline__ void fc_tree(f32x4 (&x)[N]) {
#pragma unroll
    for (int w = 1; w < N; w *= 2)
#pragma unroll
        for (int i = 0; i < N; i += 2 * w) x[i] += x[i + w];
}
template <int N>
__device__ __forceinline__ f32x4 fc_mma_tree(const f32x4 (&a)[N], const f32x4 (&b)[N]) {
    f32x4 x[N];
#pragma unroll
    for (int i = 0; i < N; ++i) x[i] = fc_mma4(a[i], b[i], zero4());
    fc_tree(x);
    return x[0];
}
__device__ __forceinline__ f32x4 fc_rows(float x, int g) {  // rows 4 g + i of a per-token value (lane n: token n)
    return f32x4{__shfl(x, 4 * g), __shfl(x, 4 * g + 1), __shfl(x, 4 * g + 2), __shfl(x, 4 * g + 3)};
}
__device__ __forceinline__ bool fc_finite(const f32x4 &x) {  // every element (a sum that overflows counts as not)
    const float z = (x[0] + x[1]) + (x[2] + x[3]);
    return z - z == 0.f;
}
__device__ __forceinline__ f32x4 fc_keep(f32x4 x, bool on) { return on ? x : zero4(); }
__device__ __forceinline__ f32x4 fc_keep4(f32x4 x, const f32x4 &on) {
#pragma unroll
    for (int i = 0; i < 4; ++i) x[i] = on[i] != 0.f ? x[i] : 0.f;
    return x;
}
// Accesses at a 32-bit byte offset from a uniform base: one instruction, with the
// base in scalar registers.
__device__ __forceinline__ const float *fc_at(const float *p, uint32_t bytes) {
    return reinterpret_cast<const float *>(reinterpret_cast<const char *>(p) + bytes);
}
__device__ __forceinline__ float *fc_at(float *p, uint32_t bytes) {
    return reinterpret_cast<float *>(reinterpret_cast<char *>(p) + bytes);
}
__device__ __forceinline__ f32x4 fc_g4(const float *p, uint32_t bytes) {
    return *reinterpret_cast<const fc_u4 *>(fc_at(p, bytes));
}
__device__ __forceinline__ void fc_p4(float *p, uint32_t bytes, const f32x4 &x) {
    *reinterpret_cast<fc_u4 *>(fc_at(p, bytes)) = x;
}
// Byte offsets of this lane's col elements (rows 4 g + i, column n) in rows of ld
// floats.
struct FcOff {
    uint32_t o[4];
    __device__ __forceinline__ explicit FcOff(uint32_t ld) {
        const uint32_t l = lane_id(), g = l >> 4, n = l & 15;
        o[0] = (4 * g * ld + n) * 4;
#pragma unroll
        for (int i = 1; i < 4; ++i) o[i] = o[i - 1] + 4 * ld;
    }
    __device__ __forceinline__ f32x4 get(const float *p, int tile = 0) const {
        p += 16 * tile;
        return f32x4{*fc_at(p, o[0]), *fc_at(p, o[1]), *fc_at(p, o[2]), *fc_at(p, o[3])};
    }
    __device__ __forceinline__ void put(float *p, const f32x4 &x, int tile = 0) const {
#pragma unroll
        for (int i = 0; i < 4; ++i) *fc_at(p + 16 * tile, o[i]) = x[i];
    }
};

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
        // Loaded whether wanted or not (the sequence's last row, the last channel), so
        // that no load waits behind a branch.
        const int tt = min(t0 + t, T - 1), cc = min(ch, W - 1);
        const float x = BF ? ld4<bf16_t>(v, b, tt, h, cc) : ld4<float>(v, b, tt, h, cc);
        return t0 + t < T && ch < W ? x : 0.f;
    }
    __device__ __forceinline__ f32x4 frag(int tau) const {
        if (VEC) {
            const char *p = base + 16 * ES * tau;  // uniform
            if (BF) {
                const uint2 x = *reinterpret_cast<const uint2 *>(p + fo);
                return f32x4{__uint_as_float(x.x << 16), __uint_as_float(x.x & 0xffff0000u),
                             __uint_as_float(x.y << 16), __uint_as_float(x.y & 0xffff0000u)};
            }
            return *reinterpret_cast<const f32x4 *>(p + fo);
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
                const char *p = base + 16 * ES * tau;  // uniform
                const uint32_t o = (uint32_t)min(4 * g + q, last) * s1 + n * ES;
                x[q] = BF ? bf16_to_f32(*reinterpret_cast<const bf16_t *>(p + o))
                          : *reinterpret_cast<const float *>(p + o);
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
    if (VEC) {
        const int es = bf16 ? 2 : 4;
        char *p = static_cast<char *>(dst) + o0 * es;
        const uint32_t row = (uint32_t)(s.H * W) * es, o = 4 * g * row + ch * es;
        if (left >= C) {
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                if (bf16) *reinterpret_cast<bf16_t *>(p + (o + i * row)) = f32_to_bf16(x[i]);
                else *reinterpret_cast<float *>(p + (o + i * row)) = x[i];
            }
            return;
        }
    }
#pragma unroll
    for (int i = 0; i < 4; ++i)
        if (4 * g + i < left && ch < W) store_out(dst, bf16, o0 + (int64_t)(4 * g + i) * s.H * W + ch, x[i]);
}

// Token n's valid and reset flags (lane (g, n); the document limits in place of
// the masks when given).
__device__ __forceinline__ void fc_flags(const SeqArgs &s, int b, int c, bool &on, bool &rst) {
    // Both words are loaded without a branch (past the sequence, the last token's).
    const int tg = c * C + (lane_id() & 15), t = min(tg, s.T - 1);
    const View &v0 = s.doc ? s.doc_start : s.valid, &v1 = s.doc ? s.doc_end : s.reset;
    const int x0 = static_cast<const int *>(v0.data)[b * v0.s0 + t * v0.s1];
    const int x1 = static_cast<const int *>(v1.data)[b * v1.s0 + t * v1.s1];
    const bool live = s.doc ? x1 >= x0 : (x0 << 1) != 0;  // x1 >= x0; a nonzero float
    const bool cut = s.doc ? x0 == tg : (x1 << 1) != 0;
    on = (tg < s.T) & live;
    rst = on & cut;
}

// T = (I + A)^-1 for A strictly lower in acc layout; returns row n of T, columns
// 4 g + r (the A operand of T x, and one 16-byte piece of the row-major T).
// T (I + A) = I by rows: from the last column on, T_nq is final and leaves T_nj
// -= T_nq A_qj for j < q (entries above the diagonal stay zero).  A's rows come
// back from LDS (the wave's own 320 floats) as broadcast 16-byte reads.
constexpr int FC_LA = 20;  // row stride
__device__ __forceinline__ f32x4 fc_inverse(const f32x4 &A, float *la, int g, int n) {
#pragma unroll
    for (int i = 0; i < 4; ++i) la[(4 * g + i) * FC_LA + n] = A[i];
    __builtin_amdgcn_wave_barrier();
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");  // the wave's own rows have landed
    __builtin_amdgcn_wave_barrier();
    float x[C];
#pragma unroll
    for (int j = 0; j < C; ++j) x[j] = j == n ? 1.f : 0.f;
#pragma unroll
    for (int q = C - 1; q > 0; --q)
#pragma unroll
        for (int j4 = 0; j4 < q; j4 += 4) {
            const f32x4 r = *reinterpret_cast<const f32x4 *>(&la[q * FC_LA + j4]);
#pragma unroll
            for (int j = j4; j < j4 + 4 && j < q; ++j) x[j] -= x[q] * r[j - j4];
        }
    f32x4 t;
#pragma unroll
    for (int r = 0; r < 4; ++r) t[r] = g == 0 ? x[r] : (g == 1 ? x[4 + r] : (g == 2 ? x[8 + r] : x[12 + r]));
    return t;
}

// A packed tile read across: register i holds row n, column 4 g + i of a
// [token][channel] tile (a frag), or row n, column 4 g + i of a state tile (four
// one-word loads that together read the tile's 1 KiB once).
__device__ __forceinline__ f32x4 fc_across(const float *tile) {
    const uint32_t l = lane_id(), n = l & 15, o = ((n >> 2) * 64 + 16 * (l >> 4) + (n & 3)) * 4;
    return f32x4{*fc_at(tile, o), *fc_at(tile, o + 16), *fc_at(tile, o + 32), *fc_at(tile, o + 48)};
}
// Row r of a chunk's gb block (16 tokens): lane (g, n)'s token n, or its rows 4 g + i.
__device__ __forceinline__ float fc_gb(const FcArgs &a, int64_t ci, int r) {
    return *fc_at(a.gb + ci * C * 8 + C * r, 4 * (lane_id() & 15));
}
__device__ __forceinline__ f32x4 fc_gb4(const FcArgs &a, int64_t ci, int r) {
    return fc_g4(a.gb + ci * C * 8 + C * r, 16 * (lane_id() >> 4));
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
