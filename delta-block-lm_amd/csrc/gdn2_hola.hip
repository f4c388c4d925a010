// HOLA exact-memory cache read on gfx950: the downstream consumer of the GDN-2
// scores.  After every chunk of `chunk` tokens each (batch, head) keeps the
// `capacity` highest-scoring valid tokens of the document of the chunk's last
// physical slot (ties: earlier position); each valid query attends with
// softmax to the previous chunk's cache plus the causal tokens of its own
// chunk in its document, next to a learned zero-value sink logit.
//
// Semantics: crates/kernels/src/hola.rs (selection_kernel, forward_kernel,
// query/key VJPs) and the scalar oracle of crates/mixers/src/hola_checks.rs.
//
// Layout and work split:
//   * schedule: two waves per (batch, head), chunks in order; one ranks a chunk's
//     eligible tokens, one chunk ahead, the other keeps the cache sorted and merges
//     them into it; it writes the cache positions before/after every chunk and the
//     end of each key's visibility ("expiry");
//   * read, query VJP: one wave per (batch, head, chunk); the rows of the chunk's
//     slots (cache positions from the schedule + the chunk's own tokens) go from
//     memory into MFMA operands, and each query's softmax over <= 80 slots stays
//     in the registers of four lanes;
//   * key VJP: four waves per (batch, head, chunk) of keys.  A selected key stays
//     in the cache without interruption until it is evicted, so its visible
//     queries are the chunks from its own up to its expiry; the waves walk them
//     with a slot map per chunk and accumulate dk, dv in registers from the
//     (probability, logit gradient) pairs the query VJP saved.  No atomics.
//   * sink gradient: a fixed-order sum over tokens per head.
#include <float.h>
#include <math.h>

#include <algorithm>
#include <initializer_list>
#include <utility>

#include "gdn2_common.h"
#include "gdn2_mfma.h"
#include "gdn2_status.h"

namespace gdn2 {
namespace {

constexpr int kMaxCapacity = 64;
constexpr int kMaxChunk = 16;
constexpr int kMaxSlots = kMaxCapacity + kMaxChunk;
constexpr int kMaxWidth = 128;

struct HolaArgs {
    int B, T, H, dk, dv, cap, chunk, nc, recency;
    float scale;
    View q, k, v, scores, valid, docs, sink, dout;
    float *schedule;         // [B*H][nc + 1][cap]
    float *expiry;           // [B*T*H]
    float *stats;            // [B*T*H][2]: softmax max, 1 / denominator
    float *out;              // [B*T*H][dv]
    const float *fwd_out;    // the forward output (backward)
    float *pairs;            // [B*T*H][cap + chunk][2]: probability, logit gradient
    float *aux;              // [B*T*H][2]: dO . o, sink gradient term
    float *gq, *gk, *gv, *gsink;  // dq, dk, dv, dsink
    float *final_positions;  // [B*H][cap] or null
};

__device__ __forceinline__ float ldf(const View &v, int64_t i0, int64_t i1 = 0, int64_t i2 = 0,
                                     int64_t i3 = 0) {
    return reinterpret_cast<const float *>(v.data)[i0 * v.s0 + i1 * v.s1 + i2 * v.s2 + i3 * v.s3];
}

template <int CTRL>
__device__ __forceinline__ float dpp_f(float v) {
    return __builtin_bit_cast(
        float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), CTRL, 0xF, 0xF, false));
}

__device__ __forceinline__ float readlane_f(float v, int lane) {
    return __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, v), lane));
}

__device__ __forceinline__ float wave_sum(float x) {
    x += dpp_f<0xB1>(x);
    x += dpp_f<0x4E>(x);
    x += dpp_f<0x141>(x);
    x += dpp_f<0x140>(x);
    return ((readlane_f(x, 0) + readlane_f(x, 16)) + readlane_f(x, 32)) + readlane_f(x, 48);
}

__device__ __forceinline__ float wave_max(float x) {
    x = fmaxf(x, dpp_f<0xB1>(x));
    x = fmaxf(x, dpp_f<0x4E>(x));
    x = fmaxf(x, dpp_f<0x141>(x));
    x = fmaxf(x, dpp_f<0x140>(x));
    return fmaxf(fmaxf(readlane_f(x, 0), readlane_f(x, 16)),
                 fmaxf(readlane_f(x, 32), readlane_f(x, 48)));
}

__device__ __forceinline__ int64_t token(const HolaArgs &a, int b, int t, int h) {
    return ((int64_t)b * a.T + t) * a.H + h;
}

// Orders a wave's own LDS traffic: what any lane wrote before is read after.
__device__ __forceinline__ void wave_fence() {
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
}

// ---- schedule ---------------------------------------------------------------------

__device__ __forceinline__ uint64_t lane_u64(uint64_t x, int lane) {
    const uint32_t lo = (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)x, lane);
    const uint32_t hi = (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)(x >> 32), lane);
    return ((uint64_t)hi << 32) | lo;
}

// One workgroup per (batch, head), chunks in order: a serial chain, bound by the
// instructions and LDS round trips of one chunk.  Wave 1 prepares chunks one ahead of
// the chain: it loads their token words (valid, document, score; kAhead chunks
// early) and leaves the eligible tokens in rank order.  Wave 0 holds the cache in
// registers, lane r the entry of rank r, so the cache is sorted at all times: an
// entry's new rank is the eligible entries before it plus the tokens that beat it,
// and the tokens fill the free ranks in their order.  128 (batch, head) pairs, 32
// chunks of 16, 64 entries: 23 us, against 62 where one wave compared every pair
// of the 80 candidates through LDS.
__global__ void __launch_bounds__(128) hola_schedule_kernel(HolaArgs a) {
    constexpr int kAhead = 4;
    // A chunk's tokens in rank order: ranking word (0 past them); position, word, document.
    __shared__ __align__(16) uint32_t word[2][kMaxChunk];
    __shared__ __align__(16) float4 tok[2][kMaxChunk];
    __shared__ float2 about[2];  // tokens, eligible document
    __shared__ __align__(16) float4 place[kMaxCapacity];  // position, ranking word, document
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int bh = blockIdx.x, b = bh / a.H, h = bh % a.H;
    float *sched = a.schedule + (int64_t)bh * (a.nc + 1) * a.cap;
    float *expiry = a.expiry ? a.expiry + (int64_t)b * a.T * a.H + h : nullptr;
    float cpos = -1.f, cdoc = 0.f;
    uint32_t cord = 0;
    if (wave == 0 && lane < a.cap) sched[lane] = -1.f;
    // Token words of a chunk: lane j < chunk holds token first + j.
    struct Words {
        float valid, doc, score;
    };
    auto fetch = [&](int c) {
        Words w{0.f, 0.f, 0.f};
        const int t = c * a.chunk + lane;
        if (lane < a.chunk && t < a.T) {
            w.valid = ldf(a.valid, b, t);
            w.doc = ldf(a.docs, b, t);
            if (!a.recency) w.score = ldf(a.scores, b, t, h);
        }
        return w;
    };
    auto prepare = [&](int c, const Words &w) {
        const int first = c * a.chunk, n = min(a.chunk, a.T - first), buf = c & 1;
        // Only the document of the chunk's last PHYSICAL slot, padding included,
        // is eligible.
        const float last_doc = readlane_f(w.doc, n - 1);
        // Ranking keys: the order-preserving bits of the score (or position)
        // above the complemented position, so "beats" (higher key, ties to the
        // earlier position) is one unsigned compare; ineligible tokens get key 0
        // and never beat.
        const float pos = (float)(first + lane);
        const bool on = lane < n && w.valid >= 0.5f && w.doc == last_doc;
        const uint32_t u = __float_as_uint(a.recency ? pos : w.score);
        const uint32_t ord = (u & 0x80000000u) ? ~u : (u | 0x80000000u);
        const uint64_t key =
            on ? ((uint64_t)ord << 32) | (uint64_t)(0xFFFFFFFFu - (uint32_t)(first + lane)) : 0;
        int rank = 0;
#pragma unroll
        for (int j = 0; j < kMaxChunk; ++j) rank += lane_u64(key, j) > key;
        const int count = __popcll(__ballot(on));
        if (lane < kMaxChunk) word[buf][lane] = 0;
        wave_fence();
        if (on) {
            word[buf][rank] = ord;
            tok[buf][rank] = make_float4(pos, __uint_as_float(ord), w.doc, 0.f);
        }
        if (lane == 0) about[buf] = make_float2((float)count, last_doc);
    };
    auto merge = [&](int c) {
        const int first = c * a.chunk, n = min(a.chunk, a.T - first), end = first + n, buf = c & 1;
        const float2 ab = about[buf];
        const int count = (int)ab.x;
        if (lane < n && expiry) expiry[(int64_t)(first + lane) * a.H] = (float)end;
        const bool on = cpos >= 0.f && cdoc == ab.y;
        const uint64_t below = (1ull << lane) - 1;
        int rank = __popcll(__ballot(on) & below);
#pragma unroll
        for (int j = 0; j < kMaxChunk; j += 4) {
            const uint4 o = *reinterpret_cast<const uint4 *>(&word[buf][j]);
            // Ties go to the earlier position, the cache's.
            rank += (int)(o.x > cord) + (int)(o.y > cord) + (int)(o.z > cord) + (int)(o.w > cord);
        }
        place[lane] = make_float4(-1.f, 0.f, 0.f, 0.f);
        wave_fence();
        if (on && rank < a.cap) place[rank] = make_float4(cpos, __uint_as_float(cord), cdoc, 0.f);
        wave_fence();
        float4 e = place[lane];
        const uint64_t used = __ballot(e.x >= 0.f);
        const int next = __popcll(~used & below);
        const float4 t = tok[buf][min(next, kMaxChunk - 1)];
        const bool take = e.x < 0.f && next < count && lane < a.cap;
        cpos = take ? t.x : e.x;
        cord = __float_as_uint(take ? t.y : e.y);
        cdoc = take ? t.z : e.z;
        wave_fence();
        if (lane < a.cap) {
            sched += a.cap;
            sched[lane] = cpos;
            if (cpos >= 0.f && expiry)
                expiry[(int64_t)(int)cpos * a.H] = (float)min(end + a.chunk, a.T);
        }
    };
    Words ring[kAhead];
    if (wave == 1) {
#pragma unroll
        for (int u = 0; u < kAhead; ++u) ring[u] = fetch(u);
    }
    for (int c0 = 0; c0 <= a.nc; c0 += kAhead) {
#pragma unroll
        for (int u = 0; u < kAhead; ++u) {
            const int c = c0 + u;
            if (c > a.nc) continue;
            if (wave == 1) {
                if (c < a.nc) prepare(c, ring[u]);
                ring[u] = fetch(c + kAhead);
            } else if (c > 0) {
                merge(c - 1);
            }
            __syncthreads();
        }
    }
    if (wave == 0 && a.final_positions && lane < a.cap)
        a.final_positions[(int64_t)bh * a.cap + lane] = cpos;
}

// ---- rows and products ------------------------------------------------------------
//
// Every product of the read and its VJP runs on v_mfma_f32_16x16x4f32 with both
// operands in registers: lane 16 g + n gives row (column) n at the reduction
// index of group g, and holds rows 4 g + i of column n of the result.  Slots (or
// keys) and queries are the rows and columns, so a result's registers are at
// once the operand of the next product over the slots (its reduction index
// 4 g + i), and no tile goes through LDS.  Rows come straight from memory: they
// are gathered in 64- to 256-byte pieces, and each is used by one wave only.

constexpr int kSlotTiles = kMaxSlots / 16;
typedef float hola_f4 __attribute__((ext_vector_type(4), aligned(4)));
typedef float hola_f2 __attribute__((ext_vector_type(2), aligned(4)));

__device__ __forceinline__ f32x4 mma(float x, float y, f32x4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x4f32(x, y, c, 0, 0, 0);
}

__device__ __forceinline__ float group_sum(float x) {  // over the four lane groups
    x += __shfl_xor(x, 16);
    return x + __shfl_xor(x, 32);
}

// Row t (its first row where t < 0: the caller drops it) of a view.
__device__ __forceinline__ const float *row_of(const View &x, int b, int t, int h) {
    return reinterpret_cast<const float *>(x.data) + b * x.s0 + max(t, 0) * x.s1 + h * x.s2;
}

// Channels i .. i + E - 1 of a row of width w, and the same with the channels past the
// width (and rows that are off) cleared; two steps, so that the loads of a whole
// set of rows are in flight before any is looked at.  VEC: unit channel stride and
// widths in whole float4, whatever the alignment.
template <int E, bool VEC>
__device__ __forceinline__ void load_row(const float *row, int64_t s3, int i, int w, float (&x)[E]) {
    if (VEC) {
        const float *p = row + (i < w ? i : 0);
        if (E == 4) {
            const hola_f4 v = *reinterpret_cast<const hola_f4 *>(p);
#pragma unroll
            for (int e = 0; e < E; ++e) x[e] = v[e];
        } else {
            const hola_f2 v = *reinterpret_cast<const hola_f2 *>(p);
#pragma unroll
            for (int e = 0; e < E; ++e) x[e] = v[e & 1];
        }
    } else {
#pragma unroll
        for (int e = 0; e < E; ++e) x[e] = row[(i + e < w ? i + e : 0) * s3];
    }
}
template <int E, bool VEC>
__device__ __forceinline__ void keep_row(int i, int w, bool on, float (&x)[E]) {
#pragma unroll
    for (int e = 0; e < E; ++e) x[e] = on && (VEC ? i : i + e) < w ? x[e] : 0.f;
}
template <int E, bool VEC>
__device__ __forceinline__ void store_row(float *row, int i, int w, const float (&x)[E]) {
    if (VEC) {
        if (i >= w) return;
        if (E == 4) *reinterpret_cast<hola_f4 *>(row + i) = hola_f4{x[0], x[1], x[E - 2], x[E - 1]};
        else *reinterpret_cast<hola_f2 *>(row + i) = hola_f2{x[0], x[1]};
    } else {
#pragma unroll
        for (int e = 0; e < E; ++e)
            if (i + e < w) row[i + e] = x[e];
    }
}

// A row as the operand of a product over its channels: lane group g holds
// channels 16 t + 4 g + q.
template <int D, bool VEC>
struct Frag {
    float x[D / 16][4];
    __device__ __forceinline__ void load(const View &v, int b, int t, int h, int w) {
        const float *row = row_of(v, b, t, h);
        const int g = lane_id() >> 4;
#pragma unroll
        for (int i = 0; i < D / 16; ++i) load_row<4, VEC>(row, v.s3, 16 * i + 4 * g, w, x[i]);
    }
    __device__ __forceinline__ void keep(bool on, int w) {
        const int g = lane_id() >> 4;
#pragma unroll
        for (int i = 0; i < D / 16; ++i) keep_row<4, VEC>(16 * i + 4 * g, w, on, x[i]);
    }
    __device__ __forceinline__ float dot(const Frag &y) const {
        float s = 0.f;
#pragma unroll
        for (int i = 0; i < D / 16; ++i)
#pragma unroll
            for (int q = 0; q < 4; ++q) s += x[i][q] * y.x[i][q];
        return group_sum(s);
    }
};

// Channels of a product over rows: tile (blk, e) has channels 16 E blk + E m + e as its
// rows m, so that a lane reads and writes E channels in one piece.
template <int D>
struct Chans {
    static constexpr int E = D >= 64 ? 4 : 2, NB = D / (16 * E);
    f32x4 x[NB][E];
    __device__ __forceinline__ void clear() {
#pragma unroll
        for (int k = 0; k < NB; ++k)
#pragma unroll
            for (int e = 0; e < E; ++e) x[k][e] = zero4();
    }
    // Column n (lane n's row of the result) to dst.
    template <bool VEC>
    __device__ __forceinline__ void store(float *row, int w, bool on) const {
        const int g = lane_id() >> 4;
#pragma unroll
        for (int k = 0; k < NB; ++k)
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                float y[E];
#pragma unroll
                for (int e = 0; e < E; ++e) y[e] = on ? x[k][e][i] : 0.f;
                store_row<E, VEC>(row, 16 * E * k + E * (4 * g + i), w, y);
            }
    }
};
// Four rows (reduction indices 4 g + q) as the operand of a product over rows.
template <int D, bool VEC>
struct Rows {
    static constexpr int E = Chans<D>::E, NB = Chans<D>::NB;
    float x[4][NB][E];
    __device__ __forceinline__ void load(const View &v, int b, const int (&t)[4], int h, int w) {
        const int n = lane_id() & 15;
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            const float *row = row_of(v, b, t[q], h);
#pragma unroll
            for (int k = 0; k < NB; ++k) load_row<E, VEC>(row, v.s3, 16 * E * k + E * n, w, x[q][k]);
        }
    }
    // out += these rows, row 4 g + q weighted by y[q] (column n); off rows (t < 0) are zero.
    __device__ __forceinline__ void mix(const f32x4 &y, const int (&t)[4], int w, Chans<D> &out) {
        const int n = lane_id() & 15;
#pragma unroll
        for (int q = 0; q < 4; ++q)
#pragma unroll
            for (int k = 0; k < NB; ++k) {
                keep_row<E, VEC>(16 * E * k + E * n, w, t[q] >= 0, x[q][k]);
#pragma unroll
                for (int e = 0; e < E; ++e) out.x[k][e] = mma(x[q][k][e], y[q], out.x[k][e]);
            }
    }
};

// (batch, head, chunk) of a workgroup: neighbouring workgroups go to the 8 XCDs in
// turn, so each XCD is given a contiguous range of the list, and a head's rows, which
// all its chunks gather from, are read into one L2 instead of into all eight.
__device__ __forceinline__ int chunk_of_block(int id, int blocks) {
    const int x = id & 7, q = blocks >> 3, r = blocks & 7;
    return x * q + min(x, r) + (id >> 3);
}

// ---- chunk slots ------------------------------------------------------------------

// Slots of a chunk (the cache before the chunk, then the chunk's tokens; empty or
// invalid slots have position -1), one wave.
struct SlotInfo {
    float pos[kMaxSlots] __attribute__((aligned(16)));
    float doc[kMaxSlots] __attribute__((aligned(16)));
    __device__ __forceinline__ void stage(const HolaArgs &a, int b, int h, int c) {
        const int lane = lane_id(), first = c * a.chunk, end = min(first + a.chunk, a.T);
        const float *sched = a.schedule + ((int64_t)(b * a.H + h) * (a.nc + 1) + c) * a.cap;
#pragma unroll
        for (int r = 0; r < 2; ++r) {
            const int j = lane + 64 * r;
            if (j >= kMaxSlots) continue;
            float p = -1.f;
            if (j < a.cap) {
                p = sched[j];
            } else {
                const int t = first + j - a.cap;
                if (t < end && ldf(a.valid, b, t) >= 0.5f) p = (float)t;
            }
            pos[j] = p;
            doc[j] = p >= 0.f ? ldf(a.docs, b, (int)p) : 0.f;
        }
        wave_fence();
    }
    __device__ __forceinline__ int at(int j) const { return (int)pos[j]; }
    __device__ __forceinline__ void rows(int s, int (&t)[4]) const {
        const f32x4 p = *reinterpret_cast<const f32x4 *>(&pos[16 * s + 4 * (lane_id() >> 4)]);
#pragma unroll
        for (int q = 0; q < 4; ++q) t[q] = (int)p[q];
    }
};

// The chunk's query of a lane (query n of lane 16 g + n).
struct Query {
    int t;
    bool in, act;  // inside the sequence; and valid
    float doc;
    __device__ __forceinline__ Query(const HolaArgs &a, int b, int c) {
        const int first = c * a.chunk, end = min(first + a.chunk, a.T);
        t = first + (lane_id() & 15);
        in = t < end;
        t = in ? t : first;
        act = in && ldf(a.valid, b, t) >= 0.5f;
        doc = ldf(a.docs, b, t);
    }
};

// Products of the slots' rows with the chunk's queries' x: slot 16 s + 4 g + i, query n.
template <int D, bool VEC>
__device__ __forceinline__ void slot_dots(const View &y, int b, int h, int w, const SlotInfo &s, int slots,
                                          const Frag<D, VEC> &x, f32x4 (&out)[kSlotTiles]) {
    const int n = lane_id() & 15;
    Frag<D, VEC> f[kSlotTiles];
#pragma unroll
    for (int k = 0; k < kSlotTiles; ++k)
        if (16 * k < slots) f[k].load(y, b, s.at(16 * k + n), h, w);
#pragma unroll
    for (int k = 0; k < kSlotTiles; ++k) {
        out[k] = zero4();
        if (16 * k >= slots) continue;
        f[k].keep(s.at(16 * k + n) >= 0, w);
#pragma unroll
        for (int i = 0; i < D / 16; ++i)
#pragma unroll
            for (int q = 0; q < 4; ++q) out[k] = mma(f[k].x[i][q], x.x[i][q], out[k]);
    }
}

// The slots' rows, for their weighted sums.
template <int D, bool VEC>
struct SlotRows {
    Rows<D, VEC> r[kSlotTiles];
    __device__ __forceinline__ void load(const View &y, int b, int h, int w, const SlotInfo &s, int slots) {
#pragma unroll
        for (int k = 0; k < kSlotTiles; ++k) {
            int t[4];
            s.rows(k, t);
            if (16 * k < slots) r[k].load(y, b, t, h, w);
        }
    }
    __device__ __forceinline__ void mix(const f32x4 (&p)[kSlotTiles], int w, const SlotInfo &s, int slots,
                                        Chans<D> &out) {
        out.clear();
#pragma unroll
        for (int k = 0; k < kSlotTiles; ++k) {
            int t[4];
            s.rows(k, t);
            if (16 * k < slots) r[k].mix(p[k], t, w, out);
        }
    }
};

// Raw logits -> scaled, -FLT_MAX where the slot is not visible: empty, later than the
// query, another document, or an inactive query.
__device__ __forceinline__ void visible_logits(const HolaArgs &a, const SlotInfo &s, const Query &q,
                                               f32x4 (&lg)[kSlotTiles]) {
    const int g = lane_id() >> 4;
#pragma unroll
    for (int k = 0; k < kSlotTiles; ++k) {
        const f32x4 p = *reinterpret_cast<const f32x4 *>(&s.pos[16 * k + 4 * g]);
        const f32x4 d = *reinterpret_cast<const f32x4 *>(&s.doc[16 * k + 4 * g]);
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const bool vis = q.act && p[i] >= 0.f && p[i] <= (float)q.t && d[i] == q.doc;
            lg[k][i] = vis ? lg[k][i] * a.scale : -FLT_MAX;
        }
    }
}

// One wave per (batch, head, chunk).  Bound by the gather of the slots' rows (40 KB
// a chunk at 64 slots + 16 and widths of 64, out of the caches) and its latency.
// B16 T512 H8, widths of 64: 31 us, against 86 with the tiles in LDS (four waves a
// chunk) and VALU products; the rows and results alone are 14 us at copy rate.  Four
// waves a SIMD hold all 4096 chunks at once (three: 33 us); they cost 1 to 12 spilled
// registers where keys or values are 64 wide (10 at 64 x 64), which is in the 31 us.
template <int DK, int DV, bool VEC>
__global__ void __launch_bounds__(64, DK + DV > 128 ? 2 : 4) hola_forward_kernel(HolaArgs a) {
    __shared__ SlotInfo s;
    const int g = lane_id() >> 4;
    const int item = chunk_of_block(blockIdx.x, gridDim.x), c = item % a.nc, bh = item / a.nc;
    const int b = bh / a.H, h = bh % a.H;
    const int slots = a.cap + a.chunk;
    const Query q(a, b, c);
    Frag<DK, VEC> qf;
    qf.load(a.q, b, q.t, h, a.dk);
    s.stage(a, b, h, c);
    qf.keep(q.in, a.dk);
    f32x4 p[kSlotTiles];
    slot_dots<DK, VEC>(a.k, b, h, a.dk, s, slots, qf, p);
    SlotRows<DV, VEC> v;
    v.load(a.v, b, h, a.dv, s, slots);
    visible_logits(a, s, q, p);
    const float sink = ldf(a.sink, h);
    float m = sink, sum = 0.f;
#pragma unroll
    for (int k = 0; k < kSlotTiles; ++k)
#pragma unroll
        for (int i = 0; i < 4; ++i) m = fmaxf(m, p[k][i]);
    m = fmaxf(m, __shfl_xor(m, 16));
    m = fmaxf(m, __shfl_xor(m, 32));
#pragma unroll
    for (int k = 0; k < kSlotTiles; ++k)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            p[k][i] = p[k][i] > -FLT_MAX ? expf(p[k][i] - m) : 0.f;
            sum += p[k][i];
        }
    const float inv = 1.f / (group_sum(sum) + expf(sink - m));
    // Normalised before the value product: finite values cannot overflow.
#pragma unroll
    for (int k = 0; k < kSlotTiles; ++k) p[k] *= inv;
    Chans<DV> o;
    v.mix(p, a.dv, s, slots, o);
    if (!q.in) return;
    const int64_t tok = token(a, b, q.t, h);
    o.template store<VEC>(a.out + tok * a.dv, a.dv, q.act);
    if (g == 0) {
        a.stats[2 * tok] = m;
        a.stats[2 * tok + 1] = inv;
    }
}

// ---- backward ---------------------------------------------------------------------

// One wave per (batch, head, chunk); bound as the read, plus the pairs that it
// leaves for the key VJP (8 bytes a query and slot).
// B16 T512 H8, widths of 64: 53 us, against 127 with the tiles in LDS; rows, pairs and
// results are 29 us at copy rate.  Three waves a SIMD: four would spill.  The element
// form spills 34 to 93 registers where keys or values are 128 wide: B16 T512 H8 128 x
// 127, the whole call, takes 778 us, against 1466 with the tiles in LDS.
template <int DK, int DV, bool VEC>
__global__ void __launch_bounds__(64, DK + DV > 128 ? 2 : 3) hola_query_backward_kernel(HolaArgs a) {
    __shared__ SlotInfo s;
    const int g = lane_id() >> 4;
    const int item = chunk_of_block(blockIdx.x, gridDim.x), c = item % a.nc, bh = item / a.nc;
    const int b = bh / a.H, h = bh % a.H;
    const int slots = a.cap + a.chunk;
    const Query q(a, b, c);
    const int64_t tok = token(a, b, q.t, h);
    const float m = a.stats[2 * tok], inv = a.stats[2 * tok + 1], sink = ldf(a.sink, h);
    Frag<DK, VEC> qf;
    Frag<DV, VEC> gf, of;
    const View ov{a.fwd_out, (int64_t)a.T * a.H * a.dv, (int64_t)a.H * a.dv, a.dv, 1};
    qf.load(a.q, b, q.t, h, a.dk);
    of.load(ov, b, q.t, h, a.dv);
    gf.load(a.dout.data ? a.dout : ov, b, q.t, h, a.dv);  // a null adjoint is zero
    s.stage(a, b, h, c);
    qf.keep(q.in, a.dk);
    gf.keep(q.in && a.dout.data, a.dv);
    of.keep(q.in, a.dv);
    float delta = gf.dot(of);
    delta = q.act ? delta : 0.f;
    f32x4 lg[kSlotTiles], dp[kSlotTiles];
    slot_dots<DK, VEC>(a.k, b, h, a.dk, s, slots, qf, lg);
    slot_dots<DV, VEC>(a.v, b, h, a.dv, s, slots, gf, dp);
    SlotRows<DK, VEC> kr;
    kr.load(a.k, b, h, a.dk, s, slots);
    visible_logits(a, s, q, lg);
    if (g == 0 && q.in) {
        a.aux[2 * tok] = delta;
        a.aux[2 * tok + 1] = q.act ? -delta * expf(sink - m) * inv : 0.f;
    }
    // p and the logit gradient d = p (dO . v - delta) / sqrt(d_k), saved as pairs.
    float *pairs = a.pairs + tok * slots * 2;
#pragma unroll
    for (int k = 0; k < kSlotTiles; ++k) {
        float pd[8];
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const bool on = lg[k][i] > -FLT_MAX;
            const float p = on ? expf(lg[k][i] - m) * inv : 0.f;
            const float d = on ? p * (dp[k][i] - delta) * a.scale : 0.f;
            pd[2 * i] = p;
            pd[2 * i + 1] = d;
            dp[k][i] = d;
        }
        const int j = 16 * k + 4 * g;
        if (q.in && j + 3 < slots) {
            *reinterpret_cast<hola_f4 *>(pairs + 2 * j) = hola_f4{pd[0], pd[1], pd[2], pd[3]};
            *reinterpret_cast<hola_f4 *>(pairs + 2 * j + 4) = hola_f4{pd[4], pd[5], pd[6], pd[7]};
        } else if (q.in) {
#pragma unroll
            for (int i = 0; i < 4; ++i)
                if (j + i < slots) {
                    pairs[2 * (j + i)] = pd[2 * i];
                    pairs[2 * (j + i) + 1] = pd[2 * i + 1];
                }
        }
    }
    Chans<DK> o;
    kr.mix(dp, a.dk, s, slots, o);
    if (q.in) o.template store<VEC>(a.gq + tok * a.dk, a.dk, q.act);
}

// kKeyWaves waves per (batch, head, chunk) of keys: the query chunks that see the keys
// run from the keys' own to the last expiry, up to the whole sequence, so wave w
// takes every kKeyWaves-th of them (one wave would leave the early chunks' walks as
// the kernel's tail) and the partial gradients are added pairwise through LDS.
// B16 T512 H8, widths of 64: 38 us, against 99 with one wave on VALU products; 50 with
// the workgroups in grid order (see chunk_of_block).
constexpr int kKeyWaves = 4;

template <int DK, int DV, bool VEC>
__global__ void __launch_bounds__(64 * kKeyWaves) hola_key_backward_kernel(HolaArgs a) {
    constexpr int NK = DK / 16, NV = DV / 16;
    __shared__ float map[kKeyWaves][kMaxChunk];
    __shared__ f32x4 part[kKeyWaves / 2][NK + NV][64];
    const int l = lane_id(), wave = threadIdx.x >> 6, n = l & 15, g = l >> 4;
    const int item = chunk_of_block(blockIdx.x, gridDim.x), c = item % a.nc, bh = item / a.nc;
    const int b = bh / a.H, h = bh % a.H;
    const int first = c * a.chunk, end = min(first + a.chunk, a.T), keys = end - first;
    const int slots = a.cap + a.chunk;
    const float *sched = a.schedule + (int64_t)bh * (a.nc + 1) * a.cap;
    Chans<DK> dka;
    Chans<DV> dva;
    dka.clear();
    dva.clear();
    // Queries that can see a key of this chunk end at its expiry.
    float lastf = (float)end;
    if (l < keys) lastf = fmaxf(lastf, a.expiry[token(a, b, first + l, h)]);
    const int last = (int)wave_max(lastf);
    auto entry = [&](int cq) {
        return l < a.cap && cq < a.nc ? sched[(int64_t)cq * a.cap + l] : -1.f;
    };
    float cached = entry(c + wave);
    for (int cq = c + wave; cq * a.chunk < last; cq += kKeyWaves) {
        const int q0 = cq * a.chunk, nq = min(q0 + a.chunk, a.T) - q0;
        // Where key n sits among the slots of query chunk cq.
        if (l < kMaxChunk) map[wave][l] = cq == c && l < keys ? (float)(a.cap + l) : -1.f;
        wave_fence();
        if (cq != c && cached >= (float)first && cached < (float)end)
            map[wave][(int)cached - first] = (float)l;
        wave_fence();
        const int sl = (int)map[wave][n];
        wave_fence();
        cached = entry(cq + kKeyWaves);
        // The chunk's queries and output adjoints, and the pairs of the mapped slots.
        int t[4];
        float p[4][2];
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            t[q] = 4 * g + q < nq ? q0 + 4 * g + q : -1;
            const float *src = a.pairs + (token(a, b, max(t[q], q0), h) * slots + max(sl, 0)) * 2;
            const hola_f2 v = *reinterpret_cast<const hola_f2 *>(src);
            p[q][0] = v[0];
            p[q][1] = v[1];
        }
        Rows<DK, VEC> qr;
        Rows<DV, VEC> gr;
        qr.load(a.q, b, t, h, a.dk);
        if (a.dout.data) gr.load(a.dout, b, t, h, a.dv);
        f32x4 pr, dl;
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            const bool on = sl >= 0 && t[q] >= 0;
            pr[q] = on ? p[q][0] : 0.f;
            dl[q] = on ? p[q][1] : 0.f;
        }
        qr.mix(dl, t, a.dk, dka);
        if (a.dout.data) gr.mix(pr, t, a.dv, dva);
    }
    // Partial gradients of waves 2, 3 to 0, 1, then of 1 to 0.
#pragma unroll
    for (int half = kKeyWaves / 2; half > 0; half /= 2) {
        if (wave >= half && wave < 2 * half) {
#pragma unroll
            for (int i = 0; i < NK; ++i) part[wave - half][i][l] = dka.x[i / Chans<DK>::E][i % Chans<DK>::E];
#pragma unroll
            for (int i = 0; i < NV; ++i)
                part[wave - half][NK + i][l] = dva.x[i / Chans<DV>::E][i % Chans<DV>::E];
        }
        __syncthreads();
        if (wave < half) {
#pragma unroll
            for (int i = 0; i < NK; ++i) dka.x[i / Chans<DK>::E][i % Chans<DK>::E] += part[wave][i][l];
#pragma unroll
            for (int i = 0; i < NV; ++i)
                dva.x[i / Chans<DV>::E][i % Chans<DV>::E] += part[wave][NK + i][l];
        }
        __syncthreads();
    }
    if (wave != 0 || n >= keys) return;
    const int64_t tok = token(a, b, first + n, h);
    dka.template store<VEC>(a.gk + tok * a.dk, a.dk, true);
    dva.template store<VEC>(a.gv + tok * a.dv, a.dv, true);
}

// dsink[h] = sum over (b, t) of aux[.][1], in a fixed order.
__global__ void __launch_bounds__(1024) hola_sink_kernel(HolaArgs a) {
    __shared__ float red[16];
    const int h = blockIdx.x, tid = threadIdx.x;
    const int64_t n = (int64_t)a.B * a.T;
    float s = 0.f;
    for (int64_t r = tid; r < n; r += 1024) s += a.aux[2 * (r * a.H + h) + 1];
    s = wave_sum(s);
    if ((tid & 63) == 0) red[tid >> 6] = s;
    __syncthreads();
    if (tid == 0) {
        float t = red[0];
        for (int i = 1; i < 16; ++i) t += red[i];
        a.gsink[h] = t;
    }
}

// ---- host ---------------------------------------------------------------------------

int pad_width(int64_t w) { return w <= 32 ? 32 : (w <= 64 ? 64 : 128); }

// Rows in whole float4 pieces: unit channel strides and widths of whole pieces.
bool vec_rows(const HolaArgs &a) {
    return a.q.s3 == 1 && a.k.s3 == 1 && a.v.s3 == 1 && (!a.dout.data || a.dout.s3 == 1) &&
           a.dk % 4 == 0 && a.dv % 4 == 0;
}

template <template <int, int, bool> class K>
void launch_widths(const HolaArgs &a, dim3 grid, hipStream_t st) {
    const int kp = pad_width(a.dk), vp = pad_width(a.dv);
    const bool vec = vec_rows(a);
#define GDN2_HOLA_CASE(P, Q)                                                                    \
    if (kp == P && vp == Q) {                                                                   \
        if (vec) hipLaunchKernelGGL((K<P, Q, true>::fn), grid, dim3(K<P, Q, true>::threads), 0, st, a); \
        else hipLaunchKernelGGL((K<P, Q, false>::fn), grid, dim3(K<P, Q, false>::threads), 0, st, a);   \
        return;                                                                                 \
    }
    GDN2_HOLA_CASE(32, 32) GDN2_HOLA_CASE(32, 64) GDN2_HOLA_CASE(32, 128)
    GDN2_HOLA_CASE(64, 32) GDN2_HOLA_CASE(64, 64) GDN2_HOLA_CASE(64, 128)
    GDN2_HOLA_CASE(128, 32) GDN2_HOLA_CASE(128, 64) GDN2_HOLA_CASE(128, 128)
#undef GDN2_HOLA_CASE
}
template <int P, int Q, bool VEC> struct Fwd {
    static constexpr auto fn = hola_forward_kernel<P, Q, VEC>;
    static constexpr int threads = 64;
};
template <int P, int Q, bool VEC> struct QBwd {
    static constexpr auto fn = hola_query_backward_kernel<P, Q, VEC>;
    static constexpr int threads = 64;
};
template <int P, int Q, bool VEC> struct KBwd {
    static constexpr auto fn = hola_key_backward_kernel<P, Q, VEC>;
    static constexpr int threads = 64 * kKeyWaves;
};

size_t align256(size_t n) { return (n + 255) & ~(size_t)255; }

int64_t chunks_of(const gdn2_hola_shape *s) { return (s->time + s->chunk - 1) / s->chunk; }

int check_hola_shape(const gdn2_hola_shape *s) {
    if (!s) return fail(GDN2_ERR_ARGUMENT, "shape is null");
    if (s->batch < 1 || s->time < 1 || s->heads < 1)
        return fail(GDN2_ERR_SHAPE, "HOLA requires nonempty batch, time and heads");
    if (s->keys < 1 || s->keys > kMaxWidth || s->values < 1 || s->values > kMaxWidth)
        return fail(GDN2_ERR_SHAPE, "HOLA key and value widths must be 1..%d", kMaxWidth);
    if (s->capacity < 1 || s->capacity > kMaxCapacity)
        return fail(GDN2_ERR_SHAPE, "HOLA capacity must be 1..%d (got %d)", kMaxCapacity,
                    s->capacity);
    if (s->chunk < 1 || s->chunk > kMaxChunk)
        return fail(GDN2_ERR_SHAPE, "HOLA chunk must be 1..%d (got %d)", kMaxChunk, s->chunk);
    if (s->batch * s->heads * chunks_of(s) > 0x7FFFFFFF || s->time > (1 << 24))
        return fail(GDN2_ERR_SHAPE, "HOLA problem too large");
    return ok();
}

struct CkLayout {
    size_t schedule, expiry, stats, total;
};

CkLayout ck_layout(const gdn2_hola_shape *s) {
    const int64_t bth = s->batch * s->time * s->heads;
    CkLayout l;
    l.schedule = 0;
    l.expiry = align256((size_t)s->batch * s->heads * (chunks_of(s) + 1) * s->capacity * 4);
    l.stats = l.expiry + align256((size_t)bth * 4);
    l.total = l.stats + align256((size_t)bth * 8);
    return l;
}

size_t ws_pairs_bytes(const gdn2_hola_shape *s) {
    return align256((size_t)s->batch * s->time * s->heads * (s->capacity + s->chunk) * 8);
}

HolaArgs hola_args(const gdn2_hola_shape *s, const gdn2_view *q, const gdn2_view *k,
                   const gdn2_view *v, const gdn2_view *valid, const gdn2_view *docs,
                   const gdn2_view *sink) {
    HolaArgs a{};
    a.B = (int)s->batch;
    a.T = (int)s->time;
    a.H = (int)s->heads;
    a.dk = (int)s->keys;
    a.dv = (int)s->values;
    a.cap = s->capacity;
    a.chunk = s->chunk;
    a.nc = (int)chunks_of(s);
    a.scale = 1.f / sqrtf((float)s->keys);
    a.q = make_view(q);
    a.k = make_view(k);
    a.v = make_view(v);
    a.valid = make_view(valid);
    a.docs = make_view(docs);
    a.sink = make_view(sink);
    return a;
}

int check_f32_views(std::initializer_list<std::pair<const gdn2_view *, const char *>> views) {
    for (auto &v : views) GDN2_TRY(check_view(v.first, v.second, GDN2_F32, false));
    return ok();
}

}  // namespace
}  // namespace gdn2

using namespace gdn2;

extern "C" {

int gdn2_hola_schedule(const gdn2_hola_shape *shape, int recency, const gdn2_view *scores,
                       const gdn2_view *valid, const gdn2_view *documents, float *schedule,
                       void *stream) {
    GDN2_TRY(check_hola_shape(shape));
    GDN2_TRY(check_f32_views({{scores, "scores"}, {valid, "valid"}, {documents, "documents"}}));
    if (!schedule) return fail(GDN2_ERR_ARGUMENT, "schedule is null");
    HolaArgs a = hola_args(shape, nullptr, nullptr, nullptr, valid, documents, nullptr);
    a.scores = make_view(scores);
    a.recency = recency != 0;
    a.schedule = schedule;
    hipLaunchKernelGGL(hola_schedule_kernel, dim3(a.B * a.H), dim3(128), 0, (hipStream_t)stream, a);
    return launch_status(hipGetLastError(), "gdn2_hola_schedule");
}

size_t gdn2_hola_checkpoint_bytes(const gdn2_hola_shape *shape) {
    if (check_hola_shape(shape)) return 0;
    return ck_layout(shape).total;
}

int gdn2_hola_read(const gdn2_hola_shape *shape, int recency, const gdn2_view *q,
                   const gdn2_view *k, const gdn2_view *v, const gdn2_view *scores,
                   const gdn2_view *valid, const gdn2_view *documents, const gdn2_view *sink,
                   float *output, float *final_positions, void *checkpoint,
                   size_t checkpoint_bytes, void *stream) {
    GDN2_TRY(check_hola_shape(shape));
    GDN2_TRY(check_f32_views({{q, "q"}, {k, "k"}, {v, "v"}, {scores, "scores"}, {valid, "valid"},
                              {documents, "documents"}, {sink, "sink"}}));
    if (!output) return fail(GDN2_ERR_ARGUMENT, "output is null");
    const CkLayout l = ck_layout(shape);
    if (!checkpoint || checkpoint_bytes < l.total)
        return fail(GDN2_ERR_WORKSPACE, "checkpoint needs %zu bytes, got %zu", l.total,
                    checkpoint_bytes);
    HolaArgs a = hola_args(shape, q, k, v, valid, documents, sink);
    char *ck = static_cast<char *>(checkpoint);
    a.scores = make_view(scores);
    a.recency = recency != 0;
    a.schedule = reinterpret_cast<float *>(ck + l.schedule);
    a.expiry = reinterpret_cast<float *>(ck + l.expiry);
    a.stats = reinterpret_cast<float *>(ck + l.stats);
    a.out = output;
    a.final_positions = final_positions;
    hipStream_t st = (hipStream_t)stream;
    hipLaunchKernelGGL(hola_schedule_kernel, dim3(a.B * a.H), dim3(128), 0, st, a);
    GDN2_TRY(launch_status(hipGetLastError(), "gdn2_hola_read (schedule)"));
    launch_widths<Fwd>(a, dim3(a.B * a.H * a.nc), st);
    return launch_status(hipGetLastError(), "gdn2_hola_read");
}

size_t gdn2_hola_workspace_bytes(const gdn2_hola_shape *shape) {
    if (check_hola_shape(shape)) return 0;
    return ws_pairs_bytes(shape) +
           align256((size_t)shape->batch * shape->time * shape->heads * 8);
}

int gdn2_hola_backward(const gdn2_hola_shape *shape, const gdn2_view *q, const gdn2_view *k,
                       const gdn2_view *v, const gdn2_view *valid, const gdn2_view *documents,
                       const gdn2_view *sink, const void *checkpoint, size_t checkpoint_bytes,
                       const float *output, const gdn2_view *d_output, float *dq, float *dk,
                       float *dv, float *dsink, void *workspace, size_t workspace_bytes,
                       void *stream) {
    GDN2_TRY(check_hola_shape(shape));
    GDN2_TRY(check_f32_views({{q, "q"}, {k, "k"}, {v, "v"}, {valid, "valid"},
                              {documents, "documents"}, {sink, "sink"}}));
    if (d_output) GDN2_TRY(check_view(d_output, "d_output", GDN2_F32, true));
    if (!output || !dq || !dk || !dv || !dsink)
        return fail(GDN2_ERR_ARGUMENT, "output, dq, dk, dv and dsink must be non-null");
    const CkLayout l = ck_layout(shape);
    if (!checkpoint || checkpoint_bytes < l.total)
        return fail(GDN2_ERR_WORKSPACE, "checkpoint needs %zu bytes, got %zu", l.total,
                    checkpoint_bytes);
    const size_t need = gdn2_hola_workspace_bytes(shape);
    if (!workspace || workspace_bytes < need)
        return fail(GDN2_ERR_WORKSPACE, "workspace needs %zu bytes, got %zu", need,
                    workspace_bytes);
    HolaArgs a = hola_args(shape, q, k, v, valid, documents, sink);
    const char *ck = static_cast<const char *>(checkpoint);
    a.schedule = const_cast<float *>(reinterpret_cast<const float *>(ck + l.schedule));
    a.expiry = const_cast<float *>(reinterpret_cast<const float *>(ck + l.expiry));
    a.stats = const_cast<float *>(reinterpret_cast<const float *>(ck + l.stats));
    if (d_output) a.dout = make_view(d_output);
    a.fwd_out = output;
    a.pairs = static_cast<float *>(workspace);
    a.aux = reinterpret_cast<float *>(static_cast<char *>(workspace) + ws_pairs_bytes(shape));
    a.gq = dq;
    a.gk = dk;
    a.gv = dv;
    a.gsink = dsink;
    hipStream_t st = (hipStream_t)stream;
    const dim3 grid(a.B * a.H * a.nc);
    launch_widths<QBwd>(a, grid, st);
    GDN2_TRY(launch_status(hipGetLastError(), "gdn2_hola_backward (queries)"));
    launch_widths<KBwd>(a, grid, st);
    GDN2_TRY(launch_status(hipGetLastError(), "gdn2_hola_backward (keys)"));
    hipLaunchKernelGGL(hola_sink_kernel, dim3(a.H), dim3(1024), 0, st, a);
    return launch_status(hipGetLastError(), "gdn2_hola_backward");
}

}  // extern "C"
