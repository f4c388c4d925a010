// Chunked channel-wise GDN-2 in f32 on gfx950: the reference's own op
// configuration (f32 q/k/v, d_k = 32, d_v = 64, 16-token chunks;
// crates/kernels/src/gdn2.rs:10-12, crates/kernels/src/gdn_training.rs:8-9), and
// every d_k, d_v <= 128, f32 or bf16 (read as its exact f32 values).
//
// Recurrence per valid token t (crates/mixers/src/reference.rs:68-111):
//   bar = diag(alpha_t) S;  delta_t = w_t.v_t - bar^T (e_t.k_t);
//   S_t = bar + k_t delta_t^T;  o_t = S_t^T q_t;  score_t = |k_t| |delta_t|.
// Per chunk of C = 16 tokens with start state S0 and, per key channel i, the
// decays as direct products of the gates, as the reference's chunked kernels
// form them (gdn2.rs:23-64), so zero and negative gates need no special case:
//   D_ts = prod_{s < u <= t} a_u (s <= t), a = alpha, 0 on a reset, 1 on padding
//   b_t = prod_{u <= t} a_u,  lam_s = prod_{s < u <= 15} a_u
//   eh = e.k,  Qhat = b.q,  Ktil = lam.k
//   A_ts = sum_i eh_t D_ts k_s (s < t),  T = (I + A)^-1,  P_ts = sum_i q_t D_ts k_s (s <= t)
//   W' = T (b.eh),  U = T (w.v),  delta = U - W' S0,  O = Qhat S0 + P delta
//   S_16 = diag(b_15) S0 + Ktil^T delta.
// Padding tokens have zero k, q, e, w (state kept, zero output).
//
// The pair sums go through matrix products by levels.  For t and s in different
// halves of an aligned block of 2 L tokens (L = 4, 8), D_ts = F_t G_s with F the
// product from t's half's start to t and G the product after s to its half's end,
// so a level is one product of scaled rows, (eh F)(k G)^T, whose other entries
// are dropped; the pairs inside a block of four tokens are summed on the VALU,
// where a lane holds four tokens of a channel.  F and G of every level are direct
// products, so nothing is divided.  The backward runs the same levels on the
// score adjoints and carries the adjoints of F and G back through the products
// that formed them, which is exact for zero gates too.
//
// Five kernels: prep (A, T, P, the map's factors), the state scan over the chunks
// of each (batch, head), out, the adjoint scan
//   X <- diag(b_15) X + Qhat^T dO - W'^T (P^T dO + c delta + Ktil X)
// and bgrad (every gradient); a wave takes one 16-channel tile of a chunk, or of a
// head in the scans.  All products are v_mfma_f32_16x16x4f32 (exact f32 products)
// on operands read in their layout (gdn2_chunk_f32_dev.h).
//
// Kernels of a forward + backward, against the LDS-tiled kernels before them
// (f32 pair sums on the VALU; bf16 64 x 64 calls on bf16 hi/lo MFMA):
//   f32 B8 T512 H4 K32 V64    75 us, was 141 (floor of its 43 MB 9 us)
//   bf16 B16 T509 H8 64 x 64  221 us, was 366 (173 MB, 35 us)
// A lone sequence per head (B1 T128 H4 K32 V64) takes 34 us, was 65: five launches
// of 4 to 9 us.  bgrad (92 us of the 221) moves 255 MB, 52 us of a copy's rate.
#include "gdn2_chunk_f32_dev.h"

#include <algorithm>

namespace gdn2 {

namespace {

// F and G of the token of lane n (see the head of the file), levels 4 and 8, of
// one channel whose gate in lane n is a.
struct FcLevels {
    float f4, g4, f8, g8;
};
__device__ __forceinline__ FcLevels fc_levels(float a, bool o1, bool o2, bool o4) {
    // Every lane move stands outside the selections: a lane that a branch has
    // switched off would read as zero.
    const float lo2 = fc_dpp<0xA0>(a), hi2 = fc_dpp<0xF5>(a);      // the pair's first and second gate
    const float f2 = o1 ? a * lo2 : a, g2 = o1 ? 1.f : hi2;
    const float lo4 = fc_dpp<0x55>(f2), hi4 = fc_dpp<0xFF>(f2);    // the quad's first and second pair
    FcLevels x;
    x.f4 = o2 ? f2 * lo4 : f2;
    x.g4 = o2 ? g2 : g2 * hi4;
    const float other = fc_dpp<0x141>(fc_dpp<0xFF>(x.f4));         // the other quad of the eight
    x.f8 = o4 ? x.f4 * other : x.f4;
    x.g8 = o4 ? x.g4 : x.g4 * other;
    return x;
}

// The same for a lane that holds tokens 4 g .. 4 g + 3 of a channel (a col tile):
// level 4's F and G are products of its own gates, x4 and x8 the whole products of
// the other quad of the eight and of the other eight.
struct FcCol {
    f32x4 f4, g4;
    float x4, x8;
    int g;
    __device__ __forceinline__ FcCol(const f32x4 &a, int g_) : g(g_) {
        f4[0] = a[0];
        f4[1] = f4[0] * a[1];
        f4[2] = f4[1] * a[2];
        f4[3] = f4[2] * a[3];
        g4[3] = 1.f;
        g4[2] = a[3];
        g4[1] = a[2] * a[3];
        g4[0] = a[1] * g4[1];
        x4 = __shfl_xor(f4[3], 16);
        x8 = __shfl_xor(f4[3] * x4, 32);
    }
    __device__ __forceinline__ float uf4() const { return (g & 1) ? x4 : 1.f; }  // F8 = F4 uf4
    __device__ __forceinline__ float ug4() const { return (g & 1) ? 1.f : x4; }  // G8 = G4 ug4
    __device__ __forceinline__ float uf8() const { return g >= 2 ? x8 : 1.f; }   // b = F8 uf8
    __device__ __forceinline__ float ug8() const { return g >= 2 ? 1.f : x8; }   // lam = G8 ug8
};

// The decay of a token from its gate: 1 on padding, 0 on a reset; NaN for a gate
// below `least` (0 where the call's contract asks for alpha >= 0, else -inf).
__device__ __forceinline__ float fc_gate(float a, bool live, float masked, float least) {
    a = a < least ? __builtin_nanf("") : a;
    return live ? a : masked;
}
__device__ __forceinline__ float fc_least(const FcArgs &a) { return a.nonneg ? 0.f : -__builtin_inff(); }

template <int KM>
struct FcGradSmem {
    static constexpr int LD = 16 * KM + 4;  // f32 row stride: rows 4 banks apart
    static constexpr int LM = 20;
    float dr[C * LD], dl[C * LD];  // [token][value]
    f32x4 m[4][64];                // dP, dA by columns t; dP, dA by rows t (one piece per lane)
    float p[2][C * LM];            // dP, dA as [t][s]
};

}  // namespace

// ---- prep: gates, A, T, P and the factored map ------------------------------------
// Wave w takes key tile w (its terms of A and P, Ktil, Qhat and W') and value
// tile w (U); blockDim is 64 max(KT, VT).  The terms of A meet in wave 0, which
// inverts, and those of P in the last wave.  (One wave per chunk measured 50 us
// where this takes 37 at 4096 chunks of 64 x 64: it holds 192 registers and waits
// for one tile's reads after another.)
struct FcPrepSmem {
    f32x4 A[8][64], P[8][64];  // each key tile's terms, in acc layout
    float la[C * FC_LA];
    f32x4 t[64];
    float ksq[8][C];
};

template <bool BF, bool VEC>
__global__ void __launch_bounds__(512) fc_prep_kernel(FcArgs a) {
    __shared__ FcPrepSmem sm;
    const SeqArgs &s = a.s;
    const int64_t ci = blockIdx.x;
    const int bh = blockIdx.x / a.nc, c = blockIdx.x % a.nc, b = bh / s.H, h = bh % s.H;
    const int K = s.K, V = s.V, KT = fc_kp(K) >> 4, VT = (V + 15) >> 4, NW = blockDim.x >> 6;
    const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), l = lane_id(), g = l >> 4, n = l & 15;
    bool on, rst;
    fc_flags(s, b, c, on, rst);
    const bool live = on && !rst;
    const float masked = on ? 0.f : 1.f, least = fc_least(a);
    f32x4 u = zero4(), be = zero4();
    if (w < VT)
        u = FcSrc<BF, VEC>(s.v, b, h, c, s.T, V).col(w) * FcSrc<false, VEC>(s.write, b, h, c, s.T, V).col(w);
    if (w < KT) {
        const FcSrc<BF, VEC> sk(s.k, b, h, c, s.T, K), sq(s.q, b, h, c, s.T, K);
        const FcSrc<false, VEC> sa(s.alpha, b, h, c, s.T, K), se(s.erase, b, h, c, s.T, K);
        f32x4 kf = sk.frag(w), qf = sq.frag(w), ef = se.frag(w), af = sa.frag(w);
        f32x4 k = sk.col(w), q = sq.col(w), e = se.col(w), al = sa.col(w);
        const bool o1 = n & 1, o2 = n & 2, o4 = n & 4;
        const f32x4 on4 = fc_rows(on ? 1.f : 0.f, g), live4 = fc_rows(live ? 1.f : 0.f, g);
        kf = fc_keep(kf, on), qf = fc_keep(qf, on), ef = fc_keep(ef, on);
        k = fc_keep4(k, on4), q = fc_keep4(q, on4), e = fc_keep4(e, on4);
        f32x4 e4, e8, q4, q8, k4, k8;
        float ksq = 0.f;
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            ksq += kf[r] * kf[r];
            const FcLevels x = fc_levels(fc_gate(af[r], live, masked, least), o1, o2, o4);
            const float eh = ef[r] * kf[r];
            e4[r] = eh * x.f4, e8[r] = eh * x.f8;
            q4[r] = qf[r] * x.f4, q8[r] = qf[r] * x.f8;
            k4[r] = kf[r] * x.g4, k8[r] = kf[r] * x.g8;
            al[r] = fc_gate(al[r], live4[r] != 0.f, 1.f - on4[r], least);
        }
        const f32x4 A4 = fc_mma4(e4, k4, zero4()), A8 = fc_mma4(e8, k8, zero4());
        const f32x4 P4 = fc_mma4(q4, k4, zero4()), P8 = fc_mma4(q8, k8, zero4());
        ksq = fc_group_sum(ksq);
        if (g == 0) sm.ksq[w][n] = ksq;
        // the pairs inside the lane's four tokens, summed over the channels
        const f32x4 eh = e * k;
        const float y10 = k[0] * al[1], y20 = y10 * al[2], y30 = y20 * al[3], y21 = k[1] * al[2], y31 = y21 * al[3],
                    y32 = k[2] * al[3];
        const float a10 = fc_row_sum(eh[1] * y10), a20 = fc_row_sum(eh[2] * y20), a21 = fc_row_sum(eh[2] * y21);
        const float a30 = fc_row_sum(eh[3] * y30), a31 = fc_row_sum(eh[3] * y31), a32 = fc_row_sum(eh[3] * y32);
        const float p10 = fc_row_sum(q[1] * y10), p20 = fc_row_sum(q[2] * y20), p21 = fc_row_sum(q[2] * y21);
        const float p30 = fc_row_sum(q[3] * y30), p31 = fc_row_sum(q[3] * y31), p32 = fc_row_sum(q[3] * y32);
        const float p00 = fc_row_sum(q[0] * k[0]), p11 = fc_row_sum(q[1] * k[1]), p22 = fc_row_sum(q[2] * k[2]),
                    p33 = fc_row_sum(q[3] * k[3]);
        // rows t = 4 g + i, column s = n: the level by the quads of t and s
        const int sq4 = n >> 2, sc = n & 3;
        const bool diag = sq4 == g, near = (sq4 < g) & ((sq4 >> 1) == (g >> 1)), far = (sq4 < g) & !near;
        const bool c0 = sc == 0, c1 = sc == 1, c2 = sc == 2;
        const f32x4 ad = {0.f, c0 ? a10 : 0.f, c0 ? a20 : (c1 ? a21 : 0.f), c0 ? a30 : (c1 ? a31 : (c2 ? a32 : 0.f))};
        const f32x4 pd = {c0 ? p00 : 0.f, c0 ? p10 : (c1 ? p11 : 0.f), c0 ? p20 : (c1 ? p21 : (c2 ? p22 : 0.f)),
                          c0 ? p30 : (c1 ? p31 : (c2 ? p32 : p33))};
        f32x4 A, P;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const float ax = far ? A8[i] : 0.f, px = far ? P8[i] : 0.f, ay = near ? A4[i] : ax, py = near ? P4[i] : px;
            A[i] = diag ? ad[i] : ay;
            P[i] = diag ? pd[i] : py;
        }
        sm.A[w][l] = A;
        sm.P[w][l] = P;
        const FcCol x(al, g);
        const f32x4 bt = x.f4 * (x.uf4() * x.uf8());
        be = bt * eh;
        fc_p4(a.fk + (ci * KT + w) * 256, 16 * l, x.g4 * (x.ug4() * x.ug8()) * k);
        fc_p4(a.fq + (ci * KT + w) * 256, 16 * l, bt * q);
        if (g == 3) *fc_at(a.gv + (ci * KT + w) * 16, 4 * n) = 16 * w + n < K ? bt[3] : 0.f;
    }
    __syncthreads();
    if (w == 0) {
        f32x4 A = sm.A[0][l];
        for (int x = 1; x < KT; ++x) A += sm.A[x][l];
        const f32x4 t = fc_inverse(A, sm.la, g, n);
        sm.t[l] = t;
        fc_p4(a.tm + ci * C * C, (n * C + 4 * g) * 4, t);
    }
    if (w == NW - 1) {
        f32x4 P = sm.P[0][l];
        float ksq = sm.ksq[0][n];
        for (int x = 1; x < KT; ++x) P += sm.P[x][l], ksq += sm.ksq[x][n];
        FcOff(C).put(a.pm + ci * C * C, P);
        if (g < 3) *fc_at(a.gb + ci * C * 8 + C * g, 4 * n) = g == 0 ? (on ? 1.f : 0.f) : (g == 1 ? (rst ? 1.f : 0.f) : ksq);
    }
    __syncthreads();
    const f32x4 t = sm.t[l];
    if (w < KT) fc_p4(a.fw + (ci * KT + w) * 256, 16 * l, fc_mma4(t, be, zero4()));
    if (w < VT)
        fc_p4(a.fu + (ci * VT + w) * 256, 16 * l, fc_mma4(t, fc_keep4(u, fc_rows(on ? 1.f : 0.f, g)), zero4()));
}

// ---- the scans over the chunks of one (batch, head) -----------------------------
// One workgroup per (batch, head, 16 value columns j = 16 cg + l % 16), one wave
// per 16-row key tile tau = w.  Wave tau holds its tile of the state in the
// accumulator layout: lane l (g = l / 16, n = l % 16) holds S[16 tau + 4 g + r][j]
// in register r.  Per chunk,
//   forward:  v = U - W' S,                  S <- diag(gv) S + Ktil^T v
//   reverse:  v = P^T dO + c delta + Ktil X,  X <- diag(gv) X + Qhat^T dO - W'^T v
// v sums over the key axis: each wave forms its tile's part (the accumulator is
// the B operand), the parts meet in LDS (double-buffered by step parity, one
// barrier per step) and every wave adds them in tile order, so all waves hold the
// same v; each then updates its own tile, v's accumulator rows as the B operand.
// The other operands are read from global memory into registers D chunks ahead.
// The scans are bound by the bytes they stream (at 128 heads of 64 x 64, 28 KiB
// per chunk forward, 4.1 TB/s).  An additive term N of the adjoint map, formed by
// a kernel of its own, cost 16 KiB written and read per chunk: that kernel and the
// scan took 27 and 42 us where the scan with the products inside takes 46.
template <bool REV>
struct FcScanOps {
    f32x4 w;           // A operand, tokens n, keys 16 tau + 4 g ..: W' or Ktil across
    f32x4 g, k, a;     // gv rows; Ktil or W', A operand over the tokens; U or Qhat
    f32x4 d, p;        // reverse: dO columns j, P rows
    f32x4 on;
    f32x4 c, e;        // reverse with a score adjoint: the coefficients c, the edits
};

// The workgroups of one (batch, head) read the same factors, so they take block
// indices of one residue mod 8 and share an XCD's L2.
// SC: with a score adjoint.
template <int KT, bool REV, bool BF, bool VEC, bool SC>
__global__ void __launch_bounds__(64 * KT) fc_scan_kernel(FcArgs a) {
    __shared__ float4 vpart[2][KT][64];  // each wave's part of v, by step parity
    const SeqArgs &s = a.s;
    const int K = s.K, V = s.V, VT = (V + 15) / 16;
    const int tau = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int wg = blockIdx.x, cg = (wg >> 3) % VT, bh = (wg & 7) + 8 * (wg / (8 * VT));
    if (bh >= s.B * s.H) return;
    const int b = bh / s.H, h = bh % s.H;
    const int l = lane_id(), g = l >> 4, n = l & 15, j = 16 * cg + n;
    const bool jv = j < V, has_do = REV && s.dout.data != nullptr;
    const View dov = has_do ? s.dout : s.v;  // a missing dO reads v, zeroed where it is used
    const int steps = REV ? a.wn : a.nc;
    if (REV && a.wbad && a.w0 + a.wn == a.nc && cg == 0 && threadIdx.x == 0) a.wbad[bh] = a.bad[bh];
    float *carry = a.carry + (((int64_t)bh * VT + cg) * KT + tau) * 256;
    f32x4 X;
    if (REV && a.w0 + a.wn < a.nc) {
        X = fc_g4(carry, 16 * l);
    } else {
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const int i = 16 * tau + 4 * g + r;
            float x = 0.f;
            if (i < K && jv) {
                if (!REV) x = s.initial.data ? ld4<float>(s.initial, b, h, i, j) : 0.f;
                else x = s.dfinal ? s.dfinal[((int64_t)bh * K + i) * V + j] : 0.f;
            }
            X[r] = x;
        }
    }
    // A ring of D chunks' operands in registers: chunk step + D is loaded (the
    // last chunk again past the end) as soon as step's operands are used.  No load
    // sits behind a branch that lanes or steps take differently.
    constexpr int D = 4;
    FcScanOps<REV> ring[D];
    auto chunk_at = [&](int step) {  // within the window (forward: all chunks)
        const int sc = step < steps ? step : steps - 1;
        return REV ? steps - 1 - sc : sc;
    };
    const FcOff oc(C);
    auto load = [&](int step, FcScanOps<REV> &o) {
        const int c = (REV ? a.w0 : 0) + chunk_at(step);
        const int64_t ci = (int64_t)bh * a.nc + c;
        const float *fw = a.fw + (ci * KT + tau) * 256, *fk = a.fk + (ci * KT + tau) * 256;
        o.w = fc_across(REV ? fk : fw);
        o.g = fc_g4(a.gv + (ci * KT + tau) * 16, 16 * g);
        o.k = fc_g4(REV ? fw : fk, 16 * l);
        o.a = fc_g4(REV ? a.fq + (ci * KT + tau) * 256 : a.fu + (ci * VT + cg) * 256, 16 * l);
        if (REV) {
            o.d = FcSrc<BF, VEC>(dov, b, h, c, s.T, V).col(cg);
            o.p = oc.get(a.pm + ci * C * C);
            o.on = fc_gb4(a, ci, 0);
            if (SC) {
                o.c = fc_g4(a.sc + ((int64_t)bh * a.wn + chunk_at(step)) * 2 * C, 16 * g);
                o.e = fc_g4(a.fu + (ci * VT + cg) * 256, 16 * l);
            }
        }
    };
    // The loads are issued in ring order, the order in which the steps wait for
    // them: a wait at the loop's head must not cover the whole ring because the
    // scheduler put the first chunk's loads last.
#pragma unroll
    for (int d = 0; d < D; ++d) {
        load(d, ring[d]);
        __builtin_amdgcn_sched_barrier(0);
    }
    // A step's masked dO and the terms of v known before X: U, or in tile 0 P^T dO
    // + c delta.
    f32x4 dnext = zero4(), base = zero4();
    auto prepare = [&](const FcScanOps<REV> &o) {
        if (!REV) {
            base = o.a;
            return;
        }
        dnext = fc_keep(fc_keep4(o.d, o.on), has_do);
        if (tau != 0) return;
        base = fc_mma4(o.p, dnext, SC ? o.c * o.e : zero4());
    };
    prepare(ring[0]);
    float *keep = REV ? a.ds : a.st;
    auto advance = [&](int step, int d) __attribute__((always_inline)) {
        const int cw = chunk_at(step);
        const int64_t ci = (int64_t)bh * a.nc + (REV ? a.w0 : 0) + cw, wi = (int64_t)bh * (REV ? a.wn : a.nc) + cw;
        const FcScanOps<REV> &cur = ring[d];
        const f32x4 dnow = dnext;
        // The state before (forward) / the adjoint after (reverse) this chunk; zero
        // outside K x V, as X0 and every term of the map are.
        fc_p4(keep + ((wi * VT + cg) * KT + tau) * 256, 16 * l, X);
        // this tile's part of v[t][j], t = 4 g + r: -W' S, or Ktil X (+ the step's
        // base in tile 0).  The four-step products that wait for X or v run as two
        // chains of two.  U and the base, the larger terms, come in last: at the head
        // of the chains every addition rounds at U's size (the edits' error at 64 x 64
        // is then 9.8e-8, against 5.0e-8, in an emulation of the sums).
        const f32x4 wm = REV ? cur.w : -cur.w;
        f32x4 vp = fc_mma(wm[1], X[1], fc_mma(wm[0], X[0], zero4()));
        vp += fc_mma(wm[3], X[3], fc_mma(wm[2], X[2], zero4()));
        if (REV && tau == 0) vp += base;
        const f32x4 u = base;
        const int par = step & 1;
        if (KT > 1) vpart[par][tau][l] = make_float4(vp[0], vp[1], vp[2], vp[3]);
        // in the shadow of the exchange: what depends on neither X nor v
        f32x4 x = cur.g * X, v = vp;
        if (REV) x = fc_mma4(cur.a, dnow, x);
        prepare(ring[(d + 1) % D]);
        if (KT > 1) {
            __syncthreads();
            float4 t0 = vpart[par][0][l];
            v = f32x4{t0.x, t0.y, t0.z, t0.w};
#pragma unroll
            for (int u = 1; u < KT; ++u) {
                const float4 t = vpart[par][u][l];
                v += f32x4{t.x, t.y, t.z, t.w};
            }
        }
        if (!REV) v += u;
        // forward: v is the chunk's edits delta, kept where U was
        if (!REV && tau == 0) fc_p4(a.fu + (ci * VT + cg) * 256, 16 * l, v);
        const f32x4 km = REV ? -cur.k : cur.k;
        x = fc_mma(km[1], v[1], fc_mma(km[0], v[0], x));
        X = x + fc_mma(km[3], v[3], fc_mma(km[2], v[2], zero4()));
        __builtin_amdgcn_sched_barrier(0);
        load(step + D, ring[d]);
        __builtin_amdgcn_sched_barrier(0);
    };
    // Whole rounds of the ring, then what is left: a round with exits between its
    // steps would make every wait at its head cover the whole ring.
    int s0 = 0;
    for (; s0 + D <= steps; s0 += D)
#pragma unroll
        for (int d = 0; d < D; ++d) advance(s0 + d, d);
#pragma unroll
    for (int d = 0; d < D - 1; ++d)
        if (s0 + d < steps) advance(s0 + d, d);
    if (REV && a.w0 > 0) {
        fc_p4(carry, 16 * l, X);
        return;
    }
    float *fin = REV ? s.dinitial : s.final_state;
    if (fin)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const int i = 16 * tau + 4 * g + r;
            if (i < K && jv) fin[((int64_t)bh * K + i) * V + j] = X[r];
        }
}

// The score adjoint's coefficients per token, one wave per chunk: c = dscore |k| /
// |delta| and c' = dscore |delta| / |k| (zero at a zero edit or key).
__global__ void __launch_bounds__(64) fc_score_kernel(FcArgs a) {
    const SeqArgs &s = a.s;
    const int bh = blockIdx.x / a.wn, c = a.w0 + blockIdx.x % a.wn, VT = (s.V + 15) >> 4;
    const int64_t ci = (int64_t)bh * a.nc + c, wi = blockIdx.x;
    const int l = lane_id(), n = l & 15, tg = c * C + n;
    f32x4 d2 = zero4();
    for (int vt = 0; vt < VT; ++vt) {
        const f32x4 d = fc_g4(a.fu + (ci * VT + vt) * 256, 16 * l);
        d2 += d * d;
    }
    float dsq = 0.f;  // token n's sum sits in group n / 4, register n % 4
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const float x = __shfl(fc_row_sum(d2[i]), 16 * (n >> 2));
        if ((n & 3) == i) dsq = x;
    }
    const float nk = sqrtf(fc_gb(a, ci, 2)), nd = sqrtf(dsq);
    const float dsc = tg < s.T ? s.dscores[((int64_t)(bh / s.H) * s.T + tg) * s.H + bh % s.H] : 0.f;
    const bool ok = fc_gb(a, ci, 0) != 0.f && nk > 0.f && nd > 0.f;
    if (l < 2 * C) *fc_at(a.sc + wi * 2 * C, 4 * l) = !ok ? 0.f : (l < C ? dsc * nk / nd : dsc * nd / nk);
}

// ---- out: O = Qhat S0 + P delta and the scores, one wave per value tile -----------
template <int KM, bool VEC>
__global__ void __launch_bounds__(512) fc_out_kernel(FcArgs a) {
    __shared__ float dd[8][C];
    const SeqArgs &s = a.s;
    const int64_t ci = blockIdx.x;
    const int bh = blockIdx.x / a.nc, c = blockIdx.x % a.nc, b = bh / s.H, h = bh % s.H;
    const int K = s.K, V = s.V, KT = fc_kp(K) >> 4, VT = (V + 15) >> 4;
    const int vt = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), l = lane_id(), g = l >> 4, n = l & 15;
    const float *fq = a.fq + ci * KT * 256, *st = a.st + (ci * VT + vt) * KT * 256;
    f32x4 q[KM], s0[KM];
#pragma unroll
    for (int tau = 0; tau < KM; ++tau) {
        q[tau] = s0[tau] = zero4();
        if (tau < KT) q[tau] = fc_across(fq + 256 * tau), s0[tau] = fc_g4(st + 256 * tau, 16 * l);
    }
    const f32x4 p = fc_g4(a.pm + ci * C * C, (n * C + 4 * g) * 4), dl = fc_g4(a.fu + (ci * VT + vt) * 256, 16 * l);
    const f32x4 on4 = fc_gb4(a, ci, 0);
    const f32x4 o = fc_mma_tree<KM>(q, s0) + fc_mma4(p, dl, zero4());
    fc_put<false, VEC>(s.out, s.out_bf16, s, b, h, c, V, vt, fc_keep4(o, on4));
    if (a.bad && !fc_finite(o + dl)) a.bad[bh] = 1;
    if (!s.scores) return;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const float x = fc_row_sum(dl[i] * dl[i]);
        if (n == 0) dd[vt][4 * g + i] = x;
    }
    __syncthreads();
    if (threadIdx.x < C && c * C + n < s.T) {
        double x = 0.;
        for (int v = 0; v < VT; ++v) x += dd[v][n];
        s.scores[((int64_t)b * s.T + c * C + n) * s.H + h] =
            fc_gb(a, ci, 0) != 0.f ? sqrtf(fc_gb(a, ci, 2) * (float)x) : 0.f;
    }
}

// ---- bgrad: every gradient of one chunk -----------------------------------------
// With S0 and delta (the forward) and dS at the chunk end (the adjoint scan):
//   ddelta = P^T dO + Ktil dS + c delta,  dR = T^T ddelta,  dw = dR.v,  dv = dR.w
//   Qg = dO S0^T,  Ag = -dR S0^T,  Kg = delta dS^T
//   dA = -strict_lower(dR delta^T),  dP = lower(dO delta^T)
// and per key channel, with the pair sums by levels (see the head of the file)
//   eA_t = sum_s dA_ts D_ts k_s,  qP_t = sum_s dP_ts D_ts k_s,
//   kAP_s = sum_t (dA_ts eh_t + dP_ts q_t) D_ts
//   dq = b Qg + qP;  deh = b Ag + eA;  de = k deh;
//   dk = lam Kg + kAP + e deh + c' k
// and dalpha from the adjoints of every F and G (b and lam, whose adjoints are
// eh.Ag + q.Qg [+ rowsum(S0 . dS) at token 15] and k.Kg, are the last level's).
// Wave w takes value tile w up to dR, then key tile w; blockDim is 64 max(KT, VT).
// Four waves a SIMD leave 128 registers, of which 1 spills (4 in the f32 element form).
template <int KM, bool BF, bool VEC>
__global__ void __launch_bounds__(64 * KM, KM == 8 ? 2 : 4) fc_bgrad_kernel(FcArgs a) {
    __shared__ FcGradSmem<KM> sm;
    constexpr int LD = FcGradSmem<KM>::LD, LM = FcGradSmem<KM>::LM;
    const SeqArgs &s = a.s;
    const int64_t ci = blockIdx.x;
    const int bh = blockIdx.x / a.nc, c = blockIdx.x % a.nc, b = bh / s.H, h = bh % s.H;
    const int K = s.K, V = s.V, KT = fc_kp(K) >> 4, VT = (V + 15) >> 4, NW = blockDim.x >> 6;
    const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), l = lane_id(), g = l >> 4, n = l & 15;
    const FcSrc<BF, VEC> sdo(s.dout, b, h, c, s.T, V);
    const bool has_do = s.dout.data != nullptr;
    const bool on = fc_gb(a, ci, 0) != 0.f;
    const f32x4 on4 = fc_gb4(a, ci, 0), rst4 = fc_gb4(a, ci, 1);
    f32x4 cs4 = zero4(), ck4 = zero4();
    if (s.dscores) cs4 = fc_g4(a.sc + ci * 2 * C, 16 * g), ck4 = fc_g4(a.sc + ci * 2 * C + C, 16 * g);
    const float *st = a.st + ci * KT * VT * 256, *ds = a.ds + ci * KT * VT * 256;
    if (w < VT) {  // ddelta and dR of value tile w
        const FcOff oc(C);
        const f32x4 p = oc.get(a.pm + ci * C * C), tb = oc.get(a.tm + ci * C * C);
        const f32x4 dl = fc_g4(a.fu + (ci * VT + w) * 256, 16 * l);
        const f32x4 v = FcSrc<BF, VEC>(s.v, b, h, c, s.T, V).col(w), wr = FcSrc<false, VEC>(s.write, b, h, c, s.T, V).col(w);
        f32x4 dO = has_do ? sdo.col(w) : zero4(), kf[KM], dsn[KM];
        const float *fk = a.fk + ci * KT * 256;
#pragma unroll
        for (int tau = 0; tau < KM; ++tau) {
            kf[tau] = dsn[tau] = zero4();
            if (tau < KT) kf[tau] = fc_across(fk + 256 * tau), dsn[tau] = fc_g4(ds + (w * KT + tau) * 256, 16 * l);
        }
        dO = fc_keep4(dO, on4);
        f32x4 dd = fc_mma4(p, dO, cs4 * dl);
#pragma unroll
        for (int tau = 0; tau < KM; ++tau) dd = fc_mma4(kf[tau], dsn[tau], dd);
        const f32x4 dr = fc_mma4(tb, dd, zero4());                                           // rows t, column j
        *reinterpret_cast<f32x4 *>(&sm.dr[n * LD + 16 * w + 4 * g]) = fc_mma4(dd, tb, zero4());  // rows j, column t
#pragma unroll
        for (int r = 0; r < 4; ++r) sm.dl[(4 * g + r) * LD + 16 * w + n] = dl[r];
        if (s.dwrite) fc_put<false, VEC>(s.dwrite, 0, s, b, h, c, V, w, fc_keep4(dr * v, on4));
        if (s.dv) fc_put<BF, VEC>(s.dv, BF, s, b, h, c, V, w, fc_keep4(dr * wr, on4));
    }
    f32x4 yf[KM];  // dO rows
#pragma unroll
    for (int vt = 0; vt < KM; ++vt) yf[vt] = (has_do && vt < VT) ? fc_keep(sdo.frag(vt), on) : zero4();
    f32x4 k = zero4(), q = zero4(), e = zero4(), al = zero4();
    if (w < KT) {
        k = FcSrc<BF, VEC>(s.k, b, h, c, s.T, K).col(w);
        q = FcSrc<BF, VEC>(s.q, b, h, c, s.T, K).col(w);
        e = FcSrc<false, VEC>(s.erase, b, h, c, s.T, K).col(w);
        al = FcSrc<false, VEC>(s.alpha, b, h, c, s.T, K).col(w);
    }
    __syncthreads();
    // The score adjoints: 0 dP, 1 dA with column t (row s); 2 dP, 3 dA with row t.
    for (int x = w; x < 4; x += NW) {
        f32x4 m = zero4();
#pragma unroll
        for (int vt = 0; vt < KM; ++vt)
            if (vt < VT) {
                const f32x4 d = *reinterpret_cast<const f32x4 *>(&sm.dl[n * LD + 16 * vt + 4 * g]);
                const f32x4 y = (x & 1) ? *reinterpret_cast<const f32x4 *>(&sm.dr[n * LD + 16 * vt + 4 * g]) : yf[vt];
                m = x < 2 ? fc_mma4(d, y, m) : fc_mma4(y, d, m);
            }
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int t = x < 2 ? n : 4 * g + i, u = x < 2 ? 4 * g + i : n;
            m[i] = (x & 1) ? (u < t ? -m[i] : 0.f) : (u <= t ? m[i] : 0.f);
            if (x >= 2) sm.p[x - 2][t * LM + u] = m[i];
        }
        sm.m[x][l] = m;
    }
    f32x4 Qg = zero4(), Ag = zero4(), Kg = zero4();  // rows t, column key 16 w + n
    float fs = 0.f;                                  // rowsum(S0 . dS) of key 16 w + n
    if (w < KT) {
#pragma unroll
        for (int vt = 0; vt < KM; ++vt)
            if (vt < VT) {
                const f32x4 s0 = fc_across(st + (vt * KT + w) * 256), d1 = fc_across(ds + (vt * KT + w) * 256);
                const f32x4 d = *reinterpret_cast<const f32x4 *>(&sm.dl[n * LD + 16 * vt + 4 * g]);
                const f32x4 r = *reinterpret_cast<const f32x4 *>(&sm.dr[n * LD + 16 * vt + 4 * g]);
                Qg = fc_mma4(yf[vt], s0, Qg);
                Ag = fc_mma4(-r, s0, Ag);
                Kg = fc_mma4(d, d1, Kg);
#pragma unroll
                for (int i = 0; i < 4; ++i) fs += s0[i] * d1[i];
            }
        fs = fc_group_sum(fs);
    }
    __syncthreads();
    if (w >= KT) return;
    k = fc_keep4(k, on4);
    q = fc_keep4(q, on4);
    e = fc_keep4(e, on4);
#pragma unroll
    for (int i = 0; i < 4; ++i) al[i] = fc_gate(al[i], on4[i] > rst4[i], 1.f - on4[i], fc_least(a));
    const f32x4 eh = e * k;
    const FcCol x(al, g);
    const f32x4 f8 = x.f4 * x.uf4(), g8 = x.g4 * x.ug4();
    // Levels: column t quad n / 4 and row s quad g (m0, m1), row t quad g and column
    // s quad n / 4 (m2, m3).
    const int n4 = n >> 2;
    const bool c4 = (n4 & 1) && g == n4 - 1, c8 = n4 >= 2 && g < 2, r4 = (g & 1) && n4 == g - 1, r8 = g >= 2 && n4 < 2;
    f32x4 e4, e8, p4, p8, k4, k8;
    {
        const f32x4 m0 = sm.m[0][l], m1 = sm.m[1][l], m2 = sm.m[2][l], m3 = sm.m[3][l];
        const f32x4 kg4 = k * x.g4, kg8 = k * g8, ef4 = eh * x.f4, ef8 = eh * f8, qf4 = q * x.f4, qf8 = q * f8;
        p4 = fc_mma4(fc_keep(m0, c4), kg4, zero4());
        e4 = fc_mma4(fc_keep(m1, c4), kg4, zero4());
        p8 = fc_mma4(fc_keep(m0, c8), kg8, zero4());
        e8 = fc_mma4(fc_keep(m1, c8), kg8, zero4());
        k4 = fc_mma4(fc_keep(m3, r4), ef4, fc_mma4(fc_keep(m2, r4), qf4, zero4()));
        k8 = fc_mma4(fc_keep(m3, r8), ef8, fc_mma4(fc_keep(m2, r8), qf8, zero4()));
    }
    f32x4 eA = x.f4 * e4 + f8 * e8, qP = x.f4 * p4 + f8 * p8, kAP = x.g4 * k4 + g8 * k8;
    // the pairs inside the lane's four tokens, and their terms of dalpha
    f32x4 da = zero4();
    {
        const float *pp = &sm.p[0][4 * g * LM + 4 * g], *pa = &sm.p[1][4 * g * LM + 4 * g];
        float cc[4][4];
#pragma unroll
        for (int t = 0; t < 4; ++t) {
            const f32x4 rp = *reinterpret_cast<const f32x4 *>(pp + t * LM), ra = *reinterpret_cast<const f32x4 *>(pa + t * LM);
            qP[t] += rp[t] * k[t];
            kAP[t] += rp[t] * q[t];
            float d = 1.f;
#pragma unroll
            for (int u = 2; u >= 0; --u) {
                if (u >= t) continue;
                d *= al[u + 1];
                const float y = d * k[u], z = ra[u] * eh[t] + rp[u] * q[t];
                eA[t] += ra[u] * y;
                qP[t] += rp[u] * y;
                kAP[u] += z * d;
                cc[t][u] = z * k[u];
            }
        }
        da[1] = cc[1][0] + al[2] * (cc[2][0] + al[3] * cc[3][0]);
        da[2] = cc[2][1] + al[1] * cc[2][0] + al[3] * (cc[3][1] + al[1] * cc[3][0]);
        da[3] = cc[3][2] + al[2] * (cc[3][1] + al[1] * cc[3][0]);
    }
    {  // adjoints of F and G, from the whole chunk down to four tokens
        f32x4 aF = eh * Ag + q * Qg, aG = k * Kg;  // of b and lam
        if (g == 3) aF[3] += fs;
        float z = 0.f;
#pragma unroll
        for (int i = 0; i < 4; ++i) z += g >= 2 ? aF[i] * f8[i] : aG[i] * g8[i];
        z += __shfl_xor(z, 16);
        const float a8 = __shfl_xor(z, 32);  // of this eight's whole product
        aF = aF * x.uf8() + eh * e8 + q * p8;
        aG = aG * x.ug8() + k * k8;
        z = 0.f;
#pragma unroll
        for (int i = 0; i < 4; ++i) z += (g & 1) ? aF[i] * x.f4[i] : aG[i] * x.g4[i];
        const float a4 = __shfl_xor(z, 16) + a8 * x.x4;  // of this quad's whole product
        aF = aF * x.uf4() + eh * e4 + q * p4;
        aG = aG * x.ug4() + k * k4;
        aF[3] += a4;
        da[3] += aF[3] * x.f4[2];
        float y = aF[2] + aF[3] * al[3];
        da[2] += y * x.f4[1];
        y = aF[1] + y * al[2];
        da[1] += y * x.f4[0];
        da[0] = aF[0] + y * al[1];
        da[1] += aG[0] * x.g4[1];
        y = aG[1] + aG[0] * al[1];
        da[2] += y * x.g4[2];
        da[3] += aG[2] + y * al[2];
    }
    const f32x4 bt = f8 * x.uf8(), lam = g8 * x.ug8();
    const f32x4 deh = bt * Ag + eA;
    if (s.dq) fc_put<BF, VEC>(s.dq, BF, s, b, h, c, K, w, fc_keep4(bt * Qg + qP, on4));
    if (s.dk) fc_put<BF, VEC>(s.dk, BF, s, b, h, c, K, w, fc_keep4(lam * Kg + kAP + e * deh + ck4 * k, on4));
    if (s.derase) fc_put<false, VEC>(s.derase, 0, s, b, h, c, K, w, fc_keep4(k * deh, on4));
    if (s.dalpha) {
#pragma unroll
        for (int i = 0; i < 4; ++i) da[i] = rst4[i] != 0.f ? 0.f : da[i];
        fc_put<false, VEC>(s.dalpha, 0, s, b, h, c, K, w, fc_keep4(da, on4));
    }
}

// ---- launches -------------------------------------------------------------------
template <bool BF, bool VEC>
static void fc_prep(const FcArgs &a, hipStream_t stream) {
    const int KT = fc_kp(a.s.K) / 16, VT = (a.s.V + 15) / 16;
    hipLaunchKernelGGL((fc_prep_kernel<BF, VEC>), dim3(a.s.B * a.s.H * a.nc), dim3(64 * std::max(KT, VT)), 0, stream, a);
}
template <int KM, bool BF, bool VEC>
static void fc_bgrad(const FcArgs &a, hipStream_t stream) {
    const int KT = fc_kp(a.s.K) / 16, VT = (a.s.V + 15) / 16;
    hipLaunchKernelGGL((fc_bgrad_kernel<KM, BF, VEC>), dim3(a.s.B * a.s.H * a.nc), dim3(64 * (KT > VT ? KT : VT)), 0,
                       stream, a);
}
template <int KM>
static void fc_out(const FcArgs &a, hipStream_t stream) {
    const dim3 grid(a.s.B * a.s.H * a.nc), block(64 * ((a.s.V + 15) / 16));
    if (a.vec) hipLaunchKernelGGL((fc_out_kernel<KM, true>), grid, block, 0, stream, a);
    else hipLaunchKernelGGL((fc_out_kernel<KM, false>), grid, block, 0, stream, a);
}

void launch_fc_out(const FcArgs &a, hipStream_t stream) {
    const int KT = fc_kp(a.s.K) / 16;
    if (KT <= 2) fc_out<2>(a, stream);
    else if (KT <= 4) fc_out<4>(a, stream);
    else fc_out<8>(a, stream);
}

template <bool REV, bool BF, bool VEC, bool SC>
static void fc_scan(const FcArgs &a, hipStream_t stream) {
    const int bh = a.s.B * a.s.H, VT = (a.s.V + 15) / 16, KT = fc_kp(a.s.K) / 16;
    const dim3 grid(8 * VT * ((bh + 7) / 8)), block(64 * KT);
#define FC_SCAN(N)                                                                                        \
    case N: hipLaunchKernelGGL((fc_scan_kernel<N, REV, BF, VEC, SC>), grid, block, 0, stream, a); break
    switch (KT) {
        FC_SCAN(1);
        FC_SCAN(2);
        FC_SCAN(3);
        FC_SCAN(4);
        FC_SCAN(5);
        FC_SCAN(6);
        FC_SCAN(7);
        FC_SCAN(8);
    }
#undef FC_SCAN
}

void launch_fc_scan(const FcArgs &a, hipStream_t stream) { fc_scan<false, false, false, false>(a, stream); }

template <bool SC>
static void fc_adjoint(const FcArgs &a, hipStream_t stream) {
    if (a.in_bf16 && a.vec) fc_scan<true, true, true, SC>(a, stream);
    else if (a.in_bf16) fc_scan<true, true, false, SC>(a, stream);
    else if (a.vec) fc_scan<true, false, true, SC>(a, stream);
    else fc_scan<true, false, false, SC>(a, stream);
}

void launch_fc_adjoint(const FcArgs &a, hipStream_t stream) {
    if (!a.s.dscores) return fc_adjoint<false>(a, stream);
    hipLaunchKernelGGL(fc_score_kernel, dim3(a.s.B * a.s.H * a.wn), dim3(64), 0, stream, a);
    fc_adjoint<true>(a, stream);
}

hipError_t launch_fc_fwd(const FcArgs &a, hipStream_t stream, const hipEvent_t *ev) {
    fc_mark(ev, 0, stream);
    if (a.in_bf16 && a.vec) fc_prep<true, true>(a, stream);
    else if (a.in_bf16) fc_prep<true, false>(a, stream);
    else if (a.vec) fc_prep<false, true>(a, stream);
    else fc_prep<false, false>(a, stream);
    fc_mark(ev, 1, stream);
    fc_mark(ev, 2, stream);
    launch_fc_scan(a, stream);
    fc_mark(ev, 3, stream);
    fc_mark(ev, 4, stream);
    launch_fc_out(a, stream);
    fc_mark(ev, 5, stream);
    return hipGetLastError();
}

hipError_t launch_fc_bwd(const FcArgs &a, hipStream_t stream, const hipEvent_t *ev) {
    fc_mark(ev, 0, stream);  // no prep stage: the adjoint scan forms its map's terms
    fc_mark(ev, 1, stream);
    fc_mark(ev, 2, stream);
    launch_fc_adjoint(a, stream);
    fc_mark(ev, 3, stream);
    fc_mark(ev, 4, stream);
    FC_DISPATCH(std::max(fc_kp(a.s.K), (a.s.V + 15) & ~15) / 16, fc_bgrad, a, stream);
    fc_mark(ev, 5, stream);
    return hipGetLastError();
}

}  // namespace gdn2
