// Chunked scalar-gate gated delta rule in f32 on gfx950: alpha = exp(g) on every
// key channel and erase = write = beta, for every d_k, d_v <= 128 (f32 q/k/v, or
// bf16 read as its exact f32 values), in 16-token chunks.
//
// The recurrence and its chunk form are those of gdn2_chunk_f32.hip with one
// decay per token, so the pair decays D_ts = prod_{s < u <= t} a_u leave the
// channel sums: A = strict_lower(beta D KK^T), P = lower(D QK^T), and every
// product of the forward and the backward is a 16 x 16 matrix product.  a_u is
// exp(g_u), 1 on padding and 0 on a reset, and D, b_t = D from the chunk start
// and lam_s = D to the chunk end are direct products, so an underflowed decay
// needs no special case.  The map's factors, the states, the scans and out are
// gdn2_chunk_f32.hip's; prep and bgrad are here.
//
// A chunk's products multiply the terms past a token by zero, so a NaN or an
// infinity at one token reaches the other tokens of its chunk, on both sides, which
// the recurrence does not.  Out and bgrad therefore mark every (batch, head) that
// gave a value that is not finite, and the token-sequential kernels (gdn2_seq.hip),
// launched behind them, walk the marked ones again (the rest return at once): such
// a sequence gets what the recurrence gives, token by token.
//
// At B8 T512 H8 K = V = 64 in f32, forward + backward takes 126 us of kernels
// (prep 18, scans 20 and 29, out 11, bgrad 44, the two launches for marked heads
// 2 each) against 885 us of the token-sequential kernels, which walk a head's tokens
// in one workgroup (forward 226, backward 658); the floor of its 69 MB is 14 us.
#include "gdn2_chunk_f32_dev.h"

#include <algorithm>

namespace gdn2 {

namespace {

// The decays are formed in f64 and rounded once.  One decay serves every channel
// of a head, so its rounding does not average out over the channel sums, as the
// token walk's does: f32 products were the largest term of the outputs' error
// (1.6e-7 of 2.5e-7 at 64 x 64, in an emulation of the sums).
__device__ __forceinline__ double fs_join(int hi, int lo) {
    return __builtin_bit_cast(double, ((uint64_t)(uint32_t)hi << 32) | (uint32_t)lo);
}
__device__ __forceinline__ int fs_hi(double x) { return (int)(__builtin_bit_cast(uint64_t, x) >> 32); }
__device__ __forceinline__ int fs_lo(double x) { return (int)__builtin_bit_cast(uint64_t, x); }
template <int CTRL>  // x of the lane that CTRL names within the 16-lane row, 1 past its start
__device__ __forceinline__ double fs_shifted(double x) {
    return fs_join(__builtin_amdgcn_update_dpp(fs_hi(1.), fs_hi(x), CTRL, 0xF, 0xF, false),
                   __builtin_amdgcn_update_dpp(0, fs_lo(x), CTRL, 0xF, 0xF, false));
}
// Inclusive product over the tokens of lanes 0 .. n of a 16-lane row.
__device__ __forceinline__ double fs_scan_mul(double x) {
    x *= fs_shifted<0x111>(x);
    x *= fs_shifted<0x112>(x);
    x *= fs_shifted<0x114>(x);
    return x * fs_shifted<0x118>(x);
}

// D_ts at t = 4 g + i, s = n (t >= s, else unspecified), and lam_n = D_15,n.
__device__ __forceinline__ f32x4 fs_decay_rows(double a, int g, int n, float &lam) {
    f32x4 d = zero4();
    double p = 0.;
#pragma unroll
    for (int t = 0; t < C; ++t) {
        const double at = fs_join(__builtin_amdgcn_readlane(fs_hi(a), t), __builtin_amdgcn_readlane(fs_lo(a), t));
        p = t == n ? 1. : p * at;
        if ((t >> 2) == g) d[t & 3] = (float)p;
    }
    lam = (float)p;
    return d;
}

template <int KM>
struct FsGradSmem {
    static constexpr int LD = 16 * KM + 4;  // f32 row stride: rows 4 banks apart
    float dr[C * LD], dl[C * LD];           // [token][value]
    f32x4 m[4][64];                         // the decayed adjoint tiles, one 16-byte piece per lane
    f32x4 e[2][64];                         // E's two terms, in acc layout
    float vd[KM][C], ys[KM][C], zs[KM][C], kd[KM][C], fr[KM];
};

}  // namespace

// ---- prep: T, P, D and the factored map, one wave per chunk ---------------------
template <int KM, bool BF, bool VEC>
__global__ void __launch_bounds__(64) fs_prep_kernel(FcArgs a) {
    __shared__ __align__(16) float la[C * FC_LA];
    const SeqArgs &s = a.s;
    const int64_t ci = blockIdx.x;
    const int bh = blockIdx.x / a.nc, c = blockIdx.x % a.nc, b = bh / s.H, h = bh % s.H;
    const int K = s.K, V = s.V, KP = fc_kp(K), KT = KP >> 4, VT = (V + 15) >> 4;
    const int l = lane_id(), g = l >> 4, n = l & 15, tg = c * C + n;
    const FcSrc<BF, VEC> sk(s.k, b, h, c, s.T, K), sq(s.q, b, h, c, s.T, K), sv(s.v, b, h, c, s.T, V);
    if (c == 0 && l == 0) a.bad[bh] = 0;
    bool on, rst;
    fc_flags(s, b, c, on, rst);
    const int tc = min(tg, s.T - 1);
    const float bv = ld4<float>(s.beta, b, tc, h, 0), gl = ld4<float>(s.g, b, tc, h, 0);
    const float beta = on ? bv : 0.f;
    const double av = on ? (rst ? 0. : exp((double)gl)) : 1.;
    const f32x4 on4 = fc_rows(on ? 1.f : 0.f, g);
    f32x4 kb[KM], qb[KM], kk[KM], qk[KM], ksq4 = zero4();
    float lam;
    const f32x4 d = fs_decay_rows(av, g, n, lam);
    const FcOff oc(C);
#pragma unroll
    for (int tau = 0; tau < KM; ++tau) {
        // Past the last key tile (vector reads) the last tile is read again and
        // zeroed, so that no load of the chunk waits behind a branch.
        const int tt = VEC ? min(tau, KT - 1) : tau;
        const bool in = tau < KT;
        const f32x4 kf = fc_keep(sk.frag(tt), on && in), qf = fc_keep(sq.frag(tt), on && in);
        kb[tau] = fc_keep4(sk.col(tt), on4);
        qb[tau] = fc_keep4(sq.col(tt), on4);
        kk[tau] = fc_mma4(kf, kf, zero4());
        qk[tau] = fc_mma4(qf, kf, zero4());  // row t = 4 g + i, column s = n
        ksq4 += kf * kf;
    }
    fc_tree(kk);
    fc_tree(qk);
    const float bn = (float)fs_scan_mul(av);
    const f32x4 be4 = fc_rows(beta, g), b4 = fc_rows(bn, g), lam4 = fc_rows(lam, g);
    f32x4 A, P, D;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        A[i] = n < 4 * g + i ? be4[i] * d[i] * kk[0][i] : 0.f;
        P[i] = n <= 4 * g + i ? d[i] * qk[0][i] : 0.f;
        D[i] = n <= 4 * g + i ? d[i] : 0.f;
    }
    const f32x4 t = fc_inverse(A, la, g, n);
    fc_p4(a.tm + ci * C * C, (n * C + 4 * g) * 4, t);
    oc.put(a.pm + ci * C * C, P);
    oc.put(a.dm + ci * C * C, D);
    const float ksq = fc_group_sum((ksq4[0] + ksq4[1]) + (ksq4[2] + ksq4[3]));
    float *gb = a.gb + ci * C * 8;
    *fc_at(gb + C * g, 4 * n) = g == 0 ? (on ? 1.f : 0.f) : (g == 1 ? (rst ? 1.f : 0.f) : (g == 2 ? ksq : beta));
    if (g < 2) *fc_at(gb + C * (4 + g), 4 * n) = g == 0 ? bn : lam;
    const float b15 = fc_lane(bn, C - 1);
    for (int i = l; i < KP; i += 64) a.gv[ci * KP + i] = b15;
    // T - I: the products with T add the rest to the operand itself, which is the
    // larger term.
    f32x4 t1 = t;
#pragma unroll
    for (int r = 0; r < 4; ++r) t1[r] = 4 * g + r == n ? 0.f : t[r];
#pragma unroll
    for (int tau = 0; tau < KM; ++tau)
        if (tau < KT) {
            const int64_t o = (ci * KT + tau) * 256;
            const f32x4 bk = b4 * be4 * kb[tau];
            fc_p4(a.fw + o, 16 * l, bk + fc_mma4(t1, bk, zero4()));
            fc_p4(a.fk + o, 16 * l, lam4 * kb[tau]);
            fc_p4(a.fq + o, 16 * l, b4 * qb[tau]);
        }
    for (int vt = 0; vt < VT; ++vt) {
        const f32x4 bv = be4 * fc_keep4(sv.col(vt), on4);
        fc_p4(a.fu + (ci * VT + vt) * 256, 16 * l, bv + fc_mma4(t1, bv, zero4()));
    }
}

// ---- bgrad: every gradient of one chunk -------------------------------------------
// With S0, delta (the forward) and dS at the chunk end (the adjoint scan):
//   ddelta = P^T dO + Ktil dS + c delta,  dR = T^T ddelta,  dv = beta dR
//   Qb = b dO S0^T,  Ab = -b dR S0^T,  Kl = lam delta dS^T
//   dA = -strict_lower(dR delta^T),  dP = lower(dO delta^T)
//   dq = Qb + (dP D) K,  deh = Ab + (dA D) K,
//   dk = Kl + beta deh + (beta dA D)^T K + (dP D)^T Q + c' k
//   dbeta = k . deh + v . dR
// and, every path of the decays through token u being a pair (lo, hi) with
// lo < u <= hi whose full product has a_u as a factor,
//   dg_u = sum_{s < u <= t} E_ts + sum_{t >= u} y_t + sum_{s < u} z_s + b_15 <S0, dS>,
//   E = beta dA D KK^T + dP P,  y_t = beta k . Ab + q . Qb,  z_s = k . Kl
// (zero on padding and resets).  Wave w takes value tile w up to dR, then key
// tile w; blockDim is 64 max(KT, VT).
template <int KM, bool BF, bool VEC>
__global__ void __launch_bounds__(64 * KM, KM == 8 ? 2 : 4) fs_bgrad_kernel(FcArgs a) {
    __shared__ FsGradSmem<KM> sm;
    constexpr int LD = FsGradSmem<KM>::LD;
    const SeqArgs &s = a.s;
    const int bh = blockIdx.x / a.wn, cw = blockIdx.x % a.wn, c = a.w0 + cw, b = bh / s.H, h = bh % s.H;
    const int64_t ci = (int64_t)bh * a.nc + c, wi = blockIdx.x;
    const int K = s.K, V = s.V, KT = fc_kp(K) >> 4, VT = (V + 15) >> 4, NW = blockDim.x >> 6;
    const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), l = lane_id(), g = l >> 4, n = l & 15, tg = c * C + n;
    const FcSrc<BF, VEC> sdo(s.dout, b, h, c, s.T, V);
    const bool has_do = s.dout.data != nullptr;
    const float bn = fc_gb(a, ci, 4), lam = fc_gb(a, ci, 5);
    const bool on = fc_gb(a, ci, 0) != 0.f;
    const f32x4 on4 = fc_gb4(a, ci, 0), be4 = fc_gb4(a, ci, 3);
    f32x4 cs4 = zero4(), ck4 = zero4();
    if (s.dscores) cs4 = fc_g4(a.sc + wi * 2 * C, 16 * g), ck4 = fc_g4(a.sc + wi * 2 * C + C, 16 * g);
    const float *st = a.st + ci * KT * VT * 256, *ds = a.ds + wi * KT * VT * 256;
    const FcOff oc(C);
    const f32x4 p = oc.get(a.pm + ci * C * C);
    if (w < VT) {  // ddelta and dR of value tile w
        const f32x4 tb = oc.get(a.tm + ci * C * C);
        const f32x4 dl = fc_g4(a.fu + (ci * VT + w) * 256, 16 * l);
        const f32x4 v = fc_keep4(FcSrc<BF, VEC>(s.v, b, h, c, s.T, V).col(w), on4);
        f32x4 dO = has_do ? sdo.col(w) : zero4(), kf[KM], dsn[KM];
        const float *fk = a.fk + ci * KT * 256;
#pragma unroll
        for (int tau = 0; tau < KM; ++tau) {
            kf[tau] = dsn[tau] = zero4();
            if (tau < KT) kf[tau] = fc_across(fk + 256 * tau), dsn[tau] = fc_g4(ds + (w * KT + tau) * 256, 16 * l);
        }
        dO = fc_keep4(dO, on4);
        const f32x4 dd = fc_mma4(p, dO, cs4 * dl) + fc_mma_tree<KM>(kf, dsn);
        f32x4 t1 = tb;  // T - I, as in prep
#pragma unroll
        for (int i = 0; i < 4; ++i) t1[i] = 4 * g + i == n ? 0.f : tb[i];
        const f32x4 dr = dd + fc_mma4(t1, dd, zero4());                                          // rows t, column j
        *reinterpret_cast<f32x4 *>(&sm.dr[n * LD + 16 * w + 4 * g]) = fc_mma4(dd, tb, zero4());  // rows j, column t
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            sm.dl[(4 * g + r) * LD + 16 * w + n] = dl[r];
            const float x = fc_row_sum(v[r] * dr[r]);
            if (n == 0) sm.vd[w][4 * g + r] = x;
        }
        const f32x4 dvt = fc_keep4(be4 * dr, on4);
        if (s.dv) fc_put<BF, VEC>(s.dv, BF, s, b, h, c, V, w, dvt);
        if (!fc_finite(dvt)) a.wbad[bh] = 1;
    }
    f32x4 yf[KM];  // dO rows
#pragma unroll
    for (int vt = 0; vt < KM; ++vt) yf[vt] = (has_do && vt < VT) ? fc_keep(sdo.frag(vt), on) : zero4();
    f32x4 kb = zero4(), qb = zero4();
    if (w < KT) {
        kb = fc_keep4(FcSrc<BF, VEC>(s.k, b, h, c, s.T, K).col(w), on4);
        qb = fc_keep4(FcSrc<BF, VEC>(s.q, b, h, c, s.T, K).col(w), on4);
    }
    __syncthreads();
    // The decayed adjoint tiles: 0 dP D and 1 dA D with column t (row s), 2 dP D
    // and 3 beta dA D with column s (row t); with the last two, E's terms.
    for (int x = w; x < 4; x += NW) {
        f32x4 mv[KM];
#pragma unroll
        for (int vt = 0; vt < KM; ++vt) {
            mv[vt] = zero4();
            if (vt < VT) {
                const f32x4 d = *reinterpret_cast<const f32x4 *>(&sm.dl[n * LD + 16 * vt + 4 * g]);
                const f32x4 y = (x & 1) ? -*reinterpret_cast<const f32x4 *>(&sm.dr[n * LD + 16 * vt + 4 * g]) : yf[vt];
                mv[vt] = x < 2 ? fc_mma4(d, y, zero4()) : fc_mma4(y, d, zero4());
            }
        }
        fc_tree(mv);
        const f32x4 m = mv[0];
        const float *dm = a.dm + ci * C * C;
        const f32x4 d = x < 2 ? fc_g4(dm, (n * C + 4 * g) * 4) : oc.get(dm);  // zero above the diagonal
        f32x4 md = m * d;
        if (x & 1)
#pragma unroll
            for (int i = 0; i < 4; ++i) md[i] = 4 * g + i == n ? 0.f : md[i];
        if (x == 2) {
            f32x4 e = m * p;
#pragma unroll
            for (int i = 0; i < 4; ++i) e[i] = 4 * g + i == n ? 0.f : e[i];
            sm.e[0][l] = e;
        }
        if (x == 3) {
            md = md * be4;
            const FcSrc<BF, VEC> sk(s.k, b, h, c, s.T, K);
            f32x4 kk[KM];
#pragma unroll
            for (int tau = 0; tau < KM; ++tau) {
                kk[tau] = zero4();
                if (tau < KT) {
                    const f32x4 kf = fc_keep(sk.frag(tau), on);
                    kk[tau] = fc_mma4(kf, kf, kk[tau]);
                }
            }
            fc_tree(kk);
            sm.e[1][l] = md * kk[0];
        }
        sm.m[x][l] = md;
    }
    f32x4 Qb[4], Ab[4], Kl[4];  // rows t, column key 16 w + n: four partial sums
#pragma unroll
    for (int i = 0; i < 4; ++i) Qb[i] = Ab[i] = Kl[i] = zero4();
    float fr = 0.f;
    if (w < KT)
#pragma unroll
        for (int vt = 0; vt < KM; ++vt)
            if (vt < VT) {
                const f32x4 s0 = fc_across(st + (vt * KT + w) * 256), d1 = fc_across(ds + (vt * KT + w) * 256);
                const f32x4 d = *reinterpret_cast<const f32x4 *>(&sm.dl[n * LD + 16 * vt + 4 * g]);
                const f32x4 r = *reinterpret_cast<const f32x4 *>(&sm.dr[n * LD + 16 * vt + 4 * g]);
                Qb[vt & 3] = fc_mma4(bn * yf[vt], s0, Qb[vt & 3]);
                Ab[vt & 3] = fc_mma4(-bn * r, s0, Ab[vt & 3]);
                Kl[vt & 3] = fc_mma4(lam * d, d1, Kl[vt & 3]);
#pragma unroll
                for (int i = 0; i < 4; ++i) fr += s0[i] * d1[i];
            }
    fc_tree(Qb);
    fc_tree(Ab);
    fc_tree(Kl);
    fr = fc_group_sum(fc_row_sum(fr));
    if (l == 0) sm.fr[w] = fr;
    __syncthreads();
    if (w < KT) {
        const f32x4 dq = Qb[0] + fc_mma4(sm.m[0][l], kb, zero4()), de = Ab[0] + fc_mma4(sm.m[1][l], kb, zero4());
        const f32x4 dk = Kl[0] + (fc_mma4(sm.m[2][l], qb, zero4()) + fc_mma4(sm.m[3][l], kb, zero4()));
        const f32x4 dqt = fc_keep4(dq, on4), dkt = fc_keep4(dk + be4 * de + ck4 * kb, on4);
        if (s.dq) fc_put<BF, VEC>(s.dq, BF, s, b, h, c, K, w, dqt);
        if (s.dk) fc_put<BF, VEC>(s.dk, BF, s, b, h, c, K, w, dkt);
        if (!fc_finite(dqt + dkt)) a.wbad[bh] = 1;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const float ys = fc_row_sum(be4[i] * kb[i] * Ab[0][i] + qb[i] * Qb[0][i]);
            const float zs = fc_row_sum(kb[i] * Kl[0][i]), kd = fc_row_sum(kb[i] * de[i]);
            if (n == 0) sm.ys[w][4 * g + i] = ys, sm.zs[w][4 * g + i] = zs, sm.kd[w][4 * g + i] = kd;
        }
    }
    float wu = 0.f;
    if (w == 0) {  // lane (g, n): sum_{s < n <= t} E_ts
        const f32x4 e = sm.e[0][l] + sm.e[1][l];
#pragma unroll
        for (int u = 1; u < C; ++u) {
            float x = 0.f;
#pragma unroll
            for (int i = 0; i < 4; ++i) x += 4 * g + i >= u ? e[i] : 0.f;
            x = fc_row_sum(n < u ? x : 0.f);
            if (u == n) wu = x;
        }
        wu = fc_group_sum(wu);
    }
    __syncthreads();
    if (threadIdx.x < C && tg < s.T) {
        double db = 0., dg = wu, f = 0.;  // one thread a token, a term for every tile
        for (int x = 0; x < VT; ++x) db += sm.vd[x][n];
        for (int x = 0; x < KT; ++x) {
            db += sm.kd[x][n];
#pragma unroll
            for (int u = 0; u < C; ++u) dg += u >= n ? sm.ys[x][u] : sm.zs[x][u];
        }
        for (int x = 0; x < NW; ++x) f += sm.fr[x];
        dg += fc_lane(bn, C - 1) * f;
        const int64_t o = ((int64_t)b * s.T + tg) * s.H + h;
        if (s.dbeta) s.dbeta[o] = on ? (float)db : 0.f;
        if (s.dg) s.dg[o] = (on && fc_gb(a, ci, 1) == 0.f) ? (float)dg : 0.f;
        if (on && !(db - db == 0. && dg - dg == 0.)) a.wbad[bh] = 1;
    }
}

template <int KM, bool BF, bool VEC>
static void fs_prep(const FcArgs &a, hipStream_t stream) {
    hipLaunchKernelGGL((fs_prep_kernel<KM, BF, VEC>), dim3(a.s.B * a.s.H * a.nc), dim3(64), 0, stream, a);
}
template <int KM, bool BF, bool VEC>
static void fs_bgrad(const FcArgs &a, hipStream_t stream) {
    const int KT = fc_kp(a.s.K) / 16, VT = (a.s.V + 15) / 16;
    hipLaunchKernelGGL((fs_bgrad_kernel<KM, BF, VEC>), dim3(a.s.B * a.s.H * a.wn), dim3(64 * (KT > VT ? KT : VT)), 0,
                       stream, a);
}

// The token walk of the marked (batch, head)s on this call's checkpoint.
static SeqArgs fs_walk(const FcArgs &a, const int *marked) {
    SeqArgs s = a.s;
    s.st = a.st;
    s.fu = a.fu;
    s.only = marked;
    return s;
}

hipError_t launch_fs_fwd(const FcArgs &a, hipStream_t stream, const hipEvent_t *ev) {
    fc_mark(ev, 0, stream);
    FC_DISPATCH(fc_kp(a.s.K) / 16, fs_prep, a, stream);
    fc_mark(ev, 1, stream);
    fc_mark(ev, 2, stream);
    launch_fc_scan(a, stream);
    fc_mark(ev, 3, stream);
    fc_mark(ev, 4, stream);
    launch_fc_out(a, stream);
    fc_mark(ev, 5, stream);
    return launch_seq_fwd(fs_walk(a, a.bad), a.in_bf16, stream);
}

hipError_t launch_fs_bwd(const FcArgs &whole, size_t ws_bytes, hipStream_t stream, const hipEvent_t *ev) {
    FcArgs a = whole;
    const int bh = a.s.B * a.s.H, VT = (a.s.V + 15) / 16, KT = fc_kp(a.s.K) / 16;
    // Chunk windows, last first: as many chunks as the workspace holds, the
    // adjoint between two windows in the carry.
    const int64_t state = (int64_t)KT * VT * 256, carry = bh * state * 4, per = bh * fc_ws_chunk(a.s.K, a.s.V) * 4;
    const int64_t words = fc_word_bytes(a.s.B, a.s.H);
    const int64_t room = ((int64_t)ws_bytes - words) & ~(int64_t)15;  // the words lie behind it
    int64_t wn = room / per;
    if (wn < a.nc) wn = (room - carry) / per;
    if (wn < 1 || room < (int64_t)seq_workspace_floats(a.s.B, a.s.H, a.s.K, a.s.V) * 4) return hipErrorInvalidValue;
    a.wbad = reinterpret_cast<int *>(reinterpret_cast<char *>(a.ds) + room);
    wn = std::min<int64_t>(wn, a.nc);
    a.sc = a.ds + wn * bh * state;
    a.carry = a.sc + wn * bh * 2 * C;
    for (int end = a.nc; end > 0; end = a.w0) {
        a.wn = (int)std::min<int64_t>(end, wn);
        a.w0 = end - a.wn;
        const hipEvent_t *e = end == a.nc ? ev : nullptr;
        fc_mark(e, 0, stream);
        fc_mark(e, 1, stream);
        fc_mark(e, 2, stream);
        launch_fc_adjoint(a, stream);
        fc_mark(e, 3, stream);
        fc_mark(e, 4, stream);
        FC_DISPATCH(std::max(KT, VT), fs_bgrad, a, stream);
        fc_mark(e, 5, stream);
    }
    SeqArgs walk = fs_walk(a, a.wbad);
    walk.replay = a.ds;  // the windows are done with it
    return launch_seq_bwd(walk, a.in_bf16, stream);
}

}  // namespace gdn2
