// Chunked scalar-gate gated delta rule in f32 on gfx950: alpha = exp(g) on every
// key channel and erase = write = beta, for every d_k, d_v <= 128 (f32 q/k/v, or
// bf16 read as its exact f32 values), in 16-token chunks.
//
// The recurrence and its chunk form are those of gdn2_chunk_f32.hip with one
// decay per token, so the pair decays D_ts = prod_{s < u <= t} a_u leave the
// channel sums: A = strict_lower(beta D KK^T), P = lower(D QK^T), and every
// product of the forward and the backward is a matrix product on
// v_mfma_f32_16x16x4f32 (exact f32 products).  a_u is exp(g_u), 1 on padding
// and 0 on a reset, and D, b_t = D from the chunk start and lam_s = D to the
// chunk end are direct products, so an underflowed decay needs no special case.
//
// The map's factors, the states and the scans are gdn2_chunk_f32.hip's
// (FcArgs); the forward scan leaves the chunk's edits delta = U - W' S0 where U
// was, so the out kernel forms neither R nor T R.
//
// Layout.  A 16-token chunk is one MFMA tile, and no product is transposed
// through LDS where an operand layout can be read instead.  With l = 16 g + n:
//   row fragment  xf[tau][r] = x[token n][16 tau + 4 g + r]   (one 16-byte load)
//     is the A operand of x Y^T and the B operand of Y x^T, reduction over channels
//   tile column   xb[q] = x[token 4 g + q][16 tau + n]
//     is the B operand of M x and the A operand of x^T Y, reduction over tokens
//   accumulator   rows 4 g + i, column n: register i is also an A or B operand
//     whose reduction slice is {4 g + i}, so products chain in registers.
// A tile-packed state (16-byte piece per lane) is a B operand as it was loaded.
// A wave owns a chunk (prep) or one 16-column tile of a chunk (the others); the
// 16 x 16 decay and score tiles are formed again by each wave, which costs less
// than a barrier to share them.
//
// At B8 T512 H8 K = V = 64 in f32, forward + backward takes 187 us (prep 17,
// scans 23 and 21, out 19, bprep 25, bgrad 65) against 885 us of the
// token-sequential kernels, which walk a head's tokens in one workgroup
// (forward 226, backward 658); the floor of its 69 MB is 14 us.  The scans are
// bound by the bytes they stream (26 KiB per chunk and head), bprep and bgrad by
// issue: 64 and 31 f32 MFMAs of 32 cycles per wave and the loads that feed them.
#include "gdn2_chunk_f32.h"
#include "gdn2_mfma.h"

namespace gdn2 {

namespace {

constexpr int C = FC_C;

template <int CTRL>
__device__ __forceinline__ float fs_dpp(float x) {
    return x + __builtin_bit_cast(
                   float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, x), CTRL, 0xF, 0xF, false));
}
// Sum over the 16 lanes n of a lane group, in all of them.
__device__ __forceinline__ float fs_row_sum(float x) {
    return fs_dpp<0x140>(fs_dpp<0x141>(fs_dpp<0x4E>(fs_dpp<0xB1>(x))));
}
// Sum over the four lane groups g, in all of them.
__device__ __forceinline__ float fs_group_sum(float x) {
    x += __shfl_xor(x, 16);
    return x + __shfl_xor(x, 32);
}
__device__ __forceinline__ float fs_lane(float x, int i) {
    return __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, x), i));
}
__device__ __forceinline__ f32x4 fs_mma(float a, float b, f32x4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
}
__device__ __forceinline__ f32x4 fs_rows(float x, int g) {  // rows 4 g + i of a per-token value (lane n: token n)
    return f32x4{__shfl(x, 4 * g), __shfl(x, 4 * g + 1), __shfl(x, 4 * g + 2), __shfl(x, 4 * g + 3)};
}
__device__ __forceinline__ f32x4 fs_keep(f32x4 x, bool on) { return on ? x : zero4(); }

// The chunk's tokens: lane (g, n) holds token n.
struct FsTok {
    float a;     // decay: exp(g), 1 on padding, 0 on a reset
    float beta;  // 0 on padding
    float on;    // 1 on a valid token of the sequence
    float rst;   // 1 on a valid reset
};

__device__ __forceinline__ FsTok fs_tok(const SeqArgs &s, int b, int h, int c) {
    const int n = lane_id() & 15, tg = c * C + n;
    float v = 0.f, r = 0.f, be = 0.f, g = 0.f;
    if (tg < s.T) {
        v = ld4<float>(s.valid, b, tg, 0, 0);
        r = ld4<float>(s.reset, b, tg, 0, 0);
        be = ld4<float>(s.beta, b, tg, h, 0);
        g = ld4<float>(s.g, b, tg, h, 0);
    }
    const bool on = v != 0.f, rs = on && r != 0.f;
    return FsTok{on ? (rs ? 0.f : expf(g)) : 1.f, on ? be : 0.f, on ? 1.f : 0.f, rs ? 1.f : 0.f};
}

// D_ts at t = 4 g + i, s = n (t >= s, else unspecified), and lam_n = D_15,n.
__device__ __forceinline__ f32x4 fs_decay_rows(float a, int g, int n, float &lam) {
    f32x4 d = zero4();
    float p = 0.f;
#pragma unroll
    for (int t = 0; t < C; ++t) {
        p = t == n ? 1.f : p * fs_lane(a, t);
        if ((t >> 2) == g) d[t & 3] = p;
    }
    lam = p;
    return d;
}
// D_ts at t = n, s = 4 g + i (s <= t, else unspecified).
__device__ __forceinline__ f32x4 fs_decay_cols(float a, int g, int n) {
    f32x4 d = zero4();
    float p = 0.f;
#pragma unroll
    for (int s = C - 1; s >= 0; --s) {
        p = s == n ? 1.f : (s < C - 1 ? p * fs_lane(a, s + 1) : 0.f);
        if ((s >> 2) == g) d[s & 3] = p;
    }
    return d;
}
// b_n = prod_{u <= n} a_u.
__device__ __forceinline__ float fs_decay_start(float a, int n) {
    float p = 1.f;
#pragma unroll
    for (int u = 0; u < C; ++u) p = u <= n ? p * fs_lane(a, u) : p;
    return p;
}

// Element and 4-channel reads of a [token][channel] input; zero past the
// sequence (in) or the width.  vec: unit channel stride, W a multiple of 4 and
// every 4-channel piece aligned to its size.
template <bool BF>
__device__ __forceinline__ float fs_ld(const View &v, int b, int t, int h, int ch, int W, bool in) {
    if (!in || ch >= W) return 0.f;
    return BF ? ld4<bf16_t>(v, b, t, h, ch) : ld4<float>(v, b, t, h, ch);
}
template <bool BF>
__device__ __forceinline__ f32x4 fs_ld4(const View &v, bool vec, int b, int t, int h, int ch, int W, bool in) {
    if (!in || ch >= W) return zero4();
    if (vec) {
        const int64_t o = b * v.s0 + t * v.s1 + h * v.s2 + ch;
        if (BF) {
            const uint2 x = *reinterpret_cast<const uint2 *>(reinterpret_cast<const bf16_t *>(v.data) + o);
            return f32x4{__uint_as_float(x.x << 16), __uint_as_float(x.x & 0xffff0000u), __uint_as_float(x.y << 16),
                         __uint_as_float(x.y & 0xffff0000u)};
        }
        return *reinterpret_cast<const f32x4 *>(reinterpret_cast<const float *>(v.data) + o);
    }
    f32x4 x;
#pragma unroll
    for (int r = 0; r < 4; ++r) x[r] = fs_ld<BF>(v, b, t, h, ch + r, W, true);
    return x;
}

// Row fragments of the chunk's tokens (KM tiles at most; not masked).
template <int KM, bool BF>
__device__ __forceinline__ void fs_frags(f32x4 (&f)[KM], const View &v, bool vec, int b, int h, int c, int T, int W) {
    const int l = lane_id(), g = l >> 4, tg = c * C + (l & 15);
#pragma unroll
    for (int tau = 0; tau < KM; ++tau) f[tau] = fs_ld4<BF>(v, vec, b, tg, h, 16 * tau + 4 * g, W, tg < T);
}
// Tile column 16 tau + n of tokens 4 g + q, zero on padding.
template <bool BF>
__device__ __forceinline__ f32x4 fs_col(const View &v, int b, int h, int c, int tau, int T, int W, f32x4 on4) {
    const int l = lane_id(), g = l >> 4;
    f32x4 x;
#pragma unroll
    for (int q = 0; q < 4; ++q) {
        const int tg = c * C + 4 * g + q;
        const float y = fs_ld<BF>(v, b, tg, h, 16 * tau + (l & 15), W, tg < T);
        x[q] = on4[q] != 0.f ? y : 0.f;
    }
    return x;
}

template <int KM>
__device__ __forceinline__ f32x4 fs_dot(const f32x4 (&x)[KM], const f32x4 (&y)[KM]) {
    f32x4 acc = zero4();
#pragma unroll
    for (int tau = 0; tau < KM; ++tau)
#pragma unroll
        for (int r = 0; r < 4; ++r) acc = fs_mma(x[tau][r], y[tau][r], acc);
    return acc;
}

// Score adjoint coefficients of token n: c = dscore |k| / |delta| and
// c' = dscore |delta| / |k| (zero at a zero edit or key).  ksq: |k_n|^2.
__device__ void fs_score_adj(const FcArgs &a, int64_t ci, int b, int h, int c, int VT, float on, float ksq, float &cs,
                             float &ck) {
    const SeqArgs &s = a.s;
    const int l = lane_id(), n = l & 15, tg = c * C + n;
    f32x4 d2 = zero4();
    for (int vt = 0; vt < VT; ++vt) {
        const f32x4 d = *reinterpret_cast<const fc_u4 *>(&a.fu[((ci * VT + vt) * 64 + l) * 4]);
        d2 += d * d;
    }
#pragma unroll
    for (int i = 0; i < 4; ++i) d2[i] = fs_row_sum(d2[i]);
    float dsq = 0.f;  // token n's sum sits in group n / 4, register n % 4
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const float x = __shfl(d2[i], 16 * (n >> 2));
        if ((n & 3) == i) dsq = x;
    }
    const float nk = sqrtf(ksq), nd = sqrtf(dsq);
    const float dsc = tg < s.T ? s.dscores[((int64_t)b * s.T + tg) * s.H + h] : 0.f;
    const bool ok = on != 0.f && nk > 0.f && nd > 0.f;
    cs = ok ? dsc * nk / nd : 0.f;
    ck = ok ? dsc * nd / nk : 0.f;
}

template <int KM>
__device__ __forceinline__ float fs_sq(const f32x4 (&x)[KM]) {  // |x_n|^2
    float p = 0.f;
#pragma unroll
    for (int tau = 0; tau < KM; ++tau)
#pragma unroll
        for (int r = 0; r < 4; ++r) p += x[tau][r] * x[tau][r];
    return fs_group_sum(p);
}

template <int KM>
struct FsGradSmem {
    static constexpr int LD = 16 * KM + 4;  // f32 row stride: rows 4 banks apart
    float s0[16 * KM * LD], ds[16 * KM * LD];  // [key][value], zero outside K x V
    float dr[C * LD], dl[C * LD];              // [token][value]
    f32x4 m[4][64];                            // the decayed adjoint tiles, one 16-byte piece per lane
    float vd[KM][C], ys[KM][C], zs[KM][C], kd[KM][C], fr[KM];
};

}  // namespace

// ---- prep: T and the factored map, one wave per chunk ---------------------------
template <int KM, bool BF>
__global__ void __launch_bounds__(64) fs_prep_kernel(FcArgs a) {
    const SeqArgs &s = a.s;
    const int64_t ci = blockIdx.x;
    const int bh = blockIdx.x / a.nc, c = blockIdx.x % a.nc, b = bh / s.H, h = bh % s.H;
    const int K = s.K, V = s.V, KP = fc_kp(K), KT = KP >> 4, VT = (V + 15) >> 4;
    const int l = lane_id(), g = l >> 4, n = l & 15;
    f32x4 kf[KM];
    fs_frags<KM, BF>(kf, s.k, a.vec & 2, b, h, c, s.T, K);
    const FsTok tk = fs_tok(s, b, h, c);
    const f32x4 on4 = fs_rows(tk.on, g);
    f32x4 kb[KM], vb[KM];
#pragma unroll
    for (int x = 0; x < KM; ++x) {
        kb[x] = x < KT ? fs_col<BF>(s.k, b, h, c, x, s.T, K, on4) : zero4();
        vb[x] = x < VT ? fs_col<BF>(s.v, b, h, c, x, s.T, V, on4) : zero4();
    }
#pragma unroll
    for (int tau = 0; tau < KM; ++tau) kf[tau] = fs_keep(kf[tau], tk.on != 0.f);
    const f32x4 kk = fs_dot<KM>(kf, kf);
    float lam;
    const f32x4 d = fs_decay_rows(tk.a, g, n, lam);
    const float bn = fs_decay_start(tk.a, n);
    const f32x4 be4 = fs_rows(tk.beta, g), b4 = fs_rows(bn, g);
    f32x4 A;
#pragma unroll
    for (int i = 0; i < 4; ++i) A[i] = n < 4 * g + i ? be4[i] * d[i] * kk[i] : 0.f;
    // T (I + A) = I by rows: lane n keeps row n of T; from the last column on,
    // T_nq is final and leaves T_nj -= T_nq A_qj for j < q (entries above the
    // diagonal stay zero).
    float x[C];
#pragma unroll
    for (int j = 0; j < C; ++j) x[j] = j == n ? 1.f : 0.f;
#pragma unroll
    for (int q = C - 1; q > 0; --q)
#pragma unroll
        for (int j = 0; j < q; ++j) x[j] -= x[q] * fs_lane(A[q & 3], 16 * (q >> 2) + j);
    f32x4 t;
#pragma unroll
    for (int r = 0; r < 4; ++r) t[r] = g == 0 ? x[r] : (g == 1 ? x[4 + r] : (g == 2 ? x[8 + r] : x[12 + r]));
    *reinterpret_cast<fc_u4 *>(&a.tm[ci * C * C + n * C + 4 * g]) = t;
    const int64_t fo = ci * C;
    for (int i = l; i < KP; i += 64) a.gv[ci * KP + i] = fs_lane(bn, C - 1);
#pragma unroll
    for (int tau = 0; tau < KM; ++tau)
        if (tau < KT) {
            *reinterpret_cast<fc_u4 *>(&a.fk[(fo + n) * KP + 16 * tau + 4 * g]) = lam * kf[tau];
            f32x4 w = zero4();
#pragma unroll
            for (int q = 0; q < 4; ++q) w = fs_mma(t[q], b4[q] * be4[q] * kb[tau][q], w);
#pragma unroll
            for (int i = 0; i < 4; ++i) a.fw[(fo + 4 * g + i) * KP + 16 * tau + n] = w[i];
        }
#pragma unroll
    for (int vt = 0; vt < KM; ++vt)
        if (vt < VT) {
            f32x4 u = zero4();
#pragma unroll
            for (int q = 0; q < 4; ++q) u = fs_mma(t[q], be4[q] * vb[vt][q], u);
            *reinterpret_cast<fc_u4 *>(&a.fu[((ci * VT + vt) * 64 + l) * 4]) = u;
        }
}

// ---- out: O = b Q S0 + P delta and the scores, one wave per value tile -----------
template <int KM, bool BF>
__global__ void __launch_bounds__(64 * KM) fs_out_kernel(FcArgs a) {
    __shared__ float dd[KM][C];
    const SeqArgs &s = a.s;
    const int64_t ci = blockIdx.x;
    const int bh = blockIdx.x / a.nc, c = blockIdx.x % a.nc, b = bh / s.H, h = bh % s.H;
    const int K = s.K, V = s.V, KT = fc_kp(K) >> 4, VT = (V + 15) >> 4;
    const int vt = threadIdx.x >> 6, l = lane_id(), g = l >> 4, n = l & 15, j = 16 * vt + n;
    f32x4 kf[KM], qf[KM], s0[KM];
    fs_frags<KM, BF>(kf, s.k, a.vec & 2, b, h, c, s.T, K);
    fs_frags<KM, BF>(qf, s.q, a.vec & 1, b, h, c, s.T, K);
#pragma unroll
    for (int tau = 0; tau < KM; ++tau)
        s0[tau] = tau < KT ? *reinterpret_cast<const fc_u4 *>(&a.st[(((ci * VT + vt) * KT + tau) * 64 + l) * 4])
                           : zero4();
    const f32x4 dl = *reinterpret_cast<const fc_u4 *>(&a.fu[((ci * VT + vt) * 64 + l) * 4]);
    const FsTok tk = fs_tok(s, b, h, c);
    const bool on = tk.on != 0.f;
#pragma unroll
    for (int tau = 0; tau < KM; ++tau) kf[tau] = fs_keep(kf[tau], on), qf[tau] = fs_keep(qf[tau], on);
    const f32x4 qk = fs_dot<KM>(kf, qf);  // row s = 4 g + i, column t = n
    const f32x4 d = fs_decay_cols(tk.a, g, n);
    const float bn = fs_decay_start(tk.a, n);
    f32x4 o = zero4();
#pragma unroll
    for (int tau = 0; tau < KM; ++tau)
#pragma unroll
        for (int r = 0; r < 4; ++r) o = fs_mma(bn * qf[tau][r], s0[tau][r], o);
#pragma unroll
    for (int q = 0; q < 4; ++q) o = fs_mma(4 * g + q <= n ? d[q] * qk[q] : 0.f, dl[q], o);
    const f32x4 on4 = fs_rows(tk.on, g);
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const int tq = c * C + 4 * g + i;
        const float p = fs_row_sum(dl[i] * dl[i]);
        if (n == 0) dd[vt][4 * g + i] = p;
        if (j < V && tq < s.T)
            store_out(s.out, s.out_bf16, (((int64_t)b * s.T + tq) * s.H + h) * V + j, on4[i] != 0.f ? o[i] : 0.f);
    }
    const float ksq = fs_sq<KM>(kf);
    __syncthreads();
    if (s.scores && threadIdx.x < C && c * C + n < s.T) {
        float x = 0.f;
        for (int v = 0; v < VT; ++v) x += dd[v][n];
        s.scores[((int64_t)b * s.T + c * C + n) * s.H + h] = on ? sqrtf(ksq * x) : 0.f;
    }
}

// ---- bprep: N = (b Q)^T dO - W'^T X, X = P^T dO + c delta, one wave per value tile
template <int KM, bool BF>
__global__ void __launch_bounds__(64 * KM) fs_bprep_kernel(FcArgs a) {
    const SeqArgs &s = a.s;
    const int bh = blockIdx.x / a.wn, cw = blockIdx.x % a.wn, c = a.w0 + cw, b = bh / s.H, h = bh % s.H;
    const int64_t ci = (int64_t)bh * a.nc + c, wi = blockIdx.x;
    const int K = s.K, V = s.V, KP = fc_kp(K), KT = KP >> 4, VT = (V + 15) >> 4;
    const int vt = threadIdx.x >> 6, l = lane_id(), g = l >> 4, n = l & 15;
    f32x4 kf[KM], qf[KM];
    fs_frags<KM, BF>(kf, s.k, a.vec & 2, b, h, c, s.T, K);
    fs_frags<KM, BF>(qf, s.q, a.vec & 1, b, h, c, s.T, K);
    const FsTok tk = fs_tok(s, b, h, c);
    const bool on = tk.on != 0.f;
    const f32x4 on4 = fs_rows(tk.on, g);
    const f32x4 dO = s.dout.data ? fs_col<BF>(s.dout, b, h, c, vt, s.T, V, on4) : zero4();
#pragma unroll
    for (int tau = 0; tau < KM; ++tau) kf[tau] = fs_keep(kf[tau], on), qf[tau] = fs_keep(qf[tau], on);
    const f32x4 qk = fs_dot<KM>(qf, kf);  // row t = 4 g + i, column s = n
    float lam;
    const f32x4 d = fs_decay_rows(tk.a, g, n, lam);
    const f32x4 b4 = fs_rows(fs_decay_start(tk.a, n), g);
    f32x4 x = zero4();
    if (s.dscores) {
        float cs, ck;
        fs_score_adj(a, ci, b, h, c, VT, tk.on, fs_sq<KM>(kf), cs, ck);
        x = fs_rows(cs, g) * *reinterpret_cast<const fc_u4 *>(&a.fu[((ci * VT + vt) * 64 + l) * 4]);
    }
#pragma unroll
    for (int q = 0; q < 4; ++q) x = fs_mma(n <= 4 * g + q ? d[q] * qk[q] : 0.f, dO[q], x);
#pragma unroll
    for (int tau = 0; tau < KM; ++tau)
        if (tau < KT) {
            const f32x4 qb = fs_col<BF>(s.q, b, h, c, tau, s.T, K, on4) * b4;
            f32x4 nn = zero4();
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                nn = fs_mma(qb[q], dO[q], nn);
                nn = fs_mma(-a.fw[(ci * C + 4 * g + q) * KP + 16 * tau + n], x[q], nn);
            }
            *reinterpret_cast<fc_u4 *>(&a.n[(((wi * VT + vt) * KT + tau) * 64 + l) * 4]) = nn;
        }
}

// ---- bgrad: every gradient of one chunk -------------------------------------------
// With S0, delta (the forward) and dS at the chunk end (the adjoint scan):
//   ddelta = P^T dO + Ktil dS + c delta,  dR = T^T ddelta,  dv = beta dR
//   Qb = b dO S0^T,  Ab = -b dR S0^T,  Kl = lam delta dS^T
//   dA = -strict_lower(dR delta^T),  dP = lower(dO delta^T)
//   dq = Qb + (dP D) K,  dehat = Ab + (dA D) K,
//   dk = Kl + beta dehat + (beta dA D)^T K + (dP D)^T Q + c' k
//   dbeta = k . dehat + v . dR
// and, every path of the decays through token u being a pair (lo, hi) with
// lo < u <= hi whose full product has a_u as a factor,
//   dg_u = sum_{s < u <= t} E_ts + sum_{t >= u} y_t + sum_{s < u} z_s + b_15 <S0, dS>,
//   E = beta dA D KK^T + dP D QK^T,  y_t = beta k . Ab + q . Qb,  z_s = k . Kl
// (zero on padding and resets).  Wave w takes value tile w for dR, then key tile
// w; blockDim is 64 max(KT, VT).
template <int KM, bool BF>
__global__ void __launch_bounds__(64 * KM) fs_bgrad_kernel(FcArgs a) {
    __shared__ FsGradSmem<KM> sm;
    constexpr int LD = FsGradSmem<KM>::LD;
    const SeqArgs &s = a.s;
    const int bh = blockIdx.x / a.wn, cw = blockIdx.x % a.wn, c = a.w0 + cw, b = bh / s.H, h = bh % s.H;
    const int64_t ci = (int64_t)bh * a.nc + c, wi = blockIdx.x;
    const int K = s.K, V = s.V, KT = fc_kp(K) >> 4, VT = (V + 15) >> 4, NW = blockDim.x >> 6;
    const int w = threadIdx.x >> 6, l = lane_id(), g = l >> 4, n = l & 15, tg = c * C + n;
    f32x4 kf[KM], qf[KM];
    fs_frags<KM, BF>(kf, s.k, a.vec & 2, b, h, c, s.T, K);
    fs_frags<KM, BF>(qf, s.q, a.vec & 1, b, h, c, s.T, K);
    const FsTok tk = fs_tok(s, b, h, c);
    const bool on = tk.on != 0.f;
    const f32x4 on4 = fs_rows(tk.on, g);
    f32x4 tb, dO = zero4(), vb = zero4(), kb = zero4(), qb = zero4();
#pragma unroll
    for (int q = 0; q < 4; ++q) tb[q] = a.tm[ci * C * C + (4 * g + q) * C + n];
    if (w < VT) {
        if (s.dout.data) dO = fs_col<BF>(s.dout, b, h, c, w, s.T, V, on4);
        vb = fs_col<BF>(s.v, b, h, c, w, s.T, V, on4);
    }
    if (w < KT) {
        kb = fs_col<BF>(s.k, b, h, c, w, s.T, K, on4);
        qb = fs_col<BF>(s.q, b, h, c, w, s.T, K, on4);
    }
    // S0, dS and delta into LDS; <S0, dS>
    float fr = 0.f;
#pragma unroll 4
    for (int x = w; x < VT * KT; x += NW) {
        const int vt = x / KT, tau = x - vt * KT;
        const f32x4 x0 = *reinterpret_cast<const fc_u4 *>(&a.st[((ci * VT * KT + x) * 64 + l) * 4]);
        const f32x4 x1 = *reinterpret_cast<const fc_u4 *>(&a.ds[((wi * VT * KT + x) * 64 + l) * 4]);
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            sm.s0[(16 * tau + 4 * g + r) * LD + 16 * vt + n] = x0[r];
            sm.ds[(16 * tau + 4 * g + r) * LD + 16 * vt + n] = x1[r];
            fr += x0[r] * x1[r];
        }
    }
    f32x4 dl = zero4();
    if (w < VT) {
        dl = *reinterpret_cast<const fc_u4 *>(&a.fu[((ci * VT + w) * 64 + l) * 4]);
#pragma unroll
        for (int r = 0; r < 4; ++r) sm.dl[(4 * g + r) * LD + 16 * w + n] = dl[r];
    }
    fr = fs_group_sum(fs_row_sum(fr));
    if (l == 0) sm.fr[w] = fr;
#pragma unroll
    for (int tau = 0; tau < KM; ++tau) kf[tau] = fs_keep(kf[tau], on), qf[tau] = fs_keep(qf[tau], on);
    const f32x4 qk = fs_dot<KM>(qf, kf);  // row t = 4 g + i, column s = n
    float lam;
    const f32x4 d = fs_decay_rows(tk.a, g, n, lam), dc = fs_decay_cols(tk.a, g, n);
    const float bn = fs_decay_start(tk.a, n);
    const f32x4 be4 = fs_rows(tk.beta, g);
    float cs = 0.f, ck = 0.f;
    if (s.dscores) fs_score_adj(a, ci, b, h, c, VT, tk.on, fs_sq<KM>(kf), cs, ck);
    __syncthreads();
    if (w < VT) {  // ddelta and dR of value tile w
        const int j = 16 * w + n;
        f32x4 dd = fs_rows(cs, g) * dl;
#pragma unroll
        for (int q = 0; q < 4; ++q) dd = fs_mma(n <= 4 * g + q ? d[q] * qk[q] : 0.f, dO[q], dd);
#pragma unroll
        for (int tau = 0; tau < KM; ++tau)
            if (tau < KT)
#pragma unroll
                for (int r = 0; r < 4; ++r)
                    dd = fs_mma(lam * kf[tau][r], sm.ds[(16 * tau + 4 * g + r) * LD + j], dd);
        f32x4 dr = zero4(), drt = zero4();  // rows t, column j; rows j, column t
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            dr = fs_mma(tb[q], dd[q], dr);
            drt = fs_mma(dd[q], tb[q], drt);
        }
        *reinterpret_cast<f32x4 *>(&sm.dr[n * LD + 16 * w + 4 * g]) = drt;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int tt = 4 * g + i, tq = c * C + tt;
            const float p = fs_row_sum(vb[i] * dr[i]);
            if (n == 0) sm.vd[w][tt] = p;
            if (s.dv && j < V && tq < s.T)
                store_out(s.dv, BF, (((int64_t)b * s.T + tq) * s.H + h) * V + j, on4[i] != 0.f ? be4[i] * dr[i] : 0.f);
        }
    }
    __syncthreads();
    // The decayed adjoint tiles: 0 dP D and 1 dA D with column t (row s), 2 dP D
    // and 3 beta dA D with column s (row t).
    for (int x = w; x < 4; x += NW) {
        f32x4 m = zero4();
        for (int vt = 0; vt < VT; ++vt) {
            const f32x4 e = *reinterpret_cast<const f32x4 *>(&sm.dl[n * LD + 16 * vt + 4 * g]);
            f32x4 y;
            if (x & 1) y = *reinterpret_cast<const f32x4 *>(&sm.dr[n * LD + 16 * vt + 4 * g]);
            else
                y = fs_keep(s.dout.data ? fs_ld4<BF>(s.dout, a.vec & 8, b, tg, h, 16 * vt + 4 * g, V, tg < s.T) : zero4(),
                            on);
#pragma unroll
            for (int r = 0; r < 4; ++r) m = x < 2 ? fs_mma(e[r], y[r], m) : fs_mma(y[r], e[r], m);
        }
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int rr = 4 * g + i, t = x < 2 ? n : rr, u = x < 2 ? rr : n;
            const float f = x < 2 ? dc[i] : d[i];
            m[i] = (x & 1) ? (u < t ? -(x == 3 ? be4[i] : 1.f) * f * m[i] : 0.f) : (u <= t ? f * m[i] : 0.f);
        }
        sm.m[x][l] = m;
    }
    f32x4 Qb = zero4(), Ab = zero4(), Kl = zero4();  // rows t, column key 16 w + n
    if (w < KT)
        for (int vt = 0; vt < VT; ++vt) {
            const int o = (16 * w + n) * LD + 16 * vt + 4 * g;
            const f32x4 s0 = *reinterpret_cast<const f32x4 *>(&sm.s0[o]);
            const f32x4 ds = *reinterpret_cast<const f32x4 *>(&sm.ds[o]);
            const f32x4 e = *reinterpret_cast<const f32x4 *>(&sm.dl[n * LD + 16 * vt + 4 * g]);
            const f32x4 r = *reinterpret_cast<const f32x4 *>(&sm.dr[n * LD + 16 * vt + 4 * g]);
            const f32x4 y = fs_keep(
                s.dout.data ? fs_ld4<BF>(s.dout, a.vec & 8, b, tg, h, 16 * vt + 4 * g, V, tg < s.T) : zero4(), on);
#pragma unroll
            for (int x = 0; x < 4; ++x) {
                Qb = fs_mma(bn * y[x], s0[x], Qb);
                Ab = fs_mma(-bn * r[x], s0[x], Ab);
                Kl = fs_mma(lam * e[x], ds[x], Kl);
            }
        }
    __syncthreads();
    if (w < KT) {
        const f32x4 m0 = sm.m[0][l], m1 = sm.m[1][l], m2 = sm.m[2][l], m3 = sm.m[3][l], ck4 = fs_rows(ck, g);
        f32x4 dq = Qb, de = Ab, dk = Kl;
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            dq = fs_mma(m0[q], kb[q], dq);
            de = fs_mma(m1[q], kb[q], de);
            dk = fs_mma(m3[q], kb[q], dk);
            dk = fs_mma(m2[q], qb[q], dk);
        }
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int tt = 4 * g + i, tq = c * C + tt, key = 16 * w + n;
            const float ys = fs_row_sum(be4[i] * kb[i] * Ab[i] + qb[i] * Qb[i]);
            const float zs = fs_row_sum(kb[i] * Kl[i]), kd = fs_row_sum(kb[i] * de[i]);
            if (n == 0) sm.ys[w][tt] = ys, sm.zs[w][tt] = zs, sm.kd[w][tt] = kd;
            if (key < K && tq < s.T) {
                const int64_t o = (((int64_t)b * s.T + tq) * s.H + h) * K + key;
                const bool v = on4[i] != 0.f;
                if (s.dq) store_out(s.dq, BF, o, v ? dq[i] : 0.f);
                if (s.dk) store_out(s.dk, BF, o, v ? dk[i] + be4[i] * de[i] + ck4[i] * kb[i] : 0.f);
            }
        }
    }
    float wu = 0.f;
    if (w == 0) {  // lane (g, n): sum_{s < n <= t} E_ts
        const f32x4 kk = fs_dot<KM>(kf, kf), m2 = sm.m[2][l], m3 = sm.m[3][l];
        f32x4 e;
#pragma unroll
        for (int i = 0; i < 4; ++i) e[i] = n < 4 * g + i ? m3[i] * kk[i] + m2[i] * qk[i] : 0.f;
#pragma unroll
        for (int u = 1; u < C; ++u) {
            float p = 0.f;
#pragma unroll
            for (int i = 0; i < 4; ++i) p += 4 * g + i >= u ? e[i] : 0.f;
            p = fs_row_sum(n < u ? p : 0.f);
            if (u == n) wu = p;
        }
        wu = fs_group_sum(wu);
    }
    __syncthreads();
    if (threadIdx.x < C && tg < s.T) {
        float db = 0.f, dg = wu, f = 0.f;
        for (int x = 0; x < VT; ++x) db += sm.vd[x][n];
        for (int x = 0; x < KT; ++x) {
            db += sm.kd[x][n];
#pragma unroll
            for (int u = 0; u < C; ++u) dg += u >= n ? sm.ys[x][u] : sm.zs[x][u];
        }
        for (int x = 0; x < NW; ++x) f += sm.fr[x];
        dg += fs_lane(bn, C - 1) * f;
        const int64_t o = ((int64_t)b * s.T + tg) * s.H + h;
        if (s.dbeta) s.dbeta[o] = on ? db : 0.f;
        if (s.dg) s.dg[o] = (on && tk.rst == 0.f) ? dg : 0.f;
    }
}

static inline void fsmark(const hipEvent_t *ev, int i, hipStream_t stream) {
    if (ev) (void)hipEventRecord(ev[i], stream);
}

template <int KM, bool BF>
static hipError_t fs_fwd(const FcArgs &a, hipStream_t stream, const hipEvent_t *ev) {
    const int n = a.s.B * a.s.H * a.nc, VT = (a.s.V + 15) / 16;
    fsmark(ev, 0, stream);
    hipLaunchKernelGGL((fs_prep_kernel<KM, BF>), dim3(n), dim3(64), 0, stream, a);
    fsmark(ev, 1, stream);
    fsmark(ev, 2, stream);
    launch_fc_scan(a, false, stream);
    fsmark(ev, 3, stream);
    fsmark(ev, 4, stream);
    hipLaunchKernelGGL((fs_out_kernel<KM, BF>), dim3(n), dim3(64 * VT), 0, stream, a);
    fsmark(ev, 5, stream);
    return hipGetLastError();
}

template <int KM, bool BF>
static hipError_t fs_bwd(FcArgs a, size_t ws_bytes, hipStream_t stream, const hipEvent_t *ev) {
    const int bh = a.s.B * a.s.H, VT = (a.s.V + 15) / 16, KT = fc_kp(a.s.K) / 16;
    // Chunk windows, last first: as many chunks as the workspace holds, the
    // adjoint between two windows in the carry.
    const int64_t tile = (int64_t)KT * VT * 256 * sizeof(float), carry = bh * tile, per = 2 * bh * tile;
    int64_t wn = (int64_t)ws_bytes / per;
    if (wn < a.nc) wn = ((int64_t)ws_bytes - carry) / per;
    if (wn < 1) return hipErrorInvalidValue;
    wn = wn < a.nc ? wn : a.nc;
    float *ws = a.ds;
    for (int end = a.nc; end > 0;) {
        a.wn = (int)(end < wn ? end : wn);
        a.w0 = end - a.wn;
        a.ds = ws;
        a.n = ws + wn * bh * tile / sizeof(float);
        a.carry = a.n + wn * bh * tile / sizeof(float);
        const hipEvent_t *e = end == a.nc ? ev : nullptr;
        fsmark(e, 0, stream);
        hipLaunchKernelGGL((fs_bprep_kernel<KM, BF>), dim3(bh * a.wn), dim3(64 * VT), 0, stream, a);
        fsmark(e, 1, stream);
        fsmark(e, 2, stream);
        launch_fc_scan(a, true, stream);
        fsmark(e, 3, stream);
        fsmark(e, 4, stream);
        hipLaunchKernelGGL((fs_bgrad_kernel<KM, BF>), dim3(bh * a.wn), dim3(64 * (KT > VT ? KT : VT)), 0, stream, a);
        fsmark(e, 5, stream);
        end = a.w0;
    }
    return hipGetLastError();
}

hipError_t launch_fs_fwd(const FcArgs &a, hipStream_t stream, const hipEvent_t *ev) {
    const bool wide = a.s.K > 64 || a.s.V > 64;
    if (a.in_bf16) return wide ? fs_fwd<8, true>(a, stream, ev) : fs_fwd<4, true>(a, stream, ev);
    return wide ? fs_fwd<8, false>(a, stream, ev) : fs_fwd<4, false>(a, stream, ev);
}

hipError_t launch_fs_bwd(const FcArgs &a, size_t ws_bytes, hipStream_t stream, const hipEvent_t *ev) {
    const bool wide = a.s.K > 64 || a.s.V > 64;
    if (a.in_bf16) return wide ? fs_bwd<8, true>(a, ws_bytes, stream, ev) : fs_bwd<4, true>(a, ws_bytes, stream, ev);
    return wide ? fs_bwd<8, false>(a, ws_bytes, stream, ev) : fs_bwd<4, false>(a, ws_bytes, stream, ev);
}

}  // namespace gdn2
