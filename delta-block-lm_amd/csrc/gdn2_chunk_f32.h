// Chunked GDN-2 in f32 (d_k, d_v <= 128, 16-token chunks): channel-wise gates
// (gdn2_chunk_f32.hip) and scalar gates (gdn2_chunk_fs.hip).
#pragma once

#include "gdn2_seq.h"

namespace gdn2 {

// Four floats of a checkpoint or workspace array: the scalar-gate entry points
// take buffers of any alignment (16-byte accesses to global memory need four).
typedef float fc_u4 __attribute__((ext_vector_type(4), aligned(4)));

constexpr int FC_C = 16;  // tokens per chunk

// The token-sequential argument block (shapes, views, outputs, gradients)
// plus the chunk path's checkpoint and workspace arrays, each indexed by
// chunk ci = (b * H + h) * nc + c:
//   st     S at the chunk start, packed tiles: [VT][KT][4][16][4], element
//          (((vt * KT + tau) * 4 + g) * 16 + n) * 4 + r = S[16 tau + 4 g + r][16 vt + n]
//          (forward scan -> out, bgrad)
//   tm     T = (I + A)^-1, [16][16]                          (prep -> bgrad)
//   pm     P, [16][16]                  (prep -> out, adjoint scan, bgrad)
//   dm     the pair decays D, [16][16], scalar gates only    (prep -> bgrad)
//   fw, fk, fq  the factored map W' = T (b . e . k) and Ktil = lam . k, and Qhat =
//          b . q, packed tiles: [KT][4][16][4], element
//          ((tau * 4 + g) * 16 + n) * 4 + r = W'[4 g + r][16 tau + n]
//   fu     U = T (w . v), packed tiles [VT][4][16][4]; the forward scan overwrites
//          it with the edits delta (-> out, bgrad)
//   gv     b_15 (the map's diagonal), [KP]
//   gb     rows of one value per token: valid, reset, |k|^2, and with scalar gates
//          beta, b, lam; [8][16]
// and, with scalar gates, one word per (batch, head):
//   bad    the forward gave a value that is not finite (out); such a (batch, head)
//          is walked by token afterwards (gdn2_chunk_fs.hip)
// KP = d_k and VP = d_v rounded up to 16 (KT = KP / 16, VT = VP / 16): the tiles
// are padded with zeros to whole 16 x 16 MFMA tiles.  Backward workspace: ds, the
// state adjoint at each chunk end, packed like st, and, with a score adjoint, sc,
// the coefficients c and c' per token [2][16], for the window of chunks w0 .. w0 +
// wn - 1 of each (batch, head) (index bh * wn + c - w0; all nc chunks unless the
// scalar-gate path walks windows); carry is the adjoint before the window, packed,
// one state per (batch, head), and wbad the backward's counterpart of bad, at the
// workspace's end.  st and ds are zero outside K x V.  Every array
// starts on a 16-byte boundary when the caller's buffer does.
struct FcArgs {
    SeqArgs s;
    int nc;
    int in_bf16;  // q, k, v, dO and dq, dk, dv are bf16 (else f32)
    int vec;      // every input of the call passes fc_vec_view
    int scalar;   // scalar gates
    int nonneg;   // a negative alpha poisons its sequence with NaN
    float *st, *fu, *tm, *pm, *dm, *fw, *fk, *fq, *gv, *gb;
    float *ds, *sc;
    int w0, wn;
    float *carry;
    int *bad, *wbad;  // null with channel-wise gates
};

inline int64_t fc_chunks(int64_t B, int64_t T, int64_t H) { return B * H * ((T + FC_C - 1) / FC_C); }
__host__ __device__ inline int fc_kp(int K) { return (K + 15) & ~15; }

// The inputs that the kernels read by whole 16-channel tiles from a uniform base
// with 32-bit offsets: unit channel stride, 4-channel pieces aligned to their
// size, and rows less than 2^24 elements apart.
inline bool fc_vec_view(const View &v, int bytes, int64_t W) {
    return v.s3 == 1 && W % 16 == 0 && ((uintptr_t)v.data & (4 * bytes - 1)) == 0 && v.s0 % 4 == 0 &&
           v.s1 % 4 == 0 && v.s2 % 4 == 0 && v.s1 < (1 << 24);
}

constexpr int FC_PARTS = 10;
// The checkpoint's arrays in order, in floats, for n chunks (each a multiple of
// four).
inline void fc_checkpoint_parts(int64_t n, int K, int V, bool scalar, size_t part[FC_PARTS]) {
    const size_t KP = fc_kp(K), VP = fc_kp(V);
    part[0] = n * KP * VP;                      // st
    part[1] = n * FC_C * VP;                    // fu
    part[2] = part[3] = n * FC_C * FC_C;        // tm, pm
    part[4] = scalar ? n * FC_C * FC_C : 0;     // dm
    part[5] = part[6] = part[7] = n * FC_C * KP;  // fw, fk, fq
    part[8] = n * KP;                           // gv
    part[9] = n * FC_C * 8;                     // gb
}

// Bytes of one word per (batch, head), whole 16-byte pieces.
inline size_t fc_word_bytes(int64_t B, int64_t H) { return ((size_t)(B * H) * 4 + 15) & ~(size_t)15; }

inline size_t fc_checkpoint_bytes(int64_t B, int64_t T, int64_t H, int K, int V, bool scalar) {
    size_t part[FC_PARTS], total = 0;
    fc_checkpoint_parts(fc_chunks(B, T, H), K, V, scalar, part);
    for (size_t x : part) total += x;
    return total * sizeof(float) + (scalar ? fc_word_bytes(B, H) : 0);
}

// Floats of the workspace per chunk.
inline int64_t fc_ws_chunk(int K, int V) { return (int64_t)fc_kp(K) * fc_kp(V) + 2 * FC_C; }

inline size_t fc_workspace_bytes(int64_t B, int64_t T, int64_t H, int K, int V) {
    return (size_t)(fc_chunks(B, T, H) * fc_ws_chunk(K, V)) * sizeof(float);
}

inline void fc_bind(FcArgs &a, void *ck, void *ws) {
    const int64_t n = fc_chunks(a.s.B, a.s.T, a.s.H);
    size_t part[FC_PARTS];
    fc_checkpoint_parts(n, a.s.K, a.s.V, a.scalar != 0, part);
    float *p = static_cast<float *>(ck);
    float **dst[FC_PARTS] = {&a.st, &a.fu, &a.tm, &a.pm, &a.dm, &a.fw, &a.fk, &a.fq, &a.gv, &a.gb};
    for (int i = 0; i < FC_PARTS; ++i) {
        *dst[i] = p;
        p += part[i];
    }
    a.bad = a.scalar ? reinterpret_cast<int *>(p) : nullptr;
    a.w0 = 0;
    a.wn = a.nc;
    if (ws) {
        a.ds = static_cast<float *>(ws);
        a.sc = a.ds + n * fc_kp(a.s.K) * fc_kp(a.s.V);
    }
}

// The stages that both gate forms share: the state scan over the chunks, out, and
// the adjoint scan over the window (with the score adjoint's coefficients).
void launch_fc_scan(const FcArgs &a, hipStream_t stream);
void launch_fc_out(const FcArgs &a, hipStream_t stream);
void launch_fc_adjoint(const FcArgs &a, hipStream_t stream);

hipError_t launch_fc_fwd(const FcArgs &a, hipStream_t stream, const hipEvent_t *ev);
hipError_t launch_fc_bwd(const FcArgs &a, hipStream_t stream, const hipEvent_t *ev);
// Scalar gates.  The backward takes any workspace that holds one chunk window, the
// carry and the words, and the words behind the token walk's workspace; with
// fc_workspace_bytes and the words it is one window.
hipError_t launch_fs_fwd(const FcArgs &a, hipStream_t stream, const hipEvent_t *ev);
hipError_t launch_fs_bwd(const FcArgs &a, size_t ws_bytes, hipStream_t stream, const hipEvent_t *ev);

}  // namespace gdn2
