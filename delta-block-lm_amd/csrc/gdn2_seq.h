// Token-sequential GDN-2 kernels (the scalar-gate walk, channel-wise decode), and the
// argument block that the chunk kernels' launchers share with them.
#pragma once

#include "gdn2_common.h"

namespace gdn2 {

constexpr int SEQ_CT = 16;  // tokens per staging block == checkpoint interval

struct SeqArgs {
    int B, T, H, K, V;
    View q, k, v, alpha, erase, write, valid, reset, initial;
    // Document limits (int32 [batch, time] views, inclusive; end < start marks
    // padding, start == t resets the state; the f32 chunk kernels).  When set they
    // replace valid/reset; the backward is the exact VJP, as with masks.
    int doc;
    View doc_start, doc_end;
    // Scalar-gate mode: alpha[i] = exp(g), erase[i] = write[j] = beta, with
    // beta and g read as [batch, time, head] views; gradients dbeta and dg.
    int scalar;
    View beta, g;
    float *dbeta, *dg;
    // forward outputs
    void *out;
    int out_bf16;
    float *final_state, *scores;
    // Checkpoint: the state at the start of every block and the edit delta of every
    // token.  A call that only walks has one block (T <= SEQ_CT): row-major
    // [B*H][K_pad][V_pad] and [B*H][SEQ_CT][V_pad].  Behind the f32 chunk kernels the
    // walk takes the (batch, head)s whose word in `only` is not zero, and these are
    // the chunk kernels' arrays of the same names, in packed 16 x 16 tiles
    // (gdn2_chunk_f32.h; whole lines a wave there, but pieces of 16 bytes in the walk's
    // own layout: at 1024 heads of 128 x 128 its forward took 62 us of them, for 53).
    float *st, *fu;
    int nck;
    const int *only;
    // backward
    View dout;
    const float *dfinal, *dscores;
    void *dq, *dk, *dv;
    float *dalpha, *derase, *dwrite, *dinitial;
    float *replay;  // [B*H][SEQ_CT][K_pad * V_pad], thread-major
};

// Padded widths used by the kernels: 32, 64 or 128.
inline int seq_pad(int n) { return n <= 32 ? 32 : (n <= 64 ? 64 : 128); }
inline int64_t seq_state_floats(int K, int V) { return (int64_t)seq_pad(K) * seq_pad(V); }

// A call of one block's checkpoint.
inline int64_t seq_checkpoint_floats(int64_t B, int64_t H, int K, int V) {
    return B * H * (seq_state_floats(K, V) + SEQ_CT * seq_pad(V));
}

inline void seq_bind_checkpoint(SeqArgs &a, const void *ck) {
    a.st = static_cast<float *>(const_cast<void *>(ck));
    a.fu = a.st + (int64_t)a.B * a.H * seq_state_floats(a.K, a.V);
}

// Offsets of S[i][j] in a block's state tiles (KT key tiles) and of token t's delta[j]
// in its edit tiles.
__host__ __device__ inline int seq_state_at(int i, int j, int KT) {
    return ((j >> 4) * KT + (i >> 4)) * 256 + ((i & 15) >> 2) * 64 + (j & 15) * 4 + (i & 3);
}
__host__ __device__ inline int seq_edit_at(int t, int j) {
    return (j >> 4) * 256 + (t >> 2) * 64 + (j & 15) * 4 + (t & 3);
}

inline int64_t seq_workspace_floats(int64_t B, int64_t H, int K, int V) {
    return B * H * SEQ_CT * seq_state_floats(K, V);
}

// Without a checkpoint (st and fu null) the outputs alone, of any length.
hipError_t launch_seq_fwd(const SeqArgs &a, bool in_bf16, hipStream_t stream);
// One token (T == 1, masks only) on a carried state; no checkpoint.
hipError_t launch_seq_decode(const SeqArgs &a, bool in_bf16, hipStream_t stream);
hipError_t launch_seq_bwd(const SeqArgs &a, bool in_bf16, hipStream_t stream);

}  // namespace gdn2
