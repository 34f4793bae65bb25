// dit_internal.hpp — shared definitions of the DiT block kernels.
#pragma once

#include "awa_internal.hpp"
#include "dit_capi.h"

namespace awa {

enum { EPI_STORE = 0, EPI_RESID = 1, EPI_SWIGLU = 2 };

struct GemmProblem {
    const uint16_t* A;     // [M][K] bf16, row stride lda (elements)
    const uint16_t* W;     // [N][K] bf16, row stride ldw
    int M, N, K, lda, ldw;
    void* C;               // EPI_STORE / EPI_SWIGLU: bf16; EPI_RESID: fp32 residual (in/out)
    int ldc;
    const float* bias;     // [N] or null (EPI_RESID)
    const float* gate0;    // [N] gate of rows < split, null = 1 (EPI_RESID)
    const float* gate1;    // [N] gate of rows >= split, null = 1
    int split;
    int n_tiles, m_tiles;  // filled by launch_gemm
};

struct GemmBatch {
    GemmProblem p[2];      // one or two independent problems in one launch
    int nprob;
    int tiles0, total_tiles;
};

// compute units of the current device (256 if it cannot be asked)
int device_cus();
hipError_t launch_gemm(int epi, GemmBatch& b, hipStream_t s);

// h[m] = bf16(RMSNorm(x[m]) * scale + shift); rows >= split use the second
// pair (null scale: plain RMSNorm, the last layer's text rows).
struct NormArgs {
    const float* x;
    uint16_t* h;
    int M, split;
    const float* scale0;
    const float* shift0;
    const float* scale1;
    const float* shift1;
    float eps;
};
hipError_t launch_norm_ada(const NormArgs& a, hipStream_t s);

// out[f][k][d] = emb[6d + K_MAP[k]] + branch_f[k][d] for the 6 vectors
// (a_sc, a_sh, a_g, m_sc, m_sh, m_g) of the two flows.
struct AdaArgs {
    const float* emb;
    const float* vec[2][6];  // branch vectors per flow, order as above
    float* out;              // [2][6][2560]
};
hipError_t launch_ada(const AdaArgs& a, hipStream_t s);

hipError_t launch_pack_mlp(const uint16_t* w_in, const uint16_t* w_gate, int mlp, uint16_t* w_cat,
                           hipStream_t s);

// The timestep embedding emb[DIT_EMB] of t: sinusoid [256], then three linears
// in fp32 ([2560][256], [2560][2560], [DIT_EMB][2560]) with SiLU after the first
// two; e1 and e2 hold 2560 values each.
hipError_t launch_time_mlp(float t, const float* const w[3], const float* const b[3], float* e1, float* e2, float* emb,
                           hipStream_t s);

// The model's ends (dit_ends.hip).  x [Lv + TXT][2560] from the latent grid
// (T, H, 2 W2, 33) and the text features [TXT][5120].
constexpr int EMBED_K = 160;  // 132 patch channels and zeros up to whole k32 steps
constexpr int EMBED_TXT_SPLIT = 16;  // parts of the text projection's K
// Up to this many text rows the embedding projects them itself; longer texts take the
// block's GEMM, since the partial products are 160 KB a row.  On 400 video rows: 58 text
// rows 17 us against 40, 320 44.3 against 45.3, 384 50.4 against 45.6, 2000 254
// against 85; the same point with 5440 video rows.
constexpr int EMBED_TXT_MAX = 320;
struct EmbedArgs {
    const float* grid;
    int H, W2;
    int Lv, TXT;  // TXT = 0: the video rows only
    const uint16_t* vid_w;  // [2560][EMBED_K] in fragment order
    const float* vid_b;
    const float* txt;
    const uint16_t* txt_w;  // [2560][5120]
    const float* txt_b;
    float* x;
    float* part;     // workspace: [EMBED_TXT_SPLIT][TXT][2560] partial products of the text
    int txt_blocks;  // filled by launch_embed
};
hipError_t launch_embed(const EmbedArgs& a, hipStream_t s);
// out (T, H, 2 W2, 16) from the first `rows` rows of x and the timestep embedding
struct FinalArgs {
    const float* x;
    const float* emb;
    const float* norm_w;
    const float* ada_scale;
    const float* ada_shift;
    const uint16_t* W;  // [64][2560] in fragment order
    const float* bias;  // [64]
    int rows, H, W2;
    float eps;
    float* out;
    int rpw;  // rows per workgroup, filled by launch_final
};
hipError_t launch_final(const FinalArgs& a, hipStream_t s);
// The video weights of both ends, [2560][132] and [64][2560], in the fragment
// order that launch_embed and launch_final read: EMBED_K per input row (zeros
// past 132), DIM per output row.
hipError_t launch_end_weights(const uint16_t* vid_in, uint16_t* vid_in_frag, const uint16_t* vid_out,
                              uint16_t* vid_out_frag, hipStream_t s);

}  // namespace awa
