// dit_ends.hip — the model's two ends, one launch each.
//
//   embed   latent grid and prompt -> the residual stream (dit_vk.cpp:486-505,
//           717-733): x = patchify(grid) W_vid^T + b, text W_txt^T + b
//   final   residual stream -> latent output (dit_vk.cpp:657-675, 735-750):
//           RMSNorm, the output modulation, the 2560 -> 64 projection, the 2x2
//           patches back to pixels
//
// Both are bound by the residual stream's bytes (56 MB fp32 at 1080p, 8-9 us
// at the rate of a device copy of that size); the products are small, and as
// tiles of the block's 256-row GEMM they left most CUs idle.  At 1080p (5440
// video rows, 58 text rows): embed 140 -> 27 us, final 76 -> 18 us against
// separate patchify, cast, zero, norm, GEMM and unpatchify launches.
#include "dit_internal.hpp"

namespace awa {

namespace {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef unsigned u32x4 __attribute__((ext_vector_type(4)));
// accesses to caller buffers that are only known to hold floats
typedef float f32x4u __attribute__((ext_vector_type(4), aligned(4)));
typedef float f32x2u __attribute__((ext_vector_type(2), aligned(4)));

__device__ inline bf16x8 pack8(const float (&v)[8]) {
    const u32x4 u = {bf16x2_rne(v[0], v[1]), bf16x2_rne(v[2], v[3]), bf16x2_rne(v[4], v[5]), bf16x2_rne(v[6], v[7])};
    return __builtin_bit_cast(bf16x8, u);
}

constexpr int NWAVE = 8;

// ---------------------------------------------------------------- final
//
// A workgroup owns rpw <= 16 RB rows, each of its 8 waves 320 of the 2560 channels, held in registers in the A-operand layout of
// v_mfma_f32_16x16x32_bf16, so a row is read once, its sum of squares is a
// per-lane sum plus one exchange through LDS, and the normalised, modulated
// row goes to the matrix cores without a trip through memory.  Within a k32
// step the four lanes of a row hold channels 4 q .. + 3 and 16 + 4 q .. + 3
// (any order that both operands share gives the same products), so each load
// instruction reads 64 contiguous bytes of a row.  The weights are stored in
// fragment order (final_w_pos).  The waves' partial products are summed in LDS
// in wave order.  The modulation vectors are formed per workgroup into LDS.
//
// The rows are spread evenly over the CUs (rpw = rows / CUs per round, two
// 16-row blocks from 17 on): a CU draws only about 30 GB/s from beyond its L2,
// so all of them must pull (32 rows on 170 CUs 22.4 us, 22 rows on 248 18.0;
// two smaller workgroups per CU read the weights twice: 17.3 us here but 13.4
// instead of 9.7 at 2720 rows).
constexpr int FIN_N = 64;
constexpr int FIN_KW = DIM / NWAVE, FIN_S = FIN_KW / 32;  // channels and k32 steps per wave
constexpr int FIN_P = 68;  // pitch of a partial row: the four lane groups of a store fall on distinct banks

template <int RB>
__global__ __launch_bounds__(512, 2) void final_kernel(FinalArgs a) {
    __shared__ float ssq[NWAVE][16 * RB];
    // the modulation vectors, then the partial products
    __shared__ __align__(16) float lds[NWAVE * 16 * RB * FIN_P];
    static_assert(sizeof(lds) >= 2 * DIM * 4, "modulation vectors fit");
    float *sc = lds, *sh = lds + DIM;
    const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
    const int r16 = lane & 15, q = lane >> 4;
    const int row0 = (int)blockIdx.x * a.rpw, row1 = min(row0 + a.rpw, a.rows);

    // scale w (emb[6d+1] + ada_scale), shift emb[6d] + ada_shift
    constexpr int NV = (DIM + 512 - 1) / 512;
    float e0[NV], e1[NV], vw[NV], vs[NV], vh[NV];
#pragma unroll
    for (int i = 0; i < NV; i++) {
        const int d = min(i * 512 + tid, DIM - 1);
        e0[i] = a.emb[6 * d]; e1[i] = a.emb[6 * d + 1];
        vw[i] = a.norm_w[d]; vs[i] = a.ada_scale[d]; vh[i] = a.ada_shift[d];
    }
    // rows past the workgroup's read nothing (zeros: their outputs are not stored)
    f32x4u v[RB][FIN_S][2];
#pragma unroll
    for (int rb = 0; rb < RB; rb++) {
        const int row = row0 + 16 * rb + r16;
        const float* xr = a.x + (size_t)row * DIM + wave * FIN_KW + 4 * q;
        if (row < row1) {
#pragma unroll
            for (int s = 0; s < FIN_S; s++)
#pragma unroll
                for (int e = 0; e < 2; e++) v[rb][s][e] = *reinterpret_cast<const f32x4u*>(xr + 32 * s + 16 * e);
        } else {
#pragma unroll
            for (int s = 0; s < FIN_S; s++) v[rb][s][0] = v[rb][s][1] = (f32x4u){0.f, 0.f, 0.f, 0.f};
        }
    }
    constexpr int PF = RB == 1 ? 3 : 2;  // k32 steps of weights loaded ahead
    const bf16x8* W = reinterpret_cast<const bf16x8*>(a.W) + (size_t)wave * FIN_S * 4 * 64 + lane;
    bf16x8 wf[PF][4];
    auto load_w = [&](int s) __attribute__((always_inline)) {
#pragma unroll
        for (int nb = 0; nb < 4; nb++)
            wf[s % PF][nb] = W[(4 * s + nb) * 64];
    };
#pragma unroll
    for (int s = 0; s < PF; s++) load_w(s);
#pragma unroll
    for (int i = 0; i < NV; i++) {
        const int d = min(i * 512 + tid, DIM - 1);  // the same value where threads repeat
        sc[d] = vw[i] * (e1[i] + vs[i]);
        sh[d] = e0[i] + vh[i];
    }
#pragma unroll
    for (int rb = 0; rb < RB; rb++) {
        float ss = 0.f;
#pragma unroll
        for (int s = 0; s < FIN_S; s++)
#pragma unroll
            for (int e = 0; e < 2; e++)
#pragma unroll
                for (int i = 0; i < 4; i++) ss += v[rb][s][e][i] * v[rb][s][e][i];
        ss += __shfl_xor(ss, 16);
        ss += __shfl_xor(ss, 32);
        if (q == 0) ssq[wave][16 * rb + r16] = ss;
    }
    __syncthreads();
    float r[RB];
#pragma unroll
    for (int rb = 0; rb < RB; rb++) {
        float tot = 0.f;
#pragma unroll
        for (int w = 0; w < NWAVE; w++) tot += ssq[w][16 * rb + r16];
        r[rb] = 1.0f / sqrtf(tot / (float)DIM + a.eps);
    }

    f32x4 acc[RB][4];
#pragma unroll
    for (int rb = 0; rb < RB; rb++)
#pragma unroll
        for (int nb = 0; nb < 4; nb++) acc[rb][nb] = (f32x4){0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int s = 0; s < FIN_S; s++) {
        const int d = wave * FIN_KW + 32 * s + 4 * q;
        f32x4 cs[2], ch[2];
#pragma unroll
        for (int e = 0; e < 2; e++) {
            cs[e] = *reinterpret_cast<const f32x4*>(sc + d + 16 * e);
            ch[e] = *reinterpret_cast<const f32x4*>(sh + d + 16 * e);
        }
#pragma unroll
        for (int rb = 0; rb < RB; rb++) {
            float h[8];
#pragma unroll
            for (int e = 0; e < 2; e++)
#pragma unroll
                for (int i = 0; i < 4; i++) h[4 * e + i] = v[rb][s][e][i] * r[rb] * cs[e][i] + ch[e][i];
            const bf16x8 hf = pack8(h);
#pragma unroll
            for (int nb = 0; nb < 4; nb++)
                acc[rb][nb] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(hf, wf[s % PF][nb], acc[rb][nb], 0, 0, 0);
        }
        if (s + PF < FIN_S) load_w(s + PF);
    }
    __syncthreads();  // every wave is done with the modulation vectors
    float* part = lds;
    // lane: output 16 nb + r16 of rows 16 rb + 4 q + t
#pragma unroll
    for (int rb = 0; rb < RB; rb++)
#pragma unroll
        for (int nb = 0; nb < 4; nb++)
#pragma unroll
            for (int t = 0; t < 4; t++) 
                    part[(wave * 16 * RB + 16 * rb + 4 * q + t) * FIN_P + 16 * nb + r16] = acc[rb][nb][t];
    __syncthreads();
    const int H2 = a.H >> 1, W2 = a.W2;
#pragma unroll
    for (int i = 0; i < 16 * RB * FIN_N / 512; i++) {
        const int o = i * 512 + tid, m = o >> 6, n = o & 63, row = row0 + m;
        if (row >= row1) continue;
        float y = part[m * FIN_P + n];
#pragma unroll
        for (int w = 1; w < NWAVE; w++) y += part[(w * 16 * RB + m) * FIN_P + n];
        y += a.bias[n];
        // value n of row (t, hh, ww) is pixel (ph, pw), channel c
        const int tt = row / (H2 * W2), hh = (row / W2) % H2, ww = row % W2;
        const int ph = n >> 5, pw = (n >> 4) & 1, c = n & 15;
        a.out[(((size_t)tt * a.H + 2 * hh + ph) * (2 * W2) + 2 * ww + pw) * 16 + c] = y;
    }
}

// The ends' weights in fragment order: the 16 bytes of every lane of a wave's
// fragment load side by side, so that a load instruction reads one contiguous
// KiB (as rows, 16 segments of 64 bytes 5 KiB apart, the 328 KB of weights that
// every CU reads from its L2 took several microseconds longer).
// final: fragment (wave, step s, block nb): lane holds output 16 nb + lane % 16,
// channels 320 wave + 32 s + 4 q + {0 .. 3, 16 .. 19}.
__global__ __launch_bounds__(256) void final_weights_kernel(const uint16_t* __restrict__ w, uint16_t* __restrict__ out) {
    const int i = blockIdx.x * 256 + threadIdx.x;
    const int e = i & 7, lane = (i >> 3) & 63, nb = (i >> 9) & 3, ws = i >> 11;  // ws = 10 wave + s
    out[i] = w[(16 * nb + (lane & 15)) * DIM + 32 * ws + 4 * (lane >> 4) + (e & 3) + 16 * (e >> 2)];
}
// embed, video: fragment (group of 64 features, step s, i): lane holds feature
// 64 group + 4 (lane % 16) + i, patch channels 32 s + 8 q .. + 7 (zeros from 132 on)
__global__ __launch_bounds__(256) void embed_weights_kernel(const uint16_t* __restrict__ w, uint16_t* __restrict__ out) {
    const int i = blockIdx.x * 256 + threadIdx.x;
    const int e = i & 7, lane = (i >> 3) & 63, b = (i >> 9) & 3, gs = i >> 11;
    const int n = 64 * (gs / 5) + 4 * (lane & 15) + b, k = 32 * (gs % 5) + 8 * (lane >> 4) + e;
    out[i] = k < 132 ? w[n * 132 + k] : (uint16_t)0;
}

// ---------------------------------------------------------------- embed
//
// One grid for both projections, the text's workgroups first, then a small
// launch that sums the text's partial products.
//
// Video: 64 rows x 512 features per workgroup, the patches (132 channels: two
// runs of 66 consecutive floats of the grid) gathered, rounded to bf16 and
// padded with zeros to 160 in LDS; a wave forms 64 rows x 64 features in five
// k32 steps (column r of product block i is feature 4 r + i; so a lane ends
// with four consecutive features and a store instruction writes 256 bytes of
// four rows).  The 56 MB written bound it; nothing is zeroed or read back.
//
// Text (K = 5120, some 26 MB of weights for a few dozen rows): 64 rows x 128
// features x 1/16 of K per workgroup, so that the weights stream through 320
// workgroups at once and are read once; fp32 partial products to the
// workspace, summed in K order.  (Whole K per workgroup, 32 rows x 32 features
// over eight waves, re-reads the text in every feature block: 28 us against 14
// for the text alone.)  Up to EMBED_TXT_MAX rows; longer texts are left to the block's
// GEMM and TXT is 0 here.
constexpr int EMB_K = 160, EMB_LP = EMB_K + 8;  // k (padded) and LDS pitch of a patch row, bf16
constexpr int EW = 8;  // waves of a workgroup
constexpr int EMB_ROWS = 64, EMB_COLS = 64 * EW;
constexpr int TXT_K = 5120, TXT_KW = TXT_K / EMBED_TXT_SPLIT, TXT_S = TXT_KW / 32;
constexpr int TXT_ROWS = 64, TXT_COLS = 16 * EW, TXT_LP = TXT_KW + 8;

__global__ __launch_bounds__(64 * EW, 4) void embed_kernel(EmbedArgs a) {
    __shared__ __align__(16) uint16_t ps[TXT_ROWS * TXT_LP];
    static_assert(TXT_LP >= EMB_LP && TXT_ROWS >= EMB_ROWS, "patch rows fit");
    const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
    const int r16 = lane & 15, q = lane >> 4;
    if ((int)blockIdx.x < a.txt_blocks) {
        const int ks = (int)blockIdx.x % EMBED_TXT_SPLIT, rest = (int)blockIdx.x / EMBED_TXT_SPLIT;
        const int n0 = (rest % (DIM / TXT_COLS)) * TXT_COLS + wave * 16, m0 = rest / (DIM / TXT_COLS) * TXT_ROWS;
        const int rows = min(TXT_ROWS, a.TXT - m0);
        const uint16_t* W = a.txt_w + (size_t)(n0 + r16) * TXT_K + ks * TXT_KW + 8 * q;
        bf16x8 wf[TXT_S];
#pragma unroll
        for (int s = 0; s < TXT_S; s++) wf[s] = *reinterpret_cast<const bf16x8*>(W + 32 * s);
        constexpr int C4 = TXT_KW / 4;  // float4 per row
#pragma unroll
        for (int i = 0; i < TXT_ROWS * C4 / (64 * EW); i++) {
            const int e = i * 64 * EW + tid, r = e / C4, c = e % C4;  // rows past the end repeat the last one
            const f32x4u v = *reinterpret_cast<const f32x4u*>(a.txt + (size_t)(m0 + min(r, rows - 1)) * TXT_K +
                                                              ks * TXT_KW + 4 * c);
            *reinterpret_cast<uint2*>(ps + r * TXT_LP + 4 * c) = make_uint2(bf16x2_rne(v[0], v[1]), bf16x2_rne(v[2], v[3]));
        }
        __syncthreads();
        f32x4 acc[4];
#pragma unroll
        for (int j = 0; j < 4; j++) acc[j] = (f32x4){0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int s = 0; s < TXT_S; s++)
#pragma unroll
            for (int j = 0; j < 4; j++) {
                const bf16x8 af = *reinterpret_cast<const bf16x8*>(ps + (16 * j + r16) * TXT_LP + 32 * s + 8 * q);
                acc[j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wf[s], af, acc[j], 0, 0, 0);
            }
        // lane: features 4 q + t of row 16 j + r16
#pragma unroll
        for (int j = 0; j < 4; j++) {
            const int m = 16 * j + r16;
            if (m < rows)
                *reinterpret_cast<f32x4*>(a.part + ((size_t)ks * a.TXT + m0 + m) * DIM + n0 + 4 * q) = acc[j];
        }
        return;
    }
    const int vb = (int)blockIdx.x - a.txt_blocks;
    constexpr int CB = DIM / EMB_COLS;
    const int row0 = (vb / CB) * EMB_ROWS, n0 = (vb % CB) * EMB_COLS + wave * 64;
    const int rows = min(EMB_ROWS, a.Lv - row0);
    // W fragments first: they do not depend on the patches
    const bf16x8* W = reinterpret_cast<const bf16x8*>(a.vid_w) + (size_t)(n0 / 64) * (EMB_K / 32) * 4 * 64 + lane;
    bf16x8 wf[2][4];
#pragma unroll
    for (int i = 0; i < 4; i++) wf[0][i] = W[i * 64];
    // the patches: pairs of channels (a run of 66 holds whole pairs), 66 per row
    const int H2 = a.H >> 1, W2 = a.W2;
    const size_t gw = (size_t)2 * W2 * 33;  // floats per grid row
#pragma unroll
    for (int i = 0; i < (EMB_ROWS * 66 + 64 * EW - 1) / (64 * EW); i++) {
        const int e = i * 64 * EW + tid;
        if (e < EMB_ROWS * 66) {
            const int r = e / 66, j = 2 * (e % 66);
            const int row = row0 + min(r, rows - 1);
            const int ph = j >= 66, tt = row / (H2 * W2), hh = (row / W2) % H2, ww = row % W2;
            const f32x2u p = *reinterpret_cast<const f32x2u*>(a.grid + ((size_t)tt * a.H + 2 * hh + ph) * gw +
                                                              (size_t)66 * ww + (j - 66 * ph));
            *reinterpret_cast<uint32_t*>(ps + r * EMB_LP + j) = bf16x2_rne(p[0], p[1]);
        }
    }
#pragma unroll
    for (int i = 0; i < (EMB_ROWS * 14 + 64 * EW - 1) / (64 * EW); i++) {  // channels 132 .. 159: zeros
        const int e = i * 64 * EW + tid;
        if (e < EMB_ROWS * 14) *reinterpret_cast<uint32_t*>(ps + (e / 14) * EMB_LP + 132 + 2 * (e % 14)) = 0;
    }
    __syncthreads();
    f32x4 acc[4][4];
#pragma unroll
    for (int i = 0; i < 4; i++)
#pragma unroll
        for (int j = 0; j < 4; j++) acc[i][j] = (f32x4){0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int s = 0; s < EMB_K / 32; s++) {
        if (s + 1 < EMB_K / 32) {
#pragma unroll
            for (int i = 0; i < 4; i++)
                wf[(s + 1) & 1][i] = W[(4 * (s + 1) + i) * 64];
        }
        bf16x8 pf[4];
#pragma unroll
        for (int j = 0; j < 4; j++)
            pf[j] = *reinterpret_cast<const bf16x8*>(ps + (16 * j + r16) * EMB_LP + 32 * s + 8 * q);
#pragma unroll
        for (int i = 0; i < 4; i++)
#pragma unroll
            for (int j = 0; j < 4; j++)
                acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(pf[j], wf[s & 1][i], acc[i][j], 0, 0, 0);
    }
    // lane: features 4 r16 + i of rows 16 j + 4 q + t
    const f32x4u b = *reinterpret_cast<const f32x4u*>(a.vid_b + n0 + 4 * r16);
#pragma unroll
    for (int j = 0; j < 4; j++)
#pragma unroll
        for (int t = 0; t < 4; t++) {
            const int m = 16 * j + 4 * q + t;
            const f32x4u y = {acc[0][j][t] + b[0], acc[1][j][t] + b[1], acc[2][j][t] + b[2], acc[3][j][t] + b[3]};
            if (m < rows) *reinterpret_cast<f32x4u*>(a.x + (size_t)(row0 + m) * DIM + n0 + 4 * r16) = y;
        }
}

// text rows of x: the partial products in K order, plus the bias
__global__ __launch_bounds__(256) void embed_sum_kernel(const float* __restrict__ part, const float* __restrict__ b,
                                                        float* __restrict__ x, int n4) {
    const int i = blockIdx.x * 256 + threadIdx.x;
    if (i >= n4) return;
    f32x4 v[EMBED_TXT_SPLIT];
#pragma unroll
    for (int k = 0; k < EMBED_TXT_SPLIT; k++) v[k] = reinterpret_cast<const f32x4*>(part)[(size_t)k * n4 + i];
    f32x4 y = v[0];
#pragma unroll
    for (int k = 1; k < EMBED_TXT_SPLIT; k++) y += v[k];
    y += *reinterpret_cast<const f32x4u*>(b + 4 * (i % (DIM / 4)));
    *reinterpret_cast<f32x4u*>(x + 4 * (size_t)i) = y;
}

}  // namespace

hipError_t launch_final(const FinalArgs& args, hipStream_t s) {
    if (args.rows <= 0) return hipSuccess;
    FinalArgs a = args;
    const int cus = device_cus(), rounds = (a.rows + 32 * cus - 1) / (32 * cus);
    a.rpw = (a.rows + rounds * cus - 1) / (rounds * cus);
    const dim3 grid((a.rows + a.rpw - 1) / a.rpw), block(512);
    if (a.rpw <= 16) hipLaunchKernelGGL(final_kernel<1>, grid, block, 0, s, a);
    else hipLaunchKernelGGL(final_kernel<2>, grid, block, 0, s, a);
    return hipGetLastError();
}

hipError_t launch_end_weights(const uint16_t* vid_in, uint16_t* vid_in_frag, const uint16_t* vid_out,
                              uint16_t* vid_out_frag, hipStream_t s) {
    static_assert(EMB_K == EMBED_K && FIN_S == 10 && EMB_K == 5 * 32 && FIN_N * DIM % 256 == 0, "fragment order");
    hipLaunchKernelGGL(embed_weights_kernel, dim3(DIM * EMB_K / 256), dim3(256), 0, s, vid_in, vid_in_frag);
    hipLaunchKernelGGL(final_weights_kernel, dim3(FIN_N * DIM / 256), dim3(256), 0, s, vid_out, vid_out_frag);
    return hipGetLastError();
}

hipError_t launch_embed(const EmbedArgs& args, hipStream_t s) {
    static_assert(EMB_K == EMBED_K && DIM % EMB_COLS == 0 && DIM % TXT_COLS == 0, "embed tiling");
    EmbedArgs a = args;
    a.txt_blocks = (a.TXT + TXT_ROWS - 1) / TXT_ROWS * (DIM / TXT_COLS) * EMBED_TXT_SPLIT;
    const int vid = (a.Lv + EMB_ROWS - 1) / EMB_ROWS * (DIM / EMB_COLS);
    hipLaunchKernelGGL(embed_kernel, dim3(a.txt_blocks + vid), dim3(64 * EW), 0, s, a);
    if (a.TXT == 0) return hipGetLastError();
    const int n4 = a.TXT * (DIM / 4);
    hipLaunchKernelGGL(embed_sum_kernel, dim3((n4 + 255) / 256), dim3(256), 0, s, a.part, a.txt_b,
                       a.x + (size_t)a.Lv * DIM, n4);
    return hipGetLastError();
}

}  // namespace awa
