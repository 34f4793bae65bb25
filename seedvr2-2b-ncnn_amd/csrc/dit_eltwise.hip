// dit_eltwise.hip — row-wise and small kernels of the DiT block.
//
//   norm_ada   RMSNorm (no affine, dit_vk.cpp:48-52) then the ada modulation
//              x * scale + shift (dit_vk.cpp:532-545, 584-597), bf16 out:
//              the A operand of the next projection.  One wave64 per row,
//              HBM-bound (reads 10 KiB fp32, writes 5 KiB bf16 per row).
//   ada        AdaCompose (ada_compose.cpp:165-235): emb[6d + K_MAP[k]] +
//              branch vector, the 12 modulation vectors of a layer.
//   pack_mlp   interleave proj_in / proj_in_gate rows for the fused SwiGLU.
//   time_in, gemv_f32   the timestep embedding and its MLP (M = 1 linears,
//              dit_vk.cpp:295-309).
#include <cmath>

#include "dit_internal.hpp"

namespace awa {

namespace {

__device__ inline float wave_sum(float v) {
#pragma unroll
    for (int o = 32; o >= 1; o >>= 1) v += __shfl_xor(v, o);
    return v;
}

constexpr int PER_LANE4 = DIM / 4 / 64;  // float4s per lane per 2560-wide row

__global__ __launch_bounds__(256) void norm_ada_kernel(NormArgs a) {
    const int row = blockIdx.x * 4 + (threadIdx.x >> 6);
    const int lane = threadIdx.x & 63;
    if (row >= a.M) return;
    const float4* x = reinterpret_cast<const float4*>(a.x + (size_t)row * DIM);
    float4 v[PER_LANE4];
    float ss = 0.f;
#pragma unroll
    for (int i = 0; i < PER_LANE4; i++) v[i] = x[i * 64 + lane];
    // the modulation vectors (cached, the same for every row) are loaded
    // while the row is in flight, not after the reduction
    const bool second = row >= a.split;
    const float* sc = second ? a.scale1 : a.scale0;
    const float* sh = second ? a.shift1 : a.shift0;
    float4 s[PER_LANE4], t[PER_LANE4];
    if (sc) {
#pragma unroll
        for (int i = 0; i < PER_LANE4; i++) {
            s[i] = reinterpret_cast<const float4*>(sc)[i * 64 + lane];
            t[i] = reinterpret_cast<const float4*>(sh)[i * 64 + lane];
        }
    }
#pragma unroll
    for (int i = 0; i < PER_LANE4; i++)
        ss += v[i].x * v[i].x + v[i].y * v[i].y + v[i].z * v[i].z + v[i].w * v[i].w;
    ss = wave_sum(ss);
    const float r = 1.0f / sqrtf(ss / (float)DIM + a.eps);
    uint2* out = reinterpret_cast<uint2*>(a.h + (size_t)row * DIM);
#pragma unroll
    for (int i = 0; i < PER_LANE4; i++) {
        float o0 = v[i].x * r, o1 = v[i].y * r, o2 = v[i].z * r, o3 = v[i].w * r;
        if (sc) {
            o0 = o0 * s[i].x + t[i].x;
            o1 = o1 * s[i].y + t[i].y;
            o2 = o2 * s[i].z + t[i].z;
            o3 = o3 * s[i].w + t[i].w;
        }
        out[i * 64 + lane] = make_uint2(bf16x2_rne(o0, o1), bf16x2_rne(o2, o3));
    }
}

// K_MAP of ada_compose.cpp:16: a_sc->1, a_sh->0, a_g->2, m_sc->4, m_sh->3, m_g->5
__constant__ int kAdaSlot[6] = {1, 0, 2, 4, 3, 5};

__global__ __launch_bounds__(256) void ada_kernel(AdaArgs a) {
    const int i = blockIdx.x * 256 + threadIdx.x;
    if (i >= 12 * DIM) return;
    const int d = i % DIM, k = (i / DIM) % 6, f = i / (6 * DIM);
    a.out[i] = a.emb[d * 6 + kAdaSlot[k]] + a.vec[f][k][d];
}

__global__ __launch_bounds__(256) void pack_mlp_kernel(const uint16_t* __restrict__ w_in,
                                                       const uint16_t* __restrict__ w_gate,
                                                       uint16_t* __restrict__ w_cat) {
    const int r = blockIdx.x;          // row of the fused weight
    const int blk = r >> 5, within = r & 31;
    const uint16_t* src = ((blk & 1) ? w_gate : w_in) + (size_t)((blk >> 1) * 32 + within) * DIM;
    const uint4* s4 = reinterpret_cast<const uint4*>(src);
    uint4* d4 = reinterpret_cast<uint4*>(w_cat + (size_t)r * DIM);
    for (int c = threadIdx.x; c < DIM / 8; c += 256) d4[c] = s4[c];
}

// y = act(W x + b): R output rows per wave, x and the rows in 16-byte pieces per
// lane, every load issued before the first use.  Bound by the weights (26 and
// 157 MB): with one value per load and lane and a row per wave 20.6 and 50 us.
typedef float f32x4u __attribute__((ext_vector_type(4), aligned(4)));  // weights are only known to hold floats
template <int IN, int R>
__device__ inline void gemv_rows(const float* __restrict__ W, const float* __restrict__ b, const float* __restrict__ x,
                                 float* __restrict__ y, int out, int silu) {
    constexpr int P = IN / 256;  // pieces per lane and row
    const int o0 = (blockIdx.x * 4 + (threadIdx.x >> 6)) * R;
    const int lane = threadIdx.x & 63;
    if (o0 >= out) return;
    f32x4u w[R][P], xv[P];
#pragma unroll
    for (int r = 0; r < R; r++) {  // rows past the end repeat the last one
        const float* row = W + (size_t)min(o0 + r, out - 1) * IN;
#pragma unroll
        for (int i = 0; i < P; i++) w[r][i] = *reinterpret_cast<const f32x4u*>(row + 4 * (i * 64 + lane));
    }
#pragma unroll
    for (int i = 0; i < P; i++) xv[i] = *reinterpret_cast<const f32x4u*>(x + 4 * (i * 64 + lane));
#pragma unroll
    for (int r = 0; r < R; r++) {
        float acc = 0.f;
#pragma unroll
        for (int i = 0; i < P; i++)
            acc += w[r][i][0] * xv[i][0] + w[r][i][1] * xv[i][1] + w[r][i][2] * xv[i][2] + w[r][i][3] * xv[i][3];
        acc = wave_sum(acc);
        if (lane == 0 && o0 + r < out) {
            float v = acc + b[o0 + r];
            if (silu) v = v / (1.f + expf(-v));
            y[o0 + r] = v;
        }
    }
}

template <int IN, int R>
__global__ __launch_bounds__(256) void gemv_f32_kernel(const float* __restrict__ W, const float* __restrict__ b,
                                                       const float* __restrict__ x, float* __restrict__ y, int out,
                                                       int silu) {
    gemv_rows<IN, R>(W, b, x, y, out, silu);
}

struct Sinusoid {
    float v[256];
};

// the first linear, its input in the kernel arguments
__global__ __launch_bounds__(256) void time_in_kernel(Sinusoid s, const float* __restrict__ W,
                                                      const float* __restrict__ b, float* __restrict__ y, int out) {
    __shared__ float x[256];
    x[threadIdx.x] = s.v[threadIdx.x];
    __syncthreads();
    gemv_rows<256, 1>(W, b, x, y, out, 1);
}

}  // namespace

hipError_t launch_norm_ada(const NormArgs& a, hipStream_t s) {
    if (a.M <= 0) return hipSuccess;
    hipLaunchKernelGGL(norm_ada_kernel, dim3((a.M + 3) / 4), dim3(256), 0, s, a);
    return hipGetLastError();
}

hipError_t launch_ada(const AdaArgs& a, hipStream_t s) {
    hipLaunchKernelGGL(ada_kernel, dim3((12 * DIM + 255) / 256), dim3(256), 0, s, a);
    return hipGetLastError();
}

hipError_t launch_pack_mlp(const uint16_t* w_in, const uint16_t* w_gate, int mlp, uint16_t* w_cat,
                           hipStream_t s) {
    hipLaunchKernelGGL(pack_mlp_kernel, dim3(2 * mlp), dim3(256), 0, s, w_in, w_gate, w_cat);
    return hipGetLastError();
}

hipError_t launch_time_mlp(float t, const float* const w[3], const float* const b[3], float* e1, float* e2, float* emb,
                           hipStream_t s) {
    // The 256 sinusoid values are formed on the host with the reference's
    // expression (dit_vk.cpp:295-302) and passed by value.
    Sinusoid v{};
    constexpr int half = 128;
    for (int j = 0; j < 2 * half; j++) {
        // float argument, double exp, rounded to float: as C's exp()
        const float freq = (float)::exp((double)(-logf(10000.f) * (j % half) / half));
        v.v[j] = (j < half) ? sinf(t * freq) : cosf(t * freq);
    }
    hipLaunchKernelGGL(time_in_kernel, dim3(DIM / 4), dim3(256), 0, s, v, w[0], b[0], e1, DIM);
    hipLaunchKernelGGL((gemv_f32_kernel<DIM, 1>), dim3(DIM / 4), dim3(256), 0, s, w[1], b[1], e1, e2, DIM, 1);
    hipLaunchKernelGGL((gemv_f32_kernel<DIM, 2>), dim3(DIT_EMB / 8), dim3(256), 0, s, w[2], b[2], e2, emb, DIT_EMB, 0);
    return hipGetLastError();
}

}  // namespace awa
