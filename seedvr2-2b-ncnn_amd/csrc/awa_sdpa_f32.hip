// awa_sdpa_f32.hip — varlen window attention with fp32 storage on CDNA4 matrix
// cores (v_mfma_f32_16x16x32_f16 on split operands).
//
// The fp32 counterpart of sdpa_bf16_kernel (awa_sdpa.hip), for AWA_F32
// storage: the reference's fp32 attention (dit_vk.cpp:406-439).  Every matrix
// operand x is carried as two fp16 values, hi = fp16(x 2^a) and lo =
// fp16(x 2^a - hi), which hold 23 of fp32's 24 significand bits (hi's rounding
// error is a multiple of 2^-24 of it, lo keeps 11 bits of that and a sign), and
// a product is three MFMAs, lo hi + hi lo + hi hi, accumulated in fp32; the
// dropped lo lo is at most 2^-22 of the product.  The fp16 MFMA does 16 times the work of
// the fp32 one, so three of them still do over five times.  Against 64 bits
// the result is no further off than a chain of fp32 MFMAs, whose 32 (here 12)
// roundings of the running sum per score outweigh the operands' last bit
// (relative error 3.2e-7 against 4.3e-7 on N(0, 1) inputs at 360p, 3.6e-7
// against 5.0e-7 at 1080p).
//
// The powers of two 2^a bring every block of 16 rows (K and V: set by the pack
// kernel per block and head; Q: per row) to at most 2^15: an element 2^-17 of
// its block's largest still has its 23 bits, smaller ones are held to 2^-40 of
// the largest.  They are undone exactly: in the factor of the scores, in P
// before its split, and in the normalisation of O.  P = exp2(s - m) is split
// like the rest.  Windows whose V spans more than that holds (SPREAD_CHANNELS,
// SPREAD_ROWS) take three bf16 values of V and P instead (wide_item), those with
// infinities, the ends of fp32's range or gains that cancel fp32 MFMAs
// (full_queries).  Up to there the error is that of N(0, 1) inputs: half of the
// rows 2^-5 of the others, or a sixteenth of the channels 2^7 times the others,
// 3.1e-7 to 3.3e-7 at 360p and at most 6.1e-7 in the worst channel, against 4.4e-7
// and 9.0e-7 as fp32 MFMAs; with 1 % of the inputs 8 times as large 5.3e-7 against
// 6.7e-7, with gains of 4 6.4e-7 against 1.1e-6.  Scores that a single channel carries
// (15 in log2 units) show the missing bit and the dropped lo lo: 9.8e-7 against
// 6.8e-7 (8.8e-7 with lo lo as a fourth MFMA, at 5 % of the op's time).
//
// The query rows are normalised and rotated here (each is read by one
// workgroup), K and V come from the pack kernel as hi and lo tiles in fragment
// order (f32_kfrag in awa_internal.hpp): the LDS DMA copies it linearly and a
// wave's fragment read is 1 KiB of consecutive LDS.  Scores are formed
// transposed, S^T = K Q^T, so that a lane owns one query column; the
// probabilities leave the accumulator in the B-operand layout of
// O^T = V^T P^T.  Video query rows are scattered back to token order
// (dit_vk.cpp:445-455); text query rows go to per-window fp32 partials that
// the coalesce kernel averages in window order (dit_vk.cpp:440-444).
#include "awa_internal.hpp"

namespace awa {

namespace {

typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));
typedef __attribute__((address_space(3))) void* lptr_t;
typedef float f32x2 __attribute__((ext_vector_type(2)));
typedef __attribute__((address_space(4))) f32x2 cfloat2_t;

// A work item (GeomPlan::sched_desc): one head, one window and one or two of its
// query tiles; the window's tiles are its video tiles, then the text tiles of
// its text set.
struct Item {
    int h, w, kq0, kq1, vbase, nvt, tbase, ntt, f, txt;
    __device__ int tile(int kk) const { return kk < nvt ? vbase + kk : tbase + (kk - nvt); }
    __device__ int nvalid(int kk) const {
        return kk < nvt ? min(TILE, f - TILE * kk) : min(TILE, txt - TILE * (kk - nvt));
    }
    // 32-key units: of the video rows, then of the text rows (a tile's empty
    // second half is none)
    __device__ int vid_units() const { return (f + 31) >> 5; }
    __device__ int units() const { return vid_units() + ((txt + 31) >> 5); }
    // half tile (2 tile + half) and valid keys of unit u
    __device__ int unit_half(int u) const {
        const int nv = vid_units();
        return u < nv ? 2 * vbase + u : 2 * tbase + (u - nv);
    }
    __device__ int unit_valid(int u) const {
        const int nv = vid_units();
        return u < nv ? f - 32 * u : txt - 32 * (u - nv);
    }
};

// Sum over the four lanes l % 16 + 16 i, as max4.
__device__ inline float sum4(float v) {
    auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
    v = __uint_as_float(r[0]) + __uint_as_float(r[1]);
    r = __builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v), false, false);
    return __uint_as_float(r[0]) + __uint_as_float(r[1]);
}

// A wave-uniform value kept in a scalar register.
__device__ inline float scalar(float v) {
    return __int_as_float(__builtin_amdgcn_readfirstlane(__float_as_int(v)));
}
// Maximum over the wave, as a scalar.
__device__ inline float wave_max(float v) {
    v = max4(v);
#pragma unroll
    for (int o = 8; o >= 1; o >>= 1) v = fmaxf(v, __shfl_xor(v, o));
    return scalar(v);
}

// P is at most 2^M_STALE (the running maximum stays until a tile's exceeds it by
// more, so that O is rarely rescaled), times 2^P_SHIFT and the V block's power of
// two relative to the window's largest (2^-SPREAD_ROWS at least, else the
// window goes to wide_item): below 2^16, and down to 2^-22 of the largest
// (2^-16 for the smallest blocks) in fp16's normal range; below that it is held
// to 2^-33 (2^-27).
constexpr float P_SHIFT = 8.f, M_STALE = 7.f;

// The largest query value times the largest key value up to which the split
// holds the scores whatever the gains.  Values are held to 2^-40 of the largest of
// their row or block, so a score is off by up to some 2^-36 of this product: far
// below the rounding of its own sum, unless the gains of q and k cancel channel by
// channel (2^10 against 2^-10: product 2^21, error 1.8e-6 for 3.2e-7).  2^13 leaves
// 2^-26 (N(0, 1) rows and gains of 1: 2^4).  Above it the largest gains must meet
// in one channel, to GAIN_SPREAD.
constexpr float QK_MAX = 8192.f, GAIN_SPREAD = 64.f;

constexpr uint32_t FU_BYTES = 32 * HEAD_D * 4;  // a K or V unit (32 keys): hi and lo, 16 KiB
constexpr uint32_t V_RING = 2 * FU_BYTES;       // LDS stage: two K units, then two V units
constexpr uint32_t STAGE_BYTES = 4 * FU_BYTES;  // 64 KiB

// A wave's quarter of a unit (4 KiB) by LDS DMA, linear: instruction offset j
// moves the global address and the LDS destination alike.  From asm, with the
// kernel's own waits (unit_barrier) before any wave reads the unit.
#pragma clang diagnostic push
#pragma clang diagnostic ignored "-Winline-asm"
__device__ inline void dma_quarter(const void* unit, uint32_t part, uint32_t lane16, uint32_t m) {
    const __amdgpu_buffer_rsrc_t r = __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(unit), 0, FU_BYTES, 0x00020000);
    asm volatile(
        "s_mov_b32 m0, %[m]\n\ts_nop 0\n\t"
        "buffer_load_dwordx4 %[v], %[r], %[so] offen lds\n\t"
        "buffer_load_dwordx4 %[v], %[r], %[so] offen offset:1024 lds\n\t"
        "buffer_load_dwordx4 %[v], %[r], %[so] offen offset:2048 lds\n\t"
        "buffer_load_dwordx4 %[v], %[r], %[so] offen offset:3072 lds"
        :
        : [v] "v"(lane16), [r] "s"(r), [so] "s"(part), [m] "s"(m + part)
        : "memory", "m0");
}
#pragma clang diagnostic pop
// This wave's DMA has landed and its LDS reads are done, then the barrier.
__device__ inline void unit_barrier() { asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory"); }

// ---- windows with infinities, values at the ends of fp32's range or gains of q
// and k that cancel (VEXP_FULL, QK_MAX, GAIN_SPREAD): fp32 MFMAs
//
// The same workgroup and the same output for its query tile t, 16 queries a wave, as
// plain fp32: K and V rows straight from vqkv / tqkv (K normalised and rotated
// as the pack kernel does) into LDS, 32 keys at a time, and
// v_mfma_f32_16x16x4_f32 for both products.  The fp32 MFMA's 32 cycles bound it,
// so it neither pipelines nor shares a unit between two query blocks.
// 1080p shifted with every window here: 454 us a pass, 360p 129.
constexpr int EX_P = HEAD_D + 4;  // LDS pitch of a row (floats)
constexpr int EX_STAGE = 2 * 32 * EX_P;  // K and V rows of a unit
template <bool kSplit>
__device__ inline void full_queries(const SdpaArgs& a, const Item& wt, float* lds, int t) {
    const int h = wt.h;
    int tid = threadIdx.x;
    asm volatile("" : "+v"(tid));  // addresses of its own, none held across
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63;
    const int half = kSplit ? wave >> 2 : 0, w4 = wave & 3, r16 = lane & 15, q = lane >> 4;
    const int nu = wt.units(), n0 = kSplit ? (nu + 1) >> 1 : nu;
    const int ubeg = half ? n0 : 0, uend = half ? nu : n0;
    float* ks = lds + half * EX_STAGE;
    float* vs = ks + 32 * EX_P;

    // query r16 of the block, channels 32 s + 8 q .. + 7 (k step 8 s + e pairs
    // channel 32 s + 8 q + e of the four lane groups, in K's fragments alike)
    const int kq = t ? wt.kq1 : wt.kq0, slot = 16 * w4 + r16;
    const bool qtxt = kq >= wt.nvt;
    const uint32_t row_ofs =
        a.vrow[(size_t)(qtxt ? a.n_vid_tiles + (kq - wt.nvt) : wt.vbase + kq) * TILE + vrow_pos(slot)];
    const int2 qmeta = reinterpret_cast<const int2*>(a.tile_meta)[wt.tile(kq)];
    float x[32];
    {
        const float* row = reinterpret_cast<const float*>(qtxt ? a.tsrc : a.vsrc) + row_ofs + h * HEAD_D + 8 * q;
        const float* cs = reinterpret_cast<const float*>(qtxt ? a.tcs : a.vcs) +
                          ((size_t)qmeta.x + min(slot, qmeta.y - 1)) * (2 * CS_STRIDE) + 8 * q;
        const float* gain = (qtxt ? a.nq_t : a.nq_v) + 8 * q;
        float ss = 0.f;
#pragma unroll
        for (int i = 0; i < 32; i++) {
            x[i] = row[32 * (i >> 3) + (i & 7)];
            ss += x[i] * x[i];
        }
        const float n = sqrtf(sum4(ss) / (float)HEAD_D + a.eps), in = 1.f / n;
#pragma unroll
        for (int i = 0; i < 32; i += 2) {
            const int c = 32 * (i >> 3) + (i & 7);
            const float x0 = div_by(x[i], n, in) * gain[c], x1 = div_by(x[i + 1], n, in) * gain[c + 1];
            x[i] = (x0 * cs[c] - x1 * cs[c + 1]) * a.qscale;
            x[i + 1] = (x1 * cs[c] + x0 * cs[c + 1]) * a.qscale;
        }
    }

    // a unit's rows: eight threads a row, 16 channels each
    const int krow = (tid & 255) >> 3, kc = 16 * (tid & 7);
    float4 rk[4], rv[4], rc[4];
    auto load_unit = [&](int u) __attribute__((always_inline)) {
        const int t2 = wt.unit_half(u), tile = t2 >> 1, sl = 32 * (t2 & 1) + krow;
        const bool txt = u >= wt.vid_units();
        const uint32_t ofs = a.vrow[(size_t)(txt ? a.n_vid_tiles + (tile - wt.tbase) : tile) * TILE + vrow_pos(sl)];
        const int2 meta = reinterpret_cast<const int2*>(a.tile_meta)[tile];
        const float* row = reinterpret_cast<const float*>(txt ? a.tsrc : a.vsrc) + ofs + DIM + h * HEAD_D + kc;
        const float* cs = reinterpret_cast<const float*>(txt ? a.tcs : a.vcs) +
                          ((size_t)meta.x + min(sl, meta.y - 1)) * (2 * CS_STRIDE) + kc;
#pragma unroll
        for (int i = 0; i < 4; i++) {
            rk[i] = reinterpret_cast<const float4*>(row)[i];
            rv[i] = reinterpret_cast<const float4*>(row + DIM)[i];
            rc[i] = reinterpret_cast<const float4*>(cs)[i];
        }
    };
    auto store_unit = [&](int u) __attribute__((always_inline)) {
        const float* gain = (u >= wt.vid_units() ? a.nk_t : a.nk_v) + kc;
        float ss = 0.f;
#pragma unroll
        for (int i = 0; i < 4; i++) ss += rk[i].x * rk[i].x + rk[i].y * rk[i].y + rk[i].z * rk[i].z + rk[i].w * rk[i].w;
#pragma unroll
        for (int o = 1; o <= 4; o <<= 1) ss += __shfl_xor(ss, o);
        const float n = sqrtf(ss / (float)HEAD_D + a.eps), in = 1.f / n;
        const bool valid = krow < wt.unit_valid(u);  // V of a masked key: 0, whatever its weight's 0 meets
#pragma unroll
        for (int i = 0; i < 4; i++) {
            const float k0 = div_by(rk[i].x, n, in) * gain[4 * i], k1 = div_by(rk[i].y, n, in) * gain[4 * i + 1];
            const float k2 = div_by(rk[i].z, n, in) * gain[4 * i + 2], k3 = div_by(rk[i].w, n, in) * gain[4 * i + 3];
            *reinterpret_cast<float4*>(ks + krow * EX_P + kc + 4 * i) =
                make_float4(k0 * rc[i].x - k1 * rc[i].y, k1 * rc[i].x + k0 * rc[i].y, k2 * rc[i].z - k3 * rc[i].w,
                            k3 * rc[i].z + k2 * rc[i].w);
            *reinterpret_cast<float4*>(vs + krow * EX_P + kc + 4 * i) = valid ? rv[i] : make_float4(0.f, 0.f, 0.f, 0.f);
        }
    };

    f32x4 oacc[8];
#pragma unroll
    for (int db = 0; db < 8; db++) oacc[db] = (f32x4){0.f, 0.f, 0.f, 0.f};
    float m = -INFINITY, l = 0.f;
    if (ubeg < uend) load_unit(ubeg);
    for (int i = 0; i < n0; i++) {  // the same iteration count in both halves
        const int u = ubeg + i;
        __syncthreads();  // every wave is done with the unit before
        if (u < uend) store_unit(u);
        __syncthreads();
        if (u + 1 < uend) load_unit(u + 1);
        if (u >= uend) continue;  // uniform per half
        f32x4 s[2];
        const int kv = wt.unit_valid(u);
        float mx = -INFINITY;
#pragma unroll
        for (int kb = 0; kb < 2; kb++) {
            s[kb] = (f32x4){0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int st = 0; st < 32; st += 4) {
                const f32x4 k4 = *reinterpret_cast<const f32x4*>(ks + (16 * kb + r16) * EX_P + 32 * (st >> 3) + 8 * q + (st & 7));
#pragma unroll
                for (int e = 0; e < 4; e++) s[kb] = __builtin_amdgcn_mfma_f32_16x16x4f32(k4[e], x[st + e], s[kb], 0, 0, 0);
            }
#pragma unroll
            for (int r = 0; r < 4; r++) {
                if (16 * kb + 4 * q + r >= kv) s[kb][r] = -INFINITY;
                mx = fmaxf(mx, s[kb][r]);
            }
        }
        const float m_new = fmaxf(m, max4(mx));  // finite: every unit has a valid key
        const float alpha = __builtin_amdgcn_exp2f(m - m_new);
        m = m_new;
        float psum = 0.f;
#pragma unroll
        for (int kb = 0; kb < 2; kb++)
#pragma unroll
            for (int r = 0; r < 4; r++) {
                s[kb][r] = __builtin_amdgcn_exp2f(s[kb][r] - m);
                psum += s[kb][r];
            }
        l = l * alpha + psum;  // this lane's keys; summed over the row at the end
#pragma unroll
        for (int db = 0; db < 8; db++) oacc[db] *= alpha;
#pragma unroll
        for (int kb = 0; kb < 2; kb++)
#pragma unroll
            for (int r = 0; r < 4; r++)
#pragma unroll
                for (int db = 0; db < 8; db++)
                    oacc[db] = __builtin_amdgcn_mfma_f32_16x16x4f32(vs[(16 * kb + 4 * q + r) * EX_P + 16 * db + r16],
                                                                    s[kb][r], oacc[db], 0, 0, 0);
    }
    l = sum4(l);
    if constexpr (kSplit) {  // half 1 leaves its share past the stages, half 0 merges it
        f32x4* pub = reinterpret_cast<f32x4*>(lds + 2 * EX_STAGE) + (size_t)w4 * (8 * 64) + lane;
        float* pml = lds + 2 * EX_STAGE + 4 * 8 * 64 * 4 + w4 * (2 * 64) + lane;
        if (half == 1) {
#pragma unroll
            for (int db = 0; db < 8; db++) pub[64 * db] = oacc[db];
            pml[0] = m;
            pml[64] = l;
        }
        __syncthreads();
        if (half == 1) return;
        const float m1 = pml[0], l1 = pml[64], mm = fmaxf(m, m1);
        const float a0 = __builtin_amdgcn_exp2f(m - mm), a1 = __builtin_amdgcn_exp2f(m1 - mm);
        l = l * a0 + l1 * a1;
#pragma unroll
        for (int db = 0; db < 8; db++) oacc[db] = oacc[db] * a0 + pub[64 * db] * a1;
    }
    if (slot >= wt.nvalid(kq)) return;  // padding
    float* dst = qtxt ? a.tpart + ((size_t)wt.w * a.txt_len + TILE * (kq - wt.nvt) + slot) * DIM
                      : reinterpret_cast<float*>(a.vattn) + row_ofs / 3;
    const float inv = 1.f / l;
#pragma unroll
    for (int db = 0; db < 8; db++) *reinterpret_cast<f32x4*>(dst + h * HEAD_D + 16 * db + 4 * q) = oacc[db] * inv;
}

// The rows of a wave's query blocks nq w4 + qb (nq = 2: blocks 4 .. 7 are of the
// second query tile): element offsets in vqkv / tqkv, and the tiles' records.
struct QueryRows {
    uint32_t ofs[2];
    int2 meta[2];
};
__device__ inline QueryRows query_rows(const SdpaArgs& a, const Item& wt, int nq, int w4, int r16) {
    QueryRows r;
#pragma unroll
    for (int qb = 0; qb < 2; qb++) {
        const int blk = nq * w4 + min(qb, nq - 1), kq = blk < 4 ? wt.kq0 : wt.kq1, slot = 16 * (blk & 3) + r16;
        const int row_tile = kq >= wt.nvt ? a.n_vid_tiles + (kq - wt.nvt) : wt.vbase + kq;
        r.ofs[qb] = a.vrow[(size_t)row_tile * TILE + vrow_pos(slot)];
        r.meta[qb] = reinterpret_cast<const int2*>(a.tile_meta)[wt.tile(kq)];
    }
    return r;
}

// This wave's queries, 16-row blocks NQ w4 + qb of the item, normalised, rotated and
// split (2^-a to cq): every load issued before the first use.
template <int NQ>
__device__ inline void load_queries(const SdpaArgs& a, const Item& wt, const QueryRows& rows, int w4, int lane,
                                    f16x8 (&qh)[NQ][4], f16x8 (&ql)[NQ][4], float (&cq)[NQ]) {
    const int h = wt.h, r16 = lane & 15, q = lane >> 4;
    float4 xr[NQ][8], cs[NQ][8];
#pragma unroll
    for (int qb = 0; qb < NQ; qb++) {
        const int blk = NQ * w4 + qb, kq = blk < 4 ? wt.kq0 : wt.kq1, slot = 16 * (blk & 3) + r16;
        const bool txt = kq >= wt.nvt;
        const float* row = reinterpret_cast<const float*>(txt ? a.tsrc : a.vsrc) + rows.ofs[qb] + h * HEAD_D + 8 * q;
        const float4* cst = reinterpret_cast<const float4*>(txt ? a.tcs : a.vcs) +
                            ((size_t)rows.meta[qb].x + min(slot, rows.meta[qb].y - 1)) * (CS_STRIDE / 2) + 2 * q;
#pragma unroll
        for (int i = 0; i < 8; i++) xr[qb][i] = *reinterpret_cast<const float4*>(row + 32 * (i >> 1) + 4 * (i & 1));
#pragma unroll
        for (int i = 0; i < 8; i++) cs[qb][i] = cst[8 * (i >> 1) + (i & 1)];
    }

#pragma unroll
    for (int qb = 0; qb < NQ; qb++) {
        float x[32];
        float ss = 0.f;
        const float* gain = ((NQ * w4 + qb < 4 ? wt.kq0 : wt.kq1) >= wt.nvt ? a.nq_t : a.nq_v) + 8 * q;
        float gr[32];
#pragma unroll
        for (int i = 0; i < 32; i++) gr[i] = gain[32 * (i >> 3) + (i & 7)];
#pragma unroll
        for (int i = 0; i < 8; i++) {
            x[4 * i] = xr[qb][i].x; x[4 * i + 1] = xr[qb][i].y; x[4 * i + 2] = xr[qb][i].z; x[4 * i + 3] = xr[qb][i].w;
        }
#pragma unroll
        for (int i = 0; i < 32; i++) ss += x[i] * x[i];
        ss = sum4(ss);
        // x / n g, rotated, times the softmax scale
        const float in = a.qscale / sqrtf(ss / (float)HEAD_D + a.eps);
        float mx = 0.f;
#pragma unroll
        for (int i = 0; i < 8; i++) {
            const float c4[4] = {cs[qb][i].x, cs[qb][i].y, cs[qb][i].z, cs[qb][i].w};
#pragma unroll
            for (int p = 0; p < 4; p += 2) {
                const float x0 = x[4 * i + p] * in * gr[4 * i + p], x1 = x[4 * i + p + 1] * in * gr[4 * i + p + 1];
                x[4 * i + p] = x0 * c4[p] - x1 * c4[p + 1];
                x[4 * i + p + 1] = x1 * c4[p] + x0 * c4[p + 1];
                mx = fmaxf(mx, fmaxf(fabsf(x[4 * i + p]), fabsf(x[4 * i + p + 1])));
            }
        }
        const float f = split_scale(max4(mx), SPLIT_FLOOR_QK);
        cq[qb] = 1.f / f;
#pragma unroll
        for (int st = 0; st < 4; st++) {
            float y[8];
            uint32_t hi[4], lo[4];
#pragma unroll
            for (int i = 0; i < 8; i++) y[i] = x[8 * st + i] * f;
            split8(y, hi, lo);
            qh[qb][st] = __builtin_bit_cast(f16x8, hi);
            ql[qb][st] = __builtin_bit_cast(f16x8, lo);
        }
        __builtin_amdgcn_sched_barrier(0);  // one block's gains at a time: registers
    }
}

// The largest V exponent of the window, in whose units P V is accumulated, or,
// where the split does not hold the window, VEXP_WIDE (wide_item) or VEXP_FULL
// (full_queries): the same in every wave.
__device__ inline float window_vmax(const SdpaArgs& a, const Item& wt, int lane) {
    const size_t head = (size_t)wt.h * a.n_tiles * 4;
    const float *ke = a.kexp + head, *ve = a.vexp + head, *vr = a.vrmin + head;
    // the largest gains of q and of k, and their largest product in one channel
    static_assert(HEAD_D == 128, "two gains per lane");
    float gq = 0.f, gk = 0.f, gqk = 0.f;
#pragma unroll
    for (int i = 0; i < 2; i++) {
        const float x = fmaxf(fabsf(a.nq_v[lane + 64 * i]), fabsf(a.nq_t[lane + 64 * i]));
        const float y = fmaxf(fabsf(a.nk_v[lane + 64 * i]), fabsf(a.nk_t[lane + 64 * i]));
        gq = fmaxf(gq, x);
        gk = fmaxf(gk, y);
        gqk = fmaxf(gqk, x * y);
    }
    float vmax = VEXP_ZERO, vmin = VEXP_WIDE, kmax = 0.f;
    for (int i = lane; i < 4 * (wt.nvt + wt.ntt); i += 64) {
        const int b = 4 * wt.tile(i >> 2) + (i & 3);
        vmax = fmaxf(vmax, ve[b]);
        vmin = fminf(vmin, vr[b]);
        kmax = fmaxf(kmax, ke[b]);
    }
    vmax = wave_max(vmax);
    vmin = -wave_max(-vmin);
    // a normalised query's largest value is below sqrt(2 128) qscale = 2.05 times
    // its largest gain, a key's below 2^15 times its block's 2^-a
    gq = wave_max(gq);
    const float qk = gq * wave_max(kmax) * 65536.f;
    if (vmax == VEXP_FULL || !(qk < 0x1p100f) || (qk > QK_MAX && gq * wave_max(gk) > GAIN_SPREAD * wave_max(gqk)))
        return VEXP_FULL;
    return vmin < vmax - SPREAD_ROWS || (wt.f < 16 && wt.txt < 16) ? VEXP_WIDE : vmax;
}

// ---- windows whose V the split does not hold
//
// run_item with P V formed from three bf16 values of V and of P (split3: all 24
// significand bits and fp32's exponents; six MFMAs a product, the dropped ones
// below 2^-25 of it).  Nothing of V is scaled, so channels do not depend on each
// other and any finite value keeps all its bits.  K comes by DMA as there; V rows
// are gathered from vqkv / tqkv a unit ahead, each thread the eight keys of two
// channels, and reach LDS as three planes of fragments.  Not pipelined between
// units.
// With every window here 1080p shifted takes 219 us a pass and 360p 60 (the fp32 MFMA
// kernel that the split replaced 371 and 60, split operands 171 and 45), with less
// error than either: 3.1e-7 at 360p, worst channel 4.3e-7.
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef unsigned u32x4 __attribute__((ext_vector_type(4)));
// eight floats = the sum of three bf16 vectors, largest first
__device__ inline void split3(const float* x, bf16x8 (&f)[3]) {
    u32x4 u[3];
#pragma unroll
    for (int i = 0; i < 4; i++) {
        float a = x[2 * i], b = x[2 * i + 1];
#pragma unroll
        for (int p = 0; p < 3; p++) {
            u[p][i] = bf16x2_rne(a, b);
            a -= __uint_as_float(u[p][i] << 16);
            b -= __uint_as_float(u[p][i] & 0xffff0000u);
        }
    }
#pragma unroll
    for (int p = 0; p < 3; p++) f[p] = __builtin_bit_cast(bf16x8, u[p]);
}

template <int NQ, bool kSplit>
__device__ inline void wide_item(const SdpaArgs& a, const Item& wt, const QueryRows& rows, unsigned char* lds) {
    const int h = wt.h;
    int tid = threadIdx.x;
    asm volatile("" : "+v"(tid));  // addresses of its own, none held across
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63;
    const int half = kSplit ? wave >> 2 : 0, w4 = wave & 3, r16 = lane & 15, q = lane >> 4;
    const int nu = wt.units(), n0 = kSplit ? (nu + 1) >> 1 : nu;
    const int ubeg = half ? n0 : 0, uend = half ? nu : n0;
    // LDS of a half: two K units, then V's planes [plane][channel block][lane]
    static_assert(V_RING + 3 * 8 * 1024 <= STAGE_BYTES, "the planes fit");
    unsigned char* stage = lds + half * STAGE_BYTES;
    const uint32_t ldsb = (uint32_t)(uintptr_t)(lptr_t)lds + half * STAGE_BYTES;
    const f16x8* kf = reinterpret_cast<const f16x8*>(stage) + lane;
    bf16x8* vf = reinterpret_cast<bf16x8*>(stage + V_RING) + lane;
    const unsigned char* Kh = reinterpret_cast<const unsigned char*>(a.Kp) + (size_t)h * a.n_tiles * (2 * FU_BYTES);
    const cfloat2_t* ke = (const cfloat2_t*)(a.kexp) + (size_t)h * a.n_tiles * 2;
    auto fetch_k = [&](int u, int slot) __attribute__((always_inline)) {
        if (u < uend)
            dma_quarter(Kh + (size_t)wt.unit_half(u) * FU_BYTES, 4096u * w4, 16u * lane, ldsb + slot * FU_BYTES);
    };
    // V of a unit: keys {4 q + e, 16 + 4 q + e} of channels 16 (w4 + 4 j) + r16
    uint32_t vofs[8];  // rows of the unit after the one in rv
    float rv[16];
    auto load_rows = [&](int u) __attribute__((always_inline)) {
        const int t2 = wt.unit_half(u), tile = t2 >> 1;
        const uint32_t* vr = a.vrow + (size_t)(u >= wt.vid_units() ? a.n_vid_tiles + (tile - wt.tbase) : tile) * TILE;
#pragma unroll
        for (int e = 0; e < 8; e++) vofs[e] = vr[vrow_pos(32 * (t2 & 1) + 16 * (e >> 2) + 4 * q + (e & 3))];
    };
    auto load_v = [&](int u) __attribute__((always_inline)) {
        const float* src =
            reinterpret_cast<const float*>(u >= wt.vid_units() ? a.tsrc : a.vsrc) + 2 * DIM + h * HEAD_D + 16 * w4 + r16;
#pragma unroll
        for (int e = 0; e < 8; e++)
#pragma unroll
            for (int j = 0; j < 2; j++) rv[8 * j + e] = src[vofs[e] + 64 * j];
    };
    fetch_k(ubeg, 0);
    if (ubeg < uend) load_rows(ubeg);
    f16x8 qh[NQ][4], ql[NQ][4];
    float cq[NQ];
    load_queries(a, wt, rows, w4, lane, qh, ql, cq);
    if (ubeg < uend) {
        load_v(ubeg);
        if (ubeg + 1 < uend) load_rows(ubeg + 1);
    }

    f32x4 oacc[8][NQ];
    float m[NQ], l[NQ];
#pragma unroll
    for (int qb = 0; qb < NQ; qb++) {
        m[qb] = -INFINITY;
        l[qb] = 0.f;
#pragma unroll
        for (int db = 0; db < 8; db++) oacc[db][qb] = (f32x4){0.f, 0.f, 0.f, 0.f};
    }
    for (int i = 0; i < n0; i++) {  // the same iteration count in both halves
        const int u = ubeg + i, slot = i & 1;
        unit_barrier();  // K(u) has landed, every wave is done with V(u - 1) and K(u - 1)
        fetch_k(u + 1, slot ^ 1);
        bf16x8 pf[NQ][3];
        if (u < uend) {  // uniform per half
#pragma unroll
            for (int j = 0; j < 2; j++) {
                bf16x8 f[3];
                split3(rv + 8 * j, f);
#pragma unroll
                for (int p = 0; p < 3; p++) vf[64 * (8 * p + w4 + 4 * j)] = f[p];
            }
            if (u + 1 < uend) load_v(u + 1);
            if (u + 2 < uend) load_rows(u + 2);
            // scores: lane has keys 16 kb + 4 q + r of query r16
            f32x4 s[2][NQ];
#pragma unroll
            for (int st = 0; st < 4; st++) {
                f16x8 f[4];
#pragma unroll
                for (int e = 0; e < 4; e++) f[e] = kf[slot * (FU_BYTES / 16) + 64 * f32_kfrag(e >> 1, st, e & 1)];
#pragma unroll
                for (int pr = 0; pr < 3; pr++)
#pragma unroll
                    for (int kb = 0; kb < 2; kb++)
#pragma unroll
                        for (int qb = 0; qb < NQ; qb++)
                            s[kb][qb] = __builtin_amdgcn_mfma_f32_16x16x32_f16(
                                f[2 * kb + (pr == 0)], pr == 1 ? ql[qb][st] : qh[qb][st],
                                st == 0 && pr == 0 ? (f32x4){0.f, 0.f, 0.f, 0.f} : s[kb][qb], 0, 0, 0);
            }
            const int kv = wt.unit_valid(u);
            const f32x2 kc = ke[wt.unit_half(u)];
#pragma unroll
            for (int qb = 0; qb < NQ; qb++) {
                float p[8], mx = -INFINITY;
#pragma unroll
                for (int e = 0; e < 8; e++) {
                    p[e] = 16 * (e >> 2) + 4 * q + (e & 3) < kv ? s[e >> 2][qb][e & 3] * (cq[qb] * kc[e >> 2]) : -INFINITY;
                    mx = fmaxf(mx, p[e]);
                }
                mx = max4(mx);
                if (__any(mx > m[qb])) {
                    const float m_new = fmaxf(m[qb], mx), alpha = __builtin_amdgcn_exp2f(m[qb] - m_new);
                    m[qb] = m_new;
                    l[qb] *= alpha;
#pragma unroll
                    for (int db = 0; db < 8; db++) oacc[db][qb] *= alpha;
                }
#pragma unroll
                for (int e = 0; e < 8; e++) {
                    p[e] = __builtin_amdgcn_exp2f(p[e] - m[qb]);
                    l[qb] += p[e];  // this lane's keys; summed over the row at the end
                }
                split3(p, pf[qb]);
            }
        }
        asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");  // V(u)'s planes are complete
        if (u < uend) {
            constexpr int order[6][2] = {{2, 0}, {0, 2}, {1, 1}, {1, 0}, {0, 1}, {0, 0}};  // small products first
#pragma unroll
            for (int db = 0; db < 8; db += 2) {
                bf16x8 f[2][3];
#pragma unroll
                for (int e = 0; e < 2; e++)
#pragma unroll
                    for (int p = 0; p < 3; p++) f[e][p] = vf[64 * (8 * p + db + e)];
#pragma unroll
                for (int o = 0; o < 6; o++)
#pragma unroll
                    for (int e = 0; e < 2; e++)
#pragma unroll
                        for (int qb = 0; qb < NQ; qb++)
                            oacc[db + e][qb] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(f[e][order[o][0]], pf[qb][order[o][1]],
                                                                                       oacc[db + e][qb], 0, 0, 0);
            }
        }
    }
#pragma unroll
    for (int qb = 0; qb < NQ; qb++) l[qb] = sum4(l[qb]);
    if constexpr (kSplit) {  // half 1 leaves its share in its stage, half 0 merges it (as run_item)
        __syncthreads();
        f32x4* pub = reinterpret_cast<f32x4*>(lds + STAGE_BYTES) + (size_t)w4 * (8 * NQ * 64) + lane;
        float* pml = reinterpret_cast<float*>(lds) + (size_t)w4 * (2 * NQ * 64) + lane;  // half 0's stage is free
        if (half == 1) {
#pragma unroll
            for (int qb = 0; qb < NQ; qb++) {
#pragma unroll
                for (int db = 0; db < 8; db++) pub[64 * (8 * qb + db)] = oacc[db][qb];
                pml[64 * (2 * qb)] = m[qb];
                pml[64 * (2 * qb + 1)] = l[qb];
            }
        }
        __syncthreads();
        if (half == 1) return;
#pragma unroll
        for (int qb = 0; qb < NQ; qb++) {
            const float m1 = pml[64 * (2 * qb)], l1 = pml[64 * (2 * qb + 1)], mm = fmaxf(m[qb], m1);
            const float a0 = __builtin_amdgcn_exp2f(m[qb] - mm), a1 = __builtin_amdgcn_exp2f(m1 - mm);
            l[qb] = l[qb] * a0 + l1 * a1;
#pragma unroll
            for (int db = 0; db < 8; db++) oacc[db][qb] = oacc[db][qb] * a0 + pub[64 * (8 * qb + db)] * a1;
        }
    }
#pragma unroll
    for (int qb = 0; qb < NQ; qb++) {
        const int blk = NQ * w4 + qb, kq = blk < 4 ? wt.kq0 : wt.kq1, slot = 16 * (blk & 3) + r16;
        if (slot >= wt.nvalid(kq)) continue;  // padding
        float* dst = kq < wt.nvt ? reinterpret_cast<float*>(a.vattn) + rows.ofs[qb] / 3
                                 : a.tpart + ((size_t)wt.w * a.txt_len + TILE * (kq - wt.nvt) + slot) * DIM;
        const float inv = 1.f / l[qb];
#pragma unroll
        for (int db = 0; db < 8; db++)
            *reinterpret_cast<f32x4*>(dst + h * HEAD_D + 16 * db + 4 * q) = oacc[db][qb] * inv;
    }
}

// One workgroup per (two query tiles of a window, head), 128 queries: four
// waves of 32 (or, for an odd window's last tile, of 16).  64 KiB of LDS and at
// most 256 registers: two workgroups per CU, two waves per SIMD.  Fewer
// queries per wave would read the fragments more often than LDS can deliver
// (32 queries: 85 of 128 bytes per clock at full MFMA rate).
//
// Measured (1080p shifted, 1,304 workgroups of 6-22 units, kernel trace): 323
// us as fp32 MFMAs, 130 here; 360p 49.5 -> 35 us.  With every window cut to two
// units it still takes 56 us: the workgroup's ends (its queries' rows from
// memory, their normalisation and split, the first units' latency, the output
// rows) are over a third of the time, the units between run at about 60 % of the
// MFMA rate.  Neither the softmax's instructions (a quarter fewer: 134 -> 128 us)
// nor HBM (112 MB read, 69 written) sets it.
//
// The window's keys run in 32-key units u, each in two phases in which the
// matrix core and the VALU work side by side:
//   A(u)  MFMA  S(u+1) = K(u+1) Q^T
//         VALU  P(u) = exp2(S(u) - m), its row sums and its split
//   B(u)  MFMA  O^T += V^T(u) P^T(u)
//         VALU  row maxima of S(u+1)
// K and V units reach LDS by DMA into rings of two; unit u's barrier makes
// K(u+1) and V(u) visible and frees the slots of K(u) and V(u-1), which the
// DMA of K(u+2) and V(u+1) refills under both phases.  Past the last unit
// phase A forms scores from whatever its slot holds, which nothing uses.
//   kSplit: eight waves in two halves of four, half 0 taking the window's
//     units [0, n0), half 1 the rest (n0 = ceil(n / 2)), each through its own
//     stage: one workgroup per CU, and a long window takes half as long; at the
//     end half 1 leaves its row maxima, sums and O^T in LDS and half 0 merges
//     them.  For grids of at most one workgroup per CU, where the longest
//     window sets the time.
//
// Lane l = 16 q + r.  Fragments (A or B operand, 16 rows x 32 k): lane holds
// row r, k 8 q .. + 7.
//   S^T block (kb: 16 keys, qb: 16 queries): A = K, B = Q, 4 k32 steps of
//     channels; out: keys 16 kb + 4 q + t of query r in register t.
//   O^T block (db: 16 channels, qb): A = V^T, B = P, one k32 step: keys
//     {4 q + e, 16 + 4 q + e}, e = 0..3, which are exactly the lane's score
//     registers of the unit's two blocks.
template <int NQ, bool kSplit>
__device__ inline void run_item(const SdpaArgs& a, const Item& wt, const QueryRows& rows, float vmax, unsigned char* lds,
                                uint32_t* out_ofs) {
    const int h = wt.h;
    const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63;
    const int half = kSplit ? wave >> 2 : 0, w4 = wave & 3;
    const int r16 = lane & 15, q = lane >> 4;
    const int nu = wt.units();
    const int n0 = kSplit ? (nu + 1) >> 1 : nu;  // iterations: half 0 has n0 units, half 1 nu - n0
    const int ubeg = half ? n0 : 0, uend = half ? nu : n0;

    const uint32_t ldsb = (uint32_t)(uintptr_t)(lptr_t)lds + half * STAGE_BYTES;
    const unsigned char* stage = lds + half * STAGE_BYTES;
    const unsigned char* Kh = reinterpret_cast<const unsigned char*>(a.Kp) + (size_t)h * a.n_tiles * (2 * FU_BYTES);
    const unsigned char* Vh = reinterpret_cast<const unsigned char*>(a.Vp) + (size_t)h * a.n_tiles * (2 * FU_BYTES);
    // 2^-a (K) and -a (V) of each 16-row block; read through the scalar cache
    // (constant address space): a vector load's wait would also wait for the
    // units' DMA
    const cfloat2_t* ke = (const cfloat2_t*)(a.kexp) + (size_t)h * a.n_tiles * 2;
    const cfloat2_t* ve2 = (const cfloat2_t*)(a.vexp) + (size_t)h * a.n_tiles * 2;
    // unit u into a ring slot (0, 1: this half's even and odd units)
    auto fetch_k = [&](int u, int slot) __attribute__((always_inline)) {
        if (u < uend)
            dma_quarter(Kh + (size_t)wt.unit_half(u) * FU_BYTES, 4096u * w4, 16u * lane, ldsb + slot * FU_BYTES);
    };
    auto fetch_v = [&](int u, int slot) __attribute__((always_inline)) {
        if (u < uend)
            dma_quarter(Vh + (size_t)wt.unit_half(u) * FU_BYTES, 4096u * w4, 16u * lane,
                        ldsb + V_RING + slot * FU_BYTES);
    };
    fetch_k(ubeg, 0);
    fetch_k(ubeg + 1, 1);
    fetch_v(ubeg, 0);
    // kept for the end in LDS (as registers they spilled), by the wave that reads it
    if (half == 0)
#pragma unroll
        for (int qb = 0; qb < NQ; qb++) out_ofs[16 * (NQ * w4 + qb) + r16] = rows.ofs[qb];

    f16x8 qh[NQ][4], ql[NQ][4];
    float cq[NQ];
    load_queries(a, wt, rows, w4, lane, qh, ql, cq);

    f32x4 oacc[8][NQ];
    float m_i[NQ], l_i[NQ];
#pragma unroll
    for (int qb = 0; qb < NQ; qb++) {
        m_i[qb] = -INFINITY;
        l_i[qb] = 0.f;
#pragma unroll
        for (int db = 0; db < 8; db++) oacc[db][qb] = (f32x4){0.f, 0.f, 0.f, 0.f};
    }

    f32x4 s[2][2][NQ];  // scores of an even and an odd unit: two 16-key blocks
    f16x8 fr[2][4];     // fragments, read a step ahead of their MFMAs
    const f16x8* frag = reinterpret_cast<const f16x8*>(stage) + lane;
    // step st of the K unit in a slot: its two key blocks, hi and lo
    auto read_k = [&](int slot, int st) __attribute__((always_inline)) {
#pragma unroll
        for (int e = 0; e < 4; e++) fr[st & 1][e] = frag[slot * (FU_BYTES / 16) + 64 * f32_kfrag(e >> 1, st, e & 1)];
    };
    // step j of the V unit in a slot: channel blocks 2 j, 2 j + 1, hi and lo
    auto read_v = [&](int slot, int j) __attribute__((always_inline)) {
#pragma unroll
        for (int e = 0; e < 4; e++)
            fr[j & 1][e] = frag[(V_RING + slot * FU_BYTES) / 16 + 64 * f32_vfrag(0, 2 * j + (e >> 1), e & 1)];
    };
    // the MFMAs of step st of S += K Q^T, the small products first
    auto score_step = [&](f32x4 (&sn)[2][NQ], int st) __attribute__((always_inline)) {
#pragma unroll
        for (int pr = 0; pr < 3; pr++)
#pragma unroll
            for (int e = 0; e < 2; e++)
#pragma unroll
                for (int qb = 0; qb < NQ; qb++)
                    sn[e][qb] = __builtin_amdgcn_mfma_f32_16x16x32_f16(
                        fr[st & 1][2 * e + (pr == 0)], pr == 1 ? ql[qb][st] : qh[qb][st],
                        st == 0 && pr == 0 ? (f32x4){0.f, 0.f, 0.f, 0.f} : sn[e][qb], 0, 0, 0);
    };
    auto mask = [&](f32x4 (&sn)[2][NQ], int u) __attribute__((always_inline)) {
        const int kv = wt.unit_valid(u);
        if (kv < 32) {
#pragma unroll
            for (int kb = 0; kb < 2; kb++)
#pragma unroll
                for (int r = 0; r < 4; r++)
                    if (16 * kb + 4 * q + r >= kv)
#pragma unroll
                        for (int qb = 0; qb < NQ; qb++) sn[kb][qb][r] = -INFINITY;
        }
    };
    // row maximum of query block qb in a unit whose K blocks have factors kc
    auto row_max = [&](const f32x4 (&sn)[2][NQ], int qb, f32x2 kc) __attribute__((always_inline)) {
        float mx = -INFINITY;
#pragma unroll
        for (int kb = 0; kb < 2; kb++)
            mx = fmaxf(mx, cq[qb] * kc[kb] * fmaxf(fmaxf(sn[kb][qb][0], sn[kb][qb][1]), fmaxf(sn[kb][qb][2], sn[kb][qb][3])));
        return max4(mx);
    };
    // the running maximum stays until a unit's exceeds it by M_STALE
    auto raise = [&](const float (&mloc)[NQ]) __attribute__((always_inline)) {
        bool up = false;
#pragma unroll
        for (int qb = 0; qb < NQ; qb++) up |= mloc[qb] > m_i[qb] + M_STALE;
        if (!__any(up)) return;
#pragma unroll
        for (int qb = 0; qb < NQ; qb++) {
            const float m_new = fmaxf(m_i[qb], mloc[qb]);
            const float alpha = __builtin_amdgcn_exp2f(m_i[qb] - m_new);
            l_i[qb] *= alpha;
#pragma unroll
            for (int db = 0; db < 8; db++) oacc[db][qb] *= alpha;
            m_i[qb] = m_new;
        }
    };
    f32x2 kc = {0.f, 0.f};  // K factors of the unit whose scores are pending
    // one unit, its V in slot sl and the next one's K in slot sl ^ 1: scores
    // s[sl] to P and O, the next unit's to s[sl ^ 1]
    auto unit = [&](int u, int sl) __attribute__((always_inline)) {
        f32x4 (&sc)[2][NQ] = s[sl];
        f32x4 (&sn)[2][NQ] = s[sl ^ 1];
        const int un = min(u + 1, uend - 1);  // past the end: any unit's factors
        const f32x2 kcn = ke[wt.unit_half(un)];
        // P leaves as exp2(s - m + vs): vs puts the block's V scale (of a block
        // of zeros any) and P_SHIFT into the exponent, vi takes them back out of
        // the row sum
        f32x2 vs = ve2[wt.unit_half(u)], vi;
#pragma unroll
        for (int kb = 0; kb < 2; kb++) {
            vs[kb] = scalar(fmaxf(vs[kb] - vmax, (float)-SPREAD_ROWS) + P_SHIFT);
            vi[kb] = scalar(__builtin_amdgcn_exp2f(-vs[kb]));  // exact: whole exponents
        }
        uint32_t hi[NQ][4], lo[NQ][4];
        // ---- phase A
        read_k(sl ^ 1, 0);
#pragma unroll
        for (int st = 0; st < 4; st++) {
            if (st < 3) read_k(sl ^ 1, st + 1);
            else read_v(sl, 0);
            __builtin_amdgcn_sched_barrier(0);
            score_step(sn, st);
            // NQ of the unit's 2 NQ (query block, key block) pairs per two steps
            if (NQ == 2 || (st & 1)) {
                const int qb = NQ == 2 ? st >> 1 : 0, kb = NQ == 2 ? st & 1 : st >> 1;
                const float c = cq[qb] * kc[kb], b = vs[kb] - m_i[qb];
                float p[4];
#pragma unroll
                for (int r = 0; r < 4; r++) p[r] = __builtin_amdgcn_exp2f(__builtin_fmaf(sc[kb][qb][r], c, b));
                // this lane's keys; summed over the row at the end
                l_i[qb] = __builtin_fmaf((p[0] + p[1]) + (p[2] + p[3]), vi[kb], l_i[qb]);
                split2(p[0], p[1], hi[qb][2 * kb], lo[qb][2 * kb]);
                split2(p[2], p[3], hi[qb][2 * kb + 1], lo[qb][2 * kb + 1]);
            }
#pragma unroll
            for (int g = 0; g < 6 * NQ; g++) {
                __builtin_amdgcn_sched_group_barrier(0x8, 1, 0);  // one MFMA
                __builtin_amdgcn_sched_group_barrier(0x2, 3, 0);  // and some of the VALU work
            }
            __builtin_amdgcn_sched_barrier(0);
        }
        mask(sn, un);
        f16x8 ph[NQ], pl[NQ];
#pragma unroll
        for (int qb = 0; qb < NQ; qb++) {
            ph[qb] = __builtin_bit_cast(f16x8, hi[qb]);
            pl[qb] = __builtin_bit_cast(f16x8, lo[qb]);
        }
        // ---- phase B
        float mloc[NQ];
#pragma unroll
        for (int j = 0; j < 4; j++) {
            if (j < 3) read_v(sl, j + 1);
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int pr = 0; pr < 3; pr++)
#pragma unroll
                for (int e = 0; e < 2; e++)
#pragma unroll
                    for (int qb = 0; qb < NQ; qb++)
                        oacc[2 * j + e][qb] = __builtin_amdgcn_mfma_f32_16x16x32_f16(
                            fr[j & 1][2 * e + (pr == 0)], pr == 1 ? pl[qb] : ph[qb], oacc[2 * j + e][qb], 0, 0, 0);
            if (j >= 1 && j <= NQ) mloc[j - 1] = row_max(sn, j - 1, kcn);
#pragma unroll
            for (int g = 0; g < 6 * NQ; g++) {
                __builtin_amdgcn_sched_group_barrier(0x8, 1, 0);
                __builtin_amdgcn_sched_group_barrier(0x2, 2, 0);
            }
            __builtin_amdgcn_sched_barrier(0);
        }
        kc = kcn;
        if (u + 1 < uend) raise(mloc);
    };

    unit_barrier();
    if (ubeg < uend) {  // the first unit's scores
        kc = ke[wt.unit_half(ubeg)];
        read_k(0, 0);
#pragma unroll
        for (int st = 0; st < 4; st++) {
            if (st < 3) read_k(0, st + 1);
            score_step(s[0], st);
        }
        mask(s[0], ubeg);
        float mloc[NQ];
#pragma unroll
        for (int qb = 0; qb < NQ; qb++) mloc[qb] = row_max(s[0], qb, kc);
        raise(mloc);
    }
    for (int i = 0; i < n0; i += 2)  // the same iteration count in both halves
#pragma unroll
        for (int e = 0; e < 2; e++) {
            const int u = ubeg + i + e;
            unit_barrier();
            fetch_k(u + 2, e);
            fetch_v(u + 1, e ^ 1);
            if (u < uend) unit(u, e);  // uniform per half
        }
    // the lane through an opaque copy: the addresses below are formed here and
    // not held in registers across the loop
    int ln = lane;
    asm volatile("" : "+v"(ln));
    float l[NQ];
#pragma unroll
    for (int qb = 0; qb < NQ; qb++) l[qb] = sum4(l_i[qb]);
    if constexpr (kSplit) {
        // merge: half 1 leaves its running maximum (-inf when it had no
        // tile), sum and O^T in its stage, half 0 rescales both to the common
        // maximum.  Rows of 16 NQ registers side by side per lane: 16-byte
        // pieces of consecutive lanes.
        __syncthreads();
        f32x4* pub = reinterpret_cast<f32x4*>(lds + STAGE_BYTES) + (size_t)w4 * (8 * NQ * 64) + ln;
        float* pml = reinterpret_cast<float*>(lds) + (size_t)w4 * (2 * NQ * 64) + ln;  // half 0's stage is free
        if (half == 1) {
#pragma unroll
            for (int qb = 0; qb < NQ; qb++) {
#pragma unroll
                for (int db = 0; db < 8; db++) pub[64 * (8 * qb + db)] = oacc[db][qb];
                pml[64 * (2 * qb)] = m_i[qb];
                pml[64 * (2 * qb + 1)] = l[qb];
            }
        }
        __syncthreads();
        if (half == 1) return;
#pragma unroll
        for (int qb = 0; qb < NQ; qb++) {
            const float m1 = pml[64 * (2 * qb)], l1 = pml[64 * (2 * qb + 1)];
            const float m = fmaxf(m_i[qb], m1);
            const float a0 = __builtin_amdgcn_exp2f(m_i[qb] - m), a1 = __builtin_amdgcn_exp2f(m1 - m);
            l[qb] = l[qb] * a0 + l1 * a1;
#pragma unroll
            for (int db = 0; db < 8; db++) oacc[db][qb] = oacc[db][qb] * a0 + pub[64 * (8 * qb + db)] * a1;
        }
    }
    // ---- O / l through LDS (each wave its own 16 rows of 512 bytes, 16-byte
    // chunk c of row r at c ^ r), so that whole rows are stored (from the
    // accumulator layout a store writes 64 bytes of 16 rows)
    if constexpr (!kSplit) __syncthreads();  // every wave is done with the K and V units
    f32x4* stg = reinterpret_cast<f32x4*>(lds + (kSplit ? 16384 : 0)) + w4 * (16 * 32);
    const float c = __builtin_amdgcn_exp2f(vmax - P_SHIFT);
#pragma unroll
    for (int qb = 0; qb < NQ; qb++) {
        const int blk = NQ * w4 + qb, kq = blk < 4 ? wt.kq0 : wt.kq1;
        // 1 / l and the V scale; the factors separately, so that neither overflows
        const float inv = 1.f / l[qb];
#pragma unroll
        for (int db = 0; db < 8; db++) stg[(ln & 15) * 32 + ((4 * db + (ln >> 4)) ^ (ln & 15))] = oacc[db][qb] * inv * c;
#pragma unroll
        for (int i = 0; i < 8; i++) {
            const int row = 2 * i + (ln >> 5), ch = ln & 31, slot = 16 * (blk & 3) + row;
            const f32x4 v = stg[row * 32 + (ch ^ row)];
            const uint32_t ofs = out_ofs[16 * blk + row];
            if (slot >= wt.nvalid(kq)) continue;  // padding
            // video: the token's row of vattn (a row is a third of its qkv row)
            float* dst = kq < wt.nvt ? reinterpret_cast<float*>(a.vattn) + ofs / 3
                                     : a.tpart + ((size_t)wt.w * a.txt_len + TILE * (kq - wt.nvt) + slot) * DIM;
            *reinterpret_cast<f32x4*>(dst + h * HEAD_D + 4 * ch) = v;
        }
    }
}

// Workgroup b: entry b of GeomPlan::f32_work.
template <bool kSplit>
__global__ __launch_bounds__(kSplit ? 512 : 256, 2) void sdpa_f32_kernel(SdpaArgs a) {
    __shared__ __align__(16) unsigned char lds[(kSplit ? 2 : 1) * STAGE_BYTES];
    __shared__ uint32_t out_ofs[2 * TILE];
    const int e = a.f32_work[blockIdx.x];
    if (e < 0) return;  // an idle entry
    const int4 d0 = reinterpret_cast<const int4*>(a.sched_desc)[2 * (e >> 2)];
    const int4 d1 = reinterpret_cast<const int4*>(a.sched_desc)[2 * (e >> 2) + 1];
    const int part = e & 3;  // 0: the item's one or two query tiles, 1, 2: one of its two
    Item it;
    it.h = d0.x & 255; it.w = d0.x >> 8; it.kq0 = part == 2 ? d0.z : d0.y; it.kq1 = part ? -1 : d0.z;
    it.vbase = d1.x; it.nvt = d1.y; it.tbase = d1.z; it.f = d1.w;
    it.ntt = a.ntt; it.txt = a.txt_len;
    const int nq = it.kq1 >= 0 ? 2 : 1;
    const QueryRows rows =
        query_rows(a, it, nq, __builtin_amdgcn_readfirstlane(threadIdx.x >> 6) & 3, threadIdx.x & 15);
    const float vmax = window_vmax(a, it, threadIdx.x & 63);
    const int mode = __builtin_amdgcn_readfirstlane(vmax == VEXP_FULL ? 2 : vmax == VEXP_WIDE);  // a scalar branch
    if (mode == 0) {
        if (nq == 2) run_item<2, kSplit>(a, it, rows, vmax, lds, out_ofs);
        else run_item<1, kSplit>(a, it, rows, vmax, lds, out_ofs);
    } else if (mode == 1) {
        if (nq == 2) wide_item<2, kSplit>(a, it, rows, lds);
        else wide_item<1, kSplit>(a, it, rows, lds);
    } else {
        for (int t = 0; t < nq; t++) full_queries<kSplit>(a, it, reinterpret_cast<float*>(lds), t);
    }
}

}  // namespace

hipError_t launch_sdpa_f32(const SdpaArgs& a, hipStream_t s) {
    if (a.n_f32_work == 0) return hipSuccess;
    // n_slots: two per CU (the persistent bf16 schedule's slot count)
    if (a.n_f32_work <= a.n_slots / 2)
        hipLaunchKernelGGL(sdpa_f32_kernel<true>, dim3(a.n_f32_work), dim3(512), 0, s, a);
    else
        hipLaunchKernelGGL(sdpa_f32_kernel<false>, dim3(a.n_f32_work), dim3(256), 0, s, a);
    return hipGetLastError();
}

}  // namespace awa
