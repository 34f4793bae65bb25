// dit_capi.cpp — C ABI of the DiT block: one layer of DitVk::forward_latent
// (dit_vk.cpp:517-632) as norm -> GEMM -> AWA -> GEMM -> norm -> GEMM -> GEMM
// on the caller's stream.
#include <algorithm>
#include <cmath>
#include <cstring>

#include "dit_internal.hpp"

using namespace awa;

namespace {

#define HIPCK(ctx, expr)                                                                     \
    do {                                                                                     \
        hipError_t e_ = (expr);                                                              \
        if (e_ != hipSuccess) {                                                              \
            set_err(ctx, "%s failed: %s (%s:%d)", #expr, hipGetErrorString(e_), __FILE__,    \
                    __LINE__);                                                               \
            return AWA_EHIP;                                                                 \
        }                                                                                    \
    } while (0)

size_t align256(size_t x) { return (x + 255) & ~(size_t)255; }

bool branch_ok(const dit_branch* b) {
    return b && b->qkv_w && b->out_w && b->out_b && b->mlp_w && b->mlp_out_w && b->nq && b->nk &&
           b->attn_shift && b->attn_scale && b->attn_gate && b->mlp_shift && b->mlp_scale && b->mlp_gate;
}

GemmProblem problem(const uint16_t* A, int lda, const uint16_t* W, int ldw, int M, int N, int K,
                    void* C, int ldc) {
    GemmProblem p{};
    p.A = A; p.lda = lda; p.W = W; p.ldw = ldw; p.M = M; p.N = N; p.K = K; p.C = C; p.ldc = ldc;
    p.split = M;
    return p;
}

constexpr int VID_OUT = 64;  // output channels 16 x 2 x 2

}  // namespace

struct dit_io {
    int device = 0;
    uint16_t* vid_in_w = nullptr;   // [2560][EMBED_K] in fragment order
    const float* vid_in_b = nullptr;
    const uint16_t* txt_in_w = nullptr;
    const float* txt_in_b = nullptr;
    const float* out_norm_w = nullptr;
    const float* out_ada_shift = nullptr;
    const float* out_ada_scale = nullptr;
    uint16_t* vid_out_w = nullptr;  // [64][2560] in fragment order
    float* vid_out_b = nullptr;     // [64]
};

extern "C" {

int dit_io_create(awa_ctx* ctx, const dit_io_weights* w, dit_io** out, awa_stream_t stream) {
    if (!ctx || !w || !out || !w->vid_in_w || !w->vid_in_b || !w->txt_in_w || !w->txt_in_b ||
        !w->out_norm_w || !w->out_ada_shift || !w->out_ada_scale || !w->vid_out_w || !w->vid_out_b) {
        set_err(ctx, "dit_io_create: null argument");
        return AWA_EARG;
    }
    *out = nullptr;
    DeviceGuard dg(ctx->device);
    hipStream_t s = reinterpret_cast<hipStream_t>(stream);
    dit_io* io = new dit_io();
    io->device = ctx->device;
    io->vid_in_b = w->vid_in_b; io->txt_in_w = w->txt_in_w; io->txt_in_b = w->txt_in_b;
    io->out_norm_w = w->out_norm_w; io->out_ada_shift = w->out_ada_shift; io->out_ada_scale = w->out_ada_scale;
    hipError_t e = hipMalloc(reinterpret_cast<void**>(&io->vid_in_w), (size_t)DIM * EMBED_K * 2);
    if (e == hipSuccess) e = hipMalloc(reinterpret_cast<void**>(&io->vid_out_w), (size_t)VID_OUT * DIM * 2);
    if (e == hipSuccess) e = hipMalloc(reinterpret_cast<void**>(&io->vid_out_b), VID_OUT * 4);
    if (e == hipSuccess) e = launch_end_weights(w->vid_in_w, io->vid_in_w, w->vid_out_w, io->vid_out_w, s);
    if (e == hipSuccess) e = hipMemcpyAsync(io->vid_out_b, w->vid_out_b, VID_OUT * 4, hipMemcpyDeviceToDevice, s);
    if (e != hipSuccess) {
        set_err(ctx, "dit_io_create: %s", hipGetErrorString(e));
        dit_io_destroy(ctx, io);
        return AWA_EHIP;
    }
    *out = io;
    return AWA_OK;
}

void dit_io_destroy(awa_ctx* ctx, dit_io* io) {
    if (!io) return;
    DeviceGuard dg(ctx ? ctx->device : io->device);
    if (io->vid_in_w) (void)hipFree(io->vid_in_w);
    if (io->vid_out_w) (void)hipFree(io->vid_out_w);
    if (io->vid_out_b) (void)hipFree(io->vid_out_b);
    delete io;
}

namespace {
// workspace bytes of each entry point (the offsets below follow the same layouts)
// embed: the text's partial products, or a long text in bf16, then copies of inputs
// that d_x lies over
size_t embed_part_bytes(int TXT) {
    return align256(TXT <= EMBED_TXT_MAX ? (size_t)EMBED_TXT_SPLIT * TXT * DIM * 4 : (size_t)TXT * 5120 * 2);
}
size_t grid_bytes(int Lv) { return (size_t)Lv * 4 * 33 * 4; }
size_t txt_bytes(int TXT) { return (size_t)TXT * 5120 * 4; }
size_t embed_ws_bytes(int Lv, int TXT) {
    return embed_part_bytes(TXT) + align256(grid_bytes(Lv)) + align256(txt_bytes(TXT));
}
// final: the output, if it lies over x or the embedding
size_t final_ws_bytes(int Lv) { return (size_t)Lv * VID_OUT * 4; }
size_t layer_ws_bytes(int M, int mlp) {
    return align256(12 * DIM * 4) + align256((size_t)M * DIM * 2) + align256((size_t)M * QKV * 2) +
           align256((size_t)M * DIM * 2) + align256((size_t)M * mlp * 2);
}
}  // namespace

int dit_reserve(awa_ctx* ctx, const awa_geom* g, int mlp) {
    if (!ctx || !g || mlp <= 0 || mlp % 128 != 0 || mlp > DIT_MLP_MAX) {
        set_err(ctx, "dit_reserve: bad argument (mlp=%d must be a positive multiple of 128, at most %d)", mlp,
                DIT_MLP_MAX);
        return AWA_EARG;
    }
    const int Lv = g->plan.Lv, TXT = g->plan.txt_len;
    DeviceGuard dg(ctx->device);
    HIPCK(ctx, ensure_buffer(&ctx->ws, &ctx->ws_bytes,
                             std::max(layer_ws_bytes(Lv + TXT, mlp), std::max(embed_ws_bytes(Lv, TXT), final_ws_bytes(Lv)))));
    return awa_reserve(ctx, g, AWA_BF16);
}

int dit_embed(awa_ctx* ctx, const dit_io* io, const float* d_grid, int T, int H, int W, const float* d_txt,
              int TXT, float* d_x, awa_stream_t stream) {
    if (!ctx || !io || !d_grid || !d_txt || !d_x || T < 1 || H < 2 || W < 2 || H % 2 || W % 2 || TXT < 1) {
        set_err(ctx, "dit_embed: bad argument (T=%d H=%d W=%d TXT=%d; H and W even)", T, H, W, TXT);
        return AWA_EARG;
    }
    DeviceGuard dg(ctx->device);
    hipStream_t s = reinterpret_cast<hipStream_t>(stream);
    EmbedArgs a{};
    a.grid = d_grid; a.H = H; a.W2 = W / 2;
    a.Lv = T * (H / 2) * (W / 2); a.TXT = TXT;
    a.vid_w = io->vid_in_w; a.vid_b = io->vid_in_b;
    a.txt = d_txt; a.txt_w = io->txt_in_w; a.txt_b = io->txt_in_b;
    a.x = d_x;
    HIPCK(ctx, ensure_buffer(&ctx->ws, &ctx->ws_bytes, embed_ws_bytes(a.Lv, TXT)));
    a.part = static_cast<float*>(ctx->ws);
    // workgroups write x while others still read the inputs: those under x are
    // copied first
    char* copy = static_cast<char*>(ctx->ws) + embed_part_bytes(TXT);
    const size_t x_bytes = (size_t)(a.Lv + TXT) * DIM * 4;
    if (overlaps(d_x, x_bytes, d_grid, grid_bytes(a.Lv))) {
        HIPCK(ctx, hipMemcpyAsync(copy, d_grid, grid_bytes(a.Lv), hipMemcpyDeviceToDevice, s));
        a.grid = reinterpret_cast<const float*>(copy);
        copy += align256(grid_bytes(a.Lv));
    }
    if (overlaps(d_x, x_bytes, d_txt, txt_bytes(TXT))) {
        HIPCK(ctx, hipMemcpyAsync(copy, d_txt, txt_bytes(TXT), hipMemcpyDeviceToDevice, s));
        a.txt = reinterpret_cast<const float*>(copy);
    }
    if (TXT <= EMBED_TXT_MAX) {
        HIPCK(ctx, launch_embed(a, s));
        return AWA_OK;
    }
    // a long text: x = A W^T + b by the residual epilogue on zeroed rows, gate 1
    uint16_t* txt16 = static_cast<uint16_t*>(ctx->ws);
    float* x_txt = d_x + (size_t)a.Lv * DIM;
    HIPCK(ctx, launch_cast_f32_bf16(a.txt, txt16, (int64_t)TXT * 5120, s));
    a.TXT = 0;
    HIPCK(ctx, launch_embed(a, s));
    HIPCK(ctx, launch_zero(x_txt, (size_t)TXT * DIM * 4, s));
    GemmBatch b{};
    b.nprob = 1;
    b.p[0] = problem(txt16, 5120, io->txt_in_w, 5120, TXT, DIM, 5120, x_txt, DIM);
    b.p[0].bias = io->txt_in_b;
    HIPCK(ctx, launch_gemm(EPI_RESID, b, s));
    return AWA_OK;
}

int dit_final(awa_ctx* ctx, const dit_io* io, const float* d_emb, const float* d_x, int T, int H, int W,
              float eps, float* d_out, awa_stream_t stream) {
    if (!ctx || !io || !d_emb || !d_x || !d_out || T < 1 || H < 2 || W < 2 || H % 2 || W % 2 || !(eps > 0.f)) {
        set_err(ctx, "dit_final: bad argument (T=%d H=%d W=%d; H and W even, eps > 0)", T, H, W);
        return AWA_EARG;
    }
    DeviceGuard dg(ctx->device);
    hipStream_t s = reinterpret_cast<hipStream_t>(stream);
    FinalArgs a{};
    a.x = d_x; a.emb = d_emb;
    a.norm_w = io->out_norm_w; a.ada_scale = io->out_ada_scale; a.ada_shift = io->out_ada_shift;
    a.W = io->vid_out_w; a.bias = io->vid_out_b;
    a.rows = T * (H / 2) * (W / 2); a.H = H; a.W2 = W / 2;
    a.eps = eps;
    a.out = d_out;
    // workgroups write out while others still read x and the embedding: over
    // those the output goes through the workspace
    const size_t out_bytes = final_ws_bytes(a.rows);
    const bool in_place = overlaps(d_out, out_bytes, d_x, (size_t)a.rows * DIM * 4) ||
                          overlaps(d_out, out_bytes, d_emb, (size_t)DIT_EMB * 4);
    if (in_place) {
        HIPCK(ctx, ensure_buffer(&ctx->ws, &ctx->ws_bytes, out_bytes));
        a.out = static_cast<float*>(ctx->ws);
    }
    HIPCK(ctx, launch_final(a, s));
    if (in_place) HIPCK(ctx, hipMemcpyAsync(d_out, a.out, out_bytes, hipMemcpyDeviceToDevice, s));
    return AWA_OK;
}

int dit_pack_mlp_weights(awa_ctx* ctx, const uint16_t* d_w_in, const uint16_t* d_w_gate, int mlp,
                         uint16_t* d_w_cat, awa_stream_t stream) {
    if (!ctx || !d_w_in || !d_w_gate || !d_w_cat || mlp <= 0 || mlp % 128 != 0 || mlp > DIT_MLP_MAX) {
        set_err(ctx, "dit_pack_mlp_weights: bad argument (mlp=%d must be a positive multiple of 128, at most %d)",
                mlp, DIT_MLP_MAX);
        return AWA_EARG;
    }
    DeviceGuard dg(ctx->device);
    HIPCK(ctx, launch_pack_mlp(d_w_in, d_w_gate, mlp, d_w_cat, reinterpret_cast<hipStream_t>(stream)));
    return AWA_OK;
}

int dit_time_embedding(awa_ctx* ctx, float t, const float* d_w_in, const float* d_b_in,
                       const float* d_w_hid, const float* d_b_hid, const float* d_w_out,
                       const float* d_b_out, float* d_emb, awa_stream_t stream) {
    if (!ctx || !d_w_in || !d_b_in || !d_w_hid || !d_b_hid || !d_w_out || !d_b_out || !d_emb) {
        set_err(ctx, "dit_time_embedding: null argument");
        return AWA_EARG;
    }
    DeviceGuard dg(ctx->device);
    hipStream_t s = reinterpret_cast<hipStream_t>(stream);
    if (!ctx->small) HIPCK(ctx, hipMalloc(reinterpret_cast<void**>(&ctx->small), 8192 * sizeof(float)));
    const float* w[3] = {d_w_in, d_w_hid, d_w_out};
    const float* b[3] = {d_b_in, d_b_hid, d_b_out};
    HIPCK(ctx, launch_time_mlp(t, w, b, ctx->small, ctx->small + DIM, d_emb, s));
    return AWA_OK;
}

int dit_gemm_bf16(awa_ctx* ctx, const uint16_t* d_A, const uint16_t* d_W, uint16_t* d_C, int M, int N,
                  int K, awa_stream_t stream) {
    if (!ctx || !d_A || !d_W || !d_C || M < 1 || N < 256 || N % 256 || N > DIT_GEMM_NK_MAX || K < 64 || K % 64 ||
        K > DIT_GEMM_NK_MAX) {
        set_err(ctx, "dit_gemm_bf16: bad argument M=%d N=%d K=%d (N %% 256 == 0, K %% 64 == 0, N, K <= %d)", M, N, K,
                DIT_GEMM_NK_MAX);
        return AWA_EARG;
    }
    DeviceGuard dg(ctx->device);
    GemmBatch b{};
    b.nprob = 1;
    b.p[0] = problem(d_A, K, d_W, K, M, N, K, d_C, N);
    HIPCK(ctx, launch_gemm(EPI_STORE, b, reinterpret_cast<hipStream_t>(stream)));
    return AWA_OK;
}

int dit_layer_forward(awa_ctx* ctx, const awa_geom* g, const dit_branch* vb, const dit_branch* tb,
                      const float* d_emb, int mlp, int txt_vid_only, float eps, float* d_x, int Lv,
                      int TXT, awa_stream_t stream) {
    if (!ctx || !g || !d_emb || !d_x || !branch_ok(vb) || !branch_ok(tb)) {
        set_err(ctx, "dit_layer_forward: null argument or incomplete branch");
        return AWA_EARG;
    }
    if (Lv != g->plan.Lv || TXT != g->plan.txt_len) {
        set_err(ctx, "dit_layer_forward: Lv=%d TXT=%d do not match the geometry (Lv=%d TXT=%d)", Lv,
                TXT, g->plan.Lv, g->plan.txt_len);
        return AWA_EARG;
    }
    if (mlp <= 0 || mlp % 128 != 0 || mlp > DIT_MLP_MAX || !(eps > 0.f)) {
        set_err(ctx, "dit_layer_forward: mlp=%d must be a positive multiple of 128 (at most %d), eps > 0", mlp,
                DIT_MLP_MAX);
        return AWA_EARG;
    }
    DeviceGuard dg(ctx->device);
    hipStream_t s = reinterpret_cast<hipStream_t>(stream);
    const bool dual = vb != tb;
    const int M = Lv + TXT;
    const int Mm = txt_vid_only ? Lv : M;  // rows that run the MLP

    // workspace: ada [12][2560] f32 | h [M][2560] | qkv [M][7680] | attn [M][2560] | u [M][mlp]
    const size_t o_h = align256(12 * DIM * 4);
    const size_t o_qkv = o_h + align256((size_t)M * DIM * 2);
    const size_t o_att = o_qkv + align256((size_t)M * QKV * 2);
    const size_t o_u = o_att + align256((size_t)M * DIM * 2);
    HIPCK(ctx, ensure_buffer(&ctx->ws, &ctx->ws_bytes, layer_ws_bytes(M, mlp)));
    char* ws = static_cast<char*>(ctx->ws);
    float* ada = reinterpret_cast<float*>(ws);
    uint16_t* h = reinterpret_cast<uint16_t*>(ws + o_h);
    uint16_t* qkv = reinterpret_cast<uint16_t*>(ws + o_qkv);
    uint16_t* att = reinterpret_cast<uint16_t*>(ws + o_att);
    uint16_t* u = reinterpret_cast<uint16_t*>(ws + o_u);
    auto V = [&](int f, int k) { return ada + (size_t)(f * 6 + k) * DIM; };  // a_sc a_sh a_g m_sc m_sh m_g
    auto mark = [&]() { return event_mark(ctx, ctx->dit_ev_used, s); };

    HIPCK(ctx, mark());
    AdaArgs aa{};
    aa.emb = d_emb;
    aa.out = ada;
    const dit_branch* br[2] = {vb, tb};
    for (int f = 0; f < 2; f++) {
        aa.vec[f][0] = br[f]->attn_scale; aa.vec[f][1] = br[f]->attn_shift; aa.vec[f][2] = br[f]->attn_gate;
        aa.vec[f][3] = br[f]->mlp_scale;  aa.vec[f][4] = br[f]->mlp_shift;  aa.vec[f][5] = br[f]->mlp_gate;
    }
    HIPCK(ctx, launch_ada(aa, s));
    // attention norm + ada (dit_vk.cpp:530-545); last layer: text rows unmodulated
    NormArgs na{};
    na.x = d_x; na.h = h; na.M = M; na.split = Lv; na.eps = eps;
    na.scale0 = V(0, 0); na.shift0 = V(0, 1);
    na.scale1 = txt_vid_only ? nullptr : V(1, 0);
    na.shift1 = txt_vid_only ? nullptr : V(1, 1);
    HIPCK(ctx, launch_norm_ada(na, s));
    HIPCK(ctx, mark());

    // qkv projections (dit_vk.cpp:321-322), no bias
    GemmBatch b{};
    if (!dual) {
        b.nprob = 1;
        b.p[0] = problem(h, DIM, vb->qkv_w, DIM, M, QKV, DIM, qkv, QKV);
    } else {
        b.nprob = 2;
        b.p[0] = problem(h, DIM, vb->qkv_w, DIM, Lv, QKV, DIM, qkv, QKV);
        b.p[1] = problem(h + (size_t)Lv * DIM, DIM, tb->qkv_w, DIM, TXT, QKV, DIM, qkv + (size_t)Lv * QKV, QKV);
    }
    HIPCK(ctx, launch_gemm(EPI_STORE, b, s));
    HIPCK(ctx, mark());

    // the AWA op, bf16 boundary (awa_layer.cpp:338-451)
    int rc = forward_impl(ctx, g, AWA_BF16, qkv, qkv + (size_t)Lv * QKV, vb->nq, vb->nk, tb->nq, tb->nk, eps,
                          att, att + (size_t)Lv * DIM, s);
    if (rc != AWA_OK) return rc;
    HIPCK(ctx, mark());

    // out projection + bias, attention gate, residual (dit_vk.cpp:461-462, 558-575)
    b = GemmBatch{};
    if (!dual) {
        b.nprob = 1;
        b.p[0] = problem(att, DIM, vb->out_w, DIM, M, DIM, DIM, d_x, DIM);
        b.p[0].bias = vb->out_b;
        b.p[0].gate0 = V(0, 2);
        b.p[0].gate1 = txt_vid_only ? nullptr : V(1, 2);
        b.p[0].split = Lv;
    } else {
        b.nprob = 2;
        b.p[0] = problem(att, DIM, vb->out_w, DIM, Lv, DIM, DIM, d_x, DIM);
        b.p[0].bias = vb->out_b;
        b.p[0].gate0 = V(0, 2);
        b.p[1] = problem(att + (size_t)Lv * DIM, DIM, tb->out_w, DIM, TXT, DIM, DIM, d_x + (size_t)Lv * DIM, DIM);
        b.p[1].bias = tb->out_b;
        b.p[1].gate0 = txt_vid_only ? nullptr : V(1, 2);
    }
    HIPCK(ctx, launch_gemm(EPI_RESID, b, s));
    HIPCK(ctx, mark());

    // MLP norm + ada (dit_vk.cpp:577-597); last layer: text rows skip the MLP
    na = NormArgs{};
    na.x = d_x; na.h = h; na.M = Mm; na.split = Lv; na.eps = eps;
    na.scale0 = V(0, 3); na.shift0 = V(0, 4);
    na.scale1 = V(1, 3); na.shift1 = V(1, 4);
    HIPCK(ctx, launch_norm_ada(na, s));
    HIPCK(ctx, mark());

    // SwiGLU (dit_vk.cpp:465-472): u = silu(h Wg^T) * (h Win^T), then out, gate, residual
    b = GemmBatch{};
    if (!dual || txt_vid_only) {
        b.nprob = 1;
        b.p[0] = problem(h, DIM, vb->mlp_w, DIM, dual ? Lv : Mm, 2 * mlp, DIM, u, mlp);
    } else {
        b.nprob = 2;
        b.p[0] = problem(h, DIM, vb->mlp_w, DIM, Lv, 2 * mlp, DIM, u, mlp);
        b.p[1] = problem(h + (size_t)Lv * DIM, DIM, tb->mlp_w, DIM, TXT, 2 * mlp, DIM, u + (size_t)Lv * mlp, mlp);
    }
    HIPCK(ctx, launch_gemm(EPI_SWIGLU, b, s));
    b = GemmBatch{};
    if (!dual || txt_vid_only) {
        b.nprob = 1;
        b.p[0] = problem(u, mlp, vb->mlp_out_w, mlp, dual ? Lv : Mm, DIM, mlp, d_x, DIM);
        b.p[0].gate0 = V(0, 5);
        b.p[0].gate1 = V(1, 5);
        b.p[0].split = Lv;
    } else {
        b.nprob = 2;
        b.p[0] = problem(u, mlp, vb->mlp_out_w, mlp, Lv, DIM, mlp, d_x, DIM);
        b.p[0].gate0 = V(0, 5);
        b.p[1] = problem(u + (size_t)Lv * mlp, mlp, tb->mlp_out_w, mlp, TXT, DIM, mlp, d_x + (size_t)Lv * DIM, DIM);
        b.p[1].gate0 = V(1, 5);
    }
    HIPCK(ctx, launch_gemm(EPI_RESID, b, s));
    HIPCK(ctx, mark());
    return AWA_OK;
}

int dit_forward_grid(awa_ctx* ctx, const dit_io* io, const dit_time_weights* tw, const dit_branch* const* vb,
                     const dit_branch* const* tb, int n_layers, const awa_geom* g_even, const awa_geom* g_odd,
                     int mlp, int last_txt_vid_only, float eps, float t, const float* d_grid, int T, int H,
                     int W, const float* d_txt, int TXT, float* d_x, float* d_out, awa_stream_t stream) {
    if (!ctx || !io || !tw || !vb || !tb || n_layers < 0 || !g_even || (n_layers > 1 && !g_odd)) {
        set_err(ctx, "dit_forward_grid: null argument or n_layers=%d < 0", n_layers);
        return AWA_EARG;
    }
    if (H % 2 || W % 2 || H < 2 || W < 2 || T < 1) {
        set_err(ctx, "dit_forward_grid: T=%d H=%d W=%d (H and W even)", T, H, W);
        return AWA_EARG;
    }
    const int Lv = T * (H / 2) * (W / 2);
    for (const awa_geom* g : {g_even, g_odd}) {
        if (g && (g->plan.Lv != Lv || g->plan.txt_len != TXT)) {
            set_err(ctx, "dit_forward_grid: geometry (Lv=%d TXT=%d) does not match the grid (Lv=%d TXT=%d)",
                    g->plan.Lv, g->plan.txt_len, Lv, TXT);
            return AWA_EARG;
        }
    }
    {
        DeviceGuard dg(ctx->device);
        if (!ctx->emb) HIPCK(ctx, hipMalloc(reinterpret_cast<void**>(&ctx->emb), DIT_EMB * sizeof(float)));
    }
    int rc = dit_embed(ctx, io, d_grid, T, H, W, d_txt, TXT, d_x, stream);
    if (rc == AWA_OK)
        rc = dit_time_embedding(ctx, t, tw->w_in, tw->b_in, tw->w_hid, tw->b_hid, tw->w_out, tw->b_out, ctx->emb,
                                stream);
    for (int i = 0; i < n_layers && rc == AWA_OK; i++)
        rc = dit_layer_forward(ctx, (i % 2 == 0) ? g_even : g_odd, vb[i], tb[i], ctx->emb, mlp,
                               (i == n_layers - 1) ? last_txt_vid_only : 0, eps, d_x, Lv, TXT, stream);
    if (rc == AWA_OK) rc = dit_final(ctx, io, ctx->emb, d_x, T, H, W, eps, d_out, stream);
    return rc;
}

int dit_timing_read(awa_ctx* ctx, double* ms_gemm, double* ms_awa, double* ms_eltwise, int* layers) {
    if (!ctx) return AWA_EARG;
    DeviceGuard dg(ctx->device);
    // per layer: e0 norm e1 qkv e2 awa e3 out e4 norm e5 mlp e6
    double gemm = 0, awa_ms = 0, elt = 0;
    const size_t n = ctx->dit_ev_used.size() / 7;
    int rc = AWA_OK;
    for (size_t i = 0; i < n && rc == AWA_OK; i++) {
        hipEvent_t* e = &ctx->dit_ev_used[7 * i];
        float d[6] = {0, 0, 0, 0, 0, 0};
        hipError_t r = hipEventSynchronize(e[6]);
        for (int k = 0; k < 6 && r == hipSuccess; k++) r = hipEventElapsedTime(&d[k], e[k], e[k + 1]);
        if (r != hipSuccess) {
            set_err(ctx, "dit_timing_read: %s", hipGetErrorString(r));
            rc = AWA_EHIP;
        }
        elt += d[0] + d[4];
        gemm += d[1] + d[3] + d[5];
        awa_ms += d[2];
    }
    ctx->ev_free.insert(ctx->ev_free.end(), ctx->dit_ev_used.begin(), ctx->dit_ev_used.end());
    ctx->dit_ev_used.clear();
    if (ms_gemm) *ms_gemm = gemm;
    if (ms_awa) *ms_awa = awa_ms;
    if (ms_eltwise) *ms_eltwise = elt;
    if (layers) *layers = (int)n;
    return rc;
}

}  // extern "C"
