// The experts of an MoE layer from one call (host code only): selection, routing, both projections and the combination, and
// the backward pass, as calls of the library's entry points.  A layer called from Python otherwise spends more time between
// its launches than in its kernels when it is small.
#include "grouped_gemm_common.h"

namespace {

using namespace xma;

struct Layer {
    const xma_moe_args& a;
    void* stream;
    int64_t M, N;
    bool gated;

    Layer(const xma_moe_args& args, void* s)
        : a(args), stream(s), M(args.tokens * args.top_k), N(args.intermediate), gated(args.epilogue != XMA_EPI_GELU_TANH) {
        if (gated) N *= 2;
    }

    xma_grouped_gemm_args gemm(int kind, int64_t n, int64_t k) const {
        xma_grouped_gemm_args g = {};
        g.struct_size = sizeof(g);
        g.kind = kind;
        g.dtype = a.dtype;
        g.num_experts = a.num_experts;
        g.rows = M;
        g.n = n;
        g.k = k;
        g.lda = kind == XMA_GEMM_MT ? n : k;
        g.ldb = kind == XMA_GEMM_NN ? n : k;
        g.ldc = kind == XMA_GEMM_MT ? k : n;
        if (kind == XMA_GEMM_MT) g.c_expert_stride = n * k;
        else g.b_expert_stride = n * k;
        g.expert_offsets = a.expert_offsets;
        g.in_fan_out = 1;
        g.workspace = a.workspace;
        g.workspace_bytes = a.workspace_bytes;
        return g;
    }
    int run(const xma_grouped_gemm_args& g) const { return xma_grouped_gemm(&g, stream); }

    int up() const {
        auto g = gemm(XMA_GEMM_TN, N, a.hidden);
        g.epilogue = a.epilogue;
        g.a = a.x;
        g.b = a.w_up;
        g.c = a.act;
        g.ldc = a.intermediate;
        g.aux = a.preact;
        g.ld_aux = a.preact ? N : 0;
        g.in_index = a.perm;
        g.in_fan_out = a.top_k;
        g.bias = a.b_up;
        g.ld_bias = a.b_up ? N : 0;
        return run(g);
    }
    int down() const {
        auto g = gemm(XMA_GEMM_TN, a.hidden, a.intermediate);
        g.a = a.act;
        g.b = a.w_down;
        g.c = a.expanded;
        g.out_index = a.perm;
        g.bias = a.b_down;
        g.ld_bias = a.b_down ? a.hidden : 0;
        return run(g);
    }
    xma_grouped_gemm_args weight_gradient(const void* d_rows, int64_t n, const void* rows, int64_t k, void* out) const {
        auto g = gemm(XMA_GEMM_MT, n, k);
        g.a = d_rows;
        g.b = rows;
        g.c = out;
        return g;
    }
    // The up-projection's weight gradient reads the tokens where they are.  That takes a type of 16 bits, whole
    // vectors and byte offsets of 32 bits; otherwise their rows are copied in grouped order first.
    xma_grouped_gemm_args d_w_up() const { return weight_gradient(a.d_preact, N, a.x, a.hidden, a.d_w_up); }
    bool gathers_tokens() const {
        int32_t kernel = 0, tile_rows, tile_cols;
        const auto g = d_w_up();
        return a.dtype != XMA_F32 && 2 * a.tokens * a.hidden < ((int64_t)1 << 32) &&
               xma_grouped_gemm_form(&g, &kernel, &tile_rows, &tile_cols) == 0 && kernel == XMA_FORM_TILED;
    }
    // fp32: the kernel that looks the rows up itself waits for the look-up in every stage, so long reductions of wide gradients
    // pay for a copy.  us, look-up / copy + plain: 8192 rows over 8 experts, N 16384, H 2048 4512 / 14 + 4038; 17728 rows over 64, N
    // 2048, H 2048 1364 / 1257, N 512 386 / 357, N 256 189 / 196; 35456 rows over 128, N 512, H 576 235 / 229, N 128 76 / 85; 2216
    // rows over 8, H 576: N 2048 73 / 83, N 512 27 / 29; 256 rows over 8, N 512, H 2048 18 / 21
    bool copies_tokens() const { return a.dtype != XMA_F32 || (N >= 512 && M * N >= (int64_t)200000 * a.num_experts); }
    int d_preact() const {
        auto g = gemm(XMA_GEMM_NN, a.intermediate, a.hidden);
        g.epilogue = a.epilogue + 1;  // the activation's backward
        g.a = a.rows;
        g.b = a.w_down;
        g.c = a.d_preact;
        g.ldc = N;
        g.aux = a.preact;
        g.ld_aux = N;
        return run(g);
    }
    int d_rows() const {
        auto g = gemm(XMA_GEMM_NN, a.hidden, N);
        g.a = a.d_preact;
        g.b = a.w_up;
        g.c = a.rows;
        g.out_index = a.perm;
        return run(g);
    }
};

static_assert(XMA_EPI_SWIGLU_BWD == XMA_EPI_SWIGLU + 1 && XMA_EPI_GLU_BWD == XMA_EPI_GLU + 1 &&
                  XMA_EPI_GELU_TANH_BWD == XMA_EPI_GELU_TANH + 1,
              "an activation's backward follows it");

int check(const char* name, const xma_moe_args* a) {
    XMA_REQUIRE(a != nullptr && a->struct_size == sizeof(xma_moe_args) && a->reserved == 0, "%s: bad args", name);
    XMA_REQUIRE(valid_dtype(a->dtype), "%s: bad dtype %d", name, a->dtype);
    XMA_REQUIRE(a->epilogue == XMA_EPI_SWIGLU || a->epilogue == XMA_EPI_GLU || a->epilogue == XMA_EPI_GELU_TANH,
                "%s: bad epilogue %d", name, a->epilogue);
    XMA_REQUIRE(a->num_experts >= 1 && a->top_k >= 1 && a->top_k <= a->num_experts && a->tokens >= 1 && a->hidden >= 1 &&
                    a->intermediate >= 1,
                "%s: bad sizes", name);
    XMA_REQUIRE(a->tokens * a->top_k < ((int64_t)1 << 31), "%s: too many routed rows", name);
    XMA_REQUIRE(a->x && a->w_up && a->w_down && a->gates && a->expert_offsets && a->perm && a->act && a->expanded && a->workspace,
                "%s: null pointer", name);
    XMA_REQUIRE(a->workspace_bytes >= xma_moe_workspace_bytes(a->tokens, a->num_experts, a->top_k), "%s: workspace too small", name);
    return 0;
}

}  // namespace

#define XMA_STEP(call)            \
    do {                          \
        const int status_ = call; \
        if (status_) return status_; \
    } while (0)

extern "C" {

int64_t xma_moe_workspace_bytes(int64_t tokens, int32_t num_experts, int32_t top_k) {
    if (tokens < 0 || num_experts < 1 || top_k < 1) return -1;
    // one user at a time: routing, then each grouped GEMM
    const int64_t route = xma_route_workspace_bytes(tokens * top_k, num_experts);
    const int64_t gemm = xma_grouped_gemm_workspace_bytes(num_experts, tokens * top_k);
    return route > gemm ? route : gemm;
}

int xma_moe_forward(const xma_moe_args* args, void* stream) {
    XMA_STEP(check("xma_moe_forward", args));
    const xma_moe_args& a = *args;
    XMA_REQUIRE(a.selected && a.counts && a.sorted_experts && a.y, "xma_moe_forward: null pointer");
    const Layer layer(a, stream);
    if (a.logits) {
        XMA_STEP(xma_topk_route(a.logits, a.dtype, a.tokens, a.num_experts, a.top_k, a.num_experts, a.gates, a.selected, a.counts,
                                a.expert_offsets, a.sorted_experts, a.perm, a.workspace, a.workspace_bytes, stream));
    } else {
        XMA_STEP(xma_route_build(a.selected, 1, layer.M, a.num_experts, a.counts, a.expert_offsets, a.sorted_experts, a.perm, 0,
                                 a.workspace, a.workspace_bytes, stream));
    }
    XMA_STEP(layer.up());
    XMA_STEP(layer.down());
    return xma_combine_topk(a.expanded, a.hidden, a.gates, a.y, a.hidden, a.tokens, a.top_k, a.hidden, a.dtype, stream);
}

int xma_moe_backward(const xma_moe_args* args, void* stream) {
    XMA_STEP(check("xma_moe_backward", args));
    const xma_moe_args& a = *args;
    XMA_REQUIRE(a.preact && a.d_y && a.d_x && a.d_gates && a.d_w_up && a.d_w_down && a.d_preact && a.rows && a.inverse,
                "xma_moe_backward: null pointer");
    const Layer layer(a, stream);
    const int64_t H = a.hidden, I = a.intermediate, N = layer.N;
    const bool gathers = layer.gathers_tokens();
    uint32_t* token_offsets = reinterpret_cast<uint32_t*>(a.inverse) + layer.M;
    if (gathers) {
        XMA_STEP(launch_invert_and_locate(a.perm, layer.M, a.top_k, (uint32_t)(2 * H), a.inverse, token_offsets, kRowOffsetsPadding,
                                          stream));
    } else {
        XMA_STEP(xma_invert_index(a.perm, 0, layer.M, a.inverse, stream));
    }
    // the output's gradient in grouped order, and the gates'
    XMA_STEP(xma_spread_rows(a.d_y, H, a.rows, H, a.perm, 0, a.inverse, a.tokens, a.top_k, H, a.dtype, a.gates, a.expanded, H,
                             a.d_gates, stream));
    if (a.d_b_down) XMA_STEP(xma_expert_colsum(a.rows, H, a.expert_offsets, a.num_experts, H, a.d_b_down, H, a.dtype, stream));
    XMA_STEP(layer.run(layer.weight_gradient(a.rows, H, a.act, I, a.d_w_down)));
    XMA_STEP(layer.d_preact());
    if (a.d_b_up) XMA_STEP(xma_expert_colsum(a.d_preact, N, a.expert_offsets, a.num_experts, N, a.d_b_up, N, a.dtype, stream));
    // `rows` holds the output's gradient, then the inputs of the up-projection where they are copied, then its input gradients
    auto d_w_up = layer.d_w_up();
    if (gathers) {
        XMA_STEP(launch_gathered_weight_gradient(d_w_up, token_offsets, (hipStream_t)stream));
    } else if (!layer.copies_tokens()) {
        d_w_up.in_index = a.perm;
        d_w_up.in_fan_out = a.top_k;
        XMA_STEP(layer.run(d_w_up));
    } else {
        XMA_STEP(xma_spread_rows(a.x, H, a.rows, H, a.perm, 0, a.inverse, a.tokens, a.top_k, H, a.dtype, nullptr, nullptr, 0,
                                 nullptr, stream));
        d_w_up.b = a.rows;
        XMA_STEP(layer.run(d_w_up));
    }
    XMA_STEP(layer.d_rows());
    return xma_combine_topk(a.rows, H, nullptr, a.d_x, H, a.tokens, a.top_k, H, a.dtype, stream);
}

}  // extern "C"
