// A post-LN encoder layer's training step, one call per direction, and its inference in bf16, one call: the order in which the kernels of the layer are launched
// and where in the two buffers their tensors lie.  Host code: launches cost 2 to 3 us each from here, 6 to 10 from Python and
// 18 to 29 through torch's products, and a layer has 9 of them forward and 18 to 20 backward, of which most last less than that.

#include <hip/hip_runtime.h>
#include <stdint.h>
#include "gemm_f32_internal.h"
#include "geo_attn_internal.h"

namespace {

enum { P_QW, P_KW, P_VW, P_QB, P_KB, P_VB, P_SPREAD, P_WO, P_G1, P_B1, P_W1, P_BIAS1, P_W2, P_BIAS2, P_G2, P_B2 };

struct Sizes {
    int Z, N, H, dk, dm, hidden;
    long rows;
    bool ok;
    Sizes(int Z_, int N_, int H_, int dk_, int hidden_) : Z(Z_), N(N_), H(H_), dk(dk_), dm(0), hidden(hidden_), rows(0), ok(false)
    {
        if (Z <= 0 || N <= 0 || H <= 0 || hidden <= 0 || hidden % 4 || (dk != 32 && dk != 64 && dk != 128) || (int64_t)H * dk > 2048) return;
        dm = H * dk; rows = (long)Z * N;
        // what the products and the attention address with 32 bits
        const int64_t widest = hidden > 3 * dm ? hidden : 3 * dm;
        ok = (rows + 512) * widest < (1LL << 29) && (int64_t)(hidden + 512) * dm < (1LL << 29) && (int64_t)(dm + 512) * widest < (1LL << 29)
             && (int64_t)Z * H <= 65535 && N <= PROTEUS_ATTN_MAX_N;
    }
};

// Buffers one behind the other on multiples of 256 bytes; with a null base, their total.
struct Carve {
    char* base;
    size_t at = 0;
    template <class T> T* take(const size_t n) { T* p = reinterpret_cast<T*>(base + at); at += (n * sizeof(T) + 255) / 256 * 256; return p; }
};

struct Kept {
    float *W, *b, *Wo, *sigma, *spread;
    uint16_t* qkv;
    float *O, *L, *y1, *stat1, *x1, *h, *a, *y2, *stat2;
    size_t bytes;
    Kept(const Sizes& s, void* base)
    {
        Carve c{static_cast<char*>(base)};
        const size_t dm = s.dm, rows = s.rows;
        W = c.take<float>(3 * dm * dm); b = c.take<float>(3 * dm); Wo = c.take<float>(dm * dm);
        sigma = c.take<float>(s.H); spread = c.take<float>(s.H);
        qkv = c.take<uint16_t>(rows * 3 * dm);
        O = c.take<float>(rows * dm); L = c.take<float>(rows * s.H);
        y1 = c.take<float>(rows * dm); stat1 = c.take<float>(rows * 2); x1 = c.take<float>(rows * dm);
        h = c.take<float>(rows * s.hidden); a = c.take<float>(rows * s.hidden);
        y2 = c.take<float>(rows * dm); stat2 = c.take<float>(rows * 2);
        bytes = c.at;
    }
};

struct Forward {
    float* branch;                 // what a residual adds: the attention's output, then the feed-forward's
    char* attn;
    size_t attn_bytes, bytes;
    Forward(const Sizes& s, void* base)
    {
        Carve c{static_cast<char*>(base)};
        branch = c.take<float>((size_t)s.rows * s.dm);
        attn_bytes = proteus_geo_attn_fwd_workspace_bytes(s.Z, s.H, s.N, s.dk, 0);
        attn = c.take<char>(attn_bytes);
        bytes = c.at;
    }
};

struct Backward {
    float *dy2, *dh, *dx1, *dy1, *dO, *D, *g, *d_sigma, *dW, *db, *dWo;
    uint16_t* dO16;
    void *lnws[2], *sums, *shares[4];                                               // of the gradients of weights: W2, W1, output projection, projections
    size_t ln_bytes, sums_bytes, shares_bytes[4], bytes;
    Backward(const Sizes& s, void* base)
    {
        Carve c{static_cast<char*>(base)};
        const size_t dm = s.dm, rows = s.rows;
        // What the feed-forward's half leaves behind the attention's half takes over: dh is read for the last time by the product that gives dx1, as is
        // dy2, and dx1 by the LayerNorm that gives dy1; g, dO and dO16 are written after that.
        dh = g = c.take<float>(rows * (s.hidden > 3 * s.dm ? s.hidden : 3 * dm));
        dy2 = dO = c.take<float>(rows * dm);
        dx1 = c.take<float>(rows * dm); dO16 = reinterpret_cast<uint16_t*>(dx1);
        dy1 = c.take<float>(rows * dm); D = c.take<float>(rows * s.H); d_sigma = c.take<float>(s.H);
        // (the second LayerNorm's partial sums are added up before the projections' gradient takes their place)
        ln_bytes = proteus_layernorm_bwd_workspace_bytes(s.rows, s.dm);
        dW = c.take<float>(3 * dm * dm > ln_bytes / 4 ? 3 * dm * dm : ln_bytes / 4); lnws[1] = dW;
        db = c.take<float>(3 * dm); dWo = c.take<float>(dm * dm);
        lnws[0] = c.take<char>(ln_bytes);
        sums_bytes = proteus_train_workspace_bytes(s.rows, s.hidden > 3 * s.dm ? s.hidden : 3 * s.dm);
        sums = c.take<char>(sums_bytes);
        const int sizes[4][2] = {{s.dm, s.hidden}, {s.hidden, s.dm}, {s.dm, s.dm}, {s.dm, 3 * s.dm}};
        for (int i = 0; i < 4; ++i) shares_bytes[i] = proteus_gemm_f32_workspace_bytes(sizes[i][0], sizes[i][1], (int)s.rows, PROTEUS_GEMM_TN);
        // (the last one's come when the others' are added up)
        shares[0] = shares[3] = c.take<char>(shares_bytes[0] > shares_bytes[3] ? shares_bytes[0] : shares_bytes[3]);
        shares[1] = c.take<char>(shares_bytes[1]); shares[2] = c.take<char>(shares_bytes[2]);
        bytes = c.at;
    }
};

bool off(const void* p, uintptr_t by) { return ((uintptr_t)p & (by - 1)) != 0; }

// strides (batch, head, token) of the heads of a [Z,N,parts,H,dk] tensor
void head_strides(int64_t* st, const Sizes& s, const int parts) { st[0] = (int64_t)s.N * parts * s.dm; st[1] = s.dk; st[2] = (int64_t)parts * s.dm; }

#define TRY(call) do { const int rc_ = (call); if (rc_ != PROTEUS_OK) return rc_; } while (0)

}  // namespace

extern "C" size_t proteus_encoder_layer_kept_bytes(int Z, int N, int H, int d_head, int hidden)
{
    const Sizes s(Z, N, H, d_head, hidden);
    return s.ok ? Kept(s, nullptr).bytes : 0;
}
extern "C" size_t proteus_encoder_layer_fwd_bytes(int Z, int N, int H, int d_head, int hidden)
{
    const Sizes s(Z, N, H, d_head, hidden);
    return s.ok ? Forward(s, nullptr).bytes : 0;
}
extern "C" size_t proteus_encoder_layer_bwd_bytes(int Z, int N, int H, int d_head, int hidden)
{
    const Sizes s(Z, N, H, d_head, hidden);
    return s.ok ? Backward(s, nullptr).bytes : 0;
}

extern "C" int proteus_encoder_layer_fwd(const float* x, const float* coords, const uint8_t* mask, const float* const* p, float min_spread,
                                         float eps1, float eps2, float* out, void* kept, size_t kept_bytes, void* ws, size_t ws_bytes,
                                         int Z, int N, int H, int d_head, int hidden, void* stream)
{
    if (!x || !coords || !p || !out || !kept || !ws) return PROTEUS_ERR_NULL_POINTER;
    for (int i = 0; i < PROTEUS_LAYER_PARAMS; ++i) {
        if (!p[i]) return PROTEUS_ERR_NULL_POINTER;
        if (off(p[i], 16)) return PROTEUS_ERR_BAD_ALIGNMENT;
    }
    const Sizes s(Z, N, H, d_head, hidden);
    if (!s.ok) return PROTEUS_ERR_BAD_SHAPE;
    if (off(x, 16) || off(out, 16) || off(kept, 256) || off(ws, 256)) return PROTEUS_ERR_BAD_ALIGNMENT;
    const Kept k(s, kept);
    const Forward f(s, ws);
    if (kept_bytes < k.bytes || ws_bytes < f.bytes) return PROTEUS_ERR_BAD_SHAPE;
    const int rows = (int)s.rows, dm = s.dm;

    float* heads[8];
    for (int i = 0; i < 8; ++i) heads[i] = const_cast<float*>(p[i]);
    heads[6] = k.spread;
    TRY(proteus_heads_layout(heads, k.W, k.b, k.Wo, k.sigma, p[P_SPREAD], dm, H, d_head, min_spread, 0, stream));
    TRY(proteus_gemm_f32(x, k.W, k.b, nullptr, k.qkv, nullptr, rows, 3 * dm, dm, dm, 3 * dm, 3 * dm, PROTEUS_GEMM_NN, PROTEUS_GEMM_BF16, stream));
    int64_t st[12];
    for (int i = 0; i < 3; ++i) head_strides(st + 3 * i, s, 3);
    head_strides(st + 9, s, 1);
    const uint16_t *q = k.qkv, *key = k.qkv + dm, *v = k.qkv + 2 * dm;
    if (f.attn_bytes) TRY(proteus_geo_attn_fwd_ws(q, key, v, st, coords, k.sigma, mask, k.O, k.L, f.attn, f.attn_bytes, Z, H, N, d_head, 0, stream));
    else              TRY(proteus_geo_attn_fwd_strided(q, key, v, st, coords, k.sigma, mask, k.O, k.L, Z, H, N, d_head, 0, stream));
    TRY(proteus_gemm_f32(k.O, k.Wo, nullptr, nullptr, f.branch, nullptr, rows, dm, dm, dm, dm, dm, PROTEUS_GEMM_NT, PROTEUS_GEMM_F32, stream));
    TRY(proteus_add_layernorm_train_fwd(x, f.branch, p[P_G1], p[P_B1], k.x1, k.y1, k.stat1, s.rows, dm, eps1, stream));
    TRY(proteus_gemm_f32(k.x1, p[P_W1], p[P_BIAS1], nullptr, k.a, k.h, rows, hidden, dm, dm, dm, hidden, PROTEUS_GEMM_NT, PROTEUS_GEMM_GELU, stream));
    TRY(proteus_gemm_f32(k.a, p[P_W2], p[P_BIAS2], nullptr, f.branch, nullptr, rows, dm, hidden, hidden, hidden, dm, PROTEUS_GEMM_NT, PROTEUS_GEMM_F32, stream));
    return proteus_add_layernorm_train_fwd(k.x1, f.branch, p[P_G2], p[P_B2], out, k.y2, k.stat2, s.rows, dm, eps2, stream);
}

extern "C" int proteus_encoder_layer_bwd(const float* x, const float* coords, const uint8_t* mask, const float* const* p, const float* dout,
                                         float* dx, float* const* g, float min_spread, const void* kept, size_t kept_bytes, void* ws, size_t ws_bytes,
                                         int Z, int N, int H, int d_head, int hidden, void* stream)
{
    if (!x || !coords || !p || !dout || !g || !kept || !ws || !p[P_G1] || !p[P_W1] || !p[P_W2] || !p[P_G2]) return PROTEUS_ERR_NULL_POINTER;
    for (int i = 0; i < PROTEUS_LAYER_PARAMS; ++i)
        if (off(g[i], 16)) return PROTEUS_ERR_BAD_ALIGNMENT;
    const Sizes s(Z, N, H, d_head, hidden);
    if (!s.ok) return PROTEUS_ERR_BAD_SHAPE;
    if (off(x, 16) || off(dout, 16) || off(dx, 16) || off(kept, 256) || off(ws, 256) || off(p[P_W1], 16) || off(p[P_W2], 16)) return PROTEUS_ERR_BAD_ALIGNMENT;
    const Kept k(s, const_cast<void*>(kept));
    const Backward b(s, ws);
    if (kept_bytes < k.bytes || ws_bytes < b.bytes) return PROTEUS_ERR_BAD_SHAPE;
    const int rows = (int)s.rows, dm = s.dm;
    auto product = [&](const float* A, const float* B, const float* h, float* C, int m, int n, int kk, int lda, int ldb, int form, int epilogue) {
        return proteus_gemm_f32(A, B, nullptr, h, C, nullptr, m, n, kk, lda, ldb, n, form, epilogue, stream);
    };
    // (The shares of several products, the last sums of the LayerNorms and the biases' in one launch, which must come before what they are of is written over.  Each of the
    // sums in a launch of its own, five per layer, took 5.3 us.)
    proteus_gemm::PendingSums pending;
    auto gradient = [&](const float* A, const float* B, float* C, int m, int n, int which) {
        return proteus_gemm::gemm_begin(A, B, C, m, n, rows, m, n, n, b.shares_bytes[which] ? b.shares[which] : nullptr, b.shares_bytes[which], pending, stream);
    };
    auto column_sums = [&](const float* a, float* out, int C) {
        return pending.add({a, out, rows, C}) ? (int)PROTEUS_OK : proteus_colsum(a, out, b.sums, b.sums_bytes, s.rows, C, stream);
    };
    auto layernorm = [&](const float* d, const float* y, const float* stat, const float* gamma, float* dy, float* dgamma_dbeta, int which) {
        proteus_train::ColumnSums sums;
        const int rc = proteus_train::layernorm_bwd_begin(d, y, stat, gamma, dy, dgamma_dbeta, b.lnws[which], b.ln_bytes, s.rows, dm, sums, stream);
        if (rc != PROTEUS_OK || !dgamma_dbeta || pending.add(sums)) return rc;
        return proteus_colsum(sums.a, sums.out, nullptr, 0, sums.rows, sums.cols, stream);
    };
    const bool projections = g[P_QW] || g[P_KW] || g[P_VW], biases = g[P_QB] || g[P_KB] || g[P_VB];
    const bool attention = dx || projections || biases || g[P_SPREAD];
    const bool first_norm = attention || g[P_WO] || g[P_G1];

    TRY(layernorm(dout, k.y2, k.stat2, p[P_G2], b.dy2, g[P_G2], 1));
    if (g[P_W2])    TRY(gradient(b.dy2, k.a, g[P_W2], dm, hidden, 0));
    if (g[P_BIAS2]) TRY(column_sums(b.dy2, g[P_BIAS2], dm));
    if (!(first_norm || g[P_W1] || g[P_BIAS1])) return proteus_gemm::gemm_sums(pending, stream);
    TRY(product(b.dy2, p[P_W2], k.h, b.dh, rows, hidden, dm, dm, hidden, PROTEUS_GEMM_NN, PROTEUS_GEMM_GELU_GRAD));
    if (g[P_W1])    TRY(gradient(b.dh, k.x1, g[P_W1], hidden, dm, 1));
    if (g[P_BIAS1]) TRY(column_sums(b.dh, g[P_BIAS1], hidden));
    if (!first_norm) return proteus_gemm::gemm_sums(pending, stream);
    TRY(product(b.dh, p[P_W1], b.dy2, b.dx1, rows, dm, hidden, hidden, dm, PROTEUS_GEMM_NN, PROTEUS_GEMM_ADD));
    TRY(layernorm(b.dx1, k.y1, k.stat1, p[P_G1], b.dy1, g[P_G1], 0));
    if (g[P_WO]) TRY(gradient(b.dy1, k.O, b.dWo, dm, dm, 2));
    if (attention) {
        TRY(proteus_gemm::gemm_sums(pending, stream));                          // dO takes dy2's place, g dh's
        TRY(product(b.dy1, k.Wo, nullptr, b.dO, rows, dm, dm, dm, dm, PROTEUS_GEMM_NN, PROTEUS_GEMM_F32));
        int64_t st[21];
        for (int i = 0; i < 3; ++i) head_strides(st + 3 * i, s, 1);          // O, dO, dO in bf16
        TRY(proteus_geo_attn_prepare_bwd(k.O, b.dO, st, b.D, b.dO16, b.d_sigma, nullptr, Z, H, N, d_head, PROTEUS_DTYPE_F32, PROTEUS_OPERAND_BF16, stream));
        for (int i = 0; i < 7; ++i) head_strides(st + 3 * i, s, i == 3 ? 1 : 3);
        TRY(proteus_geo_attn_bwd_typed(k.qkv, k.qkv + dm, k.qkv + 2 * dm, b.dO16, st, coords, k.sigma, nullptr, mask, k.L, b.D, b.g, b.g + dm, b.g + 2 * dm,
                                       b.d_sigma, nullptr, Z, H, N, d_head, 0.0f, 1.0f, PROTEUS_OPERAND_BF16, PROTEUS_GRAD_F32, stream));
        if (projections) TRY(gradient(x, b.g, b.dW, dm, 3 * dm, 3));
        if (biases)      TRY(column_sums(b.g, b.db, 3 * dm));
        if (dx)          TRY(product(b.g, k.W, b.dy1, dx, rows, dm, 3 * dm, 3 * dm, 3 * dm, PROTEUS_GEMM_NT, PROTEUS_GEMM_ADD));
    }
    TRY(proteus_gemm::gemm_sums(pending, stream));
    if (projections || biases || g[P_SPREAD] || g[P_WO])
        TRY(proteus_heads_layout(g, b.dW, b.db, b.dWo, b.d_sigma, k.spread, dm, H, d_head, min_spread, 1, stream));
    return PROTEUS_OK;
}

// ---- inference in bf16 ----

namespace {

enum { I_QKV, I_QKVB, I_WO, I_G1, I_B1, I_W1, I_BIAS1, I_W2, I_BIAS2, I_G2, I_B2, I_PARAMS };

struct Infer {
    uint16_t *wide, *O, *branch, *x1;                          // wide: Q, K and V, then the feed-forward's hidden layer
    char* attn;
    size_t attn_bytes, bytes;
    Infer(const Sizes& s, void* base)
    {
        Carve c{static_cast<char*>(base)};
        const size_t dm = s.dm, rows = s.rows;
        wide = c.take<uint16_t>(rows * (s.hidden > 3 * s.dm ? s.hidden : 3 * dm));
        O = c.take<uint16_t>(rows * dm); branch = c.take<uint16_t>(rows * dm); x1 = c.take<uint16_t>(rows * dm);
        attn_bytes = proteus_geo_attn_fwd_workspace_bytes(s.Z, s.H, s.N, s.dk, 0);
        attn = c.take<char>(attn_bytes);
        bytes = c.at;
    }
};

bool infer_ok(const Sizes& s) { return s.ok && s.hidden % 8 == 0 && s.rows < (1L << 31); }

}  // namespace

extern "C" size_t proteus_encoder_infer_bytes(int Z, int N, int H, int d_head, int hidden)
{
    const Sizes s(Z, N, H, d_head, hidden);
    return infer_ok(s) ? Infer(s, nullptr).bytes : 0;
}

extern "C" int proteus_encoder_infer(const uint16_t* x, const float* coords, const float* sigma, const uint8_t* mask, const uint16_t* const* p,
                                     float eps1, float eps2, uint16_t* out, void* ws, size_t ws_bytes, int Z, int N, int H, int d_head, int hidden, void* stream)
{
    if (!x || !coords || !sigma || !p || !out || !ws) return PROTEUS_ERR_NULL_POINTER;
    for (int i = 0; i < I_PARAMS; ++i) {
        if (!p[i]) return PROTEUS_ERR_NULL_POINTER;
        if (off(p[i], 16)) return PROTEUS_ERR_BAD_ALIGNMENT;
    }
    const Sizes s(Z, N, H, d_head, hidden);
    if (!infer_ok(s)) return PROTEUS_ERR_BAD_SHAPE;
    if (off(x, 16) || off(out, 16) || off(ws, 256)) return PROTEUS_ERR_BAD_ALIGNMENT;
    const Infer f(s, ws);
    if (ws_bytes < f.bytes) return PROTEUS_ERR_BAD_SHAPE;
    const int rows = (int)s.rows, dm = s.dm;
    auto product = [&](const uint16_t* A, int w, int b, uint16_t* C, int n, int k, int gelu) {
        return proteus_gemm_bf16(A, p[w], b < 0 ? nullptr : p[b], C, rows, n, k, k, k, n, gelu, stream);
    };
    TRY(product(x, I_QKV, I_QKVB, f.wide, 3 * dm, dm, 0));
    int64_t st[12];
    for (int i = 0; i < 3; ++i) head_strides(st + 3 * i, s, 3);
    head_strides(st + 9, s, 1);
    TRY(proteus_internal::attn_fwd_bf16_out(f.wide, f.wide + dm, f.wide + 2 * dm, st, coords, sigma, mask, f.O, f.attn_bytes ? f.attn : nullptr, f.attn_bytes, Z, H, N, d_head, stream));
    TRY(product(f.O, I_WO, -1, f.branch, dm, dm, 0));
    TRY(proteus_add_layernorm_fwd(x, f.branch, p[I_G1], p[I_B1], f.x1, s.rows, dm, eps1, PROTEUS_DTYPE_BF16, stream));
    TRY(product(f.x1, I_W1, I_BIAS1, f.wide, hidden, dm, 1));
    TRY(product(f.wide, I_W2, I_BIAS2, f.branch, dm, hidden, 0));
    return proteus_add_layernorm_fwd(f.x1, f.branch, p[I_G2], p[I_B2], out, s.rows, dm, eps2, PROTEUS_DTYPE_BF16, stream);
}
