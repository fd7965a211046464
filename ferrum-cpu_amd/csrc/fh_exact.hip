// fh_exact.hip — FH_W8A32_EXACT: the Q8_0 linear bit for bit as ferrum_core
// computes it over the expanded weights.
//
// ferrum_core expands a Q8_0 matrix to f32 at load (w = f32(f16 d) * q, exact:
// loader/decode.rs:97-100, gguf/tensors.rs:58-87) and runs linear_forward
// (ops.rs:233-256): matmul_block accumulates every output from zero, adding
// the products x[p] * w[p][j] in ascending p with a rounding after each
// product and each add (ops.rs:29-126, no fused multiply-add), and
// matmul_bias_block adds the bias after the contraction (ops.rs:132-148).  The
// row split over threads (parallel.rs:90-92) never splits an output's sum, so
// the result does not depend on the thread count.  The reference's roadmap
// names this contract for a packed Q8_0 forward
// (q8_0_packed_forward_equals_expanded).
//
// One sequential sum per output is therefore fixed: k_linear_seq and, for few
// outputs, k_linear_seq_row (fh_seq.hpp) over the Q8_0 planes or the F32 rows.  The opt-in exact mode; FH_W8A32 is the
// fast one.
#include "fh_seq.hpp"

#pragma clang fp contract(off)

namespace {

using fh_seq::kChunk;

// Thread t widens 8 positions (segment t / 16 of the chunk) of column t % 16,
// so its float4s fall on 16 different slots of a 16-lane group.
struct Q8Src {
    static constexpr int C = 16;
    static constexpr bool kBiasFirst = false, kScaled = false;
    const int8_t* qs;     // quant plane [n][k]
    const uint16_t* dsc;  // f16 scales [n][k / 32]
    struct Raw {
        uint2 q;
        uint16_t d;
    };
    __device__ __forceinline__ int column(int tile, int c, int n) const {
        const int j = tile * C + c;
        return j < n ? j : -1;
    }
    __device__ __forceinline__ void load(int tid, int tile, int c, int n, int k, Raw& r) const {
        const size_t j = static_cast<size_t>(min(tile * C + (tid & 15), n - 1));
        const int p = min(c * kChunk + (tid >> 4) * 8, k - 8);  // (k is a multiple of 32)
        r.q = *reinterpret_cast<const uint2*>(qs + j * k + p);
        r.d = dsc[j * (k >> 5) + (p >> 5)];
    }
    __device__ __forceinline__ void store(int tid, int c, int k, const Raw& r, fh_seq::f4* wt) const {
        const int col = tid & 15, seg = tid >> 4;
        // past K: d = 0 (the products are +0 or -0, and a sum that starts at +0 is never -0)
        const float d = fh_seq::inside(c, seg * 8, k) ? fh_h2f(r.d) : 0.0f;
        const uint32_t words[2] = {r.q.x, r.q.y};
#pragma unroll
        for (int v = 0; v < 2; v++) {
            float e[4];
#pragma unroll
            for (int b = 0; b < 4; b++)  // exact: an f16 value times an 8-bit integer
                e[b] = d * static_cast<float>(static_cast<int8_t>((words[v] >> (8 * b)) & 0xFFu));
            wt[(seg * 2 + v) * C + col] = fh_seq::f4{e[0], e[1], e[2], e[3]};
        }
    }
    struct Row {
        uint4 q;
        uint16_t d;
    };
    __device__ __forceinline__ void load_row(int j, int p, int k, Row& r) const {
        p = min(p, k - 16);
        r.q = *reinterpret_cast<const uint4*>(qs + static_cast<size_t>(j) * k + p);
        r.d = dsc[static_cast<size_t>(j) * (k >> 5) + (p >> 5)];
    }
    __device__ __forceinline__ fh_seq::f4 quad(const Row& r, int v) const {
        const uint32_t word = v == 0 ? r.q.x : v == 1 ? r.q.y : v == 2 ? r.q.z : r.q.w;
        const float d = fh_h2f(r.d);
        float e[4];
#pragma unroll
        for (int b = 0; b < 4; b++) e[b] = d * static_cast<float>(static_cast<int8_t>((word >> (8 * b)) & 0xFFu));
        return fh_seq::f4{e[0], e[1], e[2], e[3]};
    }
};

struct F32Src {
    static constexpr int C = 16;
    static constexpr bool kBiasFirst = false, kScaled = false;
    const float* rows;  // [n][pitch], zeros from k to pitch (k rounded up to 16)
    size_t pitch;
    struct Raw {
        fh_seq::f4 v[2];
    };
    __device__ __forceinline__ int column(int tile, int c, int n) const {
        const int j = tile * C + c;
        return j < n ? j : -1;
    }
    __device__ __forceinline__ void load(int tid, int tile, int c, int n, int k, Raw& r) const {
        const size_t j = static_cast<size_t>(min(tile * C + (tid & 15), n - 1));
        const int p = c * kChunk + (tid >> 4) * 8;
        const auto* src = reinterpret_cast<const fh_seq::f4*>(rows + j * pitch + (p < k ? p : 0));
        r.v[0] = src[0];
        r.v[1] = src[1];
    }
    __device__ __forceinline__ void store(int tid, int c, int k, const Raw& r, fh_seq::f4* wt) const {
        const int col = tid & 15, seg = tid >> 4;
        const bool in = fh_seq::inside(c, seg * 8, k);
#pragma unroll
        for (int v = 0; v < 2; v++)
            wt[(seg * 2 + v) * C + col] = in ? r.v[v] : fh_seq::f4{0.0f, 0.0f, 0.0f, 0.0f};
    }
    struct Row {
        fh_seq::f4 v[4];
    };
    __device__ __forceinline__ void load_row(int j, int p, int k, Row& r) const {
        const auto* src = reinterpret_cast<const fh_seq::f4*>(rows + j * pitch + (p < k ? p : 0));
#pragma unroll
        for (int v = 0; v < 4; v++) r.v[v] = src[v];
    }
    __device__ __forceinline__ fh_seq::f4 quad(const Row& r, int v) const { return r.v[v]; }
};

// One row of x takes the decode form (k_linear_seq_row), and so do several where
// its workgroups, one per row and 16 columns, are few per CU: they widen the
// weights for their one row again, where k_linear_seq does so for 16 to 64.  us per
// call, k_linear_seq against the decode form: up to two per CU, 768 x 3072 at m = 10
// (480) 23.5 / 13.5, 4096 x 1024 at m = 2 (512) 8.8 / 7.4; up to three per CU, from
// K = 2048 on, 768 x 3072 at m = 16 23.4 / 17.7, 1024 x 4096 at m = 12 30.5 / 22.0 (but
// 4096 x 1024 at m = 3 8.8 / 9.0, 128 x 512 at m = 96 6.2 / 6.6).  F32 rows are four times
// the bytes: up to one per CU, 768 x 3065 at m = 4 20.9 / 12.8 (at m = 16, three per CU,
// 22.4 / 28.6).  A K of one k_linear_seq chunk stays there (4096 x 128 at m = 1
// 4.1 / 4.5).
template <class Src>
void launch(fh_ctx* ctx, const Src& src, const fh_q8_0* w, const float* x, size_t m, const float* bias, float* y) {
    const size_t tiles = (w->n + Src::C - 1) / Src::C, cus = static_cast<size_t>(ctx->num_cus);
    const size_t per_cu = w->kind == FH_WEIGHT_F32 ? 1 : w->k >= 2048 ? 3 : 2;
    // (the decode form's positions run up to a chunk past K in 32 bits)
    const bool decode = (m == 1 || (m <= 65535 && tiles * m <= per_cu * cus)) && w->k > kChunk && w->k <= 0x7FFFF000u;
    auto go = [&](auto kernel) {
        hipLaunchKernelGGL(kernel, fh_seq::tile_grid(tiles, m), dim3(fh_seq::kThreads), 0, ctx->stream, src, x, bias, y,
                           static_cast<int>(w->n), static_cast<int>(w->k));
    };
    if (!decode) fh_seq::launch(ctx, src, tiles, x, m, bias, y, w->n, w->k);
    else if (tiles > 2 * cus && w->k < 2048) go(fh_seq::k_linear_seq_row<Src, 1>);
    else go(fh_seq::k_linear_seq_row<Src, 2>);
}

}  // namespace

int fh_launch_linear_exact(fh_ctx* ctx, const fh_q8_0* w, const float* x, size_t m, const float* bias, float* y) {
    if (w->n > 0x7FFFFFFFu || w->k > 0x7FFFFFFFu || m > 0x7FFFFFFFu)
        return fh_fail(ctx, FH_ERR_LIMIT, "fh_q8_0_linear: a dimension is above 2^31 - 1");
    if (w->n == 0 || m == 0) return FH_OK;
    if (w->kind == FH_WEIGHT_F32)
        launch(ctx, F32Src{w->f32, w->pitch}, w, x, m, bias, y);
    else
        launch(ctx, Q8Src{w->qs, w->d}, w, x, m, bias, y);
    FH_HIP(ctx, hipGetLastError());
    return FH_OK;
}
