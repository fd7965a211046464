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
// One sequential sum per output is therefore fixed: k_linear_seq (fh_seq.hpp)
// over the Q8_0 planes or the F32 rows.  The opt-in exact mode; FH_W8A32 is the
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
        const float d = c * kChunk + seg * 8 < k ? fh_h2f(r.d) : 0.0f;
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
        const bool in = c * kChunk + seg * 8 < k;
#pragma unroll
        for (int v = 0; v < 2; v++)
            wt[(seg * 2 + v) * C + col] = in ? r.v[v] : fh_seq::f4{0.0f, 0.0f, 0.0f, 0.0f};
    }
};

}  // namespace

int fh_launch_linear_exact(fh_ctx* ctx, const fh_q8_0* w, const float* x, size_t m, const float* bias, float* y) {
    if (w->n > 0x7FFFFFFFu || w->k > 0x7FFFFFFFu || m > 0x7FFFFFFFu)
        return fh_fail(ctx, FH_ERR_LIMIT, "fh_q8_0_linear: a dimension is above 2^31 - 1");
    if (w->n == 0 || m == 0) return FH_OK;
    if (w->kind == FH_WEIGHT_F32)
        fh_seq::launch(ctx, F32Src{w->f32, w->pitch}, (w->n + Q8Src::C - 1) / Q8Src::C, x, m, bias, y, w->n, w->k);
    else
        fh_seq::launch(ctx, Q8Src{w->qs, w->d}, (w->n + Q8Src::C - 1) / Q8Src::C, x, m, bias, y, w->n, w->k);
    FH_HIP(ctx, hipGetLastError());
    return FH_OK;
}
