// fh_attn_prefill.hip — the attention of a prompt block on the matrix cores.
//
// What it computes: the attention of TransformerBlock::forward_with_cache
// (layer/transformer.rs:242-279) for every row of a prompt block at once.
// CachedTransformer's prime (slm/cached.rs:129-136) feeds a prompt position by
// position; here row r of sequence s is position pos0 + r and attends over
// cache positions 0 .. pos0 + r of its own sequence, with the scores
// (q . k) * 1/sqrt(hd), their softmax and the weighted sum of v rows.  Keys
// before the block come from the caches, the block's own from its q|k|v rows;
// the same launch writes the block's k / v rows into the caches.
//
// How (head widths 32 and 64): one workgroup per (128 query rows, head, sequence).
// Each of its four waves owns 32 query rows and walks 32-key tiles of the
// sequence's cache up to its last row's position; the tiles are staged in LDS
// once for the four waves (double-buffered, the next tile's loads in flight
// while the current one is used).  Per tile, flash style: S^T = K Q^T on the
// matrix cores, the masked softmax with a running max and sum per query
// (exact rescaling between tiles), then O += P V on the matrix cores, P
// going in straight from the S^T accumulators as the B operand of O^T += V^T P^T,
// so that a lane keeps to one query throughout: the rescaling and the final
// division are by its own factors.  At width 64 the f32 operands ride on the
// f16 matrix cores as two terms each (k_attn_prefill_f16 below); at width 32 they stay
// as they are, on the fp32 ones (k_attn_prefill_f32).
#include "fh_internal.hpp"

#pragma clang fp contract(off)

namespace {

typedef float f32x16 __attribute__((ext_vector_type(16)));

constexpr int kHd = 64;        // k_attn_prefill_f16's head width
constexpr int kKeys = 32;      // keys per tile
constexpr int kRT = 4;         // waves of 32 query rows that share a key tile
constexpr int kPT = 64 * kRT, kQRows = 32 * kRT;

struct PrefillArgs {
    const float* qkv;   // row s * rows + r; head h's q at column h * hd
    int ld;             // qkv row stride (floats)
    float* kc;          // sequence s's caches at kc / vc + s * seq_stride, rows of kv_dim floats
    float* vc;
    size_t seq_stride;
    int kv_dim;
    int rows, pos0;
    float scale;
    float* out;         // row s * rows + r; head h at column h * hd
    int out_ld;
};

// Query row of accumulator v in a lane of half `half` (the 32 x 32 MFMA
// output layout: rows 8 (v / 4) + 4 half + v % 4).
__device__ __forceinline__ int acc_row(int v, int half) { return (v >> 2) * 8 + half * 4 + (v & 3); }

// The products on the f16 matrix cores: every f32 operand is carried as two
// f16 terms, x = h + l with l = f16(x - h) (22 significant bits), and a
// product of two such operands as the three f16 products h h' + h l' + l h'
// (the dropped l l' is 2^-22 of it), summed in f32 by v_mfma_f32_32x32x16_f16:
// 12 MFMAs per 32-key tile for S^T = K Q^T and 12 for O += P V, against 32 +
// 32 v_mfma_f32_32x32x2_f32 on the fp32 path, each of which takes twice an
// f16 one's cycles (32 prompts of 511 rows, 24 blocks: 10.6 -> 6.8 ms).
//   q, k: each query row and each key row is scaled by its own power of two
//     (its largest finite |value| into [2^14, 2^15)) before the split, and
//     the score is unscaled exactly afterwards with the 1/sqrt(hd) of the
//     reference: s = S' * (2^-eq / sqrt(hd)) * 2^-ek.  Non-finite values keep l = 0,
//     so inf and NaN reach the score as the f32 product gives them.
//   P V: P (in [0, 1]) is split as it leaves the score accumulators; a lane's
//     16 keys of its query are the B operand's two K16 steps as they stand
//     (keys 8 a + 4 half + (0..3)), and the v tile is staged transposed,
//     [dim][key] with the keys in that same order, as the A operand.  A tile
//     whose v values are not all finite and below 2^15 in magnitude is
//     finished on the vector units with only the attended keys (0 * inf would
//     otherwise turn a masked key's v into NaN), v read from the cache.
// The error is that of the 22-bit operands, ~2^-22 relative per product,
// well inside the 1e-5 rule.
// Bound: a wave's chain per tile, some 550 vector instructions, 24 dependent
// MFMAs and the waits for LDS and the barrier (a tile of its own keys: 790 vector
// instructions, shuffles through LDS for every row maximum and an LDS round trip
// for the rescaling before).  32 prompts of 511 rows, 12 heads: 176 -> 106 us, of
// which the order of the row groups (see the kernel) 40.
constexpr int kHPitch = kHd + 8;    // K tile row pitch (halves): 16-byte pieces of 8 rows on different banks
constexpr int kVPitch = kKeys + 8;  // V tile (transposed) row pitch (halves): 80-byte rows

typedef _Float16 h8f __attribute__((ext_vector_type(8)));
typedef _Float16 h2f __attribute__((ext_vector_type(2)));

// Position of key kk of a tile in the transposed V rows: K16 step s holds,
// per lane half g, the keys 8 (2 s) + 4 g + (0..3) then 8 (2 s + 1) + 4 g + (0..3).
__device__ __forceinline__ int vkey_pos(int kk) {
    const int a = kk >> 3, g = (kk >> 2) & 1, b = kk & 3;
    return 16 * (a >> 1) + 8 * g + 4 * (a & 1) + b;
}

// Offset of (dim, key position kp) in a transposed V tile: the 8-key chunks
// of dim row d are permuted by (d / 16) % 4, so the pair stores of one wave
// (16 dims 4 apart) spread over the banks; a chunk's 8 keys stay contiguous
// for the 16-byte operand loads.
__device__ __forceinline__ int vt_pos(int d, int kp) {
    return d * kVPitch + 8 * ((kp >> 3) ^ ((d >> 4) & 3)) + (kp & 7);
}

// 2^e with |x| 2^e in [2^14, 2^15) for the largest finite |x| (mx; 0 -> e = 0).
__device__ __forceinline__ int pow2_exponent(float mx) {
    if (!(mx > 0.0f)) return 0;
    const int E = static_cast<int>((__builtin_bit_cast(uint32_t, mx) >> 23) & 0xFF) - 126;
    return min(max(15 - E, -126), 126);
}
__device__ __forceinline__ float pow2f(int e) { return __builtin_bit_cast(float, static_cast<uint32_t>(e + 127) << 23); }

// e^x for x <= 0 as 2^(x log2 e) on the hardware's exp2 (v_exp_f32, 1 ulp):
// the product's rounding adds |x| 2^-24 relative, ~1e-6 for the x that carry
// weight in a softmax, far inside the 1e-5 rule; -inf gives 0, NaN stays NaN.
__device__ __forceinline__ float exp_approx(float x) { return __builtin_amdgcn_exp2f(x * 1.44269504088896341f); }

typedef float f2f __attribute__((ext_vector_type(2)));

// Two scaled f32 values as f16 h and l terms (SAFE: l = 0 for a non-finite value).
template <bool SAFE>
__device__ __forceinline__ void split2(float x0, float x1, float sc, h2f& h, h2f& l) {
    const f2f s = {x0 * sc, x1 * sc};
    h = __builtin_convertvector(s, h2f);
    f2f r = {s.x - static_cast<float>(h.x), s.y - static_cast<float>(h.y)};
    if (SAFE) {
        r.x = __builtin_isfinite(s.x) ? r.x : 0.0f;
        r.y = __builtin_isfinite(s.y) ? r.y : 0.0f;
    }
    l = __builtin_convertvector(r, h2f);
}

// Lane l's and lane l ^ 32's values, on the vector units (a shuffle goes through LDS).
__device__ __forceinline__ float max_halves(float v) {
    const auto r = __builtin_amdgcn_permlane32_swap(__builtin_bit_cast(int, v), __builtin_bit_cast(int, v), false, false);
    return fmaxf(__builtin_bit_cast(float, static_cast<int>(r[0])), __builtin_bit_cast(float, static_cast<int>(r[1])));
}
// The largest value of each 16-lane row (xor 1, xor 2, half mirror, mirror), by DPP operands.
template <int CTRL>
__device__ __forceinline__ float dpp_of(float v) {
    return __builtin_bit_cast(float, __builtin_amdgcn_mov_dpp(__builtin_bit_cast(int, v), CTRL, 0xF, 0xF, true));
}
__device__ __forceinline__ float max_row(float v) {
    v = fmaxf(v, dpp_of<0xB1>(v));
    v = fmaxf(v, dpp_of<0x4E>(v));
    v = fmaxf(v, dpp_of<0x141>(v));
    return fmaxf(v, dpp_of<0x140>(v));
}

// HALVES = 2: eight waves, the first four on the even key tiles and the others on
// the odd ones of the same 128 query rows, their sums merged at the end (a wave's
// walk over its tiles is a chain: half as long, where there are too few workgroups
// to fill the waves' waits with one another's work).
template <int HALVES>
__global__ void __launch_bounds__(kPT* HALVES, 2) k_attn_prefill_f16(PrefillArgs a) {
    constexpr int KI = kHd / 16, OT = kHd / 32;  // MFMA K steps of a score, 32-dim output tiles
    // one key tile, and per wave the P of a tile with unsafe v ([key][query])
    struct Stage {
        __align__(16) _Float16 kh[2][kKeys * kHPitch], kl[2][kKeys * kHPitch];
        __align__(16) _Float16 vh[2][kHd * kVPitch], vl[2][kHd * kVPitch];
        __align__(16) float kinv[2][kKeys];  // 2^-ek per key row
        __align__(16) float pt[kRT][kKeys * 33];
        int unsafe[3];                       // a tile's v is not safe for the split (step st: st % 3)
    };
    __shared__ Stage stages[HALVES];
    static_assert(HALVES == 1 || sizeof(Stage) >= kRT * (2 + 16 * OT) * 64 * sizeof(float), "the merge fits a stage");
    const int hf = HALVES == 1 ? 0 : __builtin_amdgcn_readfirstlane(static_cast<int>(threadIdx.x) / kPT);
    Stage& sm = stages[hf];
    auto& kh = sm.kh;
    auto& kl = sm.kl;
    auto& vh = sm.vh;
    auto& vl = sm.vl;
    auto& kinv = sm.kinv;

    const int tid = threadIdx.x % kPT, lane = tid & 63, half = lane >> 5, col = lane & 31;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    // The longest rows of every head and sequence first.  (With a head's row
    // groups next to each other, a group count of four or eight gave each XCD
    // groups of one length, since workgroups are dealt to the eight in turn.)
    const int groups = static_cast<int>(gridDim.z), g = groups - 1 - static_cast<int>(blockIdx.z);
    const int h = blockIdx.x, s = blockIdx.y;
    const int r0 = g * kQRows + wave * 32;
    const int last_row = min(a.rows - 1, g * kQRows + kQRows - 1);
    const int kmax = a.pos0 + last_row;
    const int ntiles = kmax / kKeys + 1;
    const int my_tiles = r0 < a.rows ? (a.pos0 + min(a.rows - 1, r0 + 31)) / kKeys + 1 : 0;
    const size_t sbase = static_cast<size_t>(s) * a.seq_stride + static_cast<size_t>(h) * kHd;
    float* kc = a.kc + sbase;
    float* vc = a.vc + sbase;

    // This lane's query: dims 16 i + 8 half + (0..7), i < 4 (the B
    // operand of step i), scaled by the row's power of two and split.
    h8f qh[KI], ql[KI];
    float qscale;
    {
        const int row = min(r0 + col, a.rows - 1);
        const float* qp = a.qkv + (static_cast<size_t>(s) * a.rows + row) * a.ld + h * kHd + half * 8;
        float qv[8 * KI];
#pragma unroll
        for (int i = 0; i < KI; i++) {
            const float4 u = *reinterpret_cast<const float4*>(qp + 16 * i);
            const float4 w = *reinterpret_cast<const float4*>(qp + 16 * i + 4);
            qv[8 * i] = u.x; qv[8 * i + 1] = u.y; qv[8 * i + 2] = u.z; qv[8 * i + 3] = u.w;
            qv[8 * i + 4] = w.x; qv[8 * i + 5] = w.y; qv[8 * i + 6] = w.z; qv[8 * i + 7] = w.w;
        }
        float mx = 0.0f;
#pragma unroll
        for (int i = 0; i < 8 * KI; i++)
            if (__builtin_isfinite(qv[i])) mx = fmaxf(mx, fabsf(qv[i]));
        mx = fmaxf(mx, __shfl_xor(mx, 32, 64));  // the other half of the row
        const int eq = pow2_exponent(mx);
        const float sc = pow2f(eq);
        qscale = pow2f(-eq) * a.scale;  // (a power of two: exact)
#pragma unroll
        for (int i = 0; i < KI; i++)
#pragma unroll
            for (int j = 0; j < 8; j += 2) {
                h2f hh, ll;
                split2<true>(qv[8 * i + j], qv[8 * i + j + 1], sc, hh, ll);
                qh[i][j] = hh.x; qh[i][j + 1] = hh.y;
                ql[i][j] = ll.x; ql[i][j + 1] = ll.y;
            }
    }
    const int qpos = a.pos0 + r0 + col;

    // Tile staging: thread t takes float4s t, t + kPT, ... of the k rows (row idx /
    // 16, dims 4 (idx % 16) ...); the 16 threads of a key row
    // are consecutive lanes, so its exponent is a 16-lane reduction.  Keys of
    // the block itself (pos0 on) come from its q|k|v rows, earlier ones from
    // the cache; the last row group's workgroup of each (sequence, head), which walks every tile,
    // also writes the block's k and v rows into the cache as it stages them
    // (no other workgroup of the launch reads those cache rows).
    const bool writer = g == groups - 1;
    const float* bq = a.qkv + static_cast<size_t>(s) * a.rows * a.ld + h * kHd;  // this sequence's block rows
    // The v rows go by pairs instead: thread t takes keys 2 (t / 16) and
    // 2 (t / 16) + 1, dims 4 (t % 16) ..., which sit side by side in the
    // transposed tile, so each dim is one 4-byte store per term.
    float4 pk[2], pv[2];
    auto key_row = [&](int key, int off, const float* cache) __attribute__((always_inline)) {
        return key >= a.pos0 ? bq + static_cast<size_t>(key - a.pos0) * a.ld + off
                             : cache + static_cast<size_t>(key) * a.kv_dim;
    };
    const int c0 = tid % 16 * 4;
    auto k_key = [&](int i) { return tid / 16 + i * (kPT / 16); };
    auto v_key = [&](int i) { return 2 * (tid / 16) + i; };
    const float* bk = bq + a.kv_dim + c0;
    const float* bv = bq + 2 * a.kv_dim + c0;
    auto fetch = [&](int t) __attribute__((always_inline)) {
        if (t * kKeys >= a.pos0) {  // (uniform) every key is the block's own
            const int r = t * kKeys - a.pos0, last = kmax - a.pos0;
#pragma unroll
            for (int i = 0; i < 2; i++)
                pk[i] = *reinterpret_cast<const float4*>(bk + static_cast<size_t>(min(r + k_key(i), last)) * a.ld);
#pragma unroll
            for (int i = 0; i < 2; i++)
                pv[i] = *reinterpret_cast<const float4*>(bv + static_cast<size_t>(min(r + v_key(i), last)) * a.ld);
            return;
        }
#pragma unroll
        for (int i = 0; i < 2; i++)
            pk[i] = *reinterpret_cast<const float4*>(key_row(min(t * kKeys + k_key(i), kmax), a.kv_dim, kc) + c0);
#pragma unroll
        for (int i = 0; i < 2; i++)
            pv[i] = *reinterpret_cast<const float4*>(key_row(min(t * kKeys + v_key(i), kmax), 2 * a.kv_dim, vc) + c0);
    };
    auto store_block_rows = [&](int t) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < 2; i++) {
            const int key = t * kKeys + k_key(i);
            if (key >= a.pos0 && key <= kmax)
                *reinterpret_cast<float4*>(kc + static_cast<size_t>(key) * a.kv_dim + c0) = pk[i];
        }
#pragma unroll
        for (int i = 0; i < 2; i++) {
            const int key = t * kKeys + v_key(i);
            if (key >= a.pos0 && key <= kmax)
                *reinterpret_cast<float4*>(vc + static_cast<size_t>(key) * a.kv_dim + c0) = pv[i];
        }
    };
    auto stash = [&](int st) __attribute__((always_inline)) {
        const int buf = st & 1;
#pragma unroll
        for (int i = 0; i < 2; i++) {
            const int row = k_key(i);
            const float4 k4 = pk[i];
            // fmaxf skips NaN (whose terms are NaN without a guard, as its
            // score is); an infinite maximum takes the rare guarded path.
            float mx = max_row(fmaxf(fmaxf(fabsf(k4.x), fabsf(k4.y)), fmaxf(fabsf(k4.z), fabsf(k4.w))));
            int ek;
            h2f h01, l01, h23, l23;
            if (__builtin_expect(__ballot(!__builtin_isfinite(mx)) != 0, 0)) {
                float fm = 0.0f;
                if (__builtin_isfinite(k4.x)) fm = fmaxf(fm, fabsf(k4.x));
                if (__builtin_isfinite(k4.y)) fm = fmaxf(fm, fabsf(k4.y));
                if (__builtin_isfinite(k4.z)) fm = fmaxf(fm, fabsf(k4.z));
                if (__builtin_isfinite(k4.w)) fm = fmaxf(fm, fabsf(k4.w));
                ek = pow2_exponent(max_row(fm));
                split2<true>(k4.x, k4.y, pow2f(ek), h01, l01);
                split2<true>(k4.z, k4.w, pow2f(ek), h23, l23);
            } else {
                ek = pow2_exponent(mx);
                split2<false>(k4.x, k4.y, pow2f(ek), h01, l01);
                split2<false>(k4.z, k4.w, pow2f(ek), h23, l23);
            }
            *reinterpret_cast<uint2*>(&kh[buf][row * kHPitch + c0]) =
                make_uint2(__builtin_bit_cast(uint32_t, h01), __builtin_bit_cast(uint32_t, h23));
            *reinterpret_cast<uint2*>(&kl[buf][row * kHPitch + c0]) =
                make_uint2(__builtin_bit_cast(uint32_t, l01), __builtin_bit_cast(uint32_t, l23));
            if (c0 == 0) kinv[buf][row] = pow2f(-ek);
        }
        const int kp = vkey_pos(v_key(0));  // even; the pair's second key at kp + 1
        const float va[4] = {pv[0].x, pv[0].y, pv[0].z, pv[0].w};
        const float vb[4] = {pv[1].x, pv[1].y, pv[1].z, pv[1].w};
        uint32_t top = 0;  // the largest magnitude's bits (inf and NaN above every finite one)
#pragma unroll
        for (int j = 0; j < 4; j++) {
            top = max(top, max(__builtin_bit_cast(uint32_t, va[j]) & 0x7FFFFFFFu,
                               __builtin_bit_cast(uint32_t, vb[j]) & 0x7FFFFFFFu));
            h2f hv, lv;
            split2<false>(va[j], vb[j], 1.0f, hv, lv);
            const int at = vt_pos(c0 + j, kp);
            *reinterpret_cast<uint32_t*>(&vh[buf][at]) = __builtin_bit_cast(uint32_t, hv);
            *reinterpret_cast<uint32_t*>(&vl[buf][at]) = __builtin_bit_cast(uint32_t, lv);
        }
        if (__builtin_expect(top >= 0x47000000u, 0)) sm.unsafe[st % 3] = 1;  // 2^15 or more
    };

    float m_run = -INFINITY, l_run = 0.0f;
    f32x16 o[OT];
#pragma unroll
    for (int d = 0; d < OT; d++) o[d] = f32x16{};
    // this half's tiles: hf, hf + HALVES, ... (a step past ntiles stages nothing)
    const int steps = (ntiles + HALVES - 1) / HALVES;
    if (tid < 3) sm.unsafe[tid] = 0;
    fetch(hf);
    if (writer) store_block_rows(hf);
    __syncthreads();
    stash(0);
    __syncthreads();
    for (int st = 0; st < steps; st++) {
        const int t = st * HALVES + hf, tn = t + HALVES, buf = st & 1, k0 = t * kKeys;
        if (tn < ntiles) fetch(tn);
        const bool vbad = sm.unsafe[st % 3] != 0;
        if (tid == 0) sm.unsafe[(st + 2) % 3] = 0;  // (read at step st - 1, written next at step st + 1)
        if (t < my_tiles) {
            // ---- S'^T = K Q^T (scaled terms): accumulator v of lane (half, col) is key acc_row(v, half), query col
            f32x16 sacc;
#pragma unroll
            for (int v = 0; v < 16; v++) sacc[v] = 0.0f;
            const _Float16* khr = &kh[buf][col * kHPitch + half * 8];
            const _Float16* klr = &kl[buf][col * kHPitch + half * 8];
#pragma unroll
            for (int i = 0; i < KI; i++) {
                const h8f a_h = *reinterpret_cast<const h8f*>(khr + 16 * i);
                const h8f a_l = *reinterpret_cast<const h8f*>(klr + 16 * i);
                sacc = __builtin_amdgcn_mfma_f32_32x32x16_f16(a_h, qh[i], sacc, 0, 0, 0);
                sacc = __builtin_amdgcn_mfma_f32_32x32x16_f16(a_h, ql[i], sacc, 0, 0, 0);
                sacc = __builtin_amdgcn_mfma_f32_32x32x16_f16(a_l, qh[i], sacc, 0, 0, 0);
            }
            // ---- scores, unscaled exactly, masked past the query's position
            // (only the last tiles of a wave hold masked keys)
            float sv[16];
            float mt = -INFINITY;
#pragma unroll
            for (int a4 = 0; a4 < 4; a4++) {
                const float4 ki = *reinterpret_cast<const float4*>(&kinv[buf][a4 * 8 + half * 4]);
                const float kv4[4] = {ki.x, ki.y, ki.z, ki.w};
#pragma unroll
                for (int j = 0; j < 4; j++) sv[4 * a4 + j] = sacc[4 * a4 + j] * qscale * kv4[j];
            }
            if (k0 + kKeys - 1 > a.pos0 + r0)
#pragma unroll
                for (int v = 0; v < 16; v++) sv[v] = k0 + acc_row(v, half) <= qpos ? sv[v] : -INFINITY;
#pragma unroll
            for (int v = 0; v < 16; v++) mt = fmaxf(mt, sv[v]);
            // (a query whose scores so far are all -inf, masked ones among them,
            // keeps sums of 0, and 0 / 0 = NaN if it ends so)
            const float m_new = fmaxf(m_run, max_halves(mt)), m_exp = m_new == -INFINITY ? 0.0f : m_new;
            const float corr = exp_approx(m_run - m_exp);  // 0 on the first tile (m_run = -inf)
            float ps = 0.0f;
#pragma unroll
            for (int v = 0; v < 16; v++) {
                sv[v] = exp_approx(sv[v] - m_exp);
                ps += sv[v];
            }
            l_run = l_run * corr + ps;  // (this half's keys; the halves are added at the end)
            m_run = m_new;
#pragma unroll
            for (int d = 0; d < OT; d++) o[d] *= corr;
            if (!vbad) {
                // ---- O^T += V^T P^T: step s2 takes this lane's keys acc_row(8 s2 + j, half)
#pragma unroll
                for (int s2 = 0; s2 < 2; s2++) {
                    h8f ph, pl;
#pragma unroll
                    for (int j = 0; j < 8; j += 2) {
                        h2f hh, ll;
                        split2<false>(sv[8 * s2 + j], sv[8 * s2 + j + 1], 1.0f, hh, ll);
                        ph[j] = hh.x; ph[j + 1] = hh.y;
                        pl[j] = ll.x; pl[j + 1] = ll.y;
                    }
                    const int off = 16 * s2 + 8 * half;
                    h8f v_h[OT], v_l[OT];
#pragma unroll
                    for (int d = 0; d < OT; d++) {
                        v_h[d] = *reinterpret_cast<const h8f*>(&vh[buf][vt_pos(32 * d + col, off)]);
                        v_l[d] = *reinterpret_cast<const h8f*>(&vl[buf][vt_pos(32 * d + col, off)]);
                    }
#pragma unroll
                    for (int d = 0; d < OT; d++) o[d] = __builtin_amdgcn_mfma_f32_32x32x16_f16(v_h[d], ph, o[d], 0, 0, 0);
#pragma unroll
                    for (int d = 0; d < OT; d++) o[d] = __builtin_amdgcn_mfma_f32_32x32x16_f16(v_l[d], ph, o[d], 0, 0, 0);
#pragma unroll
                    for (int d = 0; d < OT; d++) o[d] = __builtin_amdgcn_mfma_f32_32x32x16_f16(v_h[d], pl, o[d], 0, 0, 0);
                }
            } else {
                // ---- v not safe for the split: only the attended keys, on the vector units
                float* pw = sm.pt[wave];
#pragma unroll
                for (int v = 0; v < 16; v++) pw[acc_row(v, half) * 33 + col] = sv[v];
                __builtin_amdgcn_wave_barrier();
                // (lanes past the block's last row have a position past its last
                // key; they stop there, and store nothing)
                const int last = min(qpos, kmax);
                for (int kk = 0; kk < kKeys && k0 + kk <= last; kk++) {
                    const float p = pw[kk * 33 + col];
                    const float* vrow = key_row(k0 + kk, 2 * a.kv_dim, vc);
#pragma unroll
                    for (int d = 0; d < OT; d++)
#pragma unroll
                        for (int v = 0; v < 16; v++) o[d][v] += p * vrow[32 * d + acc_row(v, half)];
                }
                __builtin_amdgcn_wave_barrier();
            }
        }
        if (tn < ntiles) {
            if (writer) store_block_rows(tn);
            stash(st + 1);
        }
        __syncthreads();
    }
    float l = l_run + __shfl_xor(l_run, 32, 64);
    if constexpr (HALVES == 2) {
        // the odd tiles' maximum, sum and outputs through their stage's LDS
        // (every wave is past its last read of it), scaled to the common maximum
        float* mg = reinterpret_cast<float*>(&stages[1]) + wave * ((2 + 16 * OT) * 64) + lane;
        if (hf == 1) {
            mg[0] = m_run;
            mg[64] = l;
#pragma unroll
            for (int d = 0; d < OT; d++)
#pragma unroll
                for (int v = 0; v < 16; v++) mg[(2 + 16 * d + v) * 64] = o[d][v];
        }
        __syncthreads();
        if (hf == 1) return;
        const float m1 = mg[0], m = fmaxf(m_run, m1), m_exp = m == -INFINITY ? 0.0f : m;
        const float f0 = exp_approx(m_run - m_exp), f1 = exp_approx(m1 - m_exp);
        l = l * f0 + mg[64] * f1;
#pragma unroll
        for (int d = 0; d < OT; d++)
#pragma unroll
            for (int v = 0; v < 16; v++) o[d][v] = o[d][v] * f0 + mg[(2 + 16 * d + v) * 64] * f1;
    }

    // ---- out[row] = O / (sum of the row's exponentials): lane (half, col) holds
    // dims 8 a + 4 half + (0..3) of both 32-dim halves of query row col
    const int row = r0 + col;
    if (row >= a.rows) return;
    float* op = a.out + (static_cast<size_t>(s) * a.rows + row) * a.out_ld + h * kHd + half * 4;
#pragma unroll
    for (int d = 0; d < OT; d++)
#pragma unroll
        for (int a4 = 0; a4 < 4; a4++)
            *reinterpret_cast<float4*>(op + 32 * d + 8 * a4) =
                make_float4(o[d][4 * a4] / l, o[d][4 * a4 + 1] / l, o[d][4 * a4 + 2] / l, o[d][4 * a4 + 3] / l);
}

// e^x for x <= 0 as 2^(x log2 e), the product's rounding carried along: about 1 ulp.
__device__ __forceinline__ float exp_f32(float x) {
    x = x < -120.0f ? -120.0f : x;  // (NaN stays; 2^-173 is 0)
    const float t = x * 1.44269504088896341f;
    const float r = fmaf(x, 1.92596299e-8f, fmaf(x, 1.44269504088896341f, -t));
    const float e = __builtin_amdgcn_exp2f(t);
    return fmaf(e * r, 0.693147180559945f, e);
}

// Head width 32, on the fp32 matrix cores: the same walk, every operand as it is.
// S^T = K Q^T and O^T += V^T P^T are 16 v_mfma_f32_32x32x2_f32 each per 32-key tile (a
// step takes one dim of either half of the width, or one key of either half of the
// wave, as A and B).  The v tile is staged as it lies.  Sums in short chains, a
// tile's own products before the running sum: error against float64 over 17 shapes
// 8.4e-8, 1.19e-7 at most (the vector-unit kernel 8.8e-8 and 1.24e-7; two f16 terms per
// operand 1.27e-7 and 2.4e-7, and 3.2e-6 with v a hundredth as large, whose terms hold
// 2^-25 and no less).
// A tile with inf or NaN in v takes only the attended keys, on the vector units: 0 *
// inf would turn a masked key's v into NaN.
// Bound: the matrix cores, 32 products of 64 cycles per tile (busy 47 % of the time over
// 32 prompts of 500 rows), and some 410 vector instructions beside them.  us, d = 1024 and 32 heads: 16 prompts of 128 rows 19.3, 32
// of 500 rows 251 (vector units, one sequence at a time: 350, 10069); d = 128 with 4
// heads, 32 of 64 rows: 7.1 (182).
template <int HALVES>
__global__ void __launch_bounds__(kPT* HALVES, 2) k_attn_prefill_f32(PrefillArgs a) {
    constexpr int W = 32, kKP = W + 4, kVP = W + 8;  // pitches: 16-byte pieces of 16 keys, and two keys 4 apart, on different banks
    struct Stage {
        __align__(16) float k[2][kKeys * kKP], v[2][kKeys * kVP];
        int unsafe[3];  // a tile's v is not all finite (step st: st % 3)
    };
    __shared__ Stage stages[HALVES];
    static_assert(HALVES == 1 || sizeof(Stage) >= kRT * 18 * 64 * sizeof(float), "the merge fits a stage");
    const int hf = HALVES == 1 ? 0 : __builtin_amdgcn_readfirstlane(static_cast<int>(threadIdx.x) / kPT);
    Stage& sm = stages[hf];
    const int tid = threadIdx.x % kPT, lane = tid & 63, half = lane >> 5, col = lane & 31;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int groups = static_cast<int>(gridDim.z), g = groups - 1 - static_cast<int>(blockIdx.z);
    const int h = blockIdx.x, s = blockIdx.y;
    const int r0 = g * kQRows + wave * 32;
    const int kmax = a.pos0 + min(a.rows - 1, g * kQRows + kQRows - 1);
    const int ntiles = kmax / kKeys + 1;
    const int my_tiles = r0 < a.rows ? (a.pos0 + min(a.rows - 1, r0 + 31)) / kKeys + 1 : 0;
    const size_t sbase = static_cast<size_t>(s) * a.seq_stride + static_cast<size_t>(h) * W;
    float* kc = a.kc + sbase;
    float* vc = a.vc + sbase;
    const float* bq = a.qkv + static_cast<size_t>(s) * a.rows * a.ld + h * W;  // this sequence's block rows

    // this lane's query, dims 16 half + (0..15): step i of a score is dims i and 16 + i
    float q[16];
    {
        const float* qp = bq + static_cast<size_t>(min(r0 + col, a.rows - 1)) * a.ld + half * 16;
#pragma unroll
        for (int i = 0; i < 4; i++) {
            const float4 u = *reinterpret_cast<const float4*>(qp + 4 * i);
            q[4 * i] = u.x; q[4 * i + 1] = u.y; q[4 * i + 2] = u.z; q[4 * i + 3] = u.w;
        }
    }
    const int qpos = a.pos0 + r0 + col;

    // Staging: thread t takes 16 bytes of k and of v of key t / 8.  The last row group's
    // workgroup of each (sequence, head) also writes the block's rows into the caches.
    const bool writer = g == groups - 1;
    const int key_of = tid / 8, c0 = tid % 8 * 4;
    float4 pk, pv;
    auto fetch = [&](int t) __attribute__((always_inline)) {
        const int key = min(t * kKeys + key_of, kmax);
        const bool own = key >= a.pos0;
        const float* row = bq + static_cast<size_t>(max(key - a.pos0, 0)) * a.ld + c0;
        const size_t at = static_cast<size_t>(key) * a.kv_dim + c0;
        pk = *reinterpret_cast<const float4*>(own ? row + a.kv_dim : kc + at);
        pv = *reinterpret_cast<const float4*>(own ? row + 2 * a.kv_dim : vc + at);
    };
    auto store_block_rows = [&](int t) __attribute__((always_inline)) {
        const int key = t * kKeys + key_of;
        if (key < a.pos0 || key > kmax) return;
        const size_t at = static_cast<size_t>(key) * a.kv_dim + c0;
        *reinterpret_cast<float4*>(kc + at) = pk;
        *reinterpret_cast<float4*>(vc + at) = pv;
    };
    auto stash = [&](int st) __attribute__((always_inline)) {
        *reinterpret_cast<float4*>(&sm.k[st & 1][key_of * kKP + c0]) = pk;
        *reinterpret_cast<float4*>(&sm.v[st & 1][key_of * kVP + c0]) = pv;
        const bool finite = __builtin_isfinite(pv.x) && __builtin_isfinite(pv.y) && __builtin_isfinite(pv.z) &&
                            __builtin_isfinite(pv.w);
        if (__builtin_expect(!finite, 0)) sm.unsafe[st % 3] = 1;
    };

    float m_run = -INFINITY, l_run = 0.0f;
    f32x16 o = f32x16{};
    const int steps = (ntiles + HALVES - 1) / HALVES;
    if (tid < 3) sm.unsafe[tid] = 0;
    fetch(hf);
    if (writer) store_block_rows(hf);
    __syncthreads();
    stash(0);
    __syncthreads();
    for (int st = 0; st < steps; st++) {
        const int t = st * HALVES + hf, tn = t + HALVES, k0 = t * kKeys;
        if (tn < ntiles) fetch(tn);
        const bool vbad = sm.unsafe[st % 3] != 0;
        if (tid == 0) sm.unsafe[(st + 2) % 3] = 0;  // (read at step st - 1, written next at step st + 1)
        if (t < my_tiles) {
            const float* kt = sm.k[st & 1] + col * kKP + half * 16;
            const float* vt = sm.v[st & 1];
            f32x16 sacc[2] = {f32x16{}, f32x16{}};  // (two chains: fewer roundings in a row)
#pragma unroll
            for (int i = 0; i < 4; i++) {
                const float4 u = *reinterpret_cast<const float4*>(kt + 4 * i);
                sacc[0] = __builtin_amdgcn_mfma_f32_32x32x2f32(u.x, q[4 * i], sacc[0], 0, 0, 0);
                sacc[1] = __builtin_amdgcn_mfma_f32_32x32x2f32(u.y, q[4 * i + 1], sacc[1], 0, 0, 0);
                sacc[0] = __builtin_amdgcn_mfma_f32_32x32x2f32(u.z, q[4 * i + 2], sacc[0], 0, 0, 0);
                sacc[1] = __builtin_amdgcn_mfma_f32_32x32x2f32(u.w, q[4 * i + 3], sacc[1], 0, 0, 0);
            }
            float sv[16], mt = -INFINITY;
#pragma unroll
            for (int v = 0; v < 16; v++) sv[v] = (sacc[0][v] + sacc[1][v]) * a.scale;
            if (k0 + kKeys - 1 > a.pos0 + r0)
#pragma unroll
                for (int v = 0; v < 16; v++) sv[v] = k0 + acc_row(v, half) <= qpos ? sv[v] : -INFINITY;
#pragma unroll
            for (int v = 0; v < 16; v++) mt = fmaxf(mt, sv[v]);
            // (a query whose scores so far are all -inf keeps sums of 0, and 0 / 0 = NaN)
            const float m_new = fmaxf(m_run, max_halves(mt)), m_exp = m_new == -INFINITY ? 0.0f : m_new;
            const float corr = exp_f32(m_run - m_exp);  // 0 on the first tile (m_run = -inf)
            float ps[4] = {};
#pragma unroll
            for (int v = 0; v < 16; v++) {
                sv[v] = exp_f32(sv[v] - m_exp);
                ps[v & 3] += sv[v];
            }
            // (this half's keys; the halves are added at the end)
            l_run = fmaf(l_run, corr, (ps[0] + ps[1]) + (ps[2] + ps[3]));
            m_run = m_new;
            if (!vbad) {
                // (the tile's own sum first: a running sum of all keys' products would
                // round once per key instead of once per tile)
                f32x16 first;
#pragma unroll
                for (int v0 = 0; v0 < 16; v0 += 8) {
                    f32x16 ot[2] = {f32x16{}, f32x16{}};
#pragma unroll
                    for (int v = v0; v < v0 + 8; v++)
                        ot[v & 1] = __builtin_amdgcn_mfma_f32_32x32x2f32(vt[acc_row(v, half) * kVP + col], sv[v], ot[v & 1], 0, 0, 0);
                    if (v0 == 0) first = ot[0] + ot[1];
                    else
#pragma unroll
                        for (int d = 0; d < 16; d++) o[d] = fmaf(o[d], corr, first[d] + (ot[0][d] + ot[1][d]));
                }
            } else {
                o *= corr;
                // (keys past the query's position, or past the block's last one, are left out)
                const int last = min(qpos, kmax);
#pragma unroll
                for (int v = 0; v < 16; v++) {
                    const float other = __shfl_xor(sv[v], 32, 64);
#pragma unroll
                    for (int e = 0; e < 2; e++) {
                        const int key = acc_row(v, e);
                        const float p = e == half ? sv[v] : other;
                        if (k0 + key <= last)
#pragma unroll
                            for (int d = 0; d < 16; d++) o[d] += p * vt[key * kVP + acc_row(d, half)];
                    }
                }
            }
        }
        if (tn < ntiles) {
            if (writer) store_block_rows(tn);
            stash(st + 1);
        }
        __syncthreads();
    }
    float l = l_run + __shfl_xor(l_run, 32, 64);
    if constexpr (HALVES == 2) {
        // the odd tiles' maximum, sum and outputs, scaled to the common maximum
        float* mg = reinterpret_cast<float*>(&stages[1]) + wave * (18 * 64) + lane;
        if (hf == 1) {
            mg[0] = m_run;
            mg[64] = l;
#pragma unroll
            for (int v = 0; v < 16; v++) mg[(2 + v) * 64] = o[v];
        }
        __syncthreads();
        if (hf == 1) return;
        const float m1 = mg[0], m = fmaxf(m_run, m1), m_exp = m == -INFINITY ? 0.0f : m;
        const float f0 = exp_f32(m_run - m_exp), f1 = exp_f32(m1 - m_exp);
        l = l * f0 + mg[64] * f1;
#pragma unroll
        for (int v = 0; v < 16; v++) o[v] = o[v] * f0 + mg[(2 + v) * 64] * f1;
    }
    const int row = r0 + col;
    if (row >= a.rows) return;
    float* op = a.out + (static_cast<size_t>(s) * a.rows + row) * a.out_ld + h * W + half * 4;
#pragma unroll
    for (int a4 = 0; a4 < 4; a4++)
        *reinterpret_cast<float4*>(op + 8 * a4) =
            make_float4(o[4 * a4] / l, o[4 * a4 + 1] / l, o[4 * a4 + 2] / l, o[4 * a4 + 3] / l);
}

bool aligned16(const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15u) == 0; }

// Head width 32: whether the vector-unit kernel, two launches per sequence, should take
// less than the matrix cores' `ns`, as it does for one or a few sequences with many
// earlier positions, whose key tiles are one workgroup's chain: one row after 700, 4
// heads 7.9 us against 38, 128 rows 18.2 / 47; four of them 70.5 / 48.  A sequence takes
// 6.2 us, or 5.7 and 2.7 ns per workgroup with keys to attend (one for each row, head
// and 64 positions, 128 from 769 on), or so much per workgroup launched where the
// chunks of a row are a multiple of 4 or 8, which deals the later, often empty ones to
// the same XCDs.  It keeps partial sums in the context's areas, so a call under graph
// capture that they do not hold stays on the matrix cores.
bool few_sequences(fh_ctx* ctx, size_t heads, size_t pos0, size_t rows, size_t seqs, size_t ns) {
    const size_t len = pos0 + rows, keys = len > 768 ? 128 : len > 32 ? 64 : 32, chunks = (len + keys - 1) / keys;
    const size_t busy = heads * rows * (2 * pos0 + rows + keys) / (2 * keys) * (chunks == 1 ? 100 : 270) / 100;
    const size_t all = heads * rows * chunks * (chunks % 8 == 0 ? 300 : chunks % 4 == 0 ? 215 : 0) / 100;
    const size_t work = 5700 + (busy > all ? busy : all);
    if (1500 + seqs * (work > 6200 ? work : 6200) >= ns) return false;
    if (ctx->ws_bytes >= heads * rows * chunks * 34 * sizeof(float) && ctx->counters_bytes >= heads * rows * sizeof(unsigned))
        return true;
    hipStreamCaptureStatus cs = hipStreamCaptureStatusNone;
    return hipStreamIsCapturing(ctx->stream, &cs) == hipSuccess && cs == hipStreamCaptureStatusNone;
}

}  // namespace

int fh_launch_attention_prefill_seqs(fh_ctx* ctx, const float* qkv, float* kc, float* vc, size_t seq_stride,
                                     size_t d, size_t heads, size_t pos0, size_t rows, size_t seqs, float* out) {
    const size_t hd = d / heads;
    const bool mfma = (hd == 32 || hd == static_cast<size_t>(kHd)) && aligned16(qkv) && aligned16(kc) && aligned16(vc) &&
                      aligned16(out) && seq_stride % 4 == 0;
    // (one sequence at a time)
    auto on_vector_units = [&]() -> int {
        for (size_t s = 0; s < seqs; s++) {
            const int rc = fh_launch_attention_prefill(ctx, qkv + s * rows * 3 * d, kc + s * seq_stride,
                                                       vc + s * seq_stride, d, heads, pos0, rows, out + s * rows * d);
            if (rc) return rc;
        }
        return FH_OK;
    };
    if (!mfma) return on_vector_units();  // other head widths
    PrefillArgs a{};
    a.qkv = qkv;
    a.ld = static_cast<int>(3 * d);
    a.kc = kc;
    a.vc = vc;
    a.seq_stride = seq_stride;
    a.kv_dim = static_cast<int>(d);
    a.rows = static_cast<int>(rows);
    a.pos0 = static_cast<int>(pos0);
    a.scale = 1.0f / sqrtf(static_cast<float>(hd));
    a.out = out;
    a.out_ld = static_cast<int>(d);
    const size_t cus = static_cast<size_t>(ctx->num_cus), pairs = heads * seqs, groups = (rows + kQRows - 1) / kQRows;
    // One or two chains of key tiles per row.  Measured (ns) at head width 64: a
    // workgroup takes 2200 per tile alone on its CU, a CU of two 1750 per tile;
    // with two chains 1500 alone (one workgroup per CU) and 2300, and 1500 for the
    // merge.  8 sequences of 300 rows and 12 heads (288 workgroups of 4, 8 and 10
    // tiles): 25.2 us and 22.5; 16 heads: 25.7 and 27.5; one of 511 rows: 33.4 and
    // 25.6; 32 of 511: 106.8 and 131.4.  At width 32 1950 and 1550, 1600 and 1950: one
    // sequence of 900 rows 60.0 us and 52.7, 32 of 500 rows and 32 heads 251 and 317.
    const size_t tile1 = hd == 32 ? 1950 : 2200, tile2 = hd == 32 ? 1550 : 1750;
    const size_t half1 = hd == 32 ? 1600 : 1500, half2 = hd == 32 ? 1950 : 2300;
    size_t tiles = 0;
    for (size_t g = 1; g <= groups; g++) tiles += (pos0 + (g * kQRows < rows ? g * kQRows : rows) - 1) / kKeys + 1;
    const size_t longest = (pos0 + rows - 1) / kKeys + 1, share = tiles * pairs / cus;
    const size_t one = longest * tile1 > share * tile2 ? longest * tile1 : share * tile2;
    const size_t two = (longest * half1 > share * half2 ? longest * half1 : share * half2) + 1500;
    if (hd == 32 && few_sequences(ctx, heads, pos0, rows, seqs, 3300 + (one < two ? one : two)))
        return on_vector_units();
    auto go = [&](auto kern, int halves) {
        // (at most 65535 sequences and 512 groups of rows: the callers' limits)
        hipLaunchKernelGGL(kern, dim3(static_cast<unsigned>(heads), static_cast<unsigned>(seqs), static_cast<unsigned>(groups)),
                           dim3(static_cast<unsigned>(kPT * halves)), 0, ctx->stream, a);
    };
    if (hd == 32) two < one ? go(k_attn_prefill_f32<2>, 2) : go(k_attn_prefill_f32<1>, 1);
    else two < one ? go(k_attn_prefill_f16<2>, 2) : go(k_attn_prefill_f16<1>, 1);
    FH_HIP(ctx, hipGetLastError());
    return FH_OK;
}
