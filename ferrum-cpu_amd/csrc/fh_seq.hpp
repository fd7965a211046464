// fh_seq.hpp — linears whose every output is one sequential sum.
//
//   y[i, j] = s0 + a[i, 0] * w[0, j] + a[i, 1] * w[1, j] + ...
//
// in ascending p, each product and each add rounded (no FMA): the exact
// Q8_0 / F32 linear (fh_exact.hip) and the packed per-row linear
// (fh_qlinear.hip).  K cannot be split, so an output is a chain of K dependent
// adds and the parallelism is outputs.
//
// Bound: the vector units.  An output costs one multiply and one add per p, a
// wave issues an instruction every four cycles or so, and nothing else on the
// chip can do the rounded product and the rounded add.  So everything else is
// kept off the vector units:
//  - a wave is 64 / C rows (times TM per lane) by C columns, and the four waves
//    of a workgroup are 256 / C * TM rows of the same C columns, so a weight is
//    fetched and widened (once, into LDS) for that many rows;
//  - a lane's activation register holds 16 consecutive p of its row, one per
//    lane of its 16-lane row, and the multiply itself takes its operand from
//    lane p % 16 (DPP row_newbcast): no LDS read, no move, no scalar load;
//  - LDS holds the widened weights as float4 of four consecutive p per column:
//    one read serves four steps of a lane's chains;
//  - adds and multiplies alternate, the product four steps ahead of its add, so
//    a dependent add always has an independent multiply in front of it.
// A chunk is 128 positions, double-buffered; the next chunk's activations and
// the weights two chunks on are in flight while the current one is summed.
//
// Measured (us per call; before: one row of x per workgroup and the products
// through LDS for the exact linear, four rows with a byte read and a conversion
// per product for the packed one): exact 768 x 3072 at m = 127 190.8 -> 34.0, 2304 x 768 at m = 256 320 -> 32.7; int4 2304 x 768 at
// m = 127 38.2 -> 23.7, int8 4096 x 1024 at m = 512 247 -> 142.  At m = 512 that is
// 81 % of the rate at which the vector units issue the multiplies and adds; at
// 768 x 3072 and m = 127, where 1524 wave-wide chains meet 1024 SIMDs (two on
// some, 23.5 us of adds and multiplies), the rest is waiting: 5 us for the
// weights' way into LDS, 4 for the LDS reads.
//
// Positions past K are given a = -0 and w = +0: their product is -0, and adding
// -0 changes no value (-0 and +0 included).  The products queued before the
// first add are -0 likewise.
#pragma once

#include <type_traits>
#include <utility>

#include "fh_internal.hpp"

#pragma clang fp contract(off)

namespace fh_seq {

constexpr int kThreads = 256, kWaves = kThreads / 64;
constexpr int kChunk = 128;          // positions per chunk
constexpr int kGroups = kChunk / 4;  // float4 groups per column and chunk
constexpr int kPieces = kChunk / 16; // activation registers per row and chunk
constexpr int kQueue = 4;            // products in flight per chain

// Chunks of K.  (K goes up to 2^31 - 1: rounding it up first would overflow, and the
// position after the last chunk is 2^31, so positions are compared unsigned.)
__host__ __device__ constexpr int chunks_of(int k) { return (k - 1) / kChunk + 1; }
static_assert(chunks_of(1) == 1 && chunks_of(kChunk) == 1 && chunks_of(kChunk + 1) == 2 &&
                  chunks_of(0x7FFFFFFF) == (1 << 24) && chunks_of(0x7FFFFFE0) == (1 << 24),
              "the last chunk of the longest K starts inside it");
__device__ __forceinline__ bool inside(int chunk, int p, int k) {
    return static_cast<unsigned>(chunk) * kChunk + static_cast<unsigned>(p) < static_cast<unsigned>(k);
}

typedef float f4 __attribute__((ext_vector_type(4)));

// Lane N's value of each 16-lane row.
template <int N>
__device__ __forceinline__ float row_lane(float v) {
    return __builtin_bit_cast(float, __builtin_amdgcn_mov_dpp(__builtin_bit_cast(int, v), 0x150 + N, 0xF, 0xF, true));
}

// One position of TM chains: add the product of four positions ago, queue this
// one's.
template <int L, int TM>
__device__ __forceinline__ void step(float w, const float (&a)[TM], float (&q)[TM][kQueue], float (&acc)[TM]) {
#pragma unroll
    for (int r = 0; r < TM; r++) {
        acc[r] = acc[r] + q[r][L % kQueue];
        q[r][L % kQueue] = row_lane<L>(a[r]) * w;
    }
    __builtin_amdgcn_sched_barrier(0);
}

template <int G, int TM>
__device__ __forceinline__ void steps(f4 w, const float (&a)[TM], float (&q)[TM][kQueue], float (&acc)[TM]) {
    step<4 * G, TM>(w.x, a, q, acc);
    step<4 * G + 1, TM>(w.y, a, q, acc);
    step<4 * G + 2, TM>(w.z, a, q, acc);
    step<4 * G + 3, TM>(w.w, a, q, acc);
}

// Src (a kernel argument) says where the weights are and how they widen:
//   C                        columns per workgroup (16 or 32)
//   kBiasFirst               the bias starts the sum (else it is added last)
//   Raw                      a thread's raw weights of one chunk
//   load(tid, tile, c, n, k, Raw&)            issue their loads (c < chunks)
//   store(tid, c, k, const Raw&, f4* wt)  widen them into wt[kGroups][C]
//   kScaled, scale(p)        a factor of a[., p], rounded into it
//   column(tile, lane, n)    a lane's output column, or -1
template <class Src, int TM>
__global__ void __launch_bounds__(kThreads)
    k_linear_seq(Src src, const float* __restrict__ x, const float* __restrict__ bias, float* __restrict__ y, int m,
                 int n, int k, int tiles) {
    constexpr int C = Src::C, kWaveRows = 64 / C * TM, kTileRows = kWaves * kWaveRows;
    static_assert(C == 16 || C == 32, "a 16-lane row holds one row of x");
    __shared__ f4 wt[2][kGroups * C];
    const int tid = threadIdx.x, lane = tid & 63, l16 = tid & 15;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    // neighbouring tiles on one XCD (workgroups are dealt to the eight in turn):
    // where rows are [p][n], they read the same lines
    const int tile = blockIdx.z * gridDim.x + (blockIdx.x & 7) * (gridDim.x >> 3) + (blockIdx.x >> 3);
    if (tile >= tiles) return;
    const int chunks = chunks_of(k);
    const int col = src.column(tile, lane % C, n);
    const float b0 = bias && col >= 0 ? bias[col] : 0.0f;
    for (long i0 = static_cast<long>(blockIdx.y) * kTileRows; i0 < m; i0 += static_cast<long>(gridDim.y) * kTileRows) {
        const bool live = i0 + wave * kWaveRows < m;  // wave-uniform: a wave without rows only widens weights
        const long row = i0 + wave * kWaveRows + lane / C * TM;  // this lane's rows: row .. row + TM - 1
        const float* xr[TM];
#pragma unroll
        for (int r = 0; r < TM; r++) xr[r] = x + (row + r < m ? row + r : m - 1) * static_cast<long>(k) + l16;
        float acc[TM], q[TM][kQueue], a[2][kPieces][TM], sn[kPieces];
        typename Src::Raw raw[2];
        // Loads past the last chunk are of the last one, and are not used.
        auto load_w = [&](auto S, int c) __attribute__((always_inline)) {
            src.load(tid, tile, min(c, chunks - 1), n, k, raw[S]);
        };
        auto load_x = [&](auto S, int c) __attribute__((always_inline)) {
            if (!live) return;
            const int p0 = min(c, chunks - 1) * kChunk;
            if (p0 <= k - kChunk) {
#pragma unroll
                for (int s = 0; s < kPieces; s++) {
                    if constexpr (Src::kScaled) sn[s] = src.scale(p0 + 16 * s + l16);
#pragma unroll
                    for (int r = 0; r < TM; r++) a[S][s][r] = xr[r][p0 + 16 * s];
                }
            } else {
#pragma unroll
                for (int s = 0; s < kPieces; s++) {
                    const int p = min(p0 + 16 * s + l16, k - 1);
                    if constexpr (Src::kScaled) sn[s] = src.scale(p);
#pragma unroll
                    for (int r = 0; r < TM; r++) a[S][s][r] = xr[r][p - l16];
                }
            }
        };
        // chunk c's activations as the chains take them
        auto take_x = [&](auto S, int c) __attribute__((always_inline)) {
            if (!live) return;
            if constexpr (Src::kScaled) {
#pragma unroll
                for (int s = 0; s < kPieces; s++)
#pragma unroll
                    for (int r = 0; r < TM; r++) a[S][s][r] = a[S][s][r] * sn[s];
            }
            if (!inside(c, kChunk - 1, k)) {
#pragma unroll
                for (int s = 0; s < kPieces; s++)
#pragma unroll
                    for (int r = 0; r < TM; r++) a[S][s][r] = inside(c, 16 * s + l16, k) ? a[S][s][r] : -0.0f;
            }
        };
        auto sum = [&](auto S) __attribute__((always_inline)) {
            if (!live) return;
            const f4* wl = wt[S] + lane % C;
            f4 w[3][4];  // 16 positions each: two sets are being read while one is summed
            auto read = [&](int s) __attribute__((always_inline)) {
#pragma unroll
                for (int g = 0; g < 4; g++) w[s % 3][g] = wl[(4 * s + g) * C];
            };
            read(0);
            read(1);
#pragma unroll
            for (int s = 0; s < kPieces; s++) {
                if (s + 2 < kPieces) read(s + 2);
                __builtin_amdgcn_sched_barrier(0);
                // (an opaque copy keeps each lane read next to its multiply,
                // which then takes it as its DPP operand)
#pragma unroll
                for (int r = 0; r < TM; r++) asm volatile("" : "+v"(a[S][s][r]));
                // (one wait for the four reads)
                asm volatile("" : "+v"(w[s % 3][0]), "+v"(w[s % 3][1]), "+v"(w[s % 3][2]), "+v"(w[s % 3][3]));
                __builtin_amdgcn_sched_barrier(0);
                steps<0, TM>(w[s % 3][0], a[S][s], q, acc);
                steps<1, TM>(w[s % 3][1], a[S][s], q, acc);
                steps<2, TM>(w[s % 3][2], a[S][s], q, acc);
                steps<3, TM>(w[s % 3][3], a[S][s], q, acc);
            }
#pragma unroll
            for (int r = 0; r < TM; r++) asm volatile("" : "+v"(acc[r]));
        };
        const std::integral_constant<int, 0> even;
        const std::integral_constant<int, 1> odd;
#pragma unroll
        for (int r = 0; r < TM; r++) {
            acc[r] = Src::kBiasFirst ? b0 : 0.0f;
#pragma unroll
            for (int e = 0; e < kQueue; e++) q[r][e] = -0.0f;
        }
        // Chunk c: its successor's weights go to LDS (the other buffer's last
        // reader finished before the previous barrier), the loads of the next
        // activations and of the weights after those go out (in this order, so
        // that waiting for the activations leaves the weights outstanding),
        // and its own chains run.
        auto chunk = [&](auto S, int c) __attribute__((always_inline)) {
            const std::integral_constant<int, 1 - S> T;
            src.store(tid, c + 1, k, raw[T], wt[T]);
            load_x(T, c + 1);
            load_w(T, c + 3);
            sum(S);
            take_x(T, c + 1);
            __syncthreads();
        };
        load_w(even, 0);
        load_w(odd, 1);
        load_x(even, 0);
        src.store(tid, 0, k, raw[0], wt[0]);
        load_w(even, 2);
        take_x(even, 0);
        __syncthreads();
        for (int c = 0; c < chunks; c += 2) {
            chunk(even, c);
            if (c + 1 < chunks) chunk(odd, c + 1);
        }
        if (live && col >= 0) {
#pragma unroll
            for (int r = 0; r < TM; r++)
                if (row + r < m) {
                    float v = acc[r];
#pragma unroll
                    for (int e = 0; e < kQueue; e++) v = v + q[r][e];
                    y[(row + r) * static_cast<long>(n) + col] = Src::kBiasFirst || !bias ? v : v + b0;
                }
        }
    }
}

// Few enough outputs that every workgroup has a CU's adders to itself (one row of
// x, decode): the time is K times one step of the chain, so the summing wave
// (wave 0) does nothing but the adds, and waves 1-3 form the rounded products of
// the next chunk into LDS, as float4 of four consecutive p per column.  A
// producer's job is 16 positions of one column: its four 16-byte writes land
// beside its 15 neighbours', and the summing wave reads them the same way, both
// free of bank conflicts.
//
// JOBS, the jobs per producer and chunk: with two the chunk is 384 positions (48 KB
// of LDS, three workgroups per CU), long enough that the barrier, the first read
// and the producers' load latency are a small part of it; one (24 KB, six per CU)
// is for outputs that fill the chip many times over, where the neighbours cover
// those waits.
//
// Measured against k_linear_seq, us per call at m = 1: 768 x 3072 21.3 -> 11.8 (one
// job: 17.3, four: 12.5; the adds alone are 7.4), 3072 x 768 7.1 -> 4.9, 1024 x 4096
// 27.4 -> 15.0; with one job 50257 x 768 28.5 -> 19.4 (two: 22.1), 151936 x 896
// 79.7 -> 52.7 (66.4).
//
// Src, beside what k_linear_seq asks for (C = 16, no factor, bias last):
//   Row, load_row(column, p, k, Row&)   the raw weights of positions p .. p + 15
//   quad(Row, v)                        positions p + 4 v .. + 3 widened
// Positions past K are loaded from inside the row and never summed.
template <class Src, int JOBS>
__global__ void __launch_bounds__(kThreads)
    k_linear_seq_row(Src src, const float* __restrict__ x, const float* __restrict__ bias, float* __restrict__ y,
                     int n, int k) {
    constexpr int C = Src::C, kSegs = (kWaves - 1) * 4, kRowChunk = kSegs * 16 * JOBS, kRowGroups = kRowChunk / 4;
    static_assert(C == 16 && !Src::kBiasFirst && !Src::kScaled, "the plain sum of 16 columns");
    __shared__ f4 prod[2][kRowGroups * C];
    const int tid = threadIdx.x, lane = tid & 63, c16 = tid & 15, tile = blockIdx.z * gridDim.x + blockIdx.x;
    if (tile > (n - 1) / C) return;
    const int chunks = (k + kRowChunk - 1) / kRowChunk;
    const float* xr = x + static_cast<size_t>(blockIdx.y) * k;
    // wave-uniform role (a scalar branch: every wave meets the same barriers)
    if (__builtin_amdgcn_readfirstlane(tid >> 6) == 0) {
        const int col = src.column(tile, c16, n);
        const float b0 = bias && col >= 0 ? bias[col] : 0.0f;
        float acc = 0.0f;
        __syncthreads();  // chunk 0 is in LDS
        for (int c = 0; c < chunks; c++) {
            const f4* pb = prod[c & 1] + c16;
            const int pn = min(kRowChunk, k - c * kRowChunk);
            if (pn == kRowChunk) {
#pragma unroll 32
                for (int g = 0; g < kRowGroups; g++) {
                    const f4 v = pb[g * C];
                    acc = (((acc + v.x) + v.y) + v.z) + v.w;
                }
            } else {
                const int gn = pn >> 2, rest = pn & 3;
#pragma unroll 8
                for (int g = 0; g < gn; g++) {
                    const f4 v = pb[g * C];
                    acc = (((acc + v.x) + v.y) + v.z) + v.w;
                }
                if (rest) {
                    const f4 v = pb[gn * C];
                    acc = acc + v.x;
                    if (rest > 1) acc = acc + v.y;
                    if (rest > 2) acc = acc + v.z;
                }
            }
            __syncthreads();  // chunk c + 1 is in LDS; buffer c & 1 is free
        }
        if (lane < C && col >= 0) y[blockIdx.y * static_cast<size_t>(n) + col] = bias ? acc + b0 : acc;
        return;
    }
    // The producers: column c16 of the tile, 16-position segments seg + kSegs * i.
    const int seg = (tid - 64) >> 4, j = min(tile * C + c16, n - 1);
    typename Src::Row w[2][JOBS];
    float a[2][JOBS][16];
    auto fetch = [&](auto S, int c) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < JOBS; i++) {
            const int p = c * kRowChunk + 16 * (seg + kSegs * i);
            src.load_row(j, p, k, w[S][i]);
            if (p + 16 <= k) {
#pragma unroll
                for (int e = 0; e < 16; e++) a[S][i][e] = xr[p + e];
            } else {
#pragma unroll
                for (int e = 0; e < 16; e++) a[S][i][e] = xr[min(p + e, k - 1)];
            }
        }
    };
    auto produce = [&](auto S, int b) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < JOBS; i++)
#pragma unroll
            for (int v = 0; v < 4; v++) {
                const f4 q = src.quad(w[S][i], v);
                prod[b][(4 * (seg + kSegs * i) + v) * C + c16] =
                    f4{a[S][i][4 * v] * q.x, a[S][i][4 * v + 1] * q.y, a[S][i][4 * v + 2] * q.z,
                       a[S][i][4 * v + 3] * q.w};
            }
    };
    const std::integral_constant<int, 0> s0;
    const std::integral_constant<int, 1> s1;
    fetch(s0, 0);
    if (chunks > 1) fetch(s1, 1);
    produce(s0, 0);
    __syncthreads();
    // Step c: set c & 1 held chunk c (its products are in LDS), so it takes
    // chunk c + 2; chunk c + 1's products go to buffer (c + 1) & 1.
    auto step = [&](auto S, int c) __attribute__((always_inline)) {
        if (c + 2 < chunks) fetch(S, c + 2);
        if (c + 1 < chunks) produce(std::integral_constant<int, 1 - S>{}, (c + 1) & 1);
        __syncthreads();
    };
    for (int c = 0; c < chunks; c += 2) {
        step(s0, c);
        if (c + 1 < chunks) step(s1, c + 1);
    }
}

// TM, the rows per lane: more of them share a widened weight and a read of it,
// but make fewer workgroups.  The cost of a round of one workgroup per CU is
// about TM + 0.15, and two workgroups per CU are needed to cover one another's
// waits: int4 4096 x 1024 at m = 127 runs 45.3 / 43.1 / 39.4 us with TM = 1 / 2 /
// 4 (8, 4 and 2 whole rounds), 768 x 3072 41.8 / 41.7 / 67.7 (384, 192 and 96
// workgroups).
// Column tiles as grid.x and grid.z: a multiple of eight in x, and no more than HIP's
// 2^32 threads in that dimension.
inline dim3 tile_grid(size_t tiles, size_t y) {
    const size_t most = size_t(1) << 23, x = tiles < most ? (tiles + 7) / 8 * 8 : most;
    return dim3(static_cast<unsigned>(x), static_cast<unsigned>(y), static_cast<unsigned>((tiles + x - 1) / x));
}
inline size_t row_tiles(size_t cols, size_t m, size_t tm) { return (m + kThreads / cols * tm - 1) / (kThreads / cols * tm); }
inline size_t rows_per_lane(size_t cus, size_t cols, size_t tiles, size_t m) {
    auto blocks = [&](size_t tm) { return tiles * row_tiles(cols, m, tm); };
    auto cost = [&](size_t tm) { return ((blocks(tm) + cus - 1) / cus) * (20 * tm + 3); };
    size_t tm = 1;
    for (size_t t = 2; t <= 4; t *= 2)
        if (blocks(t) >= 2 * cus && cost(t) < cost(tm)) tm = t;
    return tm;
}

template <class Src>
void launch(fh_ctx* ctx, const Src& src, size_t tiles, const float* x, size_t m, const float* bias, float* y, size_t n,
            size_t k) {
    const size_t tm = rows_per_lane(static_cast<size_t>(ctx->num_cus), Src::C, tiles, m);
    auto go = [&](auto kernel) {
        const size_t gy = row_tiles(Src::C, m, tm);
        hipLaunchKernelGGL(kernel, tile_grid(tiles, gy < 65535 ? gy : 65535), dim3(kThreads), 0, ctx->stream, src, x, bias, y, static_cast<int>(m), static_cast<int>(n),
                           static_cast<int>(k), static_cast<int>(tiles));
    };
    if (tm == 4) go(k_linear_seq<Src, 4>);
    else if (tm == 2) go(k_linear_seq<Src, 2>);
    else go(k_linear_seq<Src, 1>);
}

}  // namespace fh_seq
