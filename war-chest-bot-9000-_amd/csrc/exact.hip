// The float32 leaf network's products in the CPU net's order.
//
// Every output is one running float32 sum over ascending inputs, a rounded
// product and a rounded addition per step (the library is built with
// -ffp-contract=off), so the result is the CPU loop's bit for bit; that rules
// out the matrix cores, whose steps round once, and splitting a sum. What is
// free is which thread takes which outputs: a workgroup takes a tile of rows x
// columns, stages 16-byte runs of both operands along the inputs in LDS, and
// each thread keeps TM x TN independent sums in registers.
//
// Bound: two VALU operations per product (about 19.7e12 products per second
// over 256 CUs without packed or fused arithmetic). A 384 -> 384 layer of 3,915
// rows takes 38 us with 64 x 32 tiles (16.9e12 products per second over a wave's
// three layers), 41 us with 32 x 32 and 319 us with one output per thread and
// its operands read through L1; the whole 512 -> 3x384 -> 567 net of 3,001 rows
// 142 us against 3,290.
#include "kernels.h"

#include <algorithm>

namespace wc {

namespace {

constexpr uint32_t THREADS = 256, SIDE = 16;  // a SIDE x SIDE grid of threads over the tile
// A larger tile reads less LDS per product but needs enough workgroups: the
// largest one with at least two per CU is taken. 3,001 rows (282 tiles of 64 x
// 64 for a 384-wide layer, 564 of 64 x 32): 142 us with 64 x 32 tiles, 148 with
// 32 x 32, 171 with 64 x 64; 8,000 rows (750 of 64 x 64): 206 us with 64 x 64
// tiles, 231 with 32 x 32. The smallest tile's k tile: 60 rows take 28.6 us
// with 128 inputs, 30.6 with 32, 33.5 with 256. Lines at 256 / 512 / 1,024 tiles
// over 100 to 8,000 rows (four runs within 2%): the same below 500 rows, then
// 512 in front (567 heads, 1,700 rows 106 / 91 / 114 us, 3,001 170 / 142 / 146)
// except near 5,600 rows (248 / 248 / 227).
constexpr uint64_t MIN_TILES = 512;

enum : uint32_t { VEC_X = 1, VEC_W = 2 };  // 16-byte loads of the operand are aligned

// Y[r, j] over X [M x K] and Wt [N x K]. HEAD: b[j] + sum_k, else
// relu(sum_k + b[j]). SKIP leaves out the terms whose x is zero, as the CPU
// loop does (engine/src/net.rs:102-122): with finite weights such a term adds
// a zero to a sum that is never -0 (it starts at +0), so only a bank holding
// an infinity or a NaN needs it. A row of the LDS tiles holds BK inputs and 4
// floats of padding: 16 rows' 16-byte runs then start in distinct banks.
// A thread's columns and rows lie SIDE apart, so a wavefront reads 16 column
// runs and 4 row runs per step, none in conflict.
template <int TM, int TN, int BK, bool HEAD, bool SKIP>
__global__ __launch_bounds__(THREADS) void k_exact(const float* __restrict__ X, uint32_t K,
                                                   const float* __restrict__ Wt, const float* __restrict__ bias,
                                                   uint32_t N, float* __restrict__ Y, uint32_t M, uint32_t vec,
                                                   const uint32_t* __restrict__ rb_n) {
    constexpr int BM = SIDE * TM, BN = SIDE * TN, LD = BK + 4, QK = BK / 4;  // QK 16-byte runs per tile row
    constexpr int RUNS = (BM + BN) * QK, PER = (RUNS + THREADS - 1) / THREADS;
    __shared__ __attribute__((aligned(16))) float lds[2][BM + BN][LD];
    const uint32_t t = threadIdx.x, m0 = blockIdx.x * BM, n0 = blockIdx.y * BN;
    if (rb_n) {  // block-uniform: no row of the tile needs these columns
        uint32_t need = 0;
        for (uint32_t r = m0; r < M && r < m0 + BM; r += SIDE) need = max(need, rb_n[r / SIDE]);
        if (n0 >= need) return;
    }
    // One run of the k tile at k0: rows past M or N and inputs past K read as zero.
    auto fetch = [&](int i, uint32_t k0) {
        float4 v = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
        const int s = (int)t + i * (int)THREADS;
        if (s >= RUNS) return v;
        const int row = s / QK;
        const uint32_t k = k0 + 4 * (s % QK);
        const bool x = row < BM;
        const uint32_t g = x ? m0 + row : n0 + row - BM;
        if (g >= (x ? M : N) || k >= K) return v;
        const float* p = (x ? X : Wt) + (size_t)g * K + k;
        if (vec & (x ? VEC_X : VEC_W)) return *(const float4*)p;  // (then K is a multiple of 4)
        v.x = p[0];
        if (k + 1 < K) v.y = p[1];
        if (k + 2 < K) v.z = p[2];
        if (k + 3 < K) v.w = p[3];
        return v;
    };
    auto store = [&](int buf, int i, const float4& v) {
        const int s = (int)t + i * (int)THREADS;
        if (s < RUNS) *(float4*)&lds[buf][s / QK][4 * (s % QK)] = v;
    };
    const uint32_t tx = t % SIDE, ty = t / SIDE;
    float acc[TM][TN];
#pragma unroll
    for (int j = 0; j < TN; j++) {
        const uint32_t n = n0 + tx + SIDE * j;
        const float b = HEAD && n < N ? bias[n] : 0.0f;
#pragma unroll
        for (int i = 0; i < TM; i++) acc[i][j] = b;
    }
    auto mac = [&](float& a, float x, float w) {
        if (SKIP)
            a = x != 0.0f ? a + x * w : a;
        else
            a += x * w;
    };
    float4 next[PER];
#pragma unroll
    for (int i = 0; i < PER; i++) store(0, i, fetch(i, 0));
    __syncthreads();
    int buf = 0;
    for (uint32_t k0 = 0; k0 < K; k0 += BK, buf ^= 1) {
        const bool more = k0 + BK < K;
        if (more) {
#pragma unroll
            for (int i = 0; i < PER; i++) next[i] = fetch(i, k0 + BK);
        }
        const uint32_t steps = min((uint32_t)BK, K - k0);
        auto four = [&](uint32_t k) {
            float4 x[TM], w[TN];
#pragma unroll
            for (int i = 0; i < TM; i++) x[i] = *(const float4*)&lds[buf][ty + SIDE * i][k];
#pragma unroll
            for (int j = 0; j < TN; j++) w[j] = *(const float4*)&lds[buf][BM + tx + SIDE * j][k];
#pragma unroll
            for (int i = 0; i < TM; i++)
#pragma unroll
                for (int j = 0; j < TN; j++) mac(acc[i][j], x[i].x, w[j].x);
#pragma unroll
            for (int i = 0; i < TM; i++)
#pragma unroll
                for (int j = 0; j < TN; j++) mac(acc[i][j], x[i].y, w[j].y);
#pragma unroll
            for (int i = 0; i < TM; i++)
#pragma unroll
                for (int j = 0; j < TN; j++) mac(acc[i][j], x[i].z, w[j].z);
#pragma unroll
            for (int i = 0; i < TM; i++)
#pragma unroll
                for (int j = 0; j < TN; j++) mac(acc[i][j], x[i].w, w[j].w);
        };
        if (steps == (uint32_t)BK) {
#pragma unroll 8
            for (uint32_t k = 0; k < (uint32_t)BK; k += 4) four(k);
        } else {  // the last tile of a K that is no multiple of BK
            uint32_t k = 0;
            for (; k + 4 <= steps; k += 4) four(k);
            for (; k < steps; k++)
#pragma unroll
                for (int i = 0; i < TM; i++)
#pragma unroll
                    for (int j = 0; j < TN; j++)
                        mac(acc[i][j], lds[buf][ty + SIDE * i][k], lds[buf][BM + tx + SIDE * j][k]);
        }
        if (more) {  // the other buffer's readers passed the last barrier
#pragma unroll
            for (int i = 0; i < PER; i++) store(buf ^ 1, i, next[i]);
        }
        __syncthreads();
    }
#pragma unroll
    for (int j = 0; j < TN; j++) {
        const uint32_t n = n0 + tx + SIDE * j;
        if (n >= N) continue;
        const float b = HEAD ? 0.0f : bias[n];
#pragma unroll
        for (int i = 0; i < TM; i++) {
            const uint32_t m = m0 + ty + SIDE * i;
            if (m >= M) continue;
            float v = acc[i][j];
            if (!HEAD) {
                v += b;
                v = v > 0.0f ? v : 0.0f;
            }
            Y[(size_t)m * N + n] = v;
        }
    }
}

template <int TM, int TN, int BK>
void launch(bool head, bool skip, const float* X, uint32_t K, const float* Wt, const float* b, uint32_t N, float* Y,
            uint32_t M, const uint32_t* rb_n, hipStream_t s) {
    constexpr uint32_t BM = SIDE * TM, BN = SIDE * TN;
    const dim3 g((M + BM - 1) / BM, (N + BN - 1) / BN);
    const bool quads = K % 4 == 0;
    const uint32_t vec = (quads && (uintptr_t)X % 16 == 0 ? VEC_X : 0u) | (quads && (uintptr_t)Wt % 16 == 0 ? VEC_W : 0u);
    if (head)
        hipLaunchKernelGGL((k_exact<TM, TN, BK, true, false>), g, dim3(THREADS), 0, s, X, K, Wt, b, N, Y, M, vec, rb_n);
    else if (skip)
        hipLaunchKernelGGL((k_exact<TM, TN, BK, false, true>), g, dim3(THREADS), 0, s, X, K, Wt, b, N, Y, M, vec, rb_n);
    else
        hipLaunchKernelGGL((k_exact<TM, TN, BK, false, false>), g, dim3(THREADS), 0, s, X, K, Wt, b, N, Y, M, vec,
                           rb_n);
}

void dispatch(bool head, bool skip, const float* X, uint32_t K, const float* Wt, const float* b, uint32_t N, float* Y,
              uint32_t M, const uint32_t* rb_n, hipStream_t s) {
    if (!M || !N) return;
    auto tiles = [&](uint32_t rows, uint32_t cols) {
        return (uint64_t)((M + rows - 1) / rows) * ((N + cols - 1) / cols);
    };
    // With per-block column bounds a finer tile also skips more columns (the
    // 64-subgame wave: 38 us per head with 64-wide tiles, about 20 with 32).
    if (tiles(64, 64) >= MIN_TILES && !rb_n)
        launch<4, 4, 32>(head, skip, X, K, Wt, b, N, Y, M, rb_n, s);
    else if (tiles(64, 32) >= MIN_TILES && !rb_n)
        launch<4, 2, 32>(head, skip, X, K, Wt, b, N, Y, M, rb_n, s);
    else if (tiles(32, 32) >= MIN_TILES)
        launch<2, 2, 64>(head, skip, X, K, Wt, b, N, Y, M, rb_n, s);
    else
        launch<1, 1, 128>(head, skip, X, K, Wt, b, N, Y, M, rb_n, s);
}

}  // namespace

void launch_dense_exact(const float* X, uint32_t K, const float* Wt, const float* b, uint32_t N, float* Y,
                        uint32_t rows, bool skip, hipStream_t s) {
    dispatch(false, skip, X, K, Wt, b, N, Y, rows, nullptr, s);
}

void launch_head_exact(const float* H, uint32_t hidden, const float* Wh, const float* bh, uint32_t heads, float* out,
                       uint32_t rows, hipStream_t s, const uint32_t* rb_n) {
    dispatch(true, false, H, hidden, Wh, bh, heads, out, rows, rb_n, s);
}

}  // namespace wc
