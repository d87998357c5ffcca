// HIP kernels of the wave executor, written for gfx950 (wave64).
//
// Every reduction whose result the CPU solver also forms is taken by one lane
// in the solver's order, with no contraction into FMA (the library is built
// with -ffp-contract=off): per-row regret updates in ascending action order,
// reverse gathers in their stored order, child sums in child order, leaf masses
// and belief normalisations in config order. That makes the CFR state
// bit-identical to the CPU restatement whenever the leaf values are.
#include "kernels.h"

#include <hip/hip_fp16.h>

#include <algorithm>

#include "../../include/wc_wave.h"

namespace wc {

// MFMA operand and accumulator vectors.
typedef _Float16 half8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float float4v __attribute__((ext_vector_type(4)));

#define EPSF 1e-6f       // regret-matching floor (engine/src/search.rs:1658)
#define SMOOTHF 1e-30f   // belief normalisation floor (engine/src/rebel.rs:359)

constexpr int BLOCK = 256;
// The subtree sweep stages a unit's values in LDS when the widest window fits this.
constexpr size_t SWEEP_LDS_MAX = 64 * 1024;
constexpr size_t REACH_LDS_MAX = 32 * 1024;  // the reach pass keeps a unit's reach window in LDS up to this

static inline unsigned grid_for(size_t n, int block = BLOCK) { return (unsigned)((n + block - 1) / block); }

// ------------------------------------------------------------------ helpers

__global__ void k_zero(float* p, size_t n) {
    size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    size_t stride = (size_t)gridDim.x * blockDim.x;
    for (; i < n; i += stride) p[i] = 0.0f;
}

void launch_zero(float* p, size_t n, hipStream_t s) {
    if (n == 0) return;
    unsigned g = grid_for(n);
    if (g > 4096) g = 4096;
    hipLaunchKernelGGL(k_zero, dim3(g), dim3(BLOCK), 0, s, p, n);
}

__device__ __forceinline__ const AccRec& decision_row(const WaveDev& w, uint32_t i, int* p) {
    if (i < w.ndec[0]) {
        *p = 0;
        return w.acc_rec[0][i];
    }
    *p = 1;
    return w.acc_rec[1][i - w.ndec[0]];
}

// ------------------------------------------------------------- CFR state

// cur = 1/len over each acting row (engine/src/search.rs:826-836).
__global__ void k_init_strategy(WaveDev w) {
    uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= w.ndec[0] + w.ndec[1]) return;
    int p;
    AccRec q = decision_row(w, i, &p);
    float u = 1.0f / (float)q.n;
    for (uint32_t g = q.lo; g < q.lo + q.n; g++) w.cur[g] = u;
}

void launch_init_strategy(const WaveDev& w, hipStream_t s) {
    uint32_t n = w.ndec[0] + w.ndec[1];
    if (n) hipLaunchKernelGGL(k_init_strategy, dim3(grid_for(n)), dim3(BLOCK), 0, s, w);
}

// Zero one tree's reach span and write its root (or carried root k) beliefs.
// Root beliefs into the zeroed reach (launch_seed_reach clears it first).
__global__ void k_seed_reach(WaveDev w, float* reach, int root_index) {
    const TreeDev t = w.trees[blockIdx.x];
    if (root_index >= (int)t.nroots) return;
    const float* src = root_index < 0 ? w.roots + t.root0 : w.carried + t.carried0 + (size_t)root_index * (t.n0 + t.n1);
    for (uint32_t i = threadIdx.x; i < t.n0 + t.n1; i += blockDim.x) {
        int p = i >= t.n0;
        uint32_t c = p ? i - t.n0 : i;
        reach[w.reach_base[2 * t.node0 + p] + c] = src[i];
    }
}

void launch_seed_reach(const WaveDev& w, float* reach, size_t reach_len, int root_index, hipStream_t s) {
    launch_zero(reach, reach_len, s);  // every tree's reach span: the trees tile [0, reach_len)
    hipLaunchKernelGGL(k_seed_reach, dim3(w.ntrees), dim3(BLOCK), 0, s, w, reach, root_index);
}

// A row's elements are contiguous and few (2 to 6 on average, rarely over 8),
// so they are taken four at a time with no branch per element: one 16-byte
// load per array and four elements (element arrays are readable 12 bytes past
// their end: another section of the same allocation follows), elements past
// the row's end redirected to an index that is valid, their terms dropped by a
// select. Every sum keeps the CPU's order. A branch per element costs ten
// instructions on top of what it guards, and these kernels were bound by them
// (3,400 instructions in the sweep, 400 of them exec-mask saves): per launch,
// branches per element against quads, the sweep 66 -> 55 us and the reach 57 ->
// 45 us on 256 depth-2 subgames, 53 -> 41 and 53 -> 41 us on 32 heavy-tailed
// ones, 21.7 -> 14.5 and 14.5 -> 12 us on a single depth-1 subgame; top regions
// 69 -> 67 us per iteration (their launches set the time).
__device__ __forceinline__ void quad(const uint32_t* p, uint32_t (&v)[4]) { __builtin_memcpy(v, p, 16); }
__device__ __forceinline__ void quad(const float* p, float (&v)[4]) { __builtin_memcpy(v, p, 16); }
// A wave-uniform pointer, held in scalar registers: a lane's choice between two
// kernel arguments would otherwise become a choice of where to load the
// pointer from, one dependent load more.
template <class T>
__device__ __forceinline__ T* scalar(T* p) {
    asm("" : "+s"(p));
    return p;
}
// The first n (at least 1) of four elements.
__device__ __forceinline__ void store_quad(float* p, const float (&v)[4], uint32_t n) {
    if (n >= 4) {
        __builtin_memcpy(p, v, 16);
        return;
    }
    p[0] = v[0];
    if (n > 1) p[1] = v[1];
    if (n > 2) p[2] = v[2];
}

constexpr uint32_t ROW_QUADS = 3;   // decision rows up to 12 actions stay in registers
constexpr uint32_t ROW_BATCH = 12;  // longer ones go 12 actions at a time
// Network-leaf slots in flight per thread in the sweep's leaf phase.
constexpr uint32_t LEAF_BATCH = 4;

// One child config's reach: the reverse gather in stored order (the CPU's
// scatter order, engine/src/serialize.rs:714-723). With LDSR the unit's reach
// window [rw, rw + rn) is also kept in LDS at lr: parent reach inside it is
// read from there (a parent's slots are all inside or all outside: the wave's
// checks hold every row to it), and the row's result goes to both.
template <bool REV>
__device__ __forceinline__ float reach_sum(const WaveDev& w, const float* reach, const float* strat, uint32_t lo,
                                           uint32_t n, uint32_t base) {
    const uint32_t* esrc = (REV ? w.rev_src : w.rvd_src) + lo;
    const uint32_t* ecell = w.rev_cell + (REV ? lo : 0);
    const float* ep = w.rvd_p + (REV ? 0 : lo);
    float v = 0.0f;
    for (uint32_t c0 = 0; c0 < n; c0 += 8) {
        const bool two = n - c0 > 4;
        uint32_t src[2][4], cell[2][4];
        float a[2][4], b[2][4];
#pragma unroll
        for (int h = 0; h < 2; h++)
            if (h == 0 || two) {
                quad(esrc + c0 + 4 * h, src[h]);
                if (REV)
                    quad(ecell + c0 + 4 * h, cell[h]);
                else
                    quad(ep + c0 + 4 * h, b[h]);
            }
#pragma unroll
        for (int h = 0; h < 2; h++)
            if (h == 0 || two)
#pragma unroll
                for (uint32_t k = 0; k < 4; k++) {
                    const bool in = c0 + 4 * h + k < n;
                    a[h][k] = reach[in ? base + src[h][k] : base];
                    if (REV) b[h][k] = strat[in ? cell[h][k] : 0u];
                }
#pragma unroll
        for (int h = 0; h < 2; h++)
            if (h == 0 || two)
#pragma unroll
                for (uint32_t k = 0; k < 4; k++) v = c0 + 4 * h + k < n ? v + a[h][k] * b[h][k] : v;
    }
    return v;
}
template <bool LDSR = false>
__device__ __forceinline__ void reach_row(const WaveDev& w, float* reach, const float* strat, ReachRec q,
                                          float* lr = nullptr, uint32_t rw = 0, uint32_t rn = 0) {
    const uint32_t lo = q.start, n = q.kn & REC_N;
    const bool rev = (q.kn >> 31) == REACH_REV;
    float v;
    if (LDSR && q.pbase - rw < rn) {
        const uint32_t base = q.pbase - rw;
        v = rev ? reach_sum<true>(w, lr, strat, lo, n, base) : reach_sum<false>(w, lr, strat, lo, n, base);
    } else {
        v = rev ? reach_sum<true>(w, reach, strat, lo, n, q.pbase) : reach_sum<false>(w, reach, strat, lo, n, q.pbase);
    }
    reach[q.out] = v;
    if (LDSR) lr[q.out - rw] = v;
}

// sum = sum * ds + reach * cur over one decision row: the DCFR discount of the
// traverser's average-strategy sum (search.rs:1770-1779, applied at the
// backprop) and this iteration's accumulation (engine/src/search.rs:1818-1835),
// the same two rounded steps in the same order, taken in one pass.
__device__ __forceinline__ void accumulate_row(const WaveDev& w, AccRec q, float ds) {
    const float r = w.reach[q.ridx];
    const uint32_t n = q.n;
    const float* cur = w.cur + q.lo;
    float* sum = w.sum + q.lo;
    for (uint32_t c0 = 0; c0 < n; c0 += 8) {
        const bool two = n - c0 > 4;
        float cu[2][4], sm[2][4];
#pragma unroll
        for (int h = 0; h < 2; h++)
            if (h == 0 || two) {
                quad(cur + c0 + 4 * h, cu[h]);
                quad(sum + c0 + 4 * h, sm[h]);
            }
#pragma unroll
        for (int h = 0; h < 2; h++)
            if (h == 0 || two) {
#pragma unroll
                for (int k = 0; k < 4; k++) sm[h][k] = sm[h][k] * ds + r * cu[h][k];
                store_quad(sum + c0 + 4 * h, sm[h], n - c0 - 4 * h);
            }
    }
}

// Both players' top-down reach of one unit, level by level under block
// barriers (their rows of a level are independent), parents read from L2:
// both players' reach windows in LDS (32 KB at the default unit budget) would
// leave room for five workgroups per CU instead of eight (88.6 against 76.4 µs
// per launch).
__device__ __forceinline__ void reach_unit_both(const WaveDev& w, const UnitDev& u, float* reach, const float* strat) {
    for (uint32_t l = 0; l < u.nlevels; l++) {
        uint32_t b0 = w.reach_lvl[0][u.lvl0 + l], e0 = w.reach_lvl[0][u.lvl0 + l + 1];
        uint32_t b1 = w.reach_lvl[1][u.lvl0 + l], e1 = w.reach_lvl[1][u.lvl0 + l + 1];
        uint32_t n0 = e0 - b0, n = n0 + (e1 - b1);
        for (uint32_t k = threadIdx.x; k < n; k += blockDim.x) {
            if (k < n0)
                reach_row(w, reach, strat, w.reach_rec[0][b0 + k]);
            else
                reach_row(w, reach, strat, w.reach_rec[1][b1 + k - n0]);
        }
        __syncthreads();
    }
}

// One player's top-down reach of one unit, the next level's bounds and each
// thread's first record of it fetched while the current level runs; with
// LDSR the unit's reach window lives in LDS as well (every slot of it is
// written by a level above the rows that read it).
template <bool LDSR>
__device__ __forceinline__ void reach_unit_one(const WaveDev& w, const UnitDev& u, float* reach, const float* strat,
                                               int p, float* lr) {
    // The player's fields by select: indexing them with the run-time p would
    // place the record in scratch memory.
    const uint32_t rw = p ? u.rwin[1] : u.rwin[0], rn = p ? u.rwin_n[1] : u.rwin_n[0];
    const ReachRec* rec = w.reach_rec[p];
    const uint32_t* lvl = w.reach_lvl[p] + u.lvl0;
    const uint32_t L = u.nlevels, t = threadIdx.x;
    uint32_t b = L ? lvl[0] : 0, e = L ? lvl[1] : 0;
    ReachRec q{};
    if (L && b + t < e) q = rec[b + t];
    for (uint32_t l = 0; l < L; l++) {
        const uint32_t lb = b, le = e;
        const bool more = l + 1 < L;
        if (more) {
            b = le;
            e = lvl[l + 2];
        }
        // Each thread's rows form one stream across the levels: the record of
        // its next row (in this level, else its first in the next level) is
        // fetched while the current row runs.
        if (lb + t >= le && more && b + t < e) q = rec[b + t];
        for (uint32_t k = lb + t; k < le;) {
            const uint32_t kn = k + blockDim.x;
            ReachRec qn{};
            if (kn < le)
                qn = rec[kn];
            else if (more && b + t < e)
                qn = rec[b + t];
            reach_row<LDSR>(w, reach, strat, q, lr, rw, rn);
            q = qn;
            k = kn;
        }
        __syncthreads();
    }
}

// Subtree units' reach: one player's, one unit per workgroup with its reach
// window in LDS when LDSR; both players' (player < 0) either as one
// workgroup per (unit, player), windows in LDS, or one per unit from L2. With
// reach2 (player >= 0), workgroup 3 u + k takes unit u's rows of player
// `player` under strat into reach (k = 0) or of player k - 1 under strat2
// into reach2: independent computations, one launch.
template <bool LDSR>
__global__ __launch_bounds__(BLOCK) void k_reach(WaveDev w, uint32_t unit0, float* reach, const float* strat,
                                               int player, float* reach2, const float* strat2) {
    extern __shared__ float lds_reach[];  // the unit's reach window of the player (when LDSR)
    if (player >= 0 && reach2) {
        const uint32_t k = blockIdx.x % 3;
        const UnitDev u = w.units[unit0 + blockIdx.x / 3];
        if (k == 0)
            reach_unit_one<LDSR>(w, u, reach, strat, player, lds_reach);
        else
            reach_unit_one<LDSR>(w, u, reach2, strat2, (int)k - 1, lds_reach);
        return;
    }
    if (LDSR && player < 0) {  // the players' rows are independent: workgroup 2 u + p
        const UnitDev u = w.units[unit0 + blockIdx.x / 2];
        reach_unit_one<true>(w, u, reach, strat, (int)(blockIdx.x & 1), lds_reach);
        return;
    }
    const UnitDev u = w.units[unit0 + blockIdx.x];
    if (player < 0)
        reach_unit_both(w, u, reach, strat);
    else
        reach_unit_one<LDSR>(w, u, reach, strat, player, lds_reach);
}

void launch_reach(const WaveDev& w, uint32_t unit0, uint32_t n, float* reach, const float* strat, int player,
                  hipStream_t s, float* reach2, const float* strat2) {
    if (!n) return;
    if (player < 0) reach2 = nullptr;  // both players already
    const size_t lds = (size_t)w.max_rwin * sizeof(float);
    const bool in_lds = w.unit_lds && lds <= REACH_LDS_MAX;
    const uint32_t grid = reach2 ? 3 * n : player < 0 && in_lds ? 2 * n : n;
    if (in_lds)
        hipLaunchKernelGGL(k_reach<true>, dim3(grid), dim3(BLOCK), lds, s, w, unit0, reach, strat, player, reach2,
                           strat2);
    else
        hipLaunchKernelGGL(k_reach<false>, dim3(grid), dim3(BLOCK), 0, s, w, unit0, reach, strat, player, reach2,
                           strat2);
}

// The average-strategy accumulation of player `acc` over all its decision rows
// (units' and top regions'), one row per thread, in workgroups of a leaf-input
// launch (both only read the final reach). The launch's pool_blocks pooling
// workgroups come longest config lists first; the accumulation's workgroups
// are dealt after the first quarter of them, so the streaming accumulation
// runs beside the long lists rather than trailing the launch (3.94 -> 3.78 ms
// per 256-subgame wave; right after the first eighth or half: 3.86 / 3.89).
// Returns true for an accumulation workgroup, else sets *pool_block to the
// workgroup's index among the pooling ones.
__device__ __forceinline__ bool accumulate_blocks(const WaveDev& w, int acc, float ds, uint32_t pool_blocks,
                                                  uint32_t* pool_block) {
    const uint32_t nacc = acc >= 0 ? gridDim.x - pool_blocks : 0, q1 = pool_blocks / 4;
    if (blockIdx.x >= q1 && blockIdx.x < q1 + nacc) {
        const uint32_t k = (blockIdx.x - q1) * blockDim.x + threadIdx.x;
        if (k < w.ndec[acc]) accumulate_row(w, w.acc_rec[acc][k], ds);
        return true;
    }
    *pool_block = blockIdx.x < q1 ? blockIdx.x : blockIdx.x - nacc;
    return false;
}

// Top-region reach at one depth, all trees together: one row per thread, the
// rows of up to three independent sets (players, reach computations).
__global__ __launch_bounds__(BLOCK) void k_reach_rows(WaveDev w, ReachSet a, ReachSet b, ReachSet c) {
    uint32_t k = blockIdx.x * blockDim.x + threadIdx.x;
    if (k < a.n) {
        reach_row(w, a.reach, a.strat, a.rows[k]);
        return;
    }
    k -= a.n;
    if (k < b.n) {
        reach_row(w, b.reach, b.strat, b.rows[k]);
        return;
    }
    k -= b.n;
    if (k < c.n) reach_row(w, c.reach, c.strat, c.rows[k]);
}

// A top depth holds 10k-50k rows, one per thread: one-wavefront workgroups
// spread them over four times as many CUs as 256-thread ones, so each CU's
// memory pipeline serves fewer of the rows' dependent loads (0.33 ms per wave
// of 256 subgames over 1,120 launches).
constexpr int TOP_BLOCK = 64;

void launch_reach_rows(const WaveDev& w, const ReachSet& a, const ReachSet& b, const ReachSet& c, hipStream_t s) {
    const size_t n = (size_t)a.n + b.n + c.n;
    if (n) hipLaunchKernelGGL(k_reach_rows, dim3(grid_for(n, TOP_BLOCK)), dim3(TOP_BLOCK), 0, s, w, a, b, c);
}

// Top-region reach at two depths in one launch, up to three independent sets
// (players, reach computations) one after another in the grid. A shallower
// row named by two chunks is computed by both: reach rows keep no state, and
// both write the same value, so each chunk reads its own result or the
// other's equal one after its barrier. A chunk names up to about 85
// shallower rows for its 64 deeper ones, so its workgroup has two wavefronts:
// one shallower row per thread (20.34 ms per 256-subgame wave, against 20.65
// with one wavefront, two rows on some threads, and 20.45 without the fused
// reach launches).
__global__ __launch_bounds__(BLOCK) void k_reach_pair(WaveDev w, ReachPair a, ReachPair b, ReachPair c) {
    uint32_t k = blockIdx.x;
    ReachPair s = a;
    if (k >= a.chunks) {
        k -= a.chunks;
        s = b;
        if (k >= b.chunks) {
            k -= b.chunks;
            s = c;
        }
    }
    const uint32_t* q = s.off + s.chunks + 1;
    for (uint32_t i = q[k] + threadIdx.x; i < q[k + 1]; i += blockDim.x)
        reach_row(w, s.reach, s.strat, s.rows[s.par[i]]);
    __syncthreads();
    for (uint32_t i = s.off[k] + threadIdx.x; i < s.off[k + 1]; i += blockDim.x)
        reach_row(w, s.reach, s.strat, s.rows[i]);
}

void launch_reach_pair(const WaveDev& w, const ReachPair& a, const ReachPair& b, const ReachPair& c, hipStream_t s) {
    const uint32_t n = a.chunks + b.chunks + c.chunks;
    if (n) hipLaunchKernelGGL(k_reach_pair, dim3(n), dim3(2 * TOP_BLOCK), 0, s, w, a, b, c);
}

// sum = reach * cur: one reach-weighted uniform strategy (engine/src/search.rs:854-870).
__global__ void k_seed_sum(WaveDev w) {
    uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= w.ndec[0] + w.ndec[1]) return;
    int p;
    AccRec q = decision_row(w, i, &p);
    float r = w.reach[q.ridx];
    for (uint32_t g = q.lo; g < q.lo + q.n; g++) w.sum[g] = r * w.cur[g];
}

void launch_seed_sum(const WaveDev& w, hipStream_t s) {
    uint32_t n = w.ndec[0] + w.ndec[1];
    if (n) hipLaunchKernelGGL(k_seed_sum, dim3(grid_for(n)), dim3(BLOCK), 0, s, w);
}

// --------------------------------------------------------------- leaf input

__device__ __forceinline__ uint16_t f32_to_bf16_rn(float x) {
    uint32_t u = __float_as_uint(x);
    if ((u & 0x7fffffffu) > 0x7f800000u) return (uint16_t)((u | 0x00400000u) >> 16);
    u += 0x7fffu + ((u >> 16) & 1u);
    return (uint16_t)(u >> 16);
}

__device__ __forceinline__ uint16_t f32_to_f16_rn(float x) {
    _Float16 h = (_Float16)x;
    return __builtin_bit_cast(uint16_t, h);
}

// One query-input element. Compensated f16 keeps two planes `plane` elements
// apart: hi = f16(v) and lo = f16(v - hi).
template <int PREC>
__device__ __forceinline__ void store_operand(void* base, size_t i, float v, size_t plane) {
    if (PREC == WC_PRECISE) {
        ((float*)base)[i] = v;
    } else if (PREC == WC_F16) {
        ((uint16_t*)base)[i] = f32_to_f16_rn(v);
    } else if (PREC == WC_BF16) {
        ((uint16_t*)base)[i] = f32_to_bf16_rn(v);
    } else {
        const uint16_t hi = f32_to_f16_rn(v);
        ((uint16_t*)base)[i] = hi;
        ((uint16_t*)base)[i + plane] = f32_to_f16_rn(v - (float)__builtin_bit_cast(_Float16, hi));
    }
}

// Query inputs are row-major float32 for the exact net, fragment-major 16-bit for MFMA.
template <int PREC>
__device__ __forceinline__ size_t operand_at(uint32_t row, uint32_t k, uint32_t K) {
    return PREC == WC_PRECISE ? (size_t)row * K + k : frag_off(row, k, K);
}

__device__ __forceinline__ float lane_value(float v, uint32_t j) {
    return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), (int)j));
}
__device__ __forceinline__ uint32_t lane_value(uint32_t v, uint32_t j) {
    return (uint32_t)__builtin_amdgcn_readlane((int)v, (int)j);
}

// tot + v's lanes 0 .. m - 1 (m <= 64), added one at a time in lane order.
// Eight lanes are read per step (independent reads ahead of the dependent
// adds); the caller sets lanes m .. 63 to +0.0, and adding +0.0 leaves a sum
// that started at +0.0 unchanged (such a sum is never -0.0), so the result is
// the plain sequential sum.
__device__ __forceinline__ float lane_sum_in_order(float tot, float v, uint32_t m) {
    for (uint32_t k0 = 0; k0 < m; k0 += 8) {
        float y[8];
#pragma unroll
        for (uint32_t i = 0; i < 8; i++) y[i] = lane_value(v, k0 + i);
#pragma unroll
        for (uint32_t i = 0; i < 8; i++) tot += y[i];
    }
    return tot;
}

// Float32 net: one wavefront per (network row, player). The leaf's reach
// mass, and the pooled belief sum_c beta(c) e(c) with beta the normalised
// reach (normalize_weights, engine/src/rebel.rs:1054-1068; accumulate,
// net.rs:161-170). Lanes load 64 configs at a time; both reductions then run
// in config order with every lane holding the running value, so the result is
// the CPU's sequential sum. Bound: the instructions of the longest list's chain
// (a lane per dimension, configs one after another), so each config costs a
// lane read, a 32-bit add and a load for its embedding (64-bit addresses cost
// five more scalar instructions) and a lane read, a product and a sum, with 16
// configs' loads in flight ahead of them: 64 depth-1 subgames 52 -> 32 us per
// launch, 32 depth-2 subgames 48 -> 30 us. WIDE: a table of 4 GiB or more.
// The pooled block goes straight into the two query inputs that carry it:
// [pooled_q | pooled_{1-q} | seat | public] for traverser q.
template <bool WIDE>
__global__ __launch_bounds__(BLOCK) void k_pool_exact(WaveDev w, int player, float* x0, float* x1, int acc,
                                                    float ds, uint32_t pool_blocks) {
    uint32_t pbk;
    if (accumulate_blocks(w, acc, ds, pool_blocks, &pbk)) return;
    const uint32_t task = __builtin_amdgcn_readfirstlane((pbk * blockDim.x + threadIdx.x) >> 6);
    const uint32_t lane = threadIdx.x & 63;
    uint32_t row, p;
    if (player < 0) {
        row = task >> 1;
        p = task & 1;
    } else {
        row = task;
        p = (uint32_t)player;
    }
    if (row >= w.rows) return;  // wave-uniform
    const uint32_t node = w.row_node[row];
    const uint32_t n = w.nc[2 * node + p];
    const float* r = w.reach + w.reach_base[2 * node + p];
    const uint32_t* cfgs = w.row_cfg + w.row_cfg_off[2 * row + p];
    float tot = 0.0f;
    for (uint32_t c0 = 0; c0 < n; c0 += 64) {
        float v = c0 + lane < n ? r[c0 + lane] : 0.0f;
        tot = lane_sum_in_order(tot, v, n - c0 < 64 ? n - c0 : 64);
    }
    float scale, flat;
    if (tot > SMOOTHF) {
        scale = 1.0f / tot;
        flat = 0.0f;
    } else {
        scale = 0.0f;
        flat = 1.0f / (float)(n > 0 ? n : 1);
    }
    if (lane == 0) w.mass[2 * row + p] = tot;
    const uint32_t pool = w.pool, in = w.in;
    float* own = p ? x1 : x0;    // pooled_p is the first block of traverser p's query
    float* other = p ? x0 : x1;  // and the second block of the other traverser's
    for (uint32_t k0 = 0; k0 < pool; k0 += 64) {
        const uint32_t k = k0 + lane;
        const bool live = k < pool;
        float acc = 0.0f;
        // 16 configs' embeddings per batch, one batch loading while the one
        // before it is added in config order. Lanes past the list hold config
        // 0, so that a batch's loads need no branch (an empty list loads none:
        // the wave may have no config at all).
        float e0[16], e1[16];
        const uint32_t kk = live ? k : 0u;
        auto index = [&](uint32_t c0) { return (c0 + lane < n ? cfgs[c0 + lane] : 0u) * (WIDE ? 1u : pool); };
        auto belief = [&](uint32_t c0) { return c0 + lane < n ? r[c0 + lane] * scale + flat : 0.0f; };
        auto fetch = [&](float (&e)[16], uint32_t cf, uint32_t j0) {
#pragma unroll
            for (uint32_t j = 0; j < 16; j++) {
                const uint32_t c = lane_value(cf, j0 + j);
                if (WIDE)
                    e[j] = w.cfg_emb[(size_t)c * pool + kk];
                else  // a 32-bit byte offset from the table
                    e[j] = *(const float*)((const char*)w.cfg_emb + 4u * (c + kk));
            }
        };
        auto add = [&](const float (&e)[16], float beta, uint32_t j0, uint32_t left) {
            if (left >= 16) {
#pragma unroll
                for (uint32_t j = 0; j < 16; j++) acc += lane_value(beta, j0 + j) * e[j];
                return;
            }
#pragma unroll
            for (uint32_t j = 0; j < 16; j++)
                if (j < left) acc += lane_value(beta, j0 + j) * e[j];
        };
        uint32_t cf = index(0);
        float beta = belief(0);
        if (n) fetch(e0, cf, 0);
        for (uint32_t c0 = 0; c0 < n; c0 += 64) {
            const uint32_t left = n - c0, cn = index(c0 + 64);
            const float bn = belief(c0 + 64);
            if (left > 16) fetch(e1, cf, 16);
            add(e0, beta, 0, left);
            if (left > 16) {
                if (left > 32) fetch(e0, cf, 32);
                add(e1, beta, 16, left - 16);
            }
            if (left > 32) {
                if (left > 48) fetch(e1, cf, 48);
                add(e0, beta, 32, left - 32);
            }
            if (left > 48) {
                if (left > 64) fetch(e0, cn, 0);
                add(e1, beta, 48, left - 48);
            }
            cf = cn;
            beta = bn;
        }
        if (live) {
            own[(size_t)row * in + k] = acc;
            other[(size_t)row * in + pool + k] = acc;
        }
    }
}

// 16-bit nets: pool groups (up to POOL_GROUP rows of one player whose configs
// are the same list) on the f32 MFMA. With A the group's reach rows (row 15:
// ones) and B the configs' embeddings, a 16x16x4 product per 16 dimensions and
// 4 configs accumulates U[r][k] = sum_c reach_r(c) e_c(k) and, in row 15, S[k]
// = sum_c e_c(k); each row's mass is summed on the VALU from the same reach
// values. Then pooled = U / mass, or S / n where the mass is below the
// smoothing floor (the uniform weights of normalize_weights). Each config's
// embedding is read once for the group. Products are exact f32; only the
// summation order differs from the CPU's, far below the 16-bit rounding of the
// stored query input.
//
// A list of up to POOL_LONG configs takes one wavefront, all its loads of a
// 64-config chunk in flight together. A longer one is a chain of chunks, each
// with dependent loads (config indices, then embeddings), so it takes a whole
// workgroup, unless there are enough of them to fill the device: the wavefronts
// split the dimensions (16 each, so that every sum keeps its one order), share
// the reach and the indices through LDS, and the next chunk's are on their way
// while the current one multiplies. Bound: the latency of those loads with four
// wavefronts per SIMD (five spill). Leaf-input time per wave, all lists on
// single wavefronts against long ones on workgroups: 32 heavy-tailed subgames
// 11.8 -> 8.2 ms, 64 depth-1 subgames in compensated f16 2.43 -> 1.37 ms, 256
// depth-2 subgames 3.50 -> 3.40 ms.

// Configs past which a list takes a workgroup, and configs per LDS chunk. Below
// the line four wavefronts wait for the loads of one or two chunks; from 128 to
// 256 it hardly matters where it lies (whole schedules at 128 / 192 / 256, 12
// runs each within 0.02 ms: 256 depth-2 subgames 18.48 / 18.32 / 18.23 ms, 64 of
// them 8.31 / 8.33 / 8.40, 32 heavy-tailed ones 33.5 at each, 64 depth-1 ones in
// compensated f16 6.94 / 6.93 / 6.94).
// POOL_FILL: wavefronts a CU holds (four per SIMD). Lists that fill the device
// with a wavefront each hide their chains behind one another, and the
// workgroups' barriers only cost: heavy-tailed subgames' leaf input per wave, on
// workgroups against single wavefronts, with 2,300 + 2,000 long lists of the two
// players 8.2 against 11.8 ms, 3,200 + 2,700 11.0 against 12.6, 5,300 + 3,900
// 16.3 against 15.3, 21,800 + 18,100 69.9 against 60.6.
constexpr uint32_t POOL_LONG = 192, POOL_CH = 64, POOL_FILL = 16;
// A chunk's reach rows in LDS: config c of a row at POOL_Q (c % 4) + c / 4, so
// that a lane's configs of four consecutive MFMA steps are one 16-byte read;
// the pitches spread a wavefront's reads and writes over the banks.
constexpr uint32_t POOL_Q = 48, POOL_ROW = 4 * POOL_Q + 4;
// A finished group in LDS as 16-bit operands: rows of 64 dimensions.
constexpr uint32_t POOL_OUT = 72;

struct PoolLds {
    union {
        struct {
            float a[2][POOL_GROUP][POOL_ROW];
            uint32_t idx[2][4][POOL_CH / 4];  // config c at [c % 4][c / 4]
        } chunk;
        uint16_t out[BLOCK / 64][2][POOL_GROUP + 1][POOL_OUT];  // per wavefront (short lists) and plane
    };
    uint32_t rbase[POOL_GROUP];
};

// Writes a group's pooled rows (the 64 dimensions from k0 on, row rr at
// src[rr], the compensated lo plane at src[16 + rr]) into both query inputs,
// eight dimensions per store: n threads, this one the t-th.
template <int PREC>
__device__ __forceinline__ void pool_store(const WaveDev& w, const PoolGroup* grp, uint32_t p, uint16_t* x0,
                                           uint16_t* x1, const uint16_t (*src)[POOL_OUT], uint32_t k0, uint32_t t,
                                           uint32_t n) {
    uint16_t* own = p ? x1 : x0;    // pooled_p is the first block of traverser p's query
    uint16_t* other = p ? x0 : x1;  // and the second block of the other traverser's
    const uint32_t G = grp->nrows, pool = w.pool;
    if (pool % 8 == 0) {
        for (uint32_t e = t; e < G * 8; e += n) {
            const uint32_t rr = e >> 3, k = k0 + 8 * (e & 7);
            if (k >= pool) continue;
            const uint32_t row = grp->row[rr];
            const size_t o = frag_off(row, k, w.in), x = frag_off(row, pool + k, w.in);
            const uint4 hi = *(const uint4*)&src[rr][k - k0];
            *(uint4*)(own + o) = hi;
            *(uint4*)(other + x) = hi;
            if (PREC == WC_F16X) {
                const uint4 lo = *(const uint4*)&src[POOL_GROUP + 1 + rr][k - k0];
                *(uint4*)(own + o + w.xplane) = lo;
                *(uint4*)(other + x + w.xplane) = lo;
            }
        }
        return;
    }
    for (uint32_t e = t; e < G * 64; e += n) {
        const uint32_t rr = e >> 6, k = k0 + (e & 63);
        if (k >= pool) continue;
        const uint32_t row = grp->row[rr];
        const size_t o = frag_off(row, k, w.in), x = frag_off(row, pool + k, w.in);
        own[o] = other[x] = src[rr][k - k0];
        if (PREC == WC_F16X) own[o + w.xplane] = other[x + w.xplane] = src[POOL_GROUP + 1 + rr][k - k0];
    }
}

// One 16-dimension tile's sums (this lane: rows 4q .. 4q + 3, dimension d of
// the 64) over their rows' masses, into the group's LDS rows.
template <int PREC>
__device__ __forceinline__ void pool_tile(const float4v& acc, const float (&tot)[4], float inv_n, uint32_t q,
                                          uint32_t i, uint32_t d, uint16_t (*dst)[POOL_OUT]) {
    const float S = __shfl(acc[3], (int)(48 + i), 64);  // row 15 of this column
#pragma unroll
    for (int v = 0; v < 4; v++) {
        const float y = tot[v] > SMOOTHF ? acc[v] * (1.0f / tot[v]) : S * inv_n;
        const uint32_t rr = 4 * q + v;  // (row 15's slot is never stored)
        store_operand<PREC>(dst, rr * POOL_OUT + d, y, (POOL_GROUP + 1) * POOL_OUT);
    }
}

// Row i's mass from the lanes' partial sums (lanes i, i + 16, i + 32, i + 48),
// to the masses of rows 4q .. 4q + 3; returns row i's.
__device__ __forceinline__ float pool_mass(float tpart, uint32_t q, float (&tot)[4]) {
    float ti = tpart + __shfl_xor(tpart, 16, 64);
    ti += __shfl_xor(ti, 32, 64);
#pragma unroll
    for (int v = 0; v < 4; v++) tot[v] = __shfl(ti, (int)(4 * q + v), 64);
    return ti;
}

// A list on one wavefront.
template <int PREC>
__device__ __forceinline__ void pool_short(const WaveDev& w, const PoolGroup* grp, uint32_t p, uint16_t* x0,
                                           uint16_t* x1, uint16_t (*dst)[POOL_OUT]) {
    const uint32_t lane = threadIdx.x & 63;
    const uint32_t n = grp->n, G = grp->nrows;
    const uint32_t i = lane & 15, q = lane >> 4;  // A row / B column, and config within a 4-step
    const float* ra = w.reach + grp->rbase[i < POOL_GROUP ? i : 0];  // lane row 15 reads no reach
    const float aconst = i == 15 ? 1.0f : 0.0f;  // rows G..14 are zero, row 15 sums the embeddings
    const uint32_t* cfgs = w.row_cfg + grp->cfg;
    const uint32_t pool = w.pool;
    float tot[4] = {0.0f, 0.0f, 0.0f, 0.0f};  // mass of rows 4q .. 4q + 3
    for (uint32_t k0 = 0; k0 < pool; k0 += 64) {
        float4v acc[4];
#pragma unroll
        for (int t = 0; t < 4; t++) acc[t] = float4v{0.0f, 0.0f, 0.0f, 0.0f};
        bool kl[4];
#pragma unroll
        for (int t = 0; t < 4; t++) kl[t] = k0 + 16 * t + i < pool;
        float tpart = 0.0f;  // this lane's share of row i's mass: configs 4 s + q
        // 64 configs per chunk: one coalesced load of their indices, the reach
        // gathers of all 16 steps in flight together, each step's index handed
        // to its lanes by a shuffle, then 8 steps' embeddings at a time. Steps
        // past the end of the list are skipped.
        for (uint32_t c0 = 0; c0 < n; c0 += 64) {
            const uint32_t cfl = c0 + lane < n ? cfgs[c0 + lane] : 0xffffffffu;
            float a[16];
#pragma unroll
            for (int s = 0; s < 16; s++) {
                const uint32_t c = c0 + 4 * s + q;
                a[s] = c < n ? (i < G ? ra[c] : aconst) : 0.0f;
            }
#pragma unroll
            for (int s = 0; s < 16; s++) tpart += a[s];
#pragma unroll
            for (int h = 0; h < 2; h++) {
                if (c0 + 32 * h >= n) break;  // wave-uniform
                uint32_t cf[8];
                float b[8][4];
#pragma unroll
                for (int s = 0; s < 8; s++) cf[s] = (uint32_t)__shfl((int)cfl, 4 * (8 * h + s) + (int)q, 64);
#pragma unroll
                for (int s = 0; s < 8; s++) {
                    const bool live = cf[s] != 0xffffffffu;
                    const float* e = w.cfg_emb + (size_t)(live ? cf[s] : 0u) * pool + k0 + i;
#pragma unroll
                    for (int t = 0; t < 4; t++) b[s][t] = live && kl[t] ? e[16 * t] : 0.0f;
                }
#pragma unroll
                for (int s = 0; s < 8; s++) {
                    if (c0 + 4 * (8 * h + s) >= n) break;  // wave-uniform
#pragma unroll
                    for (int t = 0; t < 4; t++)
                        acc[t] = __builtin_amdgcn_mfma_f32_16x16x4f32(a[8 * h + s], b[s][t], acc[t], 0, 0, 0);
                }
            }
        }
        if (k0 == 0) {
            const float ti = pool_mass(tpart, q, tot);
            if (q == 0 && i < G) w.mass[2 * grp->row[i] + p] = ti;
        }
        const float inv_n = 1.0f / (float)(n > 0 ? n : 1);
#pragma unroll
        for (int t = 0; t < 4; t++) pool_tile<PREC>(acc[t], tot, inv_n, q, i, 16 * t + i, dst);
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");  // the wavefront's own LDS rows
        pool_store<PREC>(w, grp, p, x0, x1, dst, k0, lane, 64);
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    }
}

// A list on the workgroup, one 16-dimension tile per wavefront.
template <int PREC>
__device__ __forceinline__ void pool_long(const WaveDev& w, const PoolGroup* grp, uint32_t p, uint16_t* x0,
                                          uint16_t* x1, PoolLds& sh) {
    const uint32_t t = threadIdx.x, lane = t & 63, wave = t >> 6;
    const uint32_t n = grp->n, G = min(grp->nrows, POOL_GROUP);
    const uint32_t i = lane & 15, q = lane >> 4;
    const uint32_t* cfgs = w.row_cfg + grp->cfg;
    const uint32_t pool = w.pool;
    if (t < POOL_GROUP) sh.rbase[t] = grp->rbase[t];
    __syncthreads();
    // One chunk: POOL_CH indices, and G x POOL_CH reach values, 8 per thread.
    constexpr int PER = (POOL_GROUP * POOL_CH + BLOCK - 1) / BLOCK;
    float rv[PER];
    uint32_t iv = 0xffffffffu;
    const uint32_t cc = t % POOL_CH, r0 = t / POOL_CH;  // this thread's column, and its rows r0, r0 + 4, ...
    auto fetch = [&](uint32_t c0) {
        const uint32_t c = c0 + cc;
        if (t < POOL_CH) iv = c < n ? cfgs[c] : 0xffffffffu;
#pragma unroll
        for (int j = 0; j < PER; j++) {
            const uint32_t r = r0 + j * (BLOCK / POOL_CH);
            rv[j] = r < G && c < n ? w.reach[sh.rbase[r] + c] : 0.0f;
        }
    };
    auto stage = [&](int buf) {
        if (t < POOL_CH) sh.chunk.idx[buf][cc & 3][cc >> 2] = iv;
#pragma unroll
        for (int j = 0; j < PER; j++) {
            const uint32_t r = r0 + j * (BLOCK / POOL_CH);
            if (r < G) sh.chunk.a[buf][r][POOL_Q * (cc & 3) + (cc >> 2)] = rv[j];
        }
    };
    float tot[4] = {0.0f, 0.0f, 0.0f, 0.0f};
    for (uint32_t k0 = 0; k0 < pool; k0 += 64) {
        const uint32_t k = k0 + 16 * wave + i;
        const bool kl = k < pool;
        const float* emb = w.cfg_emb + (kl ? k : 0u);
        float4v acc = float4v{0.0f, 0.0f, 0.0f, 0.0f};
        float tpart = 0.0f;
        fetch(0);
        stage(0);
        __syncthreads();
        int buf = 0;
        for (uint32_t c0 = 0; c0 < n; c0 += POOL_CH, buf ^= 1) {
            const bool more = c0 + POOL_CH < n;
            float b[POOL_CH / 4];
#pragma unroll
            for (int s4 = 0; s4 < (int)POOL_CH / 16; s4++) {
                const uint4 cf = *(const uint4*)&sh.chunk.idx[buf][q][4 * s4];
                const uint32_t f[4] = {cf.x, cf.y, cf.z, cf.w};
#pragma unroll
                for (int s = 0; s < 4; s++) {
                    const bool live = f[s] != 0xffffffffu && kl;
                    const float e = emb[(size_t)(live ? f[s] : 0u) * pool];
                    b[4 * s4 + s] = live ? e : 0.0f;
                }
            }
            if (more) fetch(c0 + POOL_CH);
#pragma unroll
            for (int s4 = 0; s4 < (int)POOL_CH / 16; s4++) {
                if (c0 + 16 * s4 >= n) break;  // block-uniform
                float4v a4 = *(const float4v*)&sh.chunk.a[buf][i < POOL_GROUP ? i : 0][POOL_Q * q + 4 * s4];
#pragma unroll
                for (int s = 0; s < 4; s++) {
                    const uint32_t c = c0 + 4 * (4 * s4 + s) + q;
                    const float a = i < G ? a4[s] : i == 15 && c < n ? 1.0f : 0.0f;
                    tpart += a;
                    if (c0 + 4 * (4 * s4 + s) < n) acc = __builtin_amdgcn_mfma_f32_16x16x4f32(a, b[4 * s4 + s], acc, 0, 0, 0);
                }
            }
            if (more) stage(buf ^ 1);
            __syncthreads();
        }
        if (k0 == 0) {
            const float ti = pool_mass(tpart, q, tot);
            if (wave == 0 && q == 0 && i < G) w.mass[2 * grp->row[i] + p] = ti;
        }
        pool_tile<PREC>(acc, tot, 1.0f / (float)n, q, i, 16 * wave + i, sh.out[0][0]);  // (the chunks are done)
        __syncthreads();
        pool_store<PREC>(w, grp, p, x0, x1, sh.out[0][0], k0, t, BLOCK);
        __syncthreads();
    }
}

template <int PREC>
__global__ __launch_bounds__(BLOCK, 4) void k_pool_mfma(WaveDev w, int player, uint16_t* x0, uint16_t* x1, int acc,
                                                   float ds, uint32_t pool_blocks) {
    __shared__ __attribute__((aligned(16))) PoolLds sh;
    uint32_t pbk;
    if (accumulate_blocks(w, acc, ds, pool_blocks, &pbk)) return;
    // One workgroup per long list (each player's lists come longest first),
    // then a wavefront per short one.
    const uint32_t l0 = player != 1 ? w.nlong[0] : 0, l1 = player != 0 ? w.nlong[1] : 0;
    if (pbk < l0 + l1) {
        const uint32_t p = pbk < l0 ? 0 : 1;
        pool_long<PREC>(w, w.pool_grp[p] + (p ? pbk - l0 : pbk), p, x0, x1, sh);
        return;
    }
    const uint32_t wave = threadIdx.x >> 6;
    uint32_t g = __builtin_amdgcn_readfirstlane((pbk - l0 - l1) * (BLOCK / 64) + wave);
    const uint32_t s0 = player != 1 ? w.npool[0] - w.nlong[0] : 0;
    const uint32_t p = g < s0 ? 0 : 1;
    g = p ? g - s0 + w.nlong[1] : g + w.nlong[0];
    if (player == 0 ? p == 1 : g >= w.npool[1] && p == 1) return;  // wave-uniform: past the last group
    pool_short<PREC>(w, w.pool_grp[p] + g, p, x0, x1, sh.out[wave][0]);
}

uint32_t pool_long_groups(const PoolGroup* grp, uint32_t n, uint32_t cus) {
    uint32_t k = 0;
    while (k < n && grp[k].n > POOL_LONG) k++;
    return k <= POOL_FILL * cus ? k : 0;
}

void launch_pool(const WaveDev& w, int player, int precision, void* x0, void* x1, hipStream_t s, int acc,
                 float ds) {
    const uint32_t accb = acc >= 0 ? grid_for(w.ndec[acc]) : 0;
    if (precision == WC_PRECISE) {
        size_t waves = (size_t)w.rows * (player < 0 ? 2 : 1);
        const uint32_t pb = grid_for(waves * 64);
        if (!(pb + accb)) return;
        if (w.emb_wide)
            hipLaunchKernelGGL(k_pool_exact<true>, dim3(pb + accb), dim3(BLOCK), 0, s, w, player, (float*)x0,
                               (float*)x1, acc, ds, pb);
        else
            hipLaunchKernelGGL(k_pool_exact<false>, dim3(pb + accb), dim3(BLOCK), 0, s, w, player, (float*)x0,
                               (float*)x1, acc, ds, pb);
        return;
    }
    size_t waves = 0, wide = 0;
    for (int p = 0; p < 2; p++)
        if (player < 0 || p == player) {
            wide += w.nlong[p];
            waves += w.npool[p] - w.nlong[p];
        }
    const uint32_t pb = (uint32_t)wide + grid_for(waves * 64);
    if (!(pb + accb)) return;
    dim3 g(pb + accb);
    if (precision == WC_F16)
        hipLaunchKernelGGL(k_pool_mfma<WC_F16>, g, dim3(BLOCK), 0, s, w, player, (uint16_t*)x0, (uint16_t*)x1, acc,
                           ds, pb);
    else if (precision == WC_BF16)
        hipLaunchKernelGGL(k_pool_mfma<WC_BF16>, g, dim3(BLOCK), 0, s, w, player, (uint16_t*)x0, (uint16_t*)x1, acc,
                           ds, pb);
    else
        hipLaunchKernelGGL(k_pool_mfma<WC_F16X>, g, dim3(BLOCK), 0, s, w, player, (uint16_t*)x0, (uint16_t*)x1, acc,
                           ds, pb);
}

// The fixed part of both traversers' query inputs: the seat (-1 for player 0,
// +1 for player 1) and the row's public features / 255.
template <int PREC>
__global__ void k_query_static(WaveDev w, void* x0, void* x1) {
    size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    const uint32_t width = w.in - 2 * w.pool;
    if (i >= (size_t)w.rows * width) return;
    uint32_t row = (uint32_t)(i / width), k = (uint32_t)(i % width);
    size_t at = operand_at<PREC>(row, 2 * w.pool + k, w.in);
    if (k == 0) {
        store_operand<PREC>(x0, at, -1.0f, w.xplane);
        store_operand<PREC>(x1, at, 1.0f, w.xplane);
    } else {
        // public features; columns past them (a 16-bit operand's k padding) are zero
        const float v = k - 1 < w.row_bytes ? (float)w.pub_raw[(size_t)row * w.row_bytes + (k - 1)] / 255.0f : 0.0f;
        store_operand<PREC>(x0, at, v, w.xplane);
        store_operand<PREC>(x1, at, v, w.xplane);
    }
}

void launch_query_static(const WaveDev& w, int precision, void* x0, void* x1, hipStream_t s) {
    size_t n = (size_t)w.rows * (w.in - 2 * w.pool);
    if (!n) return;
    if (precision == WC_PRECISE)
        hipLaunchKernelGGL(k_query_static<WC_PRECISE>, dim3(grid_for(n)), dim3(BLOCK), 0, s, w, x0, x1);
    else if (precision == WC_F16)
        hipLaunchKernelGGL(k_query_static<WC_F16>, dim3(grid_for(n)), dim3(BLOCK), 0, s, w, x0, x1);
    else if (precision == WC_BF16)
        hipLaunchKernelGGL(k_query_static<WC_BF16>, dim3(grid_for(n)), dim3(BLOCK), 0, s, w, x0, x1);
    else
        hipLaunchKernelGGL(k_query_static<WC_F16X>, dim3(grid_for(n)), dim3(BLOCK), 0, s, w, x0, x1);
}

// ------------------------------------------------------------- the sweep

// One value row of traverser p (engine/src/search.rs:1672-1803).
// Values come from the unit's LDS window when LDSV (slot i at lv[i - vw]),
// else from HBM; results go to both.
template <int MODE, bool LDSV>
__device__ __forceinline__ void backprop_row(const WaveDev& w, int p, BackRec q, float da, float db, float predict,
                                             const float* strat, float* lv, uint32_t vw) {
    float* vals = w.vals;
    // A staged unit keeps its values in LDS; only values read outside the
    // unit (REC_EXPORT) also go to HBM.
    const bool to_hbm = !LDSV || (q.kn & REC_EXPORT);
    auto get = [&](uint32_t i) { return LDSV ? lv[i - vw] : vals[i]; };
    auto put = [&](uint32_t i, float v) {
        if (to_hbm) vals[i] = v;
        if (LDSV) lv[i - vw] = v;
    };
    const uint32_t kind = q.kn >> 30, n = q.kn & REC_N, lo = q.start;
    if (kind != BACK_OWN) {
        // The traverser draws: push values through the outcome row. The
        // opponent decides: sum the children in child order.
        const bool draw = kind == BACK_DRAW;
        const uint32_t* eto = (draw ? scalar(w.draw_to) : scalar(p ? w.child_vb[1] : w.child_vb[0])) + lo;
        const float* ep = w.draw_p + (draw ? lo : 0);
        float v = 0.0f;
        for (uint32_t c0 = 0; c0 < n; c0 += 8) {
            const bool two = n - c0 > 4;
            uint32_t to[2][4];
            float pr[2][4], cv[2][4];
#pragma unroll
            for (int h = 0; h < 2; h++)
                if (h == 0 || two) {
                    quad(eto + c0 + 4 * h, to[h]);
                    if (draw) quad(ep + c0 + 4 * h, pr[h]);
                }
#pragma unroll
            for (int h = 0; h < 2; h++)
                if (h == 0 || two)
#pragma unroll
                    for (uint32_t k = 0; k < 4; k++) cv[h][k] = get(c0 + 4 * h + k < n ? q.arg + to[h][k] : q.out);
#pragma unroll
            for (int h = 0; h < 2; h++)
                if (h == 0 || two)
#pragma unroll
                    for (uint32_t k = 0; k < 4; k++)
                        v = c0 + 4 * h + k < n ? v + (draw ? pr[h][k] * cv[h][k] : cv[h][k]) : v;
        }
        put(q.out, v);
        return;
    }
    // The traverser's own row: base = sum of child value x strategy in action
    // order, then the fused regret matching with DCFR discounting
    // (search.rs:1742-1779): r = old (old > 0 ? da : db) + delta, cur = max(r +
    // predict delta, EPS), normalised by a reciprocal multiply. The sum's
    // discount (sum *= ds) is taken with the accumulation in the reach sweep.
    const float* st = MODE == MODE_VALUE ? strat : w.cur;
    // A config without actions has the value zero and owns no cell. (Leaving here
    // costs nothing; bounding the branch below to 1 to 12 actions instead, the
    // heavy-tailed wave's CFR passes took 111.7 ms for 110.5.)
    if (n == 0) {
        put(q.out, 0.0f);
        return;
    }
    if (n <= ROW_BATCH) {  // everything stays in registers
        uint32_t lvi[ROW_QUADS][4];
        float sv[ROW_QUADS][4], qv[ROW_QUADS][4], old[ROW_QUADS][4];
        const bool more[ROW_QUADS] = {true, n > 4, n > 8};
#pragma unroll
        for (uint32_t h = 0; h < ROW_QUADS; h++)
            if (more[h]) {
                quad(w.legal_value + lo + 4 * h, lvi[h]);
                quad(st + lo + 4 * h, sv[h]);
                if (MODE == MODE_REGRET) quad(w.regret + lo + 4 * h, old[h]);
            }
        // A cell past the row's end is like one without a successor, then not stored.
#pragma unroll
        for (uint32_t h = 0; h < ROW_QUADS; h++)
            if (more[h])
#pragma unroll
                for (uint32_t k = 0; k < 4; k++) {
                    if (4 * h + k >= n) lvi[h][k] = 0xffffffffu;
                    const bool live = lvi[h][k] != 0xffffffffu;
                    const float x = get(live ? lvi[h][k] : q.out);
                    qv[h][k] = live ? x : 0.0f;
                }
        float base = 0.0f;
#pragma unroll
        for (uint32_t h = 0; h < ROW_QUADS; h++)
            if (more[h])
#pragma unroll
                for (uint32_t k = 0; k < 4; k++)
                    base = lvi[h][k] != 0xffffffffu ? base + qv[h][k] * sv[h][k] : base;
        put(q.out, base);
        if (MODE == MODE_VALUE) return;
        float total = 0.0f;
#pragma unroll
        for (uint32_t h = 0; h < ROW_QUADS; h++)
            if (more[h]) {
#pragma unroll
                for (uint32_t k = 0; k < 4; k++) {
                    float delta = 0.0f;
                    delta += qv[h][k];  // (zero without a successor)
                    delta -= base;
                    const float r = old[h][k] * (old[h][k] > 0.0f ? da : db) + delta;
                    old[h][k] = r;
                    sv[h][k] = fmaxf(r + predict * delta, EPSF);
                    total = 4 * h + k < n ? total + sv[h][k] : total;
                }
                store_quad(w.regret + lo + 4 * h, old[h], n - 4 * h);
            }
        const bool pos = total > 0.0f;
        const float inv = pos ? 1.0f / total : 1.0f;
#pragma unroll
        for (uint32_t h = 0; h < ROW_QUADS; h++)
            if (more[h]) {
#pragma unroll
                for (uint32_t k = 0; k < 4; k++) sv[h][k] = pos ? sv[h][k] * inv : sv[h][k];
                store_quad(w.cur + lo + 4 * h, sv[h], n - 4 * h);
            }
        return;
    }
    // Longer rows: the same arithmetic in three batched passes (base; update,
    // with cur holding the unnormalised value; normalisation).
    float base = 0.0f;
    for (uint32_t c0 = 0; c0 < n; c0 += ROW_BATCH) {
        const uint32_t m = n - c0 < ROW_BATCH ? n - c0 : ROW_BATCH;
        uint32_t lvi[ROW_BATCH];
        float sv[ROW_BATCH], qv[ROW_BATCH];
#pragma unroll
        for (uint32_t k = 0; k < ROW_BATCH; k++)
            if (k < m) {
                lvi[k] = w.legal_value[lo + c0 + k];
                sv[k] = st[lo + c0 + k];
            }
#pragma unroll
        for (uint32_t k = 0; k < ROW_BATCH; k++)
            if (k < m) qv[k] = lvi[k] != 0xffffffffu ? get(lvi[k]) : 0.0f;
#pragma unroll
        for (uint32_t k = 0; k < ROW_BATCH; k++)
            if (k < m && lvi[k] != 0xffffffffu) base += qv[k] * sv[k];
    }
    put(q.out, base);
    if (MODE == MODE_VALUE) return;
    float total = 0.0f;
    for (uint32_t c0 = 0; c0 < n; c0 += ROW_BATCH) {
        const uint32_t m = n - c0 < ROW_BATCH ? n - c0 : ROW_BATCH;
        uint32_t lvi[ROW_BATCH];
        float qv[ROW_BATCH], old[ROW_BATCH];
#pragma unroll
        for (uint32_t k = 0; k < ROW_BATCH; k++)
            if (k < m) {
                lvi[k] = w.legal_value[lo + c0 + k];
                old[k] = w.regret[lo + c0 + k];
            }
#pragma unroll
        for (uint32_t k = 0; k < ROW_BATCH; k++)
            if (k < m) qv[k] = lvi[k] != 0xffffffffu ? get(lvi[k]) : 0.0f;
#pragma unroll
        for (uint32_t k = 0; k < ROW_BATCH; k++)
            if (k < m) {
                float delta = 0.0f;
                if (lvi[k] != 0xffffffffu) delta += qv[k];
                delta -= base;
                float r = old[k] * (old[k] > 0.0f ? da : db) + delta;
                w.regret[lo + c0 + k] = r;
                float v = fmaxf(r + predict * delta, EPSF);
                w.cur[lo + c0 + k] = v;
                total += v;
            }
    }
    if (total > 0.0f) {
        const float inv = 1.0f / total;
        for (uint32_t c0 = 0; c0 < n; c0 += ROW_BATCH) {
            const uint32_t m = n - c0 < ROW_BATCH ? n - c0 : ROW_BATCH;
            float cu[ROW_BATCH];
#pragma unroll
            for (uint32_t k = 0; k < ROW_BATCH; k++)
                if (k < m) cu[k] = w.cur[lo + c0 + k];
#pragma unroll
            for (uint32_t k = 0; k < ROW_BATCH; k++)
                if (k < m) w.cur[lo + c0 + k] = cu[k] * inv;
        }
    }
}

// Leaf values and the bottom-up value sweep of one subtree unit for traverser
// p, one workgroup per unit: leaf values first (net value x opponent reach
// mass, engine/src/search.rs:1587-1636), then levels from the deepest up, with
// the fused regret/DCFR update at the traverser's rows.
template <int MODE, bool LDSV>
__global__ __launch_bounds__(BLOCK) void k_sweep(WaveDev w, uint32_t unit0, const float* head_out, uint32_t heads,
                                               int p, float da, float db, float predict) {
    extern __shared__ float lds_vals[];  // the unit's value window of player p (when LDSV)
    const UnitDev u = w.units[unit0 + blockIdx.x];
    const int opp = 1 - p;
    // The player's fields by select, not by index: indexing the record's
    // arrays with the run-time p would place the record in scratch memory.
    const uint32_t vw = p ? u.vwin[1] : u.vwin[0];
    const uint32_t leaf0 = p ? u.leaf0[1] : u.leaf0[0], leaf1 = p ? u.leaf1[1] : u.leaf1[0];
    // The deepest level's bounds and each thread's first record of it are
    // fetched before the leaf phase: they do not depend on its values.
    const BackRec* back = w.back_rec[p];
    const uint32_t* blvl = w.back_lvl[p] + u.lvl0;
    const uint32_t t = threadIdx.x;
    uint32_t l = u.nlevels;
    uint32_t e = l ? blvl[l] : 0, b = l ? blvl[l - 1] : 0;
    BackRec q{};
    if (l && b + t < e) q = back[b + t];
    // Network leaves: one value slot per thread, LEAF_BATCH slots per thread
    // in flight (their records, then the values they name; slots past the end
    // repeat the last and are not stored).
    const LeafRec* leaves = w.leaf_rec[p];
    for (uint32_t k0 = leaf0; k0 < leaf1; k0 += LEAF_BATCH * BLOCK) {
        LeafRec lr[LEAF_BATCH];
        float h[LEAF_BATCH], m[LEAF_BATCH];
#pragma unroll
        for (uint32_t j = 0; j < LEAF_BATCH; j++) lr[j] = leaves[min(k0 + j * BLOCK + threadIdx.x, leaf1 - 1)];
#pragma unroll
        for (uint32_t j = 0; j < LEAF_BATCH; j++) {
            h[j] = head_out[lr[j].head];
            m[j] = w.mass[lr[j].mass];
        }
#pragma unroll
        for (uint32_t j = 0; j < LEAF_BATCH; j++)
            if (k0 + j * BLOCK + threadIdx.x < leaf1) {
                const float v = h[j] * m[j];
                if (!LDSV || lr[j].exported) w.vals[lr[j].out] = v;
                if (LDSV) lds_vals[lr[j].out - vw] = v;
            }
    }
    for (uint32_t x = u.term0 + threadIdx.x; x < u.term1; x += blockDim.x) {
        const uint32_t te = w.unit_term[x], k = te & TERM_INDEX;
        const bool to_hbm = !LDSV || (te & term_export(p));
        uint32_t node = w.term_node[k];
        const float* ro = w.reach + w.reach_base[2 * node + opp];
        float m = 0.0f;
        for (uint32_t c = 0; c < w.nc[2 * node + opp]; c++) m += ro[c];
        float uu = (w.node_meta[node] >> 2) == (uint32_t)p ? w.term_util[k] : -w.term_util[k];
        const uint32_t ob = w.vals_base[2 * node + p];
        for (uint32_t c = 0; c < w.nc[2 * node + p]; c++) {
            if (to_hbm) w.vals[ob + c] = uu * m;
            if (LDSV) lds_vals[ob + c - vw] = uu * m;
        }
    }
    __syncthreads();
    // Levels from the deepest up. Each thread's rows form one stream across
    // the levels: the record of its next row (in this level, else its first
    // in the next level up) is fetched while the current row runs.
    while (l-- > 0) {
        const uint32_t lb = b, le = e;
        if (l) {
            e = lb;
            b = blvl[l - 1];
        }
        if (lb + t >= le && l && b + t < e) q = back[b + t];
        for (uint32_t k = lb + t; k < le;) {
            const uint32_t kn = k + blockDim.x;
            BackRec qn{};
            if (kn < le)
                qn = back[kn];
            else if (l && b + t < e)
                qn = back[b + t];
            backprop_row<MODE, LDSV>(w, p, q, da, db, predict, w.snap, lds_vals, vw);
            q = qn;
            k = kn;
        }
        __syncthreads();
    }
}

void launch_sweep(const WaveDev& w, uint32_t unit0, uint32_t n, const float* head_out, uint32_t heads, int traverser,
                  int mode, float da, float db, float predict, hipStream_t s) {
    if (!n) return;
    const size_t lds = (size_t)w.max_vwin * sizeof(float);
    const bool staged = w.unit_lds && lds <= SWEEP_LDS_MAX;
#define WC_SWEEP(M, L)                                                                                          \
    hipLaunchKernelGGL((k_sweep<M, L>), dim3(n), dim3(BLOCK), L ? lds : 0, s, w, unit0, head_out, heads, traverser, \
                       da, db, predict)
    if (mode == MODE_VALUE) {
        if (staged)
            WC_SWEEP(MODE_VALUE, true);
        else
            WC_SWEEP(MODE_VALUE, false);
    } else {
        if (staged)
            WC_SWEEP(MODE_REGRET, true);
        else
            WC_SWEEP(MODE_REGRET, false);
    }
#undef WC_SWEEP
}

// Top-region values at one depth, all trees together: one row per thread.
template <int MODE>
__global__ __launch_bounds__(BLOCK) void k_back_rows(WaveDev w, const BackRec* rows, uint32_t n, int p, float da,
                                                   float db, float predict) {
    uint32_t k = blockIdx.x * blockDim.x + threadIdx.x;
    if (k < n) backprop_row<MODE, false>(w, p, rows[k], da, db, predict, w.snap, nullptr, 0);
}

void launch_back_rows(const WaveDev& w, const BackRec* rows, uint32_t n, int traverser, int mode, float da,
                      float db, float predict, hipStream_t s) {
    if (!n) return;
    if (mode == MODE_VALUE)
        hipLaunchKernelGGL(k_back_rows<MODE_VALUE>, dim3(grid_for(n, TOP_BLOCK)), dim3(TOP_BLOCK), 0, s, w, rows, n,
                           traverser, da, db, predict);
    else
        hipLaunchKernelGGL(k_back_rows<MODE_REGRET>, dim3(grid_for(n, TOP_BLOCK)), dim3(TOP_BLOCK), 0, s, w, rows, n,
                           traverser, da, db, predict);
}

// Two top depths in one launch: each workgroup takes one chunk's rows of the
// deeper depth, then (after a block barrier: the values it wrote are read by
// the same workgroup) that chunk's rows of the shallower depth. Sparing the
// launch boundary saves its fixed cost, about as long as a depth's own rows
// take.
template <int MODE>
__global__ __launch_bounds__(BLOCK) void k_back_pair(WaveDev w, const BackRec* rows, const uint32_t* off,
                                                   uint32_t chunks, int p, float da, float db, float predict) {
    const uint32_t k = blockIdx.x;
    for (uint32_t i = off[k] + threadIdx.x; i < off[k + 1]; i += blockDim.x)
        backprop_row<MODE, false>(w, p, rows[i], da, db, predict, w.snap, nullptr, 0);
    __syncthreads();
    const uint32_t* o = off + chunks + 1;
    for (uint32_t i = o[k] + threadIdx.x; i < o[k + 1]; i += blockDim.x)
        backprop_row<MODE, false>(w, p, rows[i], da, db, predict, w.snap, nullptr, 0);
}

void launch_back_pair(const WaveDev& w, const BackRec* rows, const uint32_t* off, uint32_t chunks, int traverser,
                      int mode, float da, float db, float predict, hipStream_t s) {
    if (!chunks) return;
    if (mode == MODE_VALUE)
        hipLaunchKernelGGL(k_back_pair<MODE_VALUE>, dim3(chunks), dim3(TOP_BLOCK), 0, s, w, rows, off, chunks,
                           traverser, da, db, predict);
    else
        hipLaunchKernelGGL(k_back_pair<MODE_REGRET>, dim3(chunks), dim3(TOP_BLOCK), 0, s, w, rows, off, chunks,
                           traverser, da, db, predict);
}

// Average strategy: sum / row sum, uniform when the sum is not positive, the
// literal current strategy for a player whose sum was never updated
// (engine/src/search.rs:899-938).
__global__ void k_normalize(WaveDev w, int touched0, int touched1) {
    uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= w.ndec[0] + w.ndec[1]) return;
    int p;
    AccRec q = decision_row(w, i, &p);
    uint32_t lo = q.lo, hi = q.lo + q.n;
    const bool touched = p ? touched1 : touched0;
    if (q.n - 1 < ROW_BATCH) {  // 1 to 12 cells: the row's loads issued together, then the same sum and quotients
        const float* src = (touched ? scalar(w.sum) : scalar(w.cur)) + lo;
        const bool more[ROW_QUADS] = {true, q.n > 4, q.n > 8};
        float x[ROW_QUADS][4];
#pragma unroll
        for (uint32_t h = 0; h < ROW_QUADS; h++)
            if (more[h]) quad(src + 4 * h, x[h]);
        float s = 0.0f;
#pragma unroll
        for (uint32_t h = 0; h < ROW_QUADS; h++)
            if (more[h])
#pragma unroll
                for (uint32_t k = 0; k < 4; k++) s = 4 * h + k < q.n ? s + x[h][k] : s;
        const float u = 1.0f / (float)q.n;
#pragma unroll
        for (uint32_t h = 0; h < ROW_QUADS; h++)
            if (more[h]) {
#pragma unroll
                for (uint32_t k = 0; k < 4; k++) {
                    const float y = s > 0.0f ? x[h][k] / s : u;
                    x[h][k] = touched ? y : x[h][k];
                }
                store_quad(w.snap + lo + 4 * h, x[h], q.n - 4 * h);
            }
        return;
    }
    if (!touched) {
        for (uint32_t g = lo; g < hi; g++) w.snap[g] = w.cur[g];
        return;
    }
    float s = 0.0f;
    for (uint32_t g = lo; g < hi; g++) s += w.sum[g];
    float k = (float)(hi > lo ? hi - lo : 1);
    for (uint32_t g = lo; g < hi; g++) w.snap[g] = s > 0.0f ? w.sum[g] / s : 1.0f / k;
}

void launch_normalize(const WaveDev& w, int touched0, int touched1, hipStream_t s) {
    uint32_t n = w.ndec[0] + w.ndec[1];
    if (n) hipLaunchKernelGGL(k_normalize, dim3(grid_for(n)), dim3(BLOCK), 0, s, w, touched0, touched1);
}

// Normalised beliefs at every exit, f16 (the carry store, engine/src/gpu/client.rs:20-111).
// One wavefront per (exit, player), task 2 e + p: its reach slot and carry
// offsets (scalar loads), then 64 configs at a time; the mass is summed in
// config order from the lanes' values.
__global__ __launch_bounds__(64) void k_gather_carry(WaveDev w, const float* reach, int slot) {
    const uint32_t lane = threadIdx.x, t = blockIdx.x;
    if (t >= 2 * w.nexit) return;  // wave-uniform
    const float* r = reach + w.exit_reach[t];
    const uint32_t cb = w.exit_coff[t], n = w.exit_coff[t + 1] - cb;
    const float v0 = lane < n ? r[lane] : 0.0f;
    float tot = 0.0f;
    for (uint32_t c0 = 0; c0 < n; c0 += 64) {
        const float x = c0 ? (c0 + lane < n ? r[c0 + lane] : 0.0f) : v0;
        tot = lane_sum_in_order(tot, x, n - c0 < 64 ? n - c0 : 64);
    }
    float scale, flat;
    if (tot > SMOOTHF) {
        scale = 1.0f / tot;
        flat = 0.0f;
    } else {
        scale = 0.0f;
        flat = 1.0f / (float)(n > 0 ? n : 1);
    }
    uint16_t* dst = w.carry + (size_t)slot * w.snapshot_configs + cb;
    for (uint32_t c = lane; c < n; c += 64) dst[c] = f32_to_f16_rn((c < 64 ? v0 : r[c]) * scale + flat);
}

void launch_gather_carry(const WaveDev& w, const float* reach, int slot, hipStream_t s) {
    const size_t tasks = (size_t)w.nexit * 2;
    // one wavefront per task, one per workgroup: a wavefront that finishes
    // frees its slot at once
    if (tasks) hipLaunchKernelGGL(k_gather_carry, dim3((uint32_t)tasks), dim3(64), 0, s, w, reach, slot);
}

__global__ void k_collect_root(WaveDev w, int root, int p) {
    const TreeDev t = w.trees[blockIdx.x];
    if (root >= (int)t.nroots) return;
    uint32_t n = p ? t.n1 : t.n0;
    float* dst = w.root_values + t.root_value0 + (size_t)root * (t.n0 + t.n1) + (p ? t.n0 : 0);
    const float* src = w.vals + w.vals_base[2 * t.node0 + p];
    for (uint32_t c = threadIdx.x; c < n; c += blockDim.x) dst[c] = src[c];
}

void launch_collect_root(const WaveDev& w, int root, int player, hipStream_t s) {
    hipLaunchKernelGGL(k_collect_root, dim3(w.ntrees), dim3(BLOCK), 0, s, w, root, player);
}

// ------------------------------------------------------- leaf MLP (MFMA)


template <int PREC>
__global__ void k_to16(const float* src, uint16_t* dst, uint32_t rows, uint32_t K, int transposed, size_t plane) {
    size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= (size_t)rows * K) return;
    uint32_t r = (uint32_t)(i / K), k = (uint32_t)(i % K);
    float v = transposed ? src[(size_t)k * rows + r] : src[i];
    store_operand<PREC>(dst, frag_off(r, k, K), v, plane);
}

void launch_to16(int precision, const float* src, void* dst, uint32_t rows, uint32_t K, bool transposed,
                 hipStream_t s) {
    size_t n = (size_t)rows * K;
    if (!n) return;
    const size_t plane = (size_t)gemm_rows(rows) * K;  // compensated f16: the lo plane follows the hi plane
#define WC_TO16(P)                                                                                              \
    hipLaunchKernelGGL(k_to16<P>, dim3(grid_for(n)), dim3(BLOCK), 0, s, src, (uint16_t*)dst, rows, K, (int)transposed, \
                       plane)
    if (precision == WC_F16)
        WC_TO16(WC_F16);
    else if (precision == WC_BF16)
        WC_TO16(WC_BF16);
    else
        WC_TO16(WC_F16X);
#undef WC_TO16
}

// 16x16x32 MFMA step over a 64 x 64 wave tile: acc[a][b] += A(a) B(b)^T.
template <int PREC>
__device__ __forceinline__ void mfma_step(float4v (&acc)[4][4], const uint4 (&af)[4], const uint4 (&bf)[4]) {
#pragma unroll
    for (int a = 0; a < 4; a++)
#pragma unroll
        for (int b = 0; b < 4; b++) {
            if (PREC == WC_F16)
                acc[a][b] = __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(half8, af[a]),
                                                                   __builtin_bit_cast(half8, bf[b]), acc[a][b], 0, 0,
                                                                   0);
            else
                acc[a][b] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, af[a]),
                                                                    __builtin_bit_cast(bf16x8, bf[b]), acc[a][b], 0,
                                                                    0, 0);
        }
}

// One 16x16x32 MFMA: acc += A(a) B(b)^T.
template <int PREC>
__device__ __forceinline__ float4v mfma_step16(const uint4& a, const uint4& b, const float4v& acc) {
    if (PREC == WC_F16)
        return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(half8, a), __builtin_bit_cast(half8, b), acc,
                                                      0, 0, 0);
    else
        return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b),
                                                       acc, 0, 0, 0);
}

// Fragment-major MFMA GEMM. A 128 x 128 output tile per workgroup, 64 x 64 per
// wavefront (4 x 4 16x16x32 tiles). Both operands are fragment-major, so each
// of a step's 8 fragment loads is one contiguous 1 KB read. Two fragment sets
// ping-pong: while one step's 16 MFMAs run, the next step's loads are in
// flight (the loop is unrolled by two so the compiler waits only for the set
// it is about to use). The epilogue adds the bias, applies ReLU and stores
// either the next layer's 16-bit fragment-major operand or row-major f32.
template <int PREC, bool RELU, bool OUT16>
__global__ __launch_bounds__(256) void k_gemm(const uint16_t* __restrict__ X, uint32_t K,
                                              const uint16_t* __restrict__ Wt, const float* __restrict__ bias,
                                              uint32_t N, void* __restrict__ Y, uint32_t M,
                                              const uint32_t* __restrict__ tile_n) {
    const uint32_t lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    if (tile_n && blockIdx.y * GEMM_ROWS >= tile_n[blockIdx.x]) return;  // block-uniform
    const uint32_t m0 = blockIdx.x * GEMM_ROWS + (wave & 1) * 64;
    const uint32_t n0 = blockIdx.y * GEMM_ROWS + (wave >> 1) * 64;
    const uint32_t ks = K >> 5;  // 32-wide k steps
    float4v acc[4][4];
#pragma unroll
    for (int a = 0; a < 4; a++)
#pragma unroll
        for (int b = 0; b < 4; b++) acc[a][b] = float4v{0.0f, 0.0f, 0.0f, 0.0f};
    // Fragment (block, step) lives at ((block * ks + step) * 64 + lane) * 8.
    const uint16_t* ap = X + ((size_t)(m0 >> 4) * ks * 64 + lane) * 8;
    const uint16_t* bp = Wt + ((size_t)(n0 >> 4) * ks * 64 + lane) * 8;
    const size_t blk = (size_t)ks * 64 * 8;  // halves between consecutive 16-row blocks
    uint4 af[4], bf[4], an[4], bn[4];
    auto load = [&](uint4 (&fa)[4], uint4 (&fb)[4], uint32_t step) {
#pragma unroll
        for (int a = 0; a < 4; a++) fa[a] = *(const uint4*)(ap + a * blk + (size_t)step * 512);
#pragma unroll
        for (int b = 0; b < 4; b++) fb[b] = *(const uint4*)(bp + b * blk + (size_t)step * 512);
    };
    load(af, bf, 0);
    uint32_t st = 0;
    for (; st + 2 <= ks; st += 2) {
        load(an, bn, st + 1);
        __builtin_amdgcn_sched_barrier(0);
        mfma_step<PREC>(acc, af, bf);
        __builtin_amdgcn_sched_barrier(0);
        load(af, bf, st + 2 < ks ? st + 2 : st + 1);  // past the end: re-read a valid step, unused
        __builtin_amdgcn_sched_barrier(0);
        mfma_step<PREC>(acc, an, bn);
        __builtin_amdgcn_sched_barrier(0);
    }
    if (st < ks) mfma_step<PREC>(acc, af, bf);  // odd step count: af holds the last step
    const uint32_t li = lane & 15, kb = lane >> 4;
#pragma unroll
    for (int a = 0; a < 4; a++)
#pragma unroll
        for (int b = 0; b < 4; b++) {
            uint32_t col = n0 + b * 16 + li;
            if (col >= N) continue;
            float bv = bias[col];
#pragma unroll
            for (int v = 0; v < 4; v++) {
                uint32_t row = m0 + a * 16 + kb * 4 + v;
                if (row >= M) continue;
                float y = acc[a][b][v] + bv;
                if (RELU) y = y > 0.0f ? y : 0.0f;
                if (OUT16)
                    ((uint16_t*)Y)[frag_off(row, col, N)] = PREC == WC_F16 ? f32_to_f16_rn(y) : f32_to_bf16_rn(y);
                else
                    ((float*)Y)[(size_t)row * N + col] = y;
            }
        }
}

// Compensated f16 GEMM: each operand is an f16 pair hi + lo in two planes
// (xplane / wplane elements apart), each product is taken as lo hi + hi lo +
// hi hi (f32 accumulation), the output likewise split when 16-bit. Tiles as
// k_gemm, without its load pipelining: this is the accuracy mode.
template <bool RELU, bool OUT16>
__global__ __launch_bounds__(256) void k_gemm_x(const uint16_t* __restrict__ X, uint32_t K,
                                                const uint16_t* __restrict__ Wt, const float* __restrict__ bias,
                                                uint32_t N, void* __restrict__ Y, uint32_t M,
                                                const uint32_t* __restrict__ tile_n, size_t xplane, size_t wplane,
                                                size_t yplane) {
    const uint32_t lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    if (tile_n && blockIdx.y * GEMM_ROWS >= tile_n[blockIdx.x]) return;  // block-uniform
    const uint32_t m0 = blockIdx.x * GEMM_ROWS + (wave & 1) * 64;
    const uint32_t n0 = blockIdx.y * GEMM_ROWS + (wave >> 1) * 64;
    const uint32_t ks = K >> 5;
    float4v acc[4][4];
#pragma unroll
    for (int a = 0; a < 4; a++)
#pragma unroll
        for (int b = 0; b < 4; b++) acc[a][b] = float4v{0.0f, 0.0f, 0.0f, 0.0f};
    const uint16_t* ap = X + ((size_t)(m0 >> 4) * ks * 64 + lane) * 8;
    const uint16_t* bp = Wt + ((size_t)(n0 >> 4) * ks * 64 + lane) * 8;
    const size_t blk = (size_t)ks * 64 * 8;
    for (uint32_t st = 0; st < ks; st++) {
        uint4 ah[4], al[4], bh[4], bl[4];
#pragma unroll
        for (int a = 0; a < 4; a++) {
            ah[a] = *(const uint4*)(ap + a * blk + (size_t)st * 512);
            al[a] = *(const uint4*)(ap + xplane + a * blk + (size_t)st * 512);
        }
#pragma unroll
        for (int b = 0; b < 4; b++) {
            bh[b] = *(const uint4*)(bp + b * blk + (size_t)st * 512);
            bl[b] = *(const uint4*)(bp + wplane + b * blk + (size_t)st * 512);
        }
#pragma unroll
        for (int a = 0; a < 4; a++)
#pragma unroll
            for (int b = 0; b < 4; b++) {
                acc[a][b] = mfma_step16<WC_F16>(al[a], bh[b], acc[a][b]);
                acc[a][b] = mfma_step16<WC_F16>(ah[a], bl[b], acc[a][b]);
                acc[a][b] = mfma_step16<WC_F16>(ah[a], bh[b], acc[a][b]);
            }
    }
    const uint32_t li = lane & 15, kb = lane >> 4;
#pragma unroll
    for (int a = 0; a < 4; a++)
#pragma unroll
        for (int b = 0; b < 4; b++) {
            uint32_t col = n0 + b * 16 + li;
            if (col >= N) continue;
            float bv = bias[col];
#pragma unroll
            for (int v = 0; v < 4; v++) {
                uint32_t row = m0 + a * 16 + kb * 4 + v;
                if (row >= M) continue;
                float y = acc[a][b][v] + bv;
                if (RELU) y = y > 0.0f ? y : 0.0f;
                if (OUT16)
                    store_operand<WC_F16X>(Y, frag_off(row, col, N), y, yplane);
                else
                    ((float*)Y)[(size_t)row * N + col] = y;
            }
        }
}

void launch_gemm16(int precision, const void* X, uint32_t K, const void* Wt, const float* b, uint32_t N, void* Y,
                   uint32_t M, bool relu, bool out16, hipStream_t s, const uint32_t* tile_n) {
    if (M == 0 || N == 0) return;
    dim3 grid(gemm_rows(M) / GEMM_ROWS, gemm_rows(N) / GEMM_ROWS);
    if (precision == WC_F16X) {
        const size_t xp = (size_t)gemm_rows(M) * K, wp = (size_t)gemm_rows(N) * K, yp = (size_t)gemm_rows(M) * N;
        const uint16_t* x = (const uint16_t*)X;
        const uint16_t* wt = (const uint16_t*)Wt;
#define WC_GEMMX(R, O) \
    hipLaunchKernelGGL((k_gemm_x<R, O>), grid, dim3(256), 0, s, x, K, wt, b, N, Y, M, tile_n, xp, wp, yp)
        if (relu && out16)
            WC_GEMMX(true, true);
        else if (relu)
            WC_GEMMX(true, false);
        else if (out16)
            WC_GEMMX(false, true);
        else
            WC_GEMMX(false, false);
#undef WC_GEMMX
        return;
    }
    const uint16_t* x = (const uint16_t*)X;
    const uint16_t* wt = (const uint16_t*)Wt;
#define WC_GEMM(P, R, O) hipLaunchKernelGGL((k_gemm<P, R, O>), grid, dim3(256), 0, s, x, K, wt, b, N, Y, M, tile_n)
    if (precision == WC_F16) {
        if (relu && out16)
            WC_GEMM(WC_F16, true, true);
        else if (relu)
            WC_GEMM(WC_F16, true, false);
        else if (out16)
            WC_GEMM(WC_F16, false, true);
        else
            WC_GEMM(WC_F16, false, false);
    } else {
        if (relu && out16)
            WC_GEMM(WC_BF16, true, true);
        else if (relu)
            WC_GEMM(WC_BF16, true, false);
        else if (out16)
            WC_GEMM(WC_BF16, false, true);
        else
            WC_GEMM(WC_BF16, false, false);
    }
#undef WC_GEMM
}


// ------------------------------------------------------------ two-tower net
//
// The two-tower leaf value of row r and infostate c is <f(c), h(r)> + b_read
// with h the public tower's output for the row's query and f(c) the private
// tower's output for the infostate's features times the readout weight
// (elementwise). f is formed once per wave and weight bank.

// F[c][k] = Hp[c][k] * wread[k]; the 16-bit nets round the product to the
// operand type (Hp fragment-major with K = width, F row-major), float32 keeps it.
template <int PREC>
__global__ void k_tower_f(const void* __restrict__ Hp, uint32_t width, uint32_t ncfg, const float* __restrict__ wread,
                          void* __restrict__ F) {
    const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= (size_t)ncfg * width) return;
    const uint32_t c = (uint32_t)(i / width), k = (uint32_t)(i % width);
    if (PREC == WC_PRECISE) {
        ((float*)F)[i] = ((const float*)Hp)[i] * wread[k];
        return;
    }
    const uint16_t hv = ((const uint16_t*)Hp)[frag_off(c, k, width)];
    float h;
    if (PREC == WC_F16)
        h = (float)__builtin_bit_cast(_Float16, hv);
    else
        h = __uint_as_float((uint32_t)hv << 16);
    const float f = h * wread[k];
    ((uint16_t*)F)[i] = PREC == WC_F16 ? f32_to_f16_rn(f) : f32_to_bf16_rn(f);
}

void launch_tower_f(int precision, const void* Hp, uint32_t width, uint32_t ncfg, const float* wread, void* F,
                    hipStream_t s) {
    const size_t n = (size_t)ncfg * width;
    if (!n) return;
    if (precision == WC_PRECISE)
        hipLaunchKernelGGL(k_tower_f<WC_PRECISE>, dim3(grid_for(n)), dim3(BLOCK), 0, s, Hp, width, ncfg, wread, F);
    else if (precision == WC_F16)
        hipLaunchKernelGGL(k_tower_f<WC_F16>, dim3(grid_for(n)), dim3(BLOCK), 0, s, Hp, width, ncfg, wread, F);
    else
        hipLaunchKernelGGL(k_tower_f<WC_BF16>, dim3(grid_for(n)), dim3(BLOCK), 0, s, Hp, width, ncfg, wread, F);
}

// Float32 readout: one workgroup per readout block of player p, one thread
// per (row, config) entry, the sum from b_read in k order as the CPU net forms
// it (engine/src/net.rs:844-853 pattern: bias, then += f[k] h[k]).
__global__ __launch_bounds__(BLOCK) void k_tower_dense_exact(WaveDev w, int p, const float* __restrict__ H,
                                                           uint32_t width, const float* __restrict__ F, float bread,
                                                           float* __restrict__ tv) {
    const TowerBlock b = w.tower_blk[p][blockIdx.x];
    const uint32_t nc = b.chi - b.clo, n = (b.r1 - b.r0) * nc;
    for (uint32_t x = threadIdx.x; x < n; x += blockDim.x) {
        const uint32_t r = b.r0 + x / nc, c = b.clo + x % nc;
        const float* h = H + (size_t)r * width;
        const float* f = F + (size_t)c * width;
        float acc = bread;
        for (uint32_t j = 0; j < width; j++) acc += f[j] * h[j];
        tv[b.dbase + x] = acc;
    }
}

// 16-bit readout on MFMA: one wavefront per 64 x 64 tile of a readout block,
// 4 x 4 16x16x32 tiles over the width. A = 16-row blocks of the public-tower
// output H (whole fragments: tile rows are 16-aligned; blocks past the tree's
// last row re-read its last block), B = 16 configs' F rows per tile (configs
// past the block re-read its last config). Entries outside the block are not
// stored.
template <int PREC>
__global__ __launch_bounds__(BLOCK) void k_tower_dense(WaveDev w, int p, const uint16_t* __restrict__ H,
                                                     uint32_t width, const uint16_t* __restrict__ F, float bread,
                                                     float* __restrict__ tv) {
    const uint32_t k = __builtin_amdgcn_readfirstlane((blockIdx.x * blockDim.x + threadIdx.x) >> 6);
    if (k >= w.ntower_unit[p]) return;  // wave-uniform
    const uint32_t lane = threadIdx.x & 63, i = lane & 15, q = lane >> 4;
    const TowerUnit u = w.tower_unit[p][k];
    const TowerBlock b = w.tower_blk[p][u.block];
    const uint32_t ks = width >> 5, last_blk = (b.r1 - 1) & ~15u;
    const uint16_t* ap[4];
    const uint16_t* bp[4];
#pragma unroll
    for (int t = 0; t < 4; t++) {
        const uint32_t rb = min(u.row + 16 * t, last_blk);
        ap[t] = H + ((size_t)(rb >> 4) * ks * 64 + lane) * 8;  // fragment (block, step) at + step * 512
        const uint32_t c = min(u.cfg + 16 * t + i, b.chi - 1);
        bp[t] = F + (size_t)c * width + 8 * q;  // this lane's 8 columns of step s at + 32 s
    }
    float4v acc[4][4];
#pragma unroll
    for (int a = 0; a < 4; a++)
#pragma unroll
        for (int c = 0; c < 4; c++) acc[a][c] = float4v{0.0f, 0.0f, 0.0f, 0.0f};
    uint4 fa[4], fb[4], na[4], nb[4];
    auto load = [&](uint4 (&xa)[4], uint4 (&xb)[4], uint32_t s) {
#pragma unroll
        for (int t = 0; t < 4; t++) {
            xa[t] = *(const uint4*)(ap[t] + (size_t)s * 512);
            xb[t] = *(const uint4*)(bp[t] + 32 * s);
        }
    };
    auto step = [&](const uint4 (&xa)[4], const uint4 (&xb)[4]) {
#pragma unroll
        for (int a = 0; a < 4; a++)
#pragma unroll
            for (int c = 0; c < 4; c++) acc[a][c] = mfma_step16<PREC>(xa[a], xb[c], acc[a][c]);
    };
    load(fa, fb, 0);
    uint32_t s = 0;
    for (; s + 2 <= ks; s += 2) {
        load(na, nb, s + 1);
        __builtin_amdgcn_sched_barrier(0);
        step(fa, fb);
        __builtin_amdgcn_sched_barrier(0);
        load(fa, fb, s + 2 < ks ? s + 2 : s + 1);  // past the end: re-read a valid step, unused
        __builtin_amdgcn_sched_barrier(0);
        step(na, nb);
        __builtin_amdgcn_sched_barrier(0);
    }
    if (s < ks) step(fa, fb);
    const uint32_t nc = b.chi - b.clo;
#pragma unroll
    for (int c = 0; c < 4; c++) {
        const uint32_t cfg = u.cfg + 16 * c + i;
        if (cfg >= b.chi) continue;
#pragma unroll
        for (int a = 0; a < 4; a++)
#pragma unroll
            for (int v = 0; v < 4; v++) {
                const uint32_t r = u.row + 16 * a + 4 * q + v;
                if (r >= b.r0 && r < b.r1) tv[b.dbase + (r - b.r0) * nc + (cfg - b.clo)] = acc[a][c][v] + bread;
            }
    }
}

void launch_tower_head(const WaveDev& w, int player, int precision, const void* H, uint32_t width, const void* F,
                       float bread, float* tv, hipStream_t s) {
    if (precision == WC_PRECISE) {
        if (w.ntower_blk[player])
            hipLaunchKernelGGL(k_tower_dense_exact, dim3(w.ntower_blk[player]), dim3(BLOCK), 0, s, w, player,
                               (const float*)H, width, (const float*)F, bread, tv);
        return;
    }
    if (!w.ntower_unit[player]) return;
    dim3 g(grid_for((size_t)w.ntower_unit[player] * 64));
    if (precision == WC_F16)
        hipLaunchKernelGGL(k_tower_dense<WC_F16>, g, dim3(BLOCK), 0, s, w, player, (const uint16_t*)H, width,
                           (const uint16_t*)F, bread, tv);
    else
        hipLaunchKernelGGL(k_tower_dense<WC_BF16>, g, dim3(BLOCK), 0, s, w, player, (const uint16_t*)H, width,
                           (const uint16_t*)F, bread, tv);
}

// ------------------------------------------------------- fused leaf network
//
// One launch runs the whole MLP, one pass of up to eight 16-row blocks per
// workgroup (the passes come from plan_chain): the pass's input operand is
// staged into LDS once, every trunk layer reads its input from LDS and writes
// its bias + ReLU output back over it (fragment-major, 16-bit: the next
// layer's operand), and the head writes row-major f32. Only the pass's input,
// the weights (shared by every pass, L2-resident) and the head outputs touch
// HBM.
//
// Products are computed transposed, D = W X^T: the weight fragment is the
// MFMA's A operand and the activation fragment its B operand, so lane l holds
// four consecutive output features 4 (l / 16) .. + 3 of one row l % 16 --
// one 8-byte LDS store per 16x16 tile in the next layer's fragment layout.
// Every output is the same f32 sum over the same 32-wide k steps, in the same
// order, as the layer-by-layer k_gemm, except in the partial-start mode, whose
// first layer adds the pooled columns' steps to the precomputed sum over the
// fixed columns (the same products, summed in another order).

constexpr uint32_t CHAIN_LDS_HALVES = GEMM_ROWS * CHAIN_MAX_WIDTH;

bool chain_fits(uint32_t in, uint32_t hidden, uint32_t layers) {
    return in % 32 == 0 && in <= CHAIN_MAX_WIDTH && hidden % 32 == 0 &&
           hidden <= CHAIN_WAVES * CHAIN_NB * 16 && layers >= 1 && layers <= CHAIN_MAX_LAYERS;
}

uint32_t chain_most(int precision) { return precision == WC_F16X ? CHAIN_PASS_BLOCKS / 2 : CHAIN_PASS_BLOCKS; }

// A compensated pass streams its head, both planes, from L2 for at most four
// row blocks, where the layer-by-layer product's tiles share it over 128 rows:
// under a wide head the fused net loses what its trunk gains. The line is on the
// columns a CU streams: the widest block's, or four blocks at a time its share
// of all. Fused against layer by layer, shapes of one to three layers 64 to 384
// wide (us): 4,000 rows with 567 heads 31 against 73 and with 1,000 39 against
// 65; 12,000 rows with 1,000 heads 115 against 111 and with 2,000 196 against
// 147; 30,000 rows with 768 heads 1.1 to 1.4 times as long; up to a block per CU
// even at about 1,500 to 2,000 heads (a row, 4,000 heads: 85 against 35).
bool chain_pays(int precision, uint32_t nrb, uint32_t widest, uint64_t columns, uint32_t cus) {
    if (precision != WC_F16X) return precision != WC_PRECISE;
    const uint64_t streamed = std::max<uint64_t>(widest, columns / (CHAIN_PASS_BLOCKS / 2 * cus));
    return streamed <= (nrb <= cus ? 1536 : 1024);
}

template <int PREC>
__device__ __forceinline__ float4v mfma16(const uint4& a, const uint4& b, const float4v& c) {
    if (PREC == WC_F16)
        return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(half8, a), __builtin_bit_cast(half8, b), c,
                                                      0, 0, 0);
    else
        return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b),
                                                       c, 0, 0, 0);
}

// acc[a][b] (a < RB, b < NB) = sum over ks steps of W(block b) X(rows 16a..)^T.
// xs: the LDS operand at this lane's fragment slot (fragment (a, s) at xs + (a
// ks + s) 512); wp: the wavefront's first weight block at this lane's slot
// (block b at wp + b wstride). Weight fragments (from L2) are fetched two
// steps ahead through a ring of four sets, activation fragments (from LDS) one
// step ahead through two; the loop is unrolled by four so every set keeps a
// fixed role. Loads past the last step re-read the last step (in bounds,
// unused).
template <int PREC, int NB, int RB, bool ZERO = true>
__device__ __forceinline__ void chain_kloop(float4v (&acc)[8][CHAIN_NB], const uint16_t* xs, uint32_t ks,
                                            const uint16_t* __restrict__ wp, size_t wstride) {
    if (ZERO) {  // else acc arrives holding the product's starting value
#pragma unroll
        for (int a = 0; a < RB; a++)
#pragma unroll
            for (int b = 0; b < NB; b++) acc[a][b] = float4v{0.0f, 0.0f, 0.0f, 0.0f};
    }
    uint4 xa[RB], xb[RB], w0[NB], w1[NB], w2[NB], w3[NB];
    auto ldw = [&](uint4 (&fw)[NB], uint32_t s) {
        s = s < ks ? s : ks - 1;
#pragma unroll
        for (int b = 0; b < NB; b++) fw[b] = *(const uint4*)(wp + b * wstride + (size_t)s * 512);
    };
    auto ldx = [&](uint4 (&fx)[RB], uint32_t s) {
        s = s < ks ? s : ks - 1;
#pragma unroll
        for (int a = 0; a < RB; a++) fx[a] = *(const uint4*)(xs + ((size_t)a * ks + s) * 512);
    };
    auto step = [&](const uint4 (&fx)[RB], const uint4 (&fw)[NB]) {
#pragma unroll
        for (int a = 0; a < RB; a++)
#pragma unroll
            for (int b = 0; b < NB; b++) acc[a][b] = mfma16<PREC>(fw[b], fx[a], acc[a][b]);
    };
    ldw(w0, 0);
    ldw(w1, 1);
    ldx(xa, 0);
    uint32_t s = 0;
    for (; s + 4 <= ks; s += 4) {
        ldw(w2, s + 2);
        ldx(xb, s + 1);
        __builtin_amdgcn_sched_barrier(0);
        step(xa, w0);
        __builtin_amdgcn_sched_barrier(0);
        ldw(w3, s + 3);
        ldx(xa, s + 2);
        __builtin_amdgcn_sched_barrier(0);
        step(xb, w1);
        __builtin_amdgcn_sched_barrier(0);
        ldw(w0, s + 4);
        ldx(xb, s + 3);
        __builtin_amdgcn_sched_barrier(0);
        step(xa, w2);
        __builtin_amdgcn_sched_barrier(0);
        ldw(w1, s + 5);
        ldx(xa, s + 4);
        __builtin_amdgcn_sched_barrier(0);
        step(xb, w3);
        __builtin_amdgcn_sched_barrier(0);
    }
    for (; s < ks; s++) {  // K not a multiple of 128: the last steps one at a time
        ldw(w0, s);
        ldx(xa, s);
        step(xa, w0);
    }
}

// The wavefront's share of one layer: 16-feature blocks blk0, blk0 + bstep,
// ... (nb of them, 0..CHAIN_NB) of RB row blocks from the LDS operand at lds,
// which holds ks k steps per row block: weight steps w0 .. w0 + ks of
// matrices with kw steps (all of them when ks == kw).
template <int PREC, int RB, bool ZERO = true>
__device__ __forceinline__ void chain_blocks(float4v (&acc)[8][CHAIN_NB], uint32_t nb, const uint16_t* lds,
                                             uint32_t ks, const uint16_t* __restrict__ W, uint32_t blk0,
                                             uint32_t bstep, uint32_t lane, uint32_t kw = 0, uint32_t w0 = 0) {
    if (!kw) kw = ks;
    const uint16_t* xs = lds + lane * 8;
    const uint16_t* wp = W + ((size_t)blk0 * kw * 64 + lane) * 8 + (size_t)w0 * 512;
    const size_t wstride = (size_t)bstep * kw * 512;
    static_assert(CHAIN_NB == 3, "dispatch below covers 1..3 blocks");
    if (nb == 1)
        chain_kloop<PREC, 1, RB, ZERO>(acc, xs, ks, wp, wstride);
    else if (nb == 2)
        chain_kloop<PREC, 2, RB, ZERO>(acc, xs, ks, wp, wstride);
    else if (nb == 3)
        chain_kloop<PREC, 3, RB, ZERO>(acc, xs, ks, wp, wstride);
}

// One (row block, feature block) tile of a first-layer partial product: the
// lane's four accumulator values.
__device__ __forceinline__ size_t part_tile(uint32_t rb, uint32_t fb, uint32_t hblk, uint32_t lane) {
    return ((size_t)rb * hblk + fb) * 256 + lane * 4;
}

__device__ __forceinline__ uint32_t pack16(uint16_t lo, uint16_t hi) { return (uint32_t)lo | ((uint32_t)hi << 16); }

// Modes: the whole net over a plan's passes; the whole net with the first
// layer started from a precomputed partial product; the partial product alone;
// the whole net over consecutive row blocks of a row-major f32 input.
constexpr int CHAIN_FULL = 0, CHAIN_PART = 1, CHAIN_STATIC = 2, CHAIN_ROWS = 3;

// The a-th 16-row block of the pass.
template <int MODE>
__device__ __forceinline__ uint32_t chain_block(const ChainPass* __restrict__ ps, uint32_t rb0, uint32_t a) {
    return MODE == CHAIN_ROWS ? rb0 + a : ps->rb[a];
}

// The head over the pass's RB row blocks (LDS operand, K = hidden): rg row
// groups of RBW blocks each (RBW = ceil(RB / rg); a group's blocks past RB are
// computed from in-bounds LDS and not stored) by 8 / rg column groups; the
// wavefront's column blocks are c, c + 8 / rg, ... in steps of CHAIN_NB of
// them. Row-major f32 out.
template <int PREC, int RB, int RBW, int MODE>
__device__ __forceinline__ void chain_head(const ChainNet& net, uint32_t rows, float* __restrict__ out,
                                           const ChainPass* __restrict__ ps, uint32_t rb0, uint32_t t0,
                                           uint32_t nt, uint32_t rg, const uint16_t* lds, uint32_t lane, uint32_t wave) {
    const uint32_t q = lane >> 4, r = lane & 15, ksn = net.hidden >> 5;
    const uint32_t cg = CHAIN_WAVES / rg, g = wave / cg, c = wave % cg, a0 = g * RBW;
    const uint16_t* wh = net.w[net.layers];
    const float* bh = net.b[net.layers];
    const uint16_t* xs = lds + (size_t)a0 * ksn * 512;
    float4v acc[8][CHAIN_NB];
    for (uint32_t c0 = t0; c0 < nt; c0 += cg * CHAIN_NB) {
        const uint32_t end = min(nt, c0 + cg * CHAIN_NB);
        const uint32_t hb = end > c0 + c ? (end - c0 - c + cg - 1) / cg : 0;
        chain_blocks<PREC, RBW>(acc, hb, xs, ksn, wh, c0 + c, cg, lane);
#pragma unroll
        for (int b = 0; b < CHAIN_NB; b++) {
            if ((uint32_t)b >= hb) break;
            const uint32_t n = (c0 + c + cg * b) * 16 + 4 * q;
            float bv[4];
#pragma unroll
            for (int v = 0; v < 4; v++) bv[v] = n + v < net.heads ? bh[n + v] : 0.0f;
            // The row indices are recomputed per column step from an opaque
            // copy of the lane's row: kept live across the loop, they spill.
            uint32_t rr = r;
            asm volatile("" : "+v"(rr));
#pragma unroll
            for (int a = 0; a < RBW; a++) {
                if (a0 + a >= RB) break;
                const uint32_t m = chain_block<MODE>(ps, rb0, a0 + a) * 16 + rr;
                if (m >= rows) continue;
                float* o = out + (size_t)m * net.heads + n;
#pragma unroll
                for (int v = 0; v < 4; v++)
                    if (n + v < net.heads) o[v] = acc[a][b][v] + bv[v];
            }
        }
    }
}

// One pass of the whole network over the pass's RB 16-row blocks (RB <= 8):
// stage their input operand in LDS, run the trunk layers in place, write the
// head.
template <int PREC, int RB, int MODE>
__device__ __forceinline__ void chain_pass(const ChainNet& net, const void* __restrict__ Xv, uint32_t rows,
                                           float* __restrict__ out, const ChainPass* __restrict__ ps, uint32_t rb0,
                                           uint16_t* lds, uint32_t lane, uint32_t wave) {
    const uint32_t q = lane >> 4, r = lane & 15;
    const uint32_t hblk = net.hidden >> 4, ksn = net.hidden >> 5;
    const uint32_t nb = hblk > wave ? (hblk - wave + CHAIN_WAVES - 1) / CHAIN_WAVES : 0;
    // head column blocks the pass needs: all of them, or (consecutive rows) the
    // blockIdx.y-th of gridDim.y shares
    const uint32_t nta = ((MODE == CHAIN_ROWS ? net.heads : min(ps->cols, net.heads)) + 15) >> 4;
    const uint32_t t0 = MODE == CHAIN_ROWS ? nta * blockIdx.y / gridDim.y : 0;
    const uint32_t nt = MODE == CHAIN_ROWS ? nta * (blockIdx.y + 1) / gridDim.y : nta;
    // The first layer's k steps [s0, s0 + sn) of each row block (a contiguous
    // run of 1 KB steps in X), packed in LDS in pass order: all of them, the
    // first dsteps (partial start) or the rest (the static product).
    const uint32_t ks0 = net.in >> 5;
    constexpr bool part = MODE == CHAIN_PART;
    const uint32_t s0 = MODE == CHAIN_STATIC ? net.dsteps : 0;
    const uint32_t sn = MODE == CHAIN_STATIC ? ks0 - net.dsteps : part ? net.dsteps : ks0;
    if constexpr (MODE == CHAIN_ROWS) {
        // One wavefront converts one (block, step) at a time: lane l reads 8
        // floats of row l % 16, so the step's 16 rows arrive as whole 128-byte
        // lines and its 64 fragments leave as one contiguous KB. Rows past the
        // last repeat it (their outputs are not stored).
        const float* X = (const float*)Xv;
#pragma unroll 4
        for (uint32_t i = wave; i < RB * ks0; i += CHAIN_WAVES) {
            const uint32_t a = i / ks0, s = i % ks0, m = min((rb0 + a) * 16 + r, rows - 1);
            const float* src = X + (size_t)m * net.in + 32 * s + 8 * q;
            float v[8];
            if (net.vec) {
                const float4v lo = *(const float4v*)src, hi = *(const float4v*)(src + 4);
#pragma unroll
                for (int k = 0; k < 4; k++) {
                    v[k] = lo[k];
                    v[4 + k] = hi[k];
                }
            } else {
#pragma unroll
                for (int k = 0; k < 8; k++) v[k] = src[k];
            }
            uint4 f;
            auto two = [&](int k) {
                return PREC == WC_F16 ? pack16(f32_to_f16_rn(v[k]), f32_to_f16_rn(v[k + 1]))
                                      : pack16(f32_to_bf16_rn(v[k]), f32_to_bf16_rn(v[k + 1]));
            };
            f.x = two(0);
            f.y = two(2);
            f.z = two(4);
            f.w = two(6);
            ((uint4*)lds)[(size_t)i * 64 + lane] = f;
        }
    } else {
        const uint16_t* X = (const uint16_t*)Xv;
        const uint32_t per = sn * 64;  // uint4 per row block
#pragma unroll
        for (int a = 0; a < RB; a++) {
            const uint4* src = (const uint4*)(X + ((size_t)ps->rb[a] * ks0 + s0) * 512);
            uint4* dst = (uint4*)lds + a * per;
            for (uint32_t i = threadIdx.x; i < per; i += CHAIN_WAVES * 64) dst[i] = src[i];
        }
    }
    float4v acc[8][CHAIN_NB];
    if constexpr (part) {  // the first layer starts from the precomputed product of its other columns
#pragma unroll
        for (int a = 0; a < RB; a++)
#pragma unroll
            for (int b = 0; b < CHAIN_NB; b++)
                if ((uint32_t)b < nb)
                    acc[a][b] = *(const float4v*)(net.part + part_tile(ps->rb[a], wave + CHAIN_WAVES * b, hblk, lane));
    }
    __syncthreads();
    if constexpr (MODE == CHAIN_STATIC) {
        chain_blocks<PREC, RB>(acc, nb, lds, sn, net.w[0], wave, CHAIN_WAVES, lane, ks0, s0);
#pragma unroll
        for (int a = 0; a < RB; a++)
#pragma unroll
            for (int b = 0; b < CHAIN_NB; b++)
                if ((uint32_t)b < nb)
                    *(float4v*)(out + part_tile(ps->rb[a], wave + CHAIN_WAVES * b, hblk, lane)) = acc[a][b];
        return;
    }
    uint32_t K = net.in;
    for (uint32_t l = 0; l < net.layers; l++) {
        if constexpr (part) {  // the later layers start from zero
            if (l > 0)
#pragma unroll
                for (int a = 0; a < RB; a++)
#pragma unroll
                    for (int b = 0; b < CHAIN_NB; b++) acc[a][b] = float4v{0.0f, 0.0f, 0.0f, 0.0f};
        }
        // (sn = ks0 without the partial start: the same call for every layer)
        chain_blocks<PREC, RB, !part>(acc, nb, lds, l ? K >> 5 : sn, net.w[l], wave, CHAIN_WAVES, lane,
                                      l ? 0 : ks0, 0);
        __syncthreads();  // the layer input is dead from here on
        // bias + ReLU, stored over the input as the next operand (K = hidden)
        const float* bias = net.b[l];
#pragma unroll
        for (int b = 0; b < CHAIN_NB; b++) {
            if ((uint32_t)b >= nb) break;
            const uint32_t n = (wave + CHAIN_WAVES * b) * 16 + 4 * q;
            const float b0 = bias[n], b1 = bias[n + 1], b2 = bias[n + 2], b3 = bias[n + 3];
            const size_t col = (size_t)(n >> 5) * 64 + r + ((n & 31) >> 3) * 16;
#pragma unroll
            for (int a = 0; a < RB; a++) {
                float y0 = acc[a][b][0] + b0, y1 = acc[a][b][1] + b1, y2 = acc[a][b][2] + b2,
                      y3 = acc[a][b][3] + b3;
                y0 = y0 > 0.0f ? y0 : 0.0f;
                y1 = y1 > 0.0f ? y1 : 0.0f;
                y2 = y2 > 0.0f ? y2 : 0.0f;
                y3 = y3 > 0.0f ? y3 : 0.0f;
                uint2 v;
                if (PREC == WC_F16) {
                    v.x = pack16(f32_to_f16_rn(y0), f32_to_f16_rn(y1));
                    v.y = pack16(f32_to_f16_rn(y2), f32_to_f16_rn(y3));
                } else {
                    v.x = pack16(f32_to_bf16_rn(y0), f32_to_bf16_rn(y1));
                    v.y = pack16(f32_to_bf16_rn(y2), f32_to_bf16_rn(y3));
                }
                *(uint2*)(lds + (((size_t)a * ksn * 64 + col) * 8 + (n & 7))) = v;
            }
        }
        __syncthreads();
        K = net.hidden;
    }
    // Head: the columns the pass's rows need, nt 16-column blocks. Few blocks go to groups of wavefronts that split the rows (rg
    // row groups of RB / rg blocks, 8 / rg blocks per column step), so that
    // every wavefront has work and reads fewer operand fragments per product.
    if (nt - t0 <= 6 && RB >= 4)
        chain_head<PREC, RB, (RB + 3) / 4, MODE>(net, rows, out, ps, rb0, t0, nt, 4, lds, lane, wave);
    else if (nt - t0 <= 12 && RB >= 2)
        chain_head<PREC, RB, (RB + 1) / 2, MODE>(net, rows, out, ps, rb0, t0, nt, 2, lds, lane, wave);
    else
        chain_head<PREC, RB, RB, MODE>(net, rows, out, ps, rb0, t0, nt, 1, lds, lane, wave);
}

// One workgroup per pass: of the plan (plan_chain orders the passes so that
// the costly ones start first), or of `per` consecutive row blocks.
template <int PREC, int MODE>
__global__ __launch_bounds__(CHAIN_WAVES * 64) __attribute__((amdgpu_waves_per_eu(CHAIN_WAVES / 4, CHAIN_WAVES / 4))) void k_chain(
    ChainNet net, const void* __restrict__ X, uint32_t rows, float* __restrict__ out,
    const ChainPass* __restrict__ plan, uint32_t per) {
    __shared__ __attribute__((aligned(16))) uint16_t lds[CHAIN_LDS_HALVES];
    const uint32_t lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const ChainPass* ps = plan + blockIdx.x;
    const uint32_t rb0 = blockIdx.x * per;
    const uint32_t n = MODE == CHAIN_ROWS ? min(per, ((rows + 15) >> 4) - rb0) : ps->n;
    switch (min(CHAIN_PASS_BLOCKS, n)) {
        case 8: chain_pass<PREC, 8, MODE>(net, X, rows, out, ps, rb0, lds, lane, wave); break;
        case 7: chain_pass<PREC, 7, MODE>(net, X, rows, out, ps, rb0, lds, lane, wave); break;
        case 6: chain_pass<PREC, 6, MODE>(net, X, rows, out, ps, rb0, lds, lane, wave); break;
        case 5: chain_pass<PREC, 5, MODE>(net, X, rows, out, ps, rb0, lds, lane, wave); break;
        case 4: chain_pass<PREC, 4, MODE>(net, X, rows, out, ps, rb0, lds, lane, wave); break;
        case 3: chain_pass<PREC, 3, MODE>(net, X, rows, out, ps, rb0, lds, lane, wave); break;
        case 2: chain_pass<PREC, 2, MODE>(net, X, rows, out, ps, rb0, lds, lane, wave); break;
        case 1: chain_pass<PREC, 1, MODE>(net, X, rows, out, ps, rb0, lds, lane, wave); break;
        default: break;
    }
}

// ------------------------------------- fused leaf network, compensated f16
//
// k_chain for operands held as f16 pairs hi + lo: both planes of up to four
// row blocks live in LDS, and each step's product is lo hi + hi lo + hi hi, as
// k_gemm_x takes it (x's lo first). Products, order and rounding are
// k_gemm_x's, so the results are too, bit for bit.
//
// Bound: a pass streams both planes of every weight matrix from L2 (2.8 MB
// for the 512 -> 3x384 -> 567 net, at 64 bytes per clock and CU) under three
// MFMAs per tile and step, against one read and write of every activation
// plane through HBM per layer and 93 workgroups for 3,915 rows in k_gemm_x. In
// the 64-subgame wave a pass (3,915 rows, head widths per block) takes 38 us
// against 133; 5,003 rows with 22 heads take 30 us against 132.

constexpr int CHAINX_RB = 4;

template <int NB, int RB>
__device__ __forceinline__ void chainx_kloop(float4v (&acc)[CHAINX_RB][CHAIN_NB], const uint16_t* xs, uint32_t xplane,
                                             uint32_t ks, const uint16_t* __restrict__ wp, size_t wstride,
                                             size_t wplane) {
#pragma unroll
    for (int a = 0; a < RB; a++)
#pragma unroll
        for (int b = 0; b < NB; b++) acc[a][b] = float4v{0.0f, 0.0f, 0.0f, 0.0f};
    uint4 xa[2][RB], xb[2][RB], w0[2][NB], w1[2][NB], w2[2][NB], w3[2][NB];
    auto ldw = [&](uint4 (&fw)[2][NB], uint32_t s) {
        s = s < ks ? s : ks - 1;
#pragma unroll
        for (int b = 0; b < NB; b++) {
            const uint16_t* p = wp + b * wstride + (size_t)s * 512;
            fw[0][b] = *(const uint4*)p;
            fw[1][b] = *(const uint4*)(p + wplane);
        }
    };
    auto ldx = [&](uint4 (&fx)[2][RB], uint32_t s) {
        s = s < ks ? s : ks - 1;
#pragma unroll
        for (int a = 0; a < RB; a++) {
            const uint16_t* p = xs + ((size_t)a * ks + s) * 512;
            fx[0][a] = *(const uint4*)p;
            fx[1][a] = *(const uint4*)(p + xplane);
        }
    };
    auto step = [&](const uint4 (&fx)[2][RB], const uint4 (&fw)[2][NB]) {
#pragma unroll
        for (int a = 0; a < RB; a++)
#pragma unroll
            for (int b = 0; b < NB; b++) acc[a][b] = mfma16<WC_F16>(fw[0][b], fx[1][a], acc[a][b]);
#pragma unroll
        for (int a = 0; a < RB; a++)
#pragma unroll
            for (int b = 0; b < NB; b++) acc[a][b] = mfma16<WC_F16>(fw[1][b], fx[0][a], acc[a][b]);
#pragma unroll
        for (int a = 0; a < RB; a++)
#pragma unroll
            for (int b = 0; b < NB; b++) acc[a][b] = mfma16<WC_F16>(fw[0][b], fx[0][a], acc[a][b]);
    };
    ldw(w0, 0);
    ldw(w1, 1);
    ldx(xa, 0);
    uint32_t s = 0;
    for (; s + 4 <= ks; s += 4) {
        ldw(w2, s + 2);
        ldx(xb, s + 1);
        __builtin_amdgcn_sched_barrier(0);
        step(xa, w0);
        __builtin_amdgcn_sched_barrier(0);
        ldw(w3, s + 3);
        ldx(xa, s + 2);
        __builtin_amdgcn_sched_barrier(0);
        step(xb, w1);
        __builtin_amdgcn_sched_barrier(0);
        ldw(w0, s + 4);
        ldx(xb, s + 3);
        __builtin_amdgcn_sched_barrier(0);
        step(xa, w2);
        __builtin_amdgcn_sched_barrier(0);
        ldw(w1, s + 5);
        ldx(xa, s + 4);
        __builtin_amdgcn_sched_barrier(0);
        step(xb, w3);
        __builtin_amdgcn_sched_barrier(0);
    }
    for (; s < ks; s++) {  // K not a multiple of 128: the last steps one at a time
        ldw(w0, s);
        ldx(xa, s);
        step(xa, w0);
    }
}

// The wavefront's column blocks blk0, blk0 + CHAIN_WAVES, ... (nb of them) of
// a matrix with N columns.
template <int RB>
__device__ __forceinline__ void chainx_blocks(float4v (&acc)[CHAINX_RB][CHAIN_NB], uint32_t nb, const uint16_t* lds,
                                              uint32_t xplane, uint32_t ks, const uint16_t* __restrict__ W,
                                              uint32_t N, uint32_t blk0, uint32_t lane) {
    const uint16_t* xs = lds + lane * 8;
    const uint16_t* wp = W + ((size_t)blk0 * ks * 64 + lane) * 8;
    const size_t wstride = (size_t)CHAIN_WAVES * ks * 512;
    const size_t wplane = (size_t)((N + GEMM_ROWS - 1) / GEMM_ROWS * GEMM_ROWS) * ks * 32;
    if (nb == 1)
        chainx_kloop<1, RB>(acc, xs, xplane, ks, wp, wstride, wplane);
    else if (nb == 2)
        chainx_kloop<2, RB>(acc, xs, xplane, ks, wp, wstride, wplane);
    else if (nb == 3)
        chainx_kloop<3, RB>(acc, xs, xplane, ks, wp, wstride, wplane);
}

// An f16 pair of v: hi = f16(v), lo = f16(v - hi).
__device__ __forceinline__ void split16(float v, uint16_t* hi, uint16_t* lo) {
    *hi = f32_to_f16_rn(v);
    *lo = f32_to_f16_rn(v - (float)__builtin_bit_cast(_Float16, *hi));
}

template <int RB, int MODE>
__device__ __forceinline__ void chainx_pass(const ChainNet& net, const void* __restrict__ Xv, uint32_t rows,
                                            float* __restrict__ out, const ChainPass* __restrict__ ps, uint32_t rb0,
                                            uint16_t* lds, uint32_t lane, uint32_t wave) {
    const uint32_t q = lane >> 4, r = lane & 15;
    const uint32_t hblk = net.hidden >> 4, ksn = net.hidden >> 5, ks0 = net.in >> 5;
    const uint32_t nb = hblk > wave ? (hblk - wave + CHAIN_WAVES - 1) / CHAIN_WAVES : 0;
    const uint32_t nta = ((MODE == CHAIN_ROWS ? net.heads : min(ps->cols, net.heads)) + 15) >> 4;
    const uint32_t t0 = MODE == CHAIN_ROWS ? nta * blockIdx.y / gridDim.y : 0;
    const uint32_t nt = MODE == CHAIN_ROWS ? nta * (blockIdx.y + 1) / gridDim.y : nta;
    const uint32_t plane = RB * max(ks0, ksn) * 512;  // halves between the planes in LDS
    if constexpr (MODE == CHAIN_ROWS) {  // as chain_pass stages it, both planes
        const float* X = (const float*)Xv;
#pragma unroll 2
        for (uint32_t i = wave; i < RB * ks0; i += CHAIN_WAVES) {
            const uint32_t a = i / ks0, s = i % ks0, m = min((rb0 + a) * 16 + r, rows - 1);
            const float* src = X + (size_t)m * net.in + 32 * s + 8 * q;
            float v[8];
            if (net.vec) {
                const float4v lo = *(const float4v*)src, hi = *(const float4v*)(src + 4);
#pragma unroll
                for (int k = 0; k < 4; k++) {
                    v[k] = lo[k];
                    v[4 + k] = hi[k];
                }
            } else {
#pragma unroll
                for (int k = 0; k < 8; k++) v[k] = src[k];
            }
            uint16_t h[8], l[8];
#pragma unroll
            for (int k = 0; k < 8; k++) split16(v[k], h + k, l + k);
            uint16_t* dst = lds + ((size_t)i * 64 + lane) * 8;
            *(uint4*)dst = make_uint4(pack16(h[0], h[1]), pack16(h[2], h[3]), pack16(h[4], h[5]), pack16(h[6], h[7]));
            *(uint4*)(dst + plane) =
                make_uint4(pack16(l[0], l[1]), pack16(l[2], l[3]), pack16(l[4], l[5]), pack16(l[6], l[7]));
        }
    } else {
        const uint16_t* X = (const uint16_t*)Xv;
        const uint32_t per = ks0 * 64;  // uint4 per row block and plane
#pragma unroll
        for (int a = 0; a < RB; a++) {
            const uint4* hi = (const uint4*)(X + (size_t)ps->rb[a] * ks0 * 512);
            const uint4* lo = (const uint4*)(X + net.xplane + (size_t)ps->rb[a] * ks0 * 512);
            uint4* dst = (uint4*)lds + a * per;
            for (uint32_t i = threadIdx.x; i < per; i += CHAIN_WAVES * 64) {
                dst[i] = hi[i];
                *(uint4*)((uint16_t*)(dst + i) + plane) = lo[i];
            }
        }
    }
    float4v acc[CHAINX_RB][CHAIN_NB];
    __syncthreads();
    for (uint32_t l = 0; l < net.layers; l++) {
        chainx_blocks<RB>(acc, nb, lds, plane, l ? ksn : ks0, net.w[l], net.hidden, wave, lane);
        __syncthreads();  // the layer input is dead from here on
        const float* bias = net.b[l];
#pragma unroll
        for (int b = 0; b < CHAIN_NB; b++) {
            if ((uint32_t)b >= nb) break;
            const uint32_t n = (wave + CHAIN_WAVES * b) * 16 + 4 * q;
            float bv[4];
#pragma unroll
            for (int v = 0; v < 4; v++) bv[v] = bias[n + v];
            const size_t col = (size_t)(n >> 5) * 64 + r + ((n & 31) >> 3) * 16;
#pragma unroll
            for (int a = 0; a < RB; a++) {
                uint16_t h[4], lo[4];
#pragma unroll
                for (int v = 0; v < 4; v++) {
                    const float y = acc[a][b][v] + bv[v];
                    split16(y > 0.0f ? y : 0.0f, h + v, lo + v);
                }
                uint16_t* dst = lds + (((size_t)a * ksn * 64 + col) * 8 + (n & 7));
                *(uint2*)dst = make_uint2(pack16(h[0], h[1]), pack16(h[2], h[3]));
                *(uint2*)(dst + plane) = make_uint2(pack16(lo[0], lo[1]), pack16(lo[2], lo[3]));
            }
        }
        __syncthreads();
    }
    const float* bh = net.b[net.layers];
    for (uint32_t c0 = t0; c0 < nt; c0 += CHAIN_WAVES * CHAIN_NB) {
        const uint32_t end = min(nt, c0 + CHAIN_WAVES * CHAIN_NB);
        const uint32_t hb = end > c0 + wave ? (end - c0 - wave + CHAIN_WAVES - 1) / CHAIN_WAVES : 0;
        chainx_blocks<RB>(acc, hb, lds, plane, ksn, net.w[net.layers], net.heads, c0 + wave, lane);
#pragma unroll
        for (int b = 0; b < CHAIN_NB; b++) {
            if ((uint32_t)b >= hb) break;
            const uint32_t n = (c0 + wave + CHAIN_WAVES * b) * 16 + 4 * q;
#pragma unroll
            for (int a = 0; a < RB; a++) {
                const uint32_t m = chain_block<MODE>(ps, rb0, a) * 16 + r;
                if (m >= rows) continue;
#pragma unroll
                for (int v = 0; v < 4; v++)
                    if (n + v < net.heads) out[(size_t)m * net.heads + n + v] = acc[a][b][v] + bh[n + v];
            }
        }
    }
}

template <int MODE>
__global__ __launch_bounds__(CHAIN_WAVES * 64) __attribute__((amdgpu_waves_per_eu(CHAIN_WAVES / 4, CHAIN_WAVES / 4))) void k_chain_x(
    ChainNet net, const void* __restrict__ X, uint32_t rows, float* __restrict__ out,
    const ChainPass* __restrict__ plan, uint32_t per) {
    __shared__ __attribute__((aligned(16))) uint16_t lds[CHAIN_LDS_HALVES];
    const uint32_t lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const ChainPass* ps = plan + blockIdx.x;
    const uint32_t rb0 = blockIdx.x * per;
    const uint32_t n = MODE == CHAIN_ROWS ? min(per, ((rows + 15) >> 4) - rb0) : ps->n;
    switch (min((uint32_t)CHAINX_RB, n)) {
        case 4: chainx_pass<4, MODE>(net, X, rows, out, ps, rb0, lds, lane, wave); break;
        case 3: chainx_pass<3, MODE>(net, X, rows, out, ps, rb0, lds, lane, wave); break;
        case 2: chainx_pass<2, MODE>(net, X, rows, out, ps, rb0, lds, lane, wave); break;
        case 1: chainx_pass<1, MODE>(net, X, rows, out, ps, rb0, lds, lane, wave); break;
        default: break;
    }
}

// ------------------------------------------------ fused public tower
//
// The two-tower net's public tower, up to TOWER_WIDTH wide, in one launch: a
// pass of up to four 16-row blocks staged in LDS, every layer in place as in
// k_chain (each wavefront owns up to four 16-feature blocks of the width), the
// last layer stored as the readout's fragment-major operand. k_gemm's products
// in k_gemm's order: bit-identical. Bound: each pass streams the weights from
// L2 (1 MB for 512 -> 2x512) and 188 registers leave one workgroup per CU;
// layer by layer every activation crossed HBM twice and a 128-wide tile filled
// 280 workgroups. 8,904 rows: 50 -> 27 us per pass; 49 row blocks (784 rows):
// 28 -> 10 us.

constexpr int TOWER_RB = 4, TOWER_NB = 4;
constexpr uint32_t TOWER_WIDTH = CHAIN_WAVES * TOWER_NB * 16;

bool tower_fits(uint32_t in, uint32_t width, uint32_t layers) {
    return in % 32 == 0 && in <= TOWER_WIDTH && width % 32 == 0 && width <= TOWER_WIDTH && layers >= 1 &&
           layers <= CHAIN_MAX_LAYERS;
}

template <int PREC, int NB, int RB>
__device__ __forceinline__ void tower_kloop(float4v (&acc)[TOWER_RB][TOWER_NB], const uint16_t* xs, uint32_t ks,
                                            const uint16_t* __restrict__ wp, size_t wstride) {
#pragma unroll
    for (int a = 0; a < RB; a++)
#pragma unroll
        for (int b = 0; b < NB; b++) acc[a][b] = float4v{0.0f, 0.0f, 0.0f, 0.0f};
    uint4 xa[RB], xb[RB], w0[NB], w1[NB], w2[NB], w3[NB];
    auto ldw = [&](uint4 (&fw)[NB], uint32_t s) {
        s = s < ks ? s : ks - 1;
#pragma unroll
        for (int b = 0; b < NB; b++) fw[b] = *(const uint4*)(wp + b * wstride + (size_t)s * 512);
    };
    auto ldx = [&](uint4 (&fx)[RB], uint32_t s) {
        s = s < ks ? s : ks - 1;
#pragma unroll
        for (int a = 0; a < RB; a++) fx[a] = *(const uint4*)(xs + ((size_t)a * ks + s) * 512);
    };
    auto step = [&](const uint4 (&fx)[RB], const uint4 (&fw)[NB]) {
#pragma unroll
        for (int a = 0; a < RB; a++)
#pragma unroll
            for (int b = 0; b < NB; b++) acc[a][b] = mfma16<PREC>(fw[b], fx[a], acc[a][b]);
    };
    ldw(w0, 0);
    ldw(w1, 1);
    ldx(xa, 0);
    uint32_t s = 0;
    for (; s + 4 <= ks; s += 4) {
        ldw(w2, s + 2);
        ldx(xb, s + 1);
        __builtin_amdgcn_sched_barrier(0);
        step(xa, w0);
        __builtin_amdgcn_sched_barrier(0);
        ldw(w3, s + 3);
        ldx(xa, s + 2);
        __builtin_amdgcn_sched_barrier(0);
        step(xb, w1);
        __builtin_amdgcn_sched_barrier(0);
        ldw(w0, s + 4);
        ldx(xb, s + 3);
        __builtin_amdgcn_sched_barrier(0);
        step(xa, w2);
        __builtin_amdgcn_sched_barrier(0);
        ldw(w1, s + 5);
        ldx(xa, s + 4);
        __builtin_amdgcn_sched_barrier(0);
        step(xb, w3);
        __builtin_amdgcn_sched_barrier(0);
    }
    for (; s < ks; s++) {  // K not a multiple of 128: the last steps one at a time
        ldw(w0, s);
        ldx(xa, s);
        step(xa, w0);
    }
}

template <int PREC, int RB>
__device__ __forceinline__ void tower_pass(const ChainNet& net, const uint16_t* __restrict__ X,
                                           uint16_t* __restrict__ Y, uint32_t rb0, uint16_t* lds, uint32_t lane,
                                           uint32_t wave) {
    const uint32_t q = lane >> 4, r = lane & 15;
    const uint32_t hblk = net.hidden >> 4, ksn = net.hidden >> 5, ks0 = net.in >> 5;
    const uint32_t nb = hblk > wave ? (hblk - wave + CHAIN_WAVES - 1) / CHAIN_WAVES : 0;
    // consecutive blocks: one contiguous run
    const uint4* src = (const uint4*)(X + (size_t)rb0 * ks0 * 512);
    for (uint32_t i = threadIdx.x; i < RB * ks0 * 64; i += CHAIN_WAVES * 64) ((uint4*)lds)[i] = src[i];
    float4v acc[TOWER_RB][TOWER_NB];
    __syncthreads();
    for (uint32_t l = 0; l < net.layers; l++) {
        const uint32_t ks = l ? ksn : ks0;
        const uint16_t* xs = lds + lane * 8;
        const uint16_t* wp = net.w[l] + ((size_t)wave * ks * 64 + lane) * 8;
        const size_t wstride = (size_t)CHAIN_WAVES * ks * 512;
        static_assert(TOWER_NB == 4, "dispatch below covers 1..4 blocks");
        if (nb == 1)
            tower_kloop<PREC, 1, RB>(acc, xs, ks, wp, wstride);
        else if (nb == 2)
            tower_kloop<PREC, 2, RB>(acc, xs, ks, wp, wstride);
        else if (nb == 3)
            tower_kloop<PREC, 3, RB>(acc, xs, ks, wp, wstride);
        else if (nb == 4)
            tower_kloop<PREC, 4, RB>(acc, xs, ks, wp, wstride);
        __syncthreads();  // the layer input is dead from here on
        const float* bias = net.b[l];
#pragma unroll
        for (int b = 0; b < TOWER_NB; b++) {
            if ((uint32_t)b >= nb) break;
            const uint32_t n = (wave + CHAIN_WAVES * b) * 16 + 4 * q;
            float bv[4];
#pragma unroll
            for (int v = 0; v < 4; v++) bv[v] = bias[n + v];
            const size_t col = (size_t)(n >> 5) * 64 + r + ((n & 31) >> 3) * 16;
#pragma unroll
            for (int a = 0; a < RB; a++) {
                uint16_t h[4];
#pragma unroll
                for (int v = 0; v < 4; v++) {
                    const float y = acc[a][b][v] + bv[v];
                    h[v] = PREC == WC_F16 ? f32_to_f16_rn(y > 0.0f ? y : 0.0f) : f32_to_bf16_rn(y > 0.0f ? y : 0.0f);
                }
                *(uint2*)(lds + (((size_t)a * ksn * 64 + col) * 8 + (n & 7))) =
                    make_uint2(pack16(h[0], h[1]), pack16(h[2], h[3]));
            }
        }
        __syncthreads();
    }
    uint4* dst = (uint4*)(Y + (size_t)rb0 * ksn * 512);
    for (uint32_t i = threadIdx.x; i < RB * ksn * 64; i += CHAIN_WAVES * 64) dst[i] = ((const uint4*)lds)[i];
}

// One workgroup per pass of `per` consecutive row blocks of nrb.
template <int PREC>
__global__ __launch_bounds__(CHAIN_WAVES * 64) void k_tower(ChainNet net, const uint16_t* __restrict__ X,
                                                            uint16_t* __restrict__ Y, uint32_t nrb, uint32_t per) {
    __shared__ __attribute__((aligned(16))) uint16_t lds[TOWER_RB * 16 * TOWER_WIDTH];
    const uint32_t lane = threadIdx.x & 63, wave = threadIdx.x >> 6, rb0 = blockIdx.x * per;
    switch (min(per, nrb - rb0)) {
        case 4: tower_pass<PREC, 4>(net, X, Y, rb0, lds, lane, wave); break;
        case 3: tower_pass<PREC, 3>(net, X, Y, rb0, lds, lane, wave); break;
        case 2: tower_pass<PREC, 2>(net, X, Y, rb0, lds, lane, wave); break;
        case 1: tower_pass<PREC, 1>(net, X, Y, rb0, lds, lane, wave); break;
        default: break;
    }
}

void launch_tower(int precision, const ChainNet& net, const void* X, void* Y, uint32_t rows, uint32_t cus,
                  hipStream_t s) {
    if (!rows) return;
    const uint32_t nrb = (rows + 15) / 16, rounds = (nrb + TOWER_RB * cus - 1) / (TOWER_RB * cus);
    const uint32_t per = (nrb + rounds * cus - 1) / (rounds * cus);  // (one workgroup's registers fill a CU)
    const dim3 grid((nrb + per - 1) / per), block(CHAIN_WAVES * 64);
    if (precision == WC_F16)
        hipLaunchKernelGGL(k_tower<WC_F16>, grid, block, 0, s, net, (const uint16_t*)X, (uint16_t*)Y, nrb, per);
    else
        hipLaunchKernelGGL(k_tower<WC_BF16>, grid, block, 0, s, net, (const uint16_t*)X, (uint16_t*)Y, nrb, per);
}

void launch_chain(int precision, const ChainNet& net, const void* X, uint32_t rows, float* out,
                  const ChainPass* plan, uint32_t npass, hipStream_t s) {
    if (rows == 0 || npass == 0) return;
    dim3 grid(npass), block(CHAIN_WAVES * 64);
    const void* x = X;
    if (precision == WC_F16X) {
        hipLaunchKernelGGL(k_chain_x<CHAIN_FULL>, grid, block, 0, s, net, x, rows, out, plan, 0u);
    } else if (precision == WC_F16) {
        if (net.part)
            hipLaunchKernelGGL((k_chain<WC_F16, CHAIN_PART>), grid, block, 0, s, net, x, rows, out, plan, 0u);
        else
            hipLaunchKernelGGL((k_chain<WC_F16, CHAIN_FULL>), grid, block, 0, s, net, x, rows, out, plan, 0u);
    } else {
        if (net.part)
            hipLaunchKernelGGL((k_chain<WC_BF16, CHAIN_PART>), grid, block, 0, s, net, x, rows, out, plan, 0u);
        else
            hipLaunchKernelGGL((k_chain<WC_BF16, CHAIN_FULL>), grid, block, 0, s, net, x, rows, out, plan, 0u);
    }
}

void launch_chain_static(int precision, const ChainNet& net, const void* X, float* part, const ChainPass* plan,
                         uint32_t npass, hipStream_t s) {
    if (npass == 0) return;
    dim3 grid(npass), block(CHAIN_WAVES * 64);
    if (precision == WC_F16)
        hipLaunchKernelGGL((k_chain<WC_F16, CHAIN_STATIC>), grid, block, 0, s, net, X, 0u, part,
                           plan, 0u);
    else
        hipLaunchKernelGGL((k_chain<WC_BF16, CHAIN_STATIC>), grid, block, 0, s, net, X, 0u, part,
                           plan, 0u);
}

void launch_chain_rows(int precision, ChainNet net, const float* X, uint32_t rows, float* out, uint32_t cus,
                       hipStream_t s) {
    if (rows == 0) return;
    net.vec = (uintptr_t)X % 16 == 0;
    const uint32_t nrb = (rows + 15) / 16, most = chain_most(precision), rounds = (nrb + most * cus - 1) / (most * cus);
    const uint32_t per = (nrb + rounds * cus - 1) / (rounds * cus);
    // Few rows: idle CUs repeat the trunk to take a share of the head columns
    // each, down to one 16-column block per wavefront (250 rows, 567 heads:
    // 15.5 us against 21.2 us with one share).
    const uint32_t passes = (nrb + per - 1) / per, blocks = (net.heads + 15) / 16;
    const uint32_t shares = std::max(1u, std::min((blocks + CHAIN_WAVES - 1) / CHAIN_WAVES, cus / passes));
    dim3 grid(passes, shares), block(CHAIN_WAVES * 64);
    if (precision == WC_F16X)
        hipLaunchKernelGGL(k_chain_x<CHAIN_ROWS>, grid, block, 0, s, net, (const void*)X, rows, out,
                           (const ChainPass*)nullptr, per);
    else if (precision == WC_F16)
        hipLaunchKernelGGL((k_chain<WC_F16, CHAIN_ROWS>), grid, block, 0, s, net, (const void*)X, rows, out,
                           (const ChainPass*)nullptr, per);
    else
        hipLaunchKernelGGL((k_chain<WC_BF16, CHAIN_ROWS>), grid, block, 0, s, net, (const void*)X, rows, out,
                           (const ChainPass*)nullptr, per);
}

}  // namespace wc
