// Domain-local RI fits per occupied pair on the device: domain_fit_pair
// (crates/ferric-mp2/src/lmp2_amplitude.rs:1707-1758),
//
//   J_ij = A_{i,D}^T V_DD^{-1} A_{j,D},   D = the aux functions within `radius`
//                                          of the centre of i or of j,
//
// with A the unwhitened (P|ia) and V the aux metric: one workgroup per pair, or several
// for large domains, gathers, factors, solves and multiplies.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstdlib>
#include <mutex>
#include <type_traits>
#include <vector>

#include "fh_device.h"
#include "fh_host.h"
#include "fh_kernels.h"

namespace fh {
namespace {

// ---- One workgroup per pair --------------------------------------------------
// With V_DD = U^T U and Y = U^-T [A_i | A_j], J = Y_i^T Y_j. The rows of
// [V_DD | A_i | A_j] are eliminated 16 at a time, looking left: a 16 x 16 block of the
// row takes the products with the rows above (v_mfma_f64_16x16x4f64, the block in the
// accumulators), wave 0 factors the diagonal block and applies the same row operations
// to the identity, and each wave multiplies its blocks by that U_kk^-T. An accumulator
// element v of a lane is row 4 v + g, which is what the B operand of step v holds, so
// the blocks stay in their registers. The finished rows lie in a slot of the workspace,
// read from the caches. A row of blocks is also a chain of two barriers and 16 dependent
// pivots (about 4 us), which the other workgroups of a CU, four to each, hide.
// 820 pairs of up to 120 aux functions and 100 virtuals: 276 us, 24% of it at the matrix
// units. The chain is eight rows, about 32 us, and all pairs are resident at once: what
// bounds the kernel is the operands, every block read again from the slot by each wave
// that needs it (530 MB past the L2). 2.5 ms of rocSOLVER and rocBLAS launches (potf2,
// trtri, lauum, symm, gemm) before. Also faster at 36 pairs of 41 (0.28 -> 0.09 ms a call)
// and 820 of 480 (26 -> 4.7 ms).
struct FitArgs {
    const int32_t *pairs;
    const uint64_t *near;  // per occupied: words of aux bits inside the radius
    int words;
    const double *v, *a;
    int64_t naux, nov;
    int nvir, nv;          // nv: 16-wide blocks of virtuals
    int cap;               // rows of a slot, a multiple of 16
    int32_t *dom;          // cap per pair
    double *u;             // cap (cap + 32 nv) per pair
    int32_t *size;         // split rows: the domain's size per pair
    int32_t *info;
    double *j;
};

constexpr int kFitWaves = 4, kFitHeld = 5;  // blocks a wave keeps while the pivots are found
constexpr int kFitThreads = kFitWaves * 64;

__device__ __forceinline__ double lane_value(double x, int lane) {
    const int64_t b = __builtin_bit_cast(int64_t, x);
    const uint32_t lo = __builtin_amdgcn_readlane((uint32_t)b, lane);
    const uint32_t hi = __builtin_amdgcn_readlane((uint32_t)((uint64_t)b >> 32), lane);
    return __builtin_bit_cast(double, (uint64_t)hi << 32 | lo);
}

// The domain: the aux functions near i or j, in aux order. Its size.
__device__ __forceinline__ int fit_domain(const FitArgs &g, int oi, int oj, int32_t *dom) {
    __shared__ int wsum[kFitWaves];
    const int tid = threadIdx.x, lane = tid % kWave;
    const int wid = __builtin_amdgcn_readfirstlane(tid / kWave);
    int d = 0;
    for (int w0 = 0; w0 < g.words; w0 += kFitThreads) {
        const int w = w0 + tid;
        uint64_t m = 0;
        if (w < g.words)
            m = g.near[(int64_t)oi * g.words + w] | g.near[(int64_t)oj * g.words + w];
        const int c = __popcll(m);
        int at = c;
        for (int k = 1; k < kWave; k *= 2) {
            const int o = __shfl_up(at, k, kWave);
            if (lane >= k) at += o;
        }
        if (lane == kWave - 1) wsum[wid] = at;
        __syncthreads();
        int total = 0;
        for (int k = 0; k < kFitWaves; ++k) {
            if (k < wid) at += wsum[k];
            total += wsum[k];
        }
        for (at += d - c; m; m &= m - 1) dom[at++] = w * 64 + __ffsll((unsigned long long)m) - 1;
        d += total;
        __syncthreads();
    }
    return __builtin_amdgcn_readfirstlane(d);
}

// Block row k of a pair's elimination: the diagonal block and the columns past it, c of C
// workgroups taking every C-th turn of kFitHeld blocks a wave (SPLIT), or all. Each of them
// factors the diagonal block for itself. The first bad pivot, from 1, or 0.
template <bool SPLIT>
__device__ __forceinline__ int fit_row(const FitArgs &g, int oi, int oj, const int32_t *dom, int d,
                                       double *u, int k, int c, int C) {
    __shared__ double diag[16][17];
    __shared__ double linv[16][17];
    __shared__ int bad;
    const int tid = threadIdx.x, lane = tid % kWave;
    const int wid = __builtin_amdgcn_readfirstlane(tid / kWave);
    const int r = lane % 16, gg = lane / 16;
    const int nd = (d + 15) / 16;
    const int64_t ldu = (int64_t)(nd + 2 * g.nv) * 16;
    const uint32_t off = (uint32_t)(gg * (int)ldu + r);
    const int nblk = nd - k + 2 * g.nv;  // block t: columns 16 (k + t) .. + 16
    int row[4];
#pragma unroll
    for (int v = 0; v < 4; ++v) row[v] = dom[min(16 * k + 4 * v + gg, d - 1)];
    // Blocks t = t0 + wid, t0 + wid + 4, ..., H of them (one past the last stands for
    // it and is not stored), as they stand before any elimination (the lower triangle
    // of V, the identity past the domain, A past V), less the products with the rows
    // above. All loads of a step are issued before the products of the last one.
    v4d acc[kFitHeld];
    auto update = [&](auto held, int t0) {
        constexpr int H = decltype(held)::value;
        int32_t first[H];  // of the column: V's row, A's column
#pragma unroll
        for (int q = 0; q < H; ++q) {
            const int t = min(t0 + wid + q * kFitWaves, nblk - 1), x = t - (nd - k);
            first[q] = x < 0 ? dom[min(16 * (k + t) + r, d - 1)]
                             : min((x < g.nv ? x : x - g.nv) * 16 + r, g.nvir - 1);
        }
#pragma unroll
        for (int q = 0; q < H; ++q) {
            const int t = min(t0 + wid + q * kFitWaves, nblk - 1), x = t - (nd - k);
            const double *base = x < 0 ? g.v : g.a + (int64_t)(x < g.nv ? oi : oj) * g.nvir;
            const int64_t sr = x < 0 ? 1 : g.nov, sc = x < 0 ? g.naux : 1;
#pragma unroll
            for (int v = 0; v < 4; ++v) acc[q][v] = base[row[v] * sr + first[q] * sc];
        }
        __builtin_amdgcn_sched_barrier(0);
        const double *um = u + 16 * k, *ut = um + 16 * (t0 + wid);
        const int last = 16 * (min(t0 + wid + (H - 1) * kFitWaves, nblk - 1) - t0 - wid);
        double fa[2][2], fb[2][2][H];
        auto fetch = [&](int h) {  // half of the 16 rows at um
#pragma unroll
            for (int s = 0; s < 2; ++s) {
                const int64_t at = 4 * (2 * h + s) * ldu;
                fa[h][s] = (um + at)[off];
#pragma unroll
                for (int q = 0; q < H; ++q)
                    fb[h][s][q] = (ut + at + (q + 1 < H ? 16 * kFitWaves * q : last))[off];
            }
            __builtin_amdgcn_sched_barrier(0);
        };
        auto products = [&](int h) {
#pragma unroll
            for (int s = 0; s < 2; ++s)
#pragma unroll
                for (int q = 0; q < H; ++q)
                    acc[q] = __builtin_amdgcn_mfma_f64_16x16x4f64(-fa[h][s], fb[h][s][q],
                                                                  acc[q], 0, 0, 0);
        };
        if (k > 0) fetch(0);
#pragma unroll
        for (int q = 0; q < H; ++q) {
            const int t = min(t0 + wid + q * kFitWaves, nblk - 1), x = t - (nd - k);
            const int C = 16 * (k + t) + r, lim = (x < g.nv ? g.nvir : g.nvir + 16 * g.nv);
#pragma unroll
            for (int v = 0; v < 4; ++v) {
                const int R = 16 * k + 4 * v + gg;
                const bool in = R < d && (x < 0 ? C < d : 16 * x + r < lim);
                acc[q][v] = in ? acc[q][v] : (R == C ? 1.0 : 0.0);
            }
        }
        for (int m = 0; m < k; ++m) {
            fetch(1);
            products(0);
            if (m + 1 < k) {
                um += 16 * ldu;
                ut += 16 * ldu;
            }
            fetch(0);
            products(1);
        }
    };
    auto finish = [&](auto held, int t0) {
        constexpr int H = decltype(held)::value;
        double fa[4];
#pragma unroll
        for (int s = 0; s < 4; ++s) fa[s] = linv[r][4 * s + gg];
#pragma unroll
        for (int q = 0; q < H; ++q) {
            const int t = t0 + wid + q * kFitWaves;
            v4d o = {0, 0, 0, 0};
#pragma unroll
            for (int s = 0; s < 4; ++s)
                o = __builtin_amdgcn_mfma_f64_16x16x4f64(fa[s], acc[q][s], o, 0, 0, 0);
            if (t >= nblk || t == 0) continue;
#pragma unroll
            for (int v = 0; v < 4; ++v)
                (u + (16 * k + 4 * v) * ldu + 16 * (k + t))[off] = o[v];
        }
    };
    auto with_held = [&](int t0, auto f) {
        const int n = (nblk - t0 + kFitWaves - 1) / kFitWaves;
        if (n >= kFitHeld) f(std::integral_constant<int, kFitHeld>{});
        else if (n == 4) f(std::integral_constant<int, 4>{});
        else if (n == 3) f(std::integral_constant<int, 3>{});
        else if (n == 2) f(std::integral_constant<int, 2>{});
        else f(std::integral_constant<int, 1>{});
    };
    if (!SPLIT || c == 0)
        with_held(0, [&](auto h) { update(h, 0); });
    else
        update(std::integral_constant<int, 1>{}, 0);
    if (wid == 0)
#pragma unroll
        for (int v = 0; v < 4; ++v) diag[4 * v + gg][r] = acc[0][v];
    __syncthreads();
    if (wid == 0) {
        // Lanes 0 .. 15 hold the block's columns, 16 .. 31 the identity's; rows below
        // the diagonal of a column are never read by another lane.
        double c[16];
#pragma unroll
        for (int i = 0; i < 16; ++i)
            c[i] = lane < 16 ? diag[i][r] : (lane < 32 && i == r ? 1.0 : 0.0);
        int fault = 0;
#pragma unroll
        for (int i = 0; i < 16; ++i) {
            const double piv = lane_value(c[i], i);
            // Not positive, NaN, or infinite: a non-finite element of the metric reaches
            // a pivot as one of them.
            if (!(piv > 0.0 && piv < INFINITY) && fault == 0) fault = 16 * k + i + 1;
            c[i] *= 1.0 / sqrt(piv);
#pragma unroll
            for (int x = i + 1; x < 16; ++x) c[x] -= lane_value(c[i], x) * c[i];
        }
        if (lane >= 16 && lane < 32)
#pragma unroll
            for (int i = 0; i < 16; ++i) linv[i][r] = c[i];
        if (lane == 0) bad = fault;
    }
    __syncthreads();
    if (bad) return bad;
    if (!SPLIT || c == 0) with_held(0, [&](auto h) { finish(h, 0); });
    const int turn = kFitHeld * kFitWaves;
    for (int t0 = (!SPLIT ? 1 : c == 0 ? C : c) * turn; t0 < nblk; t0 += (SPLIT ? C : 1) * turn) {
        with_held(t0, [&](auto h) { update(h, t0); });
        with_held(t0, [&](auto h) { finish(h, t0); });
    }
    __syncthreads();
    return 0;
}

// Turns first, first + step, ... of J = Y_i^T Y_j, 32 x 64 a wave and turn.
__device__ __forceinline__ void fit_product(const FitArgs &g, int d, const double *u, double *jp,
                                            int first, int step) {
    const int lane = threadIdx.x % kWave, r = lane % 16, gg = lane / 16;
    const int nd = (d + 15) / 16;
    const int64_t ldu = (int64_t)(nd + 2 * g.nv) * 16;
    const uint32_t off = (uint32_t)(gg * (int)ldu + r);
    const int na = (g.nv + 1) / 2, nb = (g.nv + 3) / 4;
    const double *yi = u + 16 * nd, *yj = yi + 16 * g.nv;
    for (int t = first; t < na * nb; t += step) {
        const int a0 = t / nb * 2, b0 = t % nb * 4;
        int ca[2], cb[4];  // blocks past the end repeat the last one
#pragma unroll
        for (int x = 0; x < 2; ++x) ca[x] = 16 * min(a0 + x, g.nv - 1);
#pragma unroll
        for (int y = 0; y < 4; ++y) cb[y] = 16 * min(b0 + y, g.nv - 1);
        v4d acc[2][4];
#pragma unroll
        for (int x = 0; x < 2; ++x)
#pragma unroll
            for (int y = 0; y < 4; ++y) acc[x][y] = (v4d){0, 0, 0, 0};
        double fa[2][2][2], fb[2][2][4];
        const double *ri = yi, *rj = yj;
        auto fetch = [&](int h) {  // eight rows
#pragma unroll
            for (int s = 0; s < 2; ++s) {
#pragma unroll
                for (int x = 0; x < 2; ++x) fa[h][s][x] = (ri + 4 * s * ldu + ca[x])[off];
#pragma unroll
                for (int y = 0; y < 4; ++y) fb[h][s][y] = (rj + 4 * s * ldu + cb[y])[off];
            }
            __builtin_amdgcn_sched_barrier(0);
            ri += 8 * ldu;
            rj += 8 * ldu;
        };
        auto products = [&](int h) {
#pragma unroll
            for (int s = 0; s < 2; ++s)
#pragma unroll
                for (int x = 0; x < 2; ++x)
#pragma unroll
                    for (int y = 0; y < 4; ++y)
                        acc[x][y] = __builtin_amdgcn_mfma_f64_16x16x4f64(
                            fa[h][s][x], fb[h][s][y], acc[x][y], 0, 0, 0);
        };
        fetch(0);
        for (int k = 0; k < nd; ++k) {
            fetch(1);
            products(0);
            if (k + 1 == nd) ri = yi, rj = yj;  // fetched again and not used
            fetch(0);
            products(1);
        }
#pragma unroll
        for (int x = 0; x < 2; ++x)
#pragma unroll
            for (int y = 0; y < 4; ++y) {
                const int b = 16 * (b0 + y) + r;
#pragma unroll
                for (int v = 0; v < 4; ++v) {
                    const int av = 16 * (a0 + x) + 4 * v + gg;
                    if (av < g.nvir && b < g.nvir) jp[(int64_t)av * g.nvir + b] = acc[x][y][v];
                }
            }
    }
}

__device__ __forceinline__ double *fit_slot(const FitArgs &g, int64_t p) {
    return g.u + p * g.cap * (int64_t)(g.cap + 32 * g.nv);
}

__global__ __launch_bounds__(kFitThreads, 4) void fit_pair_kernel(FitArgs g) {
    const int64_t p = blockIdx.x;
    const int oi = g.pairs[2 * p], oj = g.pairs[2 * p + 1];
    int32_t *dom = g.dom + p * g.cap;
    const int d = fit_domain(g, oi, oj, dom);
    double *u = fit_slot(g, p);
    for (int k = 0; k < (d + 15) / 16; ++k)
        if (const int bad = fit_row<false>(g, oi, oj, dom, d, u, k, 0, 1)) {
            if (threadIdx.x == 0) g.info[p] = bad;
            return;
        }
    if (threadIdx.x == 0) g.info[p] = 0;
    fit_product(g, d, u, g.j + p * (int64_t)g.nvir * g.nvir,
                __builtin_amdgcn_readfirstlane(threadIdx.x / kWave), kFitWaves);
}

// ---- Several workgroups per pair -----------------------------------------------
// The same operations in the same order, a launch to a block row, for large domains: one
// workgroup takes d^3 (359 ms for a domain of 6000, and the rest of the chip idles).
__global__ __launch_bounds__(kFitThreads) void fit_domain_kernel(FitArgs g) {
    const int64_t p = blockIdx.x;
    const int d = fit_domain(g, g.pairs[2 * p], g.pairs[2 * p + 1], g.dom + p * g.cap);
    if (threadIdx.x == 0) {
        g.size[p] = d;
        g.info[p] = 0;
    }
}

__global__ __launch_bounds__(kFitThreads, 2) void fit_row_kernel(FitArgs g, int k) {
    const int64_t p = blockIdx.x;
    const int d = g.size[p], nblk = (d + 15) / 16 - k + 2 * g.nv;
    // A pair whose bad pivot was found is of no more interest.
    if (16 * k >= d || (int)blockIdx.y * kFitHeld * kFitWaves >= nblk || g.info[p]) return;
    const int bad = fit_row<true>(g, g.pairs[2 * p], g.pairs[2 * p + 1], g.dom + p * g.cap, d,
                                  fit_slot(g, p), k, blockIdx.y, gridDim.y);
    if (bad && blockIdx.y == 0 && threadIdx.x == 0) g.info[p] = bad;
}

__global__ __launch_bounds__(kFitThreads, 2) void fit_product_kernel(FitArgs g) {
    const int64_t p = blockIdx.x;
    if (g.info[p]) return;
    fit_product(g, g.size[p], fit_slot(g, p), g.j + p * (int64_t)g.nvir * g.nvir,
                __builtin_amdgcn_readfirstlane(threadIdx.x / kWave) + kFitWaves * blockIdx.y,
                kFitWaves * gridDim.y);
}

// Where n pairs of up to dmax aux functions take several workgroups each. ms, one / several, at
// 100 virtuals: 16 pairs of 300 0.44 / 0.40, 16 of 400 0.64 / 0.58 (36 at 20 virtuals 0.48 /
// 0.50), 64 of 480 0.99 / 0.79, 136 of 480 1.02 / 1.08, 820 of 480 4.75 / 5.10, 1 of 1000 3.6 /
// 2.4, 400 of 1000 14.05 / 14.00, 300 of 1500 34.5 / 31.2, 1 of 2000 18.9 / 8.8, 400 of 2000
// 124 / 88, 4 of 3000 54 / 20, 1 of 6000 360 / 76 (100 with rocSOLVER and rocBLAS).
bool split_rows(size_t dmax, size_t n) { return dmax >= 1000 || (dmax >= 400 && n <= 64); }

hipError_t launch_fit(const FitArgs &g, size_t n, bool split, hipStream_t st, uint64_t *launches) {
    if (!split) {
        hipLaunchKernelGGL(fit_pair_kernel, dim3((unsigned)n), dim3(kFitThreads), 0, st, g);
        *launches += 1;
        return hipGetLastError();
    }
    hipLaunchKernelGGL(fit_domain_kernel, dim3((unsigned)n), dim3(kFitThreads), 0, st, g);
    auto grid = [&](int blocks, int per) {
        return dim3((unsigned)n, (unsigned)((blocks + per - 1) / per));
    };
    for (int k = 0; k < g.cap / 16; ++k)
        hipLaunchKernelGGL(fit_row_kernel,
                           grid(g.cap / 16 - k + 2 * g.nv, kFitHeld * kFitWaves),
                           dim3(kFitThreads), 0, st, g, k);
    hipLaunchKernelGGL(fit_product_kernel, grid((g.nv + 1) / 2 * ((g.nv + 3) / 4), kFitWaves),
                       dim3(kFitThreads), 0, st, g);
    *launches += (uint64_t)g.cap / 16 + 2;
    return hipGetLastError();
}

// Pairs of one batch, of `per` bytes each: 4 GiB of them.
size_t fit_batch(size_t npairs, size_t per) {
    size_t nb = 0;
    if (const char *s = std::getenv("FERRIC_FIT_BATCH")) nb = (size_t)std::strtoull(s, nullptr, 10);
    if (nb == 0) nb = std::max<size_t>(1, ((size_t)4 << 30) / (per + 64));
    return std::min(nb, npairs);
}

fh_status fit_pairs(State &s, const double *a, const double *v, size_t naux, size_t nocc,
                    size_t nvir, const std::vector<uint64_t> &near, size_t words,
                    const int32_t *pairs, size_t npairs, size_t dmax, hipStream_t stream,
                    double *j_out) {
    FitArgs g;
    g.a = a;
    g.v = v;
    g.naux = (int64_t)naux;
    g.nov = (int64_t)(nocc * nvir);
    g.nvir = (int)nvir;
    g.nv = (int)((nvir + 15) / 16);
    g.cap = (int)((dmax + 15) / 16 * 16);
    g.words = (int)words;
    const size_t cap = (size_t)g.cap, slot = cap * (cap + 32 * (size_t)g.nv);
    const size_t nb = fit_batch(npairs, sizeof(double) * slot);
    const size_t near_bytes = sizeof(uint64_t) * near.size();
    fh_status st = reserve(s, {{kSlotFitWork, sizeof(double) * nb * slot},
                               {kSlotFitMeta, near_bytes + sizeof(int32_t) * (npairs * 2 +
                                                                              nb * (cap + 2))}});
    if (st != FH_OK) return st;
    g.u = (double *)s.slots[kSlotFitWork].ptr;
    uint64_t *dnear = (uint64_t *)s.slots[kSlotFitMeta].ptr;
    int32_t *dpairs = (int32_t *)(dnear + near.size());
    g.near = dnear;
    g.dom = dpairs + 2 * npairs;
    g.size = g.dom + nb * cap;
    g.info = g.size + nb;
    st = hip_check(hipMemcpyAsync(dnear, near.data(), near_bytes, hipMemcpyHostToDevice, stream),
                   "H2D domains");
    if (st != FH_OK) return st;
    st = hip_check(hipMemcpyAsync(dpairs, pairs, sizeof(int32_t) * 2 * npairs,
                                  hipMemcpyHostToDevice, stream),
                   "H2D pairs");
    if (st != FH_OK) return st;
    s.pending.h2d_bytes += near_bytes + sizeof(int32_t) * 2 * npairs;
    std::vector<int32_t> info(nb);
    mark(s, 0, stream);
    mark(s, 1, stream);
    for (size_t p0 = 0; p0 < npairs; p0 += nb) {
        const size_t n = std::min(nb, npairs - p0);
        g.pairs = dpairs + 2 * p0;
        g.j = j_out + p0 * nvir * nvir;
        st = hip_check(launch_fit(g, n, split_rows(dmax, n), stream, &s.pending.kernel_launches),
                       "domain fit kernel");
        if (st != FH_OK) return st;
        st = hip_check(hipMemcpyAsync(info.data(), g.info, sizeof(int32_t) * n,
                                      hipMemcpyDeviceToHost, stream),
                       "D2H Cholesky info");
        if (st != FH_OK) return st;
        st = hip_check(hipStreamSynchronize(stream), "stream sync");
        if (st != FH_OK) return st;
        for (size_t k = 0; k < n; ++k)
            if (info[k] != 0)
                return fail(FH_KERNEL,
                            "domain metric of pair (%d, %d) is not positive definite (Cholesky "
                            "info %d)",
                            pairs[2 * (p0 + k)], pairs[2 * (p0 + k) + 1], info[k]);
    }
    mark(s, 2, stream);
    mark(s, 3, stream);
    finish_timing(s, (uint64_t)npairs, 0);
    return FH_OK;
}

fh_status fit_core(State &s, const double *a, const double *v, size_t naux, size_t nocc,
                   size_t nvir, const double *aux_xyz, const double *centers, double radius,
                   const int32_t *pairs, size_t npairs, hipStream_t stream, double *j_out,
                   size_t *max_domain) {
    // Aux functions near each occupied (lmp2_amplitude.rs:1726-1735), one bit each; a
    // pair's domain is the union of its two rows, in aux order.
    const double r2 = radius * radius;
    const size_t words = (naux + 63) / 64;
    std::vector<uint64_t> near(nocc * words, 0);
    std::vector<char> wanted(nocc, 0);
    for (size_t k = 0; k < 2 * npairs; ++k) wanted[pairs[k]] = 1;
    for (size_t i = 0; i < nocc; ++i) {
        if (!wanted[i]) continue;
        const double *c = centers + 3 * i;
        for (size_t p = 0; p < naux; ++p) {
            const double ux = aux_xyz[3 * p] - c[0], uy = aux_xyz[3 * p + 1] - c[1],
                         uz = aux_xyz[3 * p + 2] - c[2];
            double di = 0.0;
            di += ux * ux;
            di += uy * uy;
            di += uz * uz;
            if (di <= r2) near[i * words + p / 64] |= 1ull << (p % 64);
        }
    }
    size_t dmax = 0;
    for (size_t k = 0; k < npairs; ++k) {
        const int32_t i = pairs[2 * k], j = pairs[2 * k + 1];
        size_t d = 0;
        for (size_t w = 0; w < words; ++w)
            d += (size_t)__builtin_popcountll(near[i * words + w] | near[j * words + w]);
        if (d == 0)
            return fail(FH_LAYOUT, "empty aux domain for pair (%d, %d) at radius %g bohr", i, j,
                        radius);
        dmax = std::max(dmax, d);
    }
    if (max_domain) *max_domain = dmax;
    return fit_pairs(s, a, v, naux, nocc, nvir, near, words, pairs, npairs, dmax, stream, j_out);
}

fh_status fit_checks(size_t naux, size_t nocc, size_t nvir, const double *aux_xyz,
                     const double *centers, double radius, const int32_t *pairs, size_t npairs) {
    if (naux == 0 || nocc == 0 || nvir == 0) return fail(FH_LAYOUT, "empty dimension");
    if (!aux_xyz || !centers) return fail(FH_LAYOUT, "null aux positions or occupied centres");
    if (!(radius >= 0.0)) return fail(FH_LAYOUT, "radius must be >= 0 (got %g)", radius);
    if (npairs > 0 && !pairs) return fail(FH_LAYOUT, "null pair list");
    for (size_t k = 0; k < npairs; ++k) {
        const int32_t i = pairs[2 * k], j = pairs[2 * k + 1];
        if (i < 0 || i > j || (size_t)j >= nocc)
            return fail(FH_LAYOUT, "pair %zu is (%d, %d): need 0 <= i <= j < nocc = %zu", k, i,
                        j, nocc);
    }
    if (naux > 46340 || nocc * nvir > (size_t)INT32_MAX)
        return fail(FH_LAYOUT, "naux %zu / nocc*nvir %zu beyond the int32 BLAS range", naux,
                    nocc * nvir);
    return FH_OK;
}

}  // namespace
}  // namespace fh

using namespace fh;

extern "C" fh_status fh_domain_fit_pair_blocks_dev(const double *a_dev, const double *v_dev,
                                                   size_t naux, size_t nocc, size_t nvir,
                                                   const double *aux_xyz, const double *centers,
                                                   double radius, const int32_t *pairs,
                                                   size_t npairs, void *stream, double *j_dev,
                                                   size_t *max_domain) {
    State &s = state();
    std::lock_guard<std::mutex> lk(s.mu);
    clear_error();
    s.stats.calls++;
    s.pending = Pending{};
    fh_status st = fit_checks(naux, nocc, nvir, aux_xyz, centers, radius, pairs, npairs);
    if (st != FH_OK) return st;
    if (max_domain) *max_domain = 0;
    if (npairs == 0) return FH_OK;
    if (!a_dev || !v_dev || !j_dev) return fail(FH_LAYOUT, "null device pointer");
    st = ensure_device(s);
    if (st != FH_OK) return st;
    st = fit_core(s, a_dev, v_dev, naux, nocc, nvir, aux_xyz, centers, radius, pairs, npairs,
                  (hipStream_t)stream, j_dev, max_domain);
    if (st != FH_OK) return st;
    commit(s, Prec::F64, false, false);
    return FH_OK;
}

extern "C" fh_status fh_domain_fit_pair_blocks(const double *a, const double *v, size_t naux,
                                               size_t nocc, size_t nvir, const double *aux_xyz,
                                               const double *centers, double radius,
                                               const int32_t *pairs, size_t npairs, double *j_out,
                                               size_t *max_domain) {
    State &s = state();
    std::lock_guard<std::mutex> lk(s.mu);
    clear_error();
    s.stats.calls++;
    s.pending = Pending{};
    fh_status st = fit_checks(naux, nocc, nvir, aux_xyz, centers, radius, pairs, npairs);
    if (st != FH_OK) return st;
    if (max_domain) *max_domain = 0;
    if (npairs == 0) return FH_OK;
    if (!a || !v || !j_out) return fail(FH_LAYOUT, "null pointer");
    st = ensure_device(s);
    if (st != FH_OK) return st;
    const size_t abytes = sizeof(double) * naux * nocc * nvir;
    const size_t vbytes = sizeof(double) * naux * naux;
    const size_t jbytes = sizeof(double) * npairs * nvir * nvir;
    st = reserve(s, {{kSlotStage, abytes}, {kSlotStage2, vbytes}, {kSlotGamma, jbytes}});
    if (st != FH_OK) return st;
    st = hip_check(hipMemcpyAsync(s.slots[kSlotStage].ptr, a, abytes, hipMemcpyHostToDevice,
                                  nullptr),
                   "H2D A");
    if (st != FH_OK) return st;
    st = hip_check(hipMemcpyAsync(s.slots[kSlotStage2].ptr, v, vbytes, hipMemcpyHostToDevice,
                                  nullptr),
                   "H2D V");
    if (st != FH_OK) return st;
    s.pending.h2d_bytes += abytes + vbytes;
    double *jd = (double *)s.slots[kSlotGamma].ptr;
    st = fit_core(s, (const double *)s.slots[kSlotStage].ptr,
                  (const double *)s.slots[kSlotStage2].ptr, naux, nocc, nvir, aux_xyz, centers,
                  radius, pairs, npairs, nullptr, jd, max_domain);
    if (st != FH_OK) return st;
    st = hip_check(hipMemcpy(j_out, jd, jbytes, hipMemcpyDeviceToHost), "D2H J");
    if (st != FH_OK) return st;
    s.pending.d2h_bytes += jbytes;
    commit(s, Prec::F64, false, false);
    return FH_OK;
}
