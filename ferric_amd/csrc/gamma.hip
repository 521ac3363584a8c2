// The FP64 adjoint over whole amplitudes: dE/deps and Gamma = dE/dB (gfx950).
//
// The pair pass has stored t of every ordered occupied pair as one matrix over
// (i, a) rows and (j, b) columns. Two steps remain:
//   T~ = c_d t - c_e t^T in place (the transposed element t_ij^ba is t_ji^ab, so both
//      orders of a pair block are read and written by the same thread), with the row
//      sums of t T~ that dE/deps consists of;
//   Gamma[Q, ia] = 4 sum_jb B[Q, jb] T~[ia, jb], one FP64 product.
// At 41/209/960 one launch of each replaces 41 rounds of five launches: the adjoint
// went from 9.1 to 4.2 ms (pairs 3836 -> 1250 us in residue arithmetic, products
// 4281 -> 2320 us, the sums and folds 743 -> 240 us), 2.1 of it the products at the
// matrix rate of the clock that they leave the chip.
#include <hip/hip_runtime.h>

#include <algorithm>

#include "fh_device.h"
#include "fh_kernels.h"

namespace fh {
namespace {

// ---- B by Q, rows padded with zeros to the K panels --------------------------
template <typename Tin>
__global__ __launch_bounds__(256) void gamma_rows_kernel(const Tin *__restrict__ b, int64_t nov,
                                                         int64_t ld, double *__restrict__ out) {
    const int64_t q = blockIdx.y, c = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (c < ld) out[q * ld + c] = c < nov ? (double)b[q * nov + c] : 0.0;
}

// ---- t -> T~ in place ---------------------------------------------------------
// One workgroup per unique pair and kTRows virtuals a: a wave takes a row of the
// block (i, j) and the same row of (j, i). Bound by its traffic, one read and one
// write of the matrix: 225 us for 587 MB at 41/209, 5.2 TB/s with what the caches hold.
constexpr int kTRows = 16;
__global__ __launch_bounds__(256) void gamma_spin_kernel(GammaArgs g) {
    int i, j;
    decode_tile_pair((int)blockIdx.x, g.nocc, i, j);
    const int lane = threadIdx.x % kWave, wid = threadIdx.x / kWave;
    for (int k = wid; k < kTRows; k += 4) {
        const int a = blockIdx.y * kTRows + k;
        if (a >= g.nvir) return;
        double *x = g.t + ((int64_t)i * g.nvir + a) * g.ld + (int64_t)j * g.nvir;
        double *y = g.t + ((int64_t)j * g.nvir + a) * g.ld + (int64_t)i * g.nvir;
        double sx = 0.0, sy = 0.0;
        for (int b = lane; b < g.nvir; b += kWave) {
            const double tx = x[b], ty = y[b];
            const double ux = g.cd * tx - g.ce * ty, uy = g.cd * ty - g.ce * tx;
            sx += tx * ux;
            sy += ty * uy;
            x[b] = ux;
            if (i != j) y[b] = uy;
        }
        // Zeros up to the panel's end, for the products of the last panel.
        if (j == g.nocc - 1) {
            const int tail = (int)(g.ld - (int64_t)g.nocc * g.nvir);
            if (lane < tail) x[g.nvir + lane] = 0.0;
            if (i != j && i == g.nocc - 1 && lane < tail) y[g.nvir + lane] = 0.0;
        }
        for (int m = 1; m < kWave; m *= 2) {
            sx += __shfl_xor(sx, m, kWave);
            sy += __shfl_xor(sy, m, kWave);
        }
        if (lane == 0) {
            g.rsum[((int64_t)i * g.nvir + a) * g.nocc + j] = sx;
            if (i != j) g.rsum[((int64_t)j * g.nvir + a) * g.nocc + i] = sy;
        }
    }
}

// dE/deps from the row sums: block k < nocc adds the nvir nocc sums of occupied k,
// block nocc + c those of virtual c (nocc rows of nocc sums).
__global__ __launch_bounds__(256) void gamma_deps_kernel(GammaArgs g) {
    const int k = blockIdx.x;
    const bool occ = k < g.nocc;
    const int64_t n = (int64_t)g.nocc * (occ ? g.nvir : g.nocc);
    KSum s;
    for (int64_t e = threadIdx.x; e < n; e += 256)
        s.add(occ ? g.rsum[(int64_t)k * g.nvir * g.nocc + e]
                  : g.rsum[((e / g.nocc) * g.nvir + (k - g.nocc)) * g.nocc + e % g.nocc]);
    wave_merge(s);
    __shared__ double red[4][2];
    if (threadIdx.x % kWave == 0) {
        red[threadIdx.x / kWave][0] = s.s;
        red[threadIdx.x / kWave][1] = s.c;
    }
    __syncthreads();
    if (threadIdx.x != 0) return;
    for (int w = 1; w < 4; ++w) s.merge(red[w][0], red[w][1]);
    g.deps[k] = (occ ? -2.0 : 2.0) * s.value();
}

// ---- Gamma ------------------------------------------------------------------
// 64 Q x 128 (i, a) a workgroup of four waves, 64 x 32 each: v_mfma_f64_16x16x4f64 (64
// cycles each) bounds it: 61 TFLOP/s at 960 Q and 8569 (i, a), 83 to 89% of the issue
// slots at the 2.05 GHz that the load leaves of 2.4. A wave's 32 products a 16-deep panel
// meet 24 KB of operands, so two workgroups per CU draw 12 B a cycle. The panels come
// through three LDS stages by direct loads up to three panels ahead; a row's 16-byte
// chunk c lies at slot c ^ (row & 7), so the 16 rows of a fragment read spread over the
// banks. Every 16 panels the sums move into a second set of accumulators, which keeps the
// rounding at chains of 64 products instead of K / 4.
constexpr int kGM = 64, kGN = 128, kGK = 16, kGBuf = 3, kFlush = 16;
constexpr int kGStage = (kGM + kGN) * kGK * 8;

template <int N>
__device__ __forceinline__ void gamma_wait() {
    __builtin_amdgcn_sched_barrier(0);
    asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"(N) : "memory");
    __builtin_amdgcn_sched_barrier(0);
}

__global__ __launch_bounds__(256, 2) void gamma_gemm_kernel(GammaArgs g) {
    extern __shared__ __attribute__((aligned(16))) char lds[];
    const int64_t nov = (int64_t)g.nocc * g.nvir;
    const int mt = (g.naux + kGM - 1) / kGM;
    // Q tiles fastest, so that the workgroups of an XCD share a few rows of T~.
    const int64_t item = xcd_remap(blockIdx.x, gridDim.x);
    const int m0 = (int)(item % mt) * kGM;
    const int split = (int)(item / mt % g.splits);
    const int64_t n0 = item / mt / g.splits * kGN;
    const int np = (int)(g.ld / kGK);
    const int p0 = (int)((int64_t)np * split / g.splits);
    const int count = (int)((int64_t)np * (split + 1) / g.splits) - p0;
    const int lane = threadIdx.x % kWave;
    const int wid = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);

    // Each wave stages rows 8 wid .. 8 wid + 7 of every 32 (two instructions for A,
    // four for T~). Rows past the end repeat the last one; their sums are not stored.
    const int lr = lane / 8, lc = ((lane % 8) ^ lr) * 16;
    uint32_t off[6];
#pragma unroll
    for (int u = 0; u < 6; ++u) {
        const int row = 8 * wid + 32 * (u < 2 ? u : u - 2) + lr;
        const int64_t left = u < 2 ? (int64_t)g.naux - m0 : nov - n0;
        off[u] = (uint32_t)(std::min<int64_t>(row, left - 1) * g.ld * 8) + lc;
    }
    const char *pa = (const char *)(g.b + (int64_t)m0 * g.ld + (int64_t)p0 * kGK);
    const char *pt = (const char *)(g.t + n0 * g.ld + (int64_t)p0 * kGK);
    int ahead = count;
    uint32_t to = 0;
    // Past the last panel the first is fetched again and never read.
    auto fetch = [&] {
#pragma unroll
        for (int u = 0; u < 6; ++u) {
            const uint32_t dst = to + (8 * wid + 32 * u) * (kGK * 8);
            __builtin_amdgcn_global_load_lds((GlobalPtr)((u < 2 ? pa : pt) + off[u]),
                                             (LdsPtr)(lds + dst), 16, 0, 0);
        }
        to = to + kGStage == kGBuf * kGStage ? 0 : to + kGStage;
        const int64_t step = --ahead > 0 ? kGK * 8 : 0;
        pa += step;
        pt += step;
    };
    const int r = lane % 16, gg = lane / 16;
    const uint32_t s0 = (uint32_t)(r * (kGK * 8) + ((gg ^ (r & 7)) * 16));
    const uint32_t s1 = (uint32_t)(r * (kGK * 8) + (((4 + gg) ^ (r & 7)) * 16));
    v4d acc[4][2], sum[4][2];
#pragma unroll
    for (int x = 0; x < 4; ++x)
#pragma unroll
        for (int y = 0; y < 2; ++y) acc[x][y] = sum[x][y] = (v4d){0, 0, 0, 0};

    // Fragments of the next half panel are read while the products of this one run.
    v2d fa[2][4], ft[2][2];
    uint32_t cur = 0;
    auto read = [&](int h) {
        const char *la = lds + cur + (h ? s1 : s0), *lt = la + (kGM + 32 * wid) * (kGK * 8);
#pragma unroll
        for (int x = 0; x < 4; ++x) fa[h][x] = *(const v2d *)(la + x * 16 * (kGK * 8));
#pragma unroll
        for (int y = 0; y < 2; ++y) ft[h][y] = *(const v2d *)(lt + y * 16 * (kGK * 8));
        __builtin_amdgcn_sched_barrier(0);
    };
    auto products = [&](int h) {
#pragma unroll
        for (int e = 0; e < 2; ++e)
#pragma unroll
            for (int x = 0; x < 4; ++x)
#pragma unroll
                for (int y = 0; y < 2; ++y)
                    acc[x][y] = __builtin_amdgcn_mfma_f64_16x16x4f64(fa[h][x][e], ft[h][y][e],
                                                                     acc[x][y], 0, 0, 0);
    };
    fetch();
    fetch();
    fetch();
    gamma_wait<12>();
    read(0);
    int until = kFlush;
    for (int p = 0; p < count; ++p) {
        read(1);
        products(0);
        gamma_wait<6>();  // the next panel is in, this one is read by every wave
        fetch();
        cur = cur + kGStage == kGBuf * kGStage ? 0 : cur + kGStage;
        read(0);
        products(1);
        if (--until == 0 || p + 1 == count) {
            until = kFlush;
#pragma unroll
            for (int x = 0; x < 4; ++x)
#pragma unroll
                for (int y = 0; y < 2; ++y) {
                    sum[x][y] += acc[x][y];
                    acc[x][y] = (v4d){0, 0, 0, 0};
                }
        }
    }
    gamma_wait<0>();
    const bool part = g.splits > 1;
    double *out = part ? g.partial + (int64_t)split * g.naux * nov : g.gamma;
    const double alpha = part ? 1.0 : 4.0;
#pragma unroll
    for (int x = 0; x < 4; ++x)
#pragma unroll
        for (int y = 0; y < 2; ++y) {
            const int64_t n = n0 + 32 * wid + 16 * y + r;
#pragma unroll
            for (int v = 0; v < 4; ++v) {
                const int q = m0 + 16 * x + out_row<double>(gg, v);
                if (q < g.naux && n < nov) out[q * nov + n] = alpha * sum[x][y][v];
            }
        }
}

// Gamma = 4 sum of the K slices, in slice order.
__global__ __launch_bounds__(256) void gamma_sum_kernel(GammaArgs g) {
    const int64_t n = (int64_t)g.naux * g.nocc * g.nvir;
    const int64_t k = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (k >= n) return;
    double s = 0.0;
    for (int p = 0; p < g.splits; ++p) s += g.partial[p * n + k];
    g.gamma[k] = 4.0 * s;
}

}  // namespace

int64_t gamma_ld(int64_t nov) { return (nov + kGK - 1) / kGK * kGK; }

// K slices: the fewest that end within 2% of the shortest time, in panels of the two
// workgroups a CU holds. A slice also writes and reads its part of Gamma, the time of
// about 20 panels of a full chip per 8 M elements, and is at least one flush long.
int gamma_splits(int naux, int64_t nov, int cus) {
    const int64_t tiles = (int64_t)((naux + kGM - 1) / kGM) * ((nov + kGN - 1) / kGN);
    const int64_t np = gamma_ld(nov) / kGK, slots = 2 * (int64_t)cus;
    int best = 1;
    double least = 0.0;
    for (int s = 1; s <= 16 && (s == 1 || np / s >= kFlush); ++s) {
        const double rounds = (double)((tiles * s + slots - 1) / slots);
        const double t = rounds * (double)((np + s - 1) / s) +
                         (s > 1 ? 2.5e-6 * (double)naux * (double)nov * (s + 1) : 0.0);
        if (s == 1 || t < 0.98 * least) {
            best = s;
            least = t;
        }
    }
    return best;
}

hipError_t launch_gamma_rows(const void *b, bool in_f32, int naux, int64_t nov, int64_t ld,
                             double *out, hipStream_t st) {
    if (naux < 1 || naux > 0x7fffffff / 2 || ld < nov) return hipErrorInvalidValue;
    for (int q = 0; q < naux; q += 65535) {  // the grid's limit in y
        const dim3 grid((unsigned)((ld + 255) / 256), (unsigned)std::min(65535, naux - q));
        if (in_f32)
            hipLaunchKernelGGL(gamma_rows_kernel<float>, grid, dim3(256), 0, st,
                               (const float *)b + q * nov, nov, ld, out + q * ld);
        else
            hipLaunchKernelGGL(gamma_rows_kernel<double>, grid, dim3(256), 0, st,
                               (const double *)b + q * nov, nov, ld, out + q * ld);
    }
    return hipGetLastError();
}

hipError_t launch_gamma(const GammaArgs &g, hipStream_t st) {
    const int64_t nov = (int64_t)g.nocc * g.nvir;
    const int64_t npair = (int64_t)g.nocc * (g.nocc + 1) / 2;
    const int64_t items = (int64_t)((g.naux + kGM - 1) / kGM) * ((nov + kGN - 1) / kGN) * g.splits;
    // Row offsets inside a tile are 32-bit.
    if (g.ld % kGK != 0 || g.ld < nov || g.ld - nov >= kGK || g.ld * 8 * kGN > 0xffffffffLL ||
        g.nocc < 1 || g.nvir < 1 || g.naux < 1 || g.splits < 1 || g.splits > g.ld / kGK ||
        items > 0x7fffffffLL || npair > 0x7fffffffLL || (g.nvir + kTRows - 1) / kTRows > 65535 ||
        (g.splits > 1 && !g.partial))
        return hipErrorInvalidValue;
    hipLaunchKernelGGL(gamma_spin_kernel,
                       dim3((unsigned)npair, (unsigned)((g.nvir + kTRows - 1) / kTRows)),
                       dim3(256), 0, st, g);
    hipLaunchKernelGGL(gamma_deps_kernel, dim3((unsigned)(g.nocc + g.nvir)), dim3(256), 0, st, g);
    hipLaunchKernelGGL(gamma_gemm_kernel, dim3((unsigned)items), dim3(256), kGBuf * kGStage, st,
                       g);
    if (g.splits > 1)
        hipLaunchKernelGGL(gamma_sum_kernel,
                           dim3((unsigned)(((int64_t)g.naux * nov + 255) / 256)), dim3(256), 0, st,
                           g);
    return hipGetLastError();
}

}  // namespace fh
