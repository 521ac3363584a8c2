// MP2 one-particle densities P_oo, P_vv on the device
// (build_mp2_density, crates/ferric-mp2/src/oo_rimp2.rs:1192-1300, with the
// spin scaling of apply_spin_scaling / opposite_spin_density,
// crates/ferric-mp2/src/rimp2.rs:1917-2052):
//   P_ij = - sum_k sum_ab t_ik^ab T~_jk^ab
//   P_ab =   sum_ij sum_c t_ij^ac T~_ij^bc,   T~ = (c_os + c_ss) t - c_ss t^T.
// (c_os, c_ss) = (1, 1) gives the MP2 density (T~ = 2t - t^T); otherwise
// c_ss P_MP2 + (c_os - c_ss) P_OS.
//
// The fused FP64 energy pass runs once with an epilogue that stores
// t = g / D of every ordered occupied pair (both orientations of each unique
// pair), the layout the reference's t2 has per (i, j) block. Both densities
// are then one split-K FP64 MFMA product each over those blocks, every
// operand row K-contiguous:
//   P_vv: K = (pair ij, c); A row a = t_ij[a][.], B row b = cd t_ij[b][.] - ce t_ji[b][.]
//   P_oo: K = (k, ab);      A row i = t_ik,       B row j = cd t_jk - ce t_kj
// (t_ij^ba = t_ji^ab makes the transposed reads of T~ plain reads of the
// mirrored block). Each work item is one 64 x 64 output tile over one K slice, of
// the tiles on or above the diagonal only (both densities are symmetric; at 41/209
// that took the two products from 1848 to 1484 us); a second kernel sums the slices
// of every tile in a fixed order, so the result does not depend on scheduling.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <mutex>
#include <type_traits>
#include <vector>

#include "../../include/ferric_hip.h"
#include "fh_device.h"
#include "fh_host.h"
#include "fh_kernels.h"

namespace fh {
namespace {

constexpr int kDT = 64;   // output tile side
constexpr int kDKP = 8;   // K panel depth
constexpr int kDBuf = 3;  // LDS stages
constexpr int kDPS = kDT * kDKP * 8, kDStage = 3 * kDPS;  // bytes of an operand's panel, of all

// One 64 x 64 tile over one K slice. v_mfma_f64_16x16x4f64 bounds it (8 a wave and panel,
// 512 cycles, against 12 KB of operands): A, B1 and B2 come as they are through three LDS
// stages, loaded directly two panels ahead, and B = cd B1 - ce B2 is formed from the
// fragments of the next panel while the products of this one run; 36 KB and at most 128
// registers put four workgroups on a CU. LDS slots as in pair_f64_kernel. Where the last
// tile's columns are two blocks at most, the four waves take 16 rows each.
// 41/209: 886 us for both densities; 1384 when the panels went through registers, with
// their addresses worked out anew for each.
__global__ __launch_bounds__(256, 4) void density_gemm_kernel(DensArgs d) {
    extern __shared__ __attribute__((aligned(16))) char lds[];
    constexpr int kRow = kDKP * 8;
    const int ntp = d.ntile * (d.ntile + 1) / 2;
    const int64_t item = xcd_remap(blockIdx.x, gridDim.x);
    const int s = (int)(item / ntp);
    int tm, tn;  // both densities are symmetric: the tiles tm <= tn
    decode_tile_pair((int)(item % ntp), d.ntile, tm, tn);
    const int64_t per = (d.kpanels + d.splits - 1) / d.splits;
    const int64_t p0 = std::min(d.kpanels, (int64_t)s * per);
    const int count = (int)(std::min(d.kpanels, p0 + per) - p0);
    const int lane = threadIdx.x % kWave, r = lane % 16, g = lane / 16;
    const int wid = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
    const int limA = std::min(kDT, d.mdim - tm * kDT), limB = std::min(kDT, d.mdim - tn * kDT);
    const bool narrow = limB <= 32 && tm != tn;
    const int rowA = narrow ? 16 * wid : wid / 2 * 32, rowB = narrow ? 0 : wid % 2 * 32;

    // K runs over outer blocks o (VV: the pair (i, j); OO: the shared occupied) of `inner`
    // contiguous elements. Rows past the end repeat the last one, for elements that the
    // reduction does not read.
    const bool vv = d.mode == DensMode::VV;
    const int64_t vp = d.nvir_pad, blk = vp * vp, inner = vv ? vp : blk;
    const int row = 16 * wid + lane / 4;
    const int64_t chunk = ((lane % 4) ^ lds_spread(lane / 16)) * 2;
    const int64_t ra = tm * kDT + std::min(row, limA - 1), rb = tn * kDT + std::min(row, limB - 1);
    const int64_t s1 = vv ? vp : d.nocc * blk, s2 = vv ? vp : blk;
    const int64_t off[3] = {ra * s1 + chunk, rb * s1 + chunk, rb * s2 + chunk};
    int64_t o = p0 * kDKP / inner, f = p0 * kDKP % inner;
    int oi = (int)(o / d.nocc), oj = (int)(o % d.nocc);  // VV
    int ahead = count;
    uint32_t to = 0;
    // Past the last panel it is loaded again and not read.
    auto fetch = [&] {
        const double *b1 = d.tamp + o * blk + f;
        const double *b2 =
            d.tamp + (vv ? (int64_t)oj * d.nocc + oi : o * d.nocc) * blk + f;
#pragma unroll
        for (int op = 0; op < 3; ++op)
            __builtin_amdgcn_global_load_lds((GlobalPtr)((op == 2 ? b2 : b1) + off[op]),
                                             (LdsPtr)(lds + to + op * kDPS + 16 * wid * kRow), 16,
                                             0, 0);
        to = to + kDStage == kDBuf * kDStage ? 0 : to + kDStage;
        if (--ahead > 0) {
            f += kDKP;
            if (f == inner) {
                f = 0;
                ++o;
                if (++oj == d.nocc) {
                    oj = 0;
                    ++oi;
                }
            }
        }
    };
    const uint32_t slot = (uint32_t)(g ^ lds_spread(r / 4)) * 16;
    const uint32_t xa = (uint32_t)(rowA + r) * kRow + slot, xb = (uint32_t)(rowB + r) * kRow + slot;
    v2d fa[2][2], f1[2][2], f2[2][2];
    uint32_t cur = 0;
    auto read = [&](int h) {
        const char *q = lds + cur;
#pragma unroll
        for (int k = 0; k < 2; ++k) {
            // the narrow layout's second row block is not used
            fa[h][k] = *(const v2d *)(q + (narrow ? xa : xa + k * 16 * kRow));
            f1[h][k] = *(const v2d *)(q + kDPS + xb + k * 16 * kRow);
            f2[h][k] = *(const v2d *)(q + 2 * kDPS + xb + k * 16 * kRow);
        }
        cur = cur + kDStage == kDBuf * kDStage ? 0 : cur + kDStage;
        __builtin_amdgcn_sched_barrier(0);
    };
    v4d acc[2][2];
#pragma unroll
    for (int x = 0; x < 2; ++x)
#pragma unroll
        for (int y = 0; y < 2; ++y) acc[x][y] = (v4d){0, 0, 0, 0};
    auto products = [&](int h, auto nx, auto ny) {
#pragma unroll
        for (int e = 0; e < 2; ++e)
#pragma unroll
            for (int y = 0; y < decltype(ny)::value; ++y) {
                const double fb = d.cd * f1[h][y][e] - d.ce * f2[h][y][e];
#pragma unroll
                for (int x = 0; x < decltype(nx)::value; ++x)
                    acc[x][y] = __builtin_amdgcn_mfma_f64_16x16x4f64(fa[h][x][e], fb, acc[x][y], 0,
                                                                     0, 0);
            }
    };
    auto meet = [&] {  // the next panel is in, the last one is read by every wave
        __builtin_amdgcn_sched_barrier(0);
        asm volatile("s_waitcnt vmcnt(3) lgkmcnt(0)\n\ts_barrier" ::: "memory");
        __builtin_amdgcn_sched_barrier(0);
    };
    auto run = [&](auto nx, auto ny) {
        int p = 0;
        for (; p + 2 <= count; p += 2) {
            meet();
            fetch();
            read(1);
            products(0, nx, ny);
            meet();
            fetch();
            read(0);
            products(1, nx, ny);
        }
        if (p < count) products(0, nx, ny);
    };
    using std::integral_constant;
    const int nx = narrow ? 1 : std::min(2, std::max(0, (limA - rowA + 15) / 16));
    const int ny = std::min(2, std::max(0, (limB - rowB + 15) / 16));
    if (count > 0) {  // uniform; an empty slice stores zeros
#pragma unroll
        for (int k = 0; k < kDBuf; ++k) {
            fetch();
            __builtin_amdgcn_sched_barrier(0);
        }
        asm volatile("s_waitcnt vmcnt(6)\n\ts_barrier" ::: "memory");
        __builtin_amdgcn_sched_barrier(0);
        read(0);
        // The same barriers on every side.
        if (nx == 2 && ny == 2)
            run(integral_constant<int, 2>{}, integral_constant<int, 2>{});
        else if (nx == 1 && ny == 2)
            run(integral_constant<int, 1>{}, integral_constant<int, 2>{});
        else if (nx == 2 && ny == 1)
            run(integral_constant<int, 2>{}, integral_constant<int, 1>{});
        else if (nx == 1 && ny == 1)
            run(integral_constant<int, 1>{}, integral_constant<int, 1>{});
        else
            run(integral_constant<int, 0>{}, integral_constant<int, 0>{});
        asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory");
    }
    // partial tile, row-major 64 x 64
    double *out = d.partial + item * (int64_t)(kDT * kDT);
#pragma unroll
    for (int x = 0; x < 2; ++x) {
        if (narrow && x == 1) break;
#pragma unroll
        for (int y = 0; y < 2; ++y)
#pragma unroll
            for (int v = 0; v < 4; ++v)
                out[(rowA + x * 16 + out_row<double>(g, v)) * kDT + rowB + y * 16 + r] =
                    acc[x][y][v];
    }
}

// out[m][n] = out[n][m] = scale * sum over slices s = 0, 1, ... of the tile's partials:
// 64 elements of one tile a block, the slices dealt to sixteen groups of threads (group
// w takes s = w, w + 16, ...) whose sums are added in group order. One thread per
// element took 767 us for the 2048 slices of P_oo at 41/209, on the latency of its loads.
constexpr int kRG = 16;
__global__ __launch_bounds__(64 * kRG) void density_reduce_kernel(DensArgs d) {
    const int ntp = d.ntile * (d.ntile + 1) / 2;
    const int e = (int)(blockIdx.x % (kDT * kDT / 64)) * 64 + threadIdx.x % 64;
    const int t = (int)(blockIdx.x / (kDT * kDT / 64)), w = threadIdx.x / 64;
    int tm, tn;
    decode_tile_pair(t, d.ntile, tm, tn);
    const double *p = d.partial + (int64_t)t * kDT * kDT + e;
    double acc = 0.0;
#pragma unroll 8
    for (int s = w; s < d.splits; s += kRG) acc += p[(int64_t)s * ntp * kDT * kDT];
    __shared__ double part[kRG][64];
    part[w][threadIdx.x % 64] = acc;
    __syncthreads();
    if (w != 0) return;
    for (int k = 1; k < kRG; ++k) acc += part[k][threadIdx.x];
    const int m = tm * kDT + e / kDT, n = tn * kDT + e % kDT;
    if (m >= d.mdim || n >= d.mdim) return;
    // A diagonal tile holds both of (m, n) and (n, m): each writes its own.
    d.out[(int64_t)m * d.mdim + n] = d.scale * acc;
    if (tm != tn) d.out[(int64_t)n * d.mdim + m] = d.scale * acc;
}

}  // namespace

hipError_t launch_density(const DensArgs &d, hipStream_t st) {
    const int ntp = d.ntile * (d.ntile + 1) / 2;
    const int64_t nitems = (int64_t)ntp * d.splits;
    if (nitems <= 0 || nitems > 0x7fffffffLL || d.mdim <= 0 || d.nvir_pad % kDKP != 0 ||
        d.kpanels / d.splits >= 0x7fffffffLL)
        return hipErrorInvalidValue;
    hipLaunchKernelGGL(density_gemm_kernel, dim3((unsigned)nitems), dim3(256), kDBuf * kDStage, st,
                       d);
    hipLaunchKernelGGL(density_reduce_kernel, dim3((unsigned)(ntp * (kDT * kDT / 64))),
                       dim3(64 * kRG), 0, st, d);
    return hipGetLastError();
}

namespace {

// Slices per output tile: enough items to fill the chip (about 2048), each
// slice at least 16 panels deep.
int density_splits(int ntile, int64_t kpanels) {
    const int64_t tiles = (int64_t)ntile * (ntile + 1) / 2;
    int64_t s = std::max<int64_t>(1, 2048 / tiles);
    s = std::min<int64_t>(s, std::max<int64_t>(1, kpanels / 16));
    return (int)s;
}

fh_status density_core(State &s, const void *b_dev, fh_dtype b_dtype, size_t naux, size_t nocc,
                       size_t nvir, const double *eps, size_t first_occ, size_t nocc_total,
                       double c_os, double c_ss, hipStream_t stream, fh_spin_components *out,
                       double *p_oo, double *p_vv) {
    const EnergyPlan pl = plan_energy(nocc, nvir, naux, Prec::F64);
    const size_t vp = (size_t)pl.nvir_pad;
    const size_t amp_bytes = sizeof(double) * nocc * nocc * vp * vp;
    DensArgs vv, oo;
    vv.mode = DensMode::VV;
    vv.nocc = (int)nocc;
    vv.nvir_pad = (int)vp;
    vv.mdim = (int)vp;
    vv.ntile = (int)((vp + kDT - 1) / kDT);
    vv.kpanels = (int64_t)(nocc * nocc * vp / kDKP);
    vv.splits = density_splits(vv.ntile, vv.kpanels);
    vv.cd = c_os + c_ss;
    vv.ce = c_ss;
    vv.scale = 1.0;
    oo = vv;
    oo.mode = DensMode::OO;
    oo.mdim = (int)nocc;
    oo.ntile = (int)((nocc + kDT - 1) / kDT);
    oo.kpanels = (int64_t)(nocc * vp * vp / kDKP);
    oo.splits = density_splits(oo.ntile, oo.kpanels);
    oo.scale = -1.0;
    const size_t part_elems =
        std::max((size_t)vv.ntile * (vv.ntile + 1) / 2 * vv.splits,
                 (size_t)oo.ntile * (oo.ntile + 1) / 2 * oo.splits) *
        kDT * kDT;
    std::vector<std::pair<int, size_t>> req = {
        {kSlotDensAmp, amp_bytes},
        {kSlotDensPart, sizeof(double) * part_elems},
        {kSlotDensOut, sizeof(double) * (vp * vp + nocc * nocc)},
    };
    fh_status st = reserve(s, req);
    if (st != FH_OK) return st;
    const int64_t blk = (int64_t)(vp * vp);
    double *amp = (double *)s.slots[kSlotDensAmp].ptr;
    const AmpOut amp_out{amp, (int64_t)nocc * blk, blk, (int64_t)vp, (int)vp, true};
    st = energy_core(s, b_dev, b_dtype, naux, nocc, nvir, eps, first_occ, nocc_total, NAN,
                     Prec::F64, stream, out, nullptr, &pl, nullptr, 0, &amp_out);
    if (st != FH_OK) return st;
    double *dout = (double *)s.slots[kSlotDensOut].ptr;
    vv.tamp = oo.tamp = amp;
    vv.partial = oo.partial = (double *)s.slots[kSlotDensPart].ptr;
    vv.out = dout;
    oo.out = dout + vp * vp;
    hipError_t he = launch_density(vv, stream);
    if (he == hipSuccess) he = launch_density(oo, stream);
    if (he != hipSuccess) {
        (void)hipGetLastError();
        return fail(FH_KERNEL, "density kernels: %s", hipGetErrorString(he));
    }
    s.pending.kernel_launches += 4;
    std::vector<double> h(vp * vp + nocc * nocc);
    st = hip_check(hipMemcpyAsync(h.data(), dout, sizeof(double) * h.size(),
                                  hipMemcpyDeviceToHost, stream),
                   "D2H densities");
    if (st != FH_OK) return st;
    st = hip_check(hipStreamSynchronize(stream), "stream sync");
    if (st != FH_OK) return st;
    s.pending.d2h_bytes += sizeof(double) * h.size();
    for (size_t a = 0; a < nvir; ++a)
        for (size_t b = 0; b < nvir; ++b) p_vv[a * nvir + b] = h[a * vp + b];
    for (size_t k = 0; k < nocc * nocc; ++k) p_oo[k] = h[vp * vp + k];
    return FH_OK;
}

fh_status density_entry(const void *b, bool host, fh_dtype b_dtype, size_t naux, size_t nocc,
                        size_t nvir, const double *eps, size_t n_eps, size_t first_occ,
                        size_t nocc_total, double c_os, double c_ss, void *stream,
                        fh_spin_components *out, double *p_oo, double *p_vv) {
    State &s = state();
    std::lock_guard<std::mutex> lk(s.mu);
    clear_error();
    s.stats.calls++;
    s.pending = Pending{};
    if (!out || (nocc && !p_oo) || (nvir && !p_vv)) return fail(FH_LAYOUT, "null output pointer");
    if (!std::isfinite(c_os) || !std::isfinite(c_ss))
        return fail(FH_LAYOUT, "spin scaling coefficients must be finite");
    if (b_dtype != FH_DT_F64 && b_dtype != FH_DT_F32)
        return fail(FH_LAYOUT, "unknown b_dtype %d", (int)b_dtype);
    bool empty = false;
    fh_status st = check_shapes(naux, nocc, nvir, n_eps, first_occ, nocc_total, &empty);
    if (st != FH_OK) return st;
    if (empty) {
        *out = fh_spin_components{0.0, 0.0, 0.0};
        for (size_t k = 0; k < nocc * nocc; ++k) p_oo[k] = 0.0;
        for (size_t k = 0; k < nvir * nvir; ++k) p_vv[k] = 0.0;
        commit(s, Prec::F64, true, false);
        return FH_OK;
    }
    if (!b || !eps) return fail(FH_LAYOUT, "null input pointer");
    st = ensure_device(s);
    if (st != FH_OK) return st;
    const void *b_dev = b;
    hipStream_t strm = (hipStream_t)stream;
    if (host) {
        const size_t bbytes = sizeof(double) * naux * nocc * nvir;
        st = reserve(s, {{kSlotStage, bbytes}});
        if (st != FH_OK) return st;
        st = hip_check(hipMemcpyAsync(s.slots[kSlotStage].ptr, b, bbytes, hipMemcpyHostToDevice,
                                      strm),
                       "H2D b_ov");
        if (st != FH_OK) return st;
        s.pending.h2d_bytes += bbytes;
        b_dev = s.slots[kSlotStage].ptr;
    }
    st = density_core(s, b_dev, b_dtype, naux, nocc, nvir, eps, first_occ, nocc_total, c_os, c_ss,
                      strm, out, p_oo, p_vv);
    if (st != FH_OK) return st;
    commit(s, Prec::F64, true, false);
    return FH_OK;
}

}  // namespace
}  // namespace fh

using namespace fh;

extern "C" {

fh_status fh_rimp2_mp2_density(const double *b_ov, size_t naux, size_t nocc, size_t nvir,
                               const double *eps, size_t n_eps, size_t first_occ,
                               size_t nocc_total, double c_os, double c_ss,
                               fh_spin_components *out, double *p_oo, double *p_vv) {
    return density_entry(b_ov, true, FH_DT_F64, naux, nocc, nvir, eps, n_eps, first_occ,
                         nocc_total, c_os, c_ss, nullptr, out, p_oo, p_vv);
}

fh_status fh_rimp2_mp2_density_dev(const void *b_dev, fh_dtype b_dtype, size_t naux, size_t nocc,
                                   size_t nvir, const double *eps, size_t n_eps, size_t first_occ,
                                   size_t nocc_total, double c_os, double c_ss, void *stream,
                                   fh_spin_components *out, double *p_oo, double *p_vv) {
    return density_entry(b_dev, false, b_dtype, naux, nocc, nvir, eps, n_eps, first_occ,
                         nocc_total, c_os, c_ss, stream, out, p_oo, p_vv);
}

}  // extern "C"
