// Fused RI-MP2 pair kernels for gfx950 (CDNA4 MFMA): the energy, and phase A
// of the adjoint.
//
// Replaces the per-i tail GEMM G_i = B_i^T B_tail plus the host pair loop of
// the reference (crates/ferric-mp2/src/rimp2.rs:1399-1544; device twin
// crates/ferric-mp2/src/rimp2_gpu.rs:198-271) with one launch in which
// K_ij = B_i^T B_j never leaves the chip.
//
// Work item = (unique occupied pair i <= j, tile pair tA <= tB over the
// virtuals). A workgroup (4 waves, 2x2) computes, over the whole Q range,
//   C1(a, b) = sum_Q B_i[Q, a] B_j[Q, b] = (ia|jb)       a in A, b in B
//   C2(a, b) = sum_Q B_j[Q, a] B_i[Q, b] = (ib|ja)
// so g_ab and g_ba of every (a, b) sit in the same lane and register. The
// pair loop's terms for (a, b) and for the mirrored (b, a) are
//   OS: (g_ab^2 + g_ba^2)/D        SS: (g_ab - g_ba)^2/D
// (the reference's g_ab^2/D and g_ab(g_ab - g_ba)/D summed over both
// orientations; D is symmetric in a, b). A diagonal tile (tA == tB) covers
// each unordered {a, b} twice and takes weight 1/2; the occupied pair takes
// the reference's fac = 1 (i == j) or 2 (i < j). Every term is FP64 with one
// divide; lane sums are compensated and every reduction runs in a fixed
// order, so the result does not depend on scheduling.
//
// Adjoint epilogue (same contraction): with t = g/D and
// T~ = (c_os + c_ss) t - c_ss t^T (rimp2.rs:1987-2011), it writes the T~ block
// of the pair for the phase-B/C GEMMs (adjoint.hip) and the per-item sums of
// t*T~ by virtual row, virtual column and in total, from which dE/deps
// follows (dE/dD = -t T~).
//
// Operands come from the packed K-major layout of pack.hip:
// row (i*nvir_pad + a) holds B^Q_ia for Q = 0..naux_pad-1.
#include <hip/hip_runtime.h>
#include <math.h>
#include <stdint.h>

#include "fh_device.h"
#include "fh_kernels.h"
#include "pair_body.h"

namespace fh {

namespace {

__device__ __forceinline__ pair::Item decode_item(const EnergyArgs &a) {
    pair::Item it;
    it.id = xcd_remap((int64_t)blockIdx.x, a.nitems);
    const int64_t p = it.id / a.ntp;
    const int tp = (int)(it.id % a.ntp);
    if (a.i_fixed >= 0) {
        it.i = a.i_fixed;
        it.j = a.i_fixed + (int)p;
    } else {
        decode_pair(p, a.nocc, it.i, it.j);
    }
    decode_tile_pair(tp, a.ntile, it.ta, it.tb);
    return it;
}

template <typename T, int TILE, int KP, bool ADJ, bool SIGNED = false, bool FLUSH = false,
          bool AMP = false>
__global__ __launch_bounds__(256) void pair_k4_kernel(EnergyArgs a) {
    __shared__ __attribute__((aligned(16))) pair::K4Lds<T, TILE, KP> lds;
    pair::pair_k4_body<T, TILE, KP, ADJ, false, SIGNED, FLUSH, AMP>(a, decode_item(a), lds);
}

// FP64 at tile 64, the energies and the amplitude passes: the items, operands and
// epilogues of pair_k4_body, with 8-deep panels brought into two LDS stages by direct
// loads, a panel ahead. v_mfma_f64_16x16x4f64 holds a SIMD 64 cycles, so 16 products a
// wave and panel, for four waves, outlast a load; 32 KB and 118 registers let four
// workgroups share a CU, and cover one another's LDS reads, barriers, starts, ends and
// epilogues. The fragments are read before the next panel's loads are issued: the other
// order waits for the loads to be taken (1549 us). Where the last tile of the virtuals
// holds at most two blocks, the four waves take 16 rows each of it instead of leaving
// half of them idle (209 virtuals: 3 of 10 items).
// 41/209/960: the call takes 1500 us (54 TFLOP/s of products issued at about 2.1 GHz,
// what the load leaves of 2.4) against 2386 for the register-staged body (45% of the
// issue slots, bank conflicts, an LDS write per operand byte, two workgroups). Three
// stages, three workgroups and the next panel's fragments read ahead 1573; 16-deep panels
// in two stages, two workgroups 1677.
constexpr int kPK = 8, kPBuf = 2;      // panel depth, stages
constexpr int kPS = 64 * kPK * 8;      // one operand's panel
constexpr int kPStage = 4 * kPS;

template <bool AMP>
__global__ __launch_bounds__(256, 4) void pair_f64_kernel(EnergyArgs a) {
    extern __shared__ __attribute__((aligned(16))) char lds[];
    constexpr int TILE = 64, NB = 2, kRow = kPK * 8;
    const pair::Item it = decode_item(a);
    const int A0 = it.ta * TILE, B0 = it.tb * TILE;
    const pair::SplitQ sq(it, a.naux_pad, kPK);
    const int limA = min(TILE, a.nvir_pad - A0), limB = min(TILE, a.nvir_pad - B0);
    const int lane = threadIdx.x % kWave;
    const int wid = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
    const bool narrow = limB <= 32 && it.ta != it.tb;  // then limA = 64
    const pair::Lane L{narrow ? A0 + 16 * wid : A0, B0, narrow ? 0 : wid / 2,
                       narrow ? 0 : wid % 2, lane % 16, lane / 16};
    bool rv[NB], cv[NB];
#pragma unroll
    for (int k = 0; k < NB; ++k) {
        rv[k] = narrow ? k == 0 : L.wr * 32 + k * 16 < limA;
        cv[k] = L.wc * 32 + k * 16 < limB;
    }

    // Operands as in pair_k4_body. A wave stages rows 16 wid .. 16 wid + 15 of each;
    // rows past the tile's last repeat it, in blocks that no product reads.
    const double *b = (const double *)a.op0;
    const int64_t ld = a.naux_pad;
    const double *src[4] = {
        b + ((int64_t)it.i * a.nvir_pad + A0) * ld, b + ((int64_t)it.j * a.nvir_pad + B0) * ld,
        b + ((int64_t)(sq.single ? it.i : it.j) * a.nvir_pad + A0) * ld,
        b + ((int64_t)(sq.single ? it.j : it.i) * a.nvir_pad + B0) * ld};
    const int row = 16 * wid + lane / 4;
    const uint32_t chunk = ((lane % 4) ^ lds_spread(lane / 16)) * 16;
    const uint32_t offa = (uint32_t)min(row, limA - 1) * (uint32_t)(ld * 8) + chunk;
    const uint32_t offb = (uint32_t)min(row, limB - 1) * (uint32_t)(ld * 8) + chunk;
    // Past the last iteration its panels are loaded again and not read. (naux_pad is even
    // in panels, so a single-product item has its two in every iteration.)
    uint32_t to = 0;
    int ahead = 0;
    auto fetch = [&] {
        const int q0 = min(ahead++, sq.iters - 1) * sq.step;
#pragma unroll
        for (int op = 0; op < 4; ++op) {
            const char *p = (const char *)(src[op] + (op < 2 ? q0 : q0 + sq.off23));
            __builtin_amdgcn_global_load_lds((GlobalPtr)(p + (op & 1 ? offb : offa)),
                                             (LdsPtr)(lds + to + op * kPS + 16 * wid * kRow), 16,
                                             0, 0);
        }
        to = to + kPStage == kPBuf * kPStage ? 0 : to + kPStage;
    };
    const uint32_t slot = (uint32_t)(L.g ^ lds_spread(L.r / 4)) * 16;
    const uint32_t ra = (uint32_t)((narrow ? 16 * wid : L.wr * 32) + L.r) * kRow + slot;
    const uint32_t rb = (uint32_t)(L.wc * 32 + L.r) * kRow + slot;
    v2d f0[NB], f1[NB], f2[NB], f3[NB];
    uint32_t cur = 0;
    auto read = [&] {
        const char *s = lds + cur;
#pragma unroll
        for (int k = 0; k < NB; ++k) {
            // the narrow layout's second row block is not used: any row in the stage
            const uint32_t xa = narrow ? ra : ra + k * 16 * kRow, xb = rb + k * 16 * kRow;
            f0[k] = *(const v2d *)(s + xa);
            f1[k] = *(const v2d *)(s + kPS + xb);
            f2[k] = *(const v2d *)(s + 2 * kPS + xa);
            f3[k] = *(const v2d *)(s + 3 * kPS + xb);
        }
        cur = cur + kPStage == kPBuf * kPStage ? 0 : cur + kPStage;
        __builtin_amdgcn_sched_barrier(0);
    };
    v4d acc1[NB][NB], acc2[NB][NB];
#pragma unroll
    for (int x = 0; x < NB; ++x)
#pragma unroll
        for (int y = 0; y < NB; ++y) acc1[x][y] = acc2[x][y] = (v4d){0, 0, 0, 0};
    auto products = [&](auto nx, auto ny) {
#pragma unroll
        for (int e = 0; e < 2; ++e)
#pragma unroll
            for (int x = 0; x < decltype(nx)::value; ++x)
#pragma unroll
                for (int y = 0; y < decltype(ny)::value; ++y) {
                    acc1[x][y] = __builtin_amdgcn_mfma_f64_16x16x4f64(f0[x][e], f1[y][e],
                                                                      acc1[x][y], 0, 0, 0);
                    acc2[x][y] = __builtin_amdgcn_mfma_f64_16x16x4f64(f2[x][e], f3[y][e],
                                                                      acc2[x][y], 0, 0, 0);
                }
    };
    auto meet = [&] {  // the next panel is in, the last one is read by every wave
        __builtin_amdgcn_sched_barrier(0);
        asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory");
        __builtin_amdgcn_sched_barrier(0);
    };
    auto run = [&](auto nx, auto ny) {
        for (int f = 0; f < sq.iters; ++f) {
            meet();
            read();
            fetch();
            products(nx, ny);
        }
    };
    using std::integral_constant;
    const int nx = rv[1] ? 2 : rv[0] ? 1 : 0, ny = cv[1] ? 2 : cv[0] ? 1 : 0;
    fetch();
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
    asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory");
    if (sq.single)
        pair::derive_c2<TILE, double>(it, L, acc1, acc2, pair::RowOf<double>{}, (double *)lds);
    if constexpr (AMP)
        pair::amp_store<TILE>(a, it, L, acc1, acc2, rv, cv, pair::RowOf<double>{});
    pair::energy_epilogue<TILE>(a, it, L, acc1, acc2, rv, cv, pair::RowOf<double>{},
                                pair::NoCorr{});
}

// Opposite-spin rectangle: item (i, J, tA, tB), J and tB on the beta side;
// the items of alpha row i are contiguous.
template <typename T, int TILE, int KP, bool FLUSH = false>
__global__ __launch_bounds__(256) void pair_rect_kernel(EnergyArgs a) {
    __shared__ __attribute__((aligned(16))) pair::K4Lds<T, TILE, KP> lds;
    pair::Item it;
    it.id = xcd_remap((int64_t)blockIdx.x, a.nitems);
    const int64_t ntp = (int64_t)a.ntile * a.ntile_b;
    const int64_t p = it.id / ntp;
    const int t = (int)(it.id % ntp);
    it.i = (int)(p / a.nocc_b);
    it.j = (int)(p % a.nocc_b);
    it.ta = t / a.ntile_b;
    it.tb = t % a.ntile_b;
    pair::pair_k4_body<T, TILE, KP, false, true, false, FLUSH>(a, it, lds);
}


// BF16x3 energy on eight waves from the fragment-order operand
// (pair_bf16x3_w8f_body), TILE = 128 or 64 (at 64: 106 VGPRs, two workgroups
// per CU).
template <int TILE>
__global__ __launch_bounds__(512) void pair_bf16x3_w8f_kernel(EnergyArgs a) {
    __shared__ __attribute__((aligned(16))) pair::Bf16Lds<TILE> lds;
    pair::pair_bf16x3_w8f_body<TILE>(a, decode_item(a), lds);
}

template <int TILE, bool ADJ>
__global__ __launch_bounds__(256) void pair_bf16x3_kernel(EnergyArgs a) {
    __shared__ __attribute__((aligned(16))) pair::Bf16Lds<TILE> lds;
    pair::pair_bf16x3_body<TILE, ADJ>(a, decode_item(a), lds);
}

// ---------------------------------------------------------------------------
// Deterministic reductions: per occupied row i (items of row i are contiguous:
// pairs (i, j >= i) start at p0 = i*nocc - i(i-1)/2), then an ascending fold
// over i (the reference's i-ordered serial sum, rimp2.rs:1533-1538).
// ---------------------------------------------------------------------------
// The fold is the last row's workgroup's: a launch of its own read the rows one after
// another (11 us at 41 rows). 0 between launches; the calls that run these kernels hold
// the library's lock and wait for them.
__device__ unsigned int rows_done;

__device__ __forceinline__ void fold_rows(const double *rows, int nocc, const int *wide,
                                          double *result) {
    __shared__ double part[256][4];
    __shared__ unsigned int before;
    if (threadIdx.x == 0) {
        __threadfence();  // this row, written by this thread
        before = atomicAdd(&rows_done, 1u);
    }
    __syncthreads();
    if (before != gridDim.x - 1) return;
    __threadfence();
    KSum sum;  // thread 0: e_os, thread 64: e_ss, in row order
    const bool folds = threadIdx.x % kWave == 0 && threadIdx.x < 2 * kWave;
    const int c = 2 * (threadIdx.x / kWave);
    for (int i0 = 0; i0 < nocc; i0 += 256) {
        const int n = min(256, nocc - i0);
        if ((int)threadIdx.x < n) {
            const int64_t i = i0 + threadIdx.x;
            double v[4];
#pragma unroll
            for (int k = 0; k < 4; ++k) part[threadIdx.x][k] = v[k] = rows[4 * i + k];
            result[2 + 2 * i] = v[0] + v[1];
            result[3 + 2 * i] = v[2] + v[3];
        }
        __syncthreads();
        if (folds)
            for (int k = 0; k < n; ++k) sum.merge(part[k][c], part[k][c + 1]);
        __syncthreads();
    }
    if (folds) result[threadIdx.x / kWave] = sum.value();
    if (wide && threadIdx.x == 0) result[2 + 2 * (int64_t)nocc] = *wide ? 1.0 : 0.0;
    if (threadIdx.x == 0) rows_done = 0;
}

__global__ __launch_bounds__(256) void reduce_rows_kernel(const double *__restrict__ ip, int nocc,
                                                          int ntp, const int *wide, double *rows,
                                                          double *result) {
    const int i = blockIdx.x;
    const int64_t p0 = (int64_t)i * nocc - (int64_t)i * (i - 1) / 2;
    const int64_t w0 = p0 * ntp, w1 = (p0 + (nocc - i)) * ntp;
    KSum os, ss;
    for (int64_t w = w0 + threadIdx.x; w < w1; w += 256) {
        os.merge(ip[4 * w], ip[4 * w + 1]);
        ss.merge(ip[4 * w + 2], ip[4 * w + 3]);
    }
    pair::block_store(os, ss, 1.0, rows + 4 * i);
    fold_rows(rows, nocc, wide, result);
}

// Rectangle rows: items [i*per_row, (i+1)*per_row) belong to alpha row i.
__global__ __launch_bounds__(256) void reduce_rect_rows_kernel(const double *__restrict__ ip,
                                                               int64_t per_row, int nocc,
                                                               const int *wide, double *rows,
                                                               double *result) {
    const int i = blockIdx.x;
    KSum os, ss;
    for (int64_t w = (int64_t)i * per_row + threadIdx.x; w < (int64_t)(i + 1) * per_row;
         w += 256) {
        os.merge(ip[4 * w], ip[4 * w + 1]);
        ss.merge(ip[4 * w + 2], ip[4 * w + 3]);
    }
    pair::block_store(os, ss, 1.0, rows + 4 * i);
    fold_rows(rows, nocc, wide, result);
}

template <typename K>
hipError_t launch_items(K kern, const EnergyArgs &a, hipStream_t st, int threads = 256) {
    hipLaunchKernelGGL(kern, dim3((unsigned)a.nitems), dim3(threads), 0, st, a);
    return hipGetLastError();
}

// pair_f64_kernel's row offsets inside a tile are 32-bit: past 8388607 aux functions the
// register-staged body, whose offsets are not.
template <bool AMP>
hipError_t launch_f64(const EnergyArgs &a, hipStream_t st) {
    if (64LL * a.naux_pad * 8 > 0xffffffffLL)
        return launch_items(pair_k4_kernel<double, 64, 16, false, false, false, AMP>, a, st);
    if (a.naux_pad < 16 || a.naux_pad % 16 != 0 || a.nvir_pad % 16 != 0)
        return hipErrorInvalidValue;
    hipLaunchKernelGGL(pair_f64_kernel<AMP>, dim3((unsigned)a.nitems), dim3(256),
                       kPBuf * kPStage, st, a);
    return hipGetLastError();
}

}  // namespace

hipError_t launch_energy(const EnergyArgs &a, hipStream_t st) {
    if (a.nitems <= 0 || a.nitems > 0x7fffffffLL) return hipErrorInvalidValue;
    hipError_t e = hipErrorInvalidValue;
    if (a.amp.base) {  // FP64 energy that also stores the amplitudes
        if (a.prec != Prec::F64 || a.q_neg < a.naux_pad) return hipErrorInvalidValue;
        if (a.tile == 128) e = launch_items(pair_k4_kernel<double, 128, 16, false, false, false, true>, a, st);
        else if (a.tile == 64) e = launch_f64<true>(a, st);
        else if (a.tile == 32) e = launch_items(pair_k4_kernel<double, 32, 16, false, false, false, true>, a, st);
        return e;
    }
    if (a.q_neg < a.naux_pad) {  // signed factor: FP64 / FP32 only
        if (a.prec == Prec::F64) {
            if (a.tile == 128) e = launch_items(pair_k4_kernel<double, 128, 16, false, true>, a, st);
            else if (a.tile == 64) e = launch_items(pair_k4_kernel<double, 64, 16, false, true>, a, st);
            else if (a.tile == 32) e = launch_items(pair_k4_kernel<double, 32, 16, false, true>, a, st);
        } else if (a.prec == Prec::F32) {
            if (a.tile == 128) e = launch_items(pair_k4_kernel<float, 128, 16, false, true>, a, st);
            else if (a.tile == 64) e = launch_items(pair_k4_kernel<float, 64, 16, false, true>, a, st);
            else if (a.tile == 32) e = launch_items(pair_k4_kernel<float, 32, 16, false, true>, a, st);
        }
        return e;
    }
    switch (a.prec) {
    case Prec::F64:
        if (a.tile == 128) e = launch_items(pair_k4_kernel<double, 128, 16, false>, a, st);
        else if (a.tile == 64) e = launch_f64<false>(a, st);
        else if (a.tile == 32) e = launch_items(pair_k4_kernel<double, 32, 16, false>, a, st);
        break;
    case Prec::F32:
        if (a.tile == 128) e = launch_items(pair_k4_kernel<float, 128, 16, false>, a, st);
        else if (a.tile == 64) e = launch_items(pair_k4_kernel<float, 64, 16, false>, a, st);
        else if (a.tile == 32) e = launch_items(pair_k4_kernel<float, 32, 16, false>, a, st);
        break;
    case Prec::MIXED:
        if (a.tile == 128) e = launch_items(pair_k4_kernel<float, 128, 16, false, false, true>, a, st);
        else if (a.tile == 64) e = launch_items(pair_k4_kernel<float, 64, 16, false, false, true>, a, st);
        else if (a.tile == 32) e = launch_items(pair_k4_kernel<float, 32, 16, false, false, true>, a, st);
        break;
    case Prec::BF16X3:
        if (a.tile == 128) {
            if (a.opf) e = launch_items(pair_bf16x3_w8f_kernel<128>, a, st, 512);
        }
        else if (a.tile == 64 && a.opf) e = launch_items(pair_bf16x3_w8f_kernel<64>, a, st, 512);
        else if (a.tile == 64) e = launch_items(pair_bf16x3_kernel<64, false>, a, st);
        else if (a.tile == 32) e = launch_items(pair_bf16x3_kernel<32, false>, a, st);
        break;
    case Prec::FP8:
        e = launch_energy_fp8(a, st);
        break;
    case Prec::I8X4:
        e = launch_energy_i8x4(a, st);
        break;
    }
    return e;
}

hipError_t launch_adjoint_pairs(const EnergyArgs &a, hipStream_t st) {
    if (a.nitems <= 0 || a.nitems > 0x7fffffffLL) return hipErrorInvalidValue;
    if (a.prec == Prec::I8X4) return launch_adjoint_i8x4(a, st);
    if (a.i_fixed < 0) return hipErrorInvalidValue;
    hipError_t e = hipErrorInvalidValue;
    switch (a.prec) {
    case Prec::F64:
        // 32 or 64 wide (the host caps the FP64 adjoint tile at 64)
        if (a.tile == 64) e = launch_items(pair_k4_kernel<double, 64, 16, true>, a, st);
        else if (a.tile == 32) e = launch_items(pair_k4_kernel<double, 32, 8, true>, a, st);
        break;
    case Prec::BF16X3:
        if (a.tile == 128) e = launch_items(pair_bf16x3_kernel<128, true>, a, st);
        else if (a.tile == 64) e = launch_items(pair_bf16x3_kernel<64, true>, a, st);
        else if (a.tile == 32) e = launch_items(pair_bf16x3_kernel<32, true>, a, st);
        break;
    case Prec::I8X4:
        e = launch_adjoint_i8x4(a, st);
        break;
    default:
        break;
    }
    return e;
}

hipError_t launch_energy_rect(const EnergyArgs &a, hipStream_t st) {
    if (a.nitems <= 0 || a.nitems > 0x7fffffffLL || a.ntile_b <= 0 || a.nocc_b <= 0)
        return hipErrorInvalidValue;
    hipError_t e = hipErrorInvalidValue;
    switch (a.prec) {
    case Prec::F64:
        if (a.tile == 128) e = launch_items(pair_rect_kernel<double, 128, 16>, a, st);
        else if (a.tile == 64) e = launch_items(pair_rect_kernel<double, 64, 16>, a, st);
        else if (a.tile == 32) e = launch_items(pair_rect_kernel<double, 32, 16>, a, st);
        break;
    case Prec::F32:
        if (a.tile == 128) e = launch_items(pair_rect_kernel<float, 128, 16>, a, st);
        else if (a.tile == 64) e = launch_items(pair_rect_kernel<float, 64, 16>, a, st);
        else if (a.tile == 32) e = launch_items(pair_rect_kernel<float, 32, 16>, a, st);
        break;
    case Prec::MIXED:
        if (a.tile == 128) e = launch_items(pair_rect_kernel<float, 128, 16, true>, a, st);
        else if (a.tile == 64) e = launch_items(pair_rect_kernel<float, 64, 16, true>, a, st);
        else if (a.tile == 32) e = launch_items(pair_rect_kernel<float, 32, 16, true>, a, st);
        break;
    case Prec::I8X4:
        e = launch_energy_i8x4_rect(a, st);
        break;
    default:
        break;
    }
    return e;
}

hipError_t launch_rect_reduce(const EnergyArgs &a, hipStream_t st) {
    const int64_t per_row = (int64_t)a.nocc_b * a.ntile * a.ntile_b;
    hipLaunchKernelGGL(reduce_rect_rows_kernel, dim3((unsigned)a.nocc), dim3(256), 0, st,
                       a.item_partials, per_row, a.nocc, a.wide, a.row_partials, a.result);
    return hipGetLastError();
}

hipError_t launch_energy_reduce(const EnergyArgs &a, hipStream_t st) {
    hipLaunchKernelGGL(reduce_rows_kernel, dim3((unsigned)a.nocc), dim3(256), 0, st,
                       a.item_partials, a.nocc, a.ntp, a.wide, a.row_partials, a.result);
    return hipGetLastError();
}

}  // namespace fh
