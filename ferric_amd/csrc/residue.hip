// FP64 and MIXED pair energies in exact residue arithmetic on the INT8 matrix
// cores (residue.h has the number format; MIXED rounds B to FP32 first and takes ten
// moduli, 33 bits of each row).
//
// Why: the FP64 matrix instructions run at 1/64 of the INT8 ones' rate here, so
// sixteen exact INT8 products take about 0.4 of one FP64 product's time. Energy,
// matrix kernel / here: FP64 60/450/1800 23.8 / 14.3 ms, 100/200/2400 18.9 / 10.7,
// 100/900/3600 534 / 292; MIXED 20.0 / 9.1, 17.4 / 6.9 and 387 / 174 ms.
//
// Operand layout. For each modulus k and each 64-deep Q panel p one block of
// rows / 16 kilobytes: kilobyte rg holds the residues of packed rows
// 16 rg .. 16 rg + 15 in MFMA fragment order (lane 16 g + r at byte
// 16 (16 g + r): row r, Q = 16 g .. 16 g + 15 of the panel). A product's step
// (k, p) so reads two contiguous runs, and consecutive steps lie a fixed
// stride apart.
//
// Work item = (occupied pair i <= j, virtual tile pair tA <= tB), tiles of at
// most 16 sixteen-row blocks, split evenly; up to 128 virtuals two orbitals share a
// tile. One 512-thread workgroup per CU takes items in rounds. C1 = (iA | jB)
// and, on an off-diagonal tile pair of i < j, C2 = (jA | iB) run one after the
// other as plain 256 x 256 INT8 products: eight waves as 2 x 4, each up to 8 x 4
// blocks (128 int32 accumulators), operands straight from the L2 into four LDS
// stages, the next step's fragments read while this one's products run. After
// the last panel of a modulus every lane reduces its sums to bytes and stores
// them in the workgroup's scratch (one dword per 16 x 16 block, lane and modulus);
// after the last modulus the waves take blocks off the scratch, rebuild the
// FP64 values and add the energy terms.
//
// What bounds it: at 60/450/1800 the products alone (no reduction, no epilogue) take
// 10.6 of the kernel's 13.6 ms, 2.2 POP/s (the library's INT8 product of the same
// depth reaches 2.0), 7.8 ms with zeros for residues: the chip's power on
// random bytes, not the operand stream. Reducing the sums takes 1.5 ms, rebuilding and the
// energy terms 1.6. Tried and slower: operands staged through registers (27 ms
// then), row 1 of waves half a step behind row 0 with two barriers a step (the
// same), fetching a step's operands in one burst (0.5 ms more).
#include <hip/hip_runtime.h>
#include <math.h>
#include <stdint.h>

#include <algorithm>

#include "fh_device.h"
#include "fh_kernels.h"
#include "pair_body.h"
#include "residue.h"

namespace fh {

namespace {

constexpr int kThreads = 512;
constexpr int kNonTemporal = 2;       // buffer access that leaves the L2 to the operands
constexpr int kQueueStride = 32;      // the round counter's own line, in ints
constexpr int kMaxSplit = 5;          // most workgroups to an item
constexpr int kTB = 16;               // most 16-row blocks of a tile side
constexpr int kStage = 2 * kTB * 1024;  // LDS bytes of one panel of both operands
constexpr int kBuf = 4;                 // panels in the LDS: one in use, three in flight
constexpr int kPlane = kTB * kTB * 256;  // scratch bytes of one modulus of a product
constexpr int planes_of(int n) { return n * kPlane + 256; }  // of a product, and a dump slot

struct Recip {
    float v[res::kMaxN] = {};
};
constexpr Recip recip() {
    Recip r;
    for (int k = 0; k < res::kMaxN; ++k) r.v[k] = 1.0f / (float)res::kMod[k];
    return r;
}
__constant__ const Recip kRecip = recip();

// One orbital and one 64-deep Q panel: the largest |B| of every column (a NaN counts as an
// infinity) and, for the range test, the sum over the virtuals of B^2 at every Q. One read of
// B at the memory's rate; 16 rows of 64 columns in flight a wave.
template <typename Tin>
__global__ __launch_bounds__(256) void residue_scan_kernel(const Tin *__restrict__ b, int64_t nov,
                                                           int naux, int nvir, ResidueRange rr,
                                                           int *wide) {
    const int lane = threadIdx.x % kWave, wid = threadIdx.x / kWave;
    const int i = blockIdx.y, q0 = blockIdx.x * 64 + 16 * wid, n = min(16, naux - q0);
    if (wide && blockIdx.x == 0 && i == 0 && threadIdx.x == 0) *wide = 0;
    const Tin *p = b + (int64_t)q0 * nov + (int64_t)i * nvir;
    __shared__ double part[2][4][64];
    double sum[16];
#pragma unroll
    for (int t = 0; t < 16; ++t) sum[t] = 0.0;
    for (int a0 = 0; a0 < nvir; a0 += 64) {
        const int a = a0 + lane;
        double v[16], m = 0.0;
#pragma unroll
        for (int t = 0; t < 16; ++t) v[t] = t < n && a < nvir ? (double)p[t * nov + a] : 0.0;
#pragma unroll
        for (int t = 0; t < 16; ++t) {
            const double x = fabs(v[t]);
            const bool finite = x <= 1.7976931348623157e308;
            m = finite ? fmax(m, x) : INFINITY;
            sum[t] += finite ? x * x : 0.0;
        }
        double(*out)[64] = part[a0 / 64 % 2];
        out[wid][lane] = m;
        __syncthreads();
        if (wid == 0 && a < nvir)
            rr.pmax[(int64_t)blockIdx.x * nov + (int64_t)i * nvir + a] =
                fmax(fmax(out[0][lane], out[1][lane]), fmax(out[2][lane], out[3][lane]));
    }
#pragma unroll
    for (int t = 0; t < 16; ++t) {
        for (int m = 1; m < kWave; m *= 2) sum[t] += __shfl_xor(sum[t], m, kWave);
        if (lane == t) rr.w[((int64_t)i * gridDim.x + blockIdx.x) * 64 + 16 * wid + t] = sum[t];
    }
}

// 64 rows of an orbital: the exponent f of each is that of the INT8X4 format, the least with
// max |x| <= (1 - 2^-7) 2^(f + 1); the sum of 4^(f + 1), non-finite rows left out.
template <bool ROUND32>  // x is first rounded to FP32 (MIXED)
__global__ __launch_bounds__(256) void residue_rows_kernel(ResidueRange rr, int64_t nov, int np,
                                                           int nvir, int nvir_pad,
                                                           int *__restrict__ rexp) {
    const int lane = threadIdx.x % kWave, wid = threadIdx.x / kWave;
    const int i = blockIdx.y, a = blockIdx.x * 64 + lane;
    double m = 0.0;
    if (a < nvir) {
        const double *p = rr.pmax + (int64_t)i * nvir + a;
#pragma unroll 4
        for (int k = wid; k < np; k += 4) m = fmax(m, p[k * nov]);
    }
    __shared__ double part[4][64];
    part[wid][lane] = m;
    __syncthreads();
    if (wid != 0) return;
    double mm = fmax(fmax(part[0][lane], part[1][lane]), fmax(part[2][lane], part[3][lane]));
    if (ROUND32) mm = (double)(float)mm;
    int e = res::kZeroRow;
    double s = 0.0;
    if (mm > 1.7976931348623157e308) {
        e = kI8NonFinite;
    } else if (mm > 0.0) {
        (void)frexp(mm, &e);
        if (mm <= ldexp(1.0 - 0x1p-7, e)) e -= 1;
        s = ldexp(1.0, 2 * (e + 1));
    }
    if (a < nvir_pad) rexp[(int64_t)i * nvir_pad + a] = e;
    for (int k = 1; k < kWave; k *= 2) s += __shfl_xor(s, k, kWave);
    if (lane == 0) rr.s[(int64_t)i * rr.chunks + blockIdx.x] = s;
}

// Item order: the pair triangle in blocks of 4 x 8 pairs, cut into one run of pairs
// per XCD; each XCD takes its pairs tile pair by tile pair. Its 32 workgroups so
// run at one moment the same tile pair of about 4 i and 8 j, 12 operand tiles instead
// of 64, and all items of a round take the same time. order[position] = pair ntp + t.
__device__ void order_items(const ResidueOrder &o) {
    constexpr int BI = 4, BJ = 8;
    const int64_t n = o.nocc, npairs = o.nocc_b ? n * o.nocc_b : n * (n + 1) / 2;
    if (blockIdx.x == 0)
        for (int t = threadIdx.x; t < o.words; t += blockDim.x) o.queue[t] = 0;
    for (int64_t p = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; p < npairs;
         p += (int64_t)gridDim.x * blockDim.x) {
        int i, j;
        int64_t rank;
        if (o.nocc_b) {  // opposite spin: every (i, J)
            i = (int)(p / o.nocc_b);
            j = (int)(p % o.nocc_b);
            const int i0 = i / BI * BI, i1 = min(i0 + BI, o.nocc), j0 = j / BJ * BJ;
            rank = (int64_t)i0 * o.nocc_b + (int64_t)(i1 - i0) * j0 +
                   (i - i0) * min(BJ, o.nocc_b - j0) + j - j0;
        } else {
            decode_pair(p, o.nocc, i, j);
            const int i0 = i / BI * BI, i1 = min(i0 + BI, o.nocc);
            const int j0 = j / BJ * BJ;
            rank = i0 * n - (int64_t)i0 * (i0 - 1) / 2;  // pairs of the rows above
            for (int r = i0; r < i1; ++r) {
                rank += max(0, j0 - r);  // this band's pairs in the blocks to the left
                if (r < i) rank += max(0, min(j0 + BJ, o.nocc) - max(j0, r));
                if (r == i) rank += j - max(j0, r);
            }
        }
        int x = 0;
        while (x + 1 < kXcds && npairs * (x + 1) / kXcds <= rank) ++x;
        const int64_t lo = npairs * x / kXcds, count = npairs * (x + 1) / kXcds - lo;
        for (int t = 0; t < o.ntp; ++t)
            o.order[lo * o.ntp + t * count + rank - lo] = (int)(p * o.ntp + t);
    }
}

// One 64 x 64 tile (64 packed rows, one Q panel) to residues. Y = RN(x 2^(beta - 1 - f)).
// The rows go to row groups rg0 on, of nrg in all. ROUND32: x is first rounded to FP32
// (MIXED).
template <int N, bool ROUND32, typename Tin>
__global__ __launch_bounds__(256) void residue_pack_kernel(const Tin *__restrict__ b, int64_t nov,
                                                           int naux, int nvir, int nvir_pad,
                                                           int64_t nrows, int np, int beta,
                                                           int64_t nrg, int64_t rg0,
                                                           const int *__restrict__ rexp,
                                                           int8_t *__restrict__ out,
                                                           ResidueOrder ord, const int *wide) {
    __shared__ double tile[64][65];
    if (*wide) return;
    if ((int)blockIdx.y == np) {  // one more row of blocks: the item order and the queue words
        if (ord.order) order_items(ord);
        return;
    }
    const int tx = threadIdx.x % 64, ty = threadIdx.x / 64;
    const int64_t r0 = (int64_t)blockIdx.x * 64;
    const int q0 = blockIdx.y * 64;
    const int64_t r = r0 + tx;
    int64_t col = -1;
    if (r < nrows) {
        const int64_t i = r / nvir_pad;
        const int a = (int)(r % nvir_pad);
        if (a < nvir) col = i * nvir + a;
    }
    for (int q = ty; q < 64; q += 4) {
        const int qq = q0 + q;
        double v = 0.0;
        if (col >= 0 && qq < naux) v = (double)b[(int64_t)qq * nov + col];
        tile[q][tx] = ROUND32 ? (double)(float)v : v;
    }
    __syncthreads();
    // Thread t takes row 16 (t / 64) + t % 16 and the panel's Q = 16 g .. 16 g + 15,
    // g = (t / 16) % 4: lane t % 64 of its row group's kilobyte.
    const int t = threadIdx.x;
    const int g = (t / 16) % 4, row = (t / 64) * 16 + t % 16;
    const int64_t orow = r0 + row;
    if (orow >= nrows) return;
    const int e = rexp[orow];
    const bool bad = e == kI8NonFinite;
    const int sh = bad ? 0 : beta - 1 - e;
    uint32_t w[N][4];
#pragma unroll
    for (int k = 0; k < N; ++k)
#pragma unroll
        for (int c = 0; c < 4; ++c) w[k][c] = 0u;
#pragma unroll
    for (int q = 0; q < 16; ++q) {
        const double y = bad ? 0.0 : rint(ldexp(tile[16 * g + q][row], sh));
        // y as 64-bit two's complement: hi = floor(y / 2^32), lo = the rest
        const double h = floor(y * 0x1p-32);
        const uint64_t z =
            ((uint64_t)(uint32_t)(int)h << 32) + (uint64_t)(uint32_t)fma(h, -0x1p32, y);
        // signed base-256 digits of y
        const uint64_t d = (z + 0x8080808080808080ull) ^ 0x8080808080808080ull;
        const int dl = (int)(uint32_t)d, dh = (int)(uint32_t)(d >> 32);
#pragma unroll
        for (int k = 0; k < N; ++k) {
            uint32_t x;
            if (k == 0) {
                x = (uint32_t)dl;  // modulo 256: the lowest digit
            } else {
                const int s = __builtin_amdgcn_sdot4(
                    dl, (int)res::kDigit.v[k][0],
                    __builtin_amdgcn_sdot4(dh, (int)res::kDigit.v[k][1], 0, false), false);
                x = res::reduce_mod(s, 1.0f / (float)res::kMod[k], -res::kMod[k]);
            }
            w[k][q / 4] |= (x & 0xffu) << (8 * (q % 4));
        }
    }
    int8_t *o = out + ((int64_t)blockIdx.y * nrg + rg0 + orow / 16) * 1024 + (t % 64) * 16;
#pragma unroll
    for (int k = 0; k < N; ++k)
        *(uint4 *)(o + (int64_t)k * np * nrg * 1024) =
            make_uint4(w[k][0], w[k][1], w[k][2], w[k][3]);
}

// ---- Range test ----------------------------------------------------------------
// One exponent a row makes the rounding of g = (ia|jb) relative to the rows' largest
// elements, where the matrix kernels' is relative to the products: rows that lie on different
// aux functions (orbitals far apart) have small products of which few bits would be left. The
// mean square error of g over a and b is
//   4^-beta / 12 (s_i sum_Q w_jQ + s_j sum_Q w_iQ) + (fixed point)^2 s_i s_j,
// s_i the sum over a of the rows' squared ranges 4^(f + 1), w_iQ the sum over a of B^2, the
// sums over Q where the other orbital is not zero (zeros have no rounding error), and g^2 is
// sum_Q w_iQ w_jQ for products of random sign. A call with a pair whose error exceeds bar_of
// of that goes to the matrix kernel: the packer and the energy kernel leave at once, and the
// host sees the flag with the results, so that no wait is added (in MIXED with the range check
// of B, whose wait comes first anyway). Pairs by their own size, chain of 24 orbitals
// decaying as e^-d over 1008 aux functions: 1.9e-10 at d = 21 without the test, and 3.7e-3 in
// MIXED. What errors the bar admits the sums of the energies average down to their own rounding;
// the matrix kernels' products are off by 2^-50 (960 aux functions in FP64) and 2^-23 (panels
// of 64 in FP32) on the same scale. Normal rows, with or without hot aux functions, have
// 2^-53 to 2^-54, water in cc-pVDZ 2^-54, orbitals that reach three sites 2^-51.
// What it costs (with the tenth layer of the reconstruction): the three blocks of 21/229,
// 20/230 over 960 aux functions 1396 -> 1439 us, 60/450/1800 in MIXED 9391 -> 9328, 100/200/2400
// 9501 -> 9505; and a call that ends on the matrix kernel, over that kernel alone: 24/160/1008 in
// MIXED 497 -> 542, opposite spin 953 -> 1063, 60/450/1800 19.9 -> 20.1 and 64.2 -> 64.8 ms.
constexpr double bar_of(int n) { return n == 16 ? 0x1p-50 : 0x1p-24; }

// Orbitals i = blockIdx.y and j, a wave to each j. same: j >= i only. Sums out of the range of
// FP64's squares count as past the bar.
__global__ __launch_bounds__(256) void residue_range_kernel(const double *__restrict__ wa,
                                                            const double *__restrict__ sa,
                                                            const double *__restrict__ wb,
                                                            const double *__restrict__ sb, int nb,
                                                            int chunks, int naux_pad, bool same,
                                                            double round2, double fixed2,
                                                            int *wide) {
    const int i = blockIdx.y, j = blockIdx.x * 4 + threadIdx.x / kWave, lane = threadIdx.x % kWave;
    if (j >= nb || (same && j < i)) return;
    const double *x = wa + (int64_t)i * naux_pad, *y = wb + (int64_t)j * naux_pad;
    double gg = 0.0, ni = 0.0, nj = 0.0, si = 0.0, sj = 0.0;
#pragma unroll 4
    for (int q = lane; q < naux_pad; q += kWave) {
        const double u = x[q], v = y[q];
        gg += u * v;
        ni += v > 0.0 ? u : 0.0;
        nj += u > 0.0 ? v : 0.0;
    }
    for (int c = lane; c < chunks; c += kWave) {
        si += sa[(int64_t)i * chunks + c];
        sj += sb[(int64_t)j * chunks + c];
    }
    for (int m = 1; m < kWave; m *= 2) {
        gg += __shfl_xor(gg, m, kWave);
        ni += __shfl_xor(ni, m, kWave);
        nj += __shfl_xor(nj, m, kWave);
        si += __shfl_xor(si, m, kWave);
        sj += __shfl_xor(sj, m, kWave);
    }
    if (lane != 0 || nj == 0.0) return;  // no aux function in common: g = 0
    const double err = round2 * (si * nj + sj * ni) + fixed2 * si * sj;
    if (!(err <= gg && gg > 1e-280 && gg < 1e280)) *wide = 1;
}

// One product over a run of moduli and every panel: row groups rgA .. rgA + nA against
// rgB .. rgB + nB; the residues of block (x, y) of modulus k go to
// byte k kPlane + (16 x + y) 256 of the planes. NX x NY: the blocks of this wave (nx, ny) rounded
// up to a built size; blocks past nx or ny multiply whatever the LDS holds and
// go to the dump slot.
struct Product {
    const int8_t *op;             // residues of step 0
    int64_t step;                 // bytes from one step to the next
    int rgA, rgB;                 // first 16-row groups of the two operands
    int nA, nB, np;
    int k0, k1;                   // moduli
    int x0, y0, nx, ny;           // this wave's blocks
    __amdgpu_buffer_rsrc_t planes;  // N residue planes and the dump slot
};

template <int N>
__device__ __forceinline__ void wait_vm() {
    static_assert(N < 64, "vmcnt holds six bits");
    asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N) : "memory");
}
// All LDS reads done, then the other waves are met. One asm block between
// scheduling barriers, so that nothing moves from one phase to the next.
__device__ __forceinline__ void meet() {
    __builtin_amdgcn_sched_barrier(0);
    asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
    __builtin_amdgcn_sched_barrier(0);
}

// NL: kilobytes each wave fetches per step.
template <int N, int NX, int NY, int NL>
__device__ __forceinline__ void run_product(const Product &P, char *lds) {
    const int lane = threadIdx.x % kWave;
    const int wid = __builtin_amdgcn_readfirstlane((int)(threadIdx.x / kWave));
    const int nblk = P.nA + P.nB;
    // Kilobytes wid, wid + 8, ... of a step's nA + nB, straight into the LDS. Every
    // wave issues NL loads, so that the wait counts are the same for all: past
    // the last kilobyte it repeats it (the same bytes to the same place).
    uint32_t src[NL], dst[NL];
#pragma unroll
    for (int t = 0; t < NL; ++t) {
        const int blk = min(wid + 8 * t, nblk - 1);
        src[t] = (uint32_t)(blk < P.nA ? P.rgA + blk : P.rgB + blk - P.nA) * 1024u;
        dst[t] = (uint32_t)(blk < P.nA ? blk : kTB + blk - P.nA) * 1024u;
    }
    const int S = (P.k1 - P.k0) * P.np;
    int ahead = S;                                       // stages not yet fetched
    const int8_t *const op = P.op + P.k0 * P.np * P.step;
    const int8_t *from = op;    // the next one's residues
    uint32_t to = 0;            // and its place in the LDS
    auto fetch1 = [&](int t, uint32_t lane16) {
        const int8_t *p = from + src[t];  // uniform: a scalar base and one lane offset
        __builtin_amdgcn_global_load_lds((GlobalPtr)(p + lane16), (LdsPtr)(lds + to + dst[t]), 16,
                                         0, 0);
    };
    // Past the product's last step the first stage is fetched again and never read,
    // so that no step needs a test.
    auto advance = [&] {
        to = (to + kStage) % (kBuf * kStage);
        from = --ahead > 0 ? from + P.step : op;
    };
    uint32_t cur = 0;  // LDS place of the next stage to read
    const uint32_t offa = P.x0 * 1024, offb = (kTB + P.y0) * 1024;
    auto read = [&](v4i(&fa)[NX], v4i(&fb)[NY], uint32_t lane16) {
        const char *la = lds + cur + offa + lane16, *lb = lds + cur + offb + lane16;
#pragma unroll
        for (int y = 0; y < NY; ++y) fb[y] = *(const v4i *)(lb + y * 1024);
#pragma unroll
        for (int x = 0; x < NX; ++x) fa[x] = *(const v4i *)(la + x * 1024);
        cur = (cur + kStage) % (kBuf * kStage);
    };
    __syncthreads();  // the LDS is free
#pragma unroll
    for (int s = 0; s < kBuf; ++s) {
#pragma unroll
        for (int t = 0; t < NL; ++t) fetch1(t, lane * 16);
        advance();
    }
    wait_vm<(kBuf - 1) * NL>();
    meet();
    v4i fa[2][NX], fb[2][NY], acc[NX][NY];
    read(fa[0], fb[0], lane * 16);
    int k = P.k0, left = P.np;
    int waits = kBuf;   // since the last stores
    auto clear = [&] {
#pragma unroll
        for (int x = 0; x < NX; ++x)
#pragma unroll
            for (int y = 0; y < NY; ++y) acc[x][y] = (v4i){0, 0, 0, 0};
    };
    clear();
    // One step: the fragments of the next stage are read, and the stage after the
    // three in flight fetched into the buffer just read, while the products of
    // this one run. A stage has landed when only the kBuf - 2 younger ones are
    // out, and the stores of the last modulus while they are younger than it.
    auto step = [&](v4i(&ca)[NX], v4i(&cb)[NY], v4i(&na)[NX], v4i(&nb)[NY]) {
        if (waits < kBuf - 1)
            wait_vm<(kBuf - 2) * NL + NX * NY>();
        else
            wait_vm<(kBuf - 2) * NL>();
        ++waits;
        meet();
        // 16 x the lane, worked out anew: with both stages' fragments and the sums live
        // there is no register to keep it in.
        uint32_t lane16;
        asm volatile(
            "v_mbcnt_lo_u32_b32 %0, -1, 0\n\t"
            "v_mbcnt_hi_u32_b32 %0, -1, %0\n\t"
            "v_lshlrev_b32 %0, 4, %0"
            : "=v"(lane16));
        read(na, nb, lane16);
        __builtin_amdgcn_sched_barrier(0);
        // The loads go between rows of products: issued together they would hold the
        // wave until the memory path takes them.
#pragma unroll
        for (int x = 0; x < NX; ++x) {
#pragma unroll
            for (int y = 0; y < NY; ++y)
                acc[x][y] =
                    __builtin_amdgcn_mfma_i32_16x16x64_i8(ca[x], cb[y], acc[x][y], 0, 0, 0);
            if (x < NL) {
                __builtin_amdgcn_sched_barrier(0);
                fetch1(x, lane16);
                __builtin_amdgcn_sched_barrier(0);
            }
        }
        advance();
        if (--left || k == P.k1) return;
        const int plane = k * kPlane + (P.x0 * 16 + P.y0) * 256;
        // Exactly NX NY stores per wave (the wait counts rely on it): blocks
        // past nx or ny go to the dump slot behind the planes.
        const float inv = kRecip.v[k];
        const int neg = -res::kMod[k];
        // Kept from being worked out ahead of the loop, block by block: the registers
        // that would take are not there.
        int nx = P.nx, ny = P.ny;
        asm volatile("" : "+s"(nx), "+s"(ny));
#pragma unroll
        for (int x = 0; x < NX; ++x)
#pragma unroll
            for (int y = 0; y < NY; ++y) {
                uint32_t q[4];
#pragma unroll
                for (int v = 0; v < 4; ++v) q[v] = res::reduce_mod(acc[x][y][v], inv, neg);
                const int at = x < nx && y < ny ? plane + (x * 16 + y) * 256 : N * kPlane;
                __builtin_amdgcn_raw_buffer_store_b32(res::pack_bytes(q[0], q[1], q[2], q[3]),
                                                      P.planes, lane16 / 4, at,
                                                      kNonTemporal);
            }
        waits = 0;
        clear();
        ++k;
        left = P.np;
    };
#pragma unroll 1
    for (int s = 0; s < S; s += 2) {  // an odd S: the step past the end stores nothing
        step(fa[0], fb[0], fa[1], fb[1]);
        step(fa[1], fb[1], fa[0], fb[0]);
    }
    wait_vm<0>();
    meet();
}

template <int N, int NY>
__device__ __forceinline__ void run_rows(const Product &P, char *lds) {
    const int nblk = P.nA + P.nB, rows = (P.nA + 1) / 2;
    if (rows <= 4 && nblk <= 16)
        run_product<N, 4, NY, 2>(P, lds);
    else if (rows <= 6 && nblk <= 24)
        run_product<N, 6, NY, 3>(P, lds);
    else if (P.nx > 7)
        run_product<N, 8, NY, 4>(P, lds);
    else
        run_product<N, 7, NY, 4>(P, lds);
}

template <int N>
__device__ __forceinline__ void load_residues(const char *plane0, int bx, int by, int lane,
                                              uint32_t (&d)[N]) {
    const char *p = plane0 + (bx * 16 + by) * 256 + lane * 4;
#pragma unroll
    for (int k = 0; k < N; ++k) d[k] = *(const uint32_t *)(p + k * kPlane);
}

// One occupied pair of an item, for its epilogue: blocks (u0 + x, v0 + y) of the
// residue planes hold (i a | j b), a in the 16-row block a0 + x, b in b0 + y.
struct PairTile {
    int i, j, a0, b0, nA, nB, u0, v0;
    bool diag;  // the two tiles are the same virtuals: block (y, x) holds (i b | j a) transposed
};

struct PairTables {
    double eps[2][256];                  // virtuals of tile A and of tile B
    int exp_i[2][256], exp_j[2][256];    // row exponents of orbital i and of j there
};

// Unordered pair t of n (x <= y), y ascending.
__device__ __forceinline__ void decode_upper(int t, int &x, int &y) {
    y = (int)((sqrtf(8.0f * (float)t + 1.0f) - 1.0f) * 0.5f);
    while (y * (y + 1) / 2 > t) --y;
    while ((y + 1) * (y + 2) / 2 <= t) ++y;
    x = t - y * (y + 1) / 2;
}

// Energy terms (pair::energy_epilogue's) of one pair, block by block over the
// waves; on a diagonal tile pair the unordered block pairs, g_ba from the mirror
// block transposed through the LDS. The residues of the next block load while
// this one is rebuilt.
// AMP: also stores t = g / D of both orderings of the pair (AmpOut), each element
// from exactly one lane: inside a diagonal block
// (a, b) and (b, a) both come as t1, whose denominators need not agree to the last
// bit, so t2 is left to the other lane. At 41/209/960 the pass takes 1119 us with the
// 675 MB of amplitudes; the matrix kernel's took 2515 us.
template <int N, bool AMP>
__device__ __forceinline__ void pair_energy(const ResidueArgs &a, const PairTile &T,
                                            const char *c1, const char *c2, char *lds, KSum &os,
                                            KSum &ss) {
    const int lane = threadIdx.x % kWave;
    const int wid = __builtin_amdgcn_readfirstlane((int)(threadIdx.x / kWave));
    const int g = lane / 16, r = lane % 16;
    const int nblk = T.diag ? T.nA * (T.nA + 1) / 2 : T.nA * T.nB;
    const double eij = a.eps_occ[T.i] + a.eps_occ[T.j];
    const bool kap = !isnan(a.kappa);
    double(*tr)[17] = (double(*)[17])(lds + wid * 16 * 17 * 8);
    // What the blocks need per virtual, in the LDS: a global load here would wait
    // for the residues requested ahead of it. Virtuals past nvir take 0 energy.
    PairTables &tab = *(PairTables *)(lds + kStage);
    {
        const int h = threadIdx.x / 256, c = threadIdx.x % 256;
        if (c < 16 * (h ? T.nB : T.nA)) {
            const int v = 16 * (h ? T.b0 : T.a0) + c;
            tab.eps[h][c] = v < a.nvir ? a.eps_vir[v] : 0.0;
            tab.exp_i[h][c] = a.rexp[(int64_t)T.i * a.nvir_pad + v];
            tab.exp_j[h][c] = a.rexp[(int64_t)T.j * a.nvir_pad + v];
        }
    }
    __syncthreads();
    const int esh = -2 * (a.beta - 1);
    const bool two = T.diag || c2;
    uint32_t n1[N], n2[N];
    int bx, by;
    auto place = [&](int t) {
        if (T.diag) {
            decode_upper(t, bx, by);
        } else {
            bx = t / T.nB;
            by = t % T.nB;
        }
    };
    auto load = [&] {
        load_residues<N>(c1, T.u0 + bx, T.v0 + by, lane, n1);
        if (T.diag)
            load_residues<N>(c1, T.u0 + by, T.v0 + bx, lane, n2);
        else if (c2)
            load_residues<N>(c2, T.u0 + bx, T.v0 + by, lane, n2);
    };
    if (wid < nblk) {
        place(wid);
        load();
    }
#pragma unroll 1
    for (int t = wid; t < nblk; t += 8) {
        const int la = bx * 16, lb = by * 16;  // in the tile
        const int bx0 = bx, by0 = by;
        const double half = T.diag && bx0 == by0 ? 0.5 : 1.0;
        uint32_t d1[N], d2[N];
#pragma unroll
        for (int k = 0; k < N; ++k) {
            d1[k] = n1[k];
            d2[k] = n2[k];
        }
        if (t + 8 < nblk) {
            place(t + 8);
            load();
        }
        double g1[4], g2[4];
        res::crt4<N>(d1, g1);
        const int xb = tab.exp_j[1][lb + r] + esh;
#pragma unroll
        for (int v = 0; v < 4; ++v) g1[v] = res::scale_frac<N>(g1[v], tab.exp_i[0][la + 4 * g + v] + xb);
        if (two) {
            res::crt4<N>(d2, g2);
            if (T.diag) {
                const int xa = tab.exp_j[0][la + r] + esh;  // rows b, columns a of the pair (i, j)
#pragma unroll
                for (int v = 0; v < 4; ++v)
                    tr[4 * g + v][r] = res::scale_frac<N>(g2[v], tab.exp_i[1][lb + 4 * g + v] + xa);
                __builtin_amdgcn_wave_barrier();
#pragma unroll
                for (int v = 0; v < 4; ++v) g2[v] = tr[r][4 * g + v];
                __builtin_amdgcn_wave_barrier();
            } else {
                const int xi = tab.exp_i[1][lb + r] + esh;
#pragma unroll
                for (int v = 0; v < 4; ++v)
                    g2[v] = res::scale_frac<N>(g2[v], tab.exp_j[0][la + 4 * g + v] + xi);
            }
        } else {
#pragma unroll
            for (int v = 0; v < 4; ++v) g2[v] = g1[v];
        }
        const bool okb = T.b0 * 16 + lb + r < a.nvir;
        const double eb = tab.eps[1][lb + r];
        if constexpr (AMP) {
            const int64_t vp = a.amp.sx;
            double *bij = a.amp.base + T.i * a.amp.sp + T.j * a.amp.sq;
            double *bji = a.amp.base + T.j * a.amp.sp + T.i * a.amp.sq;
            const int64_t A = T.a0 * 16 + la + 4 * g, B = T.b0 * 16 + lb + r;
            v4d t1, t2;
#pragma unroll
            for (int v = 0; v < 4; ++v) {
                const double inv = 1.0 / (eij - tab.eps[0][la + 4 * g + v] - eb);
                const bool ok = okb && A + v < a.nvir;
                t1[v] = ok ? g1[v] * inv : 0.0;
                t2[v] = ok ? g2[v] * inv : 0.0;
            }
            const bool other = !(T.diag && bx0 == by0);
            if (a.amp.wide) {  // four of a row at once: 1119 us against 1245 at 41/209/960
#pragma unroll
                for (int v = 0; v < 4; ++v) bij[(A + v) * vp + B] = t1[v];
                if (other) *(v4d *)(bij + B * vp + A) = t2;
                if (T.i != T.j) {
                    *(v4d *)(bji + B * vp + A) = t1;
                    if (other)
#pragma unroll
                        for (int v = 0; v < 4; ++v) bji[(A + v) * vp + B] = t2[v];
                }
            } else if (B < a.amp.n) {
#pragma unroll
                for (int v = 0; v < 4; ++v) {
                    if (A + v >= a.amp.n) break;
                    bij[(A + v) * vp + B] = t1[v];
                    if (other) bij[B * vp + A + v] = t2[v];
                    if (T.i != T.j) {
                        bji[B * vp + A + v] = t1[v];
                        if (other) bji[(A + v) * vp + B] = t2[v];
                    }
                }
            }
        }
#pragma unroll
        for (int v = 0; v < 4; ++v) {
            const bool ok = okb && T.a0 * 16 + la + 4 * g + v < a.nvir;
            const double d = eij - tab.eps[0][la + 4 * g + v] - eb;
            const double inv = half / d;
            const double dd = g1[v] - g2[v];
            const double dmp = pair::damping(kap, a.kappa, d);
            const double to = dmp * ((g1[v] * g1[v] + g2[v] * g2[v]) * inv);
            const double ts = dmp * ((dd * dd) * inv);
            os.add(ok ? to : 0.0);
            ss.add(ok ? ts : 0.0);
        }
    }
}

// Opposite spin: (ia|JB)^2 / D over one (i, J) and tile pair, weight 1.
template <int N>
__device__ __forceinline__ void rect_energy(const ResidueArgs &a, const PairTile &T,
                                            const char *c1, char *lds, KSum &os) {
    const int lane = threadIdx.x % kWave;
    const int wid = __builtin_amdgcn_readfirstlane((int)(threadIdx.x / kWave));
    const int g = lane / 16, r = lane % 16;
    const int nblk = T.nA * T.nB;
    const double eij = a.eps_occ[T.i] + a.eps_occ_b[T.j];
    PairTables &tab = *(PairTables *)(lds + kStage);  // as pair_energy
    {
        const int h = threadIdx.x / 256, c = threadIdx.x % 256;
        const int v = 16 * (h ? T.b0 : T.a0) + c;
        if (c < 16 * (h ? T.nB : T.nA)) {
            tab.eps[h][c] = h ? (v < a.nvir_b ? a.eps_vir_b[v] : 0.0)
                              : (v < a.nvir ? a.eps_vir[v] : 0.0);
            tab.exp_i[h][c] = h ? a.rexp_b[(int64_t)T.j * a.nvir_pad_b + v]
                                : a.rexp[(int64_t)T.i * a.nvir_pad + v];
        }
    }
    __syncthreads();
    const int esh = -2 * (a.beta - 1);
    uint32_t n1[N];
    if (wid < nblk) load_residues<N>(c1, wid / T.nB, wid % T.nB, lane, n1);
#pragma unroll 1
    for (int t = wid; t < nblk; t += 8) {
        const int la = t / T.nB * 16, lb = t % T.nB * 16;
        uint32_t d1[N];
#pragma unroll
        for (int k = 0; k < N; ++k) d1[k] = n1[k];
        if (t + 8 < nblk) load_residues<N>(c1, (t + 8) / T.nB, (t + 8) % T.nB, lane, n1);
        double g1[4];
        res::crt4<N>(d1, g1);
        const int xb = tab.exp_i[1][lb + r] + esh;
        const bool okb = T.b0 * 16 + lb + r < a.nvir_b;
        const double eb = tab.eps[1][lb + r];
#pragma unroll
        for (int v = 0; v < 4; ++v) {
            const double x = res::scale_frac<N>(g1[v], tab.exp_i[0][la + 4 * g + v] + xb);
            const bool ok = okb && T.a0 * 16 + la + 4 * g + v < a.nvir;
            const double to = (x * x) / (eij - tab.eps[0][la + 4 * g + v] - eb);
            os.add(ok ? to : 0.0);
        }
    }
}

// RECT: opposite spin, items (i, J, tA, tB) over every alpha i, beta J and tile of
// each side, one product each; the beta rows follow the alpha rows in the operand.
// AMP: the amplitudes are stored too.
template <int N, bool RECT, bool AMP>
__global__ __launch_bounds__(kThreads) void residue_energy_kernel(ResidueArgs a) {
    extern __shared__ __attribute__((aligned(16))) char lds[];
    __shared__ int turn;
    if (*a.wide) return;
    const int tid = threadIdx.x;
    const int wid = __builtin_amdgcn_readfirstlane(tid / kWave);
    const int wr = wid >> 2;
    // The second row of waves starts one column over, so that the two waves
    // of a SIMD do not both hold a wide column.
    const int wc = wr ? (wid + 1) & 3 : wid & 3;
    const int ng = a.nvir_pad / 16;
    // XCD x takes a contiguous part of the order, its workgroups in rounds of one
    // item each. A last round of few items is shared out by moduli, split workgroups
    // to an item; the one that ends last runs the epilogue.
    const int x = blockIdx.x % kXcds, slot = blockIdx.x / kXcds;
    const int wide = gridDim.x / kXcds;
    const int pairs = (int)(a.nitems / a.ntp);
    auto first = [&](int y) { return (int)((int64_t)pairs * y / kXcds) * a.ntp; };
    const int lo = first(x), n = first(x + 1) - lo;
    for (int r = 0; r * wide < n; ++r) {
        const int m = min(wide, n - r * wide), split = min(wide / m, kMaxSplit);
        if (slot >= m * split) return;
        __syncthreads();  // scratch and LDS are free
        // The round starts together on the whole chip, so that all its workgroups go
        // through the moduli side by side: those of an XCD fetch the tiles they
        // share once into its L2, and the chip's reads stay within a modulus or two
        // of the operand (1/16 of it each), which the MALL holds. Only a matter of
        // speed, so the wait is bounded (50 us of the 100 MHz wall clock).
        if (tid == 0) {
            int target = 0;
            for (int y = 0; y < kXcds; ++y) {
                const int ny = first(y + 1) - first(y), full = ny / wide, rest = ny % wide;
                target += min(r + 1, full) * wide;
                if (r >= full && rest) target += rest * min(wide / rest, kMaxSplit);
            }
            atomicAdd(a.queue, 1);
            const uint64_t t0 = wall_clock64();
            while (__hip_atomic_load(a.queue, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) <
                       target &&
                   wall_clock64() - t0 < 5000)
                __builtin_amdgcn_s_sleep(2);
        }
        __syncthreads();
        const int at = r * wide + slot / split, part = slot % split;
        // The workgroups of one item share planes of their own (behind everybody's,
        // which another workgroup may still be reading from the round before).
        const int64_t own = split > 1 ? (int)gridDim.x + x + kXcds * (slot / split) : (int)blockIdx.x;
        char *scr = (char *)a.scratch + own * a.scratch_stride;
        const int id = a.order[lo + at];
        // Orbital groups I <= J (one orbital each unless several fit a tile).
        int I, J, ta, tb;
        if (RECT) {
            I = id / a.ntp / a.nocc_b;
            J = id / a.ntp % a.nocc_b;
            ta = id % a.ntp / a.ntile_b;
            tb = id % a.ntp % a.ntile_b;
        } else {
            decode_pair(id / a.ntp, a.ngroup, I, J);
            decode_tile_pair(id % a.ntp, a.ntile, ta, tb);
        }
        const int ngb = RECT ? a.nvir_pad_b / 16 : ng, ntb = RECT ? a.ntile_b : a.ntile;
        const int i0 = I * a.group, j0 = J * a.group;
        const int ni = min(a.group, a.nocc - i0), nj = RECT ? 1 : min(a.group, a.nocc - j0);
        const int a0 = ta * ng / a.ntile, wA = (ta + 1) * ng / a.ntile - a0;
        const int b0 = tb * ngb / ntb, wB = (tb + 1) * ngb / ntb - b0;
        Product P;
        P.op = a.op;
        P.step = ((int64_t)a.nocc * ng + (RECT ? (int64_t)a.nocc_b * ngb : 0)) * 1024;
        P.nA = ni * wA;
        P.nB = nj * wB;
        P.np = a.np;
        P.k0 = part * N / split;
        P.k1 = (part + 1) * N / split;
        P.x0 = wr ? (P.nA + 1) / 2 : 0;
        P.nx = (wr ? P.nA : (P.nA + 1) / 2) - P.x0;
        P.y0 = wc * P.nB / 4;
        P.ny = (wc + 1) * P.nB / 4 - P.y0;
        const int nprod = RECT || ta == tb || I == J ? 1 : 2;
#pragma unroll 1
        for (int c = 0; c < nprod; ++c) {
            P.rgA = (c ? j0 : i0) * ng + a0;
            P.rgB = RECT ? a.nocc * ng + j0 * ngb + b0 : (c ? i0 : j0) * ng + b0;
            P.planes = raw_rsrc(scr + (int64_t)c * planes_of(N), planes_of(N));
            if (P.ny > 3)
                run_rows<N, 4>(P, lds);
            else if (P.ny > 2)
                run_rows<N, 3>(P, lds);
            else
                run_rows<N, 2>(P, lds);
        }
        if (split > 1) {
            // Every wave has waited for its stores; the fences order them against the
            // other workgroups' and drop what this CU's L1 holds of the planes.
            __syncthreads();
            if (tid == 0) {
                __threadfence();
                turn = atomicAdd(a.queue + kQueueStride + x * wide + slot / split, 1);
                __threadfence();
            }
            __syncthreads();
            if (turn != split - 1) return;  // split rounds are last rounds
        }
        __syncthreads();  // every wave's residues are in the scratch
        if constexpr (RECT) {
            const PairTile T{I, J, a0, b0, wA, wB, 0, 0, false};
            KSum os;
            rect_energy<N>(a, T, scr, lds, os);
            pair::block_store(os, KSum{}, 1.0, a.item_partials + 4 * (int64_t)id);
            continue;
        }
        for (int u = 0; u < ni; ++u)
            for (int v = 0; v < nj; ++v) {
                PairTile T;
                T.i = i0 + u;
                T.j = j0 + v;
                if (T.i > T.j) continue;
                T.a0 = a0;
                T.b0 = b0;
                T.nA = wA;
                T.nB = wB;
                T.u0 = u * wA;
                T.v0 = v * wB;
                T.diag = ta == tb;
                KSum os, ss;
                pair_energy<N, AMP>(a, T, scr, nprod == 2 ? scr + planes_of(N) : nullptr, lds, os, ss);
                const int64_t p = (int64_t)T.i * a.nocc - (int64_t)T.i * (T.i - 1) / 2 + T.j - T.i;
                pair::block_store(os, ss, T.i == T.j ? 1.0 : 2.0,
                                  a.item_partials + 4 * (p * a.ntp + id % a.ntp));
                if (a.group > 1) __syncthreads();  // the pair's LDS is free again
            }
    }
}

template <int N, bool ROUND32>  // MIXED: ROUND32
hipError_t launch_pack_n(const PackArgs &a, const ResidueOrder &ord, const int *wide, int beta,
                         int64_t nrg, int64_t rg0, hipStream_t st) {
    const int64_t nrows = (int64_t)a.nocc * a.nvir_pad, nov = (int64_t)a.nocc * a.nvir;
    const int np = a.naux_pad / 64;
    const dim3 grid((unsigned)((nrows + 63) / 64), (unsigned)np + 1);
    if (a.in_f32)
        hipLaunchKernelGGL((residue_pack_kernel<N, ROUND32, float>), grid, dim3(256), 0, st,
                           (const float *)a.b, nov, a.naux, a.nvir, a.nvir_pad, nrows, np, beta,
                           nrg, rg0, (const int *)a.rexp, (int8_t *)a.out0, ord, wide);
    else
        hipLaunchKernelGGL((residue_pack_kernel<N, ROUND32, double>), grid, dim3(256), 0, st,
                           (const double *)a.b, nov, a.naux, a.nvir, a.nvir_pad, nrows, np, beta,
                           nrg, rg0, (const int *)a.rexp, (int8_t *)a.out0, ord, wide);
    return hipGetLastError();
}

bool pack_sizes(const PackArgs &a) {
    return a.rexp && a.nocc > 0 && a.nvir > 0 && a.naux_pad % 64 == 0 && a.naux_pad >= a.naux &&
           a.naux_pad - a.naux < 64 && a.naux_pad <= res::kMaxNauxPad && a.nvir_pad % 16 == 0 &&
           a.nvir_pad >= a.nvir;
}

}  // namespace

// The longest XCD's rounds (the last by the moduli that its split workgroups take each), in
// steps of a panel and modulus whose cost follows the blocks that the waves multiply, and in
// rebuilds, both cheaper while the chip has one round; packing; launches and the wait. Fitted
// to the 1800 of 2600 calls (65 to 560 virtuals, 4 to 90 occupied, 60 to 4608 aux functions,
// 0.15 to 20 ms) whose two routes are within 1.7 of each other: off by 5% in FP64, 4% in MIXED
// and 3% opposite spin.
double residue_estimate(const ResidueShape &p) {
    const int n = residue_moduli(p.prec), wide = p.cus / kXcds;
    double steps = 0.0, ends = 0.0;
    for (int x = 0; x < kXcds; ++x) {
        const int64_t items = (p.pairs * (x + 1) / kXcds - p.pairs * x / kXcds) * p.ntp;
        const int64_t full = items / wide;
        const int rest = (int)(items % wide), split = rest ? std::min(wide / rest, kMaxSplit) : 1;
        const double part = rest ? (double)((n + split - 1) / split) / n : 0.0;
        steps = std::max(steps, (double)full + part);
        ends = std::max(ends, (double)full + (rest ? 1 : 0));
    }
    // Off-diagonal tile pairs take two products; a single round is as long as its longest item.
    const double products =
        p.rect ? 1.0 : ends <= 1.0 && p.ntile > 1 ? 2.0 : 2.0 * p.ntile / (p.ntile + 1);
    const int rows = (p.wA + 1) / 2, blocks = p.wA + p.wB;  // run_rows' choice
    const int nx = rows <= 4 && blocks <= 16   ? 4
                   : rows <= 6 && blocks <= 24 ? 6
                   : rows <= 7                 ? 7
                                               : 8;
    const int ny = std::max(2, (p.wB + 3) / 4);
    // A call, then us of a step at 32 blocks, a step, a rebuilt tile of 16 x 16 blocks and
    // modulus with one round, the same with more, a modulus's pass, and 1e6 elements of B.
    static const double kCost[3][9] = {
        {130.5, 0.509, 0.162, 4.80, 0.480, 0.221, 8.90, -0.557, 5.86},   // FP64
        {180.0, 0.444, 0.176, 5.92, 0.279, 0.269, 10.87, 0.083, 8.46},   // MIXED
        {103.1, 0.464, 0.195, 5.36, 0.493, 0.177, 6.20, 1.119, 7.69}};   // opposite spin
    const double *k = kCost[p.rect ? 2 : p.prec == Prec::F64 ? 0 : 1];
    const double *c = ends <= 1.0 ? k + 1 : k + 4;
    const double passes = ends * products * n;
    return k[0] + steps * products * n * p.np * (c[0] * nx * ny / 32.0 + c[1]) +
           passes * (c[2] * p.wA * p.wB / 256.0 + k[7]) + p.elements * 1e-6 * k[8];
}

int residue_moduli(Prec prec) { return prec == Prec::F64 ? 16 : 10; }

int residue_beta(Prec prec, int naux_pad) {
    return prec == Prec::F64 ? res::beta_of<16>(naux_pad) : res::beta_of<10>(naux_pad);
}

int residue_scratch_sets(int blocks) { return blocks + blocks / 2; }

int residue_queue_words(int blocks) { return (kQueueStride + blocks + 31) / 32 * 32; }

size_t residue_scratch_stride(Prec prec, int products) {
    return (size_t)products * planes_of(residue_moduli(prec));
}

size_t ResidueRange::bytes(size_t nov, size_t norb, size_t nvir, int naux_pad) {
    const size_t np = (size_t)naux_pad;
    return sizeof(double) * (np / 64 * nov + norb * (np + (nvir + 63) / 64));
}

void ResidueRange::place(void *base, size_t nov, size_t norb, size_t nvir, int naux_pad) {
    pmax = (double *)base;
    w = pmax + (size_t)naux_pad / 64 * nov;
    s = w + norb * (size_t)naux_pad;
    chunks = (int)((nvir + 63) / 64);
}

hipError_t launch_residue_scan(Prec prec, const PackArgs &a, const ResidueRange &rr, int *wide,
                               hipStream_t st) {
    if (!pack_sizes(a) || !rr.pmax || rr.chunks * 64 < a.nvir) return hipErrorInvalidValue;
    const int64_t nov = (int64_t)a.nocc * a.nvir;
    const unsigned np = (unsigned)a.naux_pad / 64;
    const dim3 grid(np, (unsigned)a.nocc), rows((unsigned)rr.chunks, (unsigned)a.nocc);
    if (a.in_f32)
        hipLaunchKernelGGL(residue_scan_kernel<float>, grid, dim3(256), 0, st, (const float *)a.b,
                           nov, a.naux, a.nvir, rr, wide);
    else
        hipLaunchKernelGGL(residue_scan_kernel<double>, grid, dim3(256), 0, st,
                           (const double *)a.b, nov, a.naux, a.nvir, rr, wide);
    hipLaunchKernelGGL(prec == Prec::MIXED ? residue_rows_kernel<true> : residue_rows_kernel<false>,
                       rows, dim3(256), 0, st, rr, nov, (int)np, a.nvir, a.nvir_pad, a.rexp);
    return hipGetLastError();
}

hipError_t launch_residue_range(const ResidueArgs &a, const ResidueRange &rr, int *wide,
                                hipStream_t st) {
    const int naux_pad = a.np * 64, n = residue_moduli(a.prec);
    const bool rect = a.nocc_b > 0;
    const int nb = rect ? a.nocc_b : a.nocc;
    const double *wb = rr.w + (rect ? (int64_t)a.nocc * naux_pad : 0);
    const double *sb = rr.s + (rect ? (int64_t)a.nocc * rr.chunks : 0);
    const double bar = bar_of(n), unit = ldexp(1.0, -2 * a.beta) / (bar * bar);
    const double fixed = res::fixed_error(n) * (n == 16 ? res::kPhi<16> : res::kPhi<10>);
    hipLaunchKernelGGL(residue_range_kernel, dim3((unsigned)(nb + 3) / 4, (unsigned)a.nocc),
                       dim3(256), 0, st, rr.w, rr.s, wb, sb, nb, rr.chunks, naux_pad, !rect,
                       unit / 12.0, unit * fixed * ldexp(fixed, -2 * a.beta), wide);
    return hipGetLastError();
}

hipError_t launch_residue_pack(Prec prec, const PackArgs &a, const ResidueOrder &ord,
                               const int *wide, hipStream_t st, int64_t nrg, int64_t rg0) {
    const int64_t own = (int64_t)a.nocc * a.nvir_pad / 16;
    if (nrg == 0) nrg = own;
    if (rg0 < 0 || rg0 + own > nrg || !wide || !pack_sizes(a)) return hipErrorInvalidValue;
    const int beta = residue_beta(prec, a.naux_pad);
    switch (prec) {
    case Prec::F64: return launch_pack_n<16, false>(a, ord, wide, beta, nrg, rg0, st);
    case Prec::MIXED: return launch_pack_n<10, true>(a, ord, wide, beta, nrg, rg0, st);
    default: return hipErrorInvalidValue;
    }
}

hipError_t launch_residue_energy(const ResidueArgs &a, hipStream_t st) {
    const int ng = a.nvir_pad / 16;
    const bool rect = a.nocc_b > 0;
    const int64_t groups = (a.nocc + a.group - 1) / a.group;
    if (!a.op || !a.rexp || !a.scratch || !a.queue || !a.order || !a.wide || a.blocks <= 0 ||
        a.blocks % kXcds != 0 || a.nitems <= 0 || a.nitems > 0x7fffff00LL || a.np <= 0 ||
        a.np * 64 > res::kMaxNauxPad || a.nvir_pad % 16 != 0 || a.ntile * kTB < ng)
        return hipErrorInvalidValue;
    if (rect) {
        if (a.prec != Prec::F64 || !a.rexp_b || a.nvir_pad_b % 16 != 0 || a.group != 1 ||
            a.ntile_b * kTB < a.nvir_pad_b / 16 || a.ntp != a.ntile * a.ntile_b ||
            a.nitems != (int64_t)a.nocc * a.nocc_b * a.ntp ||
            a.scratch_stride < (int64_t)residue_scratch_stride(a.prec, 1))
            return hipErrorInvalidValue;
    } else if (a.group <= 0 || a.ngroup != groups ||
               (a.group > 1 && (a.ntile != 1 || a.group * ng > kTB)) ||
               a.ntp != a.ntile * (a.ntile + 1) / 2 ||
               a.nitems != groups * (groups + 1) / 2 * a.ntp ||
               a.scratch_stride < (int64_t)residue_scratch_stride(a.prec, a.ntile > 1 ? 2 : 1)) {
        return hipErrorInvalidValue;
    }
    if (a.amp.base && (rect || a.prec != Prec::F64)) return hipErrorInvalidValue;
    // Whole blocks, every row of four aligned.
    if (a.amp.wide && (a.amp.n != a.nvir_pad || a.amp.sx % 4 || a.amp.sp % 4 || a.amp.sq % 4 ||
                       (uintptr_t)a.amp.base % 32))
        return hipErrorInvalidValue;
    const auto kern = rect                           ? residue_energy_kernel<16, true, false>
                      : a.amp.base                   ? residue_energy_kernel<16, false, true>
                      : residue_moduli(a.prec) == 16 ? residue_energy_kernel<16, false, false>
                                                     : residue_energy_kernel<10, false, false>;
    hipLaunchKernelGGL(kern, dim3((unsigned)a.blocks), dim3(kThreads), kBuf * kStage, st, a);
    return hipGetLastError();
}

}  // namespace fh
