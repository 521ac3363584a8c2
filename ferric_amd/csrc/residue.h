// Exact residue arithmetic of the FP64 pair kernels (gfx950): the products
// sum_Q B^Q_ia B^Q_jb from INT8 matrix instructions, by the Chinese remainder
// theorem (K. Ozaki, Y. Uchino, T. Imamura, "Ozaki Scheme II: a GEMM-oriented
// emulation of floating-point matrix multiplication using an integer modular
// technique", 2025).
//
// Every packed row (i, a) is scaled by a power of two and rounded to integers
// Y with |Y| <= 2^beta, so G = sum_Q Y_ia Y_jb is an integer with 2 |G| < P =
// the product of N pairwise coprime moduli, which its residues fix. FP64 takes
// N = 16 (beta = 55 at naux = 3600, 56 at 960, 58 at 84).
// For each modulus m the residues of Y (signed, one byte) are multiplied by
// v_mfma_i32_16x16x64_i8 with exact int32 sums, and the sum reduced to a signed
// byte again. The fraction G / P is then sum_k r_k c_k modulo 1 with
// c_k = ((P / m_k)^-1 mod m_k) / m_k, taken as fixed point in ten (FP64) or nine (MIXED)
// signed byte layers (v_dot4_i32_i8 over four moduli at a time). The only rounding
// before the FP64 result is that of Y: half a unit, 2^-(beta + 1) of the row's
// power-of-two range, and about 2^-74 (FP64) or 2^-66 (MIXED) of P from the fixed point.
// With nine layers that was 2^-53 of the two rows' ranges in FP64 at naux 1000, and the
// largest error of small products: a pair energy of e^-24 of the largest was off by 1.4e-15
// of itself. The tenth costs a dword of products per four moduli and element.
//
// Why 16 moduli: with 15 a row would keep 52 bits below its largest value and
// the sums would lose the margin over the FP64 matrix instructions' rounding
// that rows of uneven size (local orbitals, hot aux rows) need. Why none above
// 239 except 256: the FP32 reciprocal that reduces a sum S has its quotient
// off by up to |S| 2^-23 / m, so the remainder leaves (m - 1) / 2 by up to
// |S| 2^-23 <= naux / 582, and it has to fit a signed byte: 119 + 8 at
// naux = 4608 (256 needs no division, its residue is the low byte).
#pragma once

#include <hip/hip_runtime.h>
#include <math.h>
#include <stdint.h>

#include "fh_device.h"
#include "fh_kernels.h"

namespace fh {
namespace res {

constexpr int kMaxN = 16;
constexpr int kMod[kMaxN] = {256, 239, 237, 235, 233, 229, 227, 223,
                             221, 217, 211, 209, 199, 197, 193, 191};
// Signed byte layers of c_k.
constexpr int layers_of(int n) { return n == 16 ? 10 : 9; }

typedef unsigned __int128 u128;
typedef __int128 i128;

// Tables of the format with the first N moduli.
constexpr int groups_of(int n) { return (n + 3) / 4; }  // moduli four to a dword

template <int N>
constexpr u128 product() {
    u128 p = 1;
    for (int k = 0; k < N; ++k) p *= (u128)kMod[k];
    return p;
}
// P as an unevaluated FP64 sum.
template <int N>
constexpr double kPhi = (double)product<N>();
template <int N>
constexpr double kPlo = (double)((i128)product<N>() - (i128)(double)product<N>());

template <int N>
struct Layers {
    // v[l][h]: byte l (0 = the highest) of c_k's fixed point, k = 4 h .. 4 h + 3.
    uint32_t v[layers_of(N)][groups_of(N)] = {};
};
template <int N>
constexpr Layers<N> make_layers() {
    Layers<N> t;
    for (int k = 0; k < N; ++k) {
        const int m = kMod[k];
        int rest = 1;  // P / m_k mod m_k
        for (int l = 0; l < N; ++l)
            if (l != k) rest = rest * (kMod[l] % m) % m;
        int inv = 0;
        for (int x = 1; x < m; ++x)
            if (rest * x % m == 1) inv = x;
        if (2 * inv > m) inv -= m;
        const i128 num = (i128)inv * ((i128)1 << 8 * layers_of(N));
        i128 f = num >= 0 ? (num + m / 2) / m : -((-num + m / 2) / m);
        for (int l = layers_of(N) - 1; l >= 0; --l) {
            const int8_t d = (int8_t)(uint8_t)(f & 0xff);
            f = (f - d) / 256;
            t.v[l][k / 4] |= (uint32_t)(uint8_t)d << (8 * (k % 4));
        }
    }
    return t;
}
template <int N>
constexpr Layers<N> kLayer = make_layers<N>();

// Largest beta with 2 naux 2^(2 beta) < P (1 - 2^-10).
template <int N>
inline int beta_of(int naux_pad) {
    int b = 0;
    while (b < 62 && (long double)naux_pad * exp2l(2 * (b + 1) + 1) <
                         (long double)kPhi<N> * (1.0L - 0x1p-10L))
        ++b;
    return b;
}

struct Digits {
    // v[k][h]: bytes 256^j mod m_k (signed, |.| <= m_k / 2), j = 4 h .. 4 h + 3, so that
    // Y mod m_k comes from Y's eight signed base-256 digits.
    uint32_t v[kMaxN][2] = {};
};
constexpr Digits make_digits() {
    Digits t;
    for (int k = 0; k < kMaxN; ++k) {
        const int m = kMod[k];
        int pw = 1;
        for (int j = 0; j < 8; ++j) {
            const int s = 2 * pw > m ? pw - m : pw;
            t.v[k][j / 4] |= (uint32_t)(uint8_t)(int8_t)s << (8 * (j % 4));
            pw = (int)((pw * 256) % m);
        }
    }
    return t;
}
constexpr Digits kDigit = make_digits();

// The exponent of a row of zeros, below every other.
constexpr int kZeroRow = -4096;

// Root mean square error of G / P from the fixed point: N residues of up to m / 2 times the
// rounding of c_k.
inline double fixed_error(int n) { return 19.0 * sqrt((double)n) * exp2(-8.0 * layers_of(n)); }

// Largest naux the int32 sums and the byte remainders allow (see above).
constexpr int kMaxNauxPad = 4608;

// S modulo m as a signed byte (in the low byte of the result). kMagic makes
// the fused multiply-add round S / m to an integer held in the low bits.
__device__ __forceinline__ uint32_t reduce_mod(int s, float inv, int neg_m) {
    const float t = __builtin_fmaf((float)s, inv, 12582912.0f);  // 1.5 2^23
    // The low 24 bits of t are q + 2^22, and 2^22 m has a zero low byte.
    return (uint32_t)(s + __mul24(__float_as_int(t), neg_m));
}

__device__ __forceinline__ uint32_t pack_bytes(uint32_t b0, uint32_t b1, uint32_t b2,
                                               uint32_t b3) {
    const uint32_t lo = __builtin_amdgcn_perm(b1, b0, 0x0c0c0400u);
    const uint32_t hi = __builtin_amdgcn_perm(b3, b2, 0x04000c0cu);
    return lo | hi;
}

// Four values from their residues: d[k] holds the signed residues modulo
// m_k of elements 0..3 in its bytes; frac[e] = G_e / P in [-1/2, 1/2).
template <int N>
__device__ __forceinline__ void crt4(const uint32_t (&d)[N], double (&frac)[4]) {
    constexpr int H = groups_of(N), L = layers_of(N);
    uint32_t t[4][H];  // [element][four moduli]
#pragma unroll
    for (int h = 0; h < H; ++h) {
        const uint32_t d0 = d[4 * h];
        const uint32_t d1 = 4 * h + 1 < N ? d[4 * h + 1] : 0u;
        const uint32_t d2 = 4 * h + 2 < N ? d[4 * h + 2] : 0u;
        const uint32_t d3 = 4 * h + 3 < N ? d[4 * h + 3] : 0u;
        const uint32_t a = __builtin_amdgcn_perm(d1, d0, 0x05010400u);  // e0: d0 d1, e1: d0 d1
        const uint32_t b = __builtin_amdgcn_perm(d1, d0, 0x07030602u);  // e2, e3
        const uint32_t c = __builtin_amdgcn_perm(d3, d2, 0x05010400u);
        const uint32_t e = __builtin_amdgcn_perm(d3, d2, 0x07030602u);
        t[0][h] = __builtin_amdgcn_perm(c, a, 0x05040100u);
        t[1][h] = __builtin_amdgcn_perm(c, a, 0x07060302u);
        t[2][h] = __builtin_amdgcn_perm(e, b, 0x05040100u);
        t[3][h] = __builtin_amdgcn_perm(e, b, 0x07060302u);
    }
#pragma unroll
    for (int x = 0; x < 4; ++x) {
        int s[L];
#pragma unroll
        for (int l = 0; l < L; ++l) {
            s[l] = 0;
#pragma unroll
            for (int h = 0; h < H; ++h)
                s[l] = __builtin_amdgcn_sdot4((int)t[x][h], (int)kLayer<N>.v[l][h], s[l], false);
        }
        // Layers 0..3 modulo 1 (the int32 wraps at 2^0), the rest exact: |s| <= 2^18.
        const uint32_t top = ((uint32_t)s[0] << 24) + ((uint32_t)s[1] << 16) +
                             ((uint32_t)s[2] << 8) + (uint32_t)s[3];
        const int m1 = s[4] * 256 + s[5], m2 = s[6] * 256 + s[7];
        const double m3 = L == 10 ? (double)(s[8] * 256 + s[L - 1]) * 0x1p-80
                                  : (double)s[8] * 0x1p-72;
        double f = fma((double)m2, 0x1p-64, m3);
        f = fma((double)m1, 0x1p-48, f);
        frac[x] = fma((double)(int)top, 0x1p-32, f);
    }
}

// G 2^e from G / P; a sum of row exponents at or above kI8NonFiniteSum marks a
// row that held a NaN or an infinity.
template <int N>
__device__ __forceinline__ double scale_frac(double frac, int e) {
    const double g = fma(frac, kPhi<N>, frac * kPlo<N>);
    return e >= kI8NonFiniteSum ? NAN : ldexp(g, e);
}

}  // namespace res
}  // namespace fh
