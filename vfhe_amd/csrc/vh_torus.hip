// vh_torus.hip -- CGGI functional bootstrapping over the 32-bit discretised torus
// (Z / 2^32) with the external product computed through an FP64 negacyclic FFT.
//
// No counterpart in the reference: its CGGI16 (modules/fhe/python/src/vfhe/fhe/
// cggi16.py:46-140) runs over RNS primes and the NTT.  This keeps that bootstrap's
// structure -- rotation amounts rounded as cggi16.py:54-86 does, the test vector
// rotated by -rot_b, one CMUX per key index with a non-zero amount (cggi16.py:76-90),
// extraction of coefficient 0 (cggi16.py:118-140) -- on the torus, with the external
// product and signed gadget decomposition of TFHE (Chillotti, Gama, Georgieva,
// Izabachene, "TFHE: fast fully homomorphic encryption over the torus",
// J. Cryptology 33 (2020): Definition 3.6 / Lemma 3.7 (decomposition), Theorem 3.13
// (external product), Algorithm 3 (blind rotation)).
//
// Negacyclic FFT.  A real polynomial p of N = 1024 coefficients is evaluated at the
// N/2 roots x of X^N = -1 with x^(N/2) = i: x = zeta * w^m, zeta = e^(i pi / N),
// w = e^(-2 pi i / M), M = N/2.  Since x^(N/2) = i,
//     p(zeta w^m) = sum_{j < M} (p_j + i p_{j+M}) zeta^j w^(jm),
// an M-point DFT of the folded and twisted sequence z_j = (p_j + i p_{j+M}) zeta^j.
// Real polynomials take conjugate values at the other N/2 roots, so products of
// these M values determine the negacyclic product; its inverse gives
// (r_j + i r_{j+M}) zeta^j, untwisted and unfolded.
//
// One wave computes one M = 512-point transform, 8 points per lane, as three
// radix-8 passes (input index j = 64 j2 + 8 j1 + j0, output k = k2 + 8 k1 + 64 k0):
//   layout A  lane = j mod 64, slot = j2       forward input, inverse output
//   layout B  lane = 8 k2 + j0, slot = j1      between the passes
//   layout C  lane = 8 k2 + k1, slot = k0      forward output (digit-reversed order),
//                                              the key's storage order, inverse input
// B<->C goes through a private LDS slice of the wave with a row pitch of 65, which spreads every
// access evenly over the banks.  A<->B swaps slot bits with lane bits 5..3: in registers where
// many waves share the LDS (64 instructions instead of 32 LDS accesses, 6.07 ms against
// 6.22 ms for 1024 samples), through LDS at pitch 72 where one workgroup has the CU and the
// chain of instructions counts (2.50 ms against 2.65 ms for 3 samples).
// Forward pass i evaluates the 8-term polynomial of a lane's slots at y_i e^(-2 pi i k / 8), k = 0..7,
//     y_1 = zeta^64   y_2 = zeta^(8 - 32 k2)   y_3 = zeta^(1 - 4 (k2 + 8 k1)),
// which covers the DFT-8, the twiddles before it and the pass's share of the twist: three radix-2
// stages by y^4, y^2 and y of 12 butterflies with 6 fused operations each, 72 per pass.  (Plain
// DFT-8s have 56, with 116 more for separate twiddles and twist: 6.33 ms for 1024 samples, 2.61 ms
// for 3, and an rms error of 3.6e-16 instead of 2.3e-16 of the values' size.)
// The inverse: a plain DFT-8 over k0, passes over k1 and k2 at y = zeta^(32 j0) and
// zeta^(4 (8 j1 + j0)) with the conjugate DFT, then the untwist by zeta^-j.
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "vh_kernels.h"

namespace {

constexpr int VT_N = 1024, VT_M = 512;
constexpr int VT_P1 = 72, VT_P2 = 65;          // exchange row pitches (doubles)
constexpr int VT_XS = 8 * VT_P2;               // doubles of an exchange array that only B<->C uses

// S = -1: X_k = sum_j x_j e^(-2 pi i jk / 8); S = +1: the same with +i (no scaling).
template <int S>
__device__ __forceinline__ void vt_dft4(double &r0, double &i0, double &r1, double &i1, double &r2, double &i2,
                                        double &r3, double &i3)
{
    const double c0r = r0 + r2, c0i = i0 + i2, d0r = r0 - r2, d0i = i0 - i2;
    const double c1r = r1 + r3, c1i = i1 + i3, er = r1 - r3, ei = i1 - i3;
    const double d1r = S > 0 ? -ei : ei, d1i = S > 0 ? er : -er;   // (r1 - r3) * (S i)
    r0 = c0r + c1r;
    i0 = c0i + c1i;
    r2 = c0r - c1r;
    i2 = c0i - c1i;
    r1 = d0r + d1r;
    i1 = d0i + d1i;
    r3 = d0r - d1r;
    i3 = d0i - d1i;
}

template <int S>
__device__ __forceinline__ void vt_dft8(double *re, double *im)
{
    const double h = 0.70710678118654752440;
    double ar[4], ai[4], br[4], bi[4];
#pragma unroll
    for (int j = 0; j < 4; j++) {
        ar[j] = re[j] + re[j + 4];
        ai[j] = im[j] + im[j + 4];
    }
    const double d0r = re[0] - re[4], d0i = im[0] - im[4];
    const double d1r = re[1] - re[5], d1i = im[1] - im[5];
    const double d2r = re[2] - re[6], d2i = im[2] - im[6];
    const double d3r = re[3] - re[7], d3i = im[3] - im[7];
    br[0] = d0r;
    bi[0] = d0i;
    br[1] = (S > 0 ? d1r - d1i : d1r + d1i) * h;          // * (1 + S i) / sqrt 2
    bi[1] = (S > 0 ? d1i + d1r : d1i - d1r) * h;
    br[2] = S > 0 ? -d2i : d2i;                           // * (S i)
    bi[2] = S > 0 ? d2r : -d2r;
    br[3] = (S > 0 ? -d3r - d3i : d3i - d3r) * h;         // * (-1 + S i) / sqrt 2
    bi[3] = (S > 0 ? d3r - d3i : -d3r - d3i) * h;
    vt_dft4<S>(ar[0], ai[0], ar[1], ai[1], ar[2], ai[2], ar[3], ai[3]);
    vt_dft4<S>(br[0], bi[0], br[1], bi[1], br[2], bi[2], br[3], bi[3]);
#pragma unroll
    for (int m = 0; m < 4; m++) {
        re[2 * m] = ar[m];
        im[2 * m] = ai[m];
        re[2 * m + 1] = br[m];
        im[2 * m + 1] = bi[m];
    }
}

__device__ __forceinline__ void vt_cmul(double &r, double &i, double wr, double wi)
{
    const double t = __fma_rn(r, wr, -(i * wi));
    i = __fma_rn(r, wi, i * wr);
    r = t;
}

// A pass's twiddles: y^4, y^2, y and y e^(S 2 pi i / 8) for y = zeta^e, from the table of zeta's powers.
struct vt_roots {
    double2 w4, w2, w1, w3;
    template <int S>
    static __device__ __forceinline__ vt_roots at(const double2 *zeta, int e)
    {
        auto p = [&](int x) { return zeta[x & (2 * VT_N - 1)]; };
        return {p(4 * e), p(2 * e), p(e), p(e + S * (VT_N / 4))};
    }
};

// (a, b) <- (a + w b, a - w b)
__device__ __forceinline__ void vt_bf(double &ar, double &ai, double &br, double &bi, double wr, double wi)
{
    const double xr = __fma_rn(wr, br, __fma_rn(-wi, bi, ar)), xi = __fma_rn(wr, bi, __fma_rn(wi, br, ai));
    br = __fma_rn(2.0, ar, -xr);
    bi = __fma_rn(2.0, ai, -xi);
    ar = xr;
    ai = xi;
}

// slot k <- sum_j (slot j) (y e^(S 2 pi i k / 8))^j
template <int S>
__device__ __forceinline__ void vt_pass(double *re, double *im, const vt_roots &t)
{
#pragma unroll
    for (int j = 0; j < 4; j++) vt_bf(re[j], im[j], re[j + 4], im[j + 4], t.w4.x, t.w4.y);
#pragma unroll
    for (int j = 0; j < 2; j++) {
        vt_bf(re[j], im[j], re[j + 2], im[j + 2], t.w2.x, t.w2.y);
        vt_bf(re[4 + j], im[4 + j], re[6 + j], im[6 + j], -S * t.w2.y, S * t.w2.x);   // times S i
    }
    vt_bf(re[0], im[0], re[1], im[1], t.w1.x, t.w1.y);                 // k = 0, 4
    vt_bf(re[2], im[2], re[3], im[3], -S * t.w1.y, S * t.w1.x);        // k = 2, 6
    vt_bf(re[4], im[4], re[5], im[5], t.w3.x, t.w3.y);                 // k = 1, 5
    vt_bf(re[6], im[6], re[7], im[7], -S * t.w3.y, S * t.w3.x);        // k = 3, 7
    auto order = [](double *v) {
        const double v1 = v[1], v3 = v[3], v4 = v[4], v5 = v[5], v6 = v[6];
        v[4] = v1; v[6] = v3; v[1] = v4; v[3] = v6; v[5] = v5;
    };
    order(re);
    order(im);
}

// The inverse's twiddles in LDS: pass 2 by lane mod 8, pass 3 and the untwist by lane.
struct vt_inv_tw {
    double2 y2[4][8], y3[4][64], untwist[8][64];
    __device__ __forceinline__ void fill(const double2 *zeta, int tid, int nthreads)
    {
        for (int l = tid; l < 64; l += nthreads) {
            const vt_roots r = vt_roots::at<1>(zeta, 4 * l);
            y3[0][l] = r.w4; y3[1][l] = r.w2; y3[2][l] = r.w1; y3[3][l] = r.w3;
            if (l < 8) {
                const vt_roots u = vt_roots::at<1>(zeta, 32 * l);
                y2[0][l] = u.w4; y2[1][l] = u.w2; y2[2][l] = u.w1; y2[3][l] = u.w3;
            }
        }
        for (int e = tid; e < VT_M; e += nthreads) {
            const double2 u = zeta[e];
            untwist[e >> 6][e & 63] = make_double2(u.x, -u.y);
        }
    }
};

// One exchange of a lane's eight complex values through LDS: written at w + ws s, read at
// r + rs s.  SEQ (the wide kernel): the real parts, then the imaginary parts, through one array (a wave's LDS
// operations complete in order), so the second write overlaps the first read.
template <bool SEQ>
__device__ __forceinline__ void vt_exchange(double *re, double *im, double *xr, double *xi, int w, int ws, int r, int rs)
{
    vh_wave_sync();
#pragma unroll
    for (int s = 0; s < 8; s++) xr[w + ws * s] = re[s];
    if (!SEQ) {
#pragma unroll
        for (int s = 0; s < 8; s++) xi[w + ws * s] = im[s];
    }
    vh_wave_sync();
#pragma unroll
    for (int s = 0; s < 8; s++) re[s] = xr[r + rs * s];
    if (SEQ) {
        vh_wave_sync();
#pragma unroll
        for (int s = 0; s < 8; s++) xr[w + ws * s] = im[s];
        vh_wave_sync();
    }
#pragma unroll
    for (int s = 0; s < 8; s++) im[s] = (SEQ ? xr : xi)[r + rs * s];
}

// The exchange A<->B in registers: slot bits 2, 1, 0 change places with lane bits 5, 4, 3.
__device__ __forceinline__ void vt_swap_bit(double &a, double &b, int bit)
{
    typedef unsigned vt_u2 __attribute__((ext_vector_type(2)));
    vt_u2 x = __builtin_bit_cast(vt_u2, a), y = __builtin_bit_cast(vt_u2, b);
#pragma unroll
    for (int h = 0; h < 2; h++) {
        if (bit == 0) {   // lanes 8..15 of a row of 16 take the other's lanes 0..7, and back
            const unsigned o = x[h];
            x[h] = __builtin_amdgcn_update_dpp(x[h], y[h], 0x128, 0xf, 0xc, false);
            y[h] = __builtin_amdgcn_update_dpp(y[h], o, 0x128, 0xf, 0x3, false);
        } else {
            const auto r = bit == 2 ? __builtin_amdgcn_permlane32_swap(x[h], y[h], false, false)
                                    : __builtin_amdgcn_permlane16_swap(x[h], y[h], false, false);
            x[h] = r[0];
            y[h] = r[1];
        }
    }
    a = __builtin_bit_cast(double, x);
    b = __builtin_bit_cast(double, y);
}

__device__ __forceinline__ void vt_swap(double *v)
{
#pragma unroll
    for (int bit = 2; bit >= 0; bit--)
#pragma unroll
        for (int s = 0; s < 8; s++)
            if (!(s & (1 << bit))) vt_swap_bit(v[s], v[s + (1 << bit)], bit);
}

// The forward twiddles of a lane: passes 2 and 3.
struct vt_fwd_tw {
    vt_roots y2, y3;
    __device__ __forceinline__ vt_fwd_tw(const double2 *zeta, int lane)
        : y2(vt_roots::at<-1>(zeta, 8 - 32 * (lane >> 3))),
          y3(vt_roots::at<-1>(zeta, 1 - 4 * ((lane >> 3) + 8 * (lane & 7))))
    {
    }
};

// Forward transform: layout A in (untwisted), layout C out.
template <bool SEQ = false>
__device__ __forceinline__ void vt_fwd(double *re, double *im, double *xr, double *xi, const vt_fwd_tw &t, int lane)
{
    // y_1 = e^(i pi / 16), correctly rounded (uniform constants, no loads)
    const vt_roots y1 = {{0x1.6a09e667f3bcdp-1, 0x1.6a09e667f3bcdp-1}, {0x1.d906bcf328d46p-1, 0x1.87de2a6aea963p-2},
                         {0x1.f6297cff75cb0p-1, 0x1.8f8b83c69a60bp-3}, {0x1.a9b66290ea1a3p-1, -0x1.1c73b39ae68c8p-1}};
    const int hi = lane >> 3, lo = lane & 7;
    vt_pass<-1>(re, im, y1);
    if (SEQ) {
        vt_exchange<true>(re, im, xr, xi, lane, VT_P1, VT_P1 * hi + lo, 8);
    } else {
        vt_swap(re);
        vt_swap(im);
    }
    vt_pass<-1>(re, im, t.y2);
    vt_exchange<SEQ>(re, im, xr, xi, VT_P2 * lo + 8 * hi, 1, lane, VT_P2);
    vt_pass<-1>(re, im, t.y3);
}

// Inverse transform (unscaled): layout C in, layout A out (untwisted).
template <bool SEQ = false>
__device__ __forceinline__ void vt_inv(double *re, double *im, double *xr, double *xi, const vt_inv_tw &t, int lane)
{
    const int hi = lane >> 3, lo = lane & 7;
    vt_dft8<1>(re, im);
    vt_exchange<SEQ>(re, im, xr, xi, lane, VT_P2, VT_P2 * lo + 8 * hi, 1);
    vt_pass<1>(re, im, {t.y2[0][lo], t.y2[1][lo], t.y2[2][lo], t.y2[3][lo]});
    if (SEQ) {
        vt_exchange<true>(re, im, xr, xi, VT_P1 * hi + lo, 8, lane, VT_P1);
    } else {
        vt_swap(re);
        vt_swap(im);
    }
    vt_pass<1>(re, im, {t.y3[0][lane], t.y3[1][lane], t.y3[2][lane], t.y3[3][lane]});
#pragma unroll
    for (int s = 0; s < 8; s++) {
        const double2 u = t.untwist[s][lane];
        vt_cmul(re[s], im[s], u.x, u.y);
    }
}

// x mod 2^32 of an integer-valued double with |x| < 2^51 (1.5 * 2^52 puts the
// rounded integer's low bits at the bottom of the mantissa).
__device__ __forceinline__ uint32_t vt_round_u32(double x)
{
    return (uint32_t)__double_as_longlong(x + 6755399441055744.0);
}

// round(x * 2N / 2^32) with ties to even, as a double quotient rounds in Python
// (cggi16.py:62,77; exact here since 2N / 2^32 is a power of two), mod 2N.
__device__ __forceinline__ uint32_t vt_mod_switch(uint64_t x, int shift, uint32_t two_n)
{
    const uint64_t q = x >> shift, rem = x & ((1ull << shift) - 1), half = 1ull << (shift - 1);
    const uint64_t r = q + ((rem > half || (rem == half && (q & 1))) ? 1 : 0);
    return (uint32_t)(r & (two_n - 1));
}

// coefficient j of X^a * p (a in [0, 2N)), mod 2^32
__device__ __forceinline__ uint32_t vt_rot(const uint32_t *p, int j, uint32_t a)
{
    const uint32_t t = ((uint32_t)j - a) & (2 * VT_N - 1);
    const uint32_t v = p[t & (VT_N - 1)], neg = 0u - (t >> 10);   // t >> 10: 1 when t >= N
    return (v ^ neg) - neg;
}

// add + coefficient j of X^a p, t = 4 (j - a): p[(j - a) mod N], negated when bit 10 of j - a is set
__device__ __forceinline__ uint32_t vt_diff(const uint32_t *p, uint32_t t, uint32_t add)
{
    const uint32_t v = *reinterpret_cast<const uint32_t *>(reinterpret_cast<const char *>(p) + (t & (4 * VT_N - 4)));
    const uint32_t neg = (uint32_t)__builtin_amdgcn_sbfe((int)t, 12, 1);
    return (v ^ neg) + (add - neg);
}

}  // namespace

// ---------------------------------------------------------------------------
// Key transform: one wave per polynomial (signed 32-bit coefficients) to layout C,
// stored [poly][slot][lane] (double2) and scaled by 1/M (exact: a power of two), so
// the blind rotation's inverse transforms need no scaling.  natural != 0: unscaled,
// in natural order [poly][k] (the transform check).
// ---------------------------------------------------------------------------
__global__ void __launch_bounds__(256) k_torus_fft(const uint32_t *__restrict__ in, double2 *__restrict__ out,
                                                   const double2 *__restrict__ consts, uint64_t count, int natural)
{
    __shared__ double lds[4][2][VT_XS];
    const int w = threadIdx.x >> 6, lane = threadIdx.x & 63;
    const uint64_t poly = (uint64_t)blockIdx.x * 4 + w;
    if (poly >= count) return;   // whole waves leave; the exchanges are wave-private
    const vt_fwd_tw tw(consts, lane);
    const uint32_t *p = in + poly * VT_N;
    double re[8], im[8];
#pragma unroll
    for (int s = 0; s < 8; s++) {   // p_j + i p_(j+M), j = 64 s + lane
        re[s] = (double)(int32_t)p[64 * s + lane];
        im[s] = (double)(int32_t)p[64 * s + lane + VT_M];
    }
    vt_fwd(re, im, lds[w][0], lds[w][1], tw, lane);
    double2 *o = out + poly * VT_M;
    const double scale = natural ? 1.0 : 1.0 / VT_M;
#pragma unroll
    for (int s = 0; s < 8; s++) {
        const int idx = natural ? (lane >> 3) + 8 * (lane & 7) + 64 * s : s * 64 + lane;
        o[idx] = make_double2(re[s] * scale, im[s] * scale);
    }
}

hipError_t vh_launch_torus_fft(hipStream_t st, const uint32_t *in, double2 *out, const double2 *consts, uint64_t count,
                               int natural)
{
    if (!count) return hipSuccess;
    VH_KL(k_torus_fft, dim3((unsigned)((count + 3) / 4)), dim3(256), 0, st, in, out, consts, count, natural);
    return hipGetLastError();
}

// ---------------------------------------------------------------------------
// Blind rotation + extraction, one workgroup per LWE sample.  Per key index with a
// non-zero amount, for each component c of the accumulator (0: the mask a, 1: the body b)
// and level l: digit polynomial of X^a_i acc_c - acc_c -> forward transform -> products with
// key row (c ell + l), output components 0 and 1; the products of all rows are summed per
// output component, inverse transform, untwist (the key rows carry the 1/M of the inverse),
// round, add into the accumulator.
//
// Few samples (k_torus_blind_rotate_wide): 2 ELL waves, one forward transform each.  Wave o < 2
// also owns component o: its accumulator in registers, the digit forming and the inverse
// transform.  acc[o] in LDS is wave o's own copy for the rotated reads, then holds the offset
// difference y every wave takes its level's digits from.  Each wave writes its partial product
// of a component it does not own to `area`; the owner adds them in wave order.  Before that a
// wave's area is its exchange slice, and the owner's inverse exchanges run through an area it
// has just read.  So an index takes two barriers: y in place, partials in place.
// The key: n x (2 ell rows) x (2 components) x [slot][lane] double2 (layout C).
// ---------------------------------------------------------------------------
template <int ELL>   // levels (1..4)
__global__ void __launch_bounds__(128 * ELL, 2) k_torus_blind_rotate_wide(vt_br_args A)
{
    constexpr int NW = 2 * ELL;
    __shared__ uint32_t acc[2][VT_N];
    __shared__ double2 area[2 * (NW - 1)][VT_M];
    __shared__ vt_inv_tw itw;
    const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
    const int l = w >> 1, mine = w == 1;   // level (of component w & 1); the component an owner wave keeps
    const uint64_t k = blockIdx.x;
    const uint32_t *in = A.lwe + k * (uint64_t)(A.n + 1);
    const uint32_t two_n = 2 * VT_N;
    const int shift = 32 - 11;   // log2(2^32 / 2N)
    // partial product of component o by wave v (v != o)
    auto part = [&](int o, int v) -> double2 * { return area[o * (NW - 1) + (v < o ? v : v - 1)]; };
    double *xs = reinterpret_cast<double *>(part(w == 0 ? 1 : 0, w));
    double *xi = reinterpret_cast<double *>(part(w & 1, NW - 1 - (w & 1) * (NW == 2)));   // read by wave w < 2 only
    const vt_fwd_tw tw(A.consts, lane);
    itw.fill(A.consts, threadIdx.x, 128 * ELL);   // read by waves 0 and 1 after the first barrier

    // acc = (0, X^-rot_b * tv): rot_b from b + floor(2^32 / (4 torus_base)) (cggi16.py:60-71)
    const uint32_t rot_b = vt_mod_switch((uint64_t)in[A.n] + A.offset, shift, two_n);
    const uint32_t rot_tv = (two_n - rot_b) & (two_n - 1);
    uint32_t own[16];   // coefficients 64 s + lane of component w
#pragma unroll
    for (int s = 0; s < 16; s++) {
        own[s] = w == 1 ? vt_rot(A.tv, 64 * s + lane, rot_tv) : 0u;
        if (w < 2) acc[w][64 * s + lane] = own[s];
    }

    // Digits: with y = x + dec_off, field_l = (y >> sh_l) mod 2^B and d_l = field_l - 2^(B-1),
    // which is the B-bit sign extension of field_l ^ 2^(B-1): one xor per coefficient, then
    // one signed bit-field extract per level.
    const uint32_t B = A.base_log;
    uint32_t xmask = 0;
#pragma unroll
    for (int e = 1; e <= ELL; e++) xmask |= (1u << (B - 1)) << (32 - B * e);
    const uint32_t sh = 32 - B * (l + 1);
    uint32_t next = in[0];
    for (uint32_t i = 0; i < A.n; i++) {
        const uint32_t ai = vt_mod_switch(next, shift, two_n);
        next = in[i + 1];   // the last one is the body
        if (ai == 0) continue;
        if (w < 2) {
            // coefficient j of X^a acc: acc[(j - a) mod N], negated when bit 10 of j - a is set
            const char *rows = reinterpret_cast<const char *>(acc[w]);
            const uint32_t t0 = 4 * ((uint32_t)lane - ai);
            uint32_t y[16];
            vh_wave_sync();
#pragma unroll
            for (int s = 0; s < 16; s++) {
                const uint32_t t = t0 + 256 * s;
                const uint32_t v = *reinterpret_cast<const uint32_t *>(rows + (t & (4 * VT_N - 4)));
                const uint32_t neg = (uint32_t)__builtin_amdgcn_sbfe((int)t, 12, 1);
                y[s] = ((v ^ neg) + (A.dec_off - own[s] - neg)) ^ xmask;
            }
            vh_wave_sync();
#pragma unroll
            for (int s = 0; s < 16; s++) acc[w][64 * s + lane] = y[s];
        }
        __syncthreads();   // y of both components is in place
        const VH_GLOBAL double *K = vh_global(reinterpret_cast<const double *>(
            A.bsk + (((uint64_t)i * (2 * ELL) + (uint64_t)((w & 1) * ELL + l)) * 2) * VT_M + lane));
        vh_f64x2 kw[8];
        auto key = [&](int o) {   // the wave's key row, output component o
#pragma unroll
            for (int s = 0; s < 8; s++) kw[s] = *(const VH_GLOBAL vh_f64x2 *)(K + o * (2 * VT_M) + 128 * s);
        };
        key(1 - mine);   // lands during the transform
        const uint32_t *yc = acc[w & 1];
        double fr[8], fi[8];
#pragma unroll
        for (int s = 0; s < 8; s++) {
            fr[s] = (double)(int)__builtin_amdgcn_sbfe((int)yc[64 * s + lane], sh, B);
            fi[s] = (double)(int)__builtin_amdgcn_sbfe((int)yc[64 * s + lane + VT_M], sh, B);
        }
        vt_fwd<true>(fr, fi, xs, nullptr, tw, lane);
        vh_wave_sync();
        double re[8], im[8];
#pragma unroll
        for (int oo = 0; oo < 2; oo++) {   // the other component's partial, then the own one
            if (oo) key(mine);
#pragma unroll
            for (int s = 0; s < 8; s++) {
                re[s] = __fma_rn(-fi[s], kw[s].y, fr[s] * kw[s].x);
                im[s] = __fma_rn(fi[s], kw[s].x, fr[s] * kw[s].y);
            }
            if (oo == 0 || w >= 2) {
                double2 *d = part(oo ? mine : 1 - mine, w) + lane;
#pragma unroll
                for (int s = 0; s < 8; s++) d[64 * s] = make_double2(re[s], im[s]);
            }
        }
        __syncthreads();   // the partials are in place, y is read
        if (w < 2) {
#pragma unroll
            for (int v = 1; v < NW; v++) {
                const double2 *d = part(w, v - (v == 1 && w == 1)) + lane;   // waves other than w, ascending
#pragma unroll
                for (int s = 0; s < 8; s++) {
                    const double2 p = d[64 * s];
                    re[s] += p.x;
                    im[s] += p.y;
                }
            }
            vt_inv<true>(re, im, xi, nullptr, itw, lane);
#pragma unroll
            for (int s = 0; s < 8; s++) {   // the key carries the 1/M of the inverse
                own[s] += vt_round_u32(re[s]);
                own[s + 8] += vt_round_u32(im[s]);
            }
#pragma unroll
            for (int s = 0; s < 16; s++) acc[w][64 * s + lane] = own[s];
        }
    }

    if (w >= 2) return;
    if (A.acc_out) {
        uint32_t *o = A.acc_out + k * 2 * VT_N + (uint64_t)w * VT_N;
#pragma unroll
        for (int s = 0; s < 16; s++) o[64 * s + lane] = own[s];
    }
    if (A.out) {
        // coefficient 0 of the phase b - a s: a'_0 = a_0, a'_j = -a_(N-j); b' = b_0
        uint32_t *o = A.out + k * (VT_N + 1);
        if (w == 0) {
#pragma unroll
            for (int s = 0; s < 16; s++) {
                const int j = 64 * s + lane;
                o[j ? VT_N - j : 0] = j ? 0u - own[s] : own[s];
            }
        } else if (lane == 0) {
            o[VT_N] = own[0];
        }
    }
}

// Many samples: two waves, wave c owns component c of the accumulator (in LDS as 32-bit words)
// and transforms its ELL digit polynomials one after another; the waves swap the partial
// product of the other's component through LDS (two barriers).
template <int ELL>   // levels (1..4)
__global__ void __launch_bounds__(128, 2) k_torus_blind_rotate(vt_br_args A)
{
    __shared__ uint32_t acc[2][VT_N];
    __shared__ double lds[2][2][VT_XS];
    __shared__ vt_inv_tw itw;
    const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
    const uint64_t k = blockIdx.x;
    const uint32_t *in = A.lwe + k * (uint64_t)(A.n + 1);
    const uint32_t two_n = 2 * VT_N;
    const int shift = 32 - 11;   // log2(2^32 / 2N)
    double *xr = lds[w][0], *xi = lds[w][1];

    itw.fill(A.consts, threadIdx.x, 128);
    const vt_fwd_tw tw(A.consts, lane);

    // acc = (0, X^-rot_b * tv): rot_b from b + floor(2^32 / (4 torus_base)) (cggi16.py:60-71)
    const uint32_t rot_b = vt_mod_switch((uint64_t)in[A.n] + A.offset, shift, two_n);
    const uint32_t rot_tv = (two_n - rot_b) & (two_n - 1);
    uint32_t *mine = acc[w];
    for (int j = lane; j < VT_N; j += 64) mine[j] = w == 0 ? 0u : vt_rot(A.tv, j, rot_tv);
    __syncthreads();

    // Digits: with y = x + dec_off, field_l = (y >> sh_l) mod 2^B and d_l = field_l - 2^(B-1),
    // which is the B-bit sign extension of field_l ^ 2^(B-1): one xor per coefficient, then
    // one signed bit-field extract per level.
    const uint32_t B = A.base_log;
    uint32_t xmask = 0;
#pragma unroll
    for (int l = 1; l <= ELL; l++) xmask |= (1u << (B - 1)) << (32 - B * l);
    const int rows = 2 * ELL;
    for (uint32_t i = 0; i < A.n; i++) {
        const uint32_t ai = vt_mod_switch(in[i], shift, two_n);
        if (ai == 0) continue;
        uint32_t dlo[8], dhi[8];
        const uint32_t t0 = 4 * ((uint32_t)lane - ai);
#pragma unroll
        for (int s = 0; s < 8; s++) {
            const int j = 64 * s + lane;
            dlo[s] = vt_diff(mine, t0 + 256 * s, A.dec_off - mine[j]) ^ xmask;
            dhi[s] = vt_diff(mine, t0 + 256 * s + 4 * VT_M, A.dec_off - mine[j + VT_M]) ^ xmask;
        }
        // own: this wave's output component (w), other: the other wave's (1 - w)
        double por[8], poi[8], pxr[8], pxi[8];
#pragma unroll
        for (int s = 0; s < 8; s++) por[s] = poi[s] = pxr[s] = pxi[s] = 0.0;
#pragma unroll
        for (int l = 0; l < ELL; l++) {
            // the level's key rows are loaded first, their latency covered by the transform
            const double2 *K = A.bsk + (((uint64_t)i * rows + (uint64_t)w * ELL + l) * 2) * VT_M + lane;
            const double2 *Ko = K + (w ? VT_M : 0), *Kx = K + (w ? 0 : VT_M);
            double2 kor[8], kxr[8];
#pragma unroll
            for (int s = 0; s < 8; s++) {
                kor[s] = Ko[s * 64];
                kxr[s] = Kx[s * 64];
            }
            const uint32_t sh = 32 - B * (l + 1);
            double re[8], im[8];
#pragma unroll
            for (int s = 0; s < 8; s++) {
                re[s] = (double)(int)__builtin_amdgcn_sbfe((int)dlo[s], sh, B);
                im[s] = (double)(int)__builtin_amdgcn_sbfe((int)dhi[s], sh, B);
            }
            vt_fwd(re, im, xr, xi, tw, lane);
#pragma unroll
            for (int s = 0; s < 8; s++) {
                const double2 ko = kor[s], kx = kxr[s];
                por[s] = __fma_rn(re[s], ko.x, por[s]);
                por[s] = __fma_rn(-im[s], ko.y, por[s]);
                poi[s] = __fma_rn(re[s], ko.y, poi[s]);
                poi[s] = __fma_rn(im[s], ko.x, poi[s]);
                pxr[s] = __fma_rn(re[s], kx.x, pxr[s]);
                pxr[s] = __fma_rn(-im[s], kx.y, pxr[s]);
                pxi[s] = __fma_rn(re[s], kx.y, pxi[s]);
                pxi[s] = __fma_rn(im[s], kx.x, pxi[s]);
            }
        }
        // swap partials; each output is wave 0's partial plus wave 1's (addition commutes)
#pragma unroll
        for (int s = 0; s < 8; s++) {
            xr[s * 64 + lane] = pxr[s];
            xi[s * 64 + lane] = pxi[s];
        }
        __syncthreads();
        const double *yr = lds[1 - w][0], *yi = lds[1 - w][1];
        double re[8], im[8];
#pragma unroll
        for (int s = 0; s < 8; s++) {
            re[s] = por[s] + yr[s * 64 + lane];
            im[s] = poi[s] + yi[s * 64 + lane];
        }
        __syncthreads();
        vt_inv(re, im, xr, xi, itw, lane);
#pragma unroll
        for (int s = 0; s < 8; s++) {   // the key carries the 1/M of the inverse
            const int j = 64 * s + lane;
            mine[j] += vt_round_u32(re[s]);
            mine[j + VT_M] += vt_round_u32(im[s]);
        }
        vh_wave_sync();
    }

    if (A.acc_out) {
        uint32_t *o = A.acc_out + k * 2 * VT_N + (uint64_t)w * VT_N;
        for (int j = lane; j < VT_N; j += 64) o[j] = mine[j];
    }
    if (A.out) {
        // coefficient 0 of the phase b - a s: a'_0 = a_0, a'_j = -a_(N-j); b' = b_0
        uint32_t *o = A.out + k * (VT_N + 1);
        if (w == 0)
            for (int j = lane; j < VT_N; j += 64) o[j] = j == 0 ? mine[0] : 0u - mine[VT_N - j];
        else if (lane == 0)
            o[VT_N] = mine[0];
    }
}

hipError_t vh_launch_torus_blind_rotate(hipStream_t st, const vt_br_args &A, uint64_t count, unsigned cus)
{
    if (!count) return hipSuccess;
    // Up to one sample per CU the levels of both components run side by side: 3 samples at
    // n = 630, 3 levels take 2.50 ms and 256 take 2.62 ms; the two-wave form takes 4.8 ms for 257, as
    // long as for fewer.  From two samples per CU on the wide form would need two rounds (5.2 ms),
    // the two-wave form has 512 side by side in 5.0 ms and 1024 in 6.1 ms, where 72% of the
    // issue slots hold vector instructions.
    const dim3 grid((unsigned)count);
    const bool wide = count <= cus;
#define VT_BR(EE)                                                                                       \
    case EE:                                                                                            \
        if (wide) VH_KL(k_torus_blind_rotate_wide<EE>, grid, dim3(128 * EE), 0, st, A);                 \
        else VH_KL(k_torus_blind_rotate<EE>, grid, dim3(128), 0, st, A);                                \
        break;
    switch (A.ell) { VT_BR(1) VT_BR(2) VT_BR(3) VT_BR(4) default: return hipErrorInvalidValue; }
#undef VT_BR
    return hipGetLastError();
}
