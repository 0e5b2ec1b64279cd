// vh_row8.h -- the last 8 stages of a transform on rows of 256 elements (FP64 path), 32 threads per
// row and 8 values per thread, 8 rows per 256-thread workgroup.
//
// Three register phases:
//   1  stages 0..2   k = t + 32 m                    (256-byte runs of the row)
//   2  stages 3..5   k = 32 (t >> 2) + 4 m + (t & 3)
//   3  stages 6..7   k = 128 (m >> 2) + 4 t + (m & 3)
// with two exchanges through LDS inside the wave (row slices of 36 doubles per 32: the reads of
// phase 2 touch every bank once).  The inverse runs them backwards.
// The row's 255 twiddles are formed once per workgroup into LDS (table head times row factor, centred,
// as in k_ntt16p).  Inverse twiddles come from the same entries: psi^-e = -psi^(N - e), so the inverse
// twiddle of entry 2^s + k is minus the forward one of entry 2^s + (2^s - 1 - k), which lies in
// the mirrored row 2^s0 - 1 - sub.
// Bounds: every twiddle is paired with w * RN(1/q), so a product is within (1/2 + |b| / 8Q) q of zero for a
// multiplied operand |b| < 4Q (Q = 2^50).  Forward: inputs centred, four stages with operands below 3.5Q,
// centring, four more.  Inverse: inputs centred, sums centred every second stage, operands below 3.9Q.
#pragma once
#include "vh_device.h"

struct vh_row8 {
    static constexpr int ROWS = 8, S = 256, T = 32, PITCH = 288;   // PITCH: doubles of a row's exchange slice
    double q, qinv;
    double *xs;          // the row's exchange slice
    const double *tw;    // the row's forward twiddles
    int t, ta, tb;

    // Entry e of row r = head e times the factor of e's stage of row sub(r); every thread takes part.
    template <typename F>
    static __device__ __forceinline__ void fill(double (*tws)[S], const vh_limb &L, F sub)
    {
        const int e = threadIdx.x, sp = e ? 31 - __builtin_clz(e) : 0;
        const double h = vh_global(reinterpret_cast<const double *>(L.tw_fwd))[2 * e];
        const VH_GLOBAL double *rf = vh_global(reinterpret_cast<const double *>(L.rowf_fwd)) + 2 * sp;
#pragma unroll
        for (int r = 0; r < ROWS; r++) {
            const size_t at = (size_t)sub(r) * 16;
            tws[r][e] = vh_center(vh_mulmod_tw(h, rf[at], rf[at + 1], L.qd), L.qd, L.qinv);
        }
    }
    __device__ __forceinline__ vh_row8(const vh_limb &L, double *lds, const double (*tws)[S])
        : q(L.qd), qinv(L.qinv), xs(lds + (threadIdx.x / T) * PITCH), tw(tws[threadIdx.x / T]), t(threadIdx.x % T),
          ta(t >> 2), tb(t & 3)
    {
    }
    __device__ __forceinline__ double centre(double x) const { return vh_center(x, q, qinv); }
    __device__ __forceinline__ void ct(double &a, double &b, double w) const
    {
        const double x = vh_mulmod_tw(b, w, w * qinv, q);
        b = a - x;
        a = a + x;
    }
    __device__ __forceinline__ void gs(double &a, double &b, double w, bool second) const   // w: minus the inverse twiddle
    {
        const double s = a + b;
        b = vh_mulmod_tw(b - a, w, w * qinv, q);
        a = second ? centre(s) : s;
    }
    // K operands at once (each twiddle read once): element t + 32 m in; 128 (m >> 2) + 4 t + (m & 3) out,
    // not centred
    template <int K>
    __device__ __forceinline__ void fwd(double (&v)[K][8]) const
    {
#pragma unroll
        for (int s = 0; s < 3; s++) {
            const int hm = 4 >> s;
#pragma unroll
            for (int m = 0; m < 8; m++) {
                if (m & hm) continue;
                const double w = tw[(1 << s) + (m >> (3 - s))];
#pragma unroll
                for (int k = 0; k < K; k++) ct(v[k][m], v[k][m + hm], w);
            }
        }
#pragma unroll
        for (int k = 0; k < K; k++) {
            vh_wave_sync();   // every read of an earlier exchange is done
#pragma unroll
            for (int m = 0; m < 8; m++) xs[t + 36 * m] = v[k][m];
            vh_wave_sync();
#pragma unroll
            for (int m = 0; m < 8; m++) v[k][m] = xs[36 * ta + 4 * m + tb];
        }
#pragma unroll
        for (int s = 3; s < 6; s++) {
            const int hm = 4 >> (s - 3);
#pragma unroll
            for (int m = 0; m < 8; m++) {
                if (m & hm) continue;
                const double w = tw[(1 << s) + (ta << (s - 3)) + (m >> (6 - s))];
#pragma unroll
                for (int k = 0; k < K; k++) ct(v[k][m], v[k][m + hm], w);
            }
            if (s == 3) {
#pragma unroll
                for (int k = 0; k < K; k++)
#pragma unroll
                    for (int m = 0; m < 8; m++) v[k][m] = centre(v[k][m]);
            }
        }
#pragma unroll
        for (int k = 0; k < K; k++) {
            if (K > 1) vh_wave_sync();   // K == 1: a thread overwrites the slots it read itself
#pragma unroll
            for (int m = 0; m < 8; m++) xs[36 * ta + 4 * m + tb] = v[k][m];
            vh_wave_sync();
#pragma unroll
            for (int m = 0; m < 8; m++) v[k][m] = xs[144 * (m >> 2) + 4 * t + 4 * (t >> 3) + (m & 3)];
        }
#pragma unroll
        for (int h = 0; h < 2; h++) {
            const double w6 = tw[64 + 32 * h + t], wa = tw[128 + 64 * h + 2 * t], wb = tw[129 + 64 * h + 2 * t];
#pragma unroll
            for (int k = 0; k < K; k++) {
                ct(v[k][4 * h], v[k][4 * h + 2], w6);
                ct(v[k][4 * h + 1], v[k][4 * h + 3], w6);
                ct(v[k][4 * h], v[k][4 * h + 1], wa);
                ct(v[k][4 * h + 2], v[k][4 * h + 3], wb);
            }
        }
    }
    // the other way; tm: the forward twiddles of the mirrored row.  |v| <= q/2 + 1 in, below 2q out.
    __device__ __forceinline__ void inv(double (&v)[8], const double *tm) const
    {
#pragma unroll
        for (int h = 0; h < 2; h++) {
            gs(v[4 * h], v[4 * h + 1], tm[255 - 64 * h - 2 * t], false);
            gs(v[4 * h + 2], v[4 * h + 3], tm[254 - 64 * h - 2 * t], false);
            const double w6 = tm[127 - 32 * h - t];
            gs(v[4 * h], v[4 * h + 2], w6, true);
            gs(v[4 * h + 1], v[4 * h + 3], w6, true);
        }
        vh_wave_sync();
#pragma unroll
        for (int m = 0; m < 8; m++) xs[144 * (m >> 2) + 4 * t + 4 * (t >> 3) + (m & 3)] = v[m];
        vh_wave_sync();
#pragma unroll
        for (int m = 0; m < 8; m++) v[m] = xs[36 * ta + 4 * m + tb];
#pragma unroll
        for (int s = 5; s >= 3; s--) {
            const int hm = 4 >> (s - 3);
#pragma unroll
            for (int m = 0; m < 8; m++)
                if (!(m & hm)) gs(v[m], v[m + hm], tm[(2 << s) - 1 - (ta << (s - 3)) - (m >> (6 - s))], s == 4);
        }
#pragma unroll
        for (int m = 0; m < 8; m++) xs[36 * ta + 4 * m + tb] = v[m];
        vh_wave_sync();
#pragma unroll
        for (int m = 0; m < 8; m++) v[m] = xs[t + 36 * m];
#pragma unroll
        for (int s = 2; s >= 0; s--) {
            const int hm = 4 >> s;
#pragma unroll
            for (int m = 0; m < 8; m++)
                if (!(m & hm)) gs(v[m], v[m + hm], tm[(2 << s) - 1 - (m >> (3 - s))], s != 1);
        }
    }
};
