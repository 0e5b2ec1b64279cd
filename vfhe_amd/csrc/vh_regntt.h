// vh_regntt.h -- register transforms of the merged negacyclic network (CT forward, natural in,
// bit-reversed out; GS inverse), 16 values per thread, over either arithmetic.
#pragma once
#include "vh_device.h"

// FP64 path (q < 2^50): integer-valued doubles.  Between centrings at most four stages, |x| < 2^52
// (vh_mulmod_tw); inverse sums are re-centred after every second stage.
struct vh_ar_fp {
    using V = double;
    static constexpr bool FP = true;
    double q, qinv;
    const VH_GLOBAL double *tw;
    __device__ __forceinline__ vh_ar_fp(const vh_limb &L, int dir)
        : q(L.qd), qinv(L.qinv), tw(vh_global(reinterpret_cast<const double *>(dir == 0 ? L.tw_fwd : L.tw_inv)))
    {
    }
    __device__ __forceinline__ static V load(uint64_t x) { return vh_u2d(x); }
    __device__ __forceinline__ void ct(V &a, V &b, unsigned i) const
    {
        const double x = vh_mulmod_tw(b, tw[2 * i], tw[2 * i + 1], q);
        b = a - x;
        a = a + x;
    }
    __device__ __forceinline__ void gs(V &a, V &b, unsigned i, bool second) const
    {
        const double s = a + b;
        b = vh_mulmod_tw(a - b, tw[2 * i], tw[2 * i + 1], q);
        a = second ? vh_center(s, q, qinv) : s;
    }
    __device__ __forceinline__ V mid(V x) const { return vh_center(x, q, qinv); }       // between forward phases
    __device__ __forceinline__ uint64_t canon(V x) const { return vh_d2u(vh_canon(x, q, qinv)); }
    __device__ __forceinline__ uint64_t scaled(V x, const vh_limb &L) const             // x n^-1, canonical
    {
        return canon(vh_mulmod_tw(x, L.ninv_d, L.ninv_q, q));
    }
    // product of two forward outputs, fit for the inverse: operands centred, |result| <= q/2 + 1
    __device__ __forceinline__ V product(V x, V y, const vh_limb &) const
    {
        const double a = vh_center(x, q, qinv), b = vh_center(y, q, qinv);
        const double hi = a * b, lo = __fma_rn(a, b, -hi);
        const double qt = __fma_rn(a, b * qinv, VH_MAGIC) - VH_MAGIC;
        return vh_center(__fma_rn(-qt, q, hi) + lo, q, qinv);
    }
};

// Integer path for q < 2^62: lazy residues (Harvey, "Faster arithmetic for number-theoretic
// transforms", J. Symbolic Computation 60 (2014)): forward values stay below 4q, inverse values
// below 2q, and a Shoup product of any 64-bit value is left in [0, 2q).
struct vh_ar_int {
    using V = uint64_t;
    static constexpr bool FP = false;
    uint64_t q, q2;
    const VH_GLOBAL uint64_t *tw;
    __device__ __forceinline__ vh_ar_int(const vh_limb &L, int dir)
        : q(L.q), q2(2 * L.q), tw(vh_global(reinterpret_cast<const uint64_t *>(dir == 0 ? L.twi_fwd : L.twi_inv)))
    {
    }
    __device__ __forceinline__ static V load(uint64_t x) { return x; }
    __device__ __forceinline__ V lazy(V a, unsigned i) const
    {
        uint64_t w, wsh;
        vh_ld2(tw + 2 * i, w, wsh);
        return a * w - vh_mulhi(a, wsh) * q;
    }
    __device__ __forceinline__ void ct(V &a, V &b, unsigned i) const
    {
        const V u = a >= q2 ? a - q2 : a, t = lazy(b, i);
        a = u + t;
        b = u - t + q2;
    }
    __device__ __forceinline__ void gs(V &a, V &b, unsigned i, bool) const
    {
        const V s = a + b;
        b = lazy(a - b + q2, i);
        a = s >= q2 ? s - q2 : s;
    }
    __device__ __forceinline__ V mid(V x) const { return x; }
    __device__ __forceinline__ uint64_t canon(V x) const
    {
        x = x >= q2 ? x - q2 : x;
        return x >= q ? x - q : x;
    }
    __device__ __forceinline__ uint64_t scaled(V x, const vh_limb &L) const { return vh_shoup(x, L.ninv, L.ninv_sh, q); }
    __device__ __forceinline__ V product(V x, V y, const vh_limb &L) const { return vh_mulmod(canon(x), canon(y), L); }
};

// Whole transforms of N = 2^9 .. 2^12 points, T = N/16 threads per transform, in three phases:
//   A  stages 0..3         stride ownership   j = t + T m            (uniform twiddles)
//   B  stages 4..7         middle ownership   j = 16U g + u + U m    (t = u + U g, U = T/16)
//   C  stages 8..logN-1    contiguous         j = 16 t + m
// with an LDS exchange between phases (one pad slot per 16 values: the contiguous reads
// stride 17 words).  A stage-s butterfly on (j, j + N/2^(s+1)) takes the twiddle of index
// 2^s + (j >> (logN - s)), so every product is the reference's and the canonical outputs
// are identical.  lds holds N + N/16 words private to the transform.  WAVE: the transform's
// threads are one wave (or part of one), so the exchanges need only the wave's own ordering.
template <int LOGN> struct vh_reg_ntt {
    static constexpr int N = 1 << LOGN, T = N / 16, U = T / 16;
    static __device__ __forceinline__ int li(int j) { return j + (j >> 4); }
    static __device__ __forceinline__ int jA(int t, int m) { return t + T * m; }
    static __device__ __forceinline__ int jB(int t, int m) { return 16 * U * (t / U) + t % U + U * m; }
    static __device__ __forceinline__ int jC(int t, int m) { return 16 * t + m; }
    template <bool WAVE> static __device__ __forceinline__ void sync()
    {
        if (WAVE) vh_wave_sync();
        else __syncthreads();
    }
    template <bool WAVE, typename V, typename FW, typename FR>
    static __device__ __forceinline__ void exchange(V (&v)[16], V *lds, FW jw, FR jr)
    {
#pragma unroll
        for (int m = 0; m < 16; m++) lds[li(jw(m))] = v[m];
        sync<WAVE>();
#pragma unroll
        for (int m = 0; m < 16; m++) v[m] = lds[li(jr(m))];
        sync<WAVE>();
    }
    // forward: v in the stride ownership -> contiguous ownership
    template <bool WAVE, typename AR>
    static __device__ __forceinline__ void fwd(typename AR::V (&v)[16], typename AR::V *lds, int t, const AR &ar)
    {
        const int g = t / U;
        auto ct = [&](int s, int hm, auto blk) {
#pragma unroll
            for (int m = 0; m < 16; m++)
                if (!(m & hm)) ar.ct(v[m], v[m + hm], (1u << s) + blk(m));
        };
        auto mid = [&]() {
#pragma unroll
            for (int m = 0; m < 16; m++) v[m] = ar.mid(v[m]);
        };
#pragma unroll
        for (int s = 0; s < 4; s++) ct(s, 8 >> s, [&](int m) { return m >> (4 - s); });
        mid();
        exchange<WAVE>(v, lds, [&](int m) { return jA(t, m); }, [&](int m) { return jB(t, m); });
#pragma unroll
        for (int s = 4; s < 8; s++) ct(s, 8 >> (s - 4), [&](int m) { return (g << (s - 4)) + (m >> (8 - s)); });
        mid();
        exchange<WAVE>(v, lds, [&](int m) { return jB(t, m); }, [&](int m) { return jC(t, m); });
#pragma unroll
        for (int s = 8; s < LOGN; s++) ct(s, 1 << (LOGN - s - 1), [&](int m) { return (16 * t + m) >> (LOGN - s); });
    }
    // inverse (before the n^-1 factor): v in the contiguous ownership (FP64: |v| <= q) -> stride ownership
    template <bool WAVE, typename AR>
    static __device__ __forceinline__ void inv(typename AR::V (&v)[16], typename AR::V *lds, int t, const AR &ar)
    {
        const int g = t / U;
        int c = 0;
        auto gs = [&](int s, int hm, auto blk) {
#pragma unroll
            for (int m = 0; m < 16; m++)
                if (!(m & hm)) ar.gs(v[m], v[m + hm], (1u << s) + blk(m), c & 1);
            c++;
        };
#pragma unroll
        for (int s = LOGN - 1; s >= 8; s--) gs(s, 1 << (LOGN - s - 1), [&](int m) { return (16 * t + m) >> (LOGN - s); });
        exchange<WAVE>(v, lds, [&](int m) { return jC(t, m); }, [&](int m) { return jB(t, m); });
#pragma unroll
        for (int s = 7; s >= 4; s--) gs(s, 8 >> (s - 4), [&](int m) { return (g << (s - 4)) + (m >> (8 - s)); });
        exchange<WAVE>(v, lds, [&](int m) { return jB(t, m); }, [&](int m) { return jA(t, m); });
#pragma unroll
        for (int s = 3; s >= 0; s--) gs(s, 8 >> s, [&](int m) { return m >> (4 - s); });
    }
};
