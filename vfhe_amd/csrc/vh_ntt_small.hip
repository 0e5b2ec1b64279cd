// vh_ntt_small.hip -- transforms and products of small rings in one pass over the data
// (N = 2^9 .. 2^12, both arithmetics), and the integer path's two-pass transforms for
// N = 2^13 .. 2^16 (q < 2^62).
#include "vh_kernels.h"
#include "vh_regntt.h"

// ---------------------------------------------------------------------------
// 4096/N transforms (or products) per 256-thread workgroup.  Rows are loaded and stored in
// the stride ownership (whole 128-byte runs per instruction); the forward pass regroups its
// output through LDS for that.
// ---------------------------------------------------------------------------
template <int DIR, int LOGN, typename AR, unsigned CAP>
__global__ void __launch_bounds__(256)
k_ntt_small(const vh_items_t<CAP> items, unsigned nitems, const vh_limb *__restrict__ limbs)
{
    using R = vh_reg_ntt<LOGN>;
    using V = typename AR::V;
    constexpr int N = R::N, T = R::T, PER = 256 / T, PAD = N + N / 16;
    constexpr bool WAVE = T <= 64;
    static_assert(LOGN >= 9 && LOGN <= 12, "k_ntt_small: N = 2^9 .. 2^12");
    __shared__ V lds_all[PER * PAD];
    const int tid = threadIdx.x, slot = tid / T, t = tid % T;
    const unsigned idx = blockIdx.x * PER + slot;
    const bool live = idx < nitems;
    // a slot past the end transforms the last item again (every thread reaches the
    // barriers) and stores nothing
    const vh_item it = items[live ? idx : nitems - 1];
    const vh_limb &L = limbs[it.limb];
    const AR ar(L, DIR);
    V *lds = lds_all + slot * PAD;
    const VH_GLOBAL uint64_t *in = vh_global(it.src);
    VH_GLOBAL uint64_t *out = vh_global(it.dst);
    V v[16];
#pragma unroll
    for (int m = 0; m < 16; m++) v[m] = AR::load(vh_ld(in + R::jA(t, m)));
    if (DIR == 0) {
        R::template fwd<WAVE>(v, lds, t, ar);
        uint64_t w[16];
#pragma unroll
        for (int m = 0; m < 16; m++) w[m] = ar.canon(v[m]);
        R::template exchange<WAVE>(w, reinterpret_cast<uint64_t *>(lds), [&](int m) { return R::jC(t, m); },
                                   [&](int m) { return R::jA(t, m); });
        if (live) {
#pragma unroll
            for (int m = 0; m < 16; m++) vh_st(out + R::jA(t, m), w[m]);
        }
    } else {
        R::template exchange<WAVE>(v, lds, [&](int m) { return R::jA(t, m); }, [&](int m) { return R::jC(t, m); });
        R::template inv<WAVE>(v, lds, t, ar);
        if (live) {
#pragma unroll
            for (int m = 0; m < 16; m++) vh_st(out + R::jA(t, m), ar.scaled(v[m], L));
        }
    }
}

// z = INTT(NTT(x) NTT(y)) of whole rows: x in it.src, y in it.src2, z in it.dst; both forward
// transforms, the product and the inverse stay in registers.  One launch and 24 N bytes per row
// where separate transforms and a product take 72 N bytes, three launches and temporaries.
// 37 pairs x 3 limbs of N = 2048: 189 us a call (24 us of it kernels, the rest a temporary
// polynomial per pair) -> 21 to 24 us.  Bound by latency at every batch: 64 pairs x 24 limbs of
// N = 4096 take 112 us for 151 MB (1.3 TB/s) and 35 us of VALU issue, two waves a SIMD (210 to 248
// VGPRs from N = 1024) waiting for 72% of their time.  The integer instances want more registers
// than that leaves and spill 48 at N = 2048 (188 bytes a lane), 82 at 4096 (324 bytes): one pair of
// 60 bits at N = 4096 takes 35 us, and took 81 in separate launches of the radix-2 kernel.
template <int LOGN, typename AR>
__global__ void __launch_bounds__(256, 2)
k_product_small(const vh_items items, unsigned nitems, const vh_limb *__restrict__ limbs)
{
    using R = vh_reg_ntt<LOGN>;
    using V = typename AR::V;
    constexpr int N = R::N, T = R::T, PER = 256 / T, PAD = N + N / 16;
    constexpr bool WAVE = T <= 64;
    __shared__ V lds_all[PER * PAD];
    const int tid = threadIdx.x, slot = tid / T, t = tid % T;
    const unsigned idx = blockIdx.x * PER + slot;
    const bool live = idx < nitems;
    const vh_item it = items[live ? idx : nitems - 1];
    const vh_limb &L = limbs[it.limb];
    const AR fw(L, 0), iv(L, 1);
    V *lds = lds_all + slot * PAD;
    const VH_GLOBAL uint64_t *x = vh_global(it.src), *y = vh_global(it.src2);
    V a[16], b[16];
#pragma unroll
    for (int m = 0; m < 16; m++) a[m] = AR::load(vh_ld(x + R::jA(t, m)));
#pragma unroll
    for (int m = 0; m < 16; m++) b[m] = AR::load(vh_ld(y + R::jA(t, m)));
    R::template fwd<WAVE>(a, lds, t, fw);
    asm volatile("" ::: "memory");   // the twiddles are read again for y rather than held in registers
    R::template fwd<WAVE>(b, lds, t, fw);
#pragma unroll
    for (int m = 0; m < 16; m++) a[m] = fw.product(a[m], b[m], L);
    R::template inv<WAVE>(a, lds, t, iv);
    VH_GLOBAL uint64_t *z = vh_global(it.dst);
    if (live) {
#pragma unroll
        for (int m = 0; m < 16; m++) vh_st(z + R::jA(t, m), iv.scaled(a[m], L));
    }
}

// ---------------------------------------------------------------------------
// Integer path, N = 2^13 .. 2^16: the two-pass split of the FP64 kernels (a column pass of the
// first logn - 8 stages over sub-transforms of stride 2^8, a row pass of the last 8 stages on
// contiguous rows of 256), 16 values per thread in registers and one exchange through LDS, in
// place of a radix-2 pass that went through LDS for every stage.  Values between the passes stay
// lazy (below 4q forward, 2q inverse).  Twiddles are read from the table: they cost less here
// than forming them would with 64-bit products.  9 products x 6 limbs of 60 bits at N = 2^14:
// 189 us in five launches of the radix-2 and elementwise kernels, 53 us in three.
// ---------------------------------------------------------------------------
template <int R, bool COL> struct vh_pass {   // one thread's part of a 2^R-point sub-transform
    static constexpr int S = 1 << R, TPS = S / 16, G = 256 / TPS;
    static constexpr int LDS = COL ? S * (G + 1) : G * (S + S / 16);
    static __device__ __forceinline__ int g(int tid) { return COL ? tid % G : tid / TPS; }
    static __device__ __forceinline__ int t(int tid) { return COL ? tid / G : tid % TPS; }
    static __device__ __forceinline__ int li(int g, int k) { return COL ? k * (G + 1) + g : g * (S + S / 16) + k + (k >> 4); }
    // a row's 16 threads are in one wave; a column's are spread over the workgroup
    static __device__ __forceinline__ void sync()
    {
        if (COL) __syncthreads();
        else vh_wave_sync();
    }
    // element t + TPS m in, 16 t + m out; tb(s', local): the twiddle index
    template <typename AR, typename TB>
    static __device__ __forceinline__ void fwd(uint64_t (&v)[16], uint64_t *lds, int g, int t, const AR &ar, TB tb)
    {
#pragma unroll
        for (int s = 0; s < 4; s++)
#pragma unroll
            for (int m = 0; m < 16; m++)
                if (!(m & (8 >> s))) ar.ct(v[m], v[m + (8 >> s)], tb(s, m >> (4 - s)));
        if (!COL) sync();   // a row's slice may still be read by an earlier exchange
#pragma unroll
        for (int m = 0; m < 16; m++) lds[li(g, t + TPS * m)] = v[m];
        sync();
#pragma unroll
        for (int m = 0; m < 16; m++) v[m] = lds[li(g, 16 * t + m)];
#pragma unroll
        for (int s = 4; s < R; s++) {
            const int hm = 1 << (R - s - 1);
#pragma unroll
            for (int m = 0; m < 16; m++)
                if (!(m & hm)) ar.ct(v[m], v[m + hm], tb(s, (16 * t + m) >> (R - s)));
        }
    }
    // element 16 t + m in, t + TPS m out
    template <typename AR, typename TB>
    static __device__ __forceinline__ void inv(uint64_t (&v)[16], uint64_t *lds, int g, int t, const AR &ar, TB tb)
    {
#pragma unroll
        for (int s = R - 1; s >= 4; s--) {
            const int hm = 1 << (R - s - 1);
#pragma unroll
            for (int m = 0; m < 16; m++)
                if (!(m & hm)) ar.gs(v[m], v[m + hm], tb(s, (16 * t + m) >> (R - s)), false);
        }
        if (!COL) sync();
#pragma unroll
        for (int m = 0; m < 16; m++) lds[li(g, 16 * t + m)] = v[m];
        sync();
#pragma unroll
        for (int m = 0; m < 16; m++) v[m] = lds[li(g, t + TPS * m)];
#pragma unroll
        for (int s = 3; s >= 0; s--)
#pragma unroll
            for (int m = 0; m < 16; m++)
                if (!(m & (8 >> s))) ar.gs(v[m], v[m + (8 >> s)], tb(s, m >> (4 - s)), false);
    }
    // row pass: between the stride and the contiguous ownership, through LDS
    static __device__ __forceinline__ void regroup(uint64_t (&v)[16], uint64_t *lds, int g, int t, bool to_contiguous)
    {
        sync();
#pragma unroll
        for (int m = 0; m < 16; m++) lds[li(g, to_contiguous ? t + TPS * m : 16 * t + m)] = v[m];
        sync();
#pragma unroll
        for (int m = 0; m < 16; m++) v[m] = lds[li(g, to_contiguous ? 16 * t + m : t + TPS * m)];
    }
};

// DIR 0: column pass (reads it.src), then row pass (in it.dst, canonical out).
// DIR 1: row pass (reads it.src), then column pass (in it.dst, times n^-1, canonical out).
template <int DIR, int R, bool COL>
__global__ void __launch_bounds__(256)
k_ntt16i(const vh_item *__restrict__ items, const vh_limb *__restrict__ limbs, int logn)
{
    using P = vh_pass<R, COL>;
    constexpr bool FIRST = COL == (DIR == 0);
    __shared__ uint64_t lds[P::LDS];
    const vh_item &it = items[blockIdx.y];
    const vh_limb &L = limbs[it.limb];
    const vh_ar_int ar(L, DIR);
    const int g = P::g(threadIdx.x), t = P::t(threadIdx.x);
    const unsigned sub = blockIdx.x * P::G + g, nsub = 1u << (logn - R);
    const VH_GLOBAL uint64_t *in = vh_global(FIRST ? it.src : it.dst);
    VH_GLOBAL uint64_t *out = vh_global(it.dst);
    auto at = [&](int k) -> unsigned { return COL ? sub + (unsigned)k * nsub : sub * P::S + (unsigned)k; };
    const int s0 = COL ? 0 : logn - 8;
    auto tb = [&](int s, int local) -> unsigned { return (1u << (s0 + s)) + ((COL ? 0u : sub) << s) + (unsigned)local; };
    uint64_t v[16];
    if (DIR == 0) {
#pragma unroll
        for (int m = 0; m < 16; m++) v[m] = vh_ld(in + at(t + P::TPS * m));
        P::fwd(v, lds, g, t, ar, tb);
        if (COL) {
#pragma unroll
            for (int m = 0; m < 16; m++) out[at(16 * t + m)] = v[m];
        } else {
#pragma unroll
            for (int m = 0; m < 16; m++) v[m] = ar.canon(v[m]);
            P::regroup(v, lds, g, t, false);
#pragma unroll
            for (int m = 0; m < 16; m++) vh_st(out + at(t + P::TPS * m), v[m]);
        }
    } else {
        if (COL) {
#pragma unroll
            for (int m = 0; m < 16; m++) v[m] = vh_ld(in + at(16 * t + m));
        } else {
#pragma unroll
            for (int m = 0; m < 16; m++) v[m] = vh_ld(in + at(t + P::TPS * m));
            P::regroup(v, lds, g, t, true);
        }
        P::inv(v, lds, g, t, ar, tb);
#pragma unroll
        for (int m = 0; m < 16; m++) {
            if (COL) vh_st(out + at(t + P::TPS * m), ar.scaled(v[m], L));
            else out[at(t + P::TPS * m)] = v[m];
        }
    }
}

// The product's middle step on the integer path: forward row stages of it.src and it.src2
// (column-pass outputs), their pointwise product and the inverse row stages, into it.dst.
__global__ void __launch_bounds__(256, 2)
k_ntt16i_row_mul(const vh_item *__restrict__ items, const vh_limb *__restrict__ limbs, int logn)
{
    using P = vh_pass<8, false>;
    __shared__ uint64_t lds[P::LDS];
    const vh_item &it = items[blockIdx.y];
    const vh_limb &L = limbs[it.limb];
    const vh_ar_int fw(L, 0), iv(L, 1);
    const int g = P::g(threadIdx.x), t = P::t(threadIdx.x);
    const unsigned sub = blockIdx.x * P::G + g;
    const int s0 = logn - 8;
    auto tb = [&](int s, int local) -> unsigned { return (1u << (s0 + s)) + (sub << s) + (unsigned)local; };
    const VH_GLOBAL uint64_t *x = vh_global(it.src) + (size_t)sub * P::S + t, *y = vh_global(it.src2) + (size_t)sub * P::S + t;
    uint64_t a[16], b[16];
#pragma unroll
    for (int m = 0; m < 16; m++) a[m] = vh_ld(x + P::TPS * m);
#pragma unroll
    for (int m = 0; m < 16; m++) b[m] = vh_ld(y + P::TPS * m);
    P::fwd(a, lds, g, t, fw, tb);
    asm volatile("" ::: "memory");   // the twiddles are read again for y rather than held in registers
    P::fwd(b, lds, g, t, fw, tb);
#pragma unroll
    for (int m = 0; m < 16; m++) a[m] = fw.product(a[m], b[m], L);
    P::inv(a, lds, g, t, iv, tb);
    VH_GLOBAL uint64_t *z = vh_global(it.dst) + (size_t)sub * P::S + t;
#pragma unroll
    for (int m = 0; m < 16; m++) z[P::TPS * m] = a[m];
}

// ---------------------------------------------------------------------------
// Launchers
// ---------------------------------------------------------------------------
// Lists in the arguments (vh_items_t): 16 polynomials x 4 limbs of N = 4096 took 11.1 us with the list in
// host memory, 7.6 us so.  The launch copies the whole block, so lists of at most 16 rows (and staged
// ones) get a short one.  That is worth little: 0.1 us of 5.5 to 7 at best on a short list, 0.2 of 19 on
// staged lists of 512 rows.  A third block of 32 rows changed nothing (17 to 32 rows alike to 0.1 us).
// A single ring product (launches of 7 and 28 rows) gains nothing either way: its kernels went from
// 15 to 11 us and the host's part, 17 to 23 us from run to run, decides.
template <int LOGN, typename AR, unsigned CAP>
static void vh_ntt_small_go(hipStream_t st, const vh_items_t<CAP> &items, unsigned nitems, const vh_limb *limbs, int dir)
{
    const unsigned per = 4096u >> LOGN, nb = (nitems + per - 1) / per;
    if (dir == 0) VH_KL((k_ntt_small<0, LOGN, AR, CAP>), dim3(nb), dim3(256), 0, st, items, nitems, limbs);
    else VH_KL((k_ntt_small<1, LOGN, AR, CAP>), dim3(nb), dim3(256), 0, st, items, nitems, limbs);
}

hipError_t vh_launch_ntt_small(hipStream_t st, const vh_items &items, unsigned nitems, const vh_limb *limbs, int dir,
                               int logn, int fp)
{
    if (logn < 9 || logn > 12 || nitems == 0) return hipErrorInvalidValue;
#define VH_SMALL(LG, AR)                                                                                    \
        if (items.p || nitems <= 16) vh_ntt_small_go<LG, AR>(st, vh_items_cut<16>(items, nitems), nitems, limbs, dir); \
        else vh_ntt_small_go<LG, AR>(st, items, nitems, limbs, dir);
#define VH_SIZE(LG) case LG: if (fp) { VH_SMALL(LG, vh_ar_fp) } else { VH_SMALL(LG, vh_ar_int) } break;
    switch (logn) { VH_SIZE(9) VH_SIZE(10) VH_SIZE(11) VH_SIZE(12) }
#undef VH_SIZE
#undef VH_SMALL
    return hipGetLastError();
}

hipError_t vh_launch_product_small(hipStream_t st, const vh_items &items, unsigned nitems, const vh_limb *limbs,
                                   int logn, int fp)
{
    if (logn < 9 || logn > 12 || nitems == 0) return hipErrorInvalidValue;
    const unsigned per = 4096u >> logn, nb = (nitems + per - 1) / per;
#define VH_PROD(LG)                                                                                         \
    case LG:                                                                                                \
        if (fp) VH_KL((k_product_small<LG, vh_ar_fp>), dim3(nb), dim3(256), 0, st, items, nitems, limbs);   \
        else VH_KL((k_product_small<LG, vh_ar_int>), dim3(nb), dim3(256), 0, st, items, nitems, limbs);     \
        break;
    switch (logn) { VH_PROD(9) VH_PROD(10) VH_PROD(11) VH_PROD(12) }
#undef VH_PROD
    return hipGetLastError();
}

hipError_t vh_launch_ntt16i(hipStream_t st, const vh_item *items, unsigned nitems, const vh_limb *limbs, int dir,
                            int logn, int col)
{
    if (logn < 13 || logn > 16 || nitems == 0) return hipErrorInvalidValue;
    const dim3 grid(1u << (logn - 12), nitems), block(256);
    if (!col) {
        if (dir == 0) VH_KL((k_ntt16i<0, 8, false>), grid, block, 0, st, items, limbs, logn);
        else VH_KL((k_ntt16i<1, 8, false>), grid, block, 0, st, items, limbs, logn);
        return hipGetLastError();
    }
#define VH_COL(RR)                                                                                          \
    case RR:                                                                                                \
        if (dir == 0) VH_KL((k_ntt16i<0, RR, true>), grid, block, 0, st, items, limbs, logn);               \
        else VH_KL((k_ntt16i<1, RR, true>), grid, block, 0, st, items, limbs, logn);                        \
        break;
    switch (logn - 8) { VH_COL(5) VH_COL(6) VH_COL(7) VH_COL(8) }
#undef VH_COL
    return hipGetLastError();
}

hipError_t vh_launch_ntt16i_row_mul(hipStream_t st, const vh_item *items, unsigned nitems, const vh_limb *limbs, int logn)
{
    if (logn < 13 || logn > 16 || nitems == 0) return hipErrorInvalidValue;
    VH_KL(k_ntt16i_row_mul, dim3(1u << (logn - 12), nitems), dim3(256), 0, st, items, limbs, logn);
    return hipGetLastError();
}
