// vh_cggi.hip -- CGGI16 blind rotation over RNS primes, every key index in one launch.
#include "vh_device.h"
#include "vh_kernels.h"

// ---------------------------------------------------------------------------
// CGGI16 blind rotation of a batch (cggi16.py:70-90 with mgsw.c:51-71 per index).
// N = 1024, FP64 limbs, one special prime.  Per key index i with a = amounts[k n + i]:
//   digit d = (component c, level limb J[jj]):  (X^a - 1) acc_c  at limb J[jj], canonical
//     (the reference's mlwe_RNSc_mul_by_xai, subtraction and gadget lift; the lift is the
//     identity on values below q_J[jj] < 2^50, which the FP64 transform accepts for any E[w]);
//   out_c' = sum_d NTT_E[w](digit_d) * bk[i][d] component c' at every extended limb E[w];
//   then per c': inverse transform, t = (x + floor(p/2)) mod p of the special limb, and every
//     level limb adds (x + floor(p/2) - t) p^-1 mod q to its accumulator row (round division
//     by p, then the CMUX's  acc + ExtProd(X^a acc - acc)).
// An exponent of 0 gives zero digits and adds zero: the reference's skipped index.
//
// Two waves per extended limb and accumulator, 8 values per lane; wave h owns the half
// [512 h, 512 h + 512) of the coefficients and of the transform.  The first forward stage
// joins the halves: both waves read both halves of the digit from LDS and compute their own
// side of it, and the other nine stages stay inside the wave (three register phases of three
// stages, exchanges through the wave's own LDS slice).  The inverse mirrors it: nine stages in
// the wave, then one exchange with the partner.  So the transforms need no workgroup barrier,
// and the 6 or 12 waves of a workgroup spread evenly over the SIMDs.
//
// A level wave keeps its half of its limb's accumulator rows in registers; `reg` holds the copy
// that rotated reads need, then the digits (formed once, read by every limb's waves), then
// the halves' exchange of the inverse transforms.  The twiddles of every extended limb sit in
// LDS, one table for both directions: psi^-e = -psi^(N - e), so the inverse twiddle of entry
// 2^s + k is minus the forward one of entry 2^s + (2^s - 1 - k).
//
// Bounds (Q = 2^50, every q < Q).  Twiddles are paired with w * RN(1/q), so for a multiplied
// operand b < 4Q the product is within (1/2 + b / 8Q) q < q of zero.  Forward: digits below Q, four
// stages reach 4.3Q with operands below 3.4Q, centring, five stages reach 4.1Q with operands
// below 3.3Q; before the tenth its operands are centred.  Inverse: sums centred every second
// stage keep every operand below 3.9Q.
//
// Bound by FP64 issue: 14.3 G VALU wave instructions for 1024 accumulators (n = 630, two level
// limbs), 25.5 ms at the clock the run holds; 36.3 ms measured.  One wave per limb with 16
// contiguous key words per lane took 69.5 ms: three waves per accumulator leave two SIMDs with
// half the work of the others, every key or twiddle load touched up to 64 lines, and each digit
// waited for its row pointers and then its key words.
// ---------------------------------------------------------------------------
namespace {
constexpr int BN = 1024, BH = 512, BSCR = 576;   // ring, half, doubles of a wave's exchange slice

// One component and one level limb: the t row lies over the digits, and the halves go through the waves'
// slices as every last component's do.  70 KiB a workgroup instead of 116, two of them on a CU: 513
// accumulators at n = 60 take 0.69 ms (0.87), 1024 take 0.70 ms (0.89).  At more level limbs still one
// workgroup would fit, and the tighter layout is slower (two limbs, 1 accumulator: 0.58 ms against 0.54).
template <int C, int NJ> constexpr bool br_lean() { return C == 1 && NJ == 1; }
template <int C, int NJ> constexpr int br_reg()   // doubles: the rows, or the exchanged halves and one t row
{
    return (br_lean<C, NJ>() || C * NJ > NJ + 2 ? C * NJ : NJ + 2) * BN;
}
template <int C, int NJ, int G> constexpr int br_per_acc()
{
    return br_reg<C, NJ>() + 2 * G * (NJ + 1) * BSCR + (br_lean<C, NJ>() ? 0 : BN);
}
template <int C, int NJ, int NA, int G> constexpr int br_lds() { return NA * br_per_acc<C, NJ, G>() + (NJ + 1) * BN; }
}  // namespace

// NA: accumulators per workgroup.  G = 2: two groups of waves per accumulator; group g takes
// half of the digits, and component g of the product after the groups have swapped partial sums.
template <int C, int NJ, int NA, int G>
__global__ void __launch_bounds__(NA * G * (NJ + 1) * 128)
k_blind_rotate(const vh_br_params P, const vh_limb *__restrict__ limbs, uint64_t *const *__restrict__ accp,
               const uint64_t *const *__restrict__ bkp, const uint64_t *__restrict__ amounts,
               const uint64_t *const *__restrict__ tvp, const uint64_t *__restrict__ rot, unsigned count)
{
    static_assert(G == 1 || (G == 2 && C == 2), "a group per component");
    constexpr int next = NJ + 1, nd = C * NJ, REG = br_reg<C, NJ>(), PER = br_per_acc<C, NJ, G>();
    constexpr int OC = C / G, ND = nd / G;   // components a wave owns, digits it transforms
    __shared__ double lds[br_lds<C, NJ, NA, G>()];
    const int lane = threadIdx.x & 63, wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int h = wv & 1, w = (wv >> 1) % next, g = (wv / (2 * next)) % G, ac = wv / (2 * next * G);
    const int c0 = g * OC, d0 = g * ND;   // the wave's first component and digit
    const unsigned k = blockIdx.x * NA + ac;
    const bool live = k < count;   // a slot past the end works on zeros and stores nothing
    double *reg = lds + ac * PER;
    double *scr = reg + REG + ((g * next + w) * 2 + h) * BSCR, *pscr = reg + REG + ((g * next + w) * 2 + 1 - h) * BSCR;
    double *tlast = br_lean<C, NJ>() ? reg : reg + REG + 2 * G * next * BSCR, *tfirst = reg + next * BN;
    const double *tw = lds + NA * PER + w * BN;
    for (int e = threadIdx.x; e < next * BN; e += blockDim.x)
        lds[NA * PER + e] =
            vh_global(reinterpret_cast<const double *>(limbs[P.E[e / BN]].tw_fwd))[2 * (e % BN)];

    const vh_limb &L = limbs[P.E[w]];
    const double q = L.qd, qinv = L.qinv;
    const int jw = P.jw[w];          // level limb index, -1: the special limb
    const bool level = jw >= 0;
    const int x0 = BH * h + lane;    // the lane's coefficients: x0 + 64 m
    double own[OC][8];
#pragma unroll
    for (int c = 0; c < OC; c++) {
#pragma unroll
        for (int m = 0; m < 8; m++) own[c][m] = 0.0;
        if (level && live) {
            const int r = (c0 + c) * NJ + jw;
            if (tvp) {   // X^rot[k] * tv: coefficient u = (x - a) mod 2N of tv, negated when u >= N
                const VH_GLOBAL uint64_t *src = vh_global(tvp[r]);
                const uint32_t a = (uint32_t)(rot[k] & (2 * BN - 1));
#pragma unroll
                for (int m = 0; m < 8; m++) {
                    const uint32_t u = (uint32_t)(x0 + 64 * m + 2 * BN - a) & (2 * BN - 1);
                    const double s = vh_u2d(src[u & (BN - 1)]);
                    own[c][m] = (u < BN || s == 0.0) ? s : q - s;
                }
            } else {
                const VH_GLOBAL uint64_t *src = vh_global(accp[((size_t)k * C + c0 + c) * NJ + jw]);
#pragma unroll
                for (int m = 0; m < 8; m++) own[c][m] = vh_u2d(src[x0 + 64 * m]);
            }
        }
        if (level) {
#pragma unroll
            for (int m = 0; m < 8; m++) reg[((c0 + c) * NJ + jw) * BN + x0 + 64 * m] = own[c][m];
        }
    }
    __syncthreads();

    const int la = lane >> 3, lb = lane & 7;
    const double w1 = tw[1], wq1 = w1 * qinv, side = h ? -1.0 : 1.0;
    auto ct = [&](double &a, double &b, double wt) {
        const double x = vh_mulmod_tw(b, wt, wt * qinv, q);
        b = a - x;
        a = a + x;
    };
    auto gs = [&](double &a, double &b, double wt, bool centre) {
        const double s = a + b;
        b = vh_mulmod_tw(b - a, wt, wt * qinv, q);   // wt = minus the inverse twiddle
        a = centre ? vh_center(s, q, qinv) : s;
    };
    // the nine in-wave stages: element 64 m + lane in, 8 lane + m out (and back)
    auto fwd9 = [&](double (&v)[8]) {
#pragma unroll
        for (int s = 0; s < 3; s++)
#pragma unroll
            for (int m = 0; m < 8; m++)
                if (!(m & (4 >> s))) ct(v[m], v[m + (4 >> s)], tw[(2 << s) + (h << s) + (m >> (3 - s))]);
        vh_wave_sync();
#pragma unroll
        for (int m = 0; m < 8; m++) scr[72 * m + lane] = vh_center(v[m], q, qinv);
        vh_wave_sync();
#pragma unroll
        for (int m = 0; m < 8; m++) v[m] = scr[72 * la + 8 * m + lb];
#pragma unroll
        for (int s = 0; s < 3; s++)
#pragma unroll
            for (int m = 0; m < 8; m++)
                if (!(m & (4 >> s))) ct(v[m], v[m + (4 >> s)], tw[(16 << s) + ((8 * h + la) << s) + (m >> (3 - s))]);
        vh_wave_sync();
#pragma unroll
        for (int m = 0; m < 8; m++) scr[72 * la + 9 * m + lb] = v[m];
        vh_wave_sync();
#pragma unroll
        for (int m = 0; m < 8; m++) v[m] = scr[9 * lane + m];
#pragma unroll
        for (int s = 0; s < 3; s++)
#pragma unroll
            for (int m = 0; m < 8; m++)
                if (!(m & (4 >> s))) {
                    if (s == 2) v[m + 1] = vh_center(v[m + 1], q, qinv);
                    ct(v[m], v[m + (4 >> s)], tw[(128 << s) + ((64 * h + lane) << s) + (m >> (3 - s))]);
                }
    };
    auto inv9 = [&](double (&v)[8]) {
#pragma unroll
        for (int s = 2; s >= 0; s--)   // stages 9, 8, 7
#pragma unroll
            for (int m = 0; m < 8; m++)
                if (!(m & (4 >> s)))
                    gs(v[m], v[m + (4 >> s)], tw[(128 << s) + ((64 * (2 - h) - lane) << s) - 1 - (m >> (3 - s))], s == 1);
        vh_wave_sync();
#pragma unroll
        for (int m = 0; m < 8; m++) scr[9 * lane + m] = v[m];
        vh_wave_sync();
#pragma unroll
        for (int m = 0; m < 8; m++) v[m] = scr[72 * la + 9 * m + lb];
#pragma unroll
        for (int s = 2; s >= 0; s--)   // stages 6, 5, 4
#pragma unroll
            for (int m = 0; m < 8; m++)
                if (!(m & (4 >> s)))
                    gs(v[m], v[m + (4 >> s)], tw[(16 << s) + ((8 * (2 - h) - la) << s) - 1 - (m >> (3 - s))], s != 1);
        vh_wave_sync();
#pragma unroll
        for (int m = 0; m < 8; m++) scr[72 * la + 8 * m + lb] = v[m];
        vh_wave_sync();
#pragma unroll
        for (int m = 0; m < 8; m++) v[m] = scr[72 * m + lane];
#pragma unroll
        for (int s = 2; s >= 0; s--)   // stages 3, 2, 1
#pragma unroll
            for (int m = 0; m < 8; m++)
                if (!(m & (4 >> s)))
                    gs(v[m], v[m + (4 >> s)], tw[(2 << s) + ((2 - h) << s) - 1 - (m >> (3 - s))], s == 1);
    };

    // Key rows are taken in the order e = i nd + d of the wave's digits: the next words load after the product of
    // the current ones, their row pointers one step earlier, the next exponent one key index earlier.
    const VH_GLOBAL uint64_t *am = vh_global(amounts + (size_t)(live ? k : 0) * P.n);
    uint64_t kw[C][8];
    const uint64_t *kp[C];
    const uint32_t n = (uint32_t)P.n;
    auto key_rows = [&](uint32_t e) {   // the wave's e-th digit over all key indices (the last one past the end)
        e = e < n * ND ? e : n * ND - 1;
        const VH_GLOBAL uint64_t *tab =
            (const VH_GLOBAL uint64_t *)(bkp + ((size_t)(e / ND) * nd + d0 + e % ND) * (C * next) + w);
#pragma unroll
        for (int c = 0; c < C; c++) kp[c] = (const uint64_t *)tab[c * next];
    };
    auto key_words = [&]() {
#pragma unroll
        for (int c = 0; c < C; c++) {
            const VH_GLOBAL uint64_t *kr = vh_global(kp[c]) + BH * h + 8 * lane;
#pragma unroll
            for (int e = 0; e < 4; e++) vh_ld2(kr + 2 * e, kw[c][2 * e], kw[c][2 * e + 1]);
        }
    };
    uint32_t anext = 0;
    if (n) {
        anext = (uint32_t)am[0];
        key_rows(0);
        key_words();
        key_rows(1);
    }
    for (uint32_t i = 0; i < n; i++) {
        const uint32_t a = anext & (2 * BN - 1);
        anext = (uint32_t)am[i + 1 < n ? i + 1 : i];
        if (level) {
            double dg[OC][8];
#pragma unroll
            for (int c = 0; c < OC; c++) {
                const double *row = reg + ((c0 + c) * NJ + jw) * BN;
#pragma unroll
                for (int m = 0; m < 8; m++) {
                    const uint32_t u = (uint32_t)(x0 + 64 * m + 2 * BN - a) & (2 * BN - 1);
                    const double s = row[u & (BN - 1)];
                    double r = (u < BN ? s : -s) - own[c][m];     // in (-2 q, q)
                    r = r < 0.0 ? r + q : r;
                    dg[c][m] = r < 0.0 ? r + q : r;
                }
            }
            __syncthreads();   // every rotated read is done
#pragma unroll
            for (int c = 0; c < OC; c++)
#pragma unroll
                for (int m = 0; m < 8; m++) reg[((c0 + c) * NJ + jw) * BN + x0 + 64 * m] = dg[c][m];
        } else {
            __syncthreads();
        }
        __syncthreads();   // the digits are in place

        double out[C][8];
#pragma unroll
        for (int c = 0; c < C; c++)
#pragma unroll
            for (int m = 0; m < 8; m++) out[c][m] = 0.0;
#pragma unroll 1
        for (int d = 0; d < ND; d++) {
            const double *row = reg + (d0 + d) * BN + lane;
            double v[8];
#pragma unroll
            for (int m = 0; m < 8; m++)
                v[m] = __fma_rn(side, vh_mulmod_tw(row[BH + 64 * m], w1, wq1, q), row[64 * m]);
            fwd9(v);
#pragma unroll
            for (int m = 0; m < 8; m++) {
                const double x = vh_center(v[m], q, qinv);
#pragma unroll
                for (int c = 0; c < C; c++) {
                    const double kk = vh_u2d(kw[c][m]);
                    const double hi = x * kk;
                    const double lo = __fma_rn(x, kk, -hi);
                    const double qt = __fma_rn(x, kk * qinv, VH_MAGIC) - VH_MAGIC;
                    out[c][m] += __fma_rn(-qt, q, hi) + lo;   // |term| <= q + 2^47
                }
            }
            key_words();
            key_rows(i * ND + d + 2);
            if (ND > 4 && d == 3) {
#pragma unroll
                for (int c = 0; c < C; c++)
#pragma unroll
                    for (int m = 0; m < 8; m++) out[c][m] = vh_center(out[c][m], q, qinv);
            }
        }
        if (G == 2) {   // swap partial sums with the other group: keep component g
            double mine[8];
            vh_wave_sync();
#pragma unroll
            for (int m = 0; m < 8; m++) {
                mine[m] = g ? out[C - 1][m] : out[0][m];
                scr[lane + 64 * m] = g ? out[0][m] : out[C - 1][m];
            }
            __syncthreads();   // the digits are read, the partial sums published
            const double *oscr = reg + REG + (((1 - g) * next + w) * 2 + h) * BSCR;
#pragma unroll
            for (int m = 0; m < 8; m++) out[0][m] = mine[m] + oscr[lane + 64 * m];   // <= 6 (q + 2^47)
            __syncthreads();   // the partial sums are read
        } else {
            __syncthreads();   // the digits are read
        }
#pragma unroll
        for (int c = 0; c < OC; c++) {
#pragma unroll
            for (int m = 0; m < 8; m++) out[c][m] = vh_center(out[c][m], q, qinv);
            inv9(out[c]);
            double *dst = c == OC - 1 ? scr : reg + (2 * w + h) * BH;
            if (c == OC - 1) vh_wave_sync();
#pragma unroll
            for (int m = 0; m < 8; m++) dst[lane + 64 * m] = out[c][m];
        }
        __syncthreads();   // every half is published
#pragma unroll
        for (int c = 0; c < OC; c++) {
            const double *src = c == OC - 1 ? pscr : reg + (2 * w + 1 - h) * BH;
            double *t = (c0 + c == C - 1 ? tlast : tfirst) + x0;
#pragma unroll
            for (int m = 0; m < 8; m++) {
                const double p = src[lane + 64 * m];
                const double x = h ? vh_mulmod_tw(out[c][m] - p, w1, wq1, q) : out[c][m] + p;
                if (level) out[c][m] = vh_mulmod_tw(x, P.ninv_inv[w], P.ninv_invq[w], q);
                else t[64 * m] = vh_canon(vh_mulmod_tw(x, L.ninv_d, L.ninv_q, q) + P.hp, q, qinv);
            }
        }
        __syncthreads();   // t of every component is published
        if (level) {
#pragma unroll
            for (int c = 0; c < OC; c++) {
                const double *t = (c0 + c == C - 1 ? tlast : tfirst) + x0;
#pragma unroll
                for (int m = 0; m < 8; m++) {
                    const double y = vh_mulmod_tw(P.hdiv[w] - t[64 * m], P.inv[w], P.invq[w], q);
                    own[c][m] = vh_canon(own[c][m] + out[c][m] + y, q, qinv);
                }
            }
        }
        __syncthreads();   // t is read
        if (level) {
#pragma unroll
            for (int c = 0; c < OC; c++)
#pragma unroll
                for (int m = 0; m < 8; m++) reg[((c0 + c) * NJ + jw) * BN + x0 + 64 * m] = own[c][m];
        }
        __syncthreads();
    }
    if (level && live) {
#pragma unroll
        for (int c = 0; c < OC; c++) {
            VH_GLOBAL uint64_t *dst = vh_global(accp[((size_t)k * C + c0 + c) * NJ + jw]);
#pragma unroll
            for (int m = 0; m < 8; m++) dst[x0 + 64 * m] = vh_d2u(own[c][m]);
        }
    }
}

hipError_t vh_launch_blind_rotate(hipStream_t st, const vh_br_params &P, const vh_limb *limbs, uint64_t *const *accp,
                                  const uint64_t *const *bkp, const uint64_t *amounts, unsigned count, unsigned cus,
                                  const uint64_t *const *tvp, const uint64_t *rot)
{
    if (P.C < 1 || P.C > 2 || P.nJ < 1 || P.nJ > VH_BR_MAXJ || P.next != P.nJ + 1 || P.next > VH_BR_MAXE ||
        P.sp < 0 || P.sp >= P.next || count == 0 || (tvp && !rot))
        return hipErrorInvalidValue;
    // One workgroup fits a CU (two at one component and one level limb).  Up to one accumulator per CU, each takes twice the waves (G = 2):
    // 8 accumulators of n = 630 take 9.0 ms (12.3 ms with G = 1).  Beyond, two accumulators
    // share a workgroup: 300 take 18.5 ms where one per CU would take two rounds of 9.
    const int na = count > cus && P.nJ < 3 ? 2 : 1, g = na == 1 && P.C == 2 && P.nJ < 3 ? 2 : 1;
#define VH_BR(CC, JJ, AA, GG)                                                                               \
    if (P.C == CC && P.nJ == JJ && na == AA && g == GG)                                                    \
        VH_KL((k_blind_rotate<CC, JJ, AA, GG>), dim3((count + AA - 1) / AA), dim3(AA * GG * (JJ + 1) * 128), 0, st, P, \
              limbs, accp, bkp, amounts, tvp, rot, count);
    VH_BR(1, 1, 1, 1) VH_BR(1, 2, 1, 1) VH_BR(1, 3, 1, 1) VH_BR(2, 1, 1, 2) VH_BR(2, 2, 1, 2) VH_BR(2, 3, 1, 1)
    VH_BR(1, 1, 2, 1) VH_BR(1, 2, 2, 1) VH_BR(2, 1, 2, 1) VH_BR(2, 2, 2, 1)
#undef VH_BR
    return hipGetLastError();
}
