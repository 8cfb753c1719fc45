// fa_ks.hip -- fmpz polynomial products beyond the eight-prime capacity, by
// Kronecker substitution onto the integer product (the route the
// reference's callers take when _fmpz_poly_mul_mid_default_mpn_ctx declines:
// fmpz_poly/mul.c:160, _fmpz_poly_mul_KS).
//
// Two routes.  The default packs signed coefficients into s-bit slots with
// borrows and needs one integer product (see the signed-slot kernels
// below).  The other packs without borrows: with a = a+ - a- (the positive
// part and the negated negative part, coefficient by coefficient)
//     a b = 2 (a+ b+ + a- b-) - |a| |b|,
// an identity of polynomials, so it holds coefficient by coefficient.  Each
// of the three products has non-negative coefficients below
// min(an, bn) 2^(|b1|+|b2|) < 2^(s-1) for the slot width
//     s = |b1| + |b2| + bitcount(min(an, bn)) + 1,
// so packing at s bits per coefficient puts every coefficient in its own
// slot with no carry between slots, at three times the product work.
// Packing is a gather per output limb; the combination is one thread per
// output coefficient.
#include <stdio.h>
#include <string.h>

#include "fa_internal.h"
#include "fa_arith.h"
#include "../../include/flint_amd.h"

enum { FA_KS_PLUS = 0, FA_KS_MINUS = 1, FA_KS_ABS = 2 };

// index of the lowest nonzero limb of each w-limb coefficient (w if zero)
__global__ void __launch_bounds__(256) fa_k_ks_low(const uint64_t* __restrict__ a, int w,
                                                   uint64_t n, int32_t* __restrict__ low)
{
    const uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const uint64_t* c = a + i * (uint64_t)w;
    int m = 0;
    while (m < w && c[m] == 0) m++;
    low[i] = m;
}

// limb m of |c| for a w-limb two's complement coefficient c: for c < 0,
// -c = ~c + 1, whose limb m takes the carry iff limbs 0..m-1 of c are zero
FA_DEV uint64_t fa_ks_mag(const uint64_t* c, int w, int m, int neg, int low)
{
    if (m >= w) return 0;
    return neg ? ~c[m] + (m <= low ? 1u : 0u) : c[m];
}

// out[j] = limb j of sum_i part(c_i) 2^(s i), part = c+, c- or |c|
__global__ void __launch_bounds__(256) fa_k_ks_pack(const uint64_t* __restrict__ a, int w,
                                                    uint64_t n, const int32_t* __restrict__ low,
                                                    uint64_t s, int mode,
                                                    uint64_t* __restrict__ out, uint64_t L)
{
    const uint64_t j = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (j >= L) return;
    const uint64_t bit0 = 64 * j;
    uint64_t i0 = bit0 / s;
    uint64_t i1 = (bit0 + 63) / s;
    if (i1 >= n) i1 = n - 1;
    uint64_t acc = 0;
    for (uint64_t i = i0; i <= i1 && i < n; i++) {
        const uint64_t* c = a + i * (uint64_t)w;
        const int neg = (int)(c[w - 1] >> 63);
        if ((mode == FA_KS_PLUS && neg) || (mode == FA_KS_MINUS && !neg)) continue;
        const int lo = low[i];
        const int64_t rel = (int64_t)bit0 - (int64_t)(s * i);   // bit of c at bit0
        if (rel >= 0) {
            if ((uint64_t)rel >= s) continue;
            const int q = (int)(rel >> 6), r = (int)(rel & 63);
            uint64_t v = fa_ks_mag(c, w, q, neg, lo) >> r;
            if (r) v |= fa_ks_mag(c, w, q + 1, neg, lo) << (64 - r);
            acc |= v;
        } else {
            acc |= fa_ks_mag(c, w, 0, neg, lo) << (int)(-rel);
        }
    }
    out[j] = acc;
}

// limb l of slot k (bits [s k, s k + s)) of a product of nP limbs
FA_DEV uint64_t fa_ks_slot(const uint64_t* __restrict__ P, uint64_t nP, uint64_t s, uint64_t k,
                           int l)
{
    const uint64_t lb = 64 * (uint64_t)l;
    if (lb >= s) return 0;
    const uint64_t off = s * k + lb;
    const uint64_t q = off >> 6;
    const int r = (int)(off & 63);
    uint64_t v = q < nP ? P[q] >> r : 0;
    if (r && q + 1 < nP) v |= P[q + 1] << (64 - r);
    if (lb + 64 > s) v &= (UINT64_C(1) << (s - lb)) - 1;
    return v;
}

// z[t] = coefficient zl + t of a b = 2 (P1 + P4) - P5 as zw limbs (two's
// complement), zero past the product's length zn
__global__ void __launch_bounds__(256) fa_k_ks_combine(const uint64_t* __restrict__ P1,
                                                       const uint64_t* __restrict__ P4,
                                                       const uint64_t* __restrict__ P5,
                                                       uint64_t nP, uint64_t s, uint64_t zl,
                                                       uint64_t cnt, uint64_t zn, int zw,
                                                       uint64_t* __restrict__ z)
{
    const uint64_t t = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= cnt) return;
    uint64_t* o = z + t * (uint64_t)zw;
    const uint64_t k = zl + t;
    if (k >= zn) {
        for (int l = 0; l < zw; l++) o[l] = 0;
        return;
    }
    unsigned carry = 0, borrow = 0;
    for (int l = 0; l < zw; l++) {
        const uint64_t e1 = fa_ks_slot(P1, nP, s, k, l);
        const uint64_t e4 = fa_ks_slot(P4, nP, s, k, l);
        const uint64_t e5 = fa_ks_slot(P5, nP, s, k, l);
        // 2 (e1 + e4) + carry, as 64 bits and a carry of at most 3
        const uint64_t h = e1 + e4;
        unsigned c1 = h < e1;
        const uint64_t d = h << 1;
        unsigned c2 = (unsigned)(h >> 63) + 2 * c1;
        const uint64_t sum = d + carry;
        c2 += sum < d;
        carry = c2;
        // minus e5 and the borrow
        const uint64_t r1 = sum - e5;
        unsigned b1 = sum < e5;
        const uint64_t r2 = r1 - borrow;
        b1 += r1 < borrow;
        borrow = b1;
        o[l] = r2;
    }
}

// ---------------------------------------------------------------------------
// Signed slots, one product (the default).  With sigma = +1 or -1 chosen so
// that sigma a has a positive top nonzero coefficient, the packed integer
//     A = sum_i sigma a_i 2^(s i)
// is positive; its base-2^s digits are d_i = (sigma a_i - br_i) mod 2^s with
// the borrow br_0 = 0, br_(i+1) = [sigma a_i - br_i < 0], i.e. generate
// [sigma a_i < 0] and propagate [a_i = 0]: a 1-bit scan over coefficients.
// The product C = A B = sum_k c_k 2^(s k) with |c_k| < 2^(s-1) (the slot
// width above) has base-2^s digits e_k, and
//     c_k = e_k + t_(k-1) - 2^s t_k,  t_k = [e_k + t_(k-1) >= 2^(s-1)].
// t_k is the top bit of e_k: they differ only for e_k = 2^(s-1) - 1 with
// t_(k-1) = 1, which would make |c_k| = 2^(s-1).  (|c_k| <= m 2^(|b1|+|b2|) for
// m terms and m < 2^bitcount(m), so the bound holds for |a_i| = 2^|b1| too.)
// So c_k is the s-bit field e_k + t_(k-1), with t_(k-1) one bit of the product
// and no scan over the slots, read as a signed s-bit number, times sigma_a
// sigma_b.
// ---------------------------------------------------------------------------

typedef __attribute__((address_space(1))) const uint64_t fa_gcw;   // global words

// The flag word of a coefficient: its lowest nonzero limb (KS_ZERO for zero)
// and in bit 30 the borrow into its slot.
#define KS_ZERO 0x3fffffff

// the lowest nonzero limb of a w-limb coefficient whose limb 0 is v0
FA_DEV int ks_low_limb(fa_gcw* c, int w, uint64_t v0)
{
    if (v0) return 0;
    int l = 1;
    while (l < w && c[l] == 0) l++;
    return l < w ? l : KS_ZERO;
}

// the carries into the 64 wave masks of a round (64 positions each, in order)
// as a mask: lane l of every wave reads mask l, whose carry-out depends on its
// carry-in only if it propagates throughout.  *c: the carry into the round, on
// return the one out of it
FA_DEV uint64_t ks_round_carries(const uint64_t* sG, const uint64_t* sP, int lane, uint32_t* c)
{
    const uint64_t g = sG[lane], p = sP[lane];
    uint32_t o, on;
    (void)fa_gp_carries(g, p, 0, &o);
    const uint64_t cin = fa_gp_carries(__ballot(o != 0), __ballot(p == ~UINT64_C(0)), *c, &on);
    *c = on;
    return cin;
}

// one workgroup per operand: the sign sigma of the top nonzero coefficient (+1
// for a zero operand), then the flag words, 4 x 1024 coefficients a round with
// the loads of a round issued together and the borrows from the ballots of its
// waves.  sG, sP: 64 words each.  Bound by the latency of one workgroup's
// loads; a run of coefficients per thread, walked limb by limb, took 159 us for
// the operands of 64 batched products (561 MB packed), the rounds 85.
FA_DEV void ks_sflags_body(const uint64_t* __restrict__ ap, int w, uint64_t n,
                           int32_t* __restrict__ low, int32_t* __restrict__ sig, uint64_t* sG,
                           uint64_t* sP)
{
    fa_gcw* a = (fa_gcw*)ap;
    typedef __attribute__((address_space(1))) int32_t gI;
    gI* lowg = (gI*)low;
    const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
    int negs = 0;
    int64_t last = -1;     // the top nonzero coefficient: above it, limb 0 tells below
    for (int64_t hi = (int64_t)n; hi > 0; hi -= 1024) {
        const int64_t i = hi - 1024 + t;
        bool nz = false, neg = false;
        if (i >= 0) {
            fa_gcw* c = a + (uint64_t)i * w;
            const uint64_t top = c[w - 1];
            neg = top >> 63;
            nz = top != 0 || ks_low_limb(c, w, c[0]) != KS_ZERO;
        }
        const uint64_t NZ = __ballot(nz), NG = __ballot(neg);
        if (lane == 0) {
            sG[wave] = NZ;
            sP[wave] = NG;
        }
        __syncthreads();
        int found = 0;
        for (int v = 15; v >= 0 && !found; v--) {
            if (sG[v]) {
                const int b = 63 - __builtin_clzll(sG[v]);
                negs = (int)((sP[v] >> b) & 1);
                last = hi - 1024 + 64 * v + b;
                found = 1;
            }
        }
        __syncthreads();
        if (found) break;
    }
    if (t == 0) *sig = negs ? -1 : 1;
    uint32_t c = 0;
    for (uint64_t base = 0; base < n; base += 4096) {
        uint64_t v0[4], vt[4];
#pragma unroll
        for (int k = 0; k < 4; k++) {
            const uint64_t i = base + 1024 * k + t;
            fa_gcw* p = a + (i < n ? i : n - 1) * (uint64_t)w;
            v0[k] = p[0];
            vt[k] = p[w - 1];
        }
        int l[4];
        uint64_t G[4], P[4];
#pragma unroll
        for (int k = 0; k < 4; k++) {
            const uint64_t i = base + 1024 * k + t;
            const bool in = i < n;
            l[k] = ks_low_limb(a + (in ? i : n - 1) * (uint64_t)w, (int64_t)i <= last ? w : 1, v0[k]);
            // generate [sigma c < 0], propagate [c = 0]
            G[k] = __ballot(in && l[k] != KS_ZERO && (int)(vt[k] >> 63) != negs);
            P[k] = __ballot(in && l[k] == KS_ZERO);
            if (lane == 0) {
                sG[16 * k + wave] = G[k];
                sP[16 * k + wave] = P[k];
            }
        }
        __syncthreads();
        const uint64_t cw = ks_round_carries(sG, sP, lane, &c);
#pragma unroll
        for (int k = 0; k < 4; k++) {
            uint32_t o;
            const uint64_t cin = fa_gp_carries(G[k], P[k], (uint32_t)(cw >> (16 * k + wave)) & 1, &o);
            const uint64_t i = base + 1024 * k + t;
            if (i < n) lowg[i] = l[k] | (int)((cin >> lane) & 1) << 30;
        }
        __syncthreads();
    }
}

__global__ void __launch_bounds__(1024) fa_k_ks_sflags(const uint64_t* __restrict__ a, int w,
                                                       uint64_t n, int32_t* __restrict__ low,
                                                       int32_t* __restrict__ sig)
{
    __shared__ uint64_t sG[64], sP[64];
    ks_sflags_body(a, w, n, low, sig, sG, sP);
}

// limb m (any m >= 0, sign-extended past w) of v = sigma c - br for a w-limb
// two's complement coefficient c with flag word f; S = 0 for sigma = +1, all
// ones for -1.  c - br subtracts br, -c - br = ~c + 1 - br adds 1 - br, in
// every limb up to the lowest nonzero one (all of them for zero).
FA_DEV uint64_t fa_ks_vlimb(fa_gcw* c, int w, int m, uint64_t S, int f)
{
    uint64_t x = c[m < w ? m : w - 1];
    if (m >= w) x = (uint64_t)((int64_t)x >> 63);
    const int64_t d = (int64_t)(S & 1) - (f >> 30);
    return (x ^ S) + (m <= (f & KS_ZERO) ? (uint64_t)d : 0);
}

// out[j] = limb j of sum_i d_i 2^(s i), d_i = (sigma c_i - br_i) mod 2^s; slots
// of fewer than 64 bits
FA_DEV uint64_t ks_spack_limb(fa_gcw* a, int w, uint64_t n, const int32_t* __restrict__ low,
                              uint64_t S, uint64_t s, uint64_t j)
{
    const uint64_t bit0 = 64 * j;
    // floor(bit0 / s) from the correctly rounded double quotient (both
    // operands below 2^53, so exact as doubles), which is at most one above
    // it: a 64-bit integer division is a long emulated sequence here
    uint64_t i0 = (uint64_t)((double)bit0 / (double)s);
    if (i0 * s > bit0) i0--;
    uint64_t acc = 0;
    for (uint64_t i = i0; i < n && s * i < bit0 + 64; i++) {
        fa_gcw* c = a + i * (uint64_t)w;
        const int f = low[i];
        const int64_t rel = (int64_t)bit0 - (int64_t)(s * i);   // slot bit at bit0
        uint64_t win;
        if (rel >= 0) {
            const int q = (int)(rel >> 6), r = (int)(rel & 63);
            win = fa_ks_vlimb(c, w, q, S, f) >> r;
            if (r) win |= fa_ks_vlimb(c, w, q + 1, S, f) << (64 - r);
        } else {
            win = fa_ks_vlimb(c, w, 0, S, f) << (int)(-rel);
        }
        // keep window positions p with 0 <= rel + p < s
        const int64_t plo = rel < 0 ? -rel : 0;
        const int64_t phi = (int64_t)s - rel < 64 ? (int64_t)s - rel : 64;
        if (phi <= plo) continue;
        uint64_t mask = phi == 64 ? ~UINT64_C(0) : ((UINT64_C(1) << phi) - 1);
        mask &= ~((UINT64_C(1) << plo) - 1);
        acc |= win & mask;
    }
    return acc;
}

// the same for K limbs j0 + 256 k + threadIdx.x of slots of at least 64 bits:
// the window [64 j, 64 j + 64) meets slot i0 = floor(64 j / s) and at most slot
// i0 + 1.  i0 comes from one reciprocal per thread and a correction by one
// (64 j < 2^46: the product of the two roundings is within 2^-11 of the
// quotient); the limbs of i0 are requested for all K windows before any is
// used, slot i0 + 1 is read only where it starts inside the window.  An
// emulated division, the limbs of both slots and their flags for every window
// took 520 us for 64 batched products (561 MB written), this 273.
template <int K>
FA_DEV void ks_spack_wide(uint64_t* v, fa_gcw* a, int w, uint64_t n,
                          const int32_t* __restrict__ lowp, uint64_t S, uint64_t s, uint64_t L,
                          uint64_t j0)
{
    typedef __attribute__((address_space(1))) const int32_t gI;
    gI* low = (gI*)lowp;
    const double inv = 1.0 / (double)s;
    uint64_t i0[K];
    int64_t rel[K];
    uint64_t lo[K], hi[K];
    int f[K];
#pragma unroll
    for (int k = 0; k < K; k++) {
        uint64_t j = j0 + 256 * (uint64_t)k + threadIdx.x;
        if (j >= L) j = L - 1;
        const uint64_t bit0 = 64 * j;
        uint64_t i = (uint64_t)((double)bit0 * inv);
        int64_t d = (int64_t)(bit0 - i * s);
        if (d < 0) {
            i--;
            d += (int64_t)s;
        } else if (d >= (int64_t)s) {
            i++;
            d -= (int64_t)s;
        }
        i0[k] = i;
        rel[k] = d;
    }
#pragma unroll
    for (int k = 0; k < K; k++) {
        const uint64_t i = i0[k] < n ? i0[k] : n - 1;
        const int q = (int)(rel[k] >> 6);
        fa_gcw* c = a + i * (uint64_t)w;
        f[k] = low[i];
        lo[k] = c[q < w ? q : w - 1];
        hi[k] = c[q + 1 < w ? q + 1 : w - 1];
    }
#pragma unroll
    for (int k = 0; k < K; k++) {
        const int q = (int)(rel[k] >> 6), r = (int)(rel[k] & 63);
        const int64_t d = (int64_t)(S & 1) - (f[k] >> 30);
        const int lw = f[k] & KS_ZERO;
        uint64_t x = q < w ? lo[k] : (uint64_t)((int64_t)lo[k] >> 63);
        uint64_t y = q + 1 < w ? hi[k] : (uint64_t)((int64_t)hi[k] >> 63);
        x = (x ^ S) + (q <= lw ? (uint64_t)d : 0);
        y = (y ^ S) + (q + 1 <= lw ? (uint64_t)d : 0);
        uint64_t win = r ? (x >> r) | (y << (64 - r)) : x;
        const uint64_t phi = s - (uint64_t)rel[k];
        if (phi < 64) {
            // positions below phi belong to slot i0, the rest to slot i0 + 1
            win &= (UINT64_C(1) << phi) - 1;
            if (i0[k] + 1 < n)
                win |= fa_ks_vlimb(a + (i0[k] + 1) * (uint64_t)w, w, 0, S, low[i0[k] + 1]) << phi;
        }
        v[k] = i0[k] < n ? win : 0;
    }
}

// packed limbs j0 + 256 k + threadIdx.x (k < K) below L: all computed
// before any is stored, so their loads can be in flight together.  A batch
// takes K = FA_KS_PACK_BLK / 256; one product alone takes K = 1, which
// leaves more waves per CU to hide the loads of a small grid.
template <int K>
FA_DEV void ks_spack_block(const uint64_t* __restrict__ ap, int w, uint64_t n,
                           const int32_t* __restrict__ low, int negs, uint64_t s,
                           uint64_t* __restrict__ out, uint64_t L, uint64_t j0)
{
    typedef __attribute__((address_space(1))) uint64_t gT;
    fa_gcw* a = (fa_gcw*)ap;
    const uint64_t S = negs ? ~UINT64_C(0) : 0;
    uint64_t v[K];
    if (s >= 64) {
        ks_spack_wide<K>(v, a, w, n, low, S, s, L, j0);
    } else {
#pragma unroll
        for (int k = 0; k < K; k++) {
            const uint64_t j = j0 + 256 * (uint64_t)k + threadIdx.x;
            v[k] = j < L ? ks_spack_limb(a, w, n, low, S, s, j) : 0;
        }
    }
#pragma unroll
    for (int k = 0; k < K; k++) {
        const uint64_t j = j0 + 256 * (uint64_t)k + threadIdx.x;
        if (j < L) ((gT*)out)[j] = v[k];
    }
}

__global__ void __launch_bounds__(256) fa_k_ks_spack(const uint64_t* __restrict__ a, int w,
                                                     uint64_t n, const int32_t* __restrict__ low,
                                                     const int32_t* __restrict__ sig, uint64_t s,
                                                     uint64_t* __restrict__ out, uint64_t L)
{
    ks_spack_block<1>(a, w, n, low, *sig < 0, s, out, L, (uint64_t)blockIdx.x * 256);
}

// limbs of each coefficient staged through LDS per step of the unpack
#define FA_KS_UC 16
// the reciprocal divisions of the unpack are exact for divisors below 64
static_assert(FA_KS_UC + 1 < 64, "unpack staging width");

// z[t] = coefficient zl + t: the s-bit field e_k + t_(k-1) read as signed,
// times sigma_a sigma_b, as zw limbs; zero past the product's length zn.
// One workgroup of 256 threads takes t = t0 .. t0 + 255 (those below cnt),
// one coefficient per thread, FA_KS_UC output limbs at a time: the slot's
// limbs are read into LDS and the output limbs written from it as runs of
// consecutive limbs, so neither side accesses memory one limb per
// coefficient at a stride of zw limbs.  buf: 256 * (FA_KS_UC + 1) words.
FA_DEV void ks_unpack_tile(const uint64_t* __restrict__ C, uint64_t nP, uint64_t s,
                           const int32_t* __restrict__ sig, uint64_t zl, uint64_t zn, uint64_t cnt, int zw,
                           uint64_t* __restrict__ z, uint64_t t0, uint64_t* __restrict__ buf)
{
    constexpr int W = FA_KS_UC + 1;
    const int c = threadIdx.x;
    const int nc = (int)(cnt - t0 < 256 ? cnt - t0 : 256);
    const uint64_t k = zl + t0 + (uint64_t)c;
    const bool mine = c < nc;
    const bool live = mine && k < zn;
    const int neg = (sig[0] < 0) != (sig[1] < 0);
    const int r = (int)((s * k) & 63);   // bit offset of the slot in its first limb
    // t_(k-1): the top bit of slot k - 1
    uint64_t carry = 0;
    if (live && k) {
        const uint64_t tb = s * k - 1;
        if (tb >> 6 < nP) carry = (C[tb >> 6] >> (tb & 63)) & 1;
    }
    uint64_t fill = 0;
    uint64_t ncarry = 1;   // two's complement negation: ~v + 1
    for (int lc = 0; lc < zw; lc += FA_KS_UC) {
        const int nl = zw - lc < FA_KS_UC ? zw - lc : FA_KS_UC;
        // limbs lc .. lc + nl of each slot's span (limb lc + nl feeds the
        // shift of limb lc + nl - 1); only those that reach the field
        // i / d for i < 256 d and d <= FA_KS_UC + 1 as (i ceil(2^20 / d)) >> 20:
        // exact (error below 256 d / 2^20 < 1 / d for d < 64) and within 32 bits
        const uint32_t m1 = ((1u << 20) + (uint32_t)nl) / (uint32_t)(nl + 1);
        const uint32_t m0 = ((1u << 20) + (uint32_t)nl - 1) / (uint32_t)nl;
        for (int i = c; i < nc * (nl + 1); i += 256) {
            const int cc = (int)(((uint32_t)i * m1) >> 20);
            const int j = i - cc * (nl + 1);
            const uint64_t kk = zl + t0 + (uint64_t)cc;
            uint64_t v = 0;
            if (kk < zn && 64 * (uint64_t)(lc + j) < s + 64) {
                const uint64_t q = ((s * kk) >> 6) + (uint64_t)(lc + j);
                if (q < nP) v = C[q];
            }
            buf[cc * W + j] = v;
        }
        __syncthreads();
        if (mine) {
            uint64_t* row = buf + c * W;
            for (int j = 0; j < nl; j++) {
                const uint64_t lb = 64 * (uint64_t)(lc + j);
                uint64_t v;
                if (!live) {
                    v = 0;
                } else {
                    if (lb < s) {
                        uint64_t e = row[j] >> r;
                        if (r) e |= row[j + 1] << (64 - r);
                        if (lb + 64 > s) e &= (UINT64_C(1) << (s - lb)) - 1;
                        v = e + carry;
                        carry = (v < carry) ? 1 : 0;
                        if (lb + 64 >= s) {
                            const uint64_t nb = s - lb;   // 1..64 field bits in this limb
                            const uint64_t m = nb == 64 ? ~UINT64_C(0) : ((UINT64_C(1) << nb) - 1);
                            v &= m;
                            fill = ((v >> (nb - 1)) & 1) ? ~UINT64_C(0) : 0;
                            v |= fill & ~m;
                        }
                    } else {
                        v = fill;
                    }
                    if (neg) {
                        v = ~v + ncarry;
                        ncarry = (ncarry && v == 0) ? 1 : 0;
                    }
                }
                row[j] = v;   // limb j + 1 is still the slot's, read next
            }
        }
        __syncthreads();
        for (int i = c; i < nc * nl; i += 256) {
            const int cc = (int)(((uint32_t)i * m0) >> 20);
            const int j = i - cc * nl;
            z[(t0 + (uint64_t)cc) * (uint64_t)zw + (uint64_t)(lc + j)] = buf[cc * W + j];
        }
        __syncthreads();
    }
}

__global__ void __launch_bounds__(256) fa_k_ks_unpack(const uint64_t* __restrict__ C,
                                                      uint64_t nP, uint64_t s,
                                                      const int32_t* __restrict__ sig,
                                                      uint64_t zl, uint64_t cnt, uint64_t zn,
                                                      int zw, uint64_t* __restrict__ z)
{
    __shared__ uint64_t buf[256 * (FA_KS_UC + 1)];
    ks_unpack_tile(C, nP, s, sig, zl, zn, cnt, zw, z, (uint64_t)blockIdx.x * 256, buf);
}

// ---------------------------------------------------------------------------
// batched signed-slot route: every KS product of a batch in one launch per
// step.  Flags take one workgroup per operand; packing and unpacking take work
// items (record | operand << 31 | block of FA_KS_PACK_BLK packed limbs or 256
// output coefficients << 32).
// ---------------------------------------------------------------------------
__global__ void __launch_bounds__(1024) fa_kb_ks_sflags(const fa_bks* __restrict__ R, unsigned nks)
{
    __shared__ uint64_t sG[64], sP[64];
    if (blockIdx.x >= 2 * nks) return;
    const fa_bks& r = R[blockIdx.x >> 1];
    if (blockIdx.x & 1)
        ks_sflags_body(r.b, (int)r.bw, r.bn, r.lowb, r.sig + 1, sG, sP);
    else
        ks_sflags_body(r.a, (int)r.aw, r.an, r.lowa, r.sig, sG, sP);
}

__global__ void __launch_bounds__(256) fa_kb_ks_spack(const fa_bks* __restrict__ R,
                                                      const uint64_t* __restrict__ work,
                                                      unsigned nwork)
{
    if (blockIdx.x >= nwork) return;
    const uint64_t wi = work[blockIdx.x];
    const fa_bks& r = R[(unsigned)(wi & 0x7fffffffu)];
    const int op = (int)((wi >> 31) & 1);
    const uint64_t j0 = (wi >> 32) * FA_KS_PACK_BLK;
    if (op)
        ks_spack_block<FA_KS_PACK_BLK / 256>(r.b, (int)r.bw, r.bn, r.lowb, r.sig[1] < 0, r.s, r.pb, r.Lb, j0);
    else
        ks_spack_block<FA_KS_PACK_BLK / 256>(r.a, (int)r.aw, r.an, r.lowa, r.sig[0] < 0, r.s, r.pa, r.La, j0);
}

__global__ void __launch_bounds__(256) fa_kb_ks_unpack(const fa_bks* __restrict__ R,
                                                       const uint64_t* __restrict__ work,
                                                       unsigned nwork)
{
    __shared__ uint64_t buf[256 * (FA_KS_UC + 1)];
    if (blockIdx.x >= nwork) return;
    const uint64_t wi = work[blockIdx.x];
    const fa_bks& r = R[(unsigned)(wi & 0x7fffffffu)];
    const uint64_t t0 = (wi >> 32) * 256;
    if (t0 < r.cnt) ks_unpack_tile(r.pr, r.nP, r.s, r.sig, r.zl, r.zn, r.cnt, (int)r.zw, r.z, t0, buf);
}

int fa_batch_ks_pre(const fa_bks* R, unsigned nks, const uint64_t* work, unsigned nwork,
                    hipStream_t s)
{
    if (!nks) return FA_OK;
    FA_LAUNCH("fa_kb_ks_sflags", fa_kb_ks_sflags, dim3(2 * nks), dim3(1024), 0, s, R, nks);
    if (nwork)
        FA_LAUNCH("fa_kb_ks_spack", fa_kb_ks_spack, dim3(nwork), dim3(256), 0, s, R, work, nwork);
    return hipGetLastError() == hipSuccess ? FA_OK : fa_set_error(FA_E_HIP, "batch ks pack launch");
}

int fa_batch_ks_post(const fa_bks* R, unsigned nks, const uint64_t* work, unsigned nwork,
                     hipStream_t s)
{
    if (!nks) return FA_OK;
    if (nwork)
        FA_LAUNCH("fa_kb_ks_unpack", fa_kb_ks_unpack, dim3(nwork), dim3(256), 0, s, R, work, nwork);
    return hipGetLastError() == hipSuccess ? FA_OK : fa_set_error(FA_E_HIP, "batch ks unpack launch");
}

static uint64_t cdiv(uint64_t a, uint64_t b) { return (a + b - 1) / b; }
static int bitcount(uint64_t x) { return x ? 64 - __builtin_clzll(x) : 0; }

// slot width for |b1|, |b2| bits and lengths an, bn
uint64_t fa_ks_slot_bits(int64_t b1, int64_t b2, uint64_t an, uint64_t bn)
{
    const uint64_t m = an < bn ? an : bn;
    return (uint64_t)(b1 < 0 ? -b1 : b1) + (uint64_t)(b2 < 0 ? -b2 : b2) + bitcount(m) + 1;
}

// 1: signed slots and one integer product (default); 0: the three products
// of non-negative parts
int fa_ks_variant = 1;
extern "C" FA_API void fa_set_ks_variant(int v) { fa_ks_variant = v ? 1 : 0; }
int fa_ks_current_variant() { return fa_ks_variant; }
int fa_ks_nprod(int variant) { return variant ? 1 : 3; }

// scratch layout of one KS product: the packed operands, the products, the
// low-limb indices (signed slots: the flag words and the two signs)
struct ks_layout {
    uint64_t La, Lb, nP;
    uint64_t* pa[3];
    uint64_t* pb[3];
    uint64_t* pr[3];
    int32_t* lowa;
    int32_t* lowb;
    int32_t* sig;
};

static ks_layout ks_lay(int variant, uint64_t sb, uint64_t an, uint64_t bn, uint64_t* scratch)
{
    ks_layout K;
    memset(&K, 0, sizeof(K));
    const int np = fa_ks_nprod(variant);
    K.La = cdiv(an * sb, 64);
    K.Lb = cdiv(bn * sb, 64);
    K.nP = K.La + K.Lb;
    uint64_t* w = scratch;
    for (int k = 0; k < np; k++) { K.pa[k] = w; w += K.La; }
    for (int k = 0; k < np; k++) { K.pb[k] = w; w += K.Lb; }
    for (int k = 0; k < np; k++) { K.pr[k] = w; w += K.nP; }
    K.lowa = (int32_t*)w;
    K.lowb = K.lowa + an;
    if (variant) K.sig = K.lowb + bn;         // two int32
    return K;
}

// scratch words of a KS product
uint64_t fa_ks_scratch_words_v(int variant, int64_t b1, int64_t b2, uint64_t an, uint64_t bn)
{
    const uint64_t sb = fa_ks_slot_bits(b1, b2, an, bn);
    const uint64_t La = cdiv(an * sb, 64), Lb = cdiv(bn * sb, 64);
    const uint64_t np = (uint64_t)fa_ks_nprod(variant);
    uint64_t w = np * (La + Lb) + np * (La + Lb) + cdiv(an + bn, 2) + 8;
    if (variant) w += 1;
    return w;
}

uint64_t fa_ks_scratch_words(int64_t b1, int64_t b2, uint64_t an, uint64_t bn)
{
    return fa_ks_scratch_words_v(fa_ks_variant, b1, b2, an, bn);
}

// the integer products of a KS product: ptrs[3k .. 3k+2] = {a, b, z} device
// pointers of product k, lens = {La, Lb}; returns the number of products
int fa_ks_products_v(int variant, uint64_t sb, uint64_t an, uint64_t bn, uint64_t* scratch,
                     uint64_t* ptrs[9], uint64_t lens[2])
{
    ks_layout K = ks_lay(variant, sb, an, bn, scratch);
    const int np = fa_ks_nprod(variant);
    for (int k = 0; k < np; k++) {
        ptrs[3 * k] = K.pa[k];
        ptrs[3 * k + 1] = K.pb[k];
        ptrs[3 * k + 2] = K.pr[k];
    }
    lens[0] = K.La;
    lens[1] = K.Lb;
    return np;
}

// the device record of a signed-slot KS product (scratch of
// fa_ks_scratch_words_v(1, ...)); operands and output as the caller's
void fa_ks_record(uint64_t sb, const uint64_t* a, uint64_t aw, uint64_t an, const uint64_t* b,
                  uint64_t bw, uint64_t bn, uint64_t* scratch, uint64_t* z, uint64_t zw,
                  uint64_t zl, uint64_t cnt, fa_bks* r)
{
    ks_layout K = ks_lay(1, sb, an, bn, scratch);
    memset(r, 0, sizeof(*r));
    r->a = a;
    r->b = b;
    r->z = z;
    r->aw = aw;
    r->an = an;
    r->bw = bw;
    r->bn = bn;
    r->s = sb;
    r->La = K.La;
    r->Lb = K.Lb;
    r->nP = K.nP;
    r->zw = zw;
    r->zl = zl;
    r->cnt = cnt;
    r->zn = an + bn - 1;
    r->lowa = K.lowa;
    r->lowb = K.lowb;
    r->sig = K.sig;
    r->pa = K.pa[0];
    r->pb = K.pb[0];
    r->pr = K.pr[0];
}

// packing before the products
int fa_ks_pre_v(int variant, const uint64_t* a, uint64_t aw, uint64_t an, const uint64_t* b,
                uint64_t bw, uint64_t bn, uint64_t sb, uint64_t* scratch, hipStream_t s)
{
    ks_layout K = ks_lay(variant, sb, an, bn, scratch);
    if (variant) {
        FA_LAUNCH("fa_k_ks_sflags", fa_k_ks_sflags, dim3(1), dim3(1024), 0, s, a, (int)aw, an,
                  K.lowa, K.sig);
        FA_LAUNCH("fa_k_ks_sflags", fa_k_ks_sflags, dim3(1), dim3(1024), 0, s, b, (int)bw, bn,
                  K.lowb, K.sig + 1);
        FA_LAUNCH("fa_k_ks_spack", fa_k_ks_spack, dim3((unsigned)cdiv(K.La, 256)), dim3(256), 0, s,
                  a, (int)aw, an, K.lowa, K.sig, sb, K.pa[0], K.La);
        FA_LAUNCH("fa_k_ks_spack", fa_k_ks_spack, dim3((unsigned)cdiv(K.Lb, 256)), dim3(256), 0, s,
                  b, (int)bw, bn, K.lowb, K.sig + 1, sb, K.pb[0], K.Lb);
        return hipGetLastError() == hipSuccess ? FA_OK : fa_set_error(FA_E_HIP, "ks pack launch");
    }
    FA_LAUNCH("fa_k_ks_low", fa_k_ks_low, dim3((unsigned)cdiv(an, 256)), dim3(256), 0, s, a,
              (int)aw, an, K.lowa);
    FA_LAUNCH("fa_k_ks_low", fa_k_ks_low, dim3((unsigned)cdiv(bn, 256)), dim3(256), 0, s, b,
              (int)bw, bn, K.lowb);
    const int modes[3] = {FA_KS_PLUS, FA_KS_MINUS, FA_KS_ABS};
    for (int k = 0; k < 3; k++) {
        FA_LAUNCH("fa_k_ks_pack", fa_k_ks_pack, dim3((unsigned)cdiv(K.La, 256)), dim3(256), 0, s,
                  a, (int)aw, an, K.lowa, sb, modes[k], K.pa[k], K.La);
        FA_LAUNCH("fa_k_ks_pack", fa_k_ks_pack, dim3((unsigned)cdiv(K.Lb, 256)), dim3(256), 0, s,
                  b, (int)bw, bn, K.lowb, sb, modes[k], K.pb[k], K.Lb);
    }
    return hipGetLastError() == hipSuccess ? FA_OK : fa_set_error(FA_E_HIP, "ks pack launch");
}

// recombination after the products
int fa_ks_post_v(int variant, uint64_t sb, uint64_t an, uint64_t bn, uint64_t* scratch,
                 uint64_t* z, uint64_t zw, uint64_t zl, uint64_t cnt, hipStream_t s)
{
    ks_layout K = ks_lay(variant, sb, an, bn, scratch);
    const uint64_t zn = an + bn - 1;
    if (variant) {
        FA_LAUNCH("fa_k_ks_unpack", fa_k_ks_unpack, dim3((unsigned)cdiv(cnt, 256)), dim3(256), 0, s,
                  K.pr[0], K.nP, sb, K.sig, zl, cnt, zn, (int)zw, z);
        return hipGetLastError() == hipSuccess ? FA_OK : fa_set_error(FA_E_HIP, "ks unpack launch");
    }
    FA_LAUNCH("fa_k_ks_combine", fa_k_ks_combine, dim3((unsigned)cdiv(cnt, 256)), dim3(256), 0, s,
              K.pr[0], K.pr[1], K.pr[2], K.nP, sb, zl, cnt, zn, (int)zw, z);
    return hipGetLastError() == hipSuccess ? FA_OK : fa_set_error(FA_E_HIP, "ks combine launch");
}

// device form: a (an x aw), b (bn x bw) resident; scratch of
// fa_ks_scratch_words; enqueued on s
int fa_ks_device(uint64_t* z, uint64_t zw, uint64_t zl, uint64_t cnt, const uint64_t* a,
                 uint64_t aw, uint64_t an, const uint64_t* b, uint64_t bw, uint64_t bn,
                 int64_t b1, int64_t b2, uint64_t* scratch, hipStream_t s)
{
    const int variant = fa_ks_variant;
    const uint64_t sb = fa_ks_slot_bits(b1, b2, an, bn);
    int rc = fa_ks_pre_v(variant, a, aw, an, b, bw, bn, sb, scratch, s);
    if (rc) return rc;
    uint64_t* ptrs[9];
    uint64_t lens[2];
    const int np = fa_ks_products_v(variant, sb, an, bn, scratch, ptrs, lens);
    for (int k = 0; k < np; k++) {
        rc = fa_mpn_mul_device(ptrs[3 * k + 2], ptrs[3 * k], (int64_t)lens[0], ptrs[3 * k + 1],
                               (int64_t)lens[1], s);
        if (rc) return rc;
    }
    return fa_ks_post_v(variant, sb, an, bn, scratch, z, zw, zl, cnt, s);
}

// host-pointer form: the product the reference's caller computes when the
// eight-prime path declines (fmpz_poly/mul.c:160); same output layout as
// fa_fmpz_poly_mul_mid, always computed (returns 1)
extern "C" int fa_fmpz_poly_mul_ks(uint64_t* z, uint64_t zw, int64_t zl, int64_t zh,
                                   const uint64_t* a, uint64_t aw, int64_t an,
                                   const uint64_t* b, uint64_t bw, int64_t bn)
{
    if (an <= 0 || bn <= 0 || !a || !b || aw == 0 || bw == 0 || zw == 0)
        return fa_set_error(FA_E_ARG, "fa_fmpz_poly_mul_ks: bad arguments");
    if (zl < 0 || zl >= zh) return 1;
    if (!z) return fa_set_error(FA_E_ARG, "fa_fmpz_poly_mul_ks: null output");
    fa_thread_state* st = fa_state();
    if (!st) return FA_E_NODEV;
    const int64_t b1 = fa_vec_max_bits(a, aw, an), b2 = fa_vec_max_bits(b, bw, bn);
    const uint64_t cnt = (uint64_t)(zh - zl);
    const uint64_t wa = (uint64_t)an * aw, wb = (uint64_t)bn * bw, wz = cnt * zw;
    const uint64_t ws = fa_ks_scratch_words(b1, b2, (uint64_t)an, (uint64_t)bn);
    // operands, output and KS scratch in the thread's grow-only staging
    // buffer (the integer product inside uses the separate scratch buffer)
    void* hb = nullptr;
    int rc0 = fa_hbuf_reserve(st, (wa + wb + wz + ws) * 8, &hb, st->stream);
    if (rc0) return rc0;
    uint64_t* d = (uint64_t*)hb;
    uint64_t *da = d, *db = d + wa, *dz = db + wb, *dw = dz + wz;
    hipStream_t s = st->stream;
    int rc = FA_OK;
    if (hipMemcpyAsync(da, a, wa * 8, hipMemcpyHostToDevice, s) != hipSuccess ||
        hipMemcpyAsync(db, b, wb * 8, hipMemcpyHostToDevice, s) != hipSuccess)
        rc = fa_set_error(FA_E_HIP, "fa_fmpz_poly_mul_ks: upload");
    if (!rc)
        rc = fa_ks_device(dz, zw, (uint64_t)zl, cnt, da, aw, (uint64_t)an, db, bw, (uint64_t)bn,
                          b1, b2, dw, s);
    if (!rc && fa_download(z, dz, wz * 8, s) != hipSuccess)
        rc = fa_set_error(FA_E_HIP, "fa_fmpz_poly_mul_ks: download");
    if (hipStreamSynchronize(s) != hipSuccess && !rc)
        rc = fa_set_error(FA_E_HIP, "fa_fmpz_poly_mul_ks: %s", hipGetErrorString(hipGetLastError()));
    return rc ? rc : 1;
}
