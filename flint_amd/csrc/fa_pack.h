// fa_pack.h -- operand import: the residue mod p of element x of an
// operand (a bit chunk of a limb array, a u64 coefficient, or a signed
// multi-limb coefficient).
#pragma once

#include "fa_internal.h"
#include "fa_arith.h"

// ------------------------------------------------------------------------
// limb splitting (mpn_mul.c:595-695, slow_mpn_to_fft :422-481)
// ------------------------------------------------------------------------

// 32-bit word of the little-endian limb array starting at byte offset
// `byte` (zero beyond the array)
FA_DEV uint32_t fa_load_u32_at(const uint32_t* __restrict__ w, uint64_t nwords, uint64_t byte)
{
    uint64_t i = byte >> 2;
    int sh = (int)(byte & 3) * 8;
    uint32_t lo = (i < nwords) ? w[i] : 0u;
    if (sh == 0) return lo;
    uint32_t hi = (i + 1 < nwords) ? w[i + 1] : 0u;
    return (lo >> sh) | (hi << (32 - sh));
}

// residue mod p of chunk j = bits [j*bits, (j+1)*bits) of the limb array
// (mpn_mul.c:595-695 splits into 32-bit pieces; here the aligned 64-bit
// words covering the chunk are read and split into 48-bit pieces, exact in
// a double): value = sum_k piece_k 2^(48k), reduced with 2^(48k) mod p.
// Result in [-p/2, p/2], or the plain value when bits <= 48.
FA_DEV uint64_t fa_word(const uint64_t* __restrict__ a, uint64_t n, uint64_t i)
{
    return i < n ? a[i] : 0;
}

FA_DEV double fa_chunk_residue(const uint64_t* __restrict__ limbs, uint64_t nlimbs, int bits,
                               uint64_t j, const double* __restrict__ pow2, double n,
                               double ninv)
{
    const uint64_t bit0 = j * (uint64_t)bits;
    const uint64_t w = bit0 >> 6;
    if (w >= nlimbs) return 0.0;
    const int sh = (int)(bit0 & 63);
    const int span = sh + bits;                  // <= 263 bits: at most five words
    uint64_t v[5];
#pragma unroll
    for (int k = 0; k < 5; k++) v[k] = (64 * k < span) ? fa_word(limbs, nlimbs, w + k) : 0;
    uint64_t u[4];
#pragma unroll
    for (int k = 0; k < 4; k++) {
        u[k] = sh ? ((v[k] >> sh) | (v[k + 1] << (64 - sh))) : v[k];
        if (64 * k >= bits) u[k] = 0;
        else if (64 * (k + 1) > bits) u[k] &= (UINT64_C(1) << (bits - 64 * k)) - 1;
    }
    const uint64_t M48 = (UINT64_C(1) << 48) - 1;
    double p0 = (double)(u[0] & M48);
    if (bits <= 48) return p0;
    double p1 = (double)(((u[0] >> 48) | (u[1] << 16)) & M48);
    double p2 = (double)(((u[1] >> 32) | (u[2] << 32)) & M48);
    double p3 = (double)((u[2] >> 16) & M48);
    double p4 = (double)(u[3] & M48);
    double acc = p0 + fa_mulmod(p1, pow2[1], n, ninv);
    if (bits > 96) acc += fa_mulmod(p2, pow2[2], n, ninv);
    if (bits > 144) acc += fa_mulmod(p3, pow2[3], n, ninv);
    if (bits > 192) acc += fa_mulmod(p4, pow2[4], n, ninv);
    return fa_reduce_pm1n(acc, n, ninv);
}

// the same for bits = 8 own (own <= 25 bytes per chunk): the chunk's bytes
// [own j, own j + own) come from two 16-byte loads at the enclosing 4-byte
// boundary, realigned with v_alignbyte, masked to own bytes and cut into
// 48-bit pieces of 32-bit words.  The result is in (-2n, 2.25n) when
// own <= 18 (at most two products) and in [-n/2, n/2] otherwise -- inside
// the (-3n, 3n) input range of the forward transform.  The last chunks,
// whose 32-byte window reaches past the array, read it word by word.
typedef uint32_t fa_u32x4 __attribute__((ext_vector_type(4)));
typedef fa_u32x4 fa_u32x4_a4 __attribute__((aligned(4)));

FA_DEV double fa_chunk_residue8(const uint64_t* __restrict__ limbs, uint64_t nlimbs, int own,
                                uint64_t j, const double* __restrict__ pow2, double n,
                                double ninv)
{
    const uint64_t B = j * (uint64_t)own;
    const uint64_t nbytes = nlimbs * 8;
    if (B >= nbytes) return 0.0;
    const uint64_t B4 = B & ~UINT64_C(3);
    uint32_t w[8];
    if (B4 + 32 <= nbytes) {
        const fa_u32x4_a4* q = (const fa_u32x4_a4*)((const char*)limbs + B4);
        const fa_u32x4 lo4 = q[0], hi4 = q[1];
        w[0] = lo4.x; w[1] = lo4.y; w[2] = lo4.z; w[3] = lo4.w;
        w[4] = hi4.x; w[5] = hi4.y; w[6] = hi4.z; w[7] = hi4.w;
    } else {
        const uint32_t* q = (const uint32_t*)((const char*)limbs + B4);
#pragma unroll
        for (int m = 0; m < 8; m++) w[m] = (B4 + 4 * m < nbytes) ? q[m] : 0u;
    }
    const uint32_t s = (uint32_t)(B & 3);
    uint32_t c[7];
#pragma unroll
    for (int m = 0; m < 7; m++) {
        c[m] = __builtin_amdgcn_alignbyte(w[m + 1], w[m], s);
        const int vb = own - 4 * m;   // valid bytes of word m
        if (vb < 4) c[m] = (vb <= 0) ? 0u : (c[m] & ((1u << (8 * vb)) - 1u));
    }
    const double T16 = 65536.0, T32 = 4294967296.0;
    double acc = __builtin_fma((double)(c[1] & 0xffffu), T32, (double)c[0]);
    if (own > 6) {
        const double p1 = __builtin_fma((double)c[2], T16, (double)(c[1] >> 16));
        acc += fa_mulmod(p1, pow2[1], n, ninv);
    }
    if (own > 12) {
        const double p2 = __builtin_fma((double)(c[4] & 0xffffu), T32, (double)c[3]);
        acc += fa_mulmod(p2, pow2[2], n, ninv);
    }
    if (own > 18) {
        const double p3 = __builtin_fma((double)c[5], T16, (double)(c[4] >> 16));
        acc += fa_mulmod(p3, pow2[3], n, ninv);
        if (own > 24) acc += fa_mulmod((double)c[6], pow2[4], n, ninv);
        acc = fa_reduce_pm1n(acc, n, ninv);
    }
    return acc;
}

// ------------------------------------------------------------------------
// operand import: the value of element x (coefficient index) of an operand
// ------------------------------------------------------------------------

struct fa_operand {
    int kind;                  // FA_PACK_*
    const uint64_t* src;
    uint64_t n;                // limbs (mpn) or coefficients
    int bits;
    int width;
};

// signed w-limb two's complement coefficient mod p: Horner over the 32-bit
// words from the top, minus 2^(64 w) for a negative coefficient
FA_DEV double fa_coeff_residue_s(const uint64_t* __restrict__ c, int w,
                                 const double* __restrict__ pow2, double n, double ninv)
{
    const uint32_t* u = (const uint32_t*)c;
    const double c32 = pow2[0];
    double r = 0.0, t = 1.0;
    for (int k = 2 * w - 1; k >= 0; k--) {
        r = fa_reduce_pm1n(fa_mulmod(r, c32, n, ninv) + (double)u[k], n, ninv);
        t = fa_reduce_pm1n(fa_mulmod(t, c32, n, ninv), n, ninv);
    }
    if ((int64_t)c[w - 1] < 0) r = fa_reduce_pm1n(r - t, n, ninv);
    return r;
}

FA_DEV double fa_operand_value(const fa_operand& op, uint64_t x,
                               const double* __restrict__ pow2, double n, double ninv)
{
    if (op.kind == FA_PACK_MPN) {
        if ((op.bits & 7) == 0 && op.bits <= 200)
            return fa_chunk_residue8(op.src, op.n, op.bits >> 3, x, pow2, n, ninv);
        return fa_chunk_residue(op.src, op.n, op.bits, x, pow2, n, ninv);
    }
    if (x >= op.n) return 0.0;
    if (op.kind == FA_PACK_U64) {
        uint64_t v = op.src[x];
        double lo = (double)(uint32_t)v, hi = (double)(uint32_t)(v >> 32);
        if (v < (UINT64_C(1) << 50)) return (double)v;
        return fa_reduce_pm1n(lo + fa_mulmod(hi, pow2[0], n, ninv), n, ninv);
    }
    return fa_coeff_residue_s(op.src + x * (uint64_t)op.width, op.width, pow2, n, ninv);
}

// whether an operand has at most len elements (chunks of a limb array,
// coefficients), len a power of two below 2^25
FA_DEV bool fa_operand_fits(const fa_operand& op, uint32_t len)
{
    if (op.kind == FA_PACK_MPN) return 64 * op.n <= (uint64_t)op.bits * len;
    return op.n <= len;
}

// import specialized at compile time (KIND = FA_PACK_*), FA_PACK_ANY
// dispatching on op.kind
template <int KIND>
FA_DEV double fa_operand_value_k(const fa_operand& op, uint64_t x,
                                 const double* __restrict__ pow2, double n, double ninv)
{
    if constexpr (KIND == FA_PACK_MPN8) {
        return fa_chunk_residue8(op.src, op.n, op.bits >> 3, x, pow2, n, ninv);
    } else if constexpr (KIND == FA_PACK_MPN) {
        return fa_chunk_residue(op.src, op.n, op.bits, x, pow2, n, ninv);
    } else if constexpr (KIND == FA_PACK_U64) {
        if (x >= op.n) return 0.0;
        uint64_t v = op.src[x];
        double lo = (double)(uint32_t)v, hi = (double)(uint32_t)(v >> 32);
        if (v < (UINT64_C(1) << 50)) return (double)v;
        return fa_reduce_pm1n(lo + fa_mulmod(hi, pow2[0], n, ninv), n, ninv);
    } else if constexpr (KIND == FA_PACK_S64W) {
        if (x >= op.n) return 0.0;
        return fa_coeff_residue_s(op.src + x * (uint64_t)op.width, op.width, pow2, n, ninv);
    } else {
        return fa_operand_value(op, x, pow2, n, ninv);
    }
}

// ------------------------------------------------------------------------
// column import: elements e0 + k step (k < NB) of an operand, e < 2^24.  All
// loads of a batch are issued before the arithmetic; a batch that lies inside
// the operand for the whole wave is read without checks, one that lies past
// its end for the whole wave is zero.  Values are below 2.75 n in size, which
// the first stage of the column transforms allows for.
// ------------------------------------------------------------------------

// byte-aligned chunks: fa_chunk_residue8 for a batch.  A chunk of own bytes
// is cut into ceil(own / 6) pieces of 48 bits; the width is uniform, so the
// higher pieces are skipped by scalar branches.
template <int NB, int OWN>
FA_DEV void fa_import_mpn8(double* x, const fa_operand& op, uint32_t e0, uint32_t step,
                           const double* __restrict__ pow2, double n, double ninv)
{
    const uint32_t own = OWN ? OWN : (uint32_t)op.bits >> 3;
    const char* base = (const char*)op.src;
    const uint32_t nbytes = op.n < (UINT64_C(1) << 29) ? (uint32_t)op.n * 8u : 0xfffffff8u;
    const uint32_t B0 = e0 * own, bstep = step * own;
    if (!__any(B0 < nbytes)) {
#pragma unroll
        for (int i = 0; i < NB; i++) x[i] = 0.0;
        return;
    }
    // 32-byte windows at the enclosing 4-byte boundary.  Lanes past the end
    // read the operand's last window instead and are cleared below; chunks
    // that straddle the end (the last one or two of an operand) send their
    // wave to word by word loads.
    uint32_t c[NB][7];
    const bool inside = __all(((B0 + (NB - 1) * bstep) & ~3u) + 32u <= nbytes);
    bool edge = nbytes < 32u;
    if (!inside) {
#pragma unroll
        for (int i = 0; i < NB; i++) {
            const uint32_t B = B0 + i * bstep;
            edge |= B < nbytes && (B & ~3u) + 32u > nbytes;
        }
    }
    if (inside || !__any(edge)) {
#pragma unroll
        for (int i = 0; i < NB; i++) {
            const uint32_t B4 = (B0 + i * bstep) & ~3u;
            const uint32_t at = B4 < nbytes - 32u ? B4 : nbytes - 32u;
            const fa_u32x4 lo4 = fa_ld<fa_u32x4_a4>(base, at);
            fa_u32x4 hi4 = {0, 0, 0, 0};
            if (own > 13) hi4 = fa_ld<fa_u32x4_a4>(base + 16, at);
            const uint32_t w[8] = {lo4.x, lo4.y, lo4.z, lo4.w, hi4.x, hi4.y, hi4.z, hi4.w};
            const uint32_t s = (B0 + i * bstep) & 3u;
#pragma unroll
            for (int m = 0; m < 7; m++) c[i][m] = __builtin_amdgcn_alignbyte(w[m + 1], w[m], s);
        }
    } else {
#pragma unroll
        for (int i = 0; i < NB; i++) {
            const uint32_t B4 = (B0 + i * bstep) & ~3u;
            uint32_t w[8];
#pragma unroll
            for (uint32_t m = 0; m < 8; m++) {
                const uint32_t at = B4 + 4 * m;
                const uint32_t v = fa_ld<uint32_t>(base, at < nbytes ? at : 0u);
                w[m] = at < nbytes ? v : 0u;
            }
            const uint32_t s = (B0 + i * bstep) & 3u;
#pragma unroll
            for (int m = 0; m < 7; m++) c[i][m] = __builtin_amdgcn_alignbyte(w[m + 1], w[m], s);
        }
    }
#pragma unroll
    for (int m = 0; m < 7; m++) {
        // bytes of word m that belong to the chunk
        const uint32_t mk = own >= 4u * m + 4 ? 0xffffffffu
                            : own <= 4u * m ? 0u : (1u << (8 * (own - 4u * m))) - 1u;
#pragma unroll
        for (int i = 0; i < NB; i++) c[i][m] &= mk;
    }
    const double T16 = 65536.0, T32 = 4294967296.0;
#pragma unroll
    for (int i = 0; i < NB; i++)
        x[i] = __builtin_fma((double)(c[i][1] & 0xffffu), T32, (double)c[i][0]);
    if (own > 6) {
#pragma unroll
        for (int i = 0; i < NB; i++) {
            const double p1 = __builtin_fma((double)c[i][2], T16, (double)(c[i][1] >> 16));
            x[i] += fa_mulmod(p1, pow2[1], n, ninv);
        }
    }
    if (own > 12) {
#pragma unroll
        for (int i = 0; i < NB; i++) {
            const double p2 = __builtin_fma((double)(c[i][4] & 0xffffu), T32, (double)c[i][3]);
            x[i] += fa_mulmod(p2, pow2[2], n, ninv);
        }
    }
    if (own > 18) {
#pragma unroll
        for (int i = 0; i < NB; i++) {
            const double p3 = __builtin_fma((double)c[i][5], T16, (double)(c[i][4] >> 16));
            x[i] += fa_mulmod(p3, pow2[3], n, ninv);
        }
        if (own > 24) {
#pragma unroll
            for (int i = 0; i < NB; i++)
                x[i] += fa_mulmod((double)c[i][6], pow2[4], n, ninv);
        }
    }
    if (!inside) {
#pragma unroll
        for (int i = 0; i < NB; i++)
            if (B0 + i * bstep >= nbytes) x[i] = 0.0;
    }
}

// u64 coefficients: v = lo + 2^32 hi as a double when the whole wave's values
// are below 2^50, else lo + (2^32 hi mod n)
template <int NB>
FA_DEV void fa_import_u64(double* x, const fa_operand& op, uint32_t e0, uint32_t step,
                          const double* __restrict__ pow2, double n, double ninv)
{
    const uint32_t len = op.n < (UINT64_C(1) << 31) ? (uint32_t)op.n : 1u << 31;
    if (!__any(e0 < len)) {
#pragma unroll
        for (int i = 0; i < NB; i++) x[i] = 0.0;
        return;
    }
    uint32_t lo[NB], hi[NB], top = 0;
#pragma unroll
    for (int i = 0; i < NB; i++) {
        const uint32_t e = e0 + i * step;
        const uint64_t v = fa_ld<uint64_t>(op.src, (e < len ? e : 0u) * 8u);
        lo[i] = e < len ? (uint32_t)v : 0u;
        hi[i] = e < len ? (uint32_t)(v >> 32) : 0u;
        top |= hi[i];
    }
    if (__any(top >> 18)) {
#pragma unroll
        for (int i = 0; i < NB; i++)
            x[i] = fa_mulmod((double)hi[i], pow2[0], n, ninv) + (double)lo[i];
    } else {
#pragma unroll
        for (int i = 0; i < NB; i++)
            x[i] = __builtin_fma((double)hi[i], 4294967296.0, (double)lo[i]);
    }
}

// two's complement coefficients of w limbs: Horner over the 32-bit words from
// the top one, which is read as signed
template <int NB>
FA_DEV void fa_import_s64w(double* x, const fa_operand& op, uint32_t e0, uint32_t step,
                           const double* __restrict__ pow2, double n, double ninv)
{
    const uint32_t len = op.n < (UINT64_C(1) << 31) ? (uint32_t)op.n : 1u << 31;
    const int w = op.width;
    if (!__any(e0 < len)) {
#pragma unroll
        for (int i = 0; i < NB; i++) x[i] = 0.0;
        return;
    }
    const double c32 = pow2[0];
    typedef __attribute__((address_space(1))) uint64_t gT;
    const gT* p[NB];
#pragma unroll
    for (int i = 0; i < NB; i++) {
        const uint32_t e = e0 + i * step;
        p[i] = (const gT*)op.src + (uint64_t)(e < len ? e : 0u) * (uint64_t)w;
        const uint64_t v = p[i][w - 1];
        x[i] = fa_mulmod((double)(int32_t)(v >> 32), c32, n, ninv) + (double)(uint32_t)v;
    }
    for (int l = w - 2; l >= 0; l--) {
        uint64_t v[NB];
#pragma unroll
        for (int i = 0; i < NB; i++) v[i] = p[i][l];
#pragma unroll
        for (int i = 0; i < NB; i++) {
            x[i] = fa_mulmod(x[i], c32, n, ninv) + (double)(uint32_t)(v[i] >> 32);
            x[i] = fa_mulmod(x[i], c32, n, ninv) + (double)(uint32_t)v[i];
        }
    }
#pragma unroll
    for (int i = 0; i < NB; i++)
        if (e0 + i * step >= len) x[i] = 0.0;
}

// elements e0 + k step, k < NEL (a multiple of the batch, or less than one)
template <int NEL, int KIND, int OWN = 0>
FA_DEV void fa_import_column(double* x, const fa_operand& op, uint32_t e0, uint32_t step,
                             const double* __restrict__ pow2, double n, double ninv)
{
    if constexpr (KIND == FA_PACK_MPN8 || KIND == FA_PACK_U64 || KIND == FA_PACK_S64W) {
        constexpr int NB = KIND == FA_PACK_U64 ? (NEL < 8 ? NEL : 8) : (NEL < 4 ? NEL : 4);
#pragma unroll
        for (int k = 0; k < NEL; k += NB) {
            const uint32_t e = e0 + (uint32_t)k * step;
            if constexpr (KIND == FA_PACK_MPN8)
                fa_import_mpn8<NB, OWN>(x + k, op, e, step, pow2, n, ninv);
            else if constexpr (KIND == FA_PACK_U64)
                fa_import_u64<NB>(x + k, op, e, step, pow2, n, ninv);
            else
                fa_import_s64w<NB>(x + k, op, e, step, pow2, n, ninv);
        }
    } else {
#pragma unroll
        for (int k = 0; k < NEL; k++)
            x[k] = fa_operand_value(op, e0 + (uint32_t)k * step, pow2, n, ninv);
    }
}

// the specialization a pair of operands can share
static inline int fa_pack_kind(const fa_operand& a, const fa_operand& b)
{
    if (a.kind != b.kind) return FA_PACK_ANY;
    if (a.kind == FA_PACK_MPN)
        return (a.bits == b.bits && (a.bits & 7) == 0 && a.bits <= 200) ? FA_PACK_MPN8
                                                                         : FA_PACK_MPN;
    return a.kind;
}
