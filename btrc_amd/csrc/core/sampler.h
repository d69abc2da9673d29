// The two samplers of the wavefront path:
//  * Halton with per-digit Owen scrambling and pixel stratification,
//    restating HaltonSampler (builtin/sampler/halton.cpp:39-133) and the
//    low-discrepancy helpers it calls (utils/low_discrepancy.cpp:10-110,
//    after pbrt-v4); every number of a path is a pure function of (pixel,
//    sample index, dimension);
//  * the independent sampler the reference's wavefront tracer uses by
//    default (renderer/wavefront/common.h:37, sampler/independent.cpp:6-25):
//    one PCG32 stream per pixel seeded by MurmurHash64A of the pixel
//    coordinates, advanced by 65536 numbers per sample index.
#pragma once

#include "vecmath.h"

namespace btrc {

constexpr int PRIME_TABLE_SIZE = 1000; // utils/prime.h:9
constexpr int MAX_HALTON_RESOLUTION = 128; // halton.cpp:9

// The first PRIME_TABLE_SIZE primes (utils/prime.cpp), produced by trial
// division at compile time.
struct PrimeTable
{
    int p[PRIME_TABLE_SIZE];
};

constexpr PrimeTable make_prime_table()
{
    PrimeTable t{};
    int n = 0;
    for(int c = 2; n < PRIME_TABLE_SIZE; ++c)
    {
        bool is_prime = true;
        for(int d = 2; d * d <= c; ++d)
        {
            if(c % d == 0)
            {
                is_prime = false;
                break;
            }
        }
        if(is_prime)
            t.p[n++] = c;
    }
    return t;
}

// pbrt-v4 MixBits, low_discrepancy.cpp:49-57
BTRC_HD uint64_t mix_bits(uint64_t v)
{
    v = v ^ (v >> 31);
    v = v * 0x7fb5d329728ea185ull;
    v = v ^ (v >> 27);
    v = v * 0x81dadef4bc2dd44dull;
    v = v ^ (v >> 33);
    return v;
}

// Kensler's hashed permutation, low_discrepancy.cpp:12-45
// the mask Kensler's permutation works in: l - 1 with every lower bit set
BTRC_HD uint32_t permutation_mask(uint32_t l)
{
    uint32_t w = l - 1;
    w = w | (w >> 1);
    w = w | (w >> 2);
    w = w | (w >> 4);
    w = w | (w >> 8);
    w = w | (w >> 16);
    return w;
}

BTRC_HD uint32_t mulhi32(uint32_t a, uint32_t b)
{
#ifdef __HIP_DEVICE_COMPILE__
    return __umulhi(a, b);
#else
    return (uint32_t)(((uint64_t)a * (uint64_t)b) >> 32);
#endif
}

// x mod l from m = floor((2^32 - 1) / l): mulhi(x, m) > x / l - 1, so one
// correction step gives the exact remainder
BTRC_HD uint32_t mod_recip(uint32_t x, uint32_t l, uint32_t m)
{
    uint32_t r = x - mulhi32(x, m) * l;
    if(r >= l)
        r = r - l;
    return r;
}

// Kensler's permutation of i over [0, l) with w = permutation_mask(l) and
// m = floor((2^32 - 1) / l)
BTRC_HD uint32_t permutation_element_masked(uint32_t i, uint32_t l, uint32_t w, uint32_t m, uint32_t p)
{
    for(;;)
    {
        i = i ^ p;
        i = i * 0xe170893du;
        i = i ^ (p >> 16);
        i = i ^ ((i & w) >> 4);
        i = i ^ (p >> 8);
        i = i * 0x0929eb3fu;
        i = i ^ (p >> 23);
        i = i ^ ((i & w) >> 1);
        i = i * (1u | p >> 27);
        i = i * 0x6935fa69u;
        i = i ^ ((i & w) >> 11);
        i = i * 0x74dcb303u;
        i = i ^ ((i & w) >> 2);
        i = i * 0x9e501cc3u;
        i = i ^ ((i & w) >> 2);
        i = i * 0xc860a3dfu;
        i = i & w;
        i = i ^ (i >> 5);
        if(i < l)
            break;
    }
    return mod_recip(i + p, l, m);
}

// Quotient and remainder of a by a small base with m = floor((2^32 - 1) /
// base): mulhi(a, m) > a / base - 1, so one correction step gives the exact
// quotient.
BTRC_HD void divmod_recip(uint32_t a, uint32_t base, uint32_t m, uint32_t *q, uint32_t *r)
{
    uint32_t q32 = mulhi32(a, m);
    uint32_t r32 = a - q32 * base;
    if(r32 >= base)
    {
        q32 = q32 + 1;
        r32 = r32 - base;
    }
    *q = q32;
    *r = r32;
}

// owen_scrambled_radical_inverse, low_discrepancy.cpp:83-101, for any a. The
// tracer's stages use halton_value below (a < 2^32, the same numbers).
BTRC_HD float owen_scrambled_radical_inverse(uint32_t base, uint64_t a, uint64_t hash)
{
    const float inv_base = 1.0f / (float)base;
    const uint32_t m = 0xffffffffu / base;
    const uint32_t w = permutation_mask(base);
    float inv_base_m = 1.0f;
    uint64_t reversed_digits = 0;
    while(1.0f - inv_base_m < 1.0f)
    {
        const uint64_t next = a / base;
        const uint32_t digit = (uint32_t)(a - next * base);
        const uint32_t digit_hash = (uint32_t)mix_bits(hash ^ reversed_digits);
        reversed_digits = reversed_digits * base + permutation_element_masked(digit, base, w, m, digit_hash);
        inv_base_m = inv_base_m * inv_base;
        a = next;
    }
    return fmin_(inv_base_m * (float)reversed_digits, 0x1.fffffep-1f);
}

// A dimension of the sampler as the tracer's stages read it (two 16-byte
// loads): the constants of its digit loop, and its first-digit table. The
// first K scrambled digits of a depend only on a mod base^K, so a table of
// base^K reversed K-digit strings (HALTON_TABLE_SPAN bounds base^K) replaces
// K steps of the loop; the rest of the digits continue from there.
struct alignas(16) HaltonDim
{
    uint32_t base;          // the dimension's prime | digits after the table << 16 | K << 20 | bits of its permutation << 28
    uint32_t recip;         // floor((2^32 - 1) / prime)
    uint32_t hash_lo, hash_hi; // mix_bits(1 + (dim << 4))
    uint32_t first;         // the table's first value
    uint32_t span;          // base^K
    uint32_t span_recip;    // floor((2^32 - 1) / span)
    float scale;            // 1 / base^digits, rounded as the digit loop rounds it
};

// Up to 2^16 entries per dimension: K = 6 for base 5, 4 for 13, 3 to 37, 2 to
// 251, 1 beyond; 5.0 million 16-bit values in all, most of a path's
// dimensions in the first megabytes.
constexpr uint32_t HALTON_TABLE_SPAN = 65536;

struct HaltonTables
{
    const uint16_t *values; // all dimensions' tables
    const HaltonDim *dims;  // PRIME_TABLE_SIZE entries
};

// one dimension's record; its table starts at `first`
BTRC_HD HaltonDim halton_dim(uint32_t base, uint32_t dim, uint32_t first)
{
    HaltonDim d;
    uint32_t span = 1, k = 0, digits = 0, bits = 0;
    while((uint64_t)span * base <= HALTON_TABLE_SPAN)
    {
        span *= base;
        ++k;
    }
    const float inv_base = 1.0f / (float)base;
    d.scale = 1.0f;
    for(; 1.0f - d.scale < 1.0f; ++digits)
        d.scale = d.scale * inv_base;
    while((permutation_mask(base) >> bits) != 0)
        ++bits;
    const uint64_t hash = mix_bits((uint64_t)(1u + (dim << 4)));
    d.base = base | ((digits - k) << 16) | (k << 20) | (bits << 28);
    d.recip = 0xffffffffu / base;
    d.hash_lo = (uint32_t)hash;
    d.hash_hi = (uint32_t)(hash >> 32);
    d.first = first;
    d.span = span;
    d.span_recip = 0xffffffffu / span;
    return d;
}

// product modulo 2^24 (its upper bits are arbitrary): 24-bit multiplies issue
// at the full rate on gfx950, 32-bit ones at a quarter of it
BTRC_HD uint32_t mul24(uint32_t a, uint32_t b)
{
#ifdef __HIP_DEVICE_COMPILE__
    return __umul24(a, b);
#else
    return (a & 0xffffffu) * (b & 0xffffffu);
#endif
}

// bits [at, at + n) of x, n >= 0 and below 32
BTRC_HD uint32_t bit_field(uint32_t x, uint32_t at, uint32_t n)
{
#ifdef __HIP_DEVICE_COMPILE__
    return __builtin_amdgcn_ubfe(x, at, n);
#else
    return (x >> at) & ((1u << n) - 1u);
#endif
}

// Digits of the scrambled radical inverse after the first ones: `n` lowest
// digits of a, each permuted by the hash of the digits reversed so far and
// appended to `reversed` (below 2^32 before every step: the loop ends once
// base^digits reaches 2^25). Kensler's permutation as in
// permutation_element_masked, restricted to what its result depends on: the
// right shifts take bits below `bits` only (the base's width, at most 13), so
// every product is needed modulo 2^bits alone and 24-bit multiplies do. Seven
// quarter-rate products a digit become full-rate ones.
BTRC_HD uint64_t halton_digits(const HaltonDim &d, uint32_t n, uint32_t a, uint32_t reversed)
{
    const uint32_t base = d.base & 0xffffu, bits = d.base >> 28;
    const uint32_t b1 = bits - 1, b2 = bits > 2 ? bits - 2 : 0, b4 = bits > 4 ? bits - 4 : 0,
                   b11 = bits > 11 ? bits - 11 : 0;
    const uint64_t hash = (uint64_t)d.hash_lo | ((uint64_t)d.hash_hi << 32);
    uint64_t rev = reversed;
    for(uint32_t k = 0; k < n; ++k)
    {
        // quotient and digit: the remainder before its correction is below
        // 2 base, so it is exact modulo 2^24
        uint32_t q = mulhi32(a, d.recip);
        uint32_t i = (a - mul24(q, base)) & 0xffffffu;
        if(i >= base)
        {
            i = i - base;
            q = q + 1;
        }
        a = q;
        const uint32_t p = (uint32_t)mix_bits(hash ^ rev);
        const uint32_t p8 = p >> 8, p16 = p >> 16, p23 = p >> 23;
        const uint32_t m27 = mul24(1u | p >> 27, 0x35fa69u);
        do
        {
            i = i ^ p;
            i = mul24(i, 0x70893du);
            i = i ^ p16;
            i = i ^ bit_field(i, 4, b4) ^ p8;
            i = mul24(i, 0x29eb3fu);
            i = i ^ p23;
            i = i ^ bit_field(i, 1, b1);
            i = mul24(i, m27);
            i = i ^ bit_field(i, 11, b11);
            i = mul24(i, 0xdcb303u);
            i = i ^ bit_field(i, 2, b2);
            i = mul24(i, 0x501cc3u);
            i = i ^ bit_field(i, 2, b2);
            i = mul24(i, 0x60a3dfu);
            i = bit_field(i, 0, bits);
            i = i ^ (i >> 5);
        } while(i >= base);
        // (i + p) mod base, again exact modulo 2^24 before the correction
        const uint32_t x = i + p;
        i = (x - mul24(mulhi32(x, d.recip), base)) & 0xffffffu;
        if(i >= base)
            i = i - base;
        rev = (uint64_t)(uint32_t)rev * base + i;
    }
    return rev;
}

// sample_halton (halton.cpp:39-44) of an index below 2^32 in two steps, so
// that the table's load can be in flight while another dimension's digits
// are computed: bit for bit owen_scrambled_radical_inverse
struct HaltonDraw
{
    HaltonDim dim;
    uint32_t high;     // index / span
    uint32_t reversed; // the table's digits
};

BTRC_HD HaltonDraw halton_begin(const HaltonTables &tab, uint32_t dim, uint32_t index)
{
    HaltonDraw w;
    w.dim = tab.dims[dim];
    uint32_t low;
    divmod_recip(index, w.dim.span, w.dim.span_recip, &w.high, &low);
    w.reversed = tab.values[w.dim.first + low];
    return w;
}

BTRC_HD float halton_end(const HaltonDraw &w)
{
    const uint64_t rev = halton_digits(w.dim, (w.dim.base >> 16) & 0xfu, w.high, w.reversed);
    return fmin_(w.dim.scale * (float)rev, 0x1.fffffep-1f);
}

BTRC_HD float halton_value(const HaltonTables &tab, uint32_t dim, uint32_t index)
{
    return halton_end(halton_begin(tab, dim, index));
}

// the same without the table
BTRC_HD float halton_value_digits(const HaltonTables &tab, uint32_t dim, uint32_t index)
{
    const HaltonDim d = tab.dims[dim];
    const uint64_t rev = halton_digits(d, ((d.base >> 16) & 0xfu) + ((d.base >> 20) & 0x1fu), index, 0);
    return fmin_(d.scale * (float)rev, 0x1.fffffep-1f);
}

// one entry of dimension d's table: the reversed digits of r < span
BTRC_HD uint16_t halton_table_entry(const HaltonDim &d, uint32_t r)
{
    return (uint16_t)halton_digits(d, (d.base >> 20) & 0x1fu, r, 0);
}

// Per-film constants of the Halton sampler (initialize_consts, halton.cpp:118-133)
struct HaltonConsts
{
    int32_t base_scales[2];
    int32_t base_exponents[2];
    int32_t mult_inverse[2];
    uint32_t offset_scale[2]; // (stride / base_scales[i]) * mult_inverse[i] mod stride
    uint32_t stride;          // base_scales[0] * base_scales[1], at most 128 * 243
};

struct HaltonState
{
    uint32_t dimension;
    uint64_t index;
};

// halton.cpp:39-44 (sample_halton)
BTRC_HD float sample_halton(const int *primes, uint32_t dim, uint64_t halton_index)
{
    return owen_scrambled_radical_inverse((uint32_t)primes[dim], halton_index,
                                          mix_bits((uint64_t)(1u + (dim << 4))));
}

// HaltonSampler(res, pixel, sample_index), halton.cpp:48-66. The pixel's
// offset fits 32 bits: each inverse is below its scale (at most 243), each
// offset_scale below the stride (at most 31,104).
BTRC_HD HaltonState halton_start(const HaltonConsts &hc, uint32_t px, uint32_t py, int32_t sample_index)
{
    HaltonState st;
    st.index = 0;
    if(hc.stride > 1)
    {
        // inverse_radical_inverse (low_discrepancy.cpp:103-114) in bases 2 and 3
        uint32_t x = px % MAX_HALTON_RESOLUTION, y = py % MAX_HALTON_RESOLUTION, ix = 0, iy = 0;
        for(int i = 0; i < hc.base_exponents[0]; ++i)
        {
            ix = ix * 2 + (x & 1u);
            x = x >> 1;
        }
        for(int i = 0; i < hc.base_exponents[1]; ++i)
        {
            iy = iy * 3 + y % 3;
            y = y / 3;
        }
        st.index = (ix * hc.offset_scale[0] + iy * hc.offset_scale[1]) % hc.stride;
    }
    st.index = st.index + (uint64_t)(int64_t)(int32_t)((uint32_t)sample_index * hc.stride);
    st.dimension = 2; // halton.cpp:64-65
    return st;
}

// The dimension where a draw of n numbers (get1d, get2d, get3d,
// halton.cpp:80-116) starts: back to 2 when it would pass the prime table
BTRC_HD uint32_t halton_wrap(uint32_t dim, uint32_t n)
{
    return dim + n > (uint32_t)PRIME_TABLE_SIZE ? 2u : dim;
}

// ---- independent sampler

// MurmurHash64A (Austin Appleby, public domain; the form of utils/hash.h:12-71)
// of the 8-byte key (x, y) as hash::hash(pixel.x, pixel.y) lays it out
// (two little-endian uint32, seed 0): one whole block, no tail bytes.
BTRC_HD uint64_t murmur_hash_pixel(uint32_t x, uint32_t y)
{
    const uint64_t m = 0xc6a4a7935bd1e995ull;
    uint64_t h = 8ull * m;
    uint64_t k = (uint64_t)x | ((uint64_t)y << 32);
    k = k * m;
    k = k ^ (k >> 47);
    k = k * m;
    h = (h ^ k) * m;
    h = h ^ (h >> 47);
    h = h * m;
    h = h ^ (h >> 47);
    return h;
}

// PCG32 (O'Neill, "PCG: A Family of Simple Fast Space-Efficient Statistically
// Good Algorithms for Random Number Generation", 2014): 64-bit LCG state,
// XSH-RR output. Seeding by stream index as pbrt-v4's RNG(seq_index).
struct Pcg32
{
    uint64_t state;
    uint64_t inc;
};

constexpr uint64_t PCG32_MULT = 0x5851f42d4c957f2dull;

BTRC_HD uint32_t pcg32_next(Pcg32 &r)
{
    const uint64_t old = r.state;
    r.state = old * PCG32_MULT + r.inc;
    const uint32_t xs = (uint32_t)(((old >> 18) ^ old) >> 27);
    const uint32_t rot = (uint32_t)(old >> 59);
    return (xs >> rot) | (xs << ((0u - rot) & 31u));
}

// stream `seq`, starting offset `offset` (pcg32_srandom_r)
BTRC_HD Pcg32 pcg32_seed(uint64_t seq, uint64_t offset)
{
    Pcg32 r;
    r.state = 0;
    r.inc = (seq << 1) | 1ull;
    (void)pcg32_next(r);
    r.state = r.state + offset;
    (void)pcg32_next(r);
    return r;
}

// jump ahead by delta numbers in O(log delta) (Brown, "Random Number
// Generation with Arbitrary Strides", 1994)
BTRC_HD void pcg32_advance(Pcg32 &r, uint64_t delta)
{
    uint64_t cur_mult = PCG32_MULT, cur_plus = r.inc;
    uint64_t acc_mult = 1, acc_plus = 0;
    while(delta > 0)
    {
        if(delta & 1ull)
        {
            acc_mult = acc_mult * cur_mult;
            acc_plus = acc_plus * cur_mult + cur_plus;
        }
        cur_plus = (cur_mult + 1ull) * cur_plus;
        cur_mult = cur_mult * cur_mult;
        delta >>= 1;
    }
    r.state = acc_mult * r.state + acc_plus;
}

// uniform float in [0, 1): 32 random bits times 2^-32, capped below 1
BTRC_HD float pcg32_uniform_float(Pcg32 &r)
{
    const float f = (float)pcg32_next(r) * 2.3283064365386963e-10f;
    return f < 0x1.fffffep-1f ? f : 0x1.fffffep-1f;
}

// IndependentSampler(res, pixel, sample_index), independent.cpp:11-15
BTRC_HD Pcg32 independent_start(uint32_t px, uint32_t py, int32_t sample_index)
{
    const uint64_t seq = murmur_hash_pixel(px, py);
    Pcg32 r = pcg32_seed(seq, mix_bits(seq));
    pcg32_advance(r, (uint64_t)((int64_t)sample_index * 65536));
    return r;
}

} // namespace btrc
