// Device-side building blocks of the spectrometer path (gfx950, FP64).
//
// One event per lane.  Every routine restates one reference routine (cited)
// with the same operation order; the file is compiled with
// -ffp-contract=off so that only the explicit __builtin_fma calls of the
// generated COSY polynomials fuse.  Uniform draws come from a per-event
// counter-based Philox4x32-10 stream or from a per-event tape.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include "simc_bm_tables.h"

namespace simcdev {

// ---------------------------------------------------------------------------
// Event arrays are addressed through buffer resources (base and size in
// SGPRs, one 32-bit byte offset per lane); accesses past the array size read
// zero and write nothing.
// ---------------------------------------------------------------------------
typedef unsigned int u32x2 __attribute__((ext_vector_type(2)));
constexpr int kBufWord3 = 0x00020000;  // raw 32-bit data format, gfx9 family

__device__ __forceinline__ __amdgpu_buffer_rsrc_t rsrc(const void* p, uint32_t bytes)
{
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(p), (short)0, (int)bytes, kBufWord3);
}
__device__ __forceinline__ double ld64(const double* p, uint32_t n, uint32_t off)
{
    return __builtin_bit_cast(double, __builtin_amdgcn_raw_buffer_load_b64(rsrc(p, n * 8u), off, 0, 0));
}
__device__ __forceinline__ uint32_t ld32(const uint32_t* p, uint32_t n, uint32_t off)
{
    return __builtin_amdgcn_raw_buffer_load_b32(rsrc(p, n * 4u), off, 0, 0);
}
__device__ __forceinline__ void st64(double* p, uint32_t n, uint32_t off, double v)
{
    __builtin_amdgcn_raw_buffer_store_b64(__builtin_bit_cast(u32x2, v), rsrc(p, n * 8u), off, 0, 0);
}
__device__ __forceinline__ void st32(void* p, uint32_t n, uint32_t off, uint32_t v)
{
    __builtin_amdgcn_raw_buffer_store_b32(v, rsrc(p, n * 4u), off, 0, 0);
}
__device__ __forceinline__ void st8(uint8_t* p, uint32_t n, uint32_t off, uint8_t v)
{
    __builtin_amdgcn_raw_buffer_store_b8(v, rsrc(p, n), off, 0, 0);
}

// constants.inc:23-42
constexpr double kPi = 3.141592653589793;
constexpr double kMpi = 139.57018;
constexpr double kMmu = 105.6583755;
constexpr double kMk = 493.677;

// ---------------------------------------------------------------------------
// Uniform sources
// ---------------------------------------------------------------------------

// Philox4x32-10 (Salmon et al., SC'11; Random123 constants).  Uniform k of an
// event is word k%4 of the block with counter (k/4, event lo, event hi, tag),
// mapped to (w + 1/2) 2^-32.
constexpr uint32_t kPhiloxTag = 0x53494d43u;  // "SIMC"
constexpr uint32_t kTargetTag = 0x54475453u;  // "TGTS"
constexpr uint32_t kHutTag = 0x48555453u;     // "HUTS": the detector huts' draws

// a ^ b ^ c in one instruction (truth table 0x96)
__device__ __forceinline__ uint32_t xor3(uint32_t a, uint32_t b, uint32_t c)
{
    return __builtin_amdgcn_bitop3_b32(a, b, c, 0x96);
}

template <bool LANE_KEY = false>
__device__ __forceinline__ void philox4x32_10(uint32_t c0, uint32_t c1, uint32_t c2, uint32_t c3,
                                              uint32_t k0, uint32_t k1, uint32_t out[4])
{
    // A launch-uniform key: without this empty statement the compiler forms
    // the 20 round keys once per kernel and keeps them in SGPRs across the
    // whole step loop, where they are spilled to VGPR lanes and read back
    // (v_readlane) in every block.  Made opaque here, they are recomputed by
    // scalar adds in each call instead.  A per-lane key (events of several
    // settings in one wavefront) is kept opaque in VGPRs for the same reason.
    // A launch-uniform key read back from memory (a stream passed to an
    // outlined function) arrives in VGPRs: readfirstlane moves it to SGPRs
    // (a copy where it is already there).
    if (LANE_KEY) {
        asm("" : "+v"(k0), "+v"(k1));
    } else {
        k0 = __builtin_amdgcn_readfirstlane(k0);
        k1 = __builtin_amdgcn_readfirstlane(k1);
        asm("" : "+s"(k0), "+s"(k1));
    }
#pragma unroll
    for (int r = 0; r < 10; ++r) {
        const uint64_t p0 = (uint64_t)0xD2511F53u * c0;
        const uint64_t p1 = (uint64_t)0xCD9E8D57u * c2;
        const uint32_t n0 = xor3((uint32_t)(p1 >> 32), c1, k0);
        const uint32_t n2 = xor3((uint32_t)(p0 >> 32), c3, k1);
        c1 = (uint32_t)p1;
        c3 = (uint32_t)p0;
        c0 = n0;
        c2 = n2;
        k0 += 0x9E3779B9u;
        k1 += 0xBB67AE85u;
    }
    out[0] = c0; out[1] = c1; out[2] = c2; out[3] = c3;
}

// Square root by one coupled (Goldschmidt) iteration from the hardware's
// reciprocal square root (2^-24) and one residual correction (Markstein);
// `y` receives 1 / sqrt(s) to 2^-47, enough for div_by's residual to round a
// quotient.  Before their last rounding both results are within 2^-42 ulp of
// the exact ones, so one in about 2^42 may round the other way than sqrt(s) and
// a / sqrt(s) (s in [2^-900, 2^1000]; no scaling and no special cases, as the
// general forms have them).  The tests hold millions of them equal in each
// range they are used in.
__device__ __forceinline__ double sqrt_inv(double s, double& y)
{
    const double y0 = __builtin_amdgcn_rsq(s);
    double g = s * y0, h = 0.5 * y0;
    const double e = __builtin_fma(-h, g, 0.5);
    g = __builtin_fma(g, e, g);
    h = __builtin_fma(h, e, h);
    y = h + h;
    return __builtin_fma(__builtin_fma(-g, g, s), h, g);
}
// a / r from y = 1 / r to 2^-47
__device__ __forceinline__ double div_by(double a, double r, double y)
{
    const double q = a * y;
    return __builtin_fma(__builtin_fma(-r, q, a), y, q);
}

// ---------------------------------------------------------------------------
// Elementary functions of the Box-Muller normal generator.  Both are fixed
// sequences of IEEE operations (explicit fma, exact reductions) over the
// tables of simc_bm_tables.h, so that the host restatement produces
// bit-identical values.
// ---------------------------------------------------------------------------
struct __attribute__((aligned(16))) BmLogEntry {
    double nhi;
    float nlo, invc;
};
static __constant__ BmLogEntry kBmLogTab[SIMC_BM_LOG_N] = SIMC_BM_LOG_TABLE;
static __constant__ __attribute__((aligned(16))) double kBmSinCosTab[SIMC_BM_SINCOS_N][2] = SIMC_BM_SINCOS_TABLE;

// A 16-byte table entry at byte offset `off` from a table in constant memory:
// one load from a scalar base and a 32-bit lane offset.
typedef unsigned int u32x4 __attribute__((ext_vector_type(4)));
__device__ __forceinline__ u32x4 table16(const void* base, uint32_t off)
{
    typedef const char __attribute__((address_space(4)))* cbytes;
    typedef const u32x4 __attribute__((address_space(4)))* centry;
    return *(centry)((cbytes)base + off);
}
__device__ __forceinline__ double double_of(uint32_t lo, uint32_t hi)
{
    return __builtin_bit_cast(double, u32x2{lo, hi});
}

// Natural logarithm of u = (w + 1/2) 2^-32: u = m 2^e with m in [sqrt(1/2),
// sqrt(2)), split on the bits (a 64-bit subtraction of sqrt(1/2)'s, whose
// exponent field is then e); c = 1 + k/64 the nearest table point, k =
// rint((m - 1) 64) taken from the low word of one fma onto 1.5 2^52 (an even
// offset, so ties go the same way); invc = 1/c to 7 bits, so t = m invc - 1
// is exact (|t| < 0.0155); log m = -log(invc) + log1p(t), log1p by its series
// to t^9 (truncation below 2^-56 relative); then e ln2 in two parts (ln2_hi
// has 21 significant bits, so e ln2_hi is exact) and the table's two-part
// -log(invc).
struct BmLog {
    double m;
    int e;
    u32x4 entry;
    __device__ __forceinline__ void load(uint32_t w)
    {
        const u32x2 x = __builtin_bit_cast(u32x2, (double)w + 0.5);  // 2^32 u, exact
        const uint32_t d = x.y - 0x3fe6a09eu - (x.x < 0x667f3bcdu ? 1u : 0u);
        e = ((int)d >> 20) - 32;
        m = double_of(x.x, x.y - (d & 0xfff00000u));
        static_assert(SIMC_BM_LOG_K0 == 19, "the table's first point");
        const double kd = __builtin_fma(m, 64.0, 0x1.8p52 - 64.0 + 20.0);  // low word: k + 20
        entry = table16((const char*)kBmLogTab - 16, __builtin_bit_cast(u32x2, kd).x << 4);
    }
    __device__ __forceinline__ double value() const
    {
        const double nhi = double_of(entry.x, entry.y);
        const float nlo = __builtin_bit_cast(float, (uint32_t)entry.z), invc = __builtin_bit_cast(float, (uint32_t)entry.w);
        const double t = __builtin_fma(m, (double)invc, -1.0);
        double q = 0x1.c71c71c71c71cp-4;                 // 1/9
        q = __builtin_fma(t, q, -0x1p-3);                // -1/8
        q = __builtin_fma(t, q, 0x1.2492492492492p-3);   // 1/7
        q = __builtin_fma(t, q, -0x1.5555555555555p-3);  // -1/6
        q = __builtin_fma(t, q, 0x1.999999999999ap-3);   // 1/5
        q = __builtin_fma(t, q, -0x1p-2);                // -1/4
        q = __builtin_fma(t, q, 0x1.5555555555555p-2);   // 1/3
        q = __builtin_fma(t, q, -0x1p-1);                // -1/2
        const double p = __builtin_fma(t * t, q, t);
        const double de = (double)e;
        return __builtin_fma(de, 0x1.62e42p-1, nhi + (p + __builtin_fma(de, 0x1.fdf473de6af28p-22, (double)nlo)));
    }
};

// sin and cos of 2 pi u for u = (w + 1/2) 2^-32: 64 u = k + r with k =
// rint(64 u) and r in [-1/2, 1/2], both read off w (its low 26 bits with
// sign are 2^26 r - 1/2), d = r pi/32 in one fma; sin d and cos d by their
// Taylor series to d^9 and d^8 (|d| <= pi/64, truncation below 2^-62), then
// the rotation by the table's sin and cos of 2 pi k/64.
struct BmSinCos {
    uint32_t w;
    u32x4 entry;
    __device__ __forceinline__ void load(uint32_t w_)
    {
        w = w_;
        entry = table16(kBmSinCosTab, ((w + (1u << 25)) >> 22) & 0x3f0u);  // entry k
    }
    __device__ __forceinline__ void value(double& sn, double& cs) const
    {
        const int rw = (int)(w << 6) >> 6;
        const double d = __builtin_fma((double)rw, 0x1.921fb54442d18p-30, 0x1.921fb54442d18p-31);
        const double z = d * d;
        double ps = 0x1.71de3a556c734p-19;                 // 1/9!
        ps = __builtin_fma(z, ps, -0x1.a01a01a01a01ap-13);  // -1/7!
        ps = __builtin_fma(z, ps, 0x1.1111111111111p-7);    // 1/5!
        ps = __builtin_fma(z, ps, -0x1.5555555555555p-3);   // -1/3!
        const double sd = __builtin_fma(d * z, ps, d);
        double pc = 0x1.a01a01a01a01ap-16;                 // 1/8!
        pc = __builtin_fma(z, pc, -0x1.6c16c16c16c17p-10);  // -1/6!
        pc = __builtin_fma(z, pc, 0x1.5555555555555p-5);    // 1/4!
        pc = __builtin_fma(z, pc, -0x1p-1);                 // -1/2
        const double cd = __builtin_fma(z, pc, 1.0);
        const double sa = double_of(entry.x, entry.y), ca = double_of(entry.z, entry.w);
        sn = __builtin_fma(sa, cd, ca * sd);
        cs = __builtin_fma(ca, cd, -(sa * sd));
    }
};

// The Box-Muller pair of two words: sqrt(-2 ln u1) (cos 2 pi u2, sin 2 pi u2).
// -2 ln u1 lies in [2^-32, 46], inside sqrt_inv's range.
struct BmPair {
    BmLog lg;
    BmSinCos sc;
    __device__ __forceinline__ void load(uint32_t w1, uint32_t w2)
    {
        lg.load(w1);
        sc.load(w2);
    }
    __device__ __forceinline__ void value(double& c, double& s) const
    {
        double y, sn, cs;
        const double r = sqrt_inv(-2.0 * lg.value(), y);
        sc.value(sn, cs);
        c = r * cs;
        s = r * sn;
    }
};
__device__ __forceinline__ void bm_pair(uint32_t w1, uint32_t w2, double& c, double& s)
{
    BmPair p;
    p.load(w1, w2);
    p.value(c, s);
}

// TAG is the fourth counter word: streams of different tags are independent
// (the arms use kPhiloxTag, the target step kTargetTag).
template <uint32_t TAG, bool LANE_KEY = false>
struct PhiloxStreamT {
    // LANE_KEY: the key (seed) may differ between the lanes of a wavefront
    static constexpr bool kLaneKey = LANE_KEY;
    uint32_t k0, k1, e0, e1;
    uint32_t pos;
    uint32_t w[4];
    int overflow;
    int have;        // a second Box-Muller normal is pending
    double pending;
    // inlined: an outlined init would leave the key in memory, no longer
    // provably uniform for the SGPR constraint of philox4x32_10
    __device__ __forceinline__ void init(uint64_t seed, uint64_t event, const double*, uint32_t, uint32_t)
    {
        k0 = (uint32_t)seed; k1 = (uint32_t)(seed >> 32);
        e0 = (uint32_t)event; e1 = (uint32_t)(event >> 32);
        pos = 0; overflow = 0; have = 0; pending = 0.0;
    }
    // Stream position for a later resume: uniforms drawn, and the pending
    // Box-Muller value.
    __device__ __forceinline__ uint32_t state_word() const { return pos | ((uint32_t)have << 31); }
    // The block's words are consumed from w[0], shifting the rest down: an
    // index by the position would put w in scratch memory (one round trip
    // per uniform), the shift is three register moves.
    __device__ __forceinline__ void shift()
    {
        w[0] = w[1];
        w[1] = w[2];
        w[2] = w[3];
    }
    // Resume at a saved position (re-forms the current Philox block when the
    // position is inside one).
    __device__ __forceinline__ void resume(uint32_t word, double pend)
    {
        pos = word & 0x7fffffffu;
        have = (int)(word >> 31);
        pending = pend;
        if (pos & 3u) {
            philox4x32_10<LANE_KEY>(pos >> 2, e0, e1, TAG, k0, k1, w);
            if ((pos & 3u) >= 1u) shift();
            if ((pos & 3u) >= 2u) shift();
            if ((pos & 3u) >= 3u) shift();
        }
    }
    __device__ __forceinline__ uint32_t next_word()
    {
        if ((pos & 3u) == 0) philox4x32_10<LANE_KEY>(pos >> 2, e0, e1, TAG, k0, k1, w);
        ++pos;
        const uint32_t v = w[0];
        shift();
        return v;
    }
    __device__ __forceinline__ double next()
    {
        return __builtin_fma((double)next_word(), 0x1p-32, 0x1p-33);  // (v + 1/2) 2^-32, exact
    }
    // Normal deviates for the counter-based stream: Box-Muller pairs
    // (u1, u2) -> sqrt(-2 ln u1) (cos 2 pi u2, sin 2 pi u2), both used, the
    // cosine value first.  There is no rejection step, so all lanes of a
    // wavefront consume uniforms in step and every Philox block is formed once
    // for the whole wavefront.  |g| <= sqrt(-2 ln 2^-33) = 6.8 always, below
    // every truncation used; a value beyond nsigmax would be skipped.
    __device__ __forceinline__ double gauss(double nsigmax)
    {
        for (;;) {
            if (have) {
                have = 0;
                if (fabs(pending) <= nsigmax) return pending;
                continue;
            }
            const uint32_t w1 = next_word();
            const uint32_t w2 = next_word();
            double g1;
            bm_pair(w1, w2, g1, pending);
            have = 1;
            if (fabs(g1) <= nsigmax) return g1;
        }
    }
    // Two consecutive gauss(nsigmax) draws for nsigmax >= 7, where no
    // Box-Muller value is ever rejected (|g| <= 6.8): with no value pending
    // that is exactly one pair, cosine value first.
    __device__ __forceinline__ void gauss_pair(double& a, double& b)
    {
        if (have) {
            a = gauss(99.0);
            b = gauss(99.0);
            return;
        }
        const uint32_t w1 = next_word();
        const uint32_t w2 = next_word();
        bm_pair(w1, w2, a, b);
        pending = b;
    }
    __device__ __forceinline__ int32_t used() const { return (int32_t)pos; }
};
using PhiloxStream = PhiloxStreamT<kPhiloxTag>;
using PhiloxLaneStream = PhiloxStreamT<kPhiloxTag, true>;

// The detector hut's own counter-based stream: uniform k of an event's hut
// is word k%4 of the Philox block (k/4, event lo, event hi, kHutTag) under
// the event's key.  A hut draws at most one uniform (resmult), before any
// other, and then Box-Muller pairs (both values used, cosine first), so
// nothing is pending between steps.  The draws depend on launch-uniform flags
// only: the position is the same in every lane of a wavefront, so refills are
// scalar branches.
//
// Pairs are formed two at a time, one Philox block, in a function of its own
// (hut_pairs): inlined at each of the hut's ~100 draws the SHMS hut was 327 KB
// of straight-line code, five times the instruction cache, and every
// wavefront streamed it from L2.  The block's first two rounds depend on the
// lane through the event id alone, so their products are formed once per
// event (a, h, l below) and the counter's part is scalar.
struct HutPairs {
    double a0, b0, a1, b1;
    uint32_t l1, l2, l3;
};

template <bool LANE_KEY>
__device__ __forceinline__ void hut_block(uint32_t blk, uint32_t a, uint32_t h, uint32_t l, uint32_t k0, uint32_t k1,
                                          uint32_t (&out)[4])
{
    blk = __builtin_amdgcn_readfirstlane(blk);
    if (LANE_KEY) {
        asm("" : "+v"(k0), "+v"(k1));
    } else {
        k0 = __builtin_amdgcn_readfirstlane(k0);
        k1 = __builtin_amdgcn_readfirstlane(k1);
        asm("" : "+s"(k0), "+s"(k1));
    }
    // rounds 1 and 2: after round 1 the counter is (X, a, s2, s3) with
    // M0 X = (h, l)
    const uint64_t b0 = (uint64_t)0xD2511F53u * blk;
    const uint32_t s2 = (uint32_t)(b0 >> 32) ^ kHutTag ^ k1, s3 = (uint32_t)b0;
    const uint64_t b1 = (uint64_t)0xCD9E8D57u * s2;
    k0 += 0x9E3779B9u;
    k1 += 0xBB67AE85u;
    uint32_t c0 = (uint32_t)(b1 >> 32) ^ a ^ k0, c1 = (uint32_t)b1, c2 = h ^ s3 ^ k1, c3 = l;
#pragma unroll
    for (int r = 2; r < 10; ++r) {
        k0 += 0x9E3779B9u;
        k1 += 0xBB67AE85u;
        const uint64_t p0 = (uint64_t)0xD2511F53u * c0;
        const uint64_t p1 = (uint64_t)0xCD9E8D57u * c2;
        const uint32_t n0 = xor3((uint32_t)(p1 >> 32), c1, k0);
        const uint32_t n2 = xor3((uint32_t)(p0 >> 32), c3, k1);
        c1 = (uint32_t)p1;
        c3 = (uint32_t)p0;
        c0 = n0;
        c2 = n2;
    }
    out[0] = c0; out[1] = c1; out[2] = c2; out[3] = c3;
}

// The next two pairs: from block blk, or with `odd` from the three words left
// of the block before and the first of blk (the others are left).
template <bool LANE_KEY>
__device__ __attribute__((noinline)) HutPairs hut_pairs(uint32_t blk, uint32_t odd, uint32_t a, uint32_t h, uint32_t l,
                                                        uint32_t k0, uint32_t k1, uint32_t l1, uint32_t l2, uint32_t l3)
{
    uint32_t w[4];
    hut_block<LANE_KEY>(blk, a, h, l, k0, k1, w);
    HutPairs r;
    r.l1 = w[1];
    r.l2 = w[2];
    r.l3 = w[3];
    if (__builtin_amdgcn_readfirstlane(odd)) {
        w[3] = w[0];
        w[0] = l1;
        w[1] = l2;
        w[2] = l3;
    }
    // all four table reads in flight before the first is waited for
    BmPair p0, p1;
    p0.load(w[0], w[1]);
    p1.load(w[2], w[3]);
    __builtin_amdgcn_sched_barrier(0);
    p0.value(r.a0, r.b0);
    p1.value(r.a1, r.b1);
    return r;
}

template <bool LANE_KEY>
struct HutPhilox {
    uint32_t k0, k1, a, h, l;
    uint32_t pos, blk;       // uniforms drawn; the next block
    uint32_t odd, half;      // one uniform was drawn first; a pair is ready
    uint32_t l1, l2, l3;
    double ra, rb;
    template <uint32_t TAG>
    __device__ __forceinline__ void init_from(const PhiloxStreamT<TAG, LANE_KEY>& g)
    {
        k0 = g.k0; k1 = g.k1;
        const uint64_t p1 = (uint64_t)0xCD9E8D57u * g.e1;
        const uint64_t p0 = (uint64_t)0xD2511F53u * ((uint32_t)(p1 >> 32) ^ g.e0 ^ g.k0);
        a = (uint32_t)p1;
        h = (uint32_t)(p0 >> 32);
        l = (uint32_t)p0;
        pos = 0; blk = 0; odd = 0; half = 0;
        l1 = l2 = l3 = 0;
        ra = rb = 0.0;
    }
    // the one uniform, before any pair
    __device__ __forceinline__ double next()
    {
        uint32_t w[4];
        hut_block<LANE_KEY>(0, a, h, l, k0, k1, w);
        l1 = w[1]; l2 = w[2]; l3 = w[3];
        pos = 1; blk = 1; odd = 1;
        return __builtin_fma((double)w[0], 0x1p-32, 0x1p-33);  // (v + 1/2) 2^-32, exact
    }
    __device__ __forceinline__ void gauss_pair(double& u, double& v)
    {
        pos += 2;
        if (half) {
            u = ra;
            v = rb;
            half = 0;
            return;
        }
        const HutPairs r = hut_pairs<LANE_KEY>(blk, odd, a, h, l, k0, k1, l1, l2, l3);
        ++blk;
        half = 1;
        u = r.a0;
        v = r.b0;
        ra = r.a1;
        rb = r.b1;
        l1 = r.l1;
        l2 = r.l2;
        l3 = r.l3;
    }
    __device__ __forceinline__ uint32_t used() const { return pos; }
};

// The stream the detector hut draws from: its own for the counter-based
// source; a tape (the reference's sequence) continues through the hut.
template <class R>
struct HutStreamOf {
    using type = R;
    static constexpr bool kOwn = false;
};
template <uint32_t TAG, bool LANE_KEY>
struct HutStreamOf<PhiloxStreamT<TAG, LANE_KEY>> {
    using type = HutPhilox<LANE_KEY>;
    static constexpr bool kOwn = true;
};

template <class R>
__device__ __forceinline__ double polar_gauss(R& g, double nsigmax);

// Tape of the launch: event slot at byte offset `base`, `stride` bytes long.
// Normal deviates use the reference's Marsaglia polar method (gauss1.f).
struct TapeStream {
    static constexpr bool kLaneKey = false;
    const double* tape;
    uint32_t base, stride, pos;
    int overflow;
    int have;          // unused (kept for a common state layout)
    double pending;
    __device__ __forceinline__ void init(uint64_t, uint64_t, const double* t, uint32_t slot_off, uint32_t s)
    {
        tape = t; base = slot_off; stride = s; pos = 0; overflow = 0; have = 0; pending = 0.0;
    }
    __device__ __forceinline__ uint32_t state_word() const { return pos; }
    __device__ __forceinline__ void resume(uint32_t word, double) { pos = word; }
    __device__ __forceinline__ double next()
    {
        if (pos >= stride) { overflow = 1; pos += 8u; return 0.5; }
        const double v = __builtin_bit_cast(
            double, __builtin_amdgcn_raw_buffer_load_b64(rsrc(tape, 0xffffffffu), base + pos, 0, 0));
        pos += 8u;
        return v;
    }
    __device__ __forceinline__ double gauss(double nsigmax) { return polar_gauss(*this, nsigmax); }
    __device__ __forceinline__ void gauss_pair(double& a, double& b)
    {
        a = polar_gauss(*this, 99.0);
        b = polar_gauss(*this, 99.0);
    }
    __device__ __forceinline__ int32_t used() const { return (int32_t)(pos / 8u); }
};

// ---------------------------------------------------------------------------
// Per-event track state: common /track/ plus the decay bookkeeping.
// ---------------------------------------------------------------------------
struct Track {
    double xs, ys, dxdzs, dydzs, dpps;
    double p, m2, pathlen, decdist;
    int dflag;
};

// Per-event settings of the run (one kinematic setting).
struct Flags {
    double ctau;     // decay length c tau (cm)
    double p_spec;   // central momentum (MeV/c)
    double sigma;    // wire-chamber resolution (cm)
    int ms, wcs, decay, coll, fit_f32;
    int sieve;       // the run's mock sieve options: bit 0 use_sieve, bit 1 the SHMS's use_2sieve
};

// Rotation constants tan/sin/cos of rotang * 0.017453292 (the truncated
// degree constant of shared/rotate_haxis.f:41), evaluated on the host with
// the same libm calls the reference makes.
struct Rot {
    double tan_th, sin_th, cos_th;
};

// ---------------------------------------------------------------------------
// gauss1, gauss1.f:17-27: Marsaglia polar method, second normal discarded.
// ---------------------------------------------------------------------------
template <class R>
__device__ __forceinline__ double polar_gauss(R& g, double nsigmax)
{
    for (;;) {
        const double u1 = g.next();
        const double u2 = g.next();
        if (g.overflow) return 0.0;
        const double v1 = 2.0 * u1 - 1.0;
        const double v2 = 2.0 * u2 - 1.0;
        const double s = v1 * v1 + v2 * v2;
        if (s > 1.0 || s == 0.0) continue;
        const double r = v1 * sqrt(-(2.0 * log(s) / s));
        if (fabs(r) > nsigmax) continue;
        return r;
    }
}

// A normal deviate from the event's stream (polar method on a tape,
// Box-Muller pairs on the counter-based stream).
template <class R>
__device__ __forceinline__ double gauss1(R& g, double nsigmax)
{
    return g.gauss(nsigmax);
}

// theta_sigma of musc / musc_ext (shared/musc.f:48-51, shared/musc_ext.f:36-39)
__device__ __forceinline__ double theta_sigma(double m2, double p, double rad_len)
{
    const double Es = 13.6, epsilon = 0.088;
    const double beta = p / sqrt(m2 + p * p);
    return Es / p / beta * sqrt(rad_len) * (1.0 + epsilon * log10(rad_len / (beta * beta)));
}

// theta_sigma for the detector-hut steps, whose radiation lengths are
// constants: sqrt(rad_len) and log10(rad_len) come with the step, the track
// factors Es/p/beta and log10(beta^2) are formed once per momentum, and
// log10(rad_len/beta^2) is taken as log10(rad_len) - log10(beta^2) (the same
// value to a few units in the last place).
struct ThetaCache {
    double p = -1.0, m2 = -1.0, a = 0.0, lb = 0.0;
    __device__ __forceinline__ void set(const Track& t)
    {
        const double Es = 13.6;
        p = t.p;
        m2 = t.m2;
        const double beta = p / sqrt(m2 + p * p);
        a = Es / p / beta;
        lb = log10(beta * beta);
    }
    // at the momentum of the last set()
    __device__ __forceinline__ double at(double sqrt_rl, double log10_rl) const
    {
        const double epsilon = 0.088;
        return a * sqrt_rl * (1.0 + epsilon * (log10_rl - lb));
    }
    __device__ __forceinline__ double theta(const Track& t, double sqrt_rl, double log10_rl)
    {
        if (t.p != p || t.m2 != m2) set(t);
        return at(sqrt_rl, log10_rl);
    }
};

// The mock sieve slit (hms/mc_hms.f:155-168, shms/mc_shms.f:276-310,
// sos/mc_sos.f:122-137, hrsl/mc_hrsl.f:122-132): the track from the target
// point is forced through the nearest hole of a sieve at z, at an offset drawn
// inside the hole (two uniforms), by changing its angles.  kind 0: holes on a
// (px, py) grid; 1: the SOS's rows (middle three at 1.016 cm, outer ones on a
// 2.54 cm pitch from 1.016); 2: the HRS's (the offset is drawn, not applied).
// NINT is round half away from zero.
template <class R>
__device__ __forceinline__ void sieve_slit(R& g, Track& t, int kind, double z, double px, double py, double r)
{
    const double x = t.xs, y = t.ys;
    double xt = x + z * t.dxdzs;
    double yt = y + z * t.dydzs;
    xt = px * round(xt / px);
    if (kind == 1) {
        if (fabs(yt) < 1.524) yt = 1.016 * round(yt / 1.016);
        else yt = yt / fabs(yt) * (2.54 * round((fabs(yt) - 1.016) / 2.54) + 1.016);
    } else {
        yt = py * round(yt / py);
    }
    const double rt = r * sqrt(g.next());
    const double tht = 2.0 * kPi * g.next();
    if (kind != 2) {
        xt = xt + rt * cos(tht);
        yt = yt + rt * sin(tht);
    }
    t.dxdzs = (xt - x) / z;
    t.dydzs = (yt - y) / z;
}

// musc(m2, p, rad_len, dth, dph), shared/musc.f:43-57
template <class R>
__device__ __forceinline__ void musc(R& g, const Track& t, double rad_len, double& dth, double& dph)
{
    if (rad_len == 0.0) return;
    const double ts = theta_sigma(t.m2, t.p, rad_len);
    dth = dth + ts * gauss1(g, 99.0);
    dph = dph + ts * gauss1(g, 99.0);
}

// musc_ext(m2, p, rad_len, x_len, dph, dth, y, x), shared/musc_ext.f:25-51.
// Every call site passes (dydzs, dxdzs, ys, xs).
template <class R>
__device__ __forceinline__ void musc_ext(R& g, Track& t, double rad_len, double x_len)
{
    if (rad_len == 0.0) return;
    if (x_len <= 0.0 || rad_len < 0.0) return;
    const double ts = theta_sigma(t.m2, t.p, rad_len);
    const double s12 = 3.4641016151377544;  // sqrt(12.)
    double g1 = gauss1(g, 99.0);
    double g2 = gauss1(g, 99.0);
    t.dxdzs = t.dxdzs + ts * g1;
    t.xs = t.xs + ts * x_len * g2 / s12 + ts * x_len * g1 / 2.0;
    g1 = gauss1(g, 99.0);
    g2 = gauss1(g, 99.0);
    t.dydzs = t.dydzs + ts * g1;
    t.ys = t.ys + ts * x_len * g2 / s12 + ts * x_len * g1 / 2.0;
}

// loren, loren.f:18-23
__device__ __forceinline__ void loren(double gam, double bx, double by, double bz, double e,
                                      double x, double y, double z, double& pxf, double& pyf,
                                      double& pzf, double& pf1)
{
    const double gam1 = gam * gam / (1.0 + gam);
    pxf = (1.0 + gam1 * (bx * bx)) * x + gam1 * bx * (by * y + bz * z) - gam * bx * e;
    pyf = (1.0 + gam1 * (by * by)) * y + gam1 * by * (bx * x + bz * z) - gam * by * e;
    pzf = (1.0 + gam1 * (bz * bz)) * z + gam1 * bz * (by * y + bx * x) - gam * bz * e;
    pf1 = sqrt(pxf * pxf + pyf * pyf + pzf * pzf);
}

// Decay products and boost: shared/project.f:72-109, shared/transp.f:146-184.
// m_kk is the final mass on the kaon two-body branch (Mk in the first half of
// transp, transp.f:158; Mpi elsewhere).
template <class R>
__device__ void decay_products(R& g, Track& t, double beta, double gamma, double p_spec, double m_kk)
{
    const double rph = g.next() * 2.0 * kPi;
    const double rth1 = g.next() * 2.0 - 1.0;
    const double rth = acos(rth1);
    double pr = 0.0, m_final = kMmu;
    if (fabs(sqrt(t.m2) - kMpi) < 2.0) pr = 29.783;
    if (fabs(sqrt(t.m2) - kMk) < 2.0) {
        if (g.next() < 0.7) {
            pr = 235.5;
        } else {
            pr = sqrt(kMk * kMk / 4.0 - kMpi * kMpi);
            m_final = m_kk;
        }
    }
    const double er = sqrt(m_final * m_final + pr * pr);
    const double pxr = pr * sin(rth) * cos(rph);
    const double pyr = pr * sin(rth) * sin(rph);
    const double pzr = pr * cos(rth);
    const double s = sqrt(1.0 + t.dxdzs * t.dxdzs + t.dydzs * t.dydzs);
    const double bx = -(beta * t.dxdzs / s);
    const double by = -(beta * t.dydzs / s);
    const double bz = -(beta * 1.0 / s);
    double pxf, pyf, pzf, pf;
    loren(gamma, bx, by, bz, er, pxr, pyr, pzr, pxf, pyf, pzf, pf);
    t.dxdzs = pxf / pzf;
    t.dydzs = pyf / pzf;
    t.dpps = 100.0 * (pf / p_spec - 1.0);
    t.p = pf;
    t.m2 = m_final * m_final;
}

// project, shared/project.f:38-119 applied to (xs, ys)
template <class R>
__device__ __forceinline__ void project(R& g, Track& t, const Flags& F, double z_drift)
{
    if (!F.decay || t.dflag) {
        t.pathlen = t.pathlen + z_drift * sqrt(1.0 + t.dxdzs * t.dxdzs + t.dydzs * t.dydzs);
        t.xs = t.xs + t.dxdzs * z_drift;
        t.ys = t.ys + t.dydzs * z_drift;
        return;
    }
    const double p_spec = t.p / (1.0 + t.dpps / 100.0);
    const double beta = t.p / sqrt(t.p * t.p + t.m2);
    const double gamma = 1.0 / sqrt(1.0 - beta * beta);
    const double dlen = F.ctau * beta * gamma;
    const double z_decay = -1.0 * dlen * log(1.0 - g.next());
    const double sq = sqrt(1.0 + t.dxdzs * t.dxdzs + t.dydzs * t.dydzs);
    if (z_decay > z_drift * sq) {
        t.decdist = t.decdist + z_drift * sq;
        t.pathlen = t.pathlen + z_drift * sq;
        t.xs = t.xs + t.dxdzs * z_drift;
        t.ys = t.ys + t.dydzs * z_drift;
    } else {
        t.dflag = 1;
        t.decdist = t.decdist + z_decay;
        t.pathlen = t.pathlen + z_decay;
        t.xs = t.xs + t.dxdzs * z_decay / sq;
        t.ys = t.ys + t.dydzs * z_decay / sq;
        decay_products(g, t, beta, gamma, p_spec, kMpi);
        const double sq2 = sqrt(1.0 + t.dxdzs * t.dxdzs + t.dydzs * t.dydzs);
        const double tmpdrift = z_drift - z_decay / sq2;
        t.pathlen = t.pathlen + tmpdrift * sq2;
        t.xs = t.xs + t.dxdzs * tmpdrift;
        t.ys = t.ys + t.dydzs * tmpdrift;
    }
}

// transp, shared/transp.f:134-279.  POLY(r0..r4, o0..o4) evaluates the class.
template <class R, class POLY>
__device__ __forceinline__ void transp(R& g, Track& t, const Flags& F, double zd, POLY poly)
{
    double p_spec = 0.0, beta = 0.0, gamma = 0.0, z_decay = 0.0;
    const bool check = F.decay && !t.dflag;
    if (check) {
        p_spec = t.p / (1.0 + t.dpps / 100.0);
        beta = t.p / sqrt(t.p * t.p + t.m2);
        gamma = 1.0 / sqrt(1.0 - beta * beta);
        const double dlen = F.ctau * beta * gamma;
        z_decay = -1.0 * dlen * log(1.0 - g.next());
        if (z_decay <= zd / 2.0) {
            t.dflag = 1;
            t.decdist = t.decdist + z_decay;
            decay_products(g, t, beta, gamma, p_spec, kMk);
        }
    }
    double o0, o1, o2, o3, o4;
    poly(t.xs, t.dxdzs * 1000.0, t.ys, t.dydzs * 1000.0, t.dpps, o0, o1, o2, o3, o4);
    t.xs = o0;
    t.dxdzs = o1 / 1000.0;
    t.ys = o2;
    t.dydzs = o3 / 1000.0;
    const double delta_z = -o4;
    if (check && !t.dflag) {
        if (z_decay > zd + delta_z) {
            t.decdist = t.decdist + (zd + delta_z);
        } else {
            t.dflag = 1;
            t.decdist = t.decdist + z_decay;
            decay_products(g, t, beta, gamma, p_spec, kMpi);
        }
    }
    t.pathlen = t.pathlen + (zd + delta_z);
}

// rotate_haxis, shared/rotate_haxis.f:43-61: new (xp0, yp0) from (xs, ys)
__device__ __forceinline__ void rotate_haxis(const Track& t, const Rot& r, double& xp0, double& yp0)
{
    const double alpha = t.dxdzs, beta = t.dydzs;
    const double alpha_p = (alpha + r.tan_th) / (1.0 - alpha * r.tan_th);
    const double beta_p = beta / (r.cos_th - alpha * r.sin_th);
    const double xi = xp0;
    xp0 = xi * (r.cos_th + alpha_p * r.sin_th);
    yp0 = yp0 + xi * beta_p * r.sin_th;
}

// rotate_vaxis, shared/rotate_vaxis.f:42-57
__device__ __forceinline__ void rotate_vaxis(const Track& t, const Rot& r, double& xp0, double& yp0)
{
    const double alpha = t.dydzs, beta = t.dxdzs;
    const double alpha_p = (alpha + r.tan_th) / (1.0 - alpha * r.tan_th);
    const double beta_p = beta / (r.cos_th - alpha * r.sin_th);
    const double yi = yp0;
    yp0 = yi * (r.cos_th + alpha_p * r.sin_th);
    xp0 = xp0 + yi * beta_p * r.sin_th;
}

// enerloss_new, enerloss_new.f:19-82, typeflag 1, in the collimator's
// tungsten: dens = 17, Z = 69.45, A = 171.56797.  Its material terms (the
// mean excitation I = 16 Z^0.9 eV, the plasma energy hnup, CO = ln hnup -
// ln I + 1/2, ln(me/I^2) + 1.063) are literals, each the correctly rounded
// value of the reference's expression; only the logarithms of the particle's
// terms are left to each step.
template <class R>
__device__ double enerloss_tungsten(R& g, double len, double epart, double mpart)
{
    const double dens = 17.0, zeff = 69.45, aeff = 171.56797;
    const double CO = -0x1.c387569315210p+0, ln10 = 0x1.26bb1bbb55516p+1, ln_me_I2 = 0x1.db05066e9762dp+3;
    const double thick = len * dens;
    const double gamma = epart / mpart;
    const double beta = sqrt(1.0 - 1.0 / (gamma * gamma));
    const double lnbg = log(beta * gamma);
    const double log10bg = lnbg / ln10;
    double denscorr;
    if (log10bg < 0.0) denscorr = 0.0;
    else if (log10bg < 3.0) {
        const double t3 = 3.0 - log10bg;
        denscorr = CO + ln10 * log10bg + fabs(CO / 27.0) * (t3 * t3 * t3);
    } else if (log10bg < 4.7) denscorr = CO + ln10 * log10bg;
    else denscorr = CO + ln10 * 4.7;
    double E;
    if (thick <= 0.0) {
        E = 0.0;
    } else {
        const double b2 = beta * beta;
        const double mp_new = 0.1536e-03 * zeff / aeff * thick / b2 *
                              (ln_me_I2 + 2.0 * lnbg + log(0.1536 * zeff / aeff * thick / b2) - b2 - denscorr);
        const double mp = mp_new * 1000.0;
        const double chsi = 0.307075 / 2.0 * zeff / aeff * thick / b2;
        const double x = fabs(gauss1(g, 10.0));
        const double lambda = x > 0.0 ? -2.0 * log(x) : 100000.0;
        E = lambda * chsi + mp;
    }
    if (E > (epart - mpart)) E = (epart - mpart) - 0.0000001;
    return E;
}

// sigA * 1.d-27 of pion_coll_absorb.f:223,229: the DOUBLE PRECISION literal is
// a 16-byte real under -fdefault-real-8, so the product is the correctly
// rounded value of sigA times the quad-precision 1e-27, formed here from a
// double-double split of that constant with an exact FMA product.
__device__ __forceinline__ double times_1em27_quad(double a)
{
    const double hi = 1.0e-27;
    const double lo = -3.849486974919184e-44;  // 1e-27 - hi, to double precision
    const double p = a * hi;
    const double e = __builtin_fma(a, hi, -p);
    return p + (e + a * lo);
}

// pion_coll_absorb, hms/pion_coll_absorb.f:54-90: transmission probability.
// The pion-nucleus cross sections sigreac * 171.57^qreac are taken per energy
// from a table (correctly rounded powers); the interval is found by counting
// the energies below the pion's, the same instructions in every lane.
struct __attribute__((aligned(16))) PionSigma {
    double T, sig;
};
static __constant__ PionSigma kPionSigma[14] = {
    {85.0, 0x1.ab340a64878aep+11},    {125.0, 0x1.3968509ef4563p+11},   {165.0, 0x1.05839ee881132p+11},
    {205.0, 0x1.ca66f5587393fp+10},   {245.0, 0x1.a50c4a4680271p+10},   {315.0, 0x1.8d13de1ddb713p+10},
    {584.02, 0x1.837068a094a21p+10},  {711.95, 0x1.830f350eff357p+10},  {870.12, 0x1.89f7ddd21c59dp+10},
    {1227.57, 0x1.8667eaf51ddc9p+10}, {1446.58, 0x1.85616242b8899p+10}, {1865.29, 0x1.7268c936690eep+10},
    {2858.0, 0x1.9f2eb6e68240ap+10},  {4159.0, 0x1.b493a5d2fff03p+10}};

__device__ __forceinline__ double pion_coll_absorb(double ppi, double thick)
{
    const double Navagadro = 6.0221367e+23, mpi = 139.56995;
    const double mate_dens = 17.0, mate_A = 171.57;
    const double Epi = sqrt(ppi * ppi + mpi * mpi);
    const double Tpi = Epi - mpi;
    int below = 0;
#pragma unroll
    for (int i = 0; i < 14; ++i) below += Tpi > kPionSigma[i].T ? 1 : 0;
    double sigA = 0.0;
    if (below == 14) {
        sigA = times_1em27_quad(kPionSigma[13].sig);
    } else if (below > 0) {
        const PionSigma lo = kPionSigma[below - 1], hi = kPionSigma[below];
        sigA = times_1em27_quad((lo.sig * (hi.T - Tpi) + hi.sig * (Tpi - lo.T)) / (hi.T - lo.T));
    }
    const double lambdai = mate_dens * Navagadro * sigA / mate_A;
    return exp(-(0.0 + thick * lambdai));
}

// mc_hms_coll / mc_shms_coll, hms/mc_hms_coll.f:50-136, shms/mc_shms_coll.f.
// Returns success; per-step slit hits go to cnt_step[0..2] (hor, vert, oct).
struct CollGeom {
    double h_entr, v_entr, h_exit, v_exit, x_off, y_off, coll_radl, step_size;
};

template <class R>
__device__ bool coll_step(R& g, Track& t, const Flags& F, const CollGeom& G, double p_spec,
                          unsigned* cnt_step)
{
    const int nstep = 20;
    double h_step = G.h_entr, v_step = G.v_entr;
    double epart = sqrt(t.p * t.p + t.m2);
#pragma unroll 1
    for (int n = 1; n <= nstep; ++n) {
        bool step_flag = false;
        if (fabs(t.ys - G.y_off) > h_step) { step_flag = true; ++cnt_step[0]; }
        if (fabs(t.xs - G.x_off) > v_step) { step_flag = true; ++cnt_step[1]; }
        if (fabs(t.xs - G.x_off) > (-(v_step / h_step * fabs(t.ys - G.y_off)) + 3.0 * v_step / 2.0)) {
            step_flag = true;
            ++cnt_step[2];
        }
        const double thick = G.step_size;
        if (step_flag) {
            if (t.m2 > 12000.0 && t.m2 < 20000.0) {
                const double trans = pion_coll_absorb(t.p, thick);
                if (g.next() > trans) return false;
            }
            musc(g, t, thick / G.coll_radl, t.dydzs, t.dxdzs);
            epart = sqrt(t.p * t.p + t.m2);
            const double eloss = enerloss_tungsten(g, thick, epart, sqrt(t.m2));
            epart = epart - eloss;
            if (epart < sqrt(t.m2)) return false;
            t.p = sqrt(epart * epart - t.m2);
            t.dpps = 100.0 * (t.p / p_spec - 1.0);
        }
        project(g, t, F, G.step_size);
        h_step = h_step + (G.h_exit - G.h_entr) / nstep;
        v_step = v_step + (G.v_exit - G.v_entr) / nstep;
    }
    return true;
}

// Fixed-collimator octagon test (hms/mc_hms.f:225-253, shms/mc_shms.f:524-565).
// Returns 0 inside, else the stop code 1 (hor), 2 (vert), 3 (oct).
__device__ __forceinline__ int slit(double x, double y, double h, double v, double x_off, double y_off)
{
    if (fabs(y - y_off) > h) return 1;
    if (fabs(x - x_off) > v) return 2;
    if (fabs(x - x_off) > (-(v / h * fabs(y - y_off)) + 3.0 * v / 2.0)) return 3;
    return 0;
}

// LFIT, cern/lfit.f:22-59 with KEY = 0.  T is float for the reference's
// REAL*4 hits (sums in FP64) or double for the FP64 fit.
template <class T, int L>
__device__ __forceinline__ void lfit(const T (&X)[L], const T (&Y)[L], T& A, T& B)
{
    double count = 0.0, sumx = 0.0, sumy = 0.0, sumxy = 0.0, sumxx = 0.0;
#pragma unroll
    for (int j = 0; j < L; ++j) {
        if (Y[j] == (T)0) continue;
        sumx = sumx + (double)X[j];
        sumy = sumy + (double)Y[j];
        count = count + 1.0;
    }
    if (count <= 1.0) { A = (T)0; B = (T)0; return; }
    const double ymed = sumy / count;
    const double xmed = sumx / count;
#pragma unroll
    for (int j = 0; j < L; ++j) {
        if (Y[j] == (T)0) continue;
        const double sx = (double)X[j] - xmed;
        const double sy = (double)Y[j] - ymed;
        sumxy = sumxy + sx * sy;
        sumxx = sumxx + sx * sx;
    }
    if (sumxx == 0.0) { A = (T)0; B = (T)0; return; }
    A = (T)(sumxy / sumxx);
    B = (T)(ymed - (double)A * xmed);
}

}  // namespace simcdev
