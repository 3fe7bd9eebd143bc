// tp_xoshiro.h -- xoshiro256+ on the device (src/random/standard.rs via
// rand_xoshiro 0.6.0 and rand 0.8.5's Standard f64), and GF(2) skip-ahead by
// a 256x256 bit matrix (256 columns of 4 words, uniform across the wavefront).
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

namespace tpd {

// rotl(x, 45) = rotr(x, 19) and x << 17 on the two 32-bit halves with
// v_alignbit_b32 (a 64-bit rotate would otherwise take a 64-bit shift plus
// two 32-bit operations).
__device__ __forceinline__ uint64_t pack64(uint32_t lo, uint32_t hi) { return ((uint64_t)hi << 32) | lo; }
__device__ __forceinline__ uint64_t rotl45(uint64_t x)
{
    const uint32_t lo = (uint32_t)x, hi = (uint32_t)(x >> 32);
    return pack64(__builtin_amdgcn_alignbit(hi, lo, 19), __builtin_amdgcn_alignbit(lo, hi, 19));
}
__device__ __forceinline__ uint64_t shl17(uint64_t x)
{
    const uint32_t lo = (uint32_t)x, hi = (uint32_t)(x >> 32);
    return pack64(lo << 17, __builtin_amdgcn_alignbit(hi, lo, 15));
}

// next_u64: output s0 + s3 before the state update.
__device__ __forceinline__ uint64_t xo_next(uint64_t s[4])
{
    const uint64_t r = s[0] + s[3];
    const uint64_t t = shl17(s[1]);
    s[2] ^= s[0];
    s[3] ^= s[1];
    s[1] ^= s[2];
    s[0] ^= s[3];
    s[2] ^= t;
    s[3] = rotl45(s[3]);
    return r;
}

// rand's Standard f64: (u64 >> 11) * 2^-53, evaluated as
// hi * 2^-32 + (lo >> 11) * 2^-53: both terms and their sum are exact, so the
// fma returns the same double as the reference's conversion.
__device__ __forceinline__ double xo_uniform(uint64_t s[4])
{
    const uint64_t x = xo_next(s);
    const uint32_t hi = (uint32_t)(x >> 32), lo = (uint32_t)x;
    return fma((double)hi, 0x1.0p-32, (double)(lo >> 11) * 0x1.0p-53);
}

// The same uniform times 2^64, i.e. (u64 >> 11) 2^11 as an exact double, for
// code that folds the 2^-64 into its own operations (masking the low bits is
// a cheaper instruction than shifting them out).
__device__ __forceinline__ double xo_uniform64(uint64_t s[4])
{
    const uint64_t x = xo_next(s);
    uint32_t hi = (uint32_t)(x >> 32);
    const uint32_t lo = (uint32_t)x;
    // (an empty asm on hi: without it the compiler matches the two 32-bit
    // conversions as a 64-bit one and adds a +0.0 term)
    asm("" : "+v"(hi));
    return fma((double)hi, 0x1.0p32, (double)(lo & 0xFFFFF800u));
}

// s <- M s.  Read through the constant address space so that the uniform
// columns come in with scalar loads into SGPRs.
typedef const __attribute__((address_space(4))) uint64_t cu64;

__device__ __forceinline__ void gf2_apply(const uint64_t *__restrict__ mg, uint64_t s[4])
{
    cu64 *m = (cu64 *)mg;
    uint64_t r0 = 0, r1 = 0, r2 = 0, r3 = 0;
#pragma unroll
    for (int w = 0; w < 4; ++w) {
        uint64_t x = s[w];
#pragma unroll 4
        for (int b = 0; b < 64; ++b) {
            uint64_t mask = 0ull - ((x >> b) & 1ull);
            cu64 *c = m + 4 * (64 * w + b);
            r0 ^= c[0] & mask;
            r1 ^= c[1] & mask;
            r2 ^= c[2] & mask;
            r3 ^= c[3] & mask;
        }
    }
    s[0] = r0;
    s[1] = r1;
    s[2] = r2;
    s[3] = r3;
}

// ---- states of a wavefront's lanes ------------------------------------------
// A wavefront whose lanes each take a run of consecutive draws needs 64 states
// a fixed number of draws apart.  A lane that skips to its own by itself
// applies one 256x256 matrix per set bit of its offset, some 2500 instructions
// each.  Instead the wavefront skips once to its first draw, all lanes on one
// matrix together (gf2_uniform), and takes the lanes' offsets from a table of
// their images of every nibble of the state (xo_lane_states): about 140
// instructions per digit of the skip and 650 for all 64 lanes.

// XOR over the wavefront's 64 lanes (all active); the result is uniform.
template <int CTRL, int ROWS> __device__ __forceinline__ uint32_t xor_dpp(uint32_t x)
{
    return x ^ (uint32_t)__builtin_amdgcn_update_dpp(0, (int)x, CTRL, ROWS, 0xf, false);
}
__device__ __forceinline__ uint32_t wave_xor(uint32_t x)
{
    x = xor_dpp<0x111, 0xf>(x); // row_shr:1, 2, 4, 8: lane 15 of each row of 16 holds the row's
    x = xor_dpp<0x112, 0xf>(x);
    x = xor_dpp<0x114, 0xf>(x);
    x = xor_dpp<0x118, 0xf>(x);
    x = xor_dpp<0x142, 0xa>(x); // row_bcast:15 into rows 1 and 3
    x = xor_dpp<0x143, 0xc>(x); // row_bcast:31 into rows 2 and 3: lane 63 holds all
    return (uint32_t)__builtin_amdgcn_readlane((int)x, 63);
}

// s <- M s for a state all lanes hold alike: lane l takes columns l, l + 64,
// l + 128 and l + 192.
__device__ __forceinline__ void gf2_uniform(const uint64_t *__restrict__ m, uint64_t s[4])
{
    const uint32_t lane = threadIdx.x & 63u;
    const uint4 *c = reinterpret_cast<const uint4 *>(m) + 2 * lane;
    uint32_t r[8] = {0, 0, 0, 0, 0, 0, 0, 0};
#pragma unroll
    for (int w = 0; w < 4; ++w) {
        const uint4 a = c[128 * w], b = c[128 * w + 1];
        const uint32_t k = 0u - ((uint32_t)(s[w] >> lane) & 1u);
        r[0] ^= a.x & k;
        r[1] ^= a.y & k;
        r[2] ^= a.z & k;
        r[3] ^= a.w & k;
        r[4] ^= b.x & k;
        r[5] ^= b.y & k;
        r[6] ^= b.z & k;
        r[7] ^= b.w & k;
    }
#pragma unroll
    for (int w = 0; w < 4; ++w)
        s[w] = pack64(wave_xor(r[2 * w]), wave_xor(r[2 * w + 1]));
}

// s <- B^e s for a state and exponent all lanes hold alike, from the table
// B^(v 16^j), v = 1..15, of e's hexadecimal digits j.
__device__ __forceinline__ void xo_advance_uniform(const uint64_t *__restrict__ tab, uint64_t e, uint64_t s[4])
{
    for (; e; e >>= 4, tab += 15 * 1024)
        if (e & 15u)
            gf2_uniform(tab + ((e & 15u) - 1) * 1024, s);
}

// The lanes' states s_l = L^l s from the table of L^l (v << 4 ch), entry
// [ch][v][2][lane][2 words] (ch the nibble of the state, v its value).
__device__ __forceinline__ void xo_lane_states(const uint64_t *__restrict__ tab, const uint64_t s[4], uint64_t st[4])
{
    const ulonglong2 *t = reinterpret_cast<const ulonglong2 *>(tab) + (threadIdx.x & 63u);
    st[0] = st[1] = st[2] = st[3] = 0;
#pragma unroll
    for (int w = 0; w < 4; ++w) {
        const uint64_t x = s[w];
#pragma unroll 8
        for (int k = 0; k < 16; ++k) {
            const ulonglong2 *e = t + 128 * (16 * (16 * w + k) + (uint32_t)((x >> (4 * k)) & 15u));
            const ulonglong2 a = e[0], b = e[64];
            st[0] ^= a.x;
            st[1] ^= a.y;
            st[2] ^= b.x;
            st[3] ^= b.y;
        }
    }
}

// ---- xoshiro128+ (the f32 generator of src/random/standard.rs) ---------------
__device__ __forceinline__ uint32_t rotl32(uint32_t x, int k) { return (x << k) | (x >> (32 - k)); }

__device__ __forceinline__ uint32_t xo128_next(uint32_t s[4])
{
    const uint32_t r = s[0] + s[3];
    const uint32_t t = s[1] << 9;
    s[2] ^= s[0];
    s[3] ^= s[1];
    s[1] ^= s[2];
    s[0] ^= s[3];
    s[2] ^= t;
    s[3] = rotl32(s[3], 11);
    return r;
}

// rand's Standard f32: (u32 >> 8) * 2^-24 (exact).
__device__ __forceinline__ float xo128_uniform(uint32_t s[4]) { return (float)(xo128_next(s) >> 8) * 0x1.0p-24f; }

// s <- M s for a 128x128 GF(2) matrix stored as 128 columns of 4 words.
typedef const __attribute__((address_space(4))) uint32_t cu32;

__device__ __forceinline__ void gf2_apply128(const uint32_t *__restrict__ mg, uint32_t s[4])
{
    cu32 *m = (cu32 *)mg;
    uint32_t r0 = 0, r1 = 0, r2 = 0, r3 = 0;
#pragma unroll
    for (int w = 0; w < 4; ++w) {
        const uint32_t x = s[w];
#pragma unroll 4
        for (int b = 0; b < 32; ++b) {
            const uint32_t mask = 0u - ((x >> b) & 1u);
            cu32 *c = m + 4 * (32 * w + b);
            r0 ^= c[0] & mask;
            r1 ^= c[1] & mask;
            r2 ^= c[2] & mask;
            r3 ^= c[3] & mask;
        }
    }
    s[0] = r0;
    s[1] = r1;
    s[2] = r2;
    s[3] = r3;
}

// The same for 128x128 matrices: lane l takes columns l and l + 64.
__device__ __forceinline__ void gf2_uniform128(const uint32_t *__restrict__ m, uint32_t s[4])
{
    const uint32_t lane = threadIdx.x & 63u;
    const uint4 *c = reinterpret_cast<const uint4 *>(m) + lane;
    const uint4 a = c[0], b = c[64];
    const uint32_t ka = 0u - ((uint32_t)(pack64(s[0], s[1]) >> lane) & 1u);
    const uint32_t kb = 0u - ((uint32_t)(pack64(s[2], s[3]) >> lane) & 1u);
    s[0] = wave_xor((a.x & ka) ^ (b.x & kb));
    s[1] = wave_xor((a.y & ka) ^ (b.y & kb));
    s[2] = wave_xor((a.z & ka) ^ (b.z & kb));
    s[3] = wave_xor((a.w & ka) ^ (b.w & kb));
}
__device__ __forceinline__ void xo128_advance_uniform(const uint32_t *__restrict__ tab, uint64_t e, uint32_t s[4])
{
    for (; e; e >>= 4, tab += 15 * 512)
        if (e & 15u)
            gf2_uniform128(tab + ((e & 15u) - 1) * 512, s);
}
// Entry [ch][v][lane][4 words] of the lane table.
__device__ __forceinline__ void xo128_lane_states(const uint32_t *__restrict__ tab, const uint32_t s[4], uint32_t st[4])
{
    const uint4 *t = reinterpret_cast<const uint4 *>(tab) + (threadIdx.x & 63u);
    st[0] = st[1] = st[2] = st[3] = 0;
#pragma unroll
    for (int w = 0; w < 4; ++w)
#pragma unroll 4
        for (int k = 0; k < 8; ++k) {
            const uint4 e = t[64 * (16 * (8 * w + k) + ((s[w] >> (4 * k)) & 15u))];
            st[0] ^= e.x;
            st[1] ^= e.y;
            st[2] ^= e.z;
            st[3] ^= e.w;
        }
}

} // namespace tpd
