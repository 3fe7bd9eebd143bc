// tp_flow.hip -- bf16-MFMA kernels of the RealNVP proposal (see tp_flow.h).
//
// Matrix products use v_mfma_f32_16x16x16_bf16.  Activations are kept
// transposed (features x samples): for H^T = W X^T the weight tile is the A
// operand and the 16-sample activation tile the B operand, and the lane
// layout of the f32 result (lane l holds rows 4(l/16)..4(l/16)+3 of column
// l%16) is exactly the B layout the next product needs, so a whole coupling
// layer runs lane-locally in registers.  The coupling state of one sample is
// spread over the four lanes l%16 + 16 g, lane group g holding features
// 4g..4g+3 -- the same rows the s and t outputs land in.
#include "tp_flow.h"
#include "tp_adjoint.h"
#include "tp_xoshiro.h"

#include <algorithm>

// The network code below is not bound to any reference operation order:
// let the compiler fuse multiply-adds.  (The physics included above keeps
// the build's contraction-free setting; it is switched back off before the
// integrand kernel at the end of this file.)
#pragma clang fp contract(fast)

namespace tpf {

typedef short s4 __attribute__((ext_vector_type(4)));
typedef short s8 __attribute__((ext_vector_type(8)));
typedef float f4 __attribute__((ext_vector_type(4)));
typedef __bf16 bf4 __attribute__((ext_vector_type(4)));
typedef __bf16 bf8 __attribute__((ext_vector_type(8)));

constexpr float LOG2E = 1.4426950408889634f, LN2 = 0.6931471805599453f;

__device__ __forceinline__ uint16_t f2bf(float x) // round to nearest even (v_cvt_pk_bf16_f32)
{
    return __builtin_bit_cast(uint16_t, (__bf16)x);
}
__device__ __forceinline__ float bf2f(uint16_t h) { return __uint_as_float((uint32_t)h << 16); }
__device__ __forceinline__ s4 pack4(f4 v)
{
    const bf4 b = {(__bf16)v.x, (__bf16)v.y, (__bf16)v.z, (__bf16)v.w};
    return __builtin_bit_cast(s4, b);
}
__device__ __forceinline__ f4 mfma(s4 a, s4 b, f4 c) { return __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(a, b, c, 0, 0, 0); }
// gfx950's 16x16x32 product (twice the K of the one above per instruction):
// lane l supplies row / column l % 16 and eight K values of group l / 16.
__device__ __forceinline__ f4 mfma32(s8 a, s8 b, f4 c)
{
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf8, a), __builtin_bit_cast(bf8, b), c, 0, 0, 0);
}
// The B operand of a K = 32 product from two 16-row activation tiles: lane
// group g holds rows 4g..4g+3 of each, the eight K values of its group.
__device__ __forceinline__ s8 cat8(s4 lo, s4 hi) { return __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7); }
// Hardware exp2 / log2 / reciprocal (about 1 ulp): the network's activations
// are rounded to bf16 anyway.
__device__ __forceinline__ float fexp(float x) { return __builtin_amdgcn_exp2f(x * LOG2E); }
__device__ __forceinline__ float flog(float x) { return __builtin_amdgcn_logf(x) * LN2; }
__device__ __forceinline__ float frcp(float x) { return __builtin_amdgcn_rcpf(x); }
__device__ __forceinline__ float sigm(float x) { return frcp(1.f + fexp(-x)); }

// Hard-swish y = c min(max(c / 6 + 1/2, 0), 1) and its derivative (0 below
// -3, c / 3 + 1/2 up to 3, 1 above; PyTorch's hardswish): three full-rate
// operations where a sigmoid-based activation takes an exp2 and a reciprocal
// at a quarter of the rate (the forward-only kernels drop d).
__device__ __forceinline__ void hswish_d(float c, float &y, float &d)
{
    y = c * fminf(fmaxf(fmaf(c, 1.f / 6.f, 0.5f), 0.f), 1.f);
    d = c < -3.f ? 0.f : (c > 3.f ? 1.f : fmaf(c, 1.f / 3.f, 0.5f));
}
__device__ __forceinline__ float ftanh(float x) { return 1.f - 2.f * frcp(__builtin_amdgcn_exp2f(x * (2.f * LOG2E)) + 1.f); }
// softplus(-x) + softplus(x) with softplus(x) = max(x, 0) + log(1 + exp(-|x|))
__device__ __forceinline__ float softplus2(float x)
{
    const float lg = __builtin_amdgcn_logf(1.f + fexp(-fabsf(x)));
    return fmaf(lg, LN2, fabsf(x)) + fmaf(lg, LN2, 0.f); // (each rounded: a product would be contracted into the sum)
}

// ---- LDS image of one layer (bf16, padded row strides against bank conflicts)
// W2 and W3 (K = 64) feed K = 32 products: their columns are stored in the
// order those products read them.  Within each 32-column half c, lane group g
// reads the eight stored columns 32c + 8g .. 32c + 8g + 7, which hold the
// original columns 32c + 4g + (0..3) and 32c + 16 + 4g + (0..3): the rows
// 4g..4g+3 of the two 16-row activation tiles 2c and 2c+1 that the lane
// holds (cat8).  Row strides of 72 keep each lane's 16-byte read aligned.
constexpr int S_W1 = 20, S_W2 = 72, S_W3 = 72, S_W1T = 68, S_W2T = 68, S_W3T = 36;
__host__ __device__ constexpr int k32_pos(int k) // stored position of original column k
{
    return 32 * (k / 32) + 8 * ((k % 16) / 4) + (k % 4) + 4 * ((k % 32) / 16);
}
constexpr int L_W1 = 0, L_W2 = L_W1 + H * S_W1, L_W3 = L_W2 + H * S_W2, L_FWD = L_W3 + O * S_W3;
constexpr int L_W1T = 0, L_W2T = L_W1T + DP * S_W1T, L_W3T = L_W2T + H * S_W2T, L_T = L_W3T + H * S_W3T;

// Forward weights only (W1, W2, W3 and the biases): the forward and inverse
// kernels keep all L layers of them resident.
struct LdsFwd {
    uint16_t w[L_FWD];
    float b[H + H + O];
};

// With W1^T, W2^T, W3^T (backward pass).
struct LdsLayer : LdsFwd {
    uint16_t wt[L_T];
};
static_assert(sizeof(LdsLayer) == WIMG_BYTES && sizeof(LdsFwd) % 16 == 0, "the weights' images are copied by 16 bytes");

// Parameter i of a layer, in bf16, into the layer's image: the kernels that
// write the weights lay them out once, so that a workgroup takes them into LDS
// as they are, 16 bytes a lane (from the parameters' own order, 2 bytes a lane
// with their places worked out, it took 10 us of the forward kernel's 31).
__device__ __forceinline__ void put_weight(LdsLayer &s, int i, uint16_t v)
{
    if (i < OFF_B1) {
        const int r = i / DP, c = i % DP;
        s.w[L_W1 + r * S_W1 + c] = v;
        s.wt[L_W1T + c * S_W1T + r] = v;
    } else if (i < OFF_W2) {
        s.b[i - OFF_B1] = bf2f(v);
    } else if (i < OFF_B2) {
        const int r = (i - OFF_W2) / H, c = (i - OFF_W2) % H;
        s.w[L_W2 + r * S_W2 + k32_pos(c)] = v;
        s.wt[L_W2T + c * S_W2T + r] = v;
    } else if (i < OFF_W3) {
        s.b[H + i - OFF_B2] = bf2f(v);
    } else if (i < OFF_B3) {
        const int r = (i - OFF_W3) / H, c = (i - OFF_W3) % H;
        s.w[L_W3 + r * S_W3 + k32_pos(c)] = v;
        s.wt[L_W3T + c * S_W3T + r] = v;
    } else {
        s.b[2 * H + i - OFF_B3] = bf2f(v);
    }
}

// A operand of a 16x16 tile of a row-major LDS matrix: rows 16 mb .., cols 16 kb ..
__device__ __forceinline__ s4 atile(const uint16_t *m, int stride, int mb, int kb)
{
    const int lane = threadIdx.x & 63;
    const int r = 16 * mb + (lane & 15), c = 16 * kb + 4 * (lane >> 4);
    return *reinterpret_cast<const s4 *>(m + r * stride + c);
}

// A operand of a K = 32 product: rows 16 mb .., stored columns 32 c + 8 g ..
__device__ __forceinline__ s8 atile8(const uint16_t *m, int stride, int mb, int c)
{
    const int lane = threadIdx.x & 63;
    const int r = 16 * mb + (lane & 15), col = 32 * c + 8 * (lane >> 4);
    return *reinterpret_cast<const s8 *>(m + r * stride + col);
}

// Bias values of rows r0 .. r0 + 3 (the lane's rows of an output tile).
template <class Lds> __device__ __forceinline__ f4 bias4(const Lds &s, int r0)
{
    return *reinterpret_cast<const f4 *>(s.b + r0);
}

struct MlpFwd {
    s4 a;          // bf16 input (features 4g..4g+3)
    f4 h1d[4];     // hard-swish'(pre-activation), 4 row blocks (backward only)
    s4 h1[4];
    f4 h2d[4];
    s4 h2[4];
    f4 o0, o1;     // s raw (rows 0..15), t raw (rows 16..31)
};

template <class Lds> __device__ __forceinline__ void mlp_forward(const Lds &s, s4 a_in, MlpFwd &r)
{
    const int g = (threadIdx.x & 63) >> 4;
    r.a = a_in;
#pragma unroll
    for (int mb = 0; mb < 4; ++mb) {
        const f4 c = mfma(atile(s.w + L_W1, S_W1, mb, 0), r.a, bias4(s, 16 * mb + 4 * g));
        f4 h, d;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            float y, dy;
            hswish_d(c[i], y, dy);
            h[i] = y;
            d[i] = dy;
        }
        r.h1d[mb] = d;
        r.h1[mb] = pack4(h);
    }
#pragma unroll
    for (int mb = 0; mb < 4; ++mb) {
        f4 c = bias4(s, H + 16 * mb + 4 * g);
#pragma unroll
        for (int kc = 0; kc < 2; ++kc)
            c = mfma32(atile8(s.w + L_W2, S_W2, mb, kc), cat8(r.h1[2 * kc], r.h1[2 * kc + 1]), c);
        f4 h, d;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            float y, dy;
            hswish_d(c[i], y, dy);
            h[i] = y;
            d[i] = dy;
        }
        r.h2d[mb] = d;
        r.h2[mb] = pack4(h);
    }
    f4 o0 = bias4(s, 2 * H + 4 * g), o1 = bias4(s, 2 * H + 16 + 4 * g);
#pragma unroll
    for (int kc = 0; kc < 2; ++kc) {
        const s8 b = cat8(r.h2[2 * kc], r.h2[2 * kc + 1]);
        o0 = mfma32(atile8(s.w + L_W3, S_W3, 0, kc), b, o0);
        o1 = mfma32(atile8(s.w + L_W3, S_W3, 1, kc), b, o1);
    }
    r.o0 = o0;
    r.o1 = o1;
}

__device__ __forceinline__ bool transformed(uint32_t cond, int j) { return j < D && !((cond >> j) & 1u); }
__device__ __forceinline__ bool conditioning(uint32_t cond, int j) { return j < D && ((cond >> j) & 1u); }

// The layer's input in bf16: the lane's conditioning features, the others 0.
struct CondMask { // all ones in the halves that stay
    uint32_t lo, hi;
};
__device__ __forceinline__ CondMask cond_mask(uint32_t cond)
{
    const uint32_t c = cond >> (4 * ((threadIdx.x & 63) >> 4)); // (no bits from D on)
    return {(c & 1u ? 0xffffu : 0u) | (c & 2u ? 0xffff0000u : 0u), (c & 4u ? 0xffffu : 0u) | (c & 8u ? 0xffff0000u : 0u)};
}
__device__ __forceinline__ s4 masked(f4 z, CondMask m)
{
    const uint2 v = __builtin_bit_cast(uint2, pack4(z));
    return __builtin_bit_cast(s4, make_uint2(v.x & m.lo, v.y & m.hi));
}

// Sum over the four lane groups of one sample (lanes l, l^16, l^32, l^48).
__device__ __forceinline__ float sample_sum(float x)
{
    x += __shfl_xor(x, 16);
    x += __shfl_xor(x, 32);
    return x;
}

// ---- counter-stream draws ----------------------------------------------------
__device__ __forceinline__ uint64_t mix64(uint64_t z)
{
    z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ull;
    z = (z ^ (z >> 27)) * 0x94D049BB133111EBull;
    return z ^ (z >> 31);
}
// The Weyl sequence of draw k; the draws after it are GOLDEN apart.
constexpr uint64_t GOLDEN = 0x9E3779B97F4A7C15ull;
__device__ __forceinline__ uint64_t stream_at(uint64_t key, uint64_t k)
{
    uint64_t w = key + (k + 1) * GOLDEN;
    asm("" : "+v"(w)); // (one product, not one for each of the draws that follow)
    return w;
}
// (2 m + 1) 2^-24 with m the top 23 bits: strictly inside (0, 1), so logit(v)
// is finite.
__device__ __forceinline__ float stream_v(uint64_t w)
{
    uint32_t hi = (uint32_t)(mix64(w) >> 32);
    asm("" : "+v"(hi)); // (a 32-bit conversion: the compiler would make it a 64-bit one)
    return (float)(hi >> 9) * 0x1.0p-23f + 0x1.0p-24f;
}
// (2 m + 1) 2^-53 with m the top 52 bits: strictly inside (0, 1).
__device__ __forceinline__ double stream_u(uint64_t w) { return (double)(mix64(w) >> 12) * 0x1.0p-52 + 0x1.0p-53; }
// u = sigmoid(z), evaluated in f32 (the density is that of the f32 network;
// the point moves by at most an f32 rounding), stored as f64 and kept inside
// (0, 1): at most 1 - 2^-53 where the f32 value rounds to 1.
__device__ __forceinline__ double sigmoid_u(float z)
{
    const double u = (double)sigm(z);
    return fmin(fmax(u, 0x1.0p-126), 0x1.fffffffffffffp-1);
}

// ---- forward ----------------------------------------------------------------
// The forward and inverse kernels load the forward weights of all L layers
// into LDS once (99.75 KiB, one block per CU) and then stride over the samples
// with no further barrier: a block takes waves x tiles x 16 samples per pass.
// Bound by VALU issue (204 instructions per tile and layer, draws and densities
// among them, next to 16 matrix instructions: 79 % of the issue slots at 4 cycles
// each) where the wavefronts cover each other's latencies,
// so three wavefronts per SIMD with two tiles each take the long runs and four
// with one tile the batches that would leave CUs idle otherwise.  1.4e7 samples
// drawn and 6e6 inverted, with the weighted event loop: 4.05 ms; 4.11 at two
// wavefronts of four tiles, 4.14 at four of one; a training batch of 65 536: 20
// us, 31 at two of two with the weights read by 2 bytes.
constexpr int FWD_WAVES = 12, FWD_TILES = 2, FWD_WAVES_SMALL = 16, FWD_TILES_SMALL = 1;
constexpr uint64_t FWD_SMALL_N = 1u << 20;

template <int WAVES> __device__ __forceinline__ void load_resident(LdsFwd (&s)[L], const void *wimg)
{
    constexpr int THREADS = 64 * WAVES;
    constexpr int N = sizeof(LdsFwd) / 16, PER = (N + THREADS - 1) / (THREADS);
    uint4 v[L][PER];
#pragma unroll
    for (int l = 0; l < L; ++l)
#pragma unroll
        for (int k = 0; k < PER; ++k)
            v[l][k] = static_cast<const uint4 *>(wimg)[l * (WIMG_BYTES / 16) + min((int)threadIdx.x + THREADS * k, N - 1)];
#pragma unroll
    for (int l = 0; l < L; ++l)
#pragma unroll
        for (int k = 0; k < PER; ++k)
            if ((int)threadIdx.x + THREADS * k < N)
                reinterpret_cast<uint4 *>(&s[l])[threadIdx.x + THREADS * k] = v[l][k];
    __syncthreads();
}

template <int TILES, int WAVES>
__global__ __launch_bounds__(64 * WAVES) void flow_forward_kernel(FlowKernelArgs a)
{
    constexpr int CHUNK = WAVES * TILES * 16;
    __shared__ __attribute__((aligned(16))) LdsFwd s[L];
    load_resident<WAVES>(s, a.wimg);
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, g = lane >> 4;
    const bool feat = g < D / 4; // lane group 3 holds padding
    for (uint64_t base = (uint64_t)blockIdx.x * CHUNK; base < a.n; base += (uint64_t)gridDim.x * CHUNK) {
        f4 z[TILES];
        float ld[TILES];
        bool valid[TILES];
        uint64_t idx[TILES];
#pragma unroll
        for (int t = 0; t < TILES; ++t) {
            idx[t] = base + (uint64_t)(wave * TILES + t) * 16 + (lane & 15);
            valid[t] = idx[t] < a.n;
            f4 vv = {0.5f, 0.5f, 0.5f, 0.5f};
            if (a.v_in) {
                if (valid[t])
                    vv = *reinterpret_cast<const f4 *>(a.v_in + 16 * idx[t] + 4 * g);
            } else if (feat) {
                const uint64_t w = stream_at(a.key, 12ull * (a.sample0 + idx[t]) + 4 * g);
#pragma unroll
                for (int i = 0; i < 4; ++i)
                    vv[i] = stream_v(w + i * GOLDEN);
            }
            float l = 0.f;
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const float x = feat ? vv[i] : 0.5f;
                // (the multiply-adds are written out: which product the compiler
                // contracts would depend on the kernel's other choices)
                const float lx = __builtin_amdgcn_logf(x), l1x = flog(1.f - x);
                z[t][i] = fmaf(lx, LN2, -l1x);
                if (feat)
                    l += fmaf(lx, LN2, l1x); // log v (1 - v)
            }
            ld[t] = l;
        }
        for (int l = 0; l < L; ++l) {
            const uint32_t cond = COND_MASK[l];
            const CondMask cm = cond_mask(cond);
#pragma unroll
            for (int t = 0; t < TILES; ++t) {
                if (a.zsave && valid[t])
                    *reinterpret_cast<f4 *>(a.zsave + ((size_t)l * a.n + idx[t]) * 16 + 4 * g) = z[t];
                MlpFwd r;
                mlp_forward(s[l], masked(z[t], cm), r);
#pragma unroll
                for (int i = 0; i < 4; ++i) { // exp(0) = 1 exactly
                    // (sv before the select: the lane groups differ in what they
                    // transform, so a branch around it is never skipped, and it
                    // keeps the features' exponentials from running side by side)
                    const bool tr = transformed(cond, 4 * g + i);
                    const float sv = FLOW_SCALE * ftanh(r.o0[i]), sc = tr ? sv : 0.f;
                    z[t][i] = z[t][i] * fexp(sc) + (tr ? r.o1[i] : 0.f);
                    ld[t] -= sc;
                }
            }
        }
#pragma unroll
        for (int t = 0; t < TILES; ++t) {
            float l = ld[t];
            if (feat)
#pragma unroll
                for (int i = 0; i < 4; ++i) // - log u (1 - u) = softplus(-z) + softplus(z)
                    l += softplus2(z[t][i]);
            l = sample_sum(l);
            if (!valid[t])
                continue;
            if (feat && a.u_out) {
                double u[4];
#pragma unroll
                for (int i = 0; i < 4; ++i)
                    u[i] = sigmoid_u(z[t][i]);
                if (a.u_stride) {
#pragma unroll
                    for (int i = 0; i < 4; ++i)
                        a.u_out[(4 * g + i) * a.u_stride + idx[t]] = u[i];
                } else {
#pragma unroll
                    for (int i = 0; i < 4; ++i)
                        a.u_out[12 * idx[t] + 4 * g + i] = u[i];
                }
            }
            if (feat && a.z_out)
#pragma unroll
                for (int i = 0; i < 4; ++i)
                    a.z_out[12 * idx[t] + 4 * g + i] = z[t][i];
            if (g == 0) {
                if (a.logq_out)
                    a.logq_out[idx[t]] = l;
                if (a.invq_out)
                    a.invq_out[idx[t]] = 1. / (a.alpha * (double)fexp(l) + (1. - a.alpha));
            }
        }
    }
}

// ---- inverse: density of given or uniformly drawn points --------------------
template <int TILES, int WAVES>
__global__ __launch_bounds__(64 * WAVES) void flow_inverse_kernel(FlowKernelArgs a)
{
    constexpr int CHUNK = WAVES * TILES * 16;
    __shared__ __attribute__((aligned(16))) LdsFwd s[L];
    load_resident<WAVES>(s, a.wimg);
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, g = lane >> 4;
    const bool feat = g < D / 4; // lane group 3 holds padding
    for (uint64_t base = (uint64_t)blockIdx.x * CHUNK; base < a.n; base += (uint64_t)gridDim.x * CHUNK) {
        f4 z[TILES];
        float ld[TILES];
        bool valid[TILES];
        uint64_t idx[TILES];
#pragma unroll
        for (int t = 0; t < TILES; ++t) {
            idx[t] = base + (uint64_t)(wave * TILES + t) * 16 + (lane & 15);
            valid[t] = idx[t] < a.n;
            double u[4] = {0.5, 0.5, 0.5, 0.5};
            if (feat && a.u_in) {
                if (valid[t])
#pragma unroll
                    for (int i = 0; i < 4; ++i)
                        u[i] = fmin(fmax(a.u_in[12 * idx[t] + 4 * g + i], 0x1.0p-126), 0x1.fffffffffffffp-1);
            } else if (feat) {
                const uint64_t w = stream_at(a.key, 12ull * (a.sample0 + idx[t]) + 4 * g);
#pragma unroll
                for (int i = 0; i < 4; ++i)
                    u[i] = stream_u(w + i * GOLDEN);
                if (a.u_out && valid[t]) {
                    if (a.u_stride) {
#pragma unroll
                        for (int i = 0; i < 4; ++i)
                            a.u_out[(4 * g + i) * a.u_stride + idx[t]] = u[i];
                    } else {
#pragma unroll
                        for (int i = 0; i < 4; ++i)
                            a.u_out[12 * idx[t] + 4 * g + i] = u[i];
                    }
                }
            }
            float l = 0.f;
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                // u and 1 - u formed in f64, logs in f32
                const float lu = __builtin_amdgcn_logf((float)u[i]), l1u = flog((float)(1. - u[i]));
                z[t][i] = fmaf(lu, LN2, -l1u);
                if (feat)
                    l -= fmaf(lu, LN2, l1u); // - log u (1 - u)
            }
            ld[t] = l;
        }
        for (int l = L - 1; l >= 0; --l) {
            const uint32_t cond = COND_MASK[l];
            const CondMask cm = cond_mask(cond);
#pragma unroll
            for (int t = 0; t < TILES; ++t) {
                MlpFwd r;
                mlp_forward(s[l], masked(z[t], cm), r);
#pragma unroll
                for (int i = 0; i < 4; ++i) { // exp(0) = 1 exactly
                    // (sv before the select: the lane groups differ in what they
                    // transform, so a branch around it is never skipped, and it
                    // keeps the features' exponentials from running side by side)
                    const bool tr = transformed(cond, 4 * g + i);
                    const float sv = FLOW_SCALE * ftanh(r.o0[i]), sc = tr ? sv : 0.f;
                    z[t][i] = (z[t][i] - (tr ? r.o1[i] : 0.f)) * fexp(-sc);
                    ld[t] -= sc;
                }
            }
        }
#pragma unroll
        for (int t = 0; t < TILES; ++t) {
            float l = ld[t];
            if (feat)
#pragma unroll
                for (int i = 0; i < 4; ++i) // log v (1 - v) = -softplus(-z) - softplus(z)
                    l -= softplus2(z[t][i]);
            l = sample_sum(l);
            if (valid[t] && g == 0) {
                if (a.logq_out)
                    a.logq_out[idx[t]] = l;
                if (a.invq_out)
                    a.invq_out[idx[t]] = 1. / (a.alpha * (double)fexp(l) + (1. - a.alpha));
            }
        }
    }
}

// ---- backward (training) -----------------------------------------------------
// loss per sample: log q(u) - log(f(u) + eps); gz = dloss/dz at the flow
// output.  Walks the layers top-down, recomputing each MLP from the saved
// layer input, and stores the bf16 activations and deltas for the batch
// weight-gradient products, by tiles of 16 samples: [layer][tile][19 row
// blocks][16 samples][16 rows], so that a wavefront stores a row block's 512
// bytes as its lanes hold them.  Bound by those stores (239 MB for a batch of
// 65 536, 35 us at the rate of a fill) and the latency of a layer's products,
// which four wavefronts per SIMD of one tile each share: 51 us; at two of two
// tiles 74; at one of four, with 2-byte stores row by row and the weights read
// and transposed by 2 bytes, 150.
//
constexpr int BWD_TILES = 1, BWD_WAVES = 16, SAVE_BLOCKS = SAVE_F / 16;
template <int TILES>
__global__ __launch_bounds__(64 * BWD_WAVES) __attribute__((amdgpu_waves_per_eu(4, 4))) void flow_backward_kernel(FlowBackArgs a)
{
    constexpr int THREADS = 64 * BWD_WAVES, CHUNK = BWD_WAVES * TILES * 16;
    constexpr int N = sizeof(LdsLayer) / 16, PER = (N + THREADS - 1) / THREADS;
    __shared__ __attribute__((aligned(16))) LdsLayer s;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, g = lane >> 4;
    const uint4 *img = static_cast<const uint4 *>(a.wimg);
    for (uint64_t base = (uint64_t)blockIdx.x * CHUNK; base < a.n; base += (uint64_t)gridDim.x * CHUNK) {
        f4 gz[TILES];
        bool valid[TILES];
        uint64_t idx[TILES];
        uint4 next[PER]; // the next layer's weights, loaded beside the products of this one
        auto fetch = [&](int l) {
#pragma unroll
            for (int k = 0; k < PER; ++k)
                next[k] = img[l * N + min((int)threadIdx.x + THREADS * k, N - 1)];
        };
        fetch(L - 1);
#pragma unroll
        for (int t = 0; t < TILES; ++t) {
            idx[t] = base + (uint64_t)(wave * TILES + t) * 16 + (lane & 15);
            valid[t] = idx[t] < a.n;
            gz[t] = valid[t] ? *reinterpret_cast<const f4 *>(a.gz + 16 * idx[t] + 4 * g) : (f4){0.f, 0.f, 0.f, 0.f};
        }
        for (int l = L - 1; l >= 0; --l) {
            __syncthreads();
#pragma unroll
            for (int k = 0; k < PER; ++k)
                if ((int)threadIdx.x + THREADS * k < N)
                    reinterpret_cast<uint4 *>(&s)[threadIdx.x + THREADS * k] = next[k];
            __syncthreads();
            if (l > 0)
                fetch(l - 1);
            const uint32_t cond = COND_MASK[l];
            const CondMask cm = cond_mask(cond);
#pragma unroll 1
            for (int t = 0; t < TILES; ++t) {
                asm volatile("" ::: "memory"); // weights come from LDS for each tile: kept over them they spill
                f4 zin = valid[t] ? *reinterpret_cast<const f4 *>(a.zsave + ((size_t)l * a.n + idx[t]) * 16 + 4 * g)
                                  : (f4){0.f, 0.f, 0.f, 0.f};
                // rows row0 + 4g .. + 3 of this lane's sample, stored as soon as
                // they are formed (short live ranges)
                const bool ok = valid[t];
                s4 *sv = reinterpret_cast<s4 *>(a.save) +
                         ((size_t)l * (a.n / 16) + idx[t] / 16) * (SAVE_BLOCKS * 64) + 4 * (lane & 15) + g;
                auto put = [&](int row0, s4 v) {
                    if (ok)
                        sv[row0 * 4] = v;
                };
                MlpFwd r;
                mlp_forward(s, masked(zin, cm), r);
                put(SAVE_A, r.a);
#pragma unroll
                for (int mb = 0; mb < 4; ++mb) {
                    put(SAVE_H1 + 16 * mb, r.h1[mb]);
                    put(SAVE_H2 + 16 * mb, r.h2[mb]);
                }
                f4 ob0, ob1, zb;
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    const int j = 4 * g + i;
                    const bool tr = transformed(cond, j);
                    const float th = ftanh(r.o0[i]);
                    const float es = fexp(FLOW_SCALE * th);
                    const float sbar = gz[t][i] * zin[i] * es - 1.f; // the -sum s term of log q
                    const float o = sbar * FLOW_SCALE * (1.f - th * th), z = gz[t][i] * es;
                    ob0[i] = tr ? o : 0.f;
                    ob1[i] = tr ? gz[t][i] : 0.f;
                    zb[i] = tr ? z : j < D ? gz[t][i] : 0.f;
                }
                const s4 obb0 = pack4(ob0), obb1 = pack4(ob1);
                put(SAVE_OB, obb0);
                put(SAVE_OB + 16, obb1);
                const f4 zero = {0.f, 0.f, 0.f, 0.f};
                s4 h2b[4], h1b[4];
#pragma unroll
                for (int mb = 0; mb < 4; ++mb) {
                    f4 c = mfma(atile(s.wt + L_W3T, S_W3T, mb, 0), obb0, zero);
                    c = mfma(atile(s.wt + L_W3T, S_W3T, mb, 1), obb1, c);
#pragma unroll
                    for (int i = 0; i < 4; ++i)
                        c[i] *= r.h2d[mb][i];
                    h2b[mb] = pack4(c);
                    put(SAVE_H2B + 16 * mb, h2b[mb]);
                }
#pragma unroll
                for (int mb = 0; mb < 4; ++mb) {
                    f4 c = zero;
#pragma unroll
                    for (int kb = 0; kb < 4; ++kb)
                        c = mfma(atile(s.wt + L_W2T, S_W2T, mb, kb), h2b[kb], c);
#pragma unroll
                    for (int i = 0; i < 4; ++i)
                        c[i] *= r.h1d[mb][i];
                    h1b[mb] = pack4(c);
                    put(SAVE_H1B + 16 * mb, h1b[mb]);
                }
                f4 ab = zero;
#pragma unroll
                for (int kb = 0; kb < 4; ++kb)
                    ab = mfma(atile(s.wt + L_W1T, S_W1T, 0, kb), h1b[kb], ab);
#pragma unroll
                for (int i = 0; i < 4; ++i)
                    if (conditioning(cond, 4 * g + i))
                        zb[i] += ab[i];
                gz[t] = zb;
            }
        }
        if (a.gv)
#pragma unroll
            for (int t = 0; t < TILES; ++t)
                if (valid[t])
                    *reinterpret_cast<f4 *>(a.gv + 16 * idx[t] + 4 * g) = gz[t];
    }
}

// ---- batch weight and bias gradients -----------------------------------------
// dW[m][k] = inv_n sum_n delta[m][n] act[k][n] and db[m] = inv_n sum_n delta[m][n]
// on MFMA, with the sample index as the reduction dimension.  One 256-thread
// block per (layer, sample range): chunks of 64 samples of all 304 saved rows
// are staged through LDS (the next chunk is loaded into registers while the
// current one is multiplied), so every saved value is read from HBM once, and
// that read is what bounds the kernel (48 us for 65 536 samples, 5.0 TB/s).  A
// row block of 16 samples lies there sample by sample; the transposing LDS read gives lane 16 g + r row r's
// samples 4g .. 4g + 3, the operand layout of the products.
// The layer's 38 output tiles -- 28 weight tiles and 10 bias tiles, whose
// B operand is a column of ones -- are spread over the four wavefronts by the
// row blocks of their deltas, so that a wavefront reads three of those and
// seven row blocks of activations for its ten products.  Each
// block writes partial sums for all of its layer's parameters, and
// flow_grad_reduce_kernel adds the partials of each parameter in block order,
// so the result does not depend on scheduling.
constexpr int GR_CHUNK = 64, GR_TILE_BYTES = SAVE_BLOCKS * 512;
constexpr int GR_PIECES = GR_CHUNK / 16 * GR_TILE_BYTES / 16, GR_LOADS = (GR_PIECES + 255) / 256;
constexpr int GR_MIN_CHUNKS = 8, GR_MAX_SPLIT = 128;

// Sample-range blocks per layer for n samples.
static int wgrad_split(uint64_t n)
{
    const uint64_t chunks = (n + GR_CHUNK - 1) / GR_CHUNK;
    const uint64_t s = (chunks + GR_MIN_CHUNKS - 1) / GR_MIN_CHUNKS;
    return (int)(s < 1 ? 1 : s > GR_MAX_SPLIT ? GR_MAX_SPLIT : s);
}

// Mean over the batch of log q - log(f + eps) by one workgroup of 256 threads,
// in a fixed order: 1024 strided sums of 4-wide loads, then a tree.
__device__ __forceinline__ void batch_loss(const FlowLossArgs &a, uint64_t n, double *red)
{
    const uint64_t n4 = n / 4;
    const float4 *q4 = reinterpret_cast<const float4 *>(a.logq), *f4p = reinterpret_cast<const float4 *>(a.logf);
    for (uint32_t v = threadIdx.x; v < 1024; v += 256) {
        double acc = 0.;
#pragma unroll 8
        for (uint64_t i = v; i < n4; i += 1024) {
            const float4 q = q4[i], f = f4p[i];
            acc += (((double)q.x - (double)f.x) + ((double)q.y - (double)f.y)) +
                   (((double)q.z - (double)f.z) + ((double)q.w - (double)f.w));
        }
        for (uint64_t i = 4 * n4 + v; i < n; i += 1024)
            acc += (double)a.logq[i] - (double)a.logf[i];
        red[v] = acc;
    }
    __syncthreads();
    for (uint32_t o = 512; o > 0; o >>= 1) {
        for (uint32_t v = threadIdx.x; v < o; v += 256)
            red[v] += red[v + o];
        __syncthreads();
    }
    if (threadIdx.x == 0)
        *a.out = (float)(red[0] / (double)n);
}

__global__ __launch_bounds__(256) void flow_wgrad_kernel(const uint16_t *save, uint64_t n, int split, float *part,
                                                         FlowLossArgs loss)
{
    __shared__ __attribute__((aligned(16))) uint16_t lds[GR_CHUNK / 16 * GR_TILE_BYTES / 2];
    const int layer = blockIdx.x / split, ks = blockIdx.x % split;
    if (layer == L) { // one block more where the training step's loss is wanted
        batch_loss(loss, n, reinterpret_cast<double *>(lds));
        return;
    }
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, g = lane >> 4, r16 = lane & 15;
    const uint64_t chunks = (n + GR_CHUNK - 1) / GR_CHUNK, per = (chunks + split - 1) / split;
    const uint64_t c0 = (uint64_t)ks * per, c1 = c0 + per < chunks ? c0 + per : chunks;
    // n is a multiple of 16: whole tiles
    const uint64_t pieces = n / 16 * (GR_TILE_BYTES / 16);
    const uint4 *sv = reinterpret_cast<const uint4 *>(save) + (size_t)layer * pieces;
    uint4 buf[GR_LOADS];
    auto load = [&](uint64_t c) {
#pragma unroll
        for (int k = 0; k < GR_LOADS; ++k) {
            const int p = threadIdx.x + 256 * k;
            const uint64_t at = c * GR_PIECES + p;
            buf[k] = make_uint4(0u, 0u, 0u, 0u);
            if (p < GR_PIECES && at < pieces)
                buf[k] = sv[at];
        }
    };
    // The wavefront's products: b1, W1 (with a) of row block H1B + wave, b2, W2
    // (with h1's four) of H2B + wave, b3 and W3 (with two of h2's) of OB.
    f4 acc[10];
#pragma unroll
    for (int j = 0; j < 10; ++j)
        acc[j] = (f4){0.f, 0.f, 0.f, 0.f};
    const short one = (short)0x3F80; // bf16 1.0
    const s4 ones = {one, one, one, one};
    const int ob = wave & 1, h2 = 2 * (wave >> 1);
    if (c0 < c1)
        load(c0);
    for (uint64_t c = c0; c < c1; ++c) {
        __syncthreads(); // the previous chunk's products are done
#pragma unroll
        for (int k = 0; k < GR_LOADS; ++k) {
            const int p = threadIdx.x + 256 * k;
            if (p < GR_PIECES)
                reinterpret_cast<uint4 *>(lds)[p] = buf[k];
        }
        __syncthreads();
        if (c + 1 < c1)
            load(c + 1);
#pragma unroll
        for (int kk = 0; kk < GR_CHUNK / 16; ++kk) {
            typedef __attribute__((address_space(3))) s4 lds_s4;
            uint16_t *tile = lds + kk * (GR_TILE_BYTES / 2) + 4 * lane;
            auto rows = [&](int row0) { // row block row0 / 16
                return __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s4 *)(tile + 16 * row0));
            };
            const s4 d1 = rows(SAVE_H1B + 16 * wave), d2 = rows(SAVE_H2B + 16 * wave), d3 = rows(SAVE_OB + 16 * ob);
            acc[0] = mfma(d1, ones, acc[0]);
            acc[1] = mfma(d1, rows(SAVE_A), acc[1]);
            acc[2] = mfma(d2, ones, acc[2]);
#pragma unroll
            for (int kb = 0; kb < 4; ++kb)
                acc[3 + kb] = mfma(d2, rows(SAVE_H1 + 16 * kb), acc[3 + kb]);
            acc[7] = mfma(d3, ones, acc[7]);
#pragma unroll
            for (int kb = 0; kb < 2; ++kb)
                acc[8 + kb] = mfma(d3, rows(SAVE_H2 + 16 * (h2 + kb)), acc[8 + kb]);
        }
    }
    float *pl = part + ((size_t)ks * L + layer) * LP;
    auto weights = [&](int off, int ld, f4 v) { // C layout: lane holds rows 4g.. of column r16
#pragma unroll
        for (int i = 0; i < 4; ++i)
            pl[off + (4 * g + i) * ld + r16] = v[i];
    };
    auto bias = [&](int off, f4 v) {
        if (r16 == 0)
#pragma unroll
            for (int i = 0; i < 4; ++i)
                pl[off + 4 * g + i] = v[i];
    };
    bias(OFF_B1 + 16 * wave, acc[0]);
    weights(OFF_W1 + 16 * wave * DP, DP, acc[1]);
    bias(OFF_B2 + 16 * wave, acc[2]);
#pragma unroll
    for (int kb = 0; kb < 4; ++kb)
        weights(OFF_W2 + 16 * wave * H + 16 * kb, H, acc[3 + kb]);
    if (wave < 2)
        bias(OFF_B3 + 16 * ob, acc[7]);
#pragma unroll
    for (int kb = 0; kb < 2; ++kb)
        weights(OFF_W3 + 16 * ob * H + 16 * (h2 + kb), H, acc[8 + kb]);
}

// grad[i] = inv_n sum over the sample-range blocks, in block order (loads
// in groups of 32 so that they are in flight together), and in training the
// parameter's Adam step from it.
__device__ __forceinline__ LdsLayer &weight_image(void *wimg, int i) { return static_cast<LdsLayer *>(wimg)[i / LP]; }
template <bool ADAM>
__global__ __launch_bounds__(256) void flow_grad_reduce_kernel(const float *part, int split, float inv_n, float *grad,
                                                               FlowAdamArgs a)
{
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= NPARAM)
        return;
    float sum = 0.f;
    for (int k0 = 0; k0 < split; k0 += 32) {
        float v[32];
#pragma unroll
        for (int j = 0; j < 32; ++j)
            v[j] = k0 + j < split ? part[(size_t)(k0 + j) * NPARAM + i] : 0.f;
#pragma unroll
        for (int j = 0; j < 32; ++j)
            sum += v[j];
    }
    const float gi = sum * inv_n;
    grad[i] = gi;
    if constexpr (ADAM) {
        const float mi = a.beta1 * a.m[i] + (1.f - a.beta1) * gi;
        const float vi = a.beta2 * a.v[i] + (1.f - a.beta2) * gi * gi;
        a.m[i] = mi;
        a.v[i] = vi;
        const float mh = mi / (1.f - powf(a.beta1, (float)a.step)), vh = vi / (1.f - powf(a.beta2, (float)a.step));
        const float wi = a.w[i] - a.lr * mh / (sqrtf(vh) + a.eps);
        a.w[i] = wi;
        put_weight(weight_image(a.wimg, i), i % LP, f2bf(wi));
    }
}

__global__ void flow_to_bf16_kernel(const float *w, void *wimg)
{
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < NPARAM)
        put_weight(weight_image(wimg, i), i % LP, f2bf(w[i]));
}

// ---- launchers ---------------------------------------------------------------
// Resident-weight kernels: one pass per block covers FWD_WAVES * TILES * 16
// samples; at most max_blocks blocks (one per CU), striding over the rest.
template <int TILES, int WAVES> static unsigned grid_resident(const FlowKernelArgs &a)
{
    const uint64_t chunk = (uint64_t)WAVES * TILES * 16, need = (a.n + chunk - 1) / chunk;
    const uint64_t cap = a.max_blocks ? a.max_blocks : need;
    return (unsigned)std::max<uint64_t>(1, std::min(need, cap));
}

void launch_flow_forward(const FlowKernelArgs &a, hipStream_t st)
{
    if (a.n < FWD_SMALL_N)
        hipLaunchKernelGGL((flow_forward_kernel<FWD_TILES_SMALL, FWD_WAVES_SMALL>),
                           dim3(grid_resident<FWD_TILES_SMALL, FWD_WAVES_SMALL>(a)), dim3(64 * FWD_WAVES_SMALL), 0, st, a);
    else
        hipLaunchKernelGGL((flow_forward_kernel<FWD_TILES, FWD_WAVES>), dim3(grid_resident<FWD_TILES, FWD_WAVES>(a)),
                           dim3(64 * FWD_WAVES), 0, st, a);
}

void launch_flow_inverse(const FlowKernelArgs &a, hipStream_t st)
{
    if (a.n < FWD_SMALL_N)
        hipLaunchKernelGGL((flow_inverse_kernel<FWD_TILES_SMALL, FWD_WAVES_SMALL>),
                           dim3(grid_resident<FWD_TILES_SMALL, FWD_WAVES_SMALL>(a)), dim3(64 * FWD_WAVES_SMALL), 0, st, a);
    else
        hipLaunchKernelGGL((flow_inverse_kernel<FWD_TILES, FWD_WAVES>), dim3(grid_resident<FWD_TILES, FWD_WAVES>(a)),
                           dim3(64 * FWD_WAVES), 0, st, a);
}

void launch_flow_backward(const FlowBackArgs &a, hipStream_t st)
{
    constexpr uint64_t chunk = BWD_WAVES * BWD_TILES * 16;
    hipLaunchKernelGGL(flow_backward_kernel<BWD_TILES>, dim3((unsigned)((a.n + chunk - 1) / chunk)), dim3(64 * BWD_WAVES), 0,
                       st, a);
}

size_t flow_wgrad_part_bytes(uint64_t n) { return (size_t)wgrad_split(n) * NPARAM * sizeof(float); }

void launch_flow_wgrad(const uint16_t *save, uint64_t n, float inv_n, float *part, float *grad, const FlowLossArgs *loss,
                       const FlowAdamArgs *adam, hipStream_t st)
{
    const int split = wgrad_split(n);
    hipLaunchKernelGGL(flow_wgrad_kernel, dim3(L * split + (loss ? 1 : 0)), dim3(256), 0, st, save, n, split, part,
                       loss ? *loss : FlowLossArgs{});
    if (adam)
        hipLaunchKernelGGL(flow_grad_reduce_kernel<true>, dim3((NPARAM + 255) / 256), dim3(256), 0, st, part, split, inv_n,
                           grad, *adam);
    else
        hipLaunchKernelGGL(flow_grad_reduce_kernel<false>, dim3((NPARAM + 255) / 256), dim3(256), 0, st, part, split, inv_n,
                           grad, FlowAdamArgs{});
}

void launch_flow_to_bf16(const float *w, void *wimg, hipStream_t st)
{
    hipLaunchKernelGGL(flow_to_bf16_kernel, dim3((NPARAM + 255) / 256), dim3(256), 0, st, w, wimg);
}

// ---- integrand and its gradient for training --------------------------------
// Physics from here on: no contraction, as in the rest of the build.
#pragma clang fp contract(off)

// f(u) = sum_c lam_c |M|^2_c(u) cut(u) from the hand-written adjoint (the
// smooth cut factor of event_adjoint when tau > 0), and
// gz = dloss/dz at the flow output for loss = log q - log(f + eps):
//   dloss/du = -(1 - 2u)/(u (1 - u)) - f'(u)/(f + eps),  dz = du * u (1 - u).
__global__ __launch_bounds__(128) void flow_integrand_kernel(tpd::Params P, double lam0, double lam1, double lam2,
                                                             double lam3, double lam4, uint64_t n, const double *u,
                                                             double eps, double tau, double fcap, int target,
                                                             float clip, float *gz, float *logf, double *f_out)
{
    const uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n)
        return;
    const tpd::AdjParams<double> A = tpd::adj_params<double>(P, 1.0);
    double uu[12], m[5], du[12], dp[12];
    const double lam[5] = {lam0, lam1, lam2, lam3, lam4};
#pragma unroll
    for (int j = 0; j < 12; ++j)
        uu[j] = u[12 * i + j];
    bool keep;
    if (target == 2)
        keep = tpd::event_adjoint<double, 2>(A, uu, lam, m, du, dp, tau, fcap);
    else if (target == 1)
        keep = tpd::event_adjoint<double, 1>(A, uu, lam, m, du, dp, tau);
    else
        keep = tpd::event_adjoint<double, 0>(A, uu, lam, m, du, dp);
    double f = 0.;
    if (keep)
        for (int c = 0; c < 5; ++c)
            f += lam[c] * m[c];
    // target 2 differentiates log f itself (du already carries the 1/f)
    const double fe = target == 2 ? (keep ? 1. : INFINITY) : f + eps;
#pragma unroll
    for (int j = 0; j < 12; ++j) {
        const double w = uu[j] * (1. - uu[j]);
        const float g = (float)(-(1. - 2. * uu[j]) - w * du[j] / fe);
        gz[16 * i + j] = fminf(fmaxf(g, -clip), clip);
    }
#pragma unroll
    for (int j = 12; j < 16; ++j)
        gz[16 * i + j] = 0.f;
    logf[i] = (float)(target == 2 ? (keep ? log(f) : -100.) : log(fe)); // dropped events: -100
    if (f_out)
        f_out[i] = f;
}

void launch_flow_integrand(const tpd::Params &P, const double lam[5], uint64_t n, const double *u, double eps,
                           double tau, double fcap, int target, float clip, float *gz, float *logf, double *f_out,
                           hipStream_t st)
{
    hipLaunchKernelGGL(flow_integrand_kernel, dim3((unsigned)((n + 127) / 128)), dim3(128), 0, st, P, lam[0], lam[1],
                       lam[2], lam[3], lam[4], n, u, eps, tau, fcap, target, clip, gz, logf, f_out);
}

} // namespace tpf
