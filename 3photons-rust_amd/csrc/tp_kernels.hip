// tp_kernels.hip -- gfx950 kernels of the 3photons event loop.
//
//  fused_kernel      one wavefront per 10 000-event batch or part of one,
//                    grid-strided over parts; uniforms from xoshiro256+ or RANF made in the
//                    loop, or read from HBM (faster-evgen, flow); RAMBO -> cuts in registers,
//                    passing events compacted through an LDS queue, spinors
//                    -> amplitudes -> weight on full wavefronts, 12 running
//                    sums per lane, butterfly reduction to one accumulator
//                    per part (batch_sums_kernel adds a batch's parts).
//  ranf_expand       RANF stream and accept bits into HBM for faster-evgen, one
//                    wavefront per segment of R rounds, 55 lanes = the 55
//                    values of a round; xo_expand, xo128_expand the same for
//                    pieces of the xoshiro streams; fe_* walk them.
//  f32_events        the all-f32 event loop, f32_accumulate its in-order sums.
//  adjoint_*         values and derivatives at given or drawn points.
//  ranf_seed         jump-mode origins, seeded_new(seed + 123456 b) per batch.
//  merge_kernel      in-order left fold of the batch accumulators.
//
// Compiled with -ffp-contract=off: nothing is fused but what the code writes as
// fma.  The f64 path keeps the reference's operation order through RAMBO and the
// sort (HadrienG2/3photons-rust src/evgen.rs); its cuts' products are fused, its
// helicity sums closed forms (evcut.rs, spinor.rs, matelems.rs), its sums taken
// per lane and part (resacc.rs).  The all-f32 path keeps the order throughout.
#include "tp_kernels.h"
#include "tp_xoshiro.h"

namespace tpk {

using namespace tpd;

struct DevAcc { // layout of tp_acc
    uint64_t selected;
    double spm2[5], vars[5], sigma, variance;
};

// ---- per-thread accumulation (resacc.rs:121-129) ---------------------------
// Sums s = (spm2[5], vars[5], sigma, variance); the mixed-precision path
// (PREC 1) keeps Kahan compensations c alongside.
template <int PREC> struct Acc {
    double s[12];
    double c[PREC ? 12 : 1];
    uint32_t n;
};

template <int PREC> __device__ __forceinline__ void acc_zero(Acc<PREC> &A)
{
#pragma unroll
    for (int j = 0; j < 12; ++j)
        A.s[j] = 0.;
#pragma unroll
    for (int j = 0; j < (PREC ? 12 : 1); ++j)
        A.c[j] = 0.;
    A.n = 0;
}

__device__ __forceinline__ void kahan(double &s, double &c, double x)
{
    double y = x - c;
    double t = s + y;
    c = (t - s) - y;
    s = t;
}

// In f64 the squares join their sums by fused multiply-adds, and the sum of
// the weights, linear in m, is formed from the sums of m at the end
// (acc_values); PREC 1 adds each of the twelve terms.
template <int PREC> __device__ __forceinline__ void acc_add(Acc<PREC> &A, const Params &P, const double m[5])
{
    const double w = weight_f64<PREC == 0>(P, m);
    A.n += 1;
    if (PREC == 0) {
#pragma unroll
        for (int k = 0; k < 5; ++k) {
            A.s[k] = A.s[k] + m[k];
            A.s[5 + k] = fma(m[k], m[k], A.s[5 + k]);
        }
        A.s[11] = fma(w, w, A.s[11]);
        return;
    }
    double x[12];
#pragma unroll
    for (int k = 0; k < 5; ++k) {
        x[k] = m[k];
        x[5 + k] = m[k] * m[k];
    }
    x[10] = w;
    x[11] = w * w;
#pragma unroll
    for (int j = 0; j < 12; ++j)
        kahan(A.s[j], A.c[PREC ? j : 0], x[j]);
}

template <int PREC> __device__ __forceinline__ void acc_values(const Acc<PREC> &A, const Params &P, double v[12])
{
#pragma unroll
    for (int j = 0; j < 12; ++j)
        v[j] = PREC ? A.s[j] - A.c[PREC ? j : 0] : A.s[j];
    if (PREC == 0)
        v[10] = weight_f64<true>(P, A.s);
}

// Fixed-shape wavefront butterfly then in-order wave combine; deterministic.
template <int NW>
__device__ __forceinline__ void block_reduce_store(double v[12], uint32_t n, DevAcc *out, double (*red)[13])
{
    const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) {
#pragma unroll
        for (int j = 0; j < 12; ++j)
            v[j] += __shfl_xor(v[j], off);
        n += __shfl_xor(n, off);
    }
    if (lane == 0) {
#pragma unroll
        for (int j = 0; j < 12; ++j)
            red[wid][j] = v[j];
        red[wid][12] = (double)n;
    }
    __syncthreads();
    if (threadIdx.x < 13) {
        const int j = threadIdx.x;
        double t = red[0][j];
#pragma unroll
        for (int w = 1; w < NW; ++w)
            t = t + red[w][j];
        if (j < 5)
            out->spm2[j] = t;
        else if (j < 10)
            out->vars[j - 5] = t;
        else if (j == 10)
            out->sigma = t;
        else if (j == 11)
            out->variance = t;
        else
            out->selected = (uint64_t)t;
    }
    __syncthreads();
}

// ---- RANF rounds -----------------------------------------------------------
constexpr int32_t MODULO = 1000000000;

// One RANF round in closed form (lane i - 1 holds X[i], i = 1..55):
//   i <= 24:  X'[i] = X[i] - X[i+31]
//   25..48:   X'[i] = X[i] - X'[i-24] = X[i] - X[i-24] + X[i+7]
//   49..55:   X'[i] = X[i] - X[i-24] + X[i-48] - X[i-17]
// (ranf.rs:106-119 applies the first two lines as in-place updates; the third
// is the second with X'[i-24] expanded once more), all mod 1e9.  Every lane
// evaluates (X[i] - b) + (c - d) with b, c, d read from other lanes of the
// same wave by ds_bpermute (no LDS storage, no barrier).  Lanes 55..63 hold 0
// and keep it, so a term a case does not have reads lane 63; each value is the
// unique representative in [0, 1e9), so the sum order does not matter.  The
// whole wave must be active: one wave holds one window.
__device__ __forceinline__ uint32_t mod_sub(uint32_t a, uint32_t b) // (a - b) mod 1e9, a, b in [0, 1e9)
{
    const uint32_t t = a - b;
    return min(t, t + (uint32_t)MODULO);
}
struct RanfLanes { // byte addresses for ds_bpermute of the lanes a lane reads
    int b, c, d;
};
__device__ __forceinline__ RanfLanes ranf_lanes()
{
    const int lane = (int)(threadIdx.x & 63u), i = lane + 1;
    const bool live = lane < 55;
    RanfLanes l;
    l.b = (live ? (i <= 24 ? i + 30 : i - 25) : 63) << 2;          // X[i+31] or X[i-24]
    l.c = (live && i > 24 ? (i <= 48 ? i + 6 : i - 49) : 63) << 2; // X[i+7] or X[i-48]
    l.d = (live && i > 48 ? i - 18 : 63) << 2;                     // X[i-17]
    return l;
}
__device__ __forceinline__ int32_t ranf_next_round(int32_t x, const RanfLanes &l)
{
    const uint32_t wb = (uint32_t)__builtin_amdgcn_ds_bpermute(l.b, x);
    const uint32_t wc = (uint32_t)__builtin_amdgcn_ds_bpermute(l.c, x);
    const uint32_t wd = (uint32_t)__builtin_amdgcn_ds_bpermute(l.d, x);
    const uint32_t v = mod_sub((uint32_t)x, wb) + mod_sub(wc, wd); // [0, 2e9)
    return (int32_t)min(v, v - (uint32_t)MODULO);
}

// X_{r+m} from X_r with c = x^(55 m) mod P: X_{r+m}[i] = sum_k c_k Y[i-1+k]
// over the window Y = (X_r, X_{r+1}).  Lane k holds c_k, so that a term waits
// for no memory but its LDS read, and those are in flight together: a part's
// start in the event loop takes some 3 us less than with the coefficients read
// term by term (closure of 10 000 events 35 -> 26 us, 1e7 events 330 -> 307).
__device__ __forceinline__ uint32_t ranf_jump_lane(const uint32_t *c) { return (threadIdx.x & 63u) < 55 ? c[threadIdx.x & 63u] : 0u; }
__device__ __forceinline__ int32_t ranf_jump(int32_t x, uint32_t ck, int32_t *win)
{
    const int lane = threadIdx.x & 63;
    int32_t nx = ranf_next_round(x, ranf_lanes());
    if (lane < 55) {
        win[lane] = x;
        win[55 + lane] = nx;
    }
    __syncthreads();
    const int32_t *w = win + (lane < 55 ? lane : 0);
    uint64_t acc = 0;
#pragma unroll
    for (int k0 = 0; k0 < 55; k0 += 16) {
        uint32_t y[16];
#pragma unroll
        for (int k = 0; k < 16; ++k)
            y[k] = k0 + k < 55 ? (uint32_t)w[k0 + k] : 0u;
#pragma unroll
        for (int k = 0; k < 16; ++k)
            if (k0 + k < 55)
                acc += (uint64_t)(uint32_t)__builtin_amdgcn_readlane((int)ck, k0 + k) * y[k];
        acc %= (uint64_t)MODULO; // 16 products and a rest stay below 2^64
    }
    __syncthreads();
    return lane < 55 ? (int32_t)acc : 0;
}

// X_{r+e} from X_r for a number of rounds e all lanes hold alike.  win: 110
// ints of LDS, free before and after.  A digit's coefficients are loaded beside
// the jump before it.
__device__ __forceinline__ int32_t ranf_advance(int32_t x, const uint32_t *__restrict__ r16, uint64_t e, int32_t *win)
{
    auto seek = [&]() { // to the next digit that is not 0
        while (e && !(e & 15u)) {
            e >>= 4;
            r16 += 15 * 55;
        }
    };
    auto coefficients = [&]() { return e ? ranf_jump_lane(r16 + 55 * ((uint32_t)(e & 15u) - 1)) : 0u; };
    seek();
    uint32_t ck = coefficients();
    while (e) {
        const uint32_t now = ck;
        e >>= 4;
        r16 += 15 * 55;
        seek();
        ck = coefficients();
        x = ranf_jump(x, now, win);
    }
    return x;
}

// A stream seeded past the modulus (faster-threading's seed + 123456 b does in
// long runs) holds values outside [0, 1e9) in its first rounds, an odd stream.
// Rounds and jumps don't commute there, so jumps are taken to whole segments of
// RANF_LATE rounds only, each straight from round 0, and rounds to every other
// place: the values don't depend on how the stream is split.
__device__ __forceinline__ bool ranf_odd(int32_t x) { return __any((uint32_t)x >= (uint32_t)MODULO); }
// Round RANF_LATE seg of an odd stream from its round 0: first the jump by the
// lowest binary digit of seg (the rounds it leads to are in range, and further
// jumps may be taken in any steps).  win: 110 ints of LDS, free before and after.
__device__ __forceinline__ int32_t ranf_odd_segment(int32_t x, const uint32_t *__restrict__ r16, uint64_t seg, int32_t *win)
{
    static_assert(RANF_LATE == 1u << 11, "seg's binary digit k is digit 11 + k of the rounds");
    if (!seg)
        return x;
    const uint32_t bit = 11u + (uint32_t)__builtin_ctzll(seg);
    x = ranf_jump(x, ranf_jump_lane(r16 + 55 * (15 * (bit / 4) + (1u << bit % 4) - 1)), win);
    return ranf_advance(x, r16, RANF_LATE * (seg & (seg - 1)), win);
}

// What bounds a round: a chain of one LDS permute and nine dependent integer
// instructions, about 180 cycles, which three wavefronts per SIMD hide behind
// the events (14 rounds of about 48 issue cycles for 64 events of 2500).
// Against a stream expanded into HBM first, 48 bytes an event written and read
// again: 1e9 events 43.4 -> 28.3 ms with the event loop's own gains, the
// expansion having been 10.4 ms of them; 1e7 events 586 -> 414 us.
//
// ODD: the run has streams with values outside [0, 1e9) (RanfSource::later),
// in kernels of their own: the places where such a stream's jumps may go cost
// every other run 2 % in the all-f32 loop, whose registers are full (1e7 events
// 395 us without them, 410 with).
template <bool ODD> struct RanfPart {
    int32_t x = 0;        // lane l: X[l + 1] of the current round
    uint32_t o = 0;       // the place of the next unread value in it: X[55 - o], o up to 55
    uint64_t round = 0;   // the number of the last round the part reads
    bool have = false;
    uint32_t late = 0;    // ODD: rounds to the next segment of RANF_LATE in an odd stream, otherwise more than the part's
    uint32_t next = 0;    // ODD: the row of RanfSource::later where it starts
    RanfLanes l = ranf_lanes();

    // To the first draw of n > 0 events from event `first` of batch b on.  win:
    // 110 ints of LDS, free before and after.
    __device__ __forceinline__ void start(const RanfSource &R, uint64_t b, uint32_t batch_size, uint32_t first,
                                          uint32_t n, int32_t *win)
    {
        const bool own = R.origin && b > 0;
        const uint64_t q = (own ? 0 : R.p0) + 12ull * (first + (R.origin ? 0 : b * batch_size));
        uint64_t skip = q / 55;
        if (!ODD && have && R.jump_rounds && round + R.jump_rounds <= skip) { // on from the previous part
            x = ranf_jump(x, ranf_jump_lane(R.jump), win);
            skip -= round + R.jump_rounds;
        } else {
            const uint32_t lane = threadIdx.x & 63u;
            x = lane < 55 ? (own ? R.origin[56 * (b - R.first) + lane + 1] : R.round[lane + 1]) : 0;
        }
        late = 0x7fffffffu;
        if (ODD && ranf_odd(x)) {
            const uint64_t seg = skip / RANF_LATE;
            skip %= RANF_LATE;
            late = RANF_LATE - (uint32_t)skip;
            next = (uint32_t)((R.origin ? b : seg) - R.first); // (with jump seeding one row serves the batch)
            if (seg)
                x = later(R);
            else
                for (; skip; --skip)
                    x = ranf_next_round(x, l);
            next += R.origin ? 0 : 1;
        }
        if (skip < 4) // (a round costs a twentieth of a jump)
            for (; skip; --skip)
                x = ranf_next_round(x, l);
        x = ranf_advance(x, R.r16, skip, win);
        o = (uint32_t)(q % 55);
        round = (q + 12ull * n - 1) / 55;
        have = true;
    }
    __device__ __forceinline__ int32_t later(const RanfSource &R) const
    {
        uint32_t lane = threadIdx.x & 63u;
        asm volatile("" : "+v"(lane)); // (its address is formed here, not kept in registers over the events)
        return lane < 55 ? R.later[56 * (uint64_t)next + lane + 1] : 0;
    }
    // The next `need` (12 .. 768) values into lds[base ..] in stream
    // order.  Lanes with nothing to write do so to lds[dump].
    __device__ __forceinline__ void fill(const RanfSource &R, uint32_t need, int32_t *lds, uint32_t base, uint32_t dump)
    {
        const int lane = (int)(threadIdx.x & 63u), at = 54 - lane - (int)o;
        lds[lane < 55 && at >= 0 ? base + (uint32_t)at : dump] = x;
        uint32_t p = lane < 55 ? base + (uint32_t)(at + 55) : dump;
        const uint32_t step = lane < 55 ? 55u : 0u, rounds = (o + need + 54) / 55 - 1;
        if (ODD && __builtin_expect(late <= rounds, 0)) { // the next segment starts among them (no two do)
            for (uint32_t r = 1; r <= rounds; ++r) {
                x = r == late ? later(R) : ranf_next_round(x, l);
                lds[p < base + need ? p : dump] = x;
                p += step;
            }
            late += RANF_LATE - rounds;
            next += R.origin ? 0 : 1;
            o = o + need - 55 * rounds;
            return;
        }
        if (ODD)
            late -= rounds;
        for (uint32_t r = 1; r < rounds; ++r) {
            x = ranf_next_round(x, l);
            lds[p] = x;
            p += step;
        }
        if (rounds) { // the last one may reach past `need`
            x = ranf_next_round(x, l);
            lds[p < base + need ? p : dump] = x;
        }
        o = o + need - 55 * rounds;
    }
};

// ---- the fused event loop ------------------------------------------------
//
// One wavefront per part of a batch, persistent: the grid holds as many
// wavefronts as are resident and each strides over parts.  Each iteration every lane generates one event
// (uniforms -> RAMBO -> cuts); the photon momenta of the events
// that pass are appended to a queue in LDS (ballot + prefix count), and whenever 64
// are queued the whole wavefront takes them and evaluates the helicity sums
// and weights on full lanes.  Cut events therefore cost no amplitude work, and
// the amplitude code never runs with masked-off lanes except for the final
// partial flush of a part.  The accumulation order is the queue order, a
// function of the data only, so results are reproducible run to run.
//
// Event assignment inside the part: with the in-register xoshiro stream each
// lane owns a contiguous run (one skip-ahead per run); the others take events
// l, l+64, ... in lane l.  The RANF stream is made by the wavefront as a whole,
// 55 values a round, into LDS (RanfPart), where each lane picks its event's 12
// values; values read from HBM then lie side by side across the lanes.
//
// What bounds it: VALU issue, at the measured issue times (f64 fma 4.9 cycles,
// add and mul 4.4, rcp and rsq 16.3, xor, mov and add_u32 2.7, shifts and
// three-operand integer instructions 4.4) about 90 % busy at 1e9 events; one
// wavefront per batch left a run of 1e7 events with one wavefront per SIMD of
// the three that fit and a closure call with one on the whole chip, most of
// whose time was the lanes' own skips of the stream (a call of 4321 events
// 381 -> 25 us, 1.23e6 events with jump seeding 677 -> 78 us, 1e9 events
// 26.8 -> 25.4 ms with parts and shared skips).
constexpr int QCAP = 128;

// Three wavefronts per SIMD (167 VGPRs at f64, no scratch): the LDS queue
// (12.4 KB per workgroup) caps a CU at 12 resident workgroups anyway, and the
// third wave hides the transcendental-table, LDS and f64 latencies better than
// two (measured 3 % faster at f64).
// The run constants re-read from the kernel-argument segment (FusedArgs::P
// sits at its start) through a pointer the compiler cannot see through, at
// each use site: scalar loads, which cost no VALU slot, instead of ~40 SGPRs
// held across the whole event loop, which the allocator spills to VGPR lanes
// and reads back with one VALU v_readlane per dword.
static_assert(offsetof(FusedArgs, P) == 0, "Params first in FusedArgs");
typedef const __attribute__((address_space(4))) Params KParams;
__device__ __forceinline__ const Params &fresh_params()
{
    KParams *k = (KParams *)__builtin_amdgcn_kernarg_segment_ptr();
    asm volatile("" : "+s"(k));
    return *(const Params *)k;
}

template <int SOURCE, int PREC, bool ODD = false>
__global__ __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(3, 8))) void fused_kernel(FusedArgs a)
{
    // momenta, structure of arrays, slots 0..63 and 64..127; between
    // iterations fewer than 64 events wait, so with the RANF source the upper
    // half holds an iteration's draws until its events are pushed
    __shared__ __align__(16) double queue[2][12][64];
    auto slot_of = [&](uint32_t s) -> double * { return &queue[0][0][0] + (s >> 6) * (12 * 64) + (s & 63u); };
    int32_t *const qints = reinterpret_cast<int32_t *>(&queue[0][0][0]);
    constexpr uint32_t RING = 2 * 12 * 64, RING_DUMP = RING + 768; // of the upper half's 1536 ints
    __shared__ uint32_t qev[SOURCE == 2 ? QCAP : 1]; // weighted source: the event's index in the chunk
    __shared__ double red[1][13];
    const uint32_t lane = threadIdx.x;
    const uint64_t lanemask_lt = (1ull << lane) - 1ull;
    uint64_t sw[4] = {a.s0[0], a.s0[1], a.s0[2], a.s0[3]}; // xoshiro state at the part's first draw (uniform)
    RanfPart<ODD> ranf;
    bool have = false;
    for (uint64_t t = blockIdx.x; t < a.nb * a.parts; t += gridDim.x) {
        const uint64_t lb = a.parts == 1 ? t : t / a.parts;
        const uint32_t first = (uint32_t)(t - lb * a.parts) * 64u * a.run; // the part's first event in the batch
        const uint64_t b = a.b_first + lb;
        const uint64_t left = a.num_events - b * a.batch_size;
        const uint32_t nbatch = left < a.batch_size ? (uint32_t)left : a.batch_size;
        const uint32_t n = first < nbatch ? min(nbatch - first, 64u * a.run) : 0u;
        uint32_t len, iters;
        uint64_t s[4] = {0, 0, 0, 0};
        if (SOURCE == 0) {
            len = lane * a.run < n ? min(n - lane * a.run, a.run) : 0u;
            iters = min(n, a.run);
            // every part of this wavefront has the same place in its batch
            // (the grid is a multiple of `parts` wherever it strides)
            xo_advance_uniform(a.b16, have ? gridDim.x / a.parts : b, sw);
            if (!have)
                xo_advance_uniform(a.m16, 12ull * first, sw);
            have = true;
            xo_lane_states(a.lanes, sw, s);
        } else {
            len = n / 64 + (lane < n % 64 ? 1u : 0u); // events lane, lane+64, ...
            iters = (n + 63) / 64;
        }
        if (SOURCE == 1 && n)
            ranf.start(a.ranf, b, a.batch_size, first, n, qints + RING);
        const size_t wbase = (size_t)lb * a.batch_size + first;
        const RerollBits rb{a.acc1, a.bbase, a.bstride ? (lb + 1) * a.bstride : a.blimit};
        Acc<PREC> A;
        acc_zero(A);
        uint32_t qn = 0; // queued events (uniform)
        // faster-evgen: the lane's next event start, loaded an event ahead
        constexpr bool FE = SOURCE == 3 || SOURCE == 4;
        uint64_t qnext = FE && len > 0 ? a.evq[wbase + lane] : 0;
        for (uint32_t k = 0; k < iters; ++k) {
            bool pass = false;
            double p[3][4];
            const uint64_t qk = qnext;
            if (FE && k + 1 < len)
                qnext = a.evq[wbase + (size_t)((k + 1) * 64 + lane)];
            int4 rd[3]; // RANF: the lane's 12 draws
            if (SOURCE == 1) {
                ranf.fill(a.ranf, 12 * min(64u, n - 64 * k), qints, RING, RING_DUMP);
                __syncthreads();
#pragma unroll
                for (int j = 0; j < 3; ++j)
                    rd[j] = reinterpret_cast<const int4 *>(qints + RING)[3 * lane + j];
                __syncthreads(); // read before the events are pushed
            }
            if (k < len && SOURCE == 3) {
                RanfWalk w{a.draws, a.qbase, qk, rb};
                pass = generate_faster_f64(fresh_params(), w, p);
            } else if (k < len && SOURCE == 4) {
                XoWalk w{a.xdraws, a.qbase, qk, rb};
                pass = generate_faster_f64(fresh_params(), w, p);
            } else if (k < len) {
                double u[12];
                if (SOURCE == 0) {
#pragma unroll
                    for (int j = 0; j < 12; ++j)
                        u[j] = xo_uniform64(s);
                } else if (SOURCE == 1) {
#pragma unroll
                    for (int j = 0; j < 3; ++j) {
                        u[4 * j] = (double)rd[j].x * 1e-9;
                        u[4 * j + 1] = (double)rd[j].y * 1e-9;
                        u[4 * j + 2] = (double)rd[j].z * 1e-9;
                        u[4 * j + 3] = (double)rd[j].w * 1e-9;
                    }
                } else {
                    const size_t e = wbase + (size_t)(k * 64 + lane);
#pragma unroll
                    for (int j = 0; j < 12; ++j)
                        u[j] = a.u[j * a.u_stride + e];
                }
                pass = generate_f64<SOURCE == 0>(fresh_params(), u, p);
            }
            const uint64_t mask = __ballot(pass);
            if (pass) {
                const uint32_t slot = qn + (uint32_t)__popcll(mask & lanemask_lt);
                int d[3] = {0, 1, 2}; // the f32 algebra of the mixed path takes the photons sorted
                if (PREC == 1)
                    sort_slots(p, fresh_params().sort, d);
#pragma unroll
                for (int i = 0; i < 3; ++i)
#pragma unroll
                    for (int j = 0; j < 4; ++j)
                        slot_of(slot)[64 * (4 * d[i] + j)] = p[i][j];
                if (SOURCE == 2)
                    qev[slot] = (uint32_t)(wbase + (size_t)(k * 64 + lane));
            }
            qn += (uint32_t)__popcll(mask);
            if (qn >= 64) {
                __syncthreads();
                const uint32_t slot = qn - 64 + lane;
                double pq[3][4], m[5];
#pragma unroll
                for (int i = 0; i < 3; ++i)
#pragma unroll
                    for (int j = 0; j < 4; ++j)
                        pq[i][j] = slot_of(slot)[64 * (4 * i + j)];
                const double wq = SOURCE == 2 ? a.invq[qev[slot]] : 1.;
                __syncthreads();
                qn -= 64;
                matrix_elements<PREC>(fresh_params(), pq, m);
                if (SOURCE == 2)
#pragma unroll
                    for (int c = 0; c < 5; ++c)
                        m[c] = m[c] * wq;
                acc_add(A, fresh_params(), m);
            }
        }
        if (qn > 0) { // partial flush
            __syncthreads();
            if (lane < qn) {
                double pq[3][4], m[5];
#pragma unroll
                for (int i = 0; i < 3; ++i)
#pragma unroll
                    for (int j = 0; j < 4; ++j)
                        pq[i][j] = slot_of(lane)[64 * (4 * i + j)];
                matrix_elements<PREC>(fresh_params(), pq, m);
                if (SOURCE == 2) {
                    const double wq = a.invq[qev[lane]];
#pragma unroll
                    for (int c = 0; c < 5; ++c)
                        m[c] = m[c] * wq;
                }
                acc_add(A, fresh_params(), m);
            }
        }
        __syncthreads();
        double v[12];
        acc_values(A, fresh_params(), v);
        block_reduce_store<1>(v, A.n, reinterpret_cast<DevAcc *>(a.parts == 1 ? a.out : a.part_out) + t, red);
    }
}

// Parts' sums into their batch's: lane l adds parts l, l + 64, ..., then the
// butterfly of block_reduce_store (the order depends on the number of parts
// only).
__global__ __launch_bounds__(64) void batch_sums_kernel(FusedArgs a)
{
    __shared__ double red[1][13];
    const uint64_t lb = blockIdx.x;
    const DevAcc *p = reinterpret_cast<const DevAcc *>(a.part_out) + lb * a.parts;
    double v[12] = {0., 0., 0., 0., 0., 0., 0., 0., 0., 0., 0., 0.};
    uint32_t n = 0;
    for (uint32_t s = threadIdx.x; s < a.parts; s += 64) {
        n += (uint32_t)p[s].selected;
#pragma unroll
        for (int j = 0; j < 5; ++j) {
            v[j] = v[j] + p[s].spm2[j];
            v[5 + j] = v[5 + j] + p[s].vars[j];
        }
        v[10] = v[10] + p[s].sigma;
        v[11] = v[11] + p[s].variance;
    }
    block_reduce_store<1>(v, n, reinterpret_cast<DevAcc *>(a.out) + lb, red);
}

void launch_batch_sums(const FusedArgs &a, hipStream_t st)
{
    hipLaunchKernelGGL(batch_sums_kernel, dim3((unsigned)a.nb), dim3(64), 0, st, a);
}

// Column `col` of B^(v 16^j), one lane per column; the matrices are uniform.
__global__ __launch_bounds__(64) void xo_digit_table_kernel(const uint64_t *pow2, uint64_t *tab16)
{
    const uint32_t j = blockIdx.x / 15, v = blockIdx.x % 15 + 1, col = 64 * blockIdx.y + threadIdx.x;
    uint64_t s[4];
#pragma unroll
    for (uint32_t w = 0; w < 4; ++w)
        s[w] = w == blockIdx.y ? 1ull << threadIdx.x : 0;
    for (uint32_t k = 0; k < 4; ++k)
        if ((v >> k) & 1u)
            gf2_apply(pow2 + XO_MAT_WORDS * (4 * j + k), s);
#pragma unroll
    for (int w = 0; w < 4; ++w)
        tab16[XO_MAT_WORDS * blockIdx.x + 4 * col + w] = s[w];
}

void launch_xo_digit_table(const uint64_t *pow2, int digits, uint64_t *tab16, hipStream_t st)
{
    hipLaunchKernelGGL(xo_digit_table_kernel, dim3(15 * digits, 4), dim3(64), 0, st, pow2, tab16);
}

struct XoRuns {
    uint32_t n[XO_NTABLES];
};
// Lane l's images of every value of nibble `threadIdx.x` of the state, for run
// length runs.n[blockIdx.y] (l = blockIdx.x, so the skip matrices are uniform).
__global__ __launch_bounds__(64) void xo_lane_table_kernel(const uint64_t *m16, uint64_t *lanes, XoRuns runs)
{
    const uint32_t l = blockIdx.x, ch = threadIdx.x;
    uint64_t img[4][4]; // of the nibble's four bits
#pragma unroll
    for (uint32_t k = 0; k < 4; ++k) {
#pragma unroll
        for (uint32_t w = 0; w < 4; ++w)
            img[k][w] = w == ch / 16 ? 1ull << (4 * (ch % 16) + k) : 0;
        const uint64_t *tab = m16;
        for (uint32_t e = 12 * runs.n[blockIdx.y] * l; e; e >>= 4, tab += 15 * XO_MAT_WORDS)
            if (e & 15u)
                gf2_apply(tab + ((e & 15u) - 1) * XO_MAT_WORDS, img[k]);
    }
    uint64_t *out = lanes + XO_LANE_WORDS * blockIdx.y + 256 * (size_t)(16 * ch) + 2 * l;
#pragma unroll
    for (uint32_t v = 0; v < 16; ++v) {
        uint64_t x[4] = {0, 0, 0, 0};
#pragma unroll
        for (uint32_t k = 0; k < 4; ++k)
#pragma unroll
            for (uint32_t w = 0; w < 4; ++w)
                x[w] ^= (v >> k) & 1u ? img[k][w] : 0;
#pragma unroll
        for (uint32_t w = 0; w < 4; ++w)
            out[256 * v + 128 * (w / 2) + w % 2] = x[w];
    }
}

void launch_xo_lane_tables(const uint64_t *m16, uint64_t *lanes, hipStream_t st)
{
    XoRuns r;
    for (int i = 0; i < XO_NRUNS; ++i)
        r.n[i] = XO_RUNS[i];
    r.n[XO_NRUNS] = XO_EXPAND_RUN;
    hipLaunchKernelGGL(xo_lane_table_kernel, dim3(64, XO_NTABLES), dim3(64), 0, st, m16, lanes, r);
}

// The xoshiro128+ tables: lane c < 64 takes columns c and c + 64; one lane per
// (nibble, half) of the state.
__global__ __launch_bounds__(64) void xo128_digit_table_kernel(const uint32_t *pow2, uint32_t *tab16)
{
    const uint32_t j = blockIdx.x / 15, v = blockIdx.x % 15 + 1, col = 64 * blockIdx.y + threadIdx.x;
    uint32_t s[4];
#pragma unroll
    for (uint32_t w = 0; w < 4; ++w)
        s[w] = w == col / 32 ? 1u << (col % 32) : 0;
    for (uint32_t k = 0; k < 4; ++k)
        if ((v >> k) & 1u)
            gf2_apply128(pow2 + XO128_MAT_WORDS * (4 * j + k), s);
#pragma unroll
    for (int w = 0; w < 4; ++w)
        tab16[XO128_MAT_WORDS * blockIdx.x + 4 * col + w] = s[w];
}

void launch_xo128_digit_table(const uint32_t *pow2, int digits, uint32_t *tab16, hipStream_t st)
{
    hipLaunchKernelGGL(xo128_digit_table_kernel, dim3(15 * digits, 2), dim3(64), 0, st, pow2, tab16);
}

__global__ __launch_bounds__(64) void xo128_lane_table_kernel(const uint32_t *m16, uint32_t *lanes, XoRuns runs)
{
    const uint32_t l = blockIdx.x, ch = threadIdx.x & 31u;
    uint32_t img[4][4]; // of the nibble's four bits
#pragma unroll
    for (uint32_t k = 0; k < 4; ++k) {
#pragma unroll
        for (uint32_t w = 0; w < 4; ++w)
            img[k][w] = w == ch / 8 ? 1u << (4 * (ch % 8) + k) : 0;
        const uint32_t *tab = m16;
        for (uint32_t e = 12 * runs.n[blockIdx.y] * l; e; e >>= 4, tab += 15 * XO128_MAT_WORDS)
            if (e & 15u)
                gf2_apply128(tab + ((e & 15u) - 1) * XO128_MAT_WORDS, img[k]);
    }
    uint32_t *out = lanes + XO128_LANE_WORDS * blockIdx.y + 256 * (size_t)(16 * ch) + 4 * l;
    const uint32_t v0 = threadIdx.x < 32 ? 0 : 8; // half of the nibble's values per lane
#pragma unroll
    for (uint32_t i = 0; i < 8; ++i) {
        const uint32_t v = v0 + i;
#pragma unroll
        for (uint32_t w = 0; w < 4; ++w) {
            uint32_t x = 0;
#pragma unroll
            for (uint32_t k = 0; k < 4; ++k)
                x ^= (v >> k) & 1u ? img[k][w] : 0;
            out[256 * v + w] = x;
        }
    }
}

void launch_xo128_lane_tables(const uint32_t *m16, uint32_t *lanes, hipStream_t st)
{
    XoRuns r;
    for (int i = 0; i < XO_NRUNS; ++i)
        r.n[i] = XO_RUNS[i];
    r.n[XO_NRUNS] = XO_EXPAND_RUN;
    hipLaunchKernelGGL(xo128_lane_table_kernel, dim3(64, XO_NTABLES), dim3(64), 0, st, m16, lanes, r);
}

template <int SOURCE, int PREC> int blocks_per_cu()
{
    int n = 0;
    hipError_t e = hipOccupancyMaxActiveBlocksPerMultiprocessor(&n, fused_kernel<SOURCE, PREC>, 64, 0);
    return (e == hipSuccess && n > 0) ? n : 1;
}

int fused_blocks_per_cu(int source, int precision)
{
    if (source == 0)
        return precision == 0 ? blocks_per_cu<0, 0>() : blocks_per_cu<0, 1>();
    if (source == 2)
        return blocks_per_cu<2, 0>();
    if (source == 3)
        return blocks_per_cu<3, 0>();
    if (source == 4)
        return blocks_per_cu<4, 0>();
    return precision == 0 ? blocks_per_cu<1, 0>() : blocks_per_cu<1, 1>();
}

void launch_fused(const FusedArgs &a, int source, int grid, hipStream_t st)
{
    const dim3 g(grid), b(64);
    if (source == 0) {
        if (a.precision == 0)
            hipLaunchKernelGGL((fused_kernel<0, 0>), g, b, 0, st, a);
        else
            hipLaunchKernelGGL((fused_kernel<0, 1>), g, b, 0, st, a);
    } else if (source == 1) {
        if (a.ranf.later && a.precision == 0)
            hipLaunchKernelGGL((fused_kernel<1, 0, true>), g, b, 0, st, a);
        else if (a.ranf.later)
            hipLaunchKernelGGL((fused_kernel<1, 1, true>), g, b, 0, st, a);
        else if (a.precision == 0)
            hipLaunchKernelGGL((fused_kernel<1, 0>), g, b, 0, st, a);
        else
            hipLaunchKernelGGL((fused_kernel<1, 1>), g, b, 0, st, a);
    } else if (source == 2) {
        hipLaunchKernelGGL((fused_kernel<2, 0>), g, b, 0, st, a);
    } else if (source == 3) {
        hipLaunchKernelGGL((fused_kernel<3, 0>), g, b, 0, st, a);
    } else {
        hipLaunchKernelGGL((fused_kernel<4, 0>), g, b, 0, st, a);
    }
}

template <int SOURCE, int PREC>
__global__ __launch_bounds__(256) void events_kernel(FusedArgs a, uint32_t n, EventOut o)
{
    const uint32_t e = blockIdx.x * blockDim.x + threadIdx.x;
    if (e >= n)
        return;
    double u[12];
    if (SOURCE == 0) {
        uint64_t s[4];
        s[0] = a.s0[0];
        s[1] = a.s0[1];
        s[2] = a.s0[2];
        s[3] = a.s0[3];
        const uint64_t off = 12ull * e;
        for (int k = 0; k < a.km; ++k)
            if ((off >> k) & 1ull)
                gf2_apply(a.mt + 1024 * k, s);
#pragma unroll
        for (int j = 0; j < 12; ++j)
            u[j] = xo_uniform64(s); // u 2^64, as the fused kernel draws them
    } else {
#pragma unroll
        for (int j = 0; j < 12; ++j)
            u[j] = (double)a.draws[12ull * e + j] * 1e-9;
    }
    double pu[3][4], p[3][4], m[5] = {0., 0., 0., 0., 0.};
    int d[3];
    const bool k = generate_f64<SOURCE == 0>(a.P, u, pu);
    sort_slots(pu, a.P.sort, d);
    to_slots(pu, d, p);
    if (SOURCE == 0)
#pragma unroll
        for (int j = 0; j < 12; ++j)
            u[j] = u[j] * 0x1.0p-64;
    if (k)
        matrix_elements<PREC>(a.P, p, m);
    if (!k) {
#pragma unroll
        for (int c = 0; c < 5; ++c)
            m[c] = 0.;
    }
    if (o.u)
#pragma unroll
        for (int j = 0; j < 12; ++j)
            o.u[12ull * e + j] = u[j];
    if (o.p)
#pragma unroll
        for (int i = 0; i < 3; ++i)
#pragma unroll
            for (int j = 0; j < 4; ++j)
                o.p[12ull * e + 4 * i + j] = p[i][j] * a.P.unit;
    if (o.keep)
        o.keep[e] = k ? 1 : 0;
    if (o.m)
#pragma unroll
        for (int c = 0; c < 5; ++c)
            o.m[5ull * e + c] = m[c];
}

void launch_events(const FusedArgs &a, int source, uint32_t n, const EventOut &o, hipStream_t st)
{
    const dim3 g((n + 255) / 256), b(256);
    if (source == 0) {
        if (a.precision == 0)
            hipLaunchKernelGGL((events_kernel<0, 0>), g, b, 0, st, a, n, o);
        else
            hipLaunchKernelGGL((events_kernel<0, 1>), g, b, 0, st, a, n, o);
    } else {
        if (a.precision == 0)
            hipLaunchKernelGGL((events_kernel<1, 0>), g, b, 0, st, a, n, o);
        else
            hipLaunchKernelGGL((events_kernel<1, 1>), g, b, 0, st, a, n, o);
    }
}

// ---- RANF expansion ------------------------------------------------------
// Outcome of the unit-disc test on the point (x, y) = 2u - 1 of two
// uniforms: r2 above 1 re-rolls, and in f64 so does r2 below MIN_POSITIVE^2
// (f32's MIN_POSITIVE^2 is 0).  The walk sums (0 + x*x) + y*y for the six
// values' points and 0 + (x*x + y*y) for a re-roll: without contraction both
// are fl(fl(x*x) + fl(y*y)).
__device__ __forceinline__ uint32_t disc_accept(double x, double y)
{
    const double min2 = 2.2250738585072014e-308 * 2.2250738585072014e-308;
    const double r2 = (0. + x * x) + y * y;
    return (r2 > 1. || r2 < min2) ? 0u : 1u;
}
__device__ __forceinline__ uint32_t disc_accept(float x, float y)
{
    const float r2 = (0.f + x * x) + y * y;
    return r2 > 1.f ? 0u : 1u;
}

// A RANF value as the walk's unit-disc test sees it: x = 2 (v * 1e-9) - 1 in
// the run's float type (ranf.rs:99), and its square.
template <class T> __device__ __forceinline__ T ranf_sq(int32_t v)
{
    const T x = fma((T)v * (T)1e-9, (T)2., (T)-1.); // 2u is exact: one rounding either way
    return x * x;
}

// Lane moves within the wavefront (DPP, no LDS): DPP_WAVE_ROR1 gives lane i
// the value of lane i - 1 (lane 0: lane 63); DPP_ROW_SHR9 gives lane i of each
// row of 16 the value of lane i - 9 of the row (lanes 61..63: lanes 52..54), 0
// to its first nine lanes.
constexpr int DPP_WAVE_ROR1 = 0x13C, DPP_ROW_SHR9 = 0x119;
template <int CTRL> __device__ __forceinline__ double lanes_dpp(double v)
{
    const uint64_t b = (uint64_t)__double_as_longlong(v);
    const uint32_t lo = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)(uint32_t)b, CTRL, 0xf, 0xf, true);
    const uint32_t hi = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)(uint32_t)(b >> 32), CTRL, 0xf, 0xf, true);
    return __longlong_as_double((long long)(((uint64_t)hi << 32) | lo));
}
template <int CTRL> __device__ __forceinline__ float lanes_dpp(float v)
{
    return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), CTRL, 0xf, 0xf, true));
}

// Accept bits of a segment's rounds.  Lane i holds the square of position
// 55 r + 54 - i (each value's square is computed once, as the next round's,
// and carried); its partners +1 and +3 come from lanes i - 1 and i - 3, or
// for the round's last positions from the next round's first ones, by lane
// moves.  Each round's two ballots, bit-reversed into position order, wait in
// LDS; every 32 rounds (1760 positions, 55 words) lanes 0..54 assemble one
// word each and store them together (barriers order lane 0's writes and the
// other lanes' reads: the workgroup is the one wavefront).
template <class T> struct RanfBits {
    uint64_t *m1, *m3;  // [32] LDS: the block's rounds' bits, bit j = position 55 r + j
    uint32_t *d1, *d3;  // the block's first words
    uint32_t k;         // rounds of the block so far
    T sq;               // this round's squares
    __device__ __forceinline__ void start(int32_t x) { sq = ranf_sq<T>(x); }
    __device__ __forceinline__ void round(int32_t xn)
    {
        const int lane = (int)(threadIdx.x & 63u);
        const T sqn = ranf_sq<T>(xn);
        // t: this round's squares in lanes 0..54 and the next round's
        // positions 2, 1, 0 (its lanes 52..54) in lanes 61..63; rotating t
        // down the wavefront by 1 and by 3 lanes gives each lane its partners
        // +1 and +3
        // (the empty asm keeps the move out of the select's branch: every
        // lane takes part, so the source lanes 52..54 are live)
        T nx = lanes_dpp<DPP_ROW_SHR9>(sqn);
        asm volatile("" : "+v"(nx));
        const T t = lane < 55 ? sq : nx;
        const T p1 = lanes_dpp<DPP_WAVE_ROR1>(t);
        const T p3 = lanes_dpp<DPP_WAVE_ROR1>(lanes_dpp<DPP_WAVE_ROR1>(p1));
        // r2 = fl(fl(x*x) + fl(y*y)), the walk's sums (0 + x*x) + y*y and
        // 0 + (x*x + y*y); a point re-rolls when r2 > 1 (the f64 test's
        // r2 < MIN_POSITIVE^2 compares with 0, which a sum of squares never
        // is below)
        const T r1 = sq + p1, r3 = sq + p3;
        constexpr uint64_t LIVE = (1ull << 55) - 1;
        const uint64_t b1 = __builtin_bitreverse64(__ballot(r1 <= (T)1.) & LIVE) >> 9;
        const uint64_t b3 = __builtin_bitreverse64(__ballot(r3 <= (T)1.) & LIVE) >> 9;
        if (lane == 0) {
            m1[k] = b1;
            m3[k] = b3;
        }
        sq = sqn;
        if (++k == 32)
            flush();
    }
    // words j of the block with 32 j < 55 k (those past the segment's last
    // round hold positions no walk reads)
    __device__ __forceinline__ void flush()
    {
        const uint32_t lane = threadIdx.x & 63u;
        __syncthreads(); // lane 0's masks are in
        if (lane < 55 && 32 * lane < 55 * k) {
            const uint32_t r0 = 32 * lane / 55, b0 = 32 * lane % 55;
            uint64_t w1 = m1[r0] >> b0, w3 = m3[r0] >> b0;
            if (55 - b0 < 32) {
                w1 |= m1[r0 + 1] << (55 - b0);
                w3 |= m3[r0 + 1] << (55 - b0);
            }
            d1[lane] = (uint32_t)w1;
            d3[lane] = (uint32_t)w3;
        }
        d1 += 55;
        d3 += 55;
        k = 0;
        __syncthreads(); // before the next block's masks overwrite these
    }
};

template <int BITS> __global__ __launch_bounds__(64) void ranf_expand_kernel(RanfArgs a)
{
    __shared__ int32_t win[112];
    const int lane = threadIdx.x;
    const uint64_t piece = blockIdx.x / a.nsegs;
    const uint64_t seg = a.seg_first + blockIdx.x % a.nsegs;
    const uint64_t p0 = (uint64_t)__builtin_amdgcn_readfirstlane(a.p0[piece]); // uniform: scalar compares below
    const uint64_t q_begin = p0 + a.d_begin, q_end = p0 + a.d_end;
    const uint64_t r_begin = seg * (uint64_t)a.R;
    if (r_begin * 55 >= q_end)
        return; // whole workgroup
    int32_t x = lane < 55 ? a.origin[56 * piece + lane + 1] : 0;
    const RanfLanes l = ranf_lanes();
    uint64_t skip = r_begin;
    if (ranf_odd(x)) { // (R divides RANF_LATE)
        const uint64_t odd_seg = skip / RANF_LATE;
        x = ranf_odd_segment(x, a.r16, odd_seg, win);
        skip %= RANF_LATE;
        for (; skip && !odd_seg; --skip)
            x = ranf_next_round(x, l);
    }
    x = ranf_advance(x, a.r16, skip, win);
    // (the empty asm makes the wait for a load of x come here: in the rounds'
    // loop, where the compiler would place it, it waits for each round's store)
    asm volatile("" : "+v"(x));
    int32_t *out = a.out + piece * a.piece_stride;
    __shared__ uint64_t bm[2][BITS ? 32 : 1];
    using BT = typename std::conditional<BITS == 2, float, double>::type;
    RanfBits<BT> bits;
    if (BITS) {
        const uint64_t w0 = piece * a.bits_piece_words + (seg - a.seg_first) * (55ull * (uint64_t)a.R / 32);
        bits.m1 = bm[0];
        bits.m3 = bm[1];
        bits.d1 = a.acc1 + w0;
        bits.d3 = a.acc3 + w0;
        bits.k = 0;
        bits.start(x);
    }
    // the round's accept bits (from it and the next round), then on to the next
    auto advance = [&](int32_t x) -> int32_t {
        const int32_t xn = ranf_next_round(x, l);
        if (BITS)
            bits.round(xn);
        return xn;
    };
    // X[lane+1] of round r is emitted at stream position 55 r + 54 - lane.
    // (A round's store is 220 bytes, not whole lines: the L2 merges them, so
    // they are ordinary stores; streaming stores took twice as long.)
    // Rounds [r_begin, r_end) reach into [q_begin, q_end); of those,
    // [f_lo, f_hi) lie wholly inside and are stored without range checks.
    const uint64_t r_end = min(r_begin + (uint64_t)a.R, (q_end + 54) / 55);
    const uint64_t f_lo = min(max((q_begin + 54) / 55, r_begin), r_end);
    const uint64_t f_hi = max(f_lo, min(r_end, q_end / 55));
    const uint64_t qq0 = (uint64_t)(54 - lane);
    uint64_t r = r_begin;
    for (; r < f_lo; ++r) {
        const uint64_t qq = 55 * r + qq0;
        if (lane < 55 && qq >= q_begin && qq < q_end)
            out[qq - q_begin] = x;
        x = advance(x);
    }
    int32_t *row = out + (55 * f_lo - q_begin); // uniform
    const int off = 54 - lane;
    const uint32_t nfull = (uint32_t)(f_hi - f_lo); // at most R
    for (uint32_t k = 0; k < nfull; ++k) {
        if (lane < 55)
            row[off] = x;
        x = advance(x);
        row += 55;
    }
    r = f_hi;
    for (; r < r_end; ++r) {
        const uint64_t qq = 55 * r + qq0;
        if (lane < 55 && qq >= q_begin && qq < q_end)
            out[qq - q_begin] = x;
        x = advance(x);
    }
    if (BITS && bits.k)
        bits.flush();
}

void launch_ranf_expand(const RanfArgs &a, uint64_t npieces, hipStream_t st)
{
    const uint64_t blocks = npieces * a.nsegs;
    if (a.bits == 1)
        hipLaunchKernelGGL(ranf_expand_kernel<1>, dim3((unsigned)blocks), dim3(64), 0, st, a);
    else if (a.bits == 2)
        hipLaunchKernelGGL(ranf_expand_kernel<2>, dim3((unsigned)blocks), dim3(64), 0, st, a);
    else
        hipLaunchKernelGGL(ranf_expand_kernel<0>, dim3((unsigned)blocks), dim3(64), 0, st, a);
}

// ---- faster-evgen stream walk --------------------------------------------------
// take(n) of random_array::<N> on the stored stream: a request that does not
// fit in the current round skips its leftovers (ranf.rs:89-92).  False (and no
// read) when the values would lie past the stored range.  T is the run's
// float type: (n as T) * 1e-9 (ranf.rs:99).
template <class T> __device__ __forceinline__ bool fe_take(const FeWalkArgs &a, uint64_t &q, int n, T *out)
{
    const uint32_t rem = 55u - (uint32_t)(q % 55u);
    if (rem < (uint32_t)n)
        q += rem;
    if (q + (uint64_t)n > a.qlimit)
        return false;
    if (out) {
        const int32_t *v = a.buf + (q - a.qbase);
        for (int k = 0; k < n; ++k)
            out[k] = (T)v[n - 1 - k] * (T)1e-9;
    }
    q += (uint64_t)n;
    return true;
}

// Consumption of one event (raw_photons_faster_f64's draws: 9, 6, then 2 per
// re-rolled point of the unit-disc test, decided in the run's float type T).
// False when the stored range ends inside the event.
template <class T = double> __device__ __forceinline__ bool fe_walk_event(const FeWalkArgs &a, uint64_t &q)
{
    T r6[6];
    if (!fe_take<T>(a, q, 9, nullptr) || !fe_take<T>(a, q, 6, r6))
        return false;
    const T minpos = sizeof(T) == 8 ? (T)2.2250738585072014e-308 : (T)1.17549435e-38f;
    const T min2 = minpos * minpos; // 0 in f32, as in the reference's f32 build
    for (int i = 0; i < 3; ++i) {
        const T x = (T)2. * r6[i] - (T)1., y = (T)2. * r6[3 + i] - (T)1.;
        T r2 = ((T)0. + x * x) + y * y;
        while (r2 > (T)1. || r2 < min2) {
            T r[2];
            if (!fe_take<T>(a, q, 2, r))
                return false;
            const T xa = (T)2. * r[0] - (T)1., ya = (T)2. * r[1] - (T)1.;
            r2 = (T)0. + (xa * xa + ya * ya);
        }
    }
    return true;
}

// Accept bit of stored position r (bit r % 32 of word r / 32).
__device__ __forceinline__ uint32_t acc_bit(const uint32_t *bits, uint64_t r) { return (bits[r >> 5] >> (r & 31)) & 1u; }

// Of the accepted re-roll pairs marked in y (bit k: the pair starting k
// positions on), the fails-th one (fails in 1..3): clearing the lowest
// fails - 1 set bits leaves it as the lowest.  0 when y has fewer.
__device__ __forceinline__ uint64_t nth_accept(uint64_t y, uint32_t fails)
{
    const uint64_t y1 = y & (y - 1), y2 = y1 & (y1 - 1);
    return fails == 1 ? y : fails == 2 ? y1 : y2;
}

// 64 bits of a bit array from bit r on: the words at w[0], w[1], w[2] hold
// bits from (r & ~31) on.
__device__ __forceinline__ uint64_t bits64(const uint32_t *w, uint64_t r)
{
    const uint32_t s = (uint32_t)(r & 31);
    const uint64_t lo = ((uint64_t)w[1] << 32) | w[0];
    return s ? (lo >> s) | ((uint64_t)w[2] << (64 - s)) : lo;
}

// One event's consumption of a xoshiro stream (xoshiro256+ in f64 or
// xoshiro128+ in f32): 9, 6, then 2 per re-rolled point of the unit-disc
// test, no discards.  The test's outcomes come from the accept bits (bit
// index = position - bbase): point i of the 6 values is (u_p, u_p+3) at
// p = q + 9 + i (acc3), a re-roll is (u_p, u_p+1) (acc1).  The re-rolls of
// the failed points form one run of pairs from q + 15 on, so with F failed
// points the event ends after the F-th accepted pair, found from 64 positions
// of acc1 bits at once (the pairs are the even offsets).  Near qlimit, or when
// the 32 pairs hold fewer than F accepted ones, the pairs are taken one at a
// time.  Every bit read pairs positions below qlimit.  False when the stored
// range ends inside the event.
__device__ __forceinline__ bool xo_walk_event(const uint32_t *acc1, const uint32_t *acc3, uint64_t bbase,
                                              uint64_t qlimit, uint64_t &q)
{
    if (q + 111 <= qlimit) { // words up to position q + 15 + 95 lie inside the stored range
        const uint64_t r3 = q + 9 - bbase, r1 = q + 15 - bbase;
        const uint32_t *p3 = acc3 + (r3 >> 5);
        const uint32_t ok3 = (uint32_t)((((uint64_t)p3[1] << 32) | p3[0]) >> (r3 & 31)) & 7u;
        const uint32_t fails = 3u - (uint32_t)__popc(ok3);
        if (fails == 0) {
            q += 15;
            return true;
        }
        const uint64_t y = nth_accept(bits64(acc1 + (r1 >> 5), r1) & 0x5555555555555555ull, fails);
        if (y) {
            q += 17 + (uint64_t)__builtin_ctzll(y);
            return true;
        }
    }
    q += 9;
    if (q + 6 > qlimit)
        return false;
    const uint64_t r = q - bbase;
    q += 6;
    for (int i = 0; i < 3; ++i) {
        if (acc_bit(acc3, r + i))
            continue;
        for (;;) {
            if (q + 2 > qlimit)
                return false;
            const uint32_t ok = acc_bit(acc1, q - bbase);
            q += 2;
            if (ok)
                break;
        }
    }
    return true;
}

// The RANF stream (frame positions: place in the round a = q % 55): take(n)
// first skips the round's leftovers when fewer than n remain (ranf.rs:89-92).
__device__ __forceinline__ void ranf_skip(uint64_t &q, uint32_t &a, uint32_t n)
{
    const uint32_t rem = 55u - a;
    if (rem < n) {
        q += rem;
        a = 0;
    }
}
__device__ __forceinline__ void ranf_step(uint64_t &q, uint32_t &a, uint32_t n)
{
    q += n;
    a += n;
    if (a == 55u)
        a = 0;
}

// One event's consumption of the RANF stream on its accept bits, as
// fe_walk_event: take(9), take(6) (its points are (p, p+3) for p the block's
// first three positions, in any order: only the count of failures matters),
// then a take(2) per re-roll until each failed point has an accepted pair.
__device__ __forceinline__ bool ranf_walk_event(const uint32_t *acc1, const uint32_t *acc3, uint64_t bbase,
                                                uint64_t qlimit, uint64_t &q, uint32_t &a)
{
    ranf_skip(q, a, 9);
    if (q + 9 > qlimit)
        return false;
    ranf_step(q, a, 9);
    ranf_skip(q, a, 6);
    if (q + 6 > qlimit)
        return false;
    const uint64_t r = q - bbase;
    ranf_step(q, a, 6);
    uint32_t fails = 3u - (acc_bit(acc3, r) + acc_bit(acc3, r + 1) + acc_bit(acc3, r + 2));
    while (fails) {
        ranf_skip(q, a, 2);
        if (q + 2 > qlimit)
            return false;
        fails -= acc_bit(acc1, q - bbase);
        ranf_step(q, a, 2);
    }
    return true;
}

// The walkers' accept bits through LDS.  Bits read straight from HBM cost
// each event several scattered loads, and a compute unit's walkers touch
// more lines than its L1 holds.  So each walking lane keeps W words of
// acc1 and acc3 (32 W positions) from the word of its next event's
// first test on in rows of its own, and takes its events' tests from there;
// the wavefront refills every lane's rows (16-byte loads) when some lane's
// next event could leave its window.  No lane reads another's rows.
constexpr int BW_THREADS = 128;
constexpr int BW_WALK = 32, BW_JOIN = 16;   // words per row of the two kernels
constexpr int bw_lds(int words) { return 2 * BW_THREADS * (words + 4); }

constexpr uint32_t FE_STUCK = 0xffffffffu; // the place of a walk that left the stored range

// The candidate pairs of an event's re-rolls by the place in the round where
// the event starts (RANF), a table in LDS of every block that walks.
struct FeLds {
    uint64_t pairs[55];
};
// Where an event that starts at place a of its round goes on after its takes of
// 9 and 6, and the positions it discards before them.
__device__ __forceinline__ void ranf_takes(uint32_t a, uint32_t &d, uint32_t &a1)
{
    d = a >= 47 ? 55 - a : a >= 41 ? 46 - a : 0;
    a1 = a >= 47 ? 15 : a >= 41 ? 6 : a == 40 ? 0 : a + 15;
}
__device__ __forceinline__ void fe_lds_fill(FeLds &t)
{
    if (threadIdx.x < 55) {
        uint32_t d, a1;
        ranf_takes(threadIdx.x, d, a1);
        t.pairs[threadIdx.x] = ranf_pair_starts(55u - a1);
    }
    __syncthreads();
}

// A walk of the RANF stream or of a xoshiro one from its walker's segment
// start, positions counted from there (p).
template <bool RANF, int W> struct FeWalker {
    // Positions past p that an event's tests may read: the 15 values, 64
    // positions of re-rolls and the rest of their last word, and on the RANF
    // stream up to 13 discarded leftovers.
    static constexpr uint32_t REACH = RANF ? 128 : 111;
    const uint32_t *acc1, *acc3;
    const FeLds *lds;
    uint64_t origin;     // bit of p = 0
    uint64_t lim;        // bits stored
    uint32_t *w1, *w3;   // the lane's rows
    uint32_t p;          // the next event's start
    uint32_t a;          // RANF: its place in the round
    uint32_t win;        // p of the rows' first bit (modulo 2^32)
    uint32_t pmax, plim; // the last p whose event's tests lie in the rows, in the stored range (+ 1)

    __device__ __forceinline__ void start(const uint32_t *b1, const uint32_t *b3, uint32_t *rows, const FeLds *t, uint64_t bit0,
                                          uint64_t limit, uint64_t q0, uint32_t p0)
    {
        acc1 = b1;
        acc3 = b3;
        lds = t;
        w1 = rows + threadIdx.x * (W + 4);
        w3 = rows + (BW_THREADS + threadIdx.x) * (W + 4);
        origin = bit0;
        lim = limit;
        p = p0;
        a = RANF ? (uint32_t)((q0 + p0) % 55u) : 0u;
        win = p0;
        pmax = 0;
        plim = limit < bit0 + REACH ? 0u : (uint32_t)min<uint64_t>(limit - bit0 - REACH + 1, 0x7fffffffu);
    }
    // Rows from the word holding position p + 9 on, in whole groups of 4
    // words below the stored range's end (past it, copies of the last group).
    // All loads go out before the first one is waited for.
    __device__ __forceinline__ void fill()
    {
        const uint64_t lim4 = (lim >> 5) & ~3ull, wb = ((origin + p + 9) >> 5) & ~3ull;
        uint4 b1[W / 4], b3[W / 4];
#pragma unroll
        for (int i = 0; i < W / 4; ++i) {
            const uint64_t w = min(wb + 4 * i, lim4 - 4);
            b1[i] = *reinterpret_cast<const uint4 *>(acc1 + w);
            b3[i] = *reinterpret_cast<const uint4 *>(acc3 + w);
        }
#pragma unroll
        for (int i = 0; i < W / 4; ++i) {
            *reinterpret_cast<uint4 *>(w1 + 4 * i) = b1[i];
            *reinterpret_cast<uint4 *>(w3 + 4 * i) = b3[i];
        }
        const uint32_t have = wb < lim4 ? 32u * (uint32_t)min<uint64_t>(lim4 - wb, W) : 0u;
        win = (uint32_t)(32 * wb - origin);
        pmax = (uint32_t)max((int32_t)(win + have - REACH + 1), 0); // (win is at most 127 below 0)
    }
    // On past one event, to FE_STUCK when the stored range ends inside it.
    // With the tests in the rows: the takes of 9 and 6 by position arithmetic,
    // the re-rolls as the F-th accepted pair past them, all as straight code
    // (a lane waits for each of its steps, and the other lanes' branches add to
    // them).
    __device__ __forceinline__ void event()
    {
        if (__any(p >= pmax && p < plim))
            fill();
        uint32_t d = 0, a1 = 0;
        if (RANF)
            ranf_takes(a, d, a1);
        // (clamped for a lane whose tests lie elsewhere)
        const uint32_t x3 = min(p + 9 - win, 32u * W - REACH + 9) + d, x1 = x3 + 6;
        const uint32_t *p3 = w3 + (x3 >> 5), *p1 = w1 + (x1 >> 5);
        const uint32_t ok3 = __builtin_amdgcn_alignbit(p3[1], p3[0], x3 & 31) & 7u;
        const uint32_t lo = __builtin_amdgcn_alignbit(p1[1], p1[0], x1 & 31), hi = __builtin_amdgcn_alignbit(p1[2], p1[1], x1 & 31);
        const uint64_t y0 = (((uint64_t)hi << 32) | lo) & (RANF ? lds->pairs[a] : 0x5555555555555555ull);
        const uint64_t y1 = y0 & (y0 - 1), y2 = y1 & (y1 - 1);
        const uint32_t good3 = (uint32_t)__popc(ok3);
        const uint64_t y = good3 == 2 ? y0 : good3 == 1 ? y1 : y2;
        const uint32_t k = good3 == 3 ? 0u : (uint32_t)__builtin_ctzll(y | 1ull << 63) + 2; // past the accepted pair
        const bool good = p < pmax && (good3 == 3 || y);
        if (__any(!good)) {
            if (!good) {
                uint64_t q = origin + p;
                const bool ok = RANF ? ranf_walk_event(acc1, acc3, 0, lim, q, a) : xo_walk_event(acc1, acc3, 0, lim, q);
                p = ok ? (uint32_t)(q - origin) : FE_STUCK;
            }
        }
        p = good ? p + d + 15 + k : p;
        if (RANF) {
            a1 += k;
            a1 = a1 >= 110u ? a1 - 110u : a1;
            a = good ? (a1 >= 55u ? a1 - 55u : a1) : a;
        }
    }
    // Records the starts below stop into list (every event takes at least 15
    // positions, so the loop ends and the list's capacity holds them).
    __device__ __forceinline__ void run(uint32_t stop, uint32_t *list, uint32_t &n)
    {
        uint32_t *o = list + n;
        while (p < stop) {
            *o++ = p;
            event();
        }
        n = (uint32_t)(o - list);
    }
};

// One event of the walk of kind a.kind: RANF with the unit-disc test in f64
// (0) or f32 (1), the xoshiro256+ stream (2) or the xoshiro128+ one (3).
__device__ __forceinline__ bool fe_walk_any(const FeWalkArgs &a, uint64_t &q)
{
    if (a.kind >= 2)
        return xo_walk_event(a.acc1, a.acc3, a.bbase, a.qlimit, q);
    return a.kind == 1 ? fe_walk_event<float>(a, q) : fe_walk_event<double>(a, q);
}

// One thread per walker, over its own segment: its list, its length and where
// the walk enters the next segment.  Bound by latency: an event is a chain of an
// LDS read and some 40 dependent integer steps, so segments are as short as the
// walks' meeting allows and a walker goes no further than that needs.  1e7 RANF
// events in 140 000 segments: 90 us here and 43 in fe_join_kernel; in 39 000
// with a fixed overlap of 24 rounds, branches and one load at a time to fill the
// rows 238 and 22.  5e7 xoshiro128+ events in 50 000: 345 and 420 us, before
// 1078 and 318.
template <bool RANF> __device__ __forceinline__ void fe_walk_segment(const FeWalkArgs &a, uint32_t *win, const FeLds *t0, uint32_t k)
{
    FeWalker<RANF, BW_WALK> w;
    const uint64_t q0 = a.seg_origin + (uint64_t)k * a.seg;
    w.start(a.acc1, a.acc3, win, t0, q0 - a.bbase, a.qlimit - a.bbase, q0, k == 0 ? (uint32_t)(a.q_start - q0) : 0u);
    uint32_t n = 0;
    w.run((uint32_t)a.seg, a.lists + (size_t)k * a.cap, n);
    a.len[k] = n;
    a.tail[k] = w.p;
}
__global__ __launch_bounds__(BW_THREADS) void fe_walk_kernel(FeWalkArgs a)
{
    __shared__ __attribute__((aligned(16))) uint32_t win[bw_lds(BW_WALK)];
    __shared__ FeLds t0;
    fe_lds_fill(t0);
    const uint32_t k = blockIdx.x * blockDim.x + threadIdx.x;
    if (k >= a.nwalkers)
        return;
    if (a.kind >= 2)
        fe_walk_segment<false>(a, win, &t0, k);
    else
        fe_walk_segment<true>(a, win, &t0, k);
}

// A walk goes on past its segment until it starts an event where a later
// segment's walker does (from there on both agree), at most to `stop`: list and
// n grow by its starts; true when they met, with j the index in that walker's
// list.  That walk, from `from` up to its segment's end `to`, is taken again
// beside this one, always the one that is behind, so that nothing waits for a
// list in memory.
template <class W>
__device__ __forceinline__ bool fe_walk_on(W &w, uint32_t from, uint32_t to, uint32_t stop, uint32_t *list, uint32_t &n,
                                           uint32_t &j)
{
    uint32_t o = from, oa = 0, p = w.p, pa = w.a; // segments start at the start of a round
    uint32_t *at = list + n;
    j = 0;
    while (p != o && o < to && p < stop) {
        const bool behind = p < o;
        if (behind)
            *at++ = p;
        w.p = behind ? p : o;
        w.a = behind ? pa : oa;
        w.event();
        p = behind ? w.p : p;
        pa = behind ? w.a : pa;
        o = behind ? o : w.p;
        oa = behind ? oa : w.a;
        j += behind ? 0u : 1u;
    }
    w.p = p;
    w.a = pa;
    n = (uint32_t)(at - list);
    return p == o && o < to;
}

// One thread per walker: on to where it meets the next one (the last one:
// `overlap` positions on).  They met within 58 events in 1.2e7 starts on the RANF
// stream, whose discards bring walkers together (each 8 events more leave an
// eighth of the walkers apart); on xoshiro streams only starting an event at the
// same place does, after a median of 22 events but at most 832 over 176 447
// walkers, and the last walker to meet is what this kernel takes its time for.
template <bool RANF> __device__ __forceinline__ void fe_join_segment(const FeWalkArgs &a, uint32_t *win, const FeLds *t0, uint32_t k)
{
    uint32_t n = a.len[k];
    const uint32_t at = a.tail[k];
    int32_t ji = -1, jj = -1;
    if (at != FE_STUCK) {
        FeWalker<RANF, BW_JOIN> w;
        const uint64_t q0 = a.seg_origin + (uint64_t)k * a.seg;
        w.start(a.acc1, a.acc3, win, t0, q0 - a.bbase, a.qlimit - a.bbase, q0, at);
        uint32_t *list = a.lists + (size_t)k * a.cap;
        const uint32_t stop = (uint32_t)(a.seg + a.overlap);
        if (k + 1 == a.nwalkers) {
            w.run(stop, list, n);
        } else {
            uint32_t j = 0;
            if (fe_walk_on(w, (uint32_t)a.seg, (uint32_t)(2 * a.seg), stop, list, n, j)) {
                ji = (int32_t)n;
                jj = (int32_t)j;
            }
        }
    }
    a.counts[k] = n;
    if (k == 0)
        a.join_prev[0] = a.join_next[0] = 0;
    if (k + 1 < a.nwalkers) {
        a.join_prev[k + 1] = ji;
        a.join_next[k + 1] = jj;
    }
}
__global__ __launch_bounds__(BW_THREADS) void fe_join_kernel(FeWalkArgs a)
{
    __shared__ __attribute__((aligned(16))) uint32_t win[bw_lds(BW_JOIN)];
    __shared__ FeLds t0;
    fe_lds_fill(t0);
    const uint32_t k = blockIdx.x * blockDim.x + threadIdx.x;
    if (k >= a.nwalkers)
        return;
    if (a.kind >= 2)
        fe_join_segment<false>(a, win, &t0, k);
    else
        fe_join_segment<true>(a, win, &t0, k);
}

void launch_fe_walk(const FeWalkArgs &a, hipStream_t st)
{
    const dim3 blocks((a.nwalkers + BW_THREADS - 1) / BW_THREADS);
    hipLaunchKernelGGL(fe_walk_kernel, blocks, dim3(BW_THREADS), 0, st, a);
    hipLaunchKernelGGL(fe_join_kernel, blocks, dim3(BW_THREADS), 0, st, a);
}

// Walker k's piece of the true walk is its list from where walker k - 1 met
// it (walker 0: from its start) to where it meets walker k + 1 (the last
// walker: to its end); it must meet walker k + 1 after that point.  The
// pieces are cut to the first `need` starts: off = min(prefix, need).  Three
// passes over blocks of FE_STITCH_BLOCK walkers (at most FE_STITCH_THREADS
// blocks): each piece and its block's sum and failure; the scan of the block
// sums (one workgroup) and the status; each block's own scan, the cut and
// start need - 1.  status[2 ..] holds the blocks' sums (then offsets) and
// status[2 + FE_STITCH_THREADS ..] their failures.
constexpr int FE_STITCH_BLOCK = 256;

__global__ __launch_bounds__(FE_STITCH_BLOCK) void fe_stitch_pieces_kernel(FeWalkArgs a, uint32_t *beg, uint32_t *len,
                                                                            uint64_t *status)
{
    __shared__ uint64_t s[FE_STITCH_BLOCK];
    __shared__ uint32_t anybad;
    const uint32_t T = a.nwalkers, k = blockIdx.x * FE_STITCH_BLOCK + threadIdx.x;
    if (threadIdx.x == 0)
        anybad = 0;
    uint32_t l = 0;
    bool ok = true;
    if (k < T) {
        const uint32_t b = k == 0 ? 0u : (uint32_t)a.join_next[k];
        const int64_t e = k + 1 < T ? (int64_t)a.join_prev[k + 1] : (int64_t)a.counts[T - 1];
        ok = e >= 0 && (uint64_t)e >= (uint64_t)b;
        l = ok ? (uint32_t)(e - (int64_t)b) : 0u;
        beg[k] = b;
        len[k] = l;
    }
    s[threadIdx.x] = l;
    __syncthreads();
    if (!ok)
        atomicOr(&anybad, 1u);
    for (uint32_t d = FE_STITCH_BLOCK / 2; d > 0; d >>= 1) {
        if (threadIdx.x < d)
            s[threadIdx.x] += s[threadIdx.x + d];
        __syncthreads();
    }
    if (threadIdx.x == 0) {
        status[2 + blockIdx.x] = s[0];
        status[2 + FE_STITCH_THREADS + blockIdx.x] = anybad;
    }
}

__global__ __launch_bounds__(FE_STITCH_THREADS) void fe_stitch_scan_kernel(uint32_t nblocks, uint64_t need,
                                                                           uint64_t *status)
{
    __shared__ uint64_t part[FE_STITCH_THREADS];
    __shared__ uint32_t anybad;
    const uint32_t t = threadIdx.x;
    if (t == 0)
        anybad = 0;
    const uint64_t v = t < nblocks ? status[2 + t] : 0;
    part[t] = v;
    __syncthreads();
    if (t < nblocks && status[2 + FE_STITCH_THREADS + t])
        atomicOr(&anybad, 1u);
    for (uint32_t d = 1; d < FE_STITCH_THREADS; d <<= 1) { // inclusive scan
        const uint64_t u = t >= d ? part[t - d] : 0;
        __syncthreads();
        part[t] += u;
        __syncthreads();
    }
    if (t < nblocks)
        status[2 + t] = part[t] - v; // the block's first walker's prefix
    if (t == 0)
        status[0] = (anybad || part[FE_STITCH_THREADS - 1] < need) ? 1u : 0u;
}

__global__ __launch_bounds__(FE_STITCH_BLOCK) void fe_stitch_cut_kernel(FeWalkArgs a, uint64_t need, const uint32_t *beg,
                                                                         uint32_t *len, uint64_t *off, uint64_t *status)
{
    __shared__ uint64_t s[FE_STITCH_BLOCK];
    const uint32_t T = a.nwalkers, t = threadIdx.x, k = blockIdx.x * FE_STITCH_BLOCK + t;
    const uint32_t l = k < T ? len[k] : 0u;
    s[t] = l;
    __syncthreads();
    for (uint32_t d = 1; d < FE_STITCH_BLOCK; d <<= 1) { // inclusive scan
        const uint64_t u = t >= d ? s[t - d] : 0;
        __syncthreads();
        s[t] += u;
        __syncthreads();
    }
    if (k >= T)
        return;
    const uint64_t o = min(status[2 + blockIdx.x] + s[t] - l, need);
    const uint32_t cut = (uint32_t)min<uint64_t>(l, need - o);
    if (o < need && need - 1 < o + cut) // this piece holds start need - 1
        status[1] = a.seg_origin + (uint64_t)k * a.seg + a.lists[(size_t)k * a.cap + beg[k] + (need - 1 - o)];
    off[k] = o;
    len[k] = cut;
}

void launch_fe_stitch(const FeWalkArgs &a, uint64_t need, uint32_t *begin, uint32_t *len, uint64_t *off,
                      uint64_t *status, hipStream_t st)
{
    const uint32_t nblocks = (a.nwalkers + FE_STITCH_BLOCK - 1) / FE_STITCH_BLOCK; // <= FE_STITCH_THREADS
    hipLaunchKernelGGL(fe_stitch_pieces_kernel, dim3(nblocks), dim3(FE_STITCH_BLOCK), 0, st, a, begin, len, status);
    hipLaunchKernelGGL(fe_stitch_scan_kernel, dim3(1), dim3(FE_STITCH_THREADS), 0, st, nblocks, need, status);
    hipLaunchKernelGGL(fe_stitch_cut_kernel, dim3(nblocks), dim3(FE_STITCH_BLOCK), 0, st, a, need, begin, len, off,
                       status);
}

// Sixteen lanes per piece.
__global__ __launch_bounds__(256) void fe_scatter_kernel(FeWalkArgs a, const uint32_t *begin, const uint32_t *len,
                                                         const uint64_t *off, uint64_t *out)
{
    const uint32_t k = 16 * blockIdx.x + threadIdx.x / 16;
    if (k >= a.nwalkers)
        return;
    const uint32_t *src = a.lists + (size_t)k * a.cap + begin[k];
    const uint64_t q0 = a.seg_origin + (uint64_t)k * a.seg;
    uint64_t *dst = out + off[k];
    const uint32_t n = len[k];
#pragma unroll 4
    for (uint32_t i = threadIdx.x % 16; i < n; i += 16)
        dst[i] = q0 + src[i];
}

void launch_fe_scatter(const FeWalkArgs &a, const uint32_t *begin, const uint32_t *len, const uint64_t *off,
                       uint64_t *out, hipStream_t st)
{
    hipLaunchKernelGGL(fe_scatter_kernel, dim3((a.nwalkers + 15) / 16), dim3(256), 0, st, a, begin, len, off, out);
}

// Events of batch b_first + k.
__device__ __forceinline__ uint32_t fe_batch_events(const FeBatchWalkArgs &a, uint64_t k)
{
    const uint64_t left = a.num_events - (a.b_first + k) * a.batch_size;
    return left < a.batch_size ? (uint32_t)left : a.batch_size;
}

// The batch's stored stream as a walk's view of it.
__device__ __forceinline__ FeWalkArgs fe_batch_view(const FeBatchWalkArgs &a, uint64_t k)
{
    FeWalkArgs w;
    w.buf = a.buf;
    w.kind = a.kind;
    w.acc1 = a.acc1;
    w.acc3 = a.acc3;
    w.bbase = 0;
    w.qbase = 0;
    w.qlimit = (k + 1) * a.piece_stride;
    return w;
}

// Walker s of batch k (thread k * S + s), as fe_walk_kernel.
template <bool RANF> __device__ __forceinline__ void fe_seg_walk(const FeBatchWalkArgs &a, uint32_t *win, const FeLds *t0, uint64_t t)
{
    const uint64_t k = t / a.S, q0 = k * a.piece_stride + (t - k * a.S) * a.seg;
    FeWalker<RANF, BW_WALK> w;
    w.start(a.acc1, a.acc3, win, t0, q0, (k + 1) * a.piece_stride, q0, t == k * a.S && a.p0 ? (uint32_t)a.p0[k] : 0u);
    uint32_t n = 0;
    w.run((uint32_t)a.seg, a.lists + t * a.cap, n);
    a.len[t] = n;
    a.tail[t] = w.p;
}
__global__ __launch_bounds__(BW_THREADS) void fe_seg_walk_kernel(FeBatchWalkArgs a)
{
    __shared__ __attribute__((aligned(16))) uint32_t win[bw_lds(BW_WALK)];
    __shared__ FeLds t0;
    fe_lds_fill(t0);
    const uint64_t t = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= a.nb * a.S)
        return;
    if (a.kind >= 2)
        fe_seg_walk<false>(a, win, &t0, t);
    else
        fe_seg_walk<true>(a, win, &t0, t);
}

// On to where the walker meets a later one of its batch, not always the next:
// next[t] that walker's number in the batch (-1: none, or the last one), met[t]
// the index in its list, counts[t] the starts of its own list up to there.
template <bool RANF> __device__ __forceinline__ void fe_seg_join(const FeBatchWalkArgs &a, uint32_t *win, const FeLds *t0, uint64_t t)
{
    const uint64_t k = t / a.S, q0 = k * a.piece_stride + (t - k * a.S) * a.seg;
    const uint32_t s = (uint32_t)(t - k * a.S), at = a.tail[t];
    uint32_t n = a.len[t], j = 0;
    int32_t next = -1;
    if (at != FE_STUCK) {
        FeWalker<RANF, BW_JOIN> w;
        w.start(a.acc1, a.acc3, win, t0, q0, (k + 1) * a.piece_stride, q0, at);
        uint32_t *list = a.lists + t * a.cap;
        const uint32_t seg = (uint32_t)a.seg, stop = (uint32_t)(a.seg + a.overlap);
        if (s + 1 == a.S)
            w.run(stop, list, n);
        for (uint32_t o = 1; s + o < a.S; ++o) {
            if (fe_walk_on(w, o * seg, (o + 1) * seg, stop, list, n, j)) {
                next = (int32_t)(s + o);
                break;
            }
            // past that list's end, within its segment: the walk goes on alone to the next one
            w.run(min(stop, (o + 1) * seg), list, n);
            if (w.p >= stop)
                break;
        }
    }
    a.counts[t] = n;
    a.next[t] = next;
    a.met[t] = j;
}
__global__ __launch_bounds__(BW_THREADS) void fe_seg_join_kernel(FeBatchWalkArgs a)
{
    __shared__ __attribute__((aligned(16))) uint32_t win[bw_lds(BW_JOIN)];
    __shared__ FeLds t0;
    fe_lds_fill(t0);
    const uint64_t t = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= a.nb * a.S)
        return;
    if (a.kind >= 2)
        fe_seg_join<false>(a, win, &t0, t);
    else
        fe_seg_join<true>(a, win, &t0, t);
}

// One wavefront per batch: the true walk is walker 0's list, then each walker's
// from where its predecessor met it.  Its first n starts go to the batch's
// slots of evq; seq[k] = 1 (nothing written) when the true walk meets no later
// walker, or the lists end, before n starts.  The chain is followed 64 walkers
// at a time, from their values in the lanes' registers, first to see whether
// it covers the batch and then to copy its pieces, 16 lanes each.
__global__ __launch_bounds__(64) void fe_seg_assemble_kernel(FeBatchWalkArgs a)
{
    const uint64_t k = blockIdx.x;
    const uint32_t lane = threadIdx.x;
    if (k >= a.nb)
        return;
    const uint32_t n = fe_batch_events(a, k), S = a.S;
    uint64_t *out = a.evq + k * a.batch_size;
    for (int pass = 0; pass < 2; ++pass) {
        uint32_t total = 0, s = 0, from = 0; // the chain's starts so far, its walker and where it enters that list
        for (uint32_t g = 0; g < S && s < S && total < n; g += 64) {
            const uint64_t t = k * S + min(g + lane, S - 1);
            const uint32_t cnt = a.counts[t];
            const int32_t next = a.next[t];
            const uint32_t met = a.met[t];
            uint32_t begin = 0, len = 0, off = 0; // this lane's walker's piece
            while (s < S && s < g + 64 && total < n) { // uniform
                const int l = (int)(s - g);
                const uint32_t c = (uint32_t)__builtin_amdgcn_readlane((int)cnt, l);
                const uint32_t piece = c > from ? c - from : 0u;
                if ((int)lane == l) {
                    begin = from;
                    len = min(piece, n - total);
                    off = total;
                }
                total += piece;
                const int32_t to = __builtin_amdgcn_readlane(next, l);
                from = (uint32_t)__builtin_amdgcn_readlane((int)met, l);
                s = to < 0 ? S : (uint32_t)to;
            }
            if (pass == 0)
                continue;
            for (uint32_t w0 = 0; w0 < 64; w0 += 4) {
                const uint32_t w = w0 + lane / 16, i0 = lane % 16;
                const uint32_t wb = (uint32_t)__shfl((int)begin, (int)w), wl = (uint32_t)__shfl((int)len, (int)w);
                const uint32_t wo = (uint32_t)__shfl((int)off, (int)w);
                const uint32_t *src = a.lists + (k * S + g + w) * a.cap + wb;
                const uint64_t q0 = k * a.piece_stride + (uint64_t)(g + w) * a.seg;
#pragma unroll 4
                for (uint32_t i = i0; i < wl; i += 16)
                    out[wo + i] = q0 + src[i];
            }
        }
        if (pass == 0) {
            if (lane == 0)
                a.seq[k] = total >= n ? 0u : 1u;
            if (total < n)
                return;
        }
    }
}

// One thread per batch that the joined walk did not cover: its walk from its
// piece's first position.  Each event consumes at least 15 positions and the
// walk stops at the piece's end, so the loop ends.
__global__ __launch_bounds__(64) void fe_seq_walk_kernel(FeBatchWalkArgs a)
{
    const uint64_t k = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (k >= a.nb || !a.seq[k])
        return;
    const uint32_t n = fe_batch_events(a, k);
    const uint64_t base = k * a.piece_stride;
    const FeWalkArgs w = fe_batch_view(a, k);
    uint64_t q = base + (a.p0 ? (uint64_t)a.p0[k] : 0);
    const uint64_t q0 = q;
    uint64_t *out = a.evq + k * a.batch_size;
    uint32_t e = 0;
    for (; e < n; ++e) {
        out[e] = q;
        if (!fe_walk_any(w, q))
            break;
    }
    if (e < n) {
        *a.overflow = 1u;
        for (; e < n; ++e)
            out[e] = q0;
    }
}

void launch_fe_walk_batches(const FeBatchWalkArgs &a, hipStream_t st)
{
    const uint64_t walkers = a.nb * a.S;
    const unsigned wb = (unsigned)((walkers + BW_THREADS - 1) / BW_THREADS), bb = (unsigned)((a.nb + 63) / 64);
    hipLaunchKernelGGL(fe_seg_walk_kernel, dim3(wb), dim3(BW_THREADS), 0, st, a);
    hipLaunchKernelGGL(fe_seg_join_kernel, dim3(wb), dim3(BW_THREADS), 0, st, a);
    hipLaunchKernelGGL(fe_seg_assemble_kernel, dim3((unsigned)a.nb), dim3(64), 0, st, a);
    hipLaunchKernelGGL(fe_seq_walk_kernel, dim3(bb), dim3(64), 0, st, a);
}

// ---- expansion of the xoshiro streams for faster-evgen ------------------------
struct Xo256Gen {
    uint64_t s[4];
    __device__ __forceinline__ double next() { return xo_uniform(s); }
};
struct Xo128Gen {
    uint32_t s[4];
    __device__ __forceinline__ float next() { return xo128_uniform(s); }
};

// Lane l of a wavefront expands positions [l * pt, (l + 1) * pt)
// of its range from its state skipped l * pt draws, one 128-byte line of
// values (16 f64 or 32 f32) at a time, with the draws of positions
// p + 1 .. p + 3 in hand when position p is stored, so that p's accept bits
// (with p + 1 and with p + 3) are known; 3 draws past the lane's range
// complete its last bits.  Each block goes out through LDS: a store then
// writes whole lines (4 lanes' blocks of f64, 2 of f32) instead of 64
// scattered values.  The bit words go out 4 at a time (128 positions) per
// lane.
template <class T, class Gen>
__device__ __forceinline__ void xo_expand_piece(Gen g, T *piece, uint32_t *acc1, uint32_t *acc3)
{
    constexpr uint32_t pt = 12 * XO_EXPAND_RUN; // positions per lane
    static_assert(pt % 128 == 0, "whole groups of 4 bit words per lane");
    constexpr int B = 128 / sizeof(T), ROW = B + 1; // values per block (a 128-byte line), padded LDS rows
    constexpr int NB = 128 / B;        // blocks per group of 4 bit words
    __shared__ T st[64 * ROW];
    __shared__ uint4 sw[2 * 64];       // the lane's bit words of the current 128 positions
    const uint32_t lane = threadIdx.x;
    T *row = st + lane * ROW;
    uint32_t *m1 = reinterpret_cast<uint32_t *>(sw + lane), *m3 = reinterpret_cast<uint32_t *>(sw + 64 + lane);
    uint4 *w1 = reinterpret_cast<uint4 *>(acc1 + (uint64_t)lane * (pt / 32));
    uint4 *w3 = reinterpret_cast<uint4 *>(acc3 + (uint64_t)lane * (pt / 32));
    T u0 = g.next(), u1 = g.next(), u2 = g.next(); // positions p, p + 1, p + 2
    for (uint32_t grp = 0; grp < pt / 128; ++grp) {
#pragma unroll 1
        for (int b = 0; b < NB; ++b) {
            uint32_t b1 = 0, b3 = 0;
#pragma unroll
            for (int i = 0; i < B; ++i) {
                const T u3 = g.next();
                const T x0 = (T)2. * u0 - (T)1.;
                b1 |= disc_accept(x0, (T)2. * u1 - (T)1.) << i;
                b3 |= disc_accept(x0, (T)2. * u3 - (T)1.) << i;
                row[i] = u0;
                u0 = u1;
                u1 = u2;
                u2 = u3;
            }
            const int wi = b * B / 32, sh = b * B % 32;
            m1[wi] = sh ? m1[wi] | (b1 << sh) : b1;
            m3[wi] = sh ? m3[wi] | (b3 << sh) : b3;
            __syncthreads();
            // each store: 64 / B lanes' blocks, B consecutive positions each
            const uint64_t pos = (uint64_t)grp * 128 + (uint64_t)b * B;
#pragma unroll 4
            for (int r = 0; r < B; ++r) { // streaming stores of whole lines: a later kernel reads them
                const uint32_t src = r * (64 / B) + lane / B, i = lane % B;
                __builtin_nontemporal_store(st[src * ROW + i], &piece[(uint64_t)src * pt + pos + i]);
            }
            __syncthreads();
        }
        w1[grp] = sw[lane];
        w3[grp] = sw[64 + lane];
    }
}

// One wavefront per XO_EXPAND draws of a piece: it skips to the piece's first
// draw, on to its own and then to its lanes' states.  Bound by the stores and,
// for few pieces, by one wavefront's draws: 5000 pieces of xoshiro128+ 750 us
// (3.65 GB), 1060 with a wavefront per piece and the skips of pieces and lanes
// thread by thread; 484 of xoshiro256+ 177 us, before 640.
constexpr uint64_t XO_EXPAND = 64 * 12 * XO_EXPAND_RUN;
__global__ __launch_bounds__(64) void xo_expand_kernel(XoPieceArgs a)
{
    const uint32_t split = (uint32_t)(a.piece_len / XO_EXPAND);
    const uint64_t k = blockIdx.x / split, b = a.b_first + k, at = XO_EXPAND * (blockIdx.x % split);
    uint64_t sw[4] = {a.s0[0], a.s0[1], a.s0[2], a.s0[3]};
    if (a.b16)
        xo_advance_uniform(a.b16, b, sw);
    xo_advance_uniform(a.m16, a.b16 ? at : b * a.piece_len + at, sw);
    Xo256Gen g;
    xo_lane_states(a.lanes, sw, g.s);
    const uint64_t o = k * a.piece_len + at;
    xo_expand_piece<double>(g, a.xbuf + o, a.acc1 + o / 32, a.acc3 + o / 32);
}
__global__ __launch_bounds__(64) void xo128_expand_kernel(Xo128PieceArgs a)
{
    const uint32_t split = (uint32_t)(a.piece_len / XO_EXPAND);
    const uint64_t k = blockIdx.x / split, b = a.b_first + k, at = XO_EXPAND * (blockIdx.x % split);
    uint32_t sw[4] = {a.s0[0], a.s0[1], a.s0[2], a.s0[3]};
    if (a.b16)
        xo128_advance_uniform(a.b16, b, sw);
    xo128_advance_uniform(a.m16, a.b16 ? at : b * a.piece_len + at, sw);
    Xo128Gen g;
    xo128_lane_states(a.lanes, sw, g.s);
    const uint64_t o = k * a.piece_len + at;
    xo_expand_piece<float>(g, a.xbuf + o, a.acc1 + o / 32, a.acc3 + o / 32);
}

void launch_xo128_expand(const Xo128PieceArgs &a, hipStream_t st)
{
    hipLaunchKernelGGL(xo128_expand_kernel, dim3((unsigned)(a.nb * (a.piece_len / XO_EXPAND))), dim3(64), 0, st, a);
}

void launch_xo_expand(const XoPieceArgs &a, hipStream_t st)
{
    hipLaunchKernelGGL(xo_expand_kernel, dim3((unsigned)(a.nb * (a.piece_len / XO_EXPAND))), dim3(64), 0, st, a);
}


// seeded_new (ranf.rs:36-66) for jump mode, one thread per batch; then the
// wavefront makes the round RANF_LATE of its odd batches (ranf_odd), if asked to.
__global__ __launch_bounds__(64) void ranf_seed_kernel(int32_t seed0, uint64_t b_first, uint64_t nb, const uint32_t *r16,
                                                       int32_t *origin, int32_t *p0, int32_t *later)
{
    __shared__ int32_t win[112];
    const uint64_t i0 = (uint64_t)blockIdx.x * 64, i = i0 + threadIdx.x;
    const uint64_t b = b_first + i;
    int32_t x[56];
    const int32_t seed = (int32_t)((uint32_t)seed0 + (uint32_t)(123456ull * b));
#pragma unroll
    for (int k = 0; k < 56; ++k)
        x[k] = 0;
    x[55] = seed;
    int32_t jj = seed, kk = 1;
    for (int t = 1; t < 55; ++t) {
        const int ii = (21 * t) % 55;
        // dynamic index into a private array: stays in scratch-free registers
        // only if unrolled; the loop is short and runs once per batch.
        x[ii] = kk;
        kk = (int32_t)((uint32_t)jj - (uint32_t)kk);
        if (kk < 0)
            kk = (int32_t)((uint32_t)kk + (uint32_t)MODULO);
        jj = x[ii];
    }
    for (int rr = 0; rr < 10; ++rr) {
        for (int t = 1; t < 25; ++t) {
            x[t] -= x[t + 31];
            if (x[t] < 0)
                x[t] += MODULO;
        }
        for (int t = 25; t < 56; ++t) {
            x[t] -= x[t - 24];
            if (x[t] < 0)
                x[t] += MODULO;
        }
    }
    bool odd = false;
    if (i < nb) {
        for (int k = 0; k < 56; ++k) {
            origin[56 * i + k] = x[k];
            odd |= (uint32_t)x[k] >= (uint32_t)MODULO;
        }
        p0[i] = 0;
    }
    uint64_t odds = __ballot(odd);
    __syncthreads(); // the lanes' origins, read by the others below
    const uint32_t lane = threadIdx.x, ck = ranf_jump_lane(r16 + 55 * RANF_LATE_R16);
    for (odds = later ? odds : 0; odds; odds &= odds - 1) {
        const uint64_t at = 56 * (i0 + (uint64_t)__builtin_ctzll(odds)) + lane + 1;
        const int32_t y = ranf_jump(lane < 55 ? origin[at] : 0, ck, win);
        if (lane < 55)
            later[at] = y;
    }
}

// The segment starts of a caller's odd stream, a wavefront each.
struct RanfRound {
    int32_t x[56];
};
__global__ __launch_bounds__(64) void ranf_late_kernel(RanfRound r, const uint32_t *r16, uint64_t first, int32_t *later)
{
    __shared__ int32_t win[112];
    const uint32_t lane = threadIdx.x;
    const int32_t y = ranf_odd_segment(lane < 55 ? r.x[lane + 1] : 0, r16, first + blockIdx.x, win);
    if (lane < 55)
        later[56 * (uint64_t)blockIdx.x + lane + 1] = y;
}
void launch_ranf_late(const int32_t round[56], const uint32_t *r16, uint64_t first, uint64_t n, int32_t *later, hipStream_t st)
{
    RanfRound r;
    for (int i = 0; i < 56; ++i)
        r.x[i] = round[i];
    hipLaunchKernelGGL(ranf_late_kernel, dim3((unsigned)n), dim3(64), 0, st, r, r16, first, later);
}

void launch_ranf_seed(int32_t seed0, uint64_t b_first, uint64_t nb, const uint32_t *r16, int32_t *origin, int32_t *p0,
                      int32_t *later, hipStream_t st)
{
    const unsigned blocks = (unsigned)((nb + 63) / 64);
    hipLaunchKernelGGL(ranf_seed_kernel, dim3(blocks), dim3(64), 0, st, seed0, b_first, nb, r16, origin, p0, later);
}

// ---- in-order merge --------------------------------------------------------
// In-order left fold of the per-batch accumulators (resacc.rs:133-139): the
// fold must stay one in batch order (its rounding is the reference's), so the
// 12 sums are 12 chains of dependent adds, and their length (nb adds of about 9
// cycles) is the floor.  Wave 0 (lanes 0..11) runs the chains over one LDS tile;
// the other waves write the next tile, which they loaded one tile ago, and load
// the one after it, so that the chains wait for neither HBM nor LDS.  The
// selected counts are integers and are summed by the loaders in any order.
// 100 000 batches: 0.55 ms; with one tile in flight and the chain's
// values moved between two sets of registers 0.80 ms, 19 cycles an add.
constexpr int MERGE_TILE = 512, MERGE_THREADS = 1024, MERGE_ROW = MERGE_TILE + 2; // rows of whole 16 bytes on distinct banks
template <class T>
__global__ __launch_bounds__(MERGE_THREADS) void merge_kernel(const DevAcc *in, uint64_t nb, DevAcc *out)
{
    __shared__ __attribute__((aligned(16))) double tile[2][12][MERGE_ROW];
    __shared__ unsigned long long cnt;
    constexpr int LOADERS = MERGE_THREADS - 64, PER = (13 * MERGE_TILE + LOADERS - 1) / LOADERS;
    const int tid = threadIdx.x;
    if (tid == 0)
        cnt = 0;
    const uint64_t *words = reinterpret_cast<const uint64_t *>(in); // 13 words per accumulator
    const uint64_t nwords = 13 * nb, ntiles = (nb + MERGE_TILE - 1) / MERGE_TILE;
    unsigned long long my_cnt = 0;
    uint64_t v[PER];
    auto load = [&](uint64_t k) {
#pragma unroll
        for (int i = 0; i < PER; ++i) {
            const uint32_t f = (uint32_t)(tid - 64) + (uint32_t)(i * LOADERS);
            const uint64_t at = 13ull * MERGE_TILE * k + f;
            v[i] = f < 13 * MERGE_TILE && at < nwords ? words[at] : 0ull;
        }
    };
    auto store = [&](uint64_t k) { // tile k -> buffer k & 1
        double(*dst)[MERGE_ROW] = tile[k & 1];
#pragma unroll
        for (int i = 0; i < PER; ++i) {
            const uint32_t f = (uint32_t)(tid - 64) + (uint32_t)(i * LOADERS), e = f / 13, w = f - 13 * e;
            if (f >= 13 * MERGE_TILE)
                continue;
            if (w == 0)
                my_cnt += v[i];
            else
                dst[w - 1][e] = __longlong_as_double((long long)v[i]);
        }
    };
    if (tid >= 64 && ntiles > 0) {
        load(0);
        store(0);
        load(1); // (zeros past the last tile)
    }
    __syncthreads();
    T t = (T)0;
    for (uint64_t k = 0; k < ntiles; ++k) {
        if (tid >= 64) {
            if (k + 1 < ntiles) {
                store(k + 1);
                load(k + 2);
            }
        } else if (tid < 12) {
            const uint64_t base = k * MERGE_TILE;
            const uint32_t m = (uint32_t)((nb - base) < (uint64_t)MERGE_TILE ? (nb - base) : (uint64_t)MERGE_TILE);
            const double *row = tile[k & 1][tid];
            uint32_t e = 0;
            if (k == 0) {
                t = (T)row[0];
                for (e = 1; e < m && e < 16; ++e)
                    t = t + (T)row[e];
            }
            // The LDS reads of the next 16 values are in flight while 16 go
            // through the chain.
            if (e + 16 <= m) {
                double2 a[8], b[8];
                auto get = [&](double2 *x, uint32_t at) {
#pragma unroll
                    for (int u = 0; u < 8; ++u)
                        x[u] = *reinterpret_cast<const double2 *>(row + at + 2 * u);
                };
                auto add = [&](const double2 *x) {
#pragma unroll
                    for (int u = 0; u < 8; ++u) {
                        t = t + (T)x[u].x;
                        t = t + (T)x[u].y;
                    }
                };
                get(a, e);
                for (e += 16; e + 32 <= m; e += 32) {
                    get(b, e);
                    __builtin_amdgcn_sched_barrier(0); // (the reads would move behind the adds)
                    add(a);
                    get(a, e + 16);
                    __builtin_amdgcn_sched_barrier(0);
                    add(b);
                }
                add(a);
            }
            for (; e < m; ++e)
                t = t + (T)row[e];
        }
        __syncthreads();
    }
    atomicAdd(&cnt, my_cnt);
    __syncthreads();
    if (tid < 12)
        reinterpret_cast<double *>(out)[1 + tid] = (double)t;
    if (tid == 0)
        out->selected = cnt;
}

void launch_merge(const void *per_batch, uint64_t nb, void *merged, hipStream_t st, int f32)
{
    if (f32)
        hipLaunchKernelGGL(merge_kernel<float>, dim3(1), dim3(MERGE_THREADS), 0, st,
                           reinterpret_cast<const DevAcc *>(per_batch), nb, reinterpret_cast<DevAcc *>(merged));
    else
        hipLaunchKernelGGL(merge_kernel<double>, dim3(1), dim3(MERGE_THREADS), 0, st,
                           reinterpret_cast<const DevAcc *>(per_batch), nb, reinterpret_cast<DevAcc *>(merged));
}

// ---- all-f32 mode --------------------------------------------------------------
// One wavefront per part of a batch (grid-stride), as in the f64 event loop:
// events that pass the cuts are queued in LDS and their helicity sums computed
// 64 at a time on dense lanes.  The batch sums are formed in event order, as
// the reference's sequential loop does in f32 (resacc.rs:121-129), where a tree
// sum would round differently.  So the queue is first in, first out: the
// oldest 64 events fill the half at `head`, and with sources whose lane l
// takes events l, l + 64, ... they leave in event order.  A wavefront with a
// whole batch (SUMS) puts the 12 summands of the 64 into the half just emptied
// and 12 lanes add them in turn: 64 dependent adds of 9 cycles that the
// other five wavefronts of the SIMD hide, against 24 bytes per event written
// and read again (7.5 of 50 ms per 1e9 events, and as much again in the
// writes).  A part of a batch hands its accepted events on in order
// (f32_accumulate_kernel).  With the xoshiro128+ stream in registers (SOURCE 0)
// a lane takes a run of events, and each event's values go to its own slot.
static_assert(offsetof(F32Args, P) == 0, "FParams first in F32Args");
typedef const __attribute__((address_space(4))) FParams KFParams;
__device__ __forceinline__ const FParams &fresh_fparams() // as fresh_params
{
    KFParams *k = (KFParams *)__builtin_amdgcn_kernarg_segment_ptr();
    asm volatile("" : "+s"(k));
    return *(const FParams *)k;
}

template <int SOURCE, bool SUMS, bool ODD = false, bool WIDE = false>
__global__ __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(6, 8))) void f32_events_kernel(F32Args a)
{
    constexpr uint32_t HALF = 12 * 64, DUMP = 2 * HALF;
    __shared__ __align__(16) float queue[2 * HALF + 4];
    __shared__ uint32_t qidx[SOURCE == 0 ? QCAP : 1];
    int32_t *const qints = reinterpret_cast<int32_t *>(queue);
    const uint32_t lane = threadIdx.x;
    const uint64_t lanemask_lt = (1ull << lane) - 1ull;
    uint32_t sw[4] = {a.s0[0], a.s0[1], a.s0[2], a.s0[3]}; // xoshiro128+ state at the part's first draw (uniform)
    RanfPart<ODD> ranf;
    bool have = false;
    for (uint64_t t = blockIdx.x; t < a.nb * a.parts; t += gridDim.x) {
        const uint64_t lb = a.parts == 1 ? t : t / a.parts;
        const uint32_t first = (uint32_t)(t - lb * a.parts) * 64u * a.run; // the part's first event in the batch
        const uint64_t b = a.b_first + lb;
        const uint64_t left = a.num_events - b * a.batch_size;
        const uint32_t nbatch = left < a.batch_size ? (uint32_t)left : a.batch_size;
        const uint32_t n = first < nbatch ? min(nbatch - first, 64u * a.run) : 0u;
        constexpr bool FE = SOURCE == 2 || SOURCE == 3;
        uint32_t len, iters;
        uint32_t s[4] = {0, 0, 0, 0};
        if (SOURCE == 0) {
            len = lane * a.run < n ? min(n - lane * a.run, a.run) : 0u;
            iters = min(n, a.run);
            xo128_advance_uniform(a.b16, have ? gridDim.x / a.parts : b, sw);
            if (!have)
                xo128_advance_uniform(a.m16, 12ull * first, sw);
            have = true;
            xo128_lane_states(a.lanes, sw, s);
        } else {
            len = n / 64 + (lane < n % 64 ? 1u : 0u);
            iters = (n + 63) / 64;
        }
        if (SOURCE == 1 && n)
            ranf.start(a.ranf, b, a.batch_size, first, n, qints);
        const uint64_t base = lb * a.batch_size + first; // the part's first slot
        uint32_t qn = 0, head = 0, done = 0; // queued events, their first slot (0 or 64), events that left (uniform)
        float sum = 0.f;                     // SUMS: lane j < 12: sum j of (spm2[5], vars[5], sigma, variance)
        // the oldest `cnt` (64, or at the part's end all) queued events
        auto flush = [&](uint32_t cnt) {
            __syncthreads();
            float *const half = queue + (head ? HALF : 0);
            auto sums = [&](float m[5]) {
                float pq[3][4];
#pragma unroll
                for (int i = 0; i < 3; ++i)
#pragma unroll
                    for (int j = 0; j < 4; ++j)
                        pq[i][j] = half[64 * (4 * i + j) + lane];
                matrix_elements_f32<WIDE>(fresh_fparams(), pq, m);
            };
            if (SUMS) {
                // summand j of event e at column (e + 4 j) % 64 of row j: the 12
                // lanes' 16-byte reads hit distinct banks.  -0.0 past the last
                // event: x + (-0.0) = x for every x.
                float m[5] = {0.f, 0.f, 0.f, 0.f, 0.f};
                const bool in = lane < cnt;
                if (in)
                    sums(m);
                const float w = weight_f32(fresh_fparams(), m), z = -0.f;
                __syncthreads();
#pragma unroll
                for (uint32_t j = 0; j < 12; ++j) {
                    const float x = j < 5 ? m[j] : j < 10 ? m[j - 5] * m[j - 5] : j == 10 ? w : w * w;
                    half[64 * j + ((lane + 4 * j) & 63u)] = in ? x : z;
                }
                __syncthreads();
                if (lane < 12) {
                    const float4 *row = reinterpret_cast<const float4 *>(half + 64 * lane);
#pragma unroll 4
                    for (uint32_t g = 0; g < 16; ++g) {
                        const float4 x = row[(g + lane) & 15u];
                        sum = sum + x.x;
                        sum = sum + x.y;
                        sum = sum + x.z;
                        sum = sum + x.w;
                    }
                }
            } else if (lane < cnt) {
                float m[5];
                sums(m);
                if (SOURCE == 0) {
                    float *o = a.ev + 6 * (size_t)qidx[head + lane];
#pragma unroll
                    for (int c = 0; c < 5; ++c)
                        o[c] = m[c];
                    o[5] = 1.f;
                } else {
#pragma unroll
                    for (int c = 0; c < 5; ++c) {
                        float *row = a.ev + (c * a.ev_stride + base + done); // uniform
                        row[lane] = m[c];
                    }
                }
            }
            __syncthreads();
            done += cnt;
            qn -= cnt;
            head ^= 64u;
        };
        // faster-evgen: the lane's next event start, loaded an event ahead
        uint64_t qnext = FE && len > 0 ? a.evq[base + lane] : 0;
        for (uint32_t i = 0; i < iters; ++i) {
            bool pass = false;
            float p[3][4];
            const uint64_t qk = qnext;
            if (FE && i + 1 < len)
                qnext = a.evq[base + 64 * (i + 1) + lane];
            int4 rd[3]; // RANF: the lane's 12 draws, through the half that is free
            if (SOURCE == 1) {
                const uint32_t ring = head ? 0 : HALF;
                ranf.fill(a.ranf, 12 * min(64u, n - 64 * i), qints, ring, DUMP);
                __syncthreads();
#pragma unroll
                for (int j = 0; j < 3; ++j)
                    rd[j] = reinterpret_cast<const int4 *>(qints + ring)[3 * lane + j];
                __syncthreads(); // read before the events are pushed
            }
            if (i < len && FE) {
                const RerollBits rb{a.acc1, a.bbase, a.bstride ? (lb + 1) * a.bstride : a.blimit};
                if constexpr (SOURCE == 2) {
                    RanfWalkF32 w{a.draws, a.qbase, qk, rb};
                    pass = generate_faster_f32<WIDE>(fresh_fparams(), w, p);
                } else {
                    Xo128WalkF32 w{a.x32draws, a.qbase, qk, rb};
                    pass = generate_faster_f32<WIDE>(fresh_fparams(), w, p);
                }
            } else if (i < len) {
                float u[12];
                if (SOURCE == 0) {
#pragma unroll
                    for (int j = 0; j < 12; ++j)
                        u[j] = xo128_uniform(s);
                } else {
#pragma unroll
                    for (int j = 0; j < 3; ++j) { // (n as f32) * INV_MODULO (ranf.rs:99)
                        u[4 * j] = (float)rd[j].x * 1e-9f;
                        u[4 * j + 1] = (float)rd[j].y * 1e-9f;
                        u[4 * j + 2] = (float)rd[j].z * 1e-9f;
                        u[4 * j + 3] = (float)rd[j].w * 1e-9f;
                    }
                }
                pass = generate_f32<WIDE>(fresh_fparams(), u, p);
            }
            if (SOURCE == 0 && i < len && !pass) {
                float *o = a.ev + 6 * (size_t)(base + lane * a.run + i);
#pragma unroll
                for (int c = 0; c < 6; ++c)
                    o[c] = 0.f;
            }
            const uint64_t mask = __ballot(pass);
            if (pass) {
                const uint32_t slot = (head + qn + (uint32_t)__popcll(mask & lanemask_lt)) & 127u;
                float *q = queue + (slot >> 6) * HALF + (slot & 63u);
#pragma unroll
                for (int k = 0; k < 3; ++k)
#pragma unroll
                    for (int j = 0; j < 4; ++j)
                        q[64 * (4 * k + j)] = p[k][j];
                if (SOURCE == 0)
                    qidx[slot] = (uint32_t)(base + lane * a.run + i);
            }
            qn += (uint32_t)__popcll(mask);
            if (qn >= 64)
                flush(64);
        }
        if (qn > 0)
            flush(qn);
        if (SUMS) {
            DevAcc *out = reinterpret_cast<DevAcc *>(a.out) + lb;
            if (lane < 12)
                reinterpret_cast<double *>(out)[1 + lane] = (double)sum;
            if (lane == 0)
                out->selected = done;
        } else if (SOURCE != 0 && lane == 0) {
            a.counts[t] = done;
        }
        __syncthreads();
    }
}

// In-order f32 batch sums (resacc.rs:121-129 with Float = f32) from the
// events' values, four wavefronts per batch: lanes 0..11 of the first add a
// tile's summands (m_c, m_c^2, w, w^2) in event order, the order that fixes the
// f32 rounding, while the other three, tile about, load the next tiles' events
// and write the accepted ones' summands to LDS side by side.  SLOTS: every event
// has a slot and a flag (source 0); otherwise the values are the accepted events
// of the batch's parts in order, tiles running on from part to part.  What bounds
// it: the chain of adds, 9 cycles an accepted event (26 us a batch, 1536 batches
// at once), or for long runs the bytes of the events.  A tile's loads have three
// tiles' time to arrive: with one loading wavefront a closure call of 10 000
// events spent 160 us here on their latency, and 54 with a rejected event's slot
// added as -0.0; 41 now (10 000 batches with slots 745 -> 445 us).
constexpr int F32_TILE = 128, F32_ROW = F32_TILE + 4; // rows 4 banks apart for the chains' 16-byte reads
constexpr int F32_BUFS = 4;                           // tiles in LDS: one being added, three being made

template <bool SLOTS> __global__ __launch_bounds__(256) void f32_accumulate_kernel(F32Args a)
{
    __shared__ __align__(16) float terms[F32_BUFS][12][F32_ROW];
    __shared__ uint32_t before[F32_MAX_PARTS + 1]; // accepted events of the parts before each
    __shared__ uint32_t kept, filled[SLOTS ? F32_BUFS : 1]; // accepted events in all, in the tiles
    const uint32_t lane = threadIdx.x & 63u, wave = threadIdx.x >> 6;
    const uint64_t lb = blockIdx.x;
    const uint64_t left = a.num_events - (a.b_first + lb) * a.batch_size;
    const uint64_t base = lb * a.batch_size;
    const uint32_t nparts = SLOTS ? 1u : a.parts; // at most F32_MAX_PARTS
    uint32_t n = left < a.batch_size ? (uint32_t)left : a.batch_size;
    if (threadIdx.x == 0)
        kept = 0;
    if (!SLOTS) {
        if (threadIdx.x < nparts)
            before[threadIdx.x + 1] = a.counts[lb * nparts + threadIdx.x];
        __syncthreads();
        if (threadIdx.x == 0) {
            before[0] = 0;
            for (uint32_t s = 0; s < nparts; ++s)
                before[s + 1] += before[s];
        }
        __syncthreads();
        n = before[nparts];
    } else {
        __syncthreads();
    }
    const uint32_t tiles = (n + F32_TILE - 1) / F32_TILE;
    constexpr int PER = F32_TILE / 64;
    float m[PER][5], flag[PER];
    bool keep[PER];
    uint32_t cnt = 0;
    auto load = [&](uint32_t k) { // (nothing in it waits for what it loads)
#pragma unroll
        for (int i = 0; i < PER; ++i) {
            const uint32_t e = k * F32_TILE + 64 * i + lane;
            keep[i] = e < n;
            uint64_t at = base + e;
            if (!SLOTS && keep[i]) {
                uint32_t lo = 0, hi = nparts; // before[lo] <= e < before[hi]
                while (hi - lo > 1) {
                    const uint32_t mid = (lo + hi) / 2;
                    if (before[mid] <= e)
                        lo = mid;
                    else
                        hi = mid;
                }
                at = base + (uint64_t)lo * 64u * a.run + (e - before[lo]);
            }
#pragma unroll
            for (int c = 0; c < 5; ++c)
                m[i][c] = !keep[i] ? 0.f : SLOTS ? a.ev[6 * at + c] : a.ev[c * a.ev_stride + at];
            flag[i] = SLOTS && keep[i] ? a.ev[6 * at + 5] : 1.f;
        }
    };
    auto write = [&](uint32_t k) {
        float(*row)[F32_ROW] = terms[k % F32_BUFS];
        if constexpr (SLOTS) { // the accepted ones side by side, in whole groups of 16
            uint32_t c = 0;
#pragma unroll
            for (int i = 0; i < PER; ++i) {
                const float w = weight_f32(a.P, m[i]);
                const bool in = keep[i] && flag[i] != 0.f;
                const uint64_t ins = __ballot(in);
                const uint32_t at = c + (uint32_t)__popcll(ins & ((1ull << lane) - 1ull));
                c += (uint32_t)__popcll(ins);
                if (in)
#pragma unroll
                    for (int j = 0; j < 12; ++j)
                        row[j][at] = j < 5 ? m[i][j] : j < 10 ? m[i][j - 5] * m[i][j - 5] : j == 10 ? w : w * w;
            }
            cnt += c;
            if (lane < (16u - c) % 16u) // x + (-0.0) = x for every x
#pragma unroll
                for (int j = 0; j < 12; ++j)
                    row[j][c + lane] = -0.f;
            if (lane == 0)
                filled[k % F32_BUFS] = c;
        } else {
#pragma unroll
            for (int i = 0; i < PER; ++i) {
                const float w = weight_f32(a.P, m[i]), z = -0.f;
                cnt += (uint32_t)__popcll(__ballot(keep[i]));
#pragma unroll
                for (int j = 0; j < 12; ++j) {
                    const float x = j < 5 ? m[i][j] : j < 10 ? m[i][j - 5] * m[i][j - 5] : j == 10 ? w : w * w;
                    row[j][64 * i + lane] = keep[i] ? x : z;
                }
            }
        }
    };
    // tile j is loaded at step j - 3, after its buffer's previous tile j - 4,
    // and written at step j - 1
    float t = 0.f; // lane j < 12 of the first wavefront: sum j of (spm2[5], vars[5], sigma, variance)
    const uint32_t p = wave - 1;
    if (wave && p < tiles)
        load(p);
    if (wave == 1 && tiles)
        write(0);
    __syncthreads();
    for (uint32_t i = 0; i < tiles; ++i) {
        if (wave) {
            if ((i + 1) % 3 == p && i + 1 < tiles)
                write(i + 1);
            if (i % 3 == p && i + 3 < tiles)
                load(i + 3);
        } else if (lane < 12) {
            const float4 *row = reinterpret_cast<const float4 *>(terms[i % F32_BUFS][lane]);
            const int groups = SLOTS ? (__builtin_amdgcn_readfirstlane((int)filled[i % F32_BUFS]) + 15) / 16 : F32_TILE / 16;
#pragma unroll 2
            for (int g = 0; g < groups; ++g) {
                float4 x[4];
#pragma unroll
                for (int u = 0; u < 4; ++u)
                    x[u] = row[4 * g + u];
#pragma unroll
                for (int u = 0; u < 4; ++u) {
                    t = t + x[u].x;
                    t = t + x[u].y;
                    t = t + x[u].z;
                    t = t + x[u].w;
                }
            }
        }
        __syncthreads();
    }
    if (wave && lane == 0)
        atomicAdd(&kept, cnt);
    __syncthreads();
    DevAcc *out = reinterpret_cast<DevAcc *>(a.out) + lb;
    if (threadIdx.x < 12)
        reinterpret_cast<double *>(out)[1 + lane] = (double)t;
    if (threadIdx.x == 0)
        out->selected = kept;
}

template <int SOURCE> static int f32_blocks()
{
    int n = 0;
    const hipError_t e = hipOccupancyMaxActiveBlocksPerMultiprocessor(&n, f32_events_kernel<SOURCE, SOURCE != 0>, 64, 0);
    return (e == hipSuccess && n > 0) ? n : 1;
}
int f32_blocks_per_cu(int source)
{
    return source == 0 ? f32_blocks<0>() : source == 1 ? f32_blocks<1>() : source == 2 ? f32_blocks<2>() : f32_blocks<3>();
}

template <int SOURCE, bool ODD = false, bool WIDE = false> static void launch_f32_source(const F32Args &a, int grid, hipStream_t st)
{
    if (f32_sums_in_kernel(a))
        hipLaunchKernelGGL((f32_events_kernel<SOURCE, true, ODD, WIDE>), dim3(grid), dim3(64), 0, st, a);
    else
        hipLaunchKernelGGL((f32_events_kernel<SOURCE, false, ODD, WIDE>), dim3(grid), dim3(64), 0, st, a);
}

void launch_f32_events(const F32Args &a, int grid, hipStream_t st)
{
    if (a.source == 0 && a.wide)
        hipLaunchKernelGGL((f32_events_kernel<0, false, false, true>), dim3(grid), dim3(64), 0, st, a);
    else if (a.source == 0)
        hipLaunchKernelGGL((f32_events_kernel<0, false>), dim3(grid), dim3(64), 0, st, a);
    else if (a.source == 1 && a.wide) // (ODD serves streams inside [0, 1e9) too)
        launch_f32_source<1, true, true>(a, grid, st);
    else if (a.source == 1 && a.ranf.later)
        launch_f32_source<1, true>(a, grid, st);
    else if (a.source == 1)
        launch_f32_source<1>(a, grid, st);
    else if (a.source == 2 && a.wide)
        launch_f32_source<2, false, true>(a, grid, st);
    else if (a.source == 2)
        launch_f32_source<2>(a, grid, st);
    else if (a.wide)
        launch_f32_source<3, false, true>(a, grid, st);
    else
        launch_f32_source<3>(a, grid, st);
}

void launch_f32_accumulate(const F32Args &a, hipStream_t st)
{
    if (a.source == 0)
        hipLaunchKernelGGL(f32_accumulate_kernel<true>, dim3((unsigned)a.nb), dim3(256), 0, st, a);
    else
        hipLaunchKernelGGL(f32_accumulate_kernel<false>, dim3((unsigned)a.nb), dim3(256), 0, st, a);
}

} // namespace tpk

// ---- adjoint ---------------------------------------------------------------
#include "tp_adjoint.h"
#include "tp_adjstore.h"

namespace tpk {

// One 64-lane workgroup per 64 consecutive points.  In f32 the sweeps run
// convergently (a cut point's lane runs them too and hands zeros on), so the
// sink can synchronise the workgroup: it stages F and dF/du in LDS for the
// whole pass and dF/dp one sweep at a time, and the stores go out with
// consecutive lanes on consecutive addresses (tp_adjstore.h), whole cache
// lines at a time for F and dF/du.
// Stage elements e = lane + 64 k, k < K, of a full workgroup (np = 64) to
// put(e, value): a fixed trip count, so the LDS loads issue back to back
// instead of one load-wait-store round trip per element.
template <int K, class T, class Put> __device__ __forceinline__ void flush_full(const T *stage, uint32_t lane, Put &&put)
{
#pragma unroll
    for (int k = 0; k < K; ++k)
        put(lane + tpa::LANES * k, stage[lane + tpa::LANES * k]);
}

// Pairs of doubles, for pointers a caller has aligned to one.
typedef double pair8 __attribute__((ext_vector_type(2), aligned(8)));

// f64: one point per lane, all derivatives from one evaluation of the closed
// forms (event_jacobian), rows staged in LDS and stored 1 KiB per instruction.
// Bound by the 1000 bytes a point writes (1.05 GB per 2^20 points: 153 us at
// the rate of a fill); its 1600 f64 instructions a point take 80 us of issue.
// One row at a time in LDS, dF/dp and then dF/du in its place: five workgroups
// per CU and 256 VGPRs.  2^20 points: 210 us; with five sweeps back through the
// amplitudes 487 (one wavefront per SIMD); with rows stored straight from
// registers, 96 B of each per sweep and lane, 620.
__global__ __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(2, 2))) void adjoint_kernel_f64(AdjArgs a)
{
    constexpr uint32_t ROW = 62; // doubles: an odd number of 16-byte units, so lanes fall on different banks
    __shared__ __attribute__((aligned(16))) double rows[ROW * tpa::LANES];
    const uint32_t lane = threadIdx.x;
    const uint64_t base = (uint64_t)blockIdx.x * tpa::LANES;
    if (base >= a.n) // whole workgroup
        return;
    const uint32_t np = tpa::points(a.n, base);
    double *F = reinterpret_cast<double *>(a.F), *Gu = reinterpret_cast<double *>(a.dF_du), *Gp = reinterpret_cast<double *>(a.dF_dp);
    const double *uu = a.u_in + 12 * (base + (lane < np ? lane : 0)); // lanes past n: a copy of point base, never stored
    double u[12];
#pragma unroll
    for (int j = 0; j < 6; ++j) {
        const pair8 x = *reinterpret_cast<const pair8 *>(uu + 2 * j);
        u[2 * j] = x.x;
        u[2 * j + 1] = x.y;
    }
    // 16-byte element e of the workgroup's rows, e < 30 np: row e / 30
    auto flush = [&](double *out) {
        double *o = out + 60 * base;
        uint32_t pt = lane / 30, r = lane % 30;
        auto put = [&](uint32_t e) {
            const double2 x = *reinterpret_cast<const double2 *>(rows + ROW * pt + 2 * r);
            *reinterpret_cast<pair8 *>(o + 2 * e) = pair8{x.x, x.y};
            r += 4; // 64 = 2 * 30 + 4
            pt += r >= 30 ? 3 : 2;
            r -= r >= 30 ? 30 : 0;
        };
        if (np == tpa::LANES)
#pragma unroll 10
            for (uint32_t k = 0; k < 30; ++k)
                put(lane + 64 * k);
        else
            for (uint32_t e = lane; e < 30 * np; e += 64)
                put(e);
    };
    event_jacobian(a.P, a.hk, a.w, u, rows + ROW * lane, Gu != nullptr, [&](const double *Fc) {
        if (F && lane < np)
#pragma unroll
            for (int c = 0; c < 5; ++c)
                F[5 * (base + lane) + c] = Fc[c];
        __syncthreads();
        if (Gp)
            flush(Gp);
        __syncthreads();
    });
    if (Gu) {
        __syncthreads();
        flush(Gu);
    }
}

// One point per lane, rows staged in LDS and stored with consecutive lanes
// on consecutive addresses (the index arithmetic is in tp_adjstore.h):
// WRITE_SIZE 1.35x the output bytes in f32 instead of 1.72x, and 13 % less
// time.  Every lane of the workgroup reaches every barrier: lanes past n
// compute a copy of point base and store nothing, and a cut point runs the
// sweeps like the others and hands zeros to the sink.
template <class T> __device__ __forceinline__ void adjoint_staged(const AdjArgs &a, T *sF, T *sU, T *sP)
{
    const uint32_t lane = threadIdx.x;
    const uint64_t base = (uint64_t)blockIdx.x * tpa::LANES;
    if (base >= a.n) // whole workgroup
        return;
    const uint32_t np = tpa::points(a.n, base);
    const bool full = np == tpa::LANES;
    const uint64_t i = base + lane;
    const bool valid = lane < np;
    const AdjParams<T> P = adj_params<T>(a.P, a.w);
    T *F = reinterpret_cast<T *>(a.F), *Gu = reinterpret_cast<T *>(a.dF_du), *Gp = reinterpret_cast<T *>(a.dF_dp);
    T u[12];
#pragma unroll
    for (int j = 0; j < 12; ++j)
        u[j] = (T)a.u_in[12 * (valid ? i : base) + j]; // lanes past n: a copy of point base, never stored
    // one forward pass, then one reverse sweep per coupling component
    T m[5], du[12], dp[12];
    event_adjoint_sweeps<T, 0, 5, true>(
        P, u, nullptr, m, du, dp, (T)0, (T)INFINITY, [&](int c, const T *mc, const T *duc, const T *dpc) {
            if (F)
                sF[tpa::slot_f(lane, c)] = P.w * (c == 0 ? mc[0] : c == 1 ? mc[1] : c == 2 ? mc[2] : c == 3 ? mc[3] : mc[4]);
            if (Gu)
#pragma unroll
                for (int j = 0; j < 12; ++j)
                    sU[tpa::slot_du(lane, c, j)] = duc[j];
            if (Gp) {
                __syncthreads(); // the previous sweep's dF/dp rows are out
#pragma unroll
                for (int j = 0; j < 12; ++j)
                    sP[tpa::slot_dp(lane, j)] = dpc[j];
                __syncthreads();
                for (uint32_t e = lane; e < 12 * np; e += tpa::LANES)
                    Gp[tpa::dst_dp(base, e, c)] = sP[e];
            }
        });
    __syncthreads();
    if (Gu) {
        if (full)
            flush_full<60>(sU, lane, [&](uint32_t e, T v) { Gu[tpa::dst_du(base, e)] = v; });
        else
            for (uint32_t e = lane; e < 60 * np; e += tpa::LANES)
                Gu[tpa::dst_du(base, e)] = sU[e];
    }
    if (F) {
        if (full)
            flush_full<5>(sF, lane, [&](uint32_t e, T v) { F[tpa::dst_f(base, e)] = v; });
        else
            for (uint32_t e = lane; e < 5 * np; e += tpa::LANES)
                F[tpa::dst_f(base, e)] = sF[e];
    }
}

// The stream's points (12 draws each, rand's Standard f64): a wavefront skips
// to its first draw, its lanes take `run` consecutive points each from there.
// Bound by latency, of the skip and of stores 96 B per lane: 46 us per 2^20
// points, 540 with one skip per thread and 256 points each.
__global__ __launch_bounds__(64) void adjoint_points_kernel(AdjArgs a)
{
    const uint64_t base = 64ull * a.run * blockIdx.x;
    uint64_t sw[4] = {a.s0[0], a.s0[1], a.s0[2], a.s0[3]}, s[4];
    xo_advance_uniform(a.m16, 12 * (a.first + base), sw);
    xo_lane_states(a.lanes, sw, s);
    const uint64_t first = base + (uint64_t)a.run * threadIdx.x, last = min(first + a.run, a.n);
    for (uint64_t k = first; k < last; ++k) {
        pair8 *out = reinterpret_cast<pair8 *>(a.u_gen + 12 * k);
#pragma unroll
        for (int j = 0; j < 6; ++j) {
            const double x = xo_uniform(s);
            out[j] = pair8{x, xo_uniform(s)};
        }
    }
}

// f32: 255 VGPRs, two wavefronts per SIMD (waves_per_eu(2, 2)), no spill;
// 19.7 KB of stage, eight workgroups per CU.
__global__ __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(2, 2))) void adjoint_kernel_f32(AdjArgs a)
{
    __shared__ float sF[5 * tpa::LANES], sU[60 * tpa::LANES], sP[12 * tpa::LANES];
    adjoint_staged<float>(a, sF, sU, sP);
}

void launch_adjoint(const AdjArgs &a0, int precision, hipStream_t st)
{
    AdjArgs a = a0;
    if (!a.u_in) {
        const uint64_t wave = 64ull * a.run;
        hipLaunchKernelGGL(adjoint_points_kernel, dim3((unsigned)((a.n + wave - 1) / wave)), dim3(64), 0, st, a);
        a.u_in = a.u_gen;
    }
    const dim3 g((unsigned)((a.n + tpa::LANES - 1) / tpa::LANES)), b(tpa::LANES);
    if (precision == 2)
        hipLaunchKernelGGL(adjoint_kernel_f32, g, b, 0, st, a);
    else
        hipLaunchKernelGGL(adjoint_kernel_f64, g, b, 0, st, a);
}

} // namespace tpk
