// tp_ctx.h -- the engine context shared by the event-loop and flow entry
// points (internal; not part of the C ABI).
#pragma once

#include "tp_guard.h"

#include <hip/hip_runtime.h>

#include <algorithm>
#include <memory>
#include <string>
#include <vector>

#include "tp.h"
#include "tp_kernels.h"
#include "tp_physics.h"
#include "tp_rng_host.h"

namespace tpe {

struct DevBuf {
    void *p = nullptr;
    size_t n = 0;
};

// Temporary device buffers of one call, freed on every return path.
template <int N> struct ScopedBufs {
    DevBuf b[N];
    ScopedBufs() = default;
    ScopedBufs(const ScopedBufs &) = delete;
    ScopedBufs &operator=(const ScopedBufs &) = delete;
    DevBuf &operator[](int i) { return b[i]; }
    ~ScopedBufs()
    {
        for (DevBuf &x : b)
            if (x.p)
                (void)hipFree(x.p);
    }
};

// xoshiro skip tables of one device, filled once by the first tp_create on
// it (the next caller, if that fails) and only read afterwards (tp_kernels.h).
struct XoTables {
    const uint64_t *m16 = nullptr;     // M^(v 16^j), M one draw
    const uint64_t *b16[2] = {nullptr, nullptr}; // B^(v 16^j): M^(12 * 10 000), the 2^128 jump (by seeding)
    const uint64_t *lanes = nullptr;   // lane tables of every run length, then of the pieces of a stream
    const uint32_t *m16_128 = nullptr, *b16_128[2] = {nullptr, nullptr}, *lanes128 = nullptr; // the same of xoshiro128+
};

struct Ctx {
    int device = 0;
    const XoTables *xo = nullptr;   // null where their set-up has failed so far
    int cus = 1;                    // compute units of the device
    int blocks_per_cu[5][2] = {{1, 1}, {1, 1}, {1, 1}, {1, 1}, {1, 1}}; // resident fused workgroups per CU [source][precision]
    int f32_blocks[4] = {1, 1, 1, 1}; // resident all-f32 wavefronts per CU [source]
    hipStream_t stream = nullptr;
    hipEvent_t ev[5] = {nullptr, nullptr, nullptr, nullptr, nullptr}; // [4]: the device walk's status copy
    std::string err;
    DevBuf mt;       // M^(2^k)
    int km = 0;
    DevBuf r16;             // RANF: jump polynomials of the digits of a number of rounds
    bool r16_ready = false;
    DevBuf draws, origin, p0, per_batch, merged, evq;
    DevBuf parts; // sums of the parts of split batches (MAX_PARTS), allocated by tp_create
    DevBuf f32ev, f32cnt;       // all-f32 mode: per-event values, accepted events of the parts
    tp_stats last{};
    bool timed = false;
    bool marking = true;        // whether mark() records its events (closure calls report no times)
    tp_acc *host_acc = nullptr; // HOST_ACCS accumulators of host memory that kernels write
    // Host staging of the RANF origin: must outlive the asynchronous copies.
    int32_t origin0[56];
    int32_t p00 = 0;
    // faster-evgen: event start positions of the last run and the state after it
    std::vector<uint64_t> fe_starts;
    tp::RanfState fe_end{};
    // device walk: walkers' start lists, their counts and join indices, the
    // joined pieces (begin, length, output offset), and host staging of them
    DevBuf fe_lists, fe_meta, fe_piece;
    DevBuf fe_flag;  // jump seeding: set by a batch walk that left its piece
    DevBuf fe_stat;  // the device walk's stitch status: failed, start n
    uint64_t *fe_stat_host = nullptr; // its pinned host copy (hipHostMalloc)
    DevBuf fe_seq;   // jump seeding: batches left to the one-thread walk
    DevBuf xo_draws, xo128_draws; // faster-evgen on xoshiro256+, on xoshiro128+ (f32): the pieces' uniforms
    DevBuf xo_acc;              // accept bits of the expanded xoshiro pieces: acc1, then acc3
    uint64_t xo_acc_words = 0;  // words per array in xo_acc
    DevBuf adj_u;               // tp_adjoint: the stream's points, expanded
    uint32_t fe_flag_host = 0;
    uint64_t fe_qnext = 0;  // the device walk's start n: where the next chunk begins
    uint64_t fe_xo_end = 0; // faster-evgen on xoshiro256+ with skip-ahead seeding: draws the last run consumed
    uint64_t fe_host_chunks = 0; // faster-evgen: chunks of the last run walked on the host
    uint64_t fe_chunks = 0;      // faster-evgen: chunks the last run was split into
};

constexpr int KM = 32;              // intra-call offsets < 2^32 draws
// RANF rounds per segment of an expansion (one wavefront and one jump each), of
// `rounds` in all: the most, up to 512, that give each SIMD six wavefronts, as a
// round waits on its LDS permutes for several times its issue.  Whole runs with
// segments of 2048, 512, 256, 128 and 64 rounds (faster-evgen): 1e7 events 1412,
// 1074, 1061, 1137, 1298 us; 1.2e6 events 987, 558, 480, 464, 470 us; 5e7 with
// jump seeding 5170, 4423, 4436, 4552, 4997 us; 1e8 8442, 8326, 8721, 9833 us.
constexpr int RANF_R_MIN = 64, RANF_R_MAX = 512;
inline int ranf_seg_rounds(const Ctx *c, uint64_t rounds)
{
    int r = RANF_R_MAX;
    while (r > RANF_R_MIN && rounds / r < 24ull * c->cus)
        r /= 2;
    return r;
}
// Where tp_guard stores an exception's message for tp_last_error.
inline std::string *ctx_err(void *ctx) { return ctx ? &static_cast<Ctx *>(ctx)->err : nullptr; }

inline int fail(Ctx *c, int code, const std::string &msg)
{
    if (c)
        c->err = msg;
    return code;
}

#define HIPCHK(ctx, expr)                                                                              \
    do {                                                                                               \
        hipError_t e_ = (expr);                                                                        \
        if (e_ != hipSuccess)                                                                          \
            return fail((ctx), TP_ERR_HIP, std::string(#expr) + ": " + hipGetErrorString(e_));         \
    } while (0)

// Records event i of the call's times.
inline int mark(Ctx *c, int i)
{
    if (c->marking)
        HIPCHK(c, hipEventRecord(c->ev[i], c->stream));
    return TP_OK;
}

// No event is recorded while one of these lives.
struct Unmarked {
    Ctx *c;
    explicit Unmarked(Ctx *ctx) : c(ctx) { c->marking = false; }
    ~Unmarked() { c->marking = true; }
    Unmarked(const Unmarked &) = delete;
    Unmarked &operator=(const Unmarked &) = delete;
};

// Results that go to the host in the end, up to this many accumulators, are
// written there by the kernels: a copy of its own waits for the last kernel and
// takes some 10 us of the 40 of a small call.
constexpr uint64_t HOST_ACCS = 4096;

inline int ensure(Ctx *c, DevBuf &b, size_t bytes)
{
    if (b.n >= bytes && b.p)
        return TP_OK;
    if (b.p) {
        (void)hipStreamSynchronize(c->stream);
        (void)hipFree(b.p);
        b.p = nullptr;
        b.n = 0;
    }
    hipError_t e = hipMalloc(&b.p, bytes);
    if (e != hipSuccess)
        return fail(c, TP_ERR_NOMEM, std::string("hipMalloc(") + std::to_string(bytes) + "): " + hipGetErrorString(e));
    b.n = bytes;
    return TP_OK;
}

// How a launch of nb batches of n events (each a wavefront's work, or split
// over several) is laid out.
struct Split {
    uint32_t parts, run; // wavefronts per batch, events per lane of each
    int grid;
};
constexpr uint64_t MAX_PARTS = 1u << 16;
// What a kernel's part costs, in issue times of one of its iterations (64
// events): `startup` iterations a part, and `wait` for latencies that other
// wavefronts do not cover, once where the SIMDs' issue is the bound (wavefronts
// that finish early leave their SIMD's time to the others), or `per_round` of
// resident wavefronts where loads are.  `join` is the kernel that joins the
// parts' sums, per `join_batches` batches, `most` the parts it takes; a split
// has to take less than `gain` of the unsplit time.
struct PartCost {
    double startup, wait;
    bool per_round;
    double gain = 1.;
    uint64_t most = MAX_PARTS;
    double join = 0.;
    uint64_t join_batches = 1;
};
// Measured at 100 to 10 000 batches with every run length.  A wavefront with a
// SIMD to itself takes 1.45 of an iteration's issue time (RANF, 1000 batches:
// 444 us in one part each, 344 in two, 317 in three, 307 in four, 308 in eight,
// 336 in sixteen), a part some 3.5 iterations beside its events (10 000 batches:
// 2.76 ms whole, 2.98 in two parts); event loops that read their draws from HBM
// wait 2.6 iterations a round (faster-evgen, 1000 batches with the walk: 1234 us
// whole, 1009 in two parts, 879 in three, which fill the chip once, 951 in
// four); the weighted loop's rows of uniforms come in best in long runs (with
// the flow, 2000 batches take 2 % longer in two parts, 1000 batches 4 % less);
// the all-f32 loop waits 0.8, its separate sums take 42 us per 1536 batches
// (1000 batches: 819 us whole, 492 in two parts, 418 in four, 395 in eight;
// 10 000: 2.99 ms whole, 3.63 in three).
inline PartCost event_part_cost(int source)
{
    return source < 2 ? PartCost{3.5, 0.45, false} : source == 2 ? PartCost{3.5, 0.45, false, 0.85} : PartCost{1.5, 2.6, true};
}
inline PartCost f32_part_cost(int source)
{
    return source == 0   ? PartCost{4., 0.8, false}
           : source == 1 ? PartCost{1., 0.8, false, 1., tpk::F32_MAX_PARTS, 21., 1536}
                         : PartCost{1., 2.6, true, 1., tpk::F32_MAX_PARTS, 21., 1536};
}
// The run length with the least estimated time for nb batches of n events on
// `blocks` resident wavefronts per CU.  lane_runs: a lane takes consecutive
// events, so a short batch leaves lanes idle.
inline Split split_for(uint64_t cus, uint64_t blocks, uint64_t nb, uint32_t n, bool lane_runs, const PartCost &k)
{
    const uint64_t simds = 4 * cus, slots = cus * blocks;
    auto up = [&](uint64_t tasks) { return (double)((tasks + simds - 1) / simds); };
    Split best{0, 0, 0};
    double least = 0.;
    for (uint32_t run : tpk::XO_RUNS) {
        const uint64_t parts = (n + 64ull * run - 1) / (64ull * run), tasks = nb * parts;
        if (parts > 1 && (parts > std::min(slots, k.most) || tasks > MAX_PARTS))
            continue;
        const uint64_t iters = lane_runs ? std::min(run, n) : std::min<uint64_t>(run, (n + 63) / 64);
        const uint64_t rest = tasks % slots;
        const double turns = !k.per_round ? up(tasks) + k.wait
                                          : (double)(tasks / slots) * ((double)slots / (double)simds + k.wait) +
                                                (rest ? up(rest) + k.wait : 0.);
        double cost = ((double)iters + k.startup) * turns;
        if (parts > 1)
            cost += k.join * (double)((nb + k.join_batches - 1) / k.join_batches);
        if (!best.parts || cost < least * (best.parts == 1 ? k.gain : 1.)) {
            least = cost;
            // a wavefront that takes several parts keeps its place in the batch
            best = Split{(uint32_t)parts, run, (int)std::min(tasks, slots / parts * parts)};
        }
    }
    if (!best.parts) // no split within the limits
        best = Split{1, (n + 63) / 64, (int)std::min(nb, slots)};
    return best;
}
inline Split split_for(const Ctx *c, int source, int precision, uint64_t nb, uint32_t n)
{
    return split_for((uint64_t)c->cus, (uint64_t)c->blocks_per_cu[source][precision], nb, n, source == 0,
                     event_part_cost(source));
}
inline Split split_for_f32(const Ctx *c, int source, uint64_t nb, uint32_t n)
{
    return split_for((uint64_t)c->cus, (uint64_t)c->f32_blocks[source], nb, n, source == 0, f32_part_cost(source));
}

// The jump of a wavefront that strides over parts of the one RANF stream.
inline void set_ranf_jump(tpk::RanfSource &R, const Split &s, uint64_t nb, uint32_t batch_size, uint32_t n)
{
    R.jump_rounds = 0;
    if (R.origin || R.later || nb * s.parts <= (uint64_t)s.grid)
        return;
    // the least number of rounds from the last one of a part to the first of
    // the wavefront's next (a part of whole runs: that or one more)
    const uint64_t stride = 12ull * batch_size * (s.grid / s.parts), part = 12ull * std::min<uint64_t>(64ull * s.run, n);
    R.jump_rounds = (stride - part + 1) / 55;
    const tp::RanfPoly q = tp::ranf_poly_rounds(R.jump_rounds);
    std::copy(q.begin(), q.end(), R.jump);
}

// The lane table of a run length, or null if there is none (split_for picks a
// run of XO_RUNS for every batch of up to 64 * 157 * the resident wavefronts).
inline const uint32_t *xo_lane_table(const uint32_t *lanes, size_t words, uint32_t run)
{
    for (int i = 0; i < tpk::XO_NRUNS; ++i)
        if (tpk::XO_RUNS[i] == run)
            return lanes + i * words;
    return nullptr;
}

// The event loop on a.nb batches of n events, split as split_for says, with
// the batches' sums in a.out.
inline int launch_event_loop(Ctx *c, tpk::FusedArgs &a, int source, uint32_t n)
{
    const Split s = split_for(c, source, a.precision, a.nb, n);
    a.parts = s.parts;
    a.run = s.run;
    a.part_out = c->parts.p;
    if (source == 0)
        a.lanes = reinterpret_cast<const uint64_t *>(
            xo_lane_table(reinterpret_cast<const uint32_t *>(c->xo->lanes), 2 * tpk::XO_LANE_WORDS, s.run));
    if (source == 0 && !a.lanes)
        return fail(c, TP_ERR_INTERNAL, "no lane table for this batch size");
    if (source == 1)
        set_ranf_jump(a.ranf, s, a.nb, a.batch_size, n);
    tpk::launch_fused(a, source, s.grid, c->stream);
    HIPCHK(c, hipGetLastError());
    if (s.parts > 1) {
        tpk::launch_batch_sums(a, c->stream);
        HIPCHK(c, hipGetLastError());
    }
    return TP_OK;
}

// The same in the all-f32 mode, with the sums in event order.
inline int launch_f32_batches(Ctx *c, tpk::F32Args &a, uint32_t n)
{
    const Split s = split_for_f32(c, a.source, a.nb, n);
    a.parts = s.parts;
    a.run = s.run;
    a.wide = tpd::f32_wide_range(a.P.e_total, a.P.e_min, a.P.cut_beam);
    if (a.source == 0)
        a.lanes = xo_lane_table(c->xo->lanes128, tpk::XO128_LANE_WORDS, s.run);
    if (a.source == 0 && !a.lanes)
        return fail(c, TP_ERR_INTERNAL, "no lane table for this batch size");
    if (a.source == 1)
        set_ranf_jump(a.ranf, s, a.nb, a.batch_size, n);
    if (!tpk::f32_sums_in_kernel(a)) {
        a.ev_stride = a.nb * a.batch_size;
        int rc = ensure(c, c->f32ev, a.ev_stride * (a.source == 0 ? 6 : 5) * sizeof(float));
        if (!rc)
            rc = ensure(c, c->f32cnt, a.nb * a.parts * sizeof(uint32_t));
        if (rc)
            return rc;
        a.ev = static_cast<float *>(c->f32ev.p);
        a.counts = static_cast<uint32_t *>(c->f32cnt.p);
    }
    tpk::launch_f32_events(a, s.grid, c->stream);
    HIPCHK(c, hipGetLastError());
    if (!tpk::f32_sums_in_kernel(a)) {
        tpk::launch_f32_accumulate(a, c->stream);
        HIPCHK(c, hipGetLastError());
    }
    return TP_OK;
}

// Device-side constants of a run, computed exactly as the reference does on
// the host (coupling.rs, resacc.rs:59-100, evgen.rs:66-69, spinor.rs:37-44).
tpd::Params make_params(const tp_params *p);
tpd::Params make_event_params(const tp_params *p, int precision);
tpd::FParams make_fparams(const tp_params *p);

} // namespace tpe
