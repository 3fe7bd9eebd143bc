// tp_ctx.h -- the engine context shared by the event-loop and flow entry
// points (internal; not part of the C ABI).
#pragma once

#include "tp_guard.h"

#include <hip/hip_runtime.h>

#include <algorithm>
#include <map>
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

struct Tables { // device copy of the powers 2^k of a GF(2) matrix
    DevBuf bt;
    int kb = 0;
};

// xoshiro256+ skip tables of one device, filled once by the first tp_create on
// it and only read afterwards (tp_kernels.h).
struct XoTables {
    int rc = TP_ERR_INTERNAL;
    std::string err;
    const uint64_t *m16 = nullptr;     // M^(v 16^j), M one draw
    const uint64_t *b16[2] = {nullptr, nullptr}; // B^(v 16^j): M^(12 * 10 000), the 2^128 jump (by seeding)
    const uint64_t *lanes = nullptr;   // lane tables of every run length
};

struct Ctx {
    int device = 0;
    const XoTables *xo = nullptr;
    int cus = 1;                    // compute units of the device
    int blocks_per_cu[5][2] = {{1, 1}, {1, 1}, {1, 1}, {1, 1}, {1, 1}}; // resident fused workgroups per CU [source][precision]
    hipStream_t stream = nullptr;
    hipEvent_t ev[5] = {nullptr, nullptr, nullptr, nullptr, nullptr}; // [4]: the device walk's status copy
    std::string err;
    DevBuf mt;       // M^(2^k)
    int km = 0;
    std::map<std::string, std::unique_ptr<Tables>> tables;
    DevBuf r16;             // RANF: jump polynomials of the digits of a number of rounds
    bool r16_ready = false;
    DevBuf draws, origin, p0, per_batch, merged, evq;
    DevBuf parts; // sums of the parts of split batches (MAX_PARTS), allocated by tp_create
    DevBuf mt128, bt128, f32ev; // all-f32 mode: xoshiro128+ tables, per-event values
    std::string bt128_key;
    int bt128_kb = 0;
    DevBuf st128;               // all-f32 mode: B^grid, the grid-stride advance
    std::string st128_key;
    tp_stats last{};
    bool timed = false;
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
    DevBuf xo_states, xo_draws; // faster-evgen on xoshiro256+: piece states and uniforms
    DevBuf xo128_states, xo128_draws, xo128_pt; // the same on xoshiro128+ (f32), and the piece matrix powers
    DevBuf xo_acc;              // accept bits of the expanded xoshiro pieces: acc1, then acc3
    DevBuf xo_lt, xo128_lt;     // the expanding lanes' skip matrices (xoshiro256+, xoshiro128+)
    uint64_t xo_acc_words = 0;  // words per array in xo_acc
    std::string xo128_pt_key;
    int xo128_pt_kb = 0;
    DevBuf adj_u;               // tp_adjoint: the stream's points, expanded
    uint32_t fe_flag_host = 0;
    uint64_t fe_qnext = 0;  // the device walk's start n: where the next chunk begins
    uint64_t fe_xo_end = 0; // faster-evgen on xoshiro256+ with skip-ahead seeding: draws the last run consumed
    uint64_t fe_host_chunks = 0; // faster-evgen: chunks of the last run walked on the host
    uint64_t fe_chunks = 0;      // faster-evgen: chunks the last run was split into
};

constexpr int KM = 32;              // intra-call offsets < 2^32 draws
constexpr int RANF_R = 2048;        // RANF rounds per expansion segment (one jump per segment)
// Batches per RANF expansion + event-loop launch: two full strides of the
// 3072-wavefront persistent grid (one wavefront per batch), so no launch ends
// on a partly idle stride; 6144 * 120000 int32 = 2.95 GB of stream.
constexpr uint64_t RANF_CHUNK_BATCHES = 6144;

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
// The run length with the least estimated time.  A wavefront takes `run`
// iterations and a start-up of about 2 (the xoshiro stream's skip; half an
// iteration for streams read from memory).  `slots` wavefronts are resident at
// once and share 4 SIMDs per CU: a SIMD with one wavefront spends 1.4 times
// the issue time of an iteration (measured: 4900 cycles against 3400), one
// with several their sum.  So 1000 batches take 2 parts each rather than leave
// two wavefronts of three idle, 10 000 take 4 rather than fill a fourth round
// of 3072 to a quarter, and one closure call takes a part per 64 events.
inline Split split_for(const Ctx *c, int source, int precision, uint64_t nb, uint32_t n)
{
    const uint64_t simds = 4ull * c->cus, slots = (uint64_t)c->cus * c->blocks_per_cu[source][precision];
    Split best{0, 0, 0};
    double least = 0.;
    for (uint32_t run : tpk::XO_RUNS) {
        const uint64_t parts = (n + 64ull * run - 1) / (64ull * run), tasks = nb * parts;
        if (parts > 1 && (parts > slots || tasks > MAX_PARTS))
            continue;
        const uint64_t iters = source == 0 ? std::min(run, n) : std::min<uint64_t>(run, (n + 63) / 64);
        const uint64_t rest = tasks % slots;
        const double turns = (double)(tasks / slots) * ((double)slots / (double)simds) +
                             (rest ? std::max(1.4, (double)((rest + simds - 1) / simds)) : 0.);
        const double cost = ((double)iters + (source == 0 ? 2. : 0.5)) * turns;
        if (!best.parts || cost < least) {
            least = cost;
            // a wavefront that takes several parts keeps its place in the batch
            best = Split{(uint32_t)parts, run, (int)std::min(tasks, slots / parts * parts)};
        }
    }
    if (!best.parts) // batches of more than 64 * 157 events, in more parts than are resident
        best = Split{1, (n + 63) / 64, (int)std::min(nb, slots)};
    return best;
}

// The event loop on a.nb batches of n events, split as split_for says, with
// the batches' sums in a.out.
inline void launch_event_loop(const Ctx *c, tpk::FusedArgs &a, int source, uint32_t n)
{
    const Split s = split_for(c, source, a.precision, a.nb, n);
    a.parts = s.parts;
    a.run = s.run;
    a.part_out = c->parts.p;
    if (source == 0) {
        a.lanes = nullptr;
        for (int i = 0; i < tpk::XO_NRUNS; ++i)
            if (tpk::XO_RUNS[i] == s.run)
                a.lanes = c->xo->lanes + (size_t)i * tpk::XO_LANE_WORDS;
    }
    a.rjump_rounds = 0;
    const uint64_t stride = 12ull * a.batch_size * (s.grid / s.parts), part = 12ull * std::min<uint64_t>(64ull * s.run, n);
    if (source == 1 && !a.rorigin && a.nb * s.parts > (uint64_t)s.grid) {
        // the least number of rounds from the last one of a part to the first
        // of the wavefront's next (a part of whole runs: that or one more)
        a.rjump_rounds = (stride - part + 1) / 55;
        const tp::RanfPoly q = tp::ranf_poly_rounds(a.rjump_rounds);
        std::copy(q.begin(), q.end(), a.rjump);
    }
    tpk::launch_fused(a, source, s.grid, c->stream);
    if (s.parts > 1)
        tpk::launch_batch_sums(a, c->stream);
}

// Device-side constants of a run, computed exactly as the reference does on
// the host (coupling.rs, resacc.rs:59-100, evgen.rs:66-69, spinor.rs:37-44).
tpd::Params make_params(const tp_params *p);
tpd::Params make_event_params(const tp_params *p, int precision);
tpd::FParams make_fparams(const tp_params *p);

} // namespace tpe
