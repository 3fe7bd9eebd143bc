// tp_kernels.h -- host-side launch interface of the gfx950 kernels
// (implemented in tp_kernels.hip).  Plain structs of device pointers; no
// ownership here.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include "tp_physics.h"

namespace tpk {


// The RANF stream of a run.  Batch b's events draw from position p0 + 12
// batch_size b on of the stream whose round 0 is `round` (X[1..55]); with jump
// seeding (origin non-null) batch b > 0 has a stream of its own, round 0 at
// origin[56 (b - first)] and positions from 0.  A stream whose round 0 holds
// values outside [0, 1e9) goes on at each multiple s of RANF_LATE rounds from
// `later`: at later[56 (b - first)] (s = 1, no batch gets further) with jump
// seeding, else at later[56 (s - first)].  Without such a stream later is null
// (the event loops then run kernels that leave the rule out).
constexpr uint32_t RANF_LATE = 2048, RANF_LATE_R16 = 2 * 15 + 7; // 8 * 16^2: its place in r16
struct RanfSource {
    int32_t round[56];
    uint32_t p0;
    const int32_t *origin, *later;
    uint64_t first;       // the first batch that origin and later hold, or the first s that later does
    const uint32_t *r16;  // x^(55 v 16^j) mod the recurrence's polynomial, 55 coefficients each, v = 1..15,
                          // for the digits of a number of rounds
    uint32_t jump[55];    // x^(55 jump_rounds): from the end of a wavefront's part to near its next one
    uint64_t jump_rounds; // (0: none)
};

// Arguments of the fused event-loop kernel.
struct FusedArgs {
    tpd::Params P;
    uint64_t nb;           // batches in this launch
    uint64_t b_first;      // global index of the first batch of this launch
    uint64_t num_events;   // events of the whole run (for the last, partial batch)
    uint32_t batch_size;   // events per full batch
    int32_t precision;     // tp_precision
    // A batch's events are split over `parts` wavefronts, each taking runs of
    // `run` events per lane: part s holds events 64 run s .. of the batch.
    // With more than one part each writes its sums to part_out[batch * parts + s]
    // and launch_batch_sums adds them up.
    uint32_t parts, run;
    void *part_out;        // tp_acc*
    // xoshiro source: part s of batch b starts at M^(12 * 64 run s) * B^b * s0
    // with B = M^(12*batch_size) or the 2^128 jump, and its lane l
    // 12 run l draws later.
    uint64_t s0[4];
    const uint64_t *m16, *b16; // M^(v 16^j), B^(v 16^j), v = 1..15: digits of an exponent (tp_xoshiro.h)
    const uint64_t *lanes;     // images of the state's nibbles under the lanes' skips for `run`
    // tp_events: M^(2^k), k < km, each 256x4 words
    const uint64_t *mt;
    int32_t km;
    RanfSource ranf;       // RANF source
    // expanded RANF values: faster-evgen (below), tp_events
    const int32_t *draws;
    // weighted source (importance sampling): uniforms (f64) and weight 1/q(u)
    // per event; event i = batch_size*(b - b_first) + e has its uniform j at
    // u[j * u_stride + i] (one row per uniform, so a wavefront's loads are
    // contiguous) and its weight at invq[i]; every |M|^2 is multiplied by
    // its weight.
    const double *u;
    const double *invq;
    uint64_t u_stride;
    // faster-evgen source (RANF, f64): stream values from position qbase in
    // draws[], event e of batch (b - b_first) starting at stream position
    // evq[batch_size*(b - b_first) + e].
    const uint64_t *evq;
    uint64_t qbase;
    // faster-evgen from the xoshiro256+ stream (source 4): its uniforms, the
    // starts evq and qbase as above
    const double *xdraws;
    // faster-evgen: the stream's accept bits (tpd::RerollBits), valid below
    // blimit, or for pieces (bstride > 0) batch k's below (k + 1) * bstride;
    // acc1 null: re-rolls one pair at a time
    const uint32_t *acc1;
    uint64_t bbase, blimit, bstride;
    // output: one accumulator per batch, index b - b_first
    void *out;             // tp_acc*
};

// Arguments of the RANF expansion kernel (one wavefront per segment of R
// rounds).  A piece is one stream origin: the reference's master stream in
// skip-ahead mode, or one reseeded batch stream in jump mode.
struct RanfArgs {
    const int32_t *origin; // [npieces][56] round X[1..55] at [1..55]
    const int32_t *p0;     // [npieces] values of the origin round already consumed
    uint64_t d_begin, d_end; // window of draws (piece-relative) to write
    uint64_t seg_first;    // first segment index of the window
    uint64_t nsegs;        // segments per piece in this launch
    uint64_t piece_stride; // output offset between pieces
    const uint32_t *r16;   // digits of a number of rounds, as FusedArgs
    int32_t R;             // rounds per segment
    int32_t *out;
    // faster-evgen: accept bits of every round the launch generates (bits 1:
    // the unit-disc test in f64, 2: in f32; 0: none), as FeWalkArgs.  Piece
    // k's segment s fills the words from k * bits_piece_words + (s - seg_first)
    // * 55 R / 32 on (55 R a multiple of 32), bit j = the segment's j-th position.
    int32_t bits;
    uint64_t bits_piece_words;
    uint32_t *acc1, *acc3;
};

void launch_fused(const FusedArgs &a,
                  int source /*0 xoshiro, 1 RANF, 2 weighted, 3 faster-evgen RANF, 4 faster-evgen xoshiro (f64 only)*/,
                  int grid, hipStream_t st);
int fused_blocks_per_cu(int source, int precision); // resident workgroups per CU (occupancy)
// The sums of a.nb batches from their parts, in the order of the parts.
void launch_batch_sums(const FusedArgs &a, hipStream_t st);

// ---- xoshiro256+ skip tables (once per device) --------------------------------
// Events per lane that a wavefront of the event loop may take, each with a
// lane table of its own: a batch of 10 000 events in 1, 2, 3, 4, 8, 16, 32, 40,
// 79 and 157 parts.
constexpr uint32_t XO_RUNS[] = {157, 79, 53, 40, 20, 10, 5, 4, 2, 1};
constexpr int XO_NRUNS = sizeof XO_RUNS / sizeof XO_RUNS[0];
// Lane tables: of every run length, and of the lanes that expand the stream for
// faster-evgen, 12 * XO_EXPAND_RUN draws each.
constexpr uint32_t XO_EXPAND_RUN = 32;
constexpr int XO_NTABLES = XO_NRUNS + 1;
// Exponents below 2^52 draws and 2^32 batches: no run is longer, as the
// accumulators of 2.8e9 batches fill 288 GB (faster-evgen: 4.7e14 draws).
constexpr int XO_M_DIGITS = 13, XO_B_DIGITS = 8;
constexpr size_t XO_MAT_WORDS = 1024;                    // 256 columns of 4 words
constexpr size_t XO_LANE_WORDS = 64 * 16 * 64 * 4;       // per run length: 2 MiB
// tab16[(15 j + v - 1) * 1024 ..] = B^(v 16^j) from pow2[k * 1024 ..] = B^(2^k), k < 4 digits.
void launch_xo_digit_table(const uint64_t *pow2, int digits, uint64_t *tab16, hipStream_t st);
// The lane tables of every run length of XO_RUNS, in that order, and XO_EXPAND_RUN's.
void launch_xo_lane_tables(const uint64_t *m16, uint64_t *lanes, hipStream_t st);
// Per-event diagnostics: one thread per event, same device code as the loop.
// Event e draws from offset 12*e (xoshiro: a.s0 with a.mt; buffer: a.draws).
struct EventOut {
    double *u;     // [n][12]
    double *p;     // [n][3][4]
    int32_t *keep; // [n]
    double *m;     // [n][5]
};
void launch_events(const FusedArgs &a, int source, uint32_t n, const EventOut &o, hipStream_t st);
void launch_ranf_expand(const RanfArgs &a, uint64_t npieces, hipStream_t st);
// Per-batch RANF origins of jump mode: seeded_new(seed0 + 123456*b).
void launch_ranf_seed(int32_t seed0, uint64_t b_first, uint64_t nb, const uint32_t *r16, int32_t *origin, int32_t *p0,
                      int32_t *later, hipStream_t st);
// The rounds RANF_LATE s, s = first .. first + n - 1, of a caller's such stream.
void launch_ranf_late(const int32_t round[56], const uint32_t *r16, uint64_t first, uint64_t n, int32_t *later, hipStream_t st);
// In-order left fold of nb accumulators (resacc.rs:133-139) into *merged.
// In-order fold of nb accumulators; f32 = 1 adds in float (all-f32 mode).
void launch_merge(const void *per_batch, uint64_t nb, void *merged, hipStream_t st, int f32 = 0);

// ---- all-f32 mode: events and per-batch sums in event order -----------------
// Batches are split over wavefronts as in FusedArgs.  A wavefront that has a
// whole batch forms its sums in event order itself (no per-event values reach
// memory), except with the xoshiro128+ stream in registers, whose lanes take
// runs of events; otherwise launch_f32_accumulate forms them from the events'
// values.
struct F32Args {
    tpd::FParams P;
    uint64_t nb, b_first, num_events;
    uint32_t batch_size;
    int32_t source;        // 0 xoshiro128+ in registers, 1 RANF, 2 faster-evgen on
                           // RANF draws, 3 faster-evgen on xoshiro128+ uniforms (x32draws)
    uint32_t parts, run;
    bool wide;             // f32_wide_range of P
    uint32_t s0[4];        // xoshiro128+ state of the run, and its skip tables as in FusedArgs
    const uint32_t *m16, *b16;
    const uint32_t *lanes;
    RanfSource ranf;       // source 1
    // faster-evgen (source 2, RANF): event starts evq[batch_size*(b - b_first) + e]
    // in draws from position qbase, as FusedArgs
    const int32_t *draws;
    const uint64_t *evq;
    uint64_t qbase;
    const float *x32draws; // faster-evgen (source 3): xoshiro128+ uniforms from position qbase
    const uint32_t *acc1;  // faster-evgen: accept bits, as FusedArgs
    uint64_t bbase, blimit, bstride;
    // Events' values.  Source 0: m[5] and keep (0/1) of event e of batch
    // b - b_first at ev[6 * (batch_size*(b - b_first) + e)].  Others: the
    // accepted events of a part in event order, m[c] of the i-th at
    // ev[c * ev_stride + batch_size*(b - b_first) + the part's first event + i],
    // their number at counts[(b - b_first) * parts + part].
    float *ev;
    uint64_t ev_stride;
    uint32_t *counts;
    void *out;             // tp_acc per batch, index b - b_first (f32 values)
};
constexpr uint32_t F32_MAX_PARTS = 256; // parts that launch_f32_accumulate joins (source 0: any number)
inline bool f32_sums_in_kernel(const F32Args &a) { return a.source != 0 && a.parts == 1; }
int f32_blocks_per_cu(int source); // resident wavefronts per CU
void launch_f32_events(const F32Args &a, int grid, hipStream_t st);
void launch_f32_accumulate(const F32Args &a, hipStream_t st); // not after f32_sums_in_kernel

// xoshiro128+ skip tables, as launch_xo_digit_table and launch_xo_lane_tables.
constexpr size_t XO128_MAT_WORDS = 512;                  // 128 columns of 4 words
constexpr size_t XO128_LANE_WORDS = 32 * 16 * 64 * 4;    // per run length: 512 KiB
void launch_xo128_digit_table(const uint32_t *pow2, int digits, uint32_t *tab16, hipStream_t st);
void launch_xo128_lane_tables(const uint32_t *m16, uint32_t *lanes, hipStream_t st);

// ---- faster-evgen stream walk on the device ----------------------------------
// Event starts of the faster-evgen draws (evgen.rs:209-255, random_array's
// discarded round leftovers ranf.rs:89-92), split like the host walk: walker
// k starts at seg_origin + k*seg (walker 0 at the true start q_start), as if
// an event started there, and records its event starts up to the next segment,
// then on to where it meets that segment's walker, at most `overlap` positions
// past the segment's end.  Positions are counted from the start of the master
// state's round; buf holds positions [qbase, qlimit).
struct FeWalkArgs {
    const int32_t *buf;    // RANF values of positions qbase .. qlimit - 1 (kinds 0, 1)
    int32_t kind;          // 0: RANF, unit-disc test in f64; 1: RANF, in f32; 2: xoshiro256+; 3: xoshiro128+ (f32)
    // The walk reads accept bits, not values.  Bit i of acc1 (word i / 32,
    // bit i % 32) is 1 when the point (2u - 1) of positions bbase + i and
    // bbase + i + 1 passes the unit-disc test; acc3 likewise for bbase + i and
    // bbase + i + 3 (the three points of each event's 6 values).  buf (RANF)
    // still serves the one-thread walk of a batch the segments leave uncovered.
    const uint32_t *acc1, *acc3;
    uint64_t bbase;        // position of bit 0 of acc1 / acc3
    uint64_t qbase, qlimit;
    uint64_t q_start;
    uint64_t seg_origin, seg, overlap;
    uint32_t nwalkers;
    uint32_t cap;          // list capacity per walker (>= its longest possible walk)
    uint32_t *lists;       // [nwalkers][cap] event starts, ascending, from the segment's start
    uint32_t *len, *tail;  // [nwalkers] starts in the own segment; where the walk enters the next one
    uint32_t *counts;      // [nwalkers] starts in all
    int32_t *join_prev;    // [nwalkers] for k >= 1: index in list k-1 of the first start >= the
    int32_t *join_next;    //   start of segment k that list k also holds, and its index there (-1: none)
};
void launch_fe_walk(const FeWalkArgs &a, hipStream_t st);
// Copies the pieces of the joined walk into out: piece k is lists[k][begin[k] ..
// begin[k] + len[k]) at out[off[k] ..].
// The chaining of the joined walk on the device: piece k of the first `need`
// starts is lists[k][begin[k] .. begin[k] + len[k]) at out[off[k] ..];
// status[0] = 1 when some walker does not meet its successor after its own
// join, or the pieces hold fewer than `need` starts; else status[1] = start
// need - 1.  status holds FE_STITCH_STATUS words (the rest: per-block sums and
// flags); at most 256 * FE_STITCH_THREADS walkers.
constexpr int FE_STITCH_THREADS = 1024;
constexpr int FE_STITCH_STATUS = 2 + 2 * FE_STITCH_THREADS;
void launch_fe_stitch(const FeWalkArgs &a, uint64_t need, uint32_t *begin, uint32_t *len, uint64_t *off,
                      uint64_t *status, hipStream_t st);
void launch_fe_scatter(const FeWalkArgs &a, const uint32_t *begin, const uint32_t *len, const uint64_t *off,
                       uint64_t *out, hipStream_t st);

// faster-evgen with jump seeding (faster-threading): every batch reseeds, so
// each batch's stream is its own piece and is walked by one thread from the
// piece's first value.  Piece k (batch b_first + k) holds the frame positions
// q of its state (q counted from the start of the state's round) at
// buf[k * piece_stride + q], piece_stride a multiple of 55, so that the
// global position G = k * piece_stride + q keeps q's place in its round
// (G % 55 = q % 55).  evq[k * batch_size + e] receives event e's start as G.
// A walk that would leave its piece sets *overflow and fills the rest of its
// batch with the piece's first position (every later read stays in bounds).
// The xoshiro pieces (kinds 2, 3) hold uniforms from position 0 of each
// batch's own stream (p0 null), and the walk reads their accept bits.
//
// Each batch is walked by S segment walkers, as the one-stream walk is
// (walker s of batch k starts at k * piece_stride + s * seg, walker 0 at the
// batch's first position), each on to where it meets a later one, not always
// the next; a batch whose chain of walkers ends before its events are covered
// is walked by one thread from its first position.
struct FeBatchWalkArgs {
    const int32_t *buf;    // RANF pieces (kinds 0, 1)
    int32_t kind;          // 0: RANF, unit-disc test in f64; 1: in f32 (all-f32 mode); 2: xoshiro256+;
                           // 3: xoshiro128+ (all-f32 mode)
    const uint32_t *acc1, *acc3; // accept bits of the pieces' positions G, as FeWalkArgs (bbase 0)
    uint64_t piece_stride;
    const int32_t *p0;     // [nb] frame position of each piece's first value (RANF)
    uint64_t nb, b_first, num_events;
    uint32_t batch_size;
    uint64_t *evq;
    uint32_t *overflow;
    uint32_t S;            // walkers per batch
    uint64_t seg, overlap; // segment length (a multiple of 55 for RANF) and overlap
    uint32_t cap;          // list capacity per walker
    uint32_t *lists;       // [nb * S][cap], len, tail and counts [nb * S] as FeWalkArgs
    uint32_t *len, *tail, *counts;
    int32_t *next;         // [nb * S] the walker of the batch it meets (-1: none)
    uint32_t *met;         // [nb * S] and the index in that one's list
    uint32_t *seq;         // [nb] 1: walk the batch with one thread
};
void launch_fe_walk_batches(const FeBatchWalkArgs &a, hipStream_t st);

// Pieces of the xoshiro256+ stream: piece k starts from J^(b_first + k) s0
// (J the 2^128 jump with jump seeding, each piece a batch's stream) or, with no
// b16, (b_first + k) * piece_len draws after s0 (the pieces tiling one stream)
// and holds its first piece_len uniforms at xbuf[k * piece_len ..], and the
// accept bits of those positions at acc1 / acc3 (the last three positions' bits
// from the draws that follow the piece: the next piece's first ones when the
// pieces tile one stream).
struct XoPieceArgs {
    uint64_t s0[4];
    const uint64_t *m16, *b16; // as FusedArgs
    const uint64_t *lanes;     // XO_EXPAND_RUN's table
    uint64_t nb, b_first;
    uint64_t piece_len;        // uniforms per piece: a multiple of 64 * 12 * XO_EXPAND_RUN, one wavefront's
    double *xbuf;              // [nb][piece_len]
    uint32_t *acc1, *acc3;     // [nb][piece_len / 32] accept bits of the positions, as FeWalkArgs
};
void launch_xo_expand(const XoPieceArgs &a, hipStream_t st);

// The same for the xoshiro128+ stream of the all-f32 mode (J the 2^64 jump; f32
// uniforms, and the unit-disc test in f32).
struct Xo128PieceArgs {
    uint32_t s0[4];
    const uint32_t *m16, *b16, *lanes;
    uint64_t nb, b_first;
    uint64_t piece_len;
    float *xbuf;
    uint32_t *acc1, *acc3;
};
void launch_xo128_expand(const Xo128PieceArgs &a, hipStream_t st);

} // namespace tpk

namespace tpk {

// Arguments of the adjoint kernel (tp_adjoint).
// The adjoint kernels run one 64-lane workgroup per 64 consecutive points,
// one point per lane, and store the rows through LDS.  Points of the
// xoshiro stream (u_in null) are first expanded into u_gen.
struct AdjArgs {
    tpd::Params P;
    tpd::HelicityK hk;     // f64: the sums in the caller's units
    double w;              // RAMBO event weight
    uint64_t n;            // points
    // uniforms: u_in (n x 12 doubles) if non-null, else xoshiro from s0,
    // expanded into u_gen (n x 12 doubles) `run` points per lane
    const double *u_in;
    double *u_gen;
    uint64_t s0[4];
    uint64_t first;        // of the stream's points, 12 draws each
    const uint64_t *m16, *lanes; // as FusedArgs
    uint32_t run;          // one of XO_RUNS
    void *F, *dF_du, *dF_dp; // [n][5], [n][5][12], [n][5][12] of double or float
};
void launch_adjoint(const AdjArgs &a, int precision /*TP_PREC_F64 or TP_PREC_F32*/, hipStream_t st);

} // namespace tpk
