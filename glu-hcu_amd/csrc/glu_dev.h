// Device-resident tables of one sparsity pattern (POD structs of device
// pointers, passed by value to kernels or stored in device memory for the
// fused multi-matrix launch).
//
// Layout in HBM (all 32-bit indices, one copy per pattern):
//   factor: per level, 16-byte update items (target, L, U and pivot
//           positions of one scalar update), merge entries with their source
//           lists, and 8-byte division items.
//   solves: row lists per level for the four triangular sweeps.
//   refine: CSR of the original A (row pointers, columns, source index into
//           the caller's CSC values), per-LU-position source index and the
//           frozen MC64 scale vectors.
// Values (FP32 L\U, FP64 A, FP64 x/b) are separate buffers indexed by
// matrix; a batch lays matrices out back to back (matrix-major).
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>

namespace glu {

// An entry updated by several pivot columns of one level: one lane owns it
// and applies the updates in increasing column order (deterministic).
struct MergeSrc {
    uint32_t lpos;     // CSC position of L(i,k) (not yet divided)
    uint32_t upos;     // CSC position of U(k,j)
    uint32_t dpos;     // CSC position of the pivot U(k,k)
    uint32_t pad;
};

constexpr uint32_t kLongTask = 0x80000000u;
// Dataflow sweeps: rows with at most this many entries are taken a lane
// each, with all their entries prefetched; longer rows a wave each.
constexpr uint32_t kDfLaneRow = 16;

// Rows / merge entries longer than this are processed by a whole wave.
constexpr uint32_t kLongRow = 64;
constexpr int kMaxKrylov = 4;     // largest restart length of the batch refinement
constexpr uint32_t kLongMerge = 32;

// Flag of a division item: the first L entry of its column, whose lane also
// stores the GESP pivot.
constexpr uint32_t kFirstBit = 0x80000000u;

// Per-level items of the right-looking factorization:
//   column task  (a wave) A(i,j) += -(A(i,k) / A(k,k) * A(k,j)) for targets
//                exactly one column of the level updates;
//   merge        all updates of an entry several columns of the level
//                update, in increasing column order (a lane, or a wave);
//   divide       A(i,k) /= A(k,k) for the columns of the previous level
//                {lpos, dpos | kFirstBit} (deferred so a level needs one
//                barrier).

// One LDS window: steps [l0, l1) with the nslot values they touch staged in
// LDS (pos[slot] is the slot's CSC position), run from per-wave streams of
// chunks: wave w takes chunks [wptr[w], wptr[w + 1]) in order, a chunk being
// 16 bytes (eight 16-bit slots) per lane and a header
// {kind << kWinKindShift | step - l0}:
//   kWinCol    {l, d, u0, t0, u1, t1, u2, t2}: S[ti] += -(S[l] / S[d] * S[ui])
//   kWinMerge  {t, flags, l0, u0, d0, l1, u1, d1}: two sources of the lane's
//              merge entry t, the running value kept by the lane from the
//              chunk with kWinFirst to the one with kWinLast
//   kWinGroup  {l0, u0, d0, l1, u1, d1, t, flags}: 16 lanes share merge entry
//              t, lane j holding sources j and 16 + j of the chunk's 32
//              (kWinGroup1: only the first 16 are used)
//   kWinOut    {l, d, u0, u1} and two 32-bit places o0, o1 (~0: none): the
//              products S[l] / S[d] * S[ui] to out[oi] (phases, after the
//              last step)
// Every wave passes one barrier per step.  Unused places address three kinds
// of extra slots after the values: a 0 (slot nslot), a 1 (nslot + 1) and one
// target a lane that nothing reads (nslot + 2 + lane), so that no chunk needs
// tests: a missing update computes 0 / 1 * 0 and a missing source subtracts
// +0, which changes no value.
constexpr uint32_t kWinExtra = 66;        // extra slots
constexpr uint32_t kWinKindShift = 29;
constexpr uint32_t kWinCol = 0, kWinMerge = 1, kWinGroup1 = 2, kWinGroup = 3, kWinOut = 4;
constexpr uint32_t kWinFirst = 1, kWinLast = 2;

struct WinDev {
    int32_t l0, l1;
    uint32_t nslot, nwave;     // nwave: streams (waves past them only pass the barriers)
    const uint32_t *pos;       // [nslot]
    const uint4 *prog;         // [64 chunks]
    const uint32_t *hdr;       // [chunks]
    const uint32_t *wptr;      // [nwave + 1]
};

// One phase of the factorization: a run of leading steps whose columns fall
// into components that share no entry (bins of components, a workgroup each,
// their columns' and rows' entries in LDS as a window's).  Updates of entries
// of later columns can come from several bins: their products go to out, the
// products of one entry in the order of the steps and columns, and are
// subtracted once the phase is done.  Entries of up to kAsmLane products come
// first in groups of 64 (a lane each, product k of lane i at base + 64 k + i),
// the rest a wave each (contiguous).
constexpr uint32_t kAsmLane = 32;

struct AsmWave {
    uint32_t tgt, base, cnt, pad;
};

struct PhaseDev {
    const WinDev *bin;         // [nbin]
    const uint2 *grp;          // [ngrp]: {base, most products of a lane}
    const uint32_t *tgt;       // [64 ngrp] entry (~0: none)
    const uint8_t *cnt;        // [64 ngrp] its products
    const AsmWave *wav;        // [nwav]
    float *out;                // the products
    uint32_t nbin, ngrp, nwav, nslot;   // nslot: the largest bin's
};

// The leading launches of a group of distinct patterns: items {member, block
// of values | bin | first wave}, phase round by phase round.
constexpr uint32_t kGroupRounds = 8;       // phases of a member taken this way, at most

struct GroupLaunch {
    const uint2 *values = nullptr, *bins[kGroupRounds] = {}, *asms[kGroupRounds] = {};
    const PhaseDev *phase[kGroupRounds] = {};   // by member
    uint32_t nvalues = 0, nbin[kGroupRounds] = {}, nasm[kGroupRounds] = {}, nslot[kGroupRounds] = {};
    uint32_t rounds = 0, threads = 0;
};

struct FactorDev {
    const uint32_t *col_ptr;   // sym_c_ptr [n+1] (GESP column sums)
    const uint32_t *gcols;     // columns, those with > kLongRow entries first [n]
    uint32_t ngl;              // number of those
    // Column tasks, by level (tasks ctask_ptr[l] .. ctask_ptr[l+1]).  Lane
    // `lane` of task t owns one L entry of a pivot column k of the level and
    // up to four consecutive entries of U_k: cln[64 t + lane] = {L(i,k)
    // position, pivot position} ({0, 0} for an unused lane); its e-th update
    // reads U(k,j) at cup[256 t + 64 e + lane] and targets ctgt[same index]
    // (~0u: no update here — an unused slot, or a merge entry does it).
    const uint32_t *ctask_ptr; // [num_lev + 2]
    const uint2 *cln;
    const uint32_t *ctgt;
    const uint32_t *cup;
    const uint32_t *ment;      // merge entries (target CSC positions), by level,
                               // entries with > kLongMerge sources first
    const uint32_t *ment_ptr;  // [num_lev + 2]
    const uint32_t *ment_long; // long merge entries at the head of each level [num_lev + 1]
    const uint32_t *msrc_ptr;  // per merge entry [entries + 1]
    const MergeSrc *msrc;      // sources in increasing column order
    // per merge entry e, its first two sources in one place (every merge
    // entry has at least two): mrec[2e] = {target, L, U, pivot position of
    // source 0}, mrec[2e + 1] = {L, U, pivot position of source 1, source
    // count}; sources from the third on are read from msrc
    const uint4 *mrec;
    // division items {L position, pivot position | kFirstBit}: those of the
    // columns of each step before the batched kernels' last grid step, step
    // by step, then the rest; each step's, and the rest, in position order
    const uint2 *dvd;
    const uint32_t *dvd_ptr;   // [num_lev + 1]: items of the columns of steps < l
    int32_t num_lev;
    uint32_t n, nnz;
    // LDS windows: runs of steps that work on values staged in LDS
    const WinDev *win;         // [nwin], in step order
    int32_t nwin;
    uint32_t win_nslot;        // the largest window's values
};

// One level-scheduled triangular sweep, row-pull form:
//   x[r] = (x[r] - sum_{e in row r} V[vpos(e)] * x[idx[e]]) [/ V[dpos[r]]]
// with row r's entries [beg[r] + begoff, end[r]) taken in ascending order,
// or descending when desc != 0.
struct TriDev {
    const uint32_t *beg;
    const uint32_t *end;
    const uint32_t *idx;
    const uint32_t *vpos;      // nullptr: identity
    const uint32_t *dpos;      // nullptr: unit diagonal
    const uint32_t *rows;      // rows grouped by level, long rows first
    const uint32_t *lvl_ptr;   // [nlev + 1]
    const uint32_t *lvl_long;  // long rows at the head of each level [nlev]
    // Dataflow schedule: tasks in topological order, each a run of <= 64
    // short rows or one long row (start position | kLongTask); task k covers
    // positions [dtask[k] & ~kLongTask, dtask[k + 1] & ~kLongTask).  Tasks
    // never cross a fused-segment boundary; seg_task gives each fused
    // segment's first task.
    const uint32_t *dtask;     // [ntask + 1]
    uint32_t ntask;
    uint32_t begoff;
    int32_t desc;
    int32_t nlev;
    int32_t pad;
};

// A pipelined dataflow sweep over a per-matrix copy of the factor values
// laid out task by task (the batch refinement).  Task k = {base, p0, z, m}:
//  - z = rows (< 2^24), no kLongTask bit: rows one per lane: lane l takes
//    position p0 + l (l < rows), its entry e at slot base + 64 e + l (e < m,
//    m = the task's longest row; shorter rows leave padding slots); a row
//    longer than kDfK is walked kDfK entries at a time;
//  - z = kLongTask | log2(gw) << 24 | rows: rows of one level (so no row of
//    the task depends on another) taken gw = 16, 32 or 64 lanes each: row
//    g at position p0 + g, its entry j at slot base + gw g + j; a 64-lane
//    row (rows = 1) may have more than 64 entries, at base + j.
// Each position's {row, entries} is in rl; entries are stored in the order
// the row consumes them.  div: U sweeps, the pivot of position p is value
// nslots + p.
constexpr uint32_t kDfK = 6;
// Rows of kDfK < len <= kDfLaneMax entries are lane rows (walked kDfK
// entries at a time) in levels that hold at least kDfWideLevel of them.
constexpr uint32_t kDfLaneMax = 64;
constexpr uint32_t kDfWideLevel = 32;

struct DfDev {
    const uint4 *task;         // [ntask]
    const uint2 *rl;           // [n]
    const uint32_t *idx;       // column of each slot [nslots]
    uint32_t ntask, nslots;
    int32_t div;
    uint32_t voff;             // this sweep's first value in the per-matrix copy
};

// A triangular sweep as streams of chunks: the layout of the sweeps whose
// vector is in LDS.  A chunk is a wave's unit: 64 lanes of four entries, rows
// of one level, which run in one step of the sweep.  A row takes 1, 2, 4, 8 or 16 lanes
// (aligned), lane j of the row its entries 4 j .. 4 j + 3 in the order the row
// consumes them, rows of any size side by side;
// a row of more than 64 summed entries takes chunks of its own, lane j of
// such a chunk holding entries j, 64 + j, 128 + j and 192 + j of its 256.
// Only the lanes a chunk uses are stored, a multiple of four (a chain of
// levels of one row each is a chunk a row): F its first lane, u its lanes.
//   meta[F + lane] = {slots of entries 0, 1 (16 bits each), of 2, 3,
//     row slot | log2 lanes << 16 | kSwTree | kSwOn, by lane: the chunk's
//     header; F and u of the wave's chunk two after}; in a chunk of a long row
//     kSwEntry << e (the lane has entry e) and its entries
//   values (L = 4, in div sweeps 5, a lane): value F L + 4 lane + e is entry
//     e's, F L + 4 u + lane the row's pivot (at the lane that stores the row)
//   a row's right-hand side: rhs[rpos[slot]], at its first lane
// Slots number the rows of a part (one workgroup's rows); the two after them
// hold 0 (places without an entry: value 0) and 1 (entries whose column is
// not in the part: their value is the finished product).  kSwTree: the
// refinement sums the row's products by lane and then across its lanes;
// other rows, and every row in the exact solve, are subtracted in order.
constexpr uint32_t kSwTree = 1u << 20, kSwOn = 1u << 21, kSwEntry = 1u << 16;
constexpr uint32_t kSwLong = 1u << 31, kSwFirst = 1u << 30, kSwLast = 1u << 29;   // header bits
constexpr uint32_t kSwHasTree = 1u << 28, kSwHasSeq = 1u << 27;
constexpr uint32_t kSwTrack = 1u << 26;   // the second of the two long rows a wave can have open
// header: the chunk's step (its rows' level among the part's levels: a chunk
// holds rows of one level, whose dependencies ran in earlier steps; a chunk of
// a long row that is not its last: a step by which its entries are set)
constexpr uint32_t kSwStepMask = 0xffffu;
// header, for the exact solve: what a wave can do ahead.  A long row's chunk:
// its first entries set more than kSwLead steps before the chunk's (64 of them
// a step, in the kSwLead steps before); other chunks: the lanes after the
// first that the running values can pass in the step before, by entries set
// two steps or more before the chunk's (pre), and those left for its own (rem).
constexpr uint32_t kSwLead = 4;
constexpr uint32_t kSwEarlyShift = 16, kSwEarlyMask = 0x1ffu;
constexpr uint32_t kSwPreShift = 16, kSwPreMask = 15u, kSwRemShift = 20, kSwRemMask = 15u;
constexpr uint32_t kSwCountShift = 20;   // meta.z of a long row's chunk: its entries

struct SwPart {
    uint32_t wp;               // wave[wp + w]: wave w's chunks
    uint32_t s0, nslot;        // rows row[s0 + slot], right-hand sides rpos[s0 + slot]
    uint32_t steps;
};

// An entry whose column belongs to an earlier launch: value[val] = lu[vpos] * x[col].
struct SwProd {
    uint32_t val, vpos, col;
};

struct SwDev {
    const uint4 *meta;         // [lanes]
    const uint4 *wave;         // {chunks, F of the first, F of the second, their u | u << 8}
    const SwPart *part;
    const uint32_t *row, *rpos;
    const SwProd *prod;
    uint32_t nprod, nwave;     // nwave: streams per part
    uint32_t voff;             // this sweep's first value in the copy
    int32_t div;
};

// The split sweeps of one matrix (a vector beyond LDS): head parts and tail
// of the first and the second sweep, over a value copy of their own.
struct SplitDev {
    SwDev head[2], tail[2];
    const uint32_t *src;       // CSC position of each value of the copy (~0: 0) [nval]
    uint32_t nval;
    uint32_t parts;            // head parts
    uint32_t head_slots;       // rows of the largest
    uint32_t tail_slots;
    const uint32_t *rsrc;      // SolveDev::df_rsrc / df_rscale, or the transposed ones
    const double *rscale;
};

struct SolveDev {
    // the vector in LDS, one part (slot = row): L, U and, for A' x = b, U', L'
    SwDev sw[4];
    TriDev lo, up;             // A x = b:   L then U
    TriDev tup, tlo;           // A' x = b:  U' then L'
    DfDev lo_df, up_df;        // L, U over the per-matrix value copy
    const uint32_t *df_src;    // value copy: CSC position of each slot (~0u: padding, holds 0) [df_nval]
    uint32_t df_nval;          // slots per matrix
    // the same copy staged in LDS, df_cpy_range slots at a time: per range
    // r, entries [df_cpy_ptr[r], df_cpy_ptr[r + 1]) of df_cpy, {CSC
    // position, slot - r df_cpy_range} in increasing position order
    const uint2 *df_cpy;
    const uint32_t *df_cpy_ptr;
    uint32_t df_cpy_range;
    // A' x = b over a second value copy (U' slots, U' pivots, L' slots),
    // the same kind of tables
    DfDev tup_df, tlo_df;
    const uint32_t *tdf_src;
    uint32_t tdf_nval;
    // the first sweep's right-hand side by row r of the factors (A x = b, and
    // A' x = b): float(v[rsrc[r]] * rscale[r]) [n]
    const uint32_t *df_rsrc, *tdf_rsrc;
    const double *df_rscale, *tdf_rscale;
    uint32_t t32_len;          // floats of a matrix's right-hand-side / correction vector scratch
    const uint32_t *row_perm, *row_perm_inv, *col_perm, *col_perm_inv;
    const double *row_scale, *col_scale_perm;
};

// The rows of A (or A') of at most kLongRow entries for products in one
// workgroup: 64 neighbouring rows a chunk, a lane each (neighbours name
// neighbouring columns, so a chunk's gathers share lines: with rows by length
// instead, n=20,000 163 us a product, 117 this way).
struct SpDev {
    const uint2 *chunk;        // [nchunk]: {first entry place, longest row}
    const uint2 *rl;           // [64 nchunk]: {row, entries} ({0, ~0}: none)
    const uint2 *ent;          // place + 64 e + lane: {value index, column} of entry e ({0, 0}: none)
    uint32_t nchunk, pad;
};

struct RefineDev {
    SpDev sp[2];               // A, A'
    const uint32_t *a_rptr;    // CSR of A [n+1]
    const uint32_t *a_cidx;    // [nnz_a]
    const uint32_t *a_src;     // index into the caller's CSC values [nnz_a]
    const uint32_t *a_cptr;    // caller CSC column pointers [n+1]
    const uint32_t *a_ridx;    // caller CSC row indices [nnz_a]
    const uint32_t *lu_src;    // LU position -> caller value index, or ~0u [nnz_lu]
    const uint32_t *row_idx;   // sym_r_idx [nnz_lu]
    const uint32_t *lu_col;    // column of each LU position [nnz_lu]
    const uint32_t *a_rows;    // rows of A, rows with > kLongRow entries first [n]
    const uint32_t *a_cols;    // columns of A, long ones first [n]
    uint32_t a_nlong;          // number of long rows
    uint32_t a_nlong_t;        // number of long columns
    const double *rs_col;      // row_scale[row_perm[c]] per GLU column c [n]
    const double *csp;         // col_scale_perm [n]
    // per caller value k: its LU position and the two scales of its entry
    const uint32_t *a_dst;     // [nnz_a]
    const double *a_rs;        // rs_col of the entry's LU column [nnz_a]
    const double *a_cs;        // csp of the entry's LU row [nnz_a]
    const uint32_t *lu_fill;   // LU positions no caller value lands on (fill-in), ascending [nfill]
    uint32_t nnz_a, nfill;
};

struct MatDesc {
    FactorDev f;
    SolveDev s;
    RefineDev r;
    uint32_t n, nnz;
    uint32_t krylov;   // Arnoldi vectors per refinement cycle (0: plain refinement)
    uint32_t a_kmax;   // most entries in a row or a column of A (rounding bound of the refinement)
};

}  // namespace glu
