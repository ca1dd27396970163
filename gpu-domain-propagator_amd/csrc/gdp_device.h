// gdp_device.h - device-side layout of a propagation problem.
//
// A problem holds one matrix layout and the state of one or more propagation
// units.  A unit is one bound vector being propagated with its own round
// count, change and infeasibility flags.  Two unit modes:
//   blocks    the matrix is a block-diagonal batch of independent instances;
//             unit u owns the rows and columns of instance u, all units share
//             the state arrays (disjoint parts of them)
//   replicas  all units share one matrix; unit u has its own copy of every
//             state array (offset u * per-unit size); a single propagation is
//             the replicas mode with one unit
// Every launch works on a step: unit u runs its round (step - start_u + 1)
// in step `step`.  Units that have converged, crossed or reached their round
// cap skip their work, so units of different ages share a step (continuous
// batching) and finished units cost nothing.
//
// Columns are relabelled internally ("internal ids") and grouped by how their
// bounds are stored:
//   ids [0, n16)      integer columns whose bounds stay integral within
//                     [-32767, 32767]: snapshot record 2 x int16 = 4 bytes
//   ids [n16, n_int)  integer columns whose bounds stay integral within the
//                     int32 range: snapshot record 2 x int32 = 8 bytes
//   ids [n_int, n)    all other columns: snapshot record 2 x double = 16 bytes
// In blocks mode each (class, instance) range is padded to a multiple of 32
// ids, so that every 32-column bitmap word belongs to one unit.  The entry
// order inside every row is unchanged, so the relabelling does not alter any
// arithmetic.
//
// HBM layout (rows grouped by length):
//   row_ptr[m'+1]  int32   start of each of the m' nonempty rows (multiple of
//                          kRowAlign) | padding entries after the row
//   sides[m']      double2 (lhs, rhs) per row
//   col[nnz']      int32   internal column id; bit 31 set for an integer column
//   val[nnz']      double  coefficients
//   items[]        int4    work items of the sweep
//   csc            col_ptr[n+1], col_rows[nnz]: rows of each column (marking)
// per unit:
//   snapshot       S16[n16] uint32, S32[n32] int2, SF[nf] double2: the bounds
//                  every row of a round reads, in one block of 16-byte chunks
//                  (S32 from byte snap_off32, SF from byte snap_offF, both
//                  multiples of 16; blocks of consecutive units snap_stride
//                  bytes apart) so that any record is read with one aligned
//                  16-byte load
//   accumulator    AI[n_int] int2 (integer atomics), AF[nf] double2 (FP64
//                  atomics), AX[n_int] double2 (exact values of integer
//                  candidates beyond the int32 range; they only arise when
//                  bounds cross)
//   bm[nwords]     uint32  columns moved in the current step (scanned by publish)
//   marks[m']      int32   step in which the row must be processed
//   lists          wl[m'], wl_seg[segments], wl_cnt: the marked rows of the
//                          next step, listed by tree width (a row once: the
//                          mark is exchanged and the first marker lists it),
//                          and the segments of split rows to recompute; a step
//                          of marked rows works through them in full passes
//                          whatever items the rows lie in
//   split rows     seg_parts, seg_state, seg_count, seg_marks: a marked split
//                  row recomputes only the segments holding a column that
//                  moved in the previous step; the others keep their stored
//                  partials
#pragma once

#include <hip/hip_runtime.h>

namespace gdp {

constexpr int kIdMask = 0x3fffffff;
constexpr int kIntFlag = static_cast<int>(0x80000000u);
constexpr int kItemGroup = 0;
constexpr int kItemLong = 1;   // one row, one wave, all segments (rows not split)
constexpr int kItemSeg = 2;    // up to kSegsPerItem consecutive segments of a split row
constexpr int kSegsPerItem = 4;
constexpr int kItemUnitShift = 12;  // items[].x >> 12: unit of the item (blocks mode)
// Units of a launch whose work a workgroup lays out in LDS at a time.
constexpr int kWindowUnits = 1024;
// Bytes of the persistent kernel's dynamic LDS in a launch of several units:
// the running sums of the units' work (one more than units) and their
// all-rows bits.
constexpr int kWindowLdsBytes = (kWindowUnits + 64) * 4 + (kWindowUnits / 32) * 4;
// Lists of marked work: class 0 the segments of split rows, 1 the unsplit
// long rows, 2 + q the rows of tree width 2^(8 - q).
constexpr int kClasses = 11;
constexpr int kListStride = 16;       // DevMatrix::list_at entries per unit
constexpr int kCountWords = 8;        // 64-bit counter words per unit and step parity, two classes each
// Binary columns (integer columns whose bound envelope lies in [0, 1]) have
// internal ids [0, n_bin) in replicas mode, and each unit keeps their bounds
// also as 2-bit codes, 16 columns to a 32-bit word: bit 0 = (lb >= 1), bit
// 1 = (ub < 1).  As bounds only tighten during a run, a code's bits are only
// ever set, so the publish of a step ORs new bits in.  A persistent launch of
// one unit copies the codes of the first n_lds binary columns into LDS at
// the start of every step and reads their bounds there instead of gathering
// their records.  At most kMaxLdsBinBytes of LDS per workgroup.
constexpr int kMaxLdsBinBytes = 64 * 1024;

// Rows start at multiples of kRowAlign entries (padding entries hold the
// column id n, whose record at the end of a snapshot block has bounds (0, 0),
// and coefficient 0: they add nothing to an activity and are never
// tightened; four of them follow the last row, for the lanes past a row's
// end); the low bits of row_ptr[r] hold
// the number of padding entries after row r.  Aligned starts let a lane load
// its 4 consecutive entries with one 16-byte column load and two 16-byte
// coefficient loads.
constexpr int kRowAlign = 4;

// Per-step status words, in a ring of kStatusRows rows (row step % kStatusRows).
constexpr int kStatusWords = 8;
constexpr int kStatusRows = 128;
constexpr int kStatusChanged = 0;  // some unit moved a bound in the step
constexpr int kStatusApply = 2;    // split-row segments queued for the apply phase
// Words of the problem-wide status block (separate from the ring).
constexpr int kGlobalError = 0;    // a bounded device wait timed out
constexpr int kGlobalTicket = 1;   // workgroups of unpack_rounds_kernel that are done
constexpr int kGlobalEnvelope = 2; // some loaded vector left the envelope (runs that then return an error)
constexpr int kGlobalWords = 8;

// Words of a run state that outlive its runs: row marks hold the step's stamp
// plus the epoch, which starts beyond every earlier mark with each run, so that
// no run has to clear them; whether an exact integer accumulator (AX) was
// written.
constexpr int kPersistEpoch = 0;
constexpr int kPersistAx = 1;
constexpr int kPersistWords = 2;
constexpr int kPersistAt = 32;    // first of them, from the global words
constexpr int kEpochStamps = 256; // stamps of a run, rounded up
// A step's stamps: of rows marked by the publish before it, and of rows marked
// by the hints of a vector that starts in it.  A server's slot may hold marks of
// its last vector for the very step in which the next one starts (the last one
// moved bounds, and crossed them or reached its cap, in the step before).
__host__ __device__ inline unsigned mark_stamp(int step, bool hint) {
    return 2u * static_cast<unsigned>(step) + (hint ? 1u : 0u);
}
// Loads and unpacks of this many vectors keep a vector to one XCD.
constexpr int kVectorsByXcd = 64;

// State of one unit (int32 words, read as 64-bit pairs).  A step's changes
// go to slot step & 1 of `changed`, and step s asks slot (s - 1) & 1 whether
// the unit moved in its previous round: writers and readers of one step
// never share a slot.
struct UnitState {
    int start;        // step of the unit's round 1; 0: no bound vector loaded
    int infeasible;   // step in which bounds crossed (0: none)
    int markall;      // step in which every row of the unit is processed
    int max_rounds;   // round cap
    int crossed;      // input bounds already crossed
    int envelope;     // input bounds outside the storage-class envelope
    int changed[2];   // last step of each parity in which the unit moved a bound
    int mark_limit;   // accepted candidates of a step from which all rows are processed
    int error;        // a bounded device wait timed out (host copy of the outcome)
    int pad[6];
};

// Accepted candidates counted per unit and step (ring of kMoveSlots steps,
// kMoveLanes counters per slot to spread the atomics); a unit whose count
// reaches its threshold processes all rows next step instead of pushing row
// marks (the count bounds the number of moved columns from above).
constexpr int kMoveSlots = 4;
constexpr int kMoveLanes = 16;
// Each counter on its own 128-byte line (ints between two counters).
constexpr int kMoveStride = 32;
// Index of counter j of unit u's slot `slot`.
__host__ __device__ inline int moved_index(int u, int slot, int j) {
    return ((u * kMoveSlots + slot) * kMoveLanes + j) * kMoveStride;
}

// Progress word of launches that stop themselves: no further step runs.
constexpr int kRoundsOver = 0x40000000;

// Grid barrier words, each counter on its own 128-byte line.
constexpr int kBarrierTop = 0;
constexpr int kBarrierGen = 32;
constexpr int kBarrierGroup = 64;  // + 32 * group, 8 groups
constexpr int kBarrierWords = 64 + 32 * 8;

// wall_clock64 runs at 100 MHz on CDNA; give up a wait after 1 s
constexpr long long kWaitTimeoutTicks = 100000000LL;

// Partial activity of one segment of a split row.
struct SegPart {
    double smin, smax, dmax;
    int infs;    // infinite contributions: min side in the low 16 bits, max side in the high
                 // (at most kSegLen each)
    int stamp;   // step in which the partial was computed (0: not in this run); written
                 // with infs as one 8-byte word
};
static_assert(kSegLen < (1 << 15), "a segment's infinite contributions fit in 16 bits");

// Activity of a split row, written by the last segment wave of a step
// when the row gate passes (read by the apply phase of that step).
struct SegState {
    double minact, maxact;
    int mininf, maxinf;  // written and read as one 8-byte word
};

struct DevMatrix {
    int m;            // nonempty rows
    int n;            // internal column ids (including padding ids)
    int n16, n_int;   // class boundaries of the internal ids
    int nwords;       // bitmap words per unit, n / 32
    int n_items;      // sweep items (of one unit in replicas mode)
    int replicas;     // 1: replicas mode, 0: blocks mode
    int mark_rows;    // 0: every step processes every row of an active unit
    const int *row_ptr;
    const double2 *sides;
    const int *col;
    const double *val;
    const int4 *items;
    const int4 *seg_rows;  // per split row: {row, first partial, segments, unit}
    const int *part_row;   // per segment of a split row: its split-row index
    int n_seg_rows;
    int n_seg_parts;
    const int *col_ptr;    // csc of the internal ids (marking)
    const int *col_rows;
    const int *col_seg;    // per csc entry: its segment of a split row, or -1 - the class of its row
    const int *list_at;    // first place in wl (class 0: in wl_seg) of each class (blocks: of each
                           // unit's classes, kListStride per unit)
    const int *unit_item;  // blocks: first sweep item of each unit, and the end
    unsigned long long class_logg, class_logk;  // lanes per row and entries per lane (log2), 4 bits a class
    const int *perm;       // internal id -> caller's column (-1: padding id)
    const int *word_unit;  // blocks mode: unit of each bitmap word
    int snap_off32;        // byte offset of S32 in a unit's snapshot block (these three: bits of a
                           // 32-bit unsigned number, below 2^31 in the rounds)
    int snap_offB;         // byte offset of SB
    int snap_offF;         // byte offset of SF
    long long snap_stride; // bytes between the snapshot blocks of two units
    int n_bin;             // binary columns: internal ids [0, n_bin) (replicas mode; blocks: 0)
    int sb_words;          // words of a unit's binary codes: ceil(n_bin / 64) * 4
    int n_padded;          // entries of the padded rows (four padding entries follow)
};

struct DevState {
    unsigned *S16;
    int2 *S32;
    double2 *SF;
    int2 *AI;
    double2 *AX;
    double2 *AF;
    unsigned *bm;
    int *marks;
    int *wl;               // marked rows of the next step, by class
    int *wl_seg;           // segments to recompute in the next step
    unsigned long long *wl_cnt;  // [units][2][kCountWords] listed rows per class, by step parity
    SegPart *seg_parts;
    int *seg_marks;        // step in which a split row's segment must be recomputed
    SegState *seg_state;
    unsigned *seg_count;   // segments reduced in the current step (a step of all rows), or still to reduce
    // shared by all units
    UnitState *units;
    int *moved;            // [units][kMoveSlots][kMoveLanes] accepted candidates, kMoveStride ints apart
    int *status;           // kStatusRows * kStatusWords ring
    int *global;           // kGlobalWords
    unsigned *barrier;     // kBarrierWords
    int *persist;          // kPersistWords
    int *apply_tasks;      // unit * n_seg_parts + segment, per step
    const int *active;     // units of the launch (replicas mode)
    int n_active;
    int n_lds;             // binary columns read from LDS (persistent launch of one unit; else 0)
    unsigned *SB;          // 2-bit codes of the binary columns (sb_words per unit)
    int n_codes;           // binary columns read from their codes in SB (kRecords)
    int *host_word;        // pinned: the step that the guarded launches have started, or kRoundsOver
};

// A vector that the units of a launch mostly agree with (the base of a
// server's requests, the majority of three node vectors): the partial
// activities of the split rows' segments are computed for it once, and a unit
// starts with them in place of its own wherever it has the same bounds.
struct ReferenceView {
    const SegPart *parts = nullptr;  // null: no reference
    const double *lbs = nullptr, *ubs = nullptr;  // by internal id
    unsigned *diff = nullptr;        // per listed unit: columns that differ (nwords each)
    int *n_diff = nullptr;           // per listed unit: words of diff that are not zero
    int start = 0;                   // step that the copied partials are stamped with
};

// Columns in which finished vectors differ from others: vector k's indices and
// bounds in region k (of cap) of cols / vl / vu, their number in cnt[k] (zero on
// entry; it may exceed cap).
struct ChangeLists {
    const double *const *lb = nullptr, *const *ub = nullptr;
    int cap = 0;
    int *cnt = nullptr, *cols = nullptr;
    double *vl = nullptr, *vu = nullptr;
};

// Up to three vectors whose bitwise majority is the reference.
struct ReferenceVectors {
    const double *lb[3], *ub[3];
    int n;
};

// ---- double-buffered rounds (one bound vector, or a batch) ----
// Two blocks of bound records take turns: round s reads the bounds S_{s-1}
// from block (s - 1) & 1 and folds its candidates into block s & 1, which
// still holds S_{s-2}; the columns that round s - 1 moved are folded into it
// in the same phase (maximum and minimum commute), so that at the end of the
// round it holds S_s.  A round is then one phase, with one kernel boundary or
// one grid barrier, in place of sweep, apply and publish.  No marks:
// from kMinTestItems items on, every workgroup copies the bitmap of the columns
// that the round before moved to LDS, and a pass looks its columns up there
// before it gathers anything; rows without a moved column would repeat the
// candidates they had.  (On average over the rounds 35 to 55% of the entries lie
// in rows with a moved column.)  Crossed bounds of round s - 1 are found
// while its moved columns are folded in round s, whose own candidates are
// then dropped with their block.
// Records: int32 pairs for the integer columns, then FP64 pairs from byte
// snap_offF (the DevMatrix of these kernels has n16 = 0, snap_off32 = 0).
constexpr int kPlanBins = 9;          // tree widths 2^8 .. 2^0
constexpr int kMaxGatherBlocks = 512; // workgroups of the persistent launch
// Items from which a round looks for unmoved rows: one a wave of the persistent
// launch.  Below, a round is the latency of one pass, which a lookup makes longer
// (77,000 nonzeros: 7.3 us a round without, 7.8 with; 2.2M: 23 without, 18 with).
constexpr int kMinTestItems = 4096;
constexpr int kMaxBitWords = 16 << 10; // LDS copy of the moved columns: 64 KB
constexpr int kMaxRoundUnits = 256;   // instances of a batch whose rounds run so (a multiple of 64)
constexpr int kMaxSlotWords = (kMaxRoundUnits + 30) / 31;
// Where each tree-width bin's rows and items start (building the item list).
struct RoundBins {
    int n_segs;
    int item0[kPlanBins + 1];         // first item of the bin of width 2^(8 - q)
    int row0[kPlanBins + 1];          // first layout row of the bin
    int rows_per_item[kPlanBins];
    int logg[kPlanBins];              // lanes per row (log2)
    int logk[kPlanBins];              // entries per lane (log2)
};
struct RoundPlan {
    int n_items;
    const int4 *items;                // as DevMatrix's: one segment of a split row, or one pass of rows
    char *block[2];
    double2 *AX[2];                   // exact integer values beyond int32, per block
    unsigned *bm[3];                  // columns moved in a round, by round % 3
    int bit_words;                    // words of a workgroup's LDS copy of one (a power of two)
    unsigned long long *slots;        // arrivals of the persistent launch's barrier, two sets
    double *lbs, *ubs;                // the caller's vectors
    int mark_limit, max_rounds;
    UnitState *host_state;            // pinned: the outcome (of every unit)
    // a batch: its instances side by side in the blocks
    int n_units = 1;
    int slot_words = 1;               // words of an arrival: 31 units each
    const int *unit_item = nullptr;   // first item of each unit, and the end
    int *run = nullptr, *upto = nullptr;  // launches: units of the round, running totals of their items
};

// State arrays of unit u (replicas mode); the shared arrays are unchanged.
__device__ __forceinline__ DevState unit_view(const DevMatrix &M, const DevState &D, int u) {
    if (!M.replicas) return D;
    DevState V = D;
    const size_t k = static_cast<size_t>(u);
    const size_t snap = k * static_cast<size_t>(M.snap_stride);
    V.S16 = reinterpret_cast<unsigned *>(reinterpret_cast<char *>(D.S16) + snap);
    V.S32 = reinterpret_cast<int2 *>(reinterpret_cast<char *>(D.S32) + snap);
    V.SF = reinterpret_cast<double2 *>(reinterpret_cast<char *>(D.SF) + snap);
    V.AI += k * M.n_int;
    V.AX += k * M.n_int;
    V.AF += k * (M.n - M.n_int);
    V.bm += k * M.nwords;
    V.marks += k * M.m;
    V.wl += k * M.m;
    V.wl_seg += k * M.n_seg_parts;
    V.seg_parts += k * M.n_seg_parts;
    V.seg_marks += k * M.n_seg_parts;
    V.seg_state += k * M.n_seg_rows;
    V.seg_count += k * M.n_seg_rows;
    V.SB = reinterpret_cast<unsigned *>(reinterpret_cast<char *>(D.SB) + snap);
    return V;
}

}  // namespace gdp
