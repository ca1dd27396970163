// gdp_kernels.hip - CDNA4 (gfx950) kernels of the propagation steps.
//
// A step advances every active unit (bound vector) by one round, in three
// phases:
//   sweep    every marked row of every active unit reads the unit's bound
//            snapshot, computes its activities and the candidate bounds of
//            its columns, and folds accepted candidates into the unit's
//            accumulator with native atomics (int32 max/min for compact
//            integer columns, global_atomic_{max,min}_f64 for the others); the
//            first candidate of a 32-column word queues the word for publish.
//   apply    split rows (longer than kSegLen) whose gate passed apply the
//            candidates of their segments (long rows rarely pass the gate,
//            so this phase is mostly empty).
//   publish  the queued words' moved columns are copied from the accumulator
//            into the snapshot, checked for crossed bounds (lb > ub + eps),
//            and the rows of the moved columns are marked for the next step.
// Rows therefore see exactly the bounds at the end of the unit's previous
// round: the round-synchronous semantics of the oracle.  A row none of whose
// columns moved in the previous round is skipped; it would reproduce
// candidates that were already applied, so skipping it changes no result.
//
// Sweep work is split into 64-lane wave items:
//   group item  rows of tree width w = next_pow2(len) <= kSegLen, processed by
//               groups of g = 2^logg lanes with K = w / g consecutive entries
//               per lane; a row's activity is the pairwise tree over its
//               entries in natural order: K entries in registers, then an
//               xor butterfly over the g lanes.
//   seg item    up to kSegsPerItem kSegLen-entry segments of a longer row;
//               segment sums are added left to right by the wave that
//               completes the row.
//   long item   a row that is not split (a tuning option), reduced segment
//               by segment by one wave.
// The summation order is thus a function of the row length only, whatever
// (g, K) a bin uses, which makes results reproducible bit for bit.
//
// Reference counterpart: GPUAtomicDomainPropagation
// (src/kernels/atomic_kernel.cuh:9-450) and the megakernel
// (src/kernels/atomic_megakernel.cuh:14-490).
#include <hip/hip_runtime.h>

#include "gdp_arith.h"
#include "gdp_device.h"

namespace gdp {

__device__ __forceinline__ double shfl_xor_d(double v, int mask) { return __shfl_xor(v, mask, 64); }

__device__ __forceinline__ void atomic_max_d(double *p, double v) {
    __hip_atomic_fetch_max(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ void atomic_min_d(double *p, double v) {
    __hip_atomic_fetch_min(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ void atomic_max_i(int *p, int v) {
    __hip_atomic_fetch_max(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ void atomic_min_i(int *p, int v) {
    __hip_atomic_fetch_min(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ unsigned atomic_or_u(unsigned *p, unsigned v) {
    return __hip_atomic_fetch_or(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ int atomic_add_i(int *p, int v) {
    return __hip_atomic_fetch_add(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ void atomic_or_i(int *p, int v) {
    __hip_atomic_fetch_or(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// Device-coherent plain accesses.  Relaxed agent-scope atomic loads and
// stores are single memory operations marked device-coherent (no whole-cache
// write-back or invalidate, unlike acquire/release fences at agent scope,
// which on this target maintain the entire L2).  Data exchanged between
// waves of one launch uses these; ordering comes from waiting for the
// wave's outstanding memory operations (mem_wait) before the operation that
// publishes them.
template <typename T>
__device__ __forceinline__ T coherent_load(const T *p) {
    return __hip_atomic_load(const_cast<T *>(p), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
template <typename T>
__device__ __forceinline__ void coherent_store(T *p, T v) {
    __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ double coherent_load_d(const double *p) {
    return __longlong_as_double(coherent_load(reinterpret_cast<const long long *>(p)));
}
__device__ __forceinline__ void coherent_store_d(double *p, double v) {
    coherent_store(reinterpret_cast<long long *>(p), __double_as_longlong(v));
}
// Two adjacent ints (8-byte aligned, first in the low word) in one
// device-coherent access.
__device__ __forceinline__ void coherent_store_2i(int *p, int a, int b) {
    coherent_store(reinterpret_cast<long long *>(p),
                   static_cast<long long>(static_cast<unsigned long long>(static_cast<unsigned>(a)) |
                                          (static_cast<unsigned long long>(static_cast<unsigned>(b)) << 32)));
}
__device__ __forceinline__ void coherent_load_2i(const int *p, int &a, int &b) {
    const unsigned long long w =
        static_cast<unsigned long long>(coherent_load(reinterpret_cast<const long long *>(p)));
    a = static_cast<int>(w & 0xffffffffull);
    b = static_cast<int>(w >> 32);
}
// waits until every memory operation this wave issued has completed
__device__ __forceinline__ void mem_wait() { __builtin_amdgcn_s_waitcnt(0); }

// ---------------------------------------------------------------------------
// bounds snapshot and accumulator
// ---------------------------------------------------------------------------

// How a kernel reads the snapshot.
//   kRecords        int16, int32 and FP64 records (DevMatrix's three classes)
//   kWide           int32 and FP64 records only (the double-buffered rounds)
//   kWideCoherent   the same with device-coherent loads (sc1: past the L1,
//                   coherent across the XCDs' L2s), for a launch in which other
//                   workgroups wrote the records and nothing is invalidated
constexpr int kRecords = 0, kWide = 1, kWideCoherent = 2;

// Byte offset of the record of internal column `id` in the unit's block: the
// record's size and the class's base picked by class, then one shift and add
// (picking among the three finished offsets becomes branches).
// Binary columns id < D.n_codes are read from their 2-bit codes, 16 columns a
// word: 50,000 of them take 12.5 KB where the records take 200, so that a
// compute unit at work on one vector of many finds them in its L1: a sweep is
// bound by its requests to the L2 (116 a ns, half of what 128 channels could
// take at one a clock), one per gathered record.  256 vectors, 200,000 rows:
// 2.09 -> 1.94 ms in the persistent launch; one vector of 1M rows in the loop, whose
// 62 KB of codes fit an L1 by half: 3.02 -> 2.67.
template <int kMode>
__device__ __forceinline__ unsigned record_offset(const DevMatrix &M, const DevState &D, int id) {
    const unsigned uid = static_cast<unsigned>(id);
    const unsigned base32 = static_cast<unsigned>(M.snap_off32) - static_cast<unsigned>(M.n16) * 8u;
    const unsigned baseF = static_cast<unsigned>(M.snap_offF) - static_cast<unsigned>(M.n_int) * 16u;
    unsigned shift = id < M.n_int ? 3u : 4u;
    unsigned base = id < M.n_int ? (kMode == kRecords ? base32 : 0u) : baseF;
    if constexpr (kMode == kRecords) {
        shift = id < M.n16 ? 2u : shift;
        base = id < M.n16 ? 0u : base;
        const unsigned code_word = static_cast<unsigned>(M.snap_offB) + (uid >> 4 << 2);
        return id < D.n_codes ? code_word : (uid << shift) + base;
    }
    return (uid << shift) + base;
}

// Dynamic LDS of the persistent kernel: the sweep's window in a launch
// of several units, else the 2-bit codes of the first D.n_lds binary columns
// (other kernels run with D.n_lds = 0 and never touch it).
extern __shared__ __align__(16) unsigned dyn_lds[];

// The bytes from byte `off` of the unit's snapshot block (a multiple of the
// record's size), the record's own first, zeros from kNoRecord.  One 16-byte
// buffer load whatever the record's class: the address takes no 64-bit
// arithmetic, and the lanes without an entry are cut off by the bounds check
// instead of by masks.  Of blocks with 4-byte records it is the aligned 16 bytes
// that hold the record, picked apart: from the record's own first byte every
// tenth load crossed into a second line, and a sweep is bound by such requests
// (ms a call: 12.4M entries over 2M columns 8.11 -> 7.90 persistent, 8.00 -> 7.79 in
// the loop; 16M with rows of up to 50,000 3.54 -> 3.53 and 3.54 -> 3.45; 1M rows 2.83
// -> 2.84 and 2.86 -> 2.80; 256 node vectors 2.84 -> 2.86).  Where records have 8
// bytes or 16, every sixteenth crosses, and picking gains nothing.
constexpr unsigned kNoRecord = 0xfffffff0u;
template <int kMode>
__device__ __forceinline__ uint4 load_record(const DevMatrix &M, const DevState &D, unsigned off) {
    const auto rsrc = __builtin_amdgcn_make_buffer_rsrc(D.S16, 0, static_cast<int>(M.snap_stride), 0x00020000);
    constexpr int kSc1 = 16;
    const unsigned at = kMode == kRecords ? off & ~15u : off;
    const auto v = __builtin_amdgcn_raw_buffer_load_b128(rsrc, static_cast<int>(at), 0,
                                                         kMode == kWideCoherent ? kSc1 : 0);
    if constexpr (kMode == kRecords) {
        // bits 3 and 2 of the offset as masks: two bit-field extracts, three inserts
        const unsigned upper = static_cast<unsigned>(static_cast<int>(off << 28) >> 31);
        const unsigned odd = static_cast<unsigned>(static_cast<int>(off << 29) >> 31);
        const unsigned x = (v[2] & upper) | (v[0] & ~upper), y = (v[3] & upper) | (v[1] & ~upper);
        return make_uint4((y & odd) | (x & ~odd), y, v[2], v[3]);
    }
    return make_uint4(v[0], v[1], v[2], v[3]);
}

// Bounds of `id` from its record; of a binary column id < D.n_lds from its
// 2-bit code in LDS instead, of one id < D.n_codes from its code in `c`.
template <int kMode>
__device__ __forceinline__ void decode_bounds(const DevMatrix &M, const DevState &D, int id, const uint4 c, double &l,
                                              double &u) {
    int il = static_cast<int>(c.x), iu = static_cast<int>(c.y);
    if constexpr (kMode == kRecords) {
        const bool c16 = id < M.n16;
        il = c16 ? static_cast<short>(c.x & 0xffffu) : il;
        iu = c16 ? static_cast<int>(c.x) >> 16 : iu;
        if (id < D.n_lds || id < D.n_codes) {
            const unsigned code = (id < D.n_lds ? dyn_lds[id >> 4] : c.x) >> ((id & 15) * 2);
            il = static_cast<int>(code & 1u);
            iu = static_cast<int>(((code >> 1) & 1u) ^ 1u);
        }
    }
    const double lf = __hiloint2double(static_cast<int>(c.y), static_cast<int>(c.x));
    const double uf = __hiloint2double(static_cast<int>(c.w), static_cast<int>(c.z));
    const bool whole = id < M.n_int;
    l = whole ? static_cast<double>(il) : lf;
    u = whole ? static_cast<double>(iu) : uf;
}

// Bounds of internal column `id` at the start of the round.
template <int kMode>
__device__ __forceinline__ void load_bounds(const DevMatrix &M, const DevState &D, int id, double &l, double &u) {
    const unsigned off = id < D.n_lds ? kNoRecord : record_offset<kMode>(M, D, id);
    decode_bounds<kMode>(M, D, id, load_record<kMode>(M, D, off), l, u);
}

__device__ __forceinline__ bool fits_int32(double v) { return v >= -2147483647.0 && v <= 2147483647.0; }

// Where accepted candidates go: the unit's accumulator and bitmap.
struct Sink {
    DevState V;
};

// Sentinels of the integer accumulator: a candidate beyond the int32 range
// goes to AX, and AI's side is pushed to its sentinel so that readers know
// to consult AX (AI.x == kAiHigh may also be a genuine bound; reading AX
// then is merely redundant).  Integer candidates are integral, so those
// beyond the range are >= 2^31 or <= -2^31 and the max / min with the
// sentinel is the candidate itself.
constexpr int kAiHigh = 2147483647;
constexpr int kAiLow = -2147483647 - 1;

// Folds an accepted lower / upper candidate into the accumulator and marks
// the column in the unit's bitmap of moved columns.
__device__ __forceinline__ void accumulate(const DevMatrix &M, const Sink &K, int id, int t, double nl, double nu) {
    const DevState &D = K.V;
    if (id < M.n_int) {
        if (t & 1) {
            if (fits_int32(nl)) {
                atomic_max_i(&D.AI[id].x, static_cast<int>(nl));
            } else {
                coherent_store(&D.persist[kPersistAx], 1);
                atomic_max_d(&D.AX[id].x, nl);
                atomic_max_i(&D.AI[id].x, kAiHigh);
            }
        }
        if (t & 2) {
            if (fits_int32(nu)) {
                atomic_min_i(&D.AI[id].y, static_cast<int>(nu));
            } else {
                coherent_store(&D.persist[kPersistAx], 1);
                atomic_min_d(&D.AX[id].y, nu);
                atomic_min_i(&D.AI[id].y, kAiLow);
            }
        }
    } else {
        double2 *a = &D.AF[id - M.n_int];
        if (t & 1) atomic_max_d(&a->x, nl);
        if (t & 2) atomic_min_d(&a->y, nu);
    }
    __hip_atomic_fetch_or(&D.bm[id >> 5], 1u << (id & 31), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// The accumulator words of internal column `id` as read (device-coherent):
// both int32 sides in one access, or the FP64 pair.  acc_resolve() turns
// them into bounds; issuing the reads of several columns first lets their
// latencies overlap.
struct AccRaw {
    long long w;
    double fl, fu;
};
__device__ __forceinline__ AccRaw acc_load(const DevMatrix &M, const DevState &D, int id) {
    AccRaw a{0, 0.0, 0.0};
    if (id < M.n_int) {
        a.w = coherent_load(reinterpret_cast<const long long *>(&D.AI[id]));
    } else {
        const double2 *p = &D.AF[id - M.n_int];
        a.fl = coherent_load_d(&p->x);
        a.fu = coherent_load_d(&p->y);
    }
    return a;
}
__device__ __forceinline__ void acc_resolve(const DevMatrix &M, const DevState &D, int id, const AccRaw &a,
                                            double &l, double &u) {
    if (id < M.n_int) {
        const int lo = static_cast<int>(static_cast<unsigned long long>(a.w) & 0xffffffffull);
        const int hi = static_cast<int>(static_cast<unsigned long long>(a.w) >> 32);
        l = static_cast<double>(lo);
        u = static_cast<double>(hi);
        if (lo == kAiHigh || hi == kAiLow) {  // AX only behind a sentinel
            const double xl = coherent_load_d(&D.AX[id].x);
            const double xu = coherent_load_d(&D.AX[id].y);
            l = xl > l ? xl : l;
            u = xu < u ? xu : u;
        }
    } else {
        l = a.fl;
        u = a.fu;
    }
}

// Current accumulated bounds of internal column `id` (device-coherent).
__device__ __forceinline__ void accumulated(const DevMatrix &M, const DevState &D, int id, double &l, double &u) {
    if (id < M.n_int) {
        // both int32 sides in one device-coherent access; AX only behind a sentinel
        const long long w = coherent_load(reinterpret_cast<const long long *>(&D.AI[id]));
        const int lo = static_cast<int>(static_cast<unsigned long long>(w) & 0xffffffffull);
        const int hi = static_cast<int>(static_cast<unsigned long long>(w) >> 32);
        l = static_cast<double>(lo);
        u = static_cast<double>(hi);
        if (lo == kAiHigh || hi == kAiLow) {
            const double xl = coherent_load_d(&D.AX[id].x);
            const double xu = coherent_load_d(&D.AX[id].y);
            l = xl > l ? xl : l;
            u = xu < u ? xu : u;
        }
    } else {
        const double2 *a = &D.AF[id - M.n_int];
        l = coherent_load_d(&a->x);
        u = coherent_load_d(&a->y);
    }
}

__device__ __forceinline__ short clamp16(double v) {
    return static_cast<short>(v < -32767.0 ? -32767.0 : (v > 32767.0 ? 32767.0 : v));
}

__device__ __forceinline__ unsigned pack16(double l, double u) {
    return static_cast<unsigned short>(clamp16(l)) | (static_cast<unsigned>(static_cast<unsigned short>(clamp16(u))) << 16);
}

// Writes bounds into the snapshot record of `id` (device-coherent).  Values
// out of a record's range only occur once bounds have crossed, after which
// the run stops and the snapshot is not read again.
__device__ __forceinline__ void store_snapshot(const DevMatrix &M, const DevState &D, int id, double l, double u) {
    if (id < M.n16) {
        coherent_store(&D.S16[id], pack16(l, u));
    } else if (id < M.n_int) {
        // both sides in one device-coherent 8-byte store (x in the low word)
        const int lo = fits_int32(l) ? static_cast<int>(l) : -2147483647;
        const int hi = fits_int32(u) ? static_cast<int>(u) : 2147483647;
        const unsigned long long w = static_cast<unsigned long long>(static_cast<unsigned>(lo)) |
                                     (static_cast<unsigned long long>(static_cast<unsigned>(hi)) << 32);
        coherent_store(reinterpret_cast<long long *>(&D.S32[id - M.n16]), static_cast<long long>(w));
    } else {
        double2 *s = &D.SF[id - M.n_int];
        coherent_store_d(&s->x, l);
        coherent_store_d(&s->y, u);
    }
}

// ---------------------------------------------------------------------------
// row gate
// ---------------------------------------------------------------------------

// Row gate with the sequential propagator's epsilon-maximum of |a|(u-l).
// That maximum depends on the order of the entries (a later term replaces
// the running value only when larger by more than the tolerance) but always
// lies in [lo, M] with M the exact maximum (computed in parallel, order-free)
// and lo = M minus a little more than the tolerance.  row_gate is monotone in
// its last argument, so when row_gate(lo) == row_gate(M) the answer is known;
// otherwise (entries within 2*eps of the decision threshold) the
// order-dependent maximum is computed exactly by a sequential scan.
struct GateBounds {
    bool hi, lo;
    __device__ __forceinline__ bool decided() const { return hi == lo; }
};

__device__ __forceinline__ GateBounds gate_bounds(double minact, double maxact, int mininf, int maxinf, double lhs,
                                                  double rhs, double dmax) {
    GateBounds g;
    g.hi = row_gate(minact, maxact, mininf, maxinf, lhs, rhs, dmax);
    double lo_d = dmax;
    if (isfinite(dmax)) lo_d = dmax - 4e-9 - fabs(dmax) * 0x1p-48;
    g.lo = row_gate(minact, maxact, mininf, maxinf, lhs, rhs, lo_d);
    return g;
}

// Sequential epsilon-maximum of a whole row read from memory, in CSR order
// (rows that are not split, whose entries are not held in registers).
__device__ __forceinline__ double seq_eps_max(const DevMatrix &M, const DevState &D, int start, int len) {
    double run = 0.0;
    for (int e = 0; e < len; e++) {
        double l, u;
        load_bounds<kRecords>(M, D, M.col[start + e] & kIdMask, l, u);
        run = eps_max_step(run, fabs(M.val[start + e]) * (u - l));
    }
    return run;
}

__device__ __forceinline__ bool decide_gate(const DevMatrix &M, const DevState &D, int start, int len,
                                            double minact, double maxact, int mininf, int maxinf, double lhs,
                                            double rhs, double dmax) {
    const GateBounds g = gate_bounds(minact, maxact, mininf, maxinf, lhs, rhs, dmax);
    if (g.decided()) return g.hi;
    const double m = seq_eps_max(M, D, start, len);
    return row_gate(minact, maxact, mininf, maxinf, lhs, rhs, m);
}

// Applies the candidates of one entry; returns true when a bound moved.
__device__ __forceinline__ bool apply_entry(const DevMatrix &M, const Sink &K, int jp, double a, double l, double u,
                                            double lhs, double rhs, double minact, double maxact, int mininf,
                                            int maxinf) {
    const bool is_cont = jp >= 0;  // bit 31 set marks an integer column
    double nl = l, nu = u;
    const int t = tighten_variable(a, lhs, rhs, minact, maxact, mininf, maxinf, is_cont, l, u, nl, nu);
    if (t == 0) return false;
    accumulate(M, K, jp & kIdMask, t, nl, nu);
    return true;
}

// ---------------------------------------------------------------------------
// lane entries
// ---------------------------------------------------------------------------

// First entry and length of row r (starts are multiples of kRowAlign; the
// low bits of row_ptr[r] count the padding entries after the row).
__device__ __forceinline__ void row_extent(const DevMatrix &M, int r, int &start, int &len) {
    const int a = M.row_ptr[r], b = M.row_ptr[r + 1];
    start = a & ~(kRowAlign - 1);
    len = (b & ~(kRowAlign - 1)) - start - (a & (kRowAlign - 1));
}

// The lane's number, opaque to the optimizer: what is derived from it is
// computed where it is used instead of being kept in registers across the
// loops around (the sweep's registers decide its waves per SIMD).
__device__ __forceinline__ int lane_here() {
    int lane = threadIdx.x & 63;
    asm volatile("" : "+v"(lane));
    return lane;
}

// The values of a lane and of its partner in step h = 2^k of a butterfly whose
// earlier steps ran (lanes of a group of h hold the same value): lane i ^ h,
// or, where that is cheaper, another lane of the same partner group.  In
// registers: DPP within 16 lanes, the row swaps of this target beyond.
template <int h>
__device__ __forceinline__ void partner(int v, int &a, int &b) {
    if constexpr (h <= 8) {
        constexpr int kCtrl = h == 1 ? 0xB1 : (h == 2 ? 0x4E : (h == 4 ? 0x141 : 0x140));
        a = v;
        b = __builtin_amdgcn_update_dpp(v, v, kCtrl, 0xf, 0xf, false);
    } else if constexpr (h == 16) {
        const auto r = __builtin_amdgcn_permlane16_swap(static_cast<unsigned>(v), static_cast<unsigned>(v), false, false);
        a = static_cast<int>(r[0]);
        b = static_cast<int>(r[1]);
    } else {
        const auto r = __builtin_amdgcn_permlane32_swap(static_cast<unsigned>(v), static_cast<unsigned>(v), false, false);
        a = static_cast<int>(r[0]);
        b = static_cast<int>(r[1]);
    }
}
template <int h>
__device__ __forceinline__ void partner_d(double v, double &a, double &b) {
    int al, ah, bl, bh;
    partner<h>(__double2loint(v), al, bl);
    partner<h>(__double2hiint(v), ah, bh);
    a = __hiloint2double(ah, al);
    b = __hiloint2double(bh, bl);
}
template <int h>
__device__ __forceinline__ double step_add(double v) {
    double a, b;
    partner_d<h>(v, a, b);
    return a + b;
}
template <int h>
__device__ __forceinline__ double step_max(double v) {
    double a, b;
    partner_d<h>(v, a, b);
    return fmax(a, b);
}
template <int h>
__device__ __forceinline__ int step_add(int v) {
    int a, b;
    partner<h>(v, a, b);
    return a + b;
}

// The columns that the previous round moved, a bit each, in LDS: bit id of
// word (id / 32) & mask (larger problems share words, which lets rows through
// that have no moved column).  words null: every row counts as moved.
struct MovedBits {
    const unsigned *words;
    unsigned mask;
};

// K consecutive entries of one lane: loads, contributions, pairwise tree of
// the K contributions in natural order, and the cross-lane reduction.
// A sweep is bound by its instructions as much as by its gathers (200,000
// rows, 2.2M nonzeros, nothing moving: 500 vector instructions per pass, 45%
// of the 19 us), so the entries past the row's end are ordinary entries of a
// zero column with a zero coefficient, infinite contributions are looked at
// only where a lane of the wave has one, and their two counts share a word
// (at most kSegLen each).
template <int K, int kMode>
struct LaneEntries {
    int jp[K];
    double a[K], l[K], u[K];
    double tmin, tmax, dmax;
    int infs;     // infinite contributions: minimum side in the low 16 bits, maximum side in the high
    bool some;    // some lane of the wave has one

    __device__ __forceinline__ int min_inf() const { return infs & 0xffff; }
    __device__ __forceinline__ int max_inf() const { return infs >> 16; }

    __device__ __forceinline__ void load(const DevMatrix &M, const DevState &D, int base, int first, int len) {
        const int e = place(M, base, first, len);
        columns(M, e);
        coefficients(M, e);
        bounds(M, D);
    }
    // Where the lane's K entries lie (base + first is a multiple of K and the
    // row is padded to a multiple of kRowAlign, a multiple of K): for a lane
    // past the end, the padding entries behind the last row.
    static __device__ __forceinline__ int place(const DevMatrix &M, int base, int first, int len) {
        return first < len ? base + first : M.n_padded;
    }
    __device__ __forceinline__ void columns(const DevMatrix &M, int e) {
        const int *cp = M.col + static_cast<size_t>(e);
        if constexpr (K == 4) {
            const int4 c = *reinterpret_cast<const int4 *>(cp);
            jp[0] = c.x; jp[1] = c.y; jp[2] = c.z; jp[3] = c.w;
        } else if constexpr (K == 2) {
            const int2 c = *reinterpret_cast<const int2 *>(cp);
            jp[0] = c.x; jp[1] = c.y;
        } else {
            jp[0] = *cp;
        }
    }
    // Whether a bound of one of the lane's columns moved.
    __device__ __forceinline__ bool moved(const MovedBits &B) const {
        unsigned any = 0u;
#pragma unroll
        for (int k = 0; k < K; k++) {
            const unsigned id = static_cast<unsigned>(jp[k] & kIdMask);
            any |= B.words[(id >> 5) & B.mask] >> (id & 31);
        }
        return any & 1u;
    }
    __device__ __forceinline__ void coefficients(const DevMatrix &M, int e) {
        const double *vp = M.val + static_cast<size_t>(e);
        if constexpr (K == 4) {
            const double2 v0 = *reinterpret_cast<const double2 *>(vp);
            const double2 v1 = *reinterpret_cast<const double2 *>(vp + 2);
            a[0] = v0.x; a[1] = v0.y; a[2] = v1.x; a[3] = v1.y;
        } else if constexpr (K == 2) {
            const double2 v0 = *reinterpret_cast<const double2 *>(vp);
            a[0] = v0.x; a[1] = v0.y;
        } else {
            a[0] = *vp;
        }
    }
    // The bounds, and the lane's contributions.
    __device__ __forceinline__ void bounds(const DevMatrix &M, const DevState &D) {
        // every gather first, then the decoding and the contributions; binary
        // columns held in LDS are read there instead
        uint4 rec[K];
#pragma unroll
        for (int k = 0; k < K; k++) {
            const int id = jp[k] & kIdMask;
            rec[k] = load_record<kMode>(M, D, id < D.n_lds ? kNoRecord : record_offset<kMode>(M, D, id));
        }
        dmax = 0.0;
        bool any = false;
#pragma unroll
        for (int k = 0; k < K; k++) {
            decode_bounds<kMode>(M, D, jp[k] & kIdMask, rec[k], l[k], u[k]);
            dmax = fmax(dmax, fabs(a[k]) * (u[k] - l[k]));
            any |= is_neg_inf(l[k]) | is_pos_inf(u[k]);
        }
        infs = 0;
        some = __any(any);
        double smin[K], smax[K];
        if (some) {
#pragma unroll
            for (int k = 0; k < K; k++) {
                const bool lo = is_neg_inf(l[k]), up = is_pos_inf(u[k]);
                const bool pos = a[k] > kEps;
                const bool mi = pos ? lo : up, xi = pos ? up : lo;
                smin[k] = mi ? 0.0 : a[k] * (a[k] > 0.0 ? l[k] : u[k]);
                smax[k] = xi ? 0.0 : a[k] * (a[k] > 0.0 ? u[k] : l[k]);
                infs += (mi ? 1 : 0) + (xi ? 0x10000 : 0);
            }
        } else {
#pragma unroll
            for (int k = 0; k < K; k++) {
                smin[k] = a[k] * (a[k] > 0.0 ? l[k] : u[k]);
                smax[k] = a[k] * (a[k] > 0.0 ? u[k] : l[k]);
            }
        }
#pragma unroll
        for (int w = 1; w < K; w <<= 1) {
#pragma unroll
            for (int k = 0; k < K; k += 2 * w) {
                smin[k] = smin[k] + smin[k + w];
                smax[k] = smax[k] + smax[k + w];
            }
        }
        tmin = smin[0];
        tmax = smax[0];
    }

    // One step of the butterfly; kMax: the largest width too.
    template <int h, bool kMax>
    __device__ __forceinline__ void step() {
        tmin = step_add<h>(tmin);
        tmax = step_add<h>(tmax);
        if (some) infs = step_add<h>(infs);
        if constexpr (kMax) dmax = step_max<h>(dmax);
    }
    // xor butterfly over groups of g lanes (natural pairwise order)
    template <bool kMax>
    __device__ __forceinline__ void reduce(int g) {
        if (g > 1) step<1, kMax>();
        if (g > 2) step<2, kMax>();
        if (g > 4) step<4, kMax>();
        if (g > 8) step<8, kMax>();
        if (g > 16) step<16, kMax>();
        if (g > 32) step<32, kMax>();
    }

    // Sequential epsilon-maximum over the entries of each group of g lanes in
    // natural order (lane by lane, K entries each), starting from `run`;
    // all lanes of a group return the same value.  Entries past the end of
    // the row hold zeros, which never replace the running value.
    __device__ __forceinline__ double eps_scan(int g, double run) const {
        const int gbase = lane_here() & ~(g - 1);
        for (int j = 0; j < g; j++) {
#pragma unroll
            for (int k = 0; k < K; k++) run = eps_max_step(run, __shfl(fabs(a[k]) * (u[k] - l[k]), gbase + j, 64));
        }
        return run;
    }

    // number of accepted candidates
    __device__ __forceinline__ int apply(const DevMatrix &M, const Sink &S, int first, int len, double lhs,
                                         double rhs, double minact, double maxact, int ni, int xi) {
        int moved = 0;
#pragma unroll
        for (int k = 0; k < K; k++)
        {
            if (first + k < len) moved += apply_entry(M, S, jp[k], a[k], l[k], u[k], lhs, rhs, minact, maxact, ni, xi);
            __builtin_amdgcn_sched_barrier(0);
        }
        return moved;
    }
};

// ---------------------------------------------------------------------------
// units and steps
// ---------------------------------------------------------------------------

// Value known to be the same on every lane of the wave (kept in a scalar
// register).
__device__ __forceinline__ int uniform(int v) { return __builtin_amdgcn_readfirstlane(v); }

__device__ __forceinline__ int *status_row(const DevState &D, int step) {
    return D.status + kStatusWords * (step % kStatusRows);
}

// Whether unit u works in `step`, and whether it processes every row.
struct UnitStep {
    bool active;
    bool all_rows;
    int start;  // step of the unit's round 1
};

// The rule for a unit working in `step`, from its state words: loaded, not
// stopped by its load, under its round cap, and in its first round or moved a
// bound in the previous step without becoming infeasible.
__device__ __forceinline__ bool unit_works(int step, int start, int infeasible, int max_rounds, int crossed,
                                           int envelope, int prev_changed) {
    return start > 0 && step >= start && !crossed && !envelope && step - start < max_rounds &&
           (step == start || (prev_changed == step - 1 && infeasible == 0));
}

// unit_step for a different unit on every lane.
__device__ __forceinline__ UnitStep unit_step_lane(const DevMatrix &M, const DevState &D, int u, int step) {
    const long long *p = reinterpret_cast<const long long *>(&D.units[u]);
    const long long w0 = coherent_load(p), w1 = coherent_load(p + 1), w2 = coherent_load(p + 2),
                    w3 = coherent_load(p + 3);
    const int start = static_cast<int>(w0), infeasible = static_cast<int>(w0 >> 32);
    const int markall = static_cast<int>(w1), max_rounds = static_cast<int>(w1 >> 32);
    const int crossed = static_cast<int>(w2), envelope = static_cast<int>(w2 >> 32);
    const int prev_changed = static_cast<int>((step - 1) & 1 ? (w3 >> 32) : w3);
    UnitStep r;
    r.active = unit_works(step, start, infeasible, max_rounds, crossed, envelope, prev_changed);
    r.all_rows = !M.mark_rows || markall == step;
    r.start = start;
    return r;
}

// The same unit on every lane of the wave (result in scalar registers).
__device__ __forceinline__ UnitStep unit_step(const DevMatrix &M, const DevState &D, int u, int step) {
    const UnitStep l = unit_step_lane(M, D, uniform(u), step);
    UnitStep r;
    r.active = uniform(l.active ? 1 : 0) != 0;
    r.all_rows = uniform(l.all_rows ? 1 : 0) != 0;
    r.start = uniform(l.start);
    return r;
}

// Counts the wave's accepted candidates (`moved` per lane) of unit u in
// `step` in one of the unit's kMoveLanes counters of the step (one
// non-returning atomic per wave).  Whether the unit moved at all is recorded
// by the publish phase, from its bitmap, so that nothing writes the unit's
// state words while the items of a step read them.
__device__ __forceinline__ void note_change(const DevState &D, int u, int step, int moved) {
    if (!__any(moved != 0)) return;
#pragma unroll
    for (int h = 1; h < 64; h <<= 1) moved += __shfl_xor(moved, h, 64);
    if ((threadIdx.x & 63) == 0) {
        const int lane_slot = (blockIdx.x * (blockDim.x >> 6) + (threadIdx.x >> 6)) % kMoveLanes;
        atomic_add_i(&D.moved[moved_index(u, step % kMoveSlots, lane_slot)], moved);
    }
}

__device__ __forceinline__ Sink make_sink(const DevState &V) {
    Sink k;
    k.V = V;
    return k;
}

// ---------------------------------------------------------------------------
// sweep items
// ---------------------------------------------------------------------------

// Rows [first, first + nrows) of one tree-width bin, or the nrows rows listed
// at list[first ..]: groups of 2^logg lanes, K consecutive entries per lane.
// With kTest, rows none of whose columns moved are left out: their lanes take
// the padding entries.
template <int K, int kMode, bool kTest = false>
__device__ __forceinline__ int group_item(const DevMatrix &M, const Sink &S, int first, int nrows, int logg,
                                          const int *list, const MovedBits &B = MovedBits{nullptr, 0u}) {
    const DevState &V = S.V;
    const int lane = lane_here();
    const int g = 1 << logg;
    const int gl = lane & (g - 1);
    const int per_pass = 64 >> logg;
    const unsigned long long gmask = (g == 64 ? ~0ull : (1ull << g) - 1ull) << (lane & ~(g - 1) & 63);
    const int end = first + nrows;
    int moved = 0;
    for (int base = first; base < end; base += per_pass) {
        int r = base + (lane >> logg);
        const bool take = r < end;
        if (list != nullptr && take) r = coherent_load(&list[r]);
        int start = 0, len = 0;
        double lhs = 0.0, rhs = 0.0;
        if (take) {
            row_extent(M, r, start, len);
            const double2 sd = M.sides[r];
            lhs = sd.x;
            rhs = sd.y;
        }
        LaneEntries<K, kMode> E;
        int e = E.place(M, start, gl * K, len);
        E.columns(M, e);
        if constexpr (kTest) {
            if (B.words != nullptr) {
                const unsigned long long rows = __ballot(E.moved(B));
                if (rows == 0ull) continue;
                if ((rows & gmask) == 0ull) {
                    len = 0;
                    e = M.n_padded;
#pragma unroll
                    for (int k = 0; k < K; k++) E.jp[k] = M.n;
                }
            }
        }
        E.coefficients(M, e);
        E.bounds(M, V);
        E.template reduce<false>(g);
        const double minact = 0.0 + E.tmin;
        const double maxact = 0.0 + E.tmax;
        const int ni = E.min_inf(), xi = E.max_inf();
        // The gate is monotone in the largest width, so a row passes it when
        // one of its lanes does with its own largest: one ballot in place of
        // a maximum over the lanes.
        const GateBounds gb = gate_bounds(minact, maxact, ni, xi, lhs, rhs, E.dmax);
        const unsigned long long hi = __ballot(gb.hi && len > 0);
        if (hi == 0ull) continue;
        const unsigned long long lo = __ballot(gb.lo && len > 0);
        bool gate = (hi & gmask) != 0ull;
        const bool undecided = gate && (lo & gmask) == 0ull;
        if (__any(undecided)) {
            const double dm = E.eps_scan(g, 0.0);
            if (undecided) gate = row_gate(minact, maxact, ni, xi, lhs, rhs, dm);
        }
        if (gate) moved += E.apply(M, S, gl * K, len, lhs, rhs, minact, maxact, ni, xi);
    }
    return moved;
}

// One row that is not split: one wave, segment by segment, then a second
// pass for the candidates.
__device__ __forceinline__ int long_item(const DevMatrix &M, const Sink &S, int r) {
    constexpr int K = kSegLen / 64;
    const DevState &V = S.V;
    const int lane = lane_here();
    int start, len;
    row_extent(M, r, start, len);
    const double2 sd = M.sides[r];
    double acc_min = 0.0, acc_max = 0.0, dmax = 0.0;
    int mininf = 0, maxinf = 0;
    for (int s0 = 0; s0 < len; s0 += kSegLen) {
        LaneEntries<K, kRecords> E;
        E.load(M, V, start + s0, lane * K, len - s0);
        E.template reduce<true>(64);
        acc_min = acc_min + E.tmin;
        acc_max = acc_max + E.tmax;
        mininf += E.min_inf();
        maxinf += E.max_inf();
        dmax = fmax(dmax, E.dmax);
    }
    int moved = 0;
    if (decide_gate(M, V, start, len, acc_min, acc_max, mininf, maxinf, sd.x, sd.y, dmax)) {
        for (int e = lane; e < len; e += 64) {
            const int jp = M.col[start + e];
            double l, u;
            load_bounds<kRecords>(M, V, jp & kIdMask, l, u);
            moved += apply_entry(M, S, jp, M.val[start + e], l, u, sd.x, sd.y, acc_min, acc_max, mininf, maxinf);
        }
    }
    return moved;
}

// Sequential epsilon-maximum of a split row, computed by its last segment
// wave.  A segment whose exact maximum Ms satisfies !(Ms - run > eps) cannot
// replace the running value (floating-point subtraction is monotone), so it
// is skipped; the others are scanned entry by entry in order.
template <int kMode>
__device__ __forceinline__ double split_eps_scan(const DevMatrix &M, const DevState &V, const int4 info, int start, int len) {
    constexpr int K = kSegLen / 64;
    const int lane = lane_here();
    double run = 0.0;
    for (int b = 0; b < info.z; b += 64) {
        const int q = b + lane;
        const double ms = q < info.z ? coherent_load_d(&V.seg_parts[info.y + q].dmax) : 0.0;
        const int cnt = min(64, info.z - b);
        for (int t = 0; t < cnt; t++) {
            const double mt = __shfl(ms, t, 64);
            if (!eps_gt(mt, run)) continue;
            const int s0 = (b + t) * kSegLen;
            LaneEntries<K, kMode> E;
            E.load(M, V, start + s0, lane * K, len - s0);
            run = E.eps_scan(64, run);
        }
    }
    return run;
}

// Stores the activity partial of segment `part` and the step that computed
// it (lane 0 of the wave).
template <int kMode>
__device__ __forceinline__ void store_part(const DevState &V, int part, const LaneEntries<kSegLen / 64, kMode> &E,
                                           int step) {
    SegPart *p = &V.seg_parts[part];
    coherent_store_d(&p->smin, E.tmin);
    coherent_store_d(&p->smax, E.tmax);
    coherent_store_d(&p->dmax, E.dmax);
    coherent_store_2i(&p->infs, E.infs, step);
}

// Reduces segment s of the split row (rows from `start`, `len` entries) whose
// partials begin at part0 and stores the partial.
template <int kMode>
__device__ __forceinline__ void segment_partial(const DevMatrix &M, const DevState &V, int part0, int s, int start,
                                                int len, int step) {
    constexpr int K = kSegLen / 64;
    const int lane = lane_here();
    const int s0 = s * kSegLen;
    LaneEntries<K, kMode> E;
    E.load(M, V, start + s0, lane * K, len - s0);
    E.template reduce<true>(64);
    if (lane == 0) store_part(V, part0 + s, E, step);
}

// Segments [s, s + cnt) of split row lr (cnt <= kSegsPerItem; cnt < 0: the
// one listed segment s of a step of marked rows) for unit u.  The wave
// reduces each kSegLen-entry segment like a kSegLen-wide group row, stores
// the partials and counts them in (a listed segment: off the segments that
// the row has listed); nobody waits.  The wave that completes the row's count
// adds the partials in segment order and decides the row gate; when it
// passes, the row's activity is stored and its segments are queued for the
// apply phase that follows the sweep.
template <int kMode, bool kTest = false>
__device__ __forceinline__ void seg_item(const DevMatrix &M, const DevState &D, const DevState &V, int u, int lr, int s,
                                         int cnt, int *st, int step, const MovedBits &B = MovedBits{nullptr, 0u}) {
    const int lane = lane_here();
    const int4 info = M.seg_rows[lr];
    const int r = info.x;
    int start, len;
    row_extent(M, r, start, len);
    const bool listed = cnt < 0;
    const int end = s + (listed ? 1 : cnt);
    unsigned add = static_cast<unsigned>(listed ? -1 : cnt);
    if constexpr (kTest) {
        // a segment without moved columns keeps its partial of the round
        // before; the upper half of the row's count holds the others
        constexpr int K = kSegLen / 64;
        const bool countable = info.z < 0x8000;
        for (int q = s; q < end; q++) {
            if (B.words != nullptr && countable) {
                LaneEntries<K, kMode> E;
                E.columns(M, E.place(M, start + q * kSegLen, lane * K, len - q * kSegLen));
                if (!__any(E.moved(B))) continue;
            }
            if (countable) add += 0x10000u;
            segment_partial<kMode>(M, V, info.y, q, start, len, step);
        }
    } else {
        for (int q = s; q < end; q++) segment_partial<kMode>(M, V, info.y, q, start, len, step);
    }
    unsigned old = 0;
    if (lane == 0) {
        mem_wait();
        old = __hip_atomic_fetch_add(&V.seg_count[lr], add, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
    old = __shfl(old, 0, 64);
    if constexpr (kTest) {
        const unsigned now = old + add;
        const bool countable = info.z < 0x8000;
        if ((countable ? now & 0xffffu : now) != static_cast<unsigned>(info.z)) return;
        if (countable && now >> 16 == 0u) {  // nothing of the row moved
            if (lane == 0) coherent_store(&V.seg_count[lr], 0u);
            return;
        }
    } else {
        if (listed ? old != 1u : old + cnt != static_cast<unsigned>(info.z)) return;
    }

    // the row is complete: the lanes load 64 partials at a time
    // (independent loads), which are then added in segment order
    double am = 0.0, ax = 0.0, dm = 0.0;
    int ni = 0, xi = 0;
    for (int b = 0; b < info.z; b += 64) {
        const int q = b + lane;
        double pmin = 0.0, pmax = 0.0;
        if (q < info.z) {
            const SegPart *pq = &V.seg_parts[info.y + q];
            pmin = coherent_load_d(&pq->smin);
            pmax = coherent_load_d(&pq->smax);
            dm = fmax(dm, coherent_load_d(&pq->dmax));
            int infs, stamp;
            coherent_load_2i(&pq->infs, infs, stamp);
            (void)stamp;
            ni += infs & 0xffff;
            xi += infs >> 16;
        }
        const int n_here = min(64, info.z - b);
        for (int t = 0; t < n_here; t++) {
            am = am + __shfl(pmin, t, 64);
            ax = ax + __shfl(pmax, t, 64);
        }
    }
#pragma unroll
    for (int h = 1; h < 64; h <<= 1) {
        ni += __shfl_xor(ni, h, 64);
        xi += __shfl_xor(xi, h, 64);
        dm = fmax(dm, shfl_xor_d(dm, h));
    }
    const double2 sd = M.sides[r];
    const GateBounds gb = gate_bounds(am, ax, ni, xi, sd.x, sd.y, dm);
    bool gate = gb.hi;
    if (!gb.decided()) gate = row_gate(am, ax, ni, xi, sd.x, sd.y, split_eps_scan<kMode>(M, V, info, start, len));
    int pos = 0;
    if (lane == 0) {
        coherent_store(&V.seg_count[lr], 0u);
        if (gate) {
            SegState *stp = &V.seg_state[lr];
            coherent_store_d(&stp->minact, am);
            coherent_store_d(&stp->maxact, ax);
            coherent_store_2i(&stp->mininf, ni, xi);
            pos = atomic_add_i(&st[kStatusApply], info.z);
        }
    }
    if (!gate) return;
    pos = __shfl(pos, 0, 64);
    const int base = u * M.n_seg_parts + info.y;
    for (int q = lane; q < info.z; q += 64) coherent_store(&D.apply_tasks[pos + q], base + q);
}

// Lanes per row and entries per lane (log2) of a class of rows.
__device__ __forceinline__ int class_logg(const DevMatrix &M, int c) {
    return static_cast<int>(M.class_logg >> (4 * c)) & 15;
}
__device__ __forceinline__ int class_logk(const DevMatrix &M, int c) {
    return static_cast<int>(M.class_logk >> (4 * c)) & 15;
}

// The counters of unit u's lists for `step`, and the first place of class c's.
__device__ __forceinline__ unsigned long long *list_counts(const DevState &D, int u, int step) {
    return D.wl_cnt + (static_cast<size_t>(u) * 2 + (step & 1)) * kCountWords;
}
__device__ __forceinline__ int list_start(const DevMatrix &M, int u, int c) {
    return M.list_at[(M.replicas ? 0 : u * kListStride) + c];
}

// Listed rows (class 0: segments) of unit u in `step`, lane c holding class
// c's; the passes they take (segments and unsplit rows one each).
__device__ __forceinline__ int listed_rows(const DevState &D, int u, int step) {
    const int lane = lane_here();
    if (lane >= kClasses) return 0;
    const unsigned long long w = coherent_load(&list_counts(D, u, step)[lane >> 1]);
    return static_cast<int>(lane & 1 ? w >> 32 : w & 0xffffffffull);
}
__device__ __forceinline__ int class_passes(const DevMatrix &M, int c, int rows) {
    if (c < 2) return rows;
    const int log_rows = 6 - class_logg(M, c);
    return (rows + (1 << log_rows) - 1) >> log_rows;
}
// Passes of unit u's lists in `step`, by one lane.
__device__ __forceinline__ int list_passes(const DevMatrix &M, const DevState &D, int u, int step) {
    const unsigned long long *w = list_counts(D, u, step);
    unsigned long long v[(kClasses + 1) / 2];
#pragma unroll
    for (int q = 0; q < (kClasses + 1) / 2; q++) v[q] = coherent_load(&w[q]);
    int n = 0;
#pragma unroll
    for (int c = 0; c < kClasses; c++)
        n += class_passes(M, c, static_cast<int>(c & 1 ? v[c >> 1] >> 32 : v[c >> 1] & 0xffffffffull));
    return n;
}

// Sweep items of unit u (a step of all rows).
__device__ __forceinline__ int unit_items(const DevMatrix &M, int u) {
    return M.replicas ? M.n_items : M.unit_item[u + 1] - M.unit_item[u];
}

// Piece `q` of the work of unit u in `step`: its q-th sweep item when every
// row is processed, else the q-th pass of its lists (segments first, then
// wide to narrow).  With 2^log_parts parts to an item, part `part` of it.
// Records the unit's accepted candidates.
__device__ __forceinline__ void sweep_piece(const DevMatrix &M, const DevState &D, int u, int q, bool all_rows,
                                            int part, int log_parts, int step, int *st) {
    u = uniform(u);
    q = uniform(q);
    const DevState V = unit_view(M, D, u);
    const Sink S = make_sink(V);
    const int *list = nullptr;
    int kind = kItemGroup, first = 0, n = 0, cnt = 0, logg = 0, logk = 0;
    if (all_rows) {
        const int4 d = M.items[(M.replicas ? 0 : uniform(M.unit_item[u])) + q];
        kind = uniform(d.x) & 15;
        logg = (uniform(d.x) >> 4) & 15;
        logk = (uniform(d.x) >> 8) & 15;
        first = uniform(d.y);
        n = uniform(d.z);
        cnt = uniform(d.w);
        if (kind == kItemSeg) {
            const int per = (cnt + (1 << log_parts) - 1) >> log_parts;
            n += part * per;
            cnt = min(per, cnt - part * per);
            if (cnt <= 0) return;
        } else if (kind == kItemGroup) {
            const int log_unit = 6 - logg + log_parts;  // rows of one pass of every part
            const int per = ((n + (1 << log_unit) - 1) >> log_unit) << (6 - logg);
            first += part * per;
            n = min(per, n - part * per);
            if (n <= 0) return;
        } else if (part > 0) {
            return;
        }
    } else {
        if (part > 0) return;  // a pass
        const int lane = lane_here();
        const int rows = listed_rows(D, u, step);
        const int passes = lane < kClasses ? class_passes(M, lane, rows) : 0;
        int upto = passes;  // inclusive running sum over the classes
#pragma unroll
        for (int h = 1; h < 16; h <<= 1) {
            const int v = __shfl_up(upto, h, 64);
            if (lane >= h) upto += v;
        }
        const unsigned long long above = __ballot(lane < kClasses && upto > q);
        if (above == 0ull) return;
        const int c = __ffsll(static_cast<long long>(above)) - 1;
        const int at = q - (__shfl(upto, c, 64) - __shfl(passes, c, 64));
        const int have = uniform(__shfl(rows, c, 64));
        const int start = uniform(list_start(M, u, c));
        if (c == 0) {
            const int part = uniform(coherent_load(&V.wl_seg[start + at]));
            kind = kItemSeg;
            first = uniform(M.part_row[part]);
            n = part - uniform(M.seg_rows[first].y);
            cnt = -1;
        } else if (c == 1) {
            kind = kItemLong;
            first = uniform(coherent_load(&V.wl[start + at]));
        } else {
            logg = class_logg(M, c);
            logk = class_logk(M, c);
            const int per_pass = 64 >> logg;
            list = V.wl + start;
            first = uniform(at * per_pass);
            n = min(per_pass, have - first);
        }
    }
    int moved = 0;
    if (kind == kItemSeg) {
        seg_item<kRecords>(M, D, V, u, first, n, cnt, st, step);
        return;
    }
    if (kind == kItemLong) {
        moved = long_item(M, S, first);
    } else {
        switch (logk) {
            case 0: moved = group_item<1, kRecords>(M, S, first, n, logg, list); break;
            case 1: moved = group_item<2, kRecords>(M, S, first, n, logg, list); break;
            default: moved = group_item<4, kRecords>(M, S, first, n, logg, list); break;
        }
    }
    note_change(D, u, step, moved);
}

// Running sums of the pieces of the units of slots [base, base + win), and
// their all-rows bits, in LDS (the whole workgroup).
__device__ __forceinline__ void lay_out_window(const DevMatrix &M, const DevState &D, int step, int base, int win,
                                               int *sums, unsigned *dense) {
    const int lane = threadIdx.x & 63;
    const int wg_wave = threadIdx.x >> 6;
    __syncthreads();  // nobody still reads the previous window
    for (int g = wg_wave * 64; g < win; g += blockDim.x) {
        const int k = g + lane;
        int n = 0;
        UnitStep us{};
        if (k < win) {
            const int slot = base + k;
            const int u = M.replicas ? D.active[slot] : slot;
            us = unit_step_lane(M, D, u, step);
            if (us.active) n = us.all_rows ? unit_items(M, u) : list_passes(M, D, u, step);
        }
        const unsigned long long b = __ballot(us.all_rows);
        if (lane == 0) {
            dense[g >> 5] = static_cast<unsigned>(b);
            dense[(g >> 5) + 1] = static_cast<unsigned>(b >> 32);
        }
        sums[k] = n;
    }
    __syncthreads();
    if (wg_wave == 0) {
        int carry = 0;
        for (int g = 0; g < win; g += 64) {
            int v = sums[g + lane];
#pragma unroll
            for (int h = 1; h < 64; h <<= 1) {
                const int o = __shfl_up(v, h, 64);
                if (lane >= h) v += o;
            }
            sums[g + lane] = v + carry;
            carry += __shfl(v, 63, 64);
        }
    }
    __syncthreads();
}

// The sweep of a step over the waves of the grid: the pieces of every working
// unit, one unit after the other, dealt out with the grid's stride.  With
// several units, each workgroup lays out the running sums of their pieces in
// LDS (`window`, kWindowLdsBytes) for up to kWindowUnits of them at a time;
// a wave then finds its piece's unit with two ballots.  Also clears the
// counters of the lists that the step's publish will fill.
__device__ __forceinline__ void sweep_phase(const DevMatrix &M, const DevState &D, int step, int wave, int nwaves,
                                            int n_units, unsigned *window, const UnitStep &one) {
    int *st = status_row(D, step);
    const int n_slots = M.replicas ? D.n_active : n_units;
    if (M.mark_rows) {
        const int tid = blockIdx.x * blockDim.x + threadIdx.x;
        for (int k = tid; k < n_slots * kCountWords; k += gridDim.x * blockDim.x) {
            const int slot = k / kCountWords;
            const int u = M.replicas ? D.active[slot] : slot;
            coherent_store(&list_counts(D, u, step + 1)[k - slot * kCountWords], 0ull);
        }
    }
    const bool single = n_slots == 1;
    if (single && !one.active) return;
    const int u1 = M.replicas ? uniform(D.active[0]) : 0;
    int *sums = reinterpret_cast<int *>(window);            // kWindowUnits + 64
    unsigned *dense = window + kWindowUnits + 64;           // all-rows bits
    // Many bound vectors of one matrix: the workgroups of an XCD (they go round
    // the 8 XCDs) take an eighth of the pieces that lies together, so that an
    // L2 holds the snapshots of an eighth of the vectors in work, and every
    // workgroup has work whichever vectors still need any (one vector of 64 with
    // 4.4M nonzeros and 32 rounds of work: 2.5 ms; 5.8 with every eighth vector
    // to an XCD).  Only the locality hangs on where a workgroup really runs.
    const bool by_xcd = M.replicas && n_slots >= 64 && gridDim.x % 8 == 0;
    const int xcd = blockIdx.x & 7;
    const int chip_waves = nwaves;
    if (by_xcd) {
        const int waves = blockDim.x >> 6;
        wave = uniform((blockIdx.x >> 3) * waves + (threadIdx.x >> 6));
        nwaves = (gridDim.x >> 3) * waves;
    }
    int shift = 0;  // pieces of the windows before
    for (int base = 0; base < n_slots; base += kWindowUnits) {
        const int win = min(kWindowUnits, n_slots - base);
        const int blocks = (win + 63) / 64;
        int total;
        if (single) {
            total = one.all_rows ? unit_items(M, u1) : uniform(list_passes(M, D, u1, step));
        } else {
            lay_out_window(M, D, step, base, win, sums, dense);
            total = uniform(sums[blocks * 64 - 1]);
        }
        // items in up to 4 parts while the waves outnumber them: an item is
        // four passes or more, a chain of about 4 us each
        const int log_parts = total * 4 <= chip_waves ? 2 : (total * 2 <= chip_waves ? 1 : 0);
        const int parts = total << log_parts;
        const int begin = by_xcd ? (parts >> 3) * xcd + ((parts & 7) * xcd >> 3) : 0;
        const int end = by_xcd ? (parts >> 3) * (xcd + 1) + ((parts & 7) * (xcd + 1) >> 3) : parts;
        // the grid's stride goes on across the windows
        int q = (wave - shift) % nwaves;
        if (q < 0) q += nwaves;
        for (q += begin; q < end; q += nwaves) {
            const int piece = q >> log_parts;
            int u = u1, before = 0;
            bool all_rows = one.all_rows;
            if (!single) {
                const int lane = lane_here();
                int blk = 0;
                if (blocks > 1)
                    blk = uniform(__ffsll(static_cast<long long>(__ballot(
                                      lane < blocks && sums[min(lane, blocks - 1) * 64 + 63] > piece))) - 1);
                const int upto = sums[blk * 64 + lane];
                const int k = uniform(__ffsll(static_cast<long long>(__ballot(upto > piece))) - 1);
                before = uniform(k == 0 ? (blk == 0 ? 0 : sums[blk * 64 - 1]) : __shfl(upto, k - 1, 64));
                const int at = blk * 64 + k;
                const int slot = base + at;
                u = M.replicas ? uniform(D.active[slot]) : slot;
                all_rows = uniform((dense[at >> 5] >> (at & 31)) & 1u) != 0;
            }
            sweep_piece(M, D, u, piece - before, all_rows, q & ((1 << log_parts) - 1), log_parts, step, st);
        }
        shift = (shift + end - begin) % nwaves;
    }
}

// Applies the candidates of queued task `task` = unit * n_seg_parts + segment
// (one wave; the row's activity is read back from its SegState).  Returns the
// lane's accepted candidates; u: the task's unit.
template <int kMode>
__device__ __forceinline__ int apply_split_task(const DevMatrix &M, const DevState &D, int task, int &u) {
    constexpr int K = kSegLen / 64;
    const int lane = threadIdx.x & 63;
    task = uniform(task);
    u = task / M.n_seg_parts;
    const int part = task - u * M.n_seg_parts;
    const DevState V = unit_view(M, D, u);
    const Sink S = make_sink(V);
    const int lr = M.part_row[part];
    const int4 info = M.seg_rows[lr];
    const int r = info.x;
    int start, len;
    row_extent(M, r, start, len);
    const int s0 = (part - info.y) * kSegLen;
    const SegState *stp = &V.seg_state[lr];
    const double minact = coherent_load_d(&stp->minact);
    const double maxact = coherent_load_d(&stp->maxact);
    int ni, xi;
    coherent_load_2i(&stp->mininf, ni, xi);
    const double2 sd = M.sides[r];
    int moved = 0;
#pragma unroll
    for (int k = 0; k < K; k++) {
        const int e = s0 + lane * K + k;
        if (e < len) {
            const int jp = M.col[start + e];
            double l, uu;
            load_bounds<kMode>(M, V, jp & kIdMask, l, uu);
            moved += apply_entry(M, S, jp, M.val[start + e], l, uu, sd.x, sd.y, minact, maxact, ni, xi);
        }
    }
    return moved;
}

// The apply phase: the waves of the grid take the queued segments in turn.
__device__ __forceinline__ void apply_phase(const DevMatrix &M, const DevState &D, int step, int wave, int nwaves) {
    int *st = status_row(D, step);
    const int count = coherent_load(&st[kStatusApply]);
    for (int t = wave; t < count; t += nwaves) {
        int u;
        const int moved = apply_split_task<kRecords>(M, D, coherent_load(&D.apply_tasks[t]), u);
        note_change(D, u, step, moved);
    }
}

// ---------------------------------------------------------------------------
// publish phase
// ---------------------------------------------------------------------------

// Publishes bitmap word w of unit u (one half-wave of 32 lanes, lane b owns
// column 32 w + b; `bits` is the word as read by the scan): copies the
// accumulated bounds of the moved columns into the unit's snapshot, records
// a crossing as the unit's infeasible step and marks the rows of the moved
// columns for the next step.  A unit whose accepted candidates in this step
// reach its threshold processes all rows next step instead (no marks are
// pushed then).  Clears the word.
// Whether unit u processes all rows in the step after `step` (its accepted
// candidates of `step` reached its limit; the unit's all-rows step is set
// from the same counters by the publish phase's per-unit pass).  Lanes 0..15
// of each half-wave read the unit's counters: call with every lane of the
// wave, `valid` per half.
__device__ __forceinline__ bool decide_all_rows(const DevMatrix &M, const DevState &D, int u, bool valid, int step) {
    const int b = threadIdx.x & 31;
    int cnt = 0;
    if (valid && M.mark_rows && b < kMoveLanes)
        cnt = coherent_load(&D.moved[moved_index(u, step % kMoveSlots, b)]);
#pragma unroll
    for (int h = 1; h < kMoveLanes; h <<= 1) cnt += __shfl_xor(cnt, h, 64);
    cnt = __shfl(cnt, threadIdx.x & 32, 64);
    const int limit = valid ? coherent_load(&D.units[u].mark_limit) : 0;
    return valid && M.mark_rows && cnt >= limit;
}

// Marks column-to-row entries, N per lane (row[q], and its col_seg code, where
// valid[q]), for `step` of unit u, the same unit on the lanes of each half of
// the wave: the first to mark a row (a segment of a split row) lists it.  The
// entries take their ranks within the half and class in LDS, and the places
// of all classes in the unit's lists come from one atomic instruction (two
// classes a word, six lanes) per N entries a lane: the counters of a unit lie
// in one line, and every addition to it by a wave costs tens of nanoseconds.
// kHint: marks of a vector's first step (mark_stamp).
template <bool kHint, int N>
__device__ __forceinline__ void mark_entries(const DevMatrix &M, const DevState &V, int u, const bool (&valid)[N],
                                             const int (&row)[N], const int (&code)[N], int step) {
    __shared__ unsigned ranks[16][2][16];  // per wave and half: rows per class, then their first places
    const int lane = lane_here();
    const int b = lane & 31;
    unsigned *mine = ranks[threadIdx.x >> 6][lane >> 5];
    const int stamp = static_cast<int>(mark_stamp(step, kHint) + static_cast<unsigned>(V.persist[kPersistEpoch]));
    bool first[N], any = false;
#pragma unroll
    for (int q = 0; q < N; q++) {
        first[q] = false;
        if (valid[q]) {
            int *mark = code[q] >= 0 ? &V.seg_marks[code[q]] : &V.marks[row[q]];
            first[q] = __hip_atomic_exchange(mark, stamp, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) != stamp;
        }
        any |= first[q];
    }
    if (!__any(any)) return;
    if (b < 16) mine[b] = 0u;
    __builtin_amdgcn_wave_barrier();
    unsigned rank[N];
#pragma unroll
    for (int q = 0; q < N; q++) {
        rank[q] = 0u;
        if (first[q])
            rank[q] = __hip_atomic_fetch_add(&mine[code[q] >= 0 ? 0 : -1 - code[q]], 1u, __ATOMIC_RELAXED,
                                             __HIP_MEMORY_SCOPE_WORKGROUP);
    }
    __builtin_amdgcn_wave_barrier();
    if (b < (kClasses + 1) / 2) {
        const unsigned n0 = __hip_atomic_load(&mine[2 * b], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
        const unsigned n1 = __hip_atomic_load(&mine[2 * b + 1], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
        if ((n0 | n1) != 0u) {
            const unsigned long long old =
                __hip_atomic_fetch_add(&list_counts(V, u, step)[b], n0 | (static_cast<unsigned long long>(n1) << 32),
                                       __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            mine[2 * b] = static_cast<unsigned>(list_start(M, u, 2 * b)) + static_cast<unsigned>(old);
            mine[2 * b + 1] = static_cast<unsigned>(list_start(M, u, 2 * b + 1)) + static_cast<unsigned>(old >> 32);
        }
    }
    __builtin_amdgcn_wave_barrier();
#pragma unroll
    for (int q = 0; q < N; q++) {
        if (!first[q]) continue;
        if (code[q] >= 0) {
            coherent_store(&V.wl_seg[__hip_atomic_load(&mine[0], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP) + rank[q]],
                           code[q]);
            atomic_add_i(reinterpret_cast<int *>(&V.seg_count[M.part_row[code[q]]]), 1);
        } else {
            const unsigned at = __hip_atomic_load(&mine[-1 - code[q]], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
            coherent_store(&V.wl[at + rank[q]], row[q]);
        }
    }
    __builtin_amdgcn_wave_barrier();
}

__device__ __forceinline__ void publish_word(const DevMatrix &M, const DevState &D, int u, int w, unsigned bits,
                                             bool valid, int step, int all_rows_known) {
    const int lane = threadIdx.x & 63;
    const int b = lane & 31;
    if (valid && !M.replicas) u = M.word_unit[w];
    const DevState V = unit_view(M, D, u);
    if (valid && b == 0) coherent_store(&V.bm[w], 0u);
    const bool all_rows = all_rows_known >= 0 ? all_rows_known != 0 : decide_all_rows(M, D, u, valid, step);
    const bool moved = valid && ((bits >> b) & 1u);
    const int id = w * 32 + b;
    unsigned code = 0u;
    if (moved) {
        double l, uu;
        accumulated(M, V, id, l, uu);
        store_snapshot(M, V, id, l, uu);
        if (eps_gt(l, uu)) atomic_max_i(&D.units[u].infeasible, step);
        if (id < D.n_lds || id < D.n_codes) code = (l >= 1.0 ? 1u : 0u) | (uu < 1.0 ? 2u : 0u);
    }
    if (__any(code != 0u)) {
        // the new code bits of each 16 columns, ORed into their table word
        unsigned cw = code << ((id & 15) * 2);
#pragma unroll
        for (int h = 1; h < 16; h <<= 1) cw |= static_cast<unsigned>(__shfl_xor(static_cast<int>(cw), h, 64));
        if ((b & 15) == 0 && cw != 0u) atomic_or_u(&V.SB[id >> 4], cw);
    }
    const bool marks = M.mark_rows && valid && !all_rows;
    if (!__any(marks)) return;
    // rows of the moved columns, flattened over the 32 lanes of the half:
    // exclusive prefix of the columns' lengths, then lane i marks entries
    // i, i + 32, ... found by a binary search over the prefix
    const int c0 = moved && marks ? M.col_ptr[id] : 0;
    const int cn = moved && marks ? M.col_ptr[id + 1] - c0 : 0;
    int pre = cn;
#pragma unroll
    for (int d = 1; d < 32; d <<= 1) {
        const int v = __shfl_up(pre, d, 32);
        if (b >= d) pre += v;
    }
    const int total = __shfl(pre, 31, 32);
    const int longest = max(total, __shfl_xor(total, 32, 64));  // of both halves, which go together
    pre -= cn;  // exclusive
    // kMarkBatch entries per lane at a time: their index loads are all issued
    // before the marks they name are stored
    constexpr int kMarkBatch = 4;
    for (int base = 0; base < longest; base += 32 * kMarkBatch) {
        int row[kMarkBatch], sp[kMarkBatch];
        bool in[kMarkBatch];
#pragma unroll
        for (int q = 0; q < kMarkBatch; q++) {
            const int i = base + q * 32 + b;
            int lo = 0;
#pragma unroll
            for (int st = 16; st > 0; st >>= 1) {
                const int cand = lo + st;
                if (cand < 32 && __shfl(pre, cand, 32) <= i) lo = cand;
            }
            const int k = __shfl(c0, lo, 32) + i - __shfl(pre, lo, 32);
            row[q] = 0;
            sp[q] = -1;
            in[q] = i < total;
            if (in[q]) {
                row[q] = M.col_rows[k];
                sp[q] = M.col_seg[k];
            }
        }
        mark_entries<false>(M, V, u, in, row, sp, step + 1);
    }
}

// Publish phase of `step` over the waves of the grid: every wave scans 8
// bitmap words of one unit (replicas: the launch's units; blocks: the one
// shared bitmap), 64 where many units give every wave more to scan than that
// (the scan is a chain of loads per visit, 1 us each: 256 vectors of 100,000
// columns, dense steps 64 -> 52 us, late ones 24 ->
// 10), and publishes the nonzero ones two at a time; a unit with
// accepted candidates records that it, and the step, changed.  Also clears
// the next step's status row and the candidate counters two steps ahead.
__device__ __forceinline__ void publish_phase(const DevMatrix &M, const DevState &D, int step, int wave,
                                              int nwaves, int n_units) {
    constexpr int kChunk = 8;
    const int lane = threadIdx.x & 63;
    const int half = lane >> 5;
    const bool wide = M.replicas && D.n_active * ((M.nwords + 63LL) / 64) + 3 >= nwaves;
    const int span = wide ? 64 : kChunk;  // bitmap words per wave
    const int chunks = (M.nwords + span - 1) / span;
    const int n_chunks = (M.replicas ? D.n_active : 1) * chunks;
    // One unit in the launch (a single problem): the all-rows decision is
    // taken once per workgroup (its first wave reads the unit's counters,
    // final after the sweep's barrier) and shared through LDS instead of
    // once per chunk after the chunk's words arrive.
    __shared__ int single_all_rows;
    const bool single = M.replicas && D.n_active == 1;
    if (single) {
        if (threadIdx.x < 64) {
            const bool all_rows = decide_all_rows(M, D, uniform(D.active[0]), true, step);
            if (threadIdx.x == 0) single_all_rows = all_rows ? 1 : 0;
        }
        __syncthreads();
    }
    for (int c = wave; c < n_chunks; c += nwaves) {
        const int k = c / chunks;
        const int q = c - k * chunks;
        const int u = M.replicas ? uniform(D.active[k]) : 0;
        const DevState V = unit_view(M, D, u);
        const int w = q * span + lane;
        const unsigned bits = lane < span && w < M.nwords ? coherent_load(&V.bm[w]) : 0u;
        unsigned long long pending = __ballot(bits != 0u);
        if (!pending) continue;
        // one decision for the chunk's unit (replicas; blocks: when the
        // chunk's words all belong to one unit, as in a single problem)
        int known = -1;
        if (single) {
            known = uniform(single_all_rows);
        } else if (M.replicas) {
            known = decide_all_rows(M, D, u, true, step) ? 1 : 0;
        } else {
            const int u0 = uniform(M.word_unit[q * span]);
            const bool other = lane < span && w < M.nwords && M.word_unit[w] != u0;
            if (!__ballot(other)) known = decide_all_rows(M, D, u0, true, step) ? 1 : 0;
        }
        if (M.replicas && (known == 1 || !M.mark_rows)) {
            // no row marks to push: eight of the nonzero words at once,
            // their accumulator reads issued before any is used (lane b of
            // each half takes bit b of the half's word of every pair)
            constexpr int kPairs = kChunk / 2;
            do {
                int ids[kPairs];
                bool mv[kPairs];
                AccRaw raw[kPairs];
#pragma unroll
                for (int i = 0; i < kPairs; i++) {
                    int t0 = -1, t1 = -1;
                    if (pending) {
                        t0 = __ffsll(static_cast<long long>(pending)) - 1;
                        pending &= pending - 1;
                    }
                    if (pending) {
                        t1 = __ffsll(static_cast<long long>(pending)) - 1;
                        pending &= pending - 1;
                    }
                    const int t = half ? t1 : t0;
                    const int wt = q * span + (t < 0 ? 0 : t);
                    const unsigned wb = __shfl(bits, t < 0 ? 0 : t, 64);
                    if (t >= 0 && (lane & 31) == 0) coherent_store(&V.bm[wt], 0u);
                    ids[i] = wt * 32 + (lane & 31);
                    mv[i] = t >= 0 && ((wb >> (lane & 31)) & 1u);
                    raw[i] = mv[i] ? acc_load(M, V, ids[i]) : AccRaw{0, 0.0, 0.0};
                }
#pragma unroll
                for (int i = 0; i < kPairs; i++) {
                    unsigned code = 0u;
                    if (mv[i]) {
                        double l, uu;
                        acc_resolve(M, V, ids[i], raw[i], l, uu);
                        store_snapshot(M, V, ids[i], l, uu);
                        if (eps_gt(l, uu)) atomic_max_i(&D.units[u].infeasible, step);
                        if (ids[i] < D.n_lds || ids[i] < D.n_codes) code = (l >= 1.0 ? 1u : 0u) | (uu < 1.0 ? 2u : 0u);
                    }
                    if (__any(code != 0u)) {
                        unsigned cw = code << ((ids[i] & 15) * 2);
#pragma unroll
                        for (int h = 1; h < 16; h <<= 1)
                            cw |= static_cast<unsigned>(__shfl_xor(static_cast<int>(cw), h, 64));
                        if ((lane & 15) == 0 && cw != 0u) atomic_or_u(&V.SB[ids[i] >> 4], cw);
                    }
                }
            } while (pending);
            continue;
        }
        while (pending) {
            const int t0 = __ffsll(static_cast<long long>(pending)) - 1;
            pending &= pending - 1;
            int t1 = -1;
            if (pending) {
                t1 = __ffsll(static_cast<long long>(pending)) - 1;
                pending &= pending - 1;
            }
            const int t = half ? t1 : t0;
            const unsigned wb = __shfl(bits, t < 0 ? 0 : t, 64);
            publish_word(M, D, u, q * span + (t < 0 ? 0 : t), wb, t >= 0, step, known);
        }
    }
    // The units that accepted candidates in this step moved a bound: their
    // candidate counters (final since the sweep's barrier) set the unit's
    // and the step's changed flags, and the unit's all-rows step when they
    // reach its limit, one wave per unit, so that the words above need no
    // flag reads.
    const int n_flag_units = M.replicas ? D.n_active : n_units;
    for (int k = wave; k < n_flag_units; k += nwaves) {
        const int uu = M.replicas ? uniform(D.active[k]) : k;
        int cnt = lane < kMoveLanes
                      ? coherent_load(&D.moved[moved_index(uu, step % kMoveSlots, lane)])
                      : 0;
        const int limit = lane == 0 ? coherent_load(&D.units[uu].mark_limit) : 0;
#pragma unroll
        for (int h = 1; h < kMoveLanes; h <<= 1) cnt += __shfl_xor(cnt, h, 64);
        if (lane == 0 && cnt > 0) {
            coherent_store(&D.units[uu].changed[step & 1], step);
            if (M.mark_rows && cnt >= limit) coherent_store(&D.units[uu].markall, step + 1);
            // read first: many units set it
            if (coherent_load(&status_row(D, step)[kStatusChanged]) == 0)
                atomic_or_i(&status_row(D, step)[kStatusChanged], 1);
        }
    }
    const int tid = blockIdx.x * blockDim.x + threadIdx.x;
    const int stride = gridDim.x * blockDim.x;
    if (tid < kStatusWords) coherent_store(&status_row(D, step + 1)[tid], 0);
    for (int k = tid; k < n_units * kMoveLanes; k += stride) {
        const int uu = k / kMoveLanes, j = k - uu * kMoveLanes;
        coherent_store(&D.moved[moved_index(uu, (step + 2) % kMoveSlots, j)], 0);
    }
}

// ---------------------------------------------------------------------------
// step kernels (CPU_LOOP, GPU_LOOP)
// ---------------------------------------------------------------------------

// With `guard`, a launch first checks on the device whether
// the previous step changed anything; if not, the run is over and the launch
// does nothing.
__device__ __forceinline__ bool step_skipped(const DevState &D, int step, int first_step) {
    if (coherent_load(&D.global[kGlobalError]) != 0) return true;
    if (step <= first_step) return false;
    return coherent_load(&status_row(D, step - 1)[kStatusChanged]) == 0;
}

// The sweep of one step over a grid sized to the device.
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(5))) void sweep_kernel(
    DevMatrix M, DevState D_arg, int step, int guard, int first_step, int n_units) {
    // no LDS codes in the step kernels (a constant, so that the LDS reads compile out)
    DevState D = D_arg;
    D.n_lds = 0;
    __shared__ unsigned window[kWindowLdsBytes / 4];
    const bool skipped = guard && step_skipped(D, step, first_step);
    if (guard && blockIdx.x == 0 && threadIdx.x == 0)  // tells the host
        __hip_atomic_store(D.host_word, skipped ? kRoundsOver : step, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
    if (skipped) return;
    const int waves = blockDim.x >> 6;
    const int wave = uniform(blockIdx.x * waves + (threadIdx.x >> 6));
    UnitStep one{};
    if ((M.replicas ? D.n_active : n_units) == 1) one = unit_step(M, D, M.replicas ? D.active[0] : 0, step);
    sweep_phase(M, D, step, wave, gridDim.x * waves, n_units, window, one);
}

__global__ __launch_bounds__(256) void apply_split_kernel(DevMatrix M, DevState D_arg, int step, int guard,
                                                          int first_step) {
    DevState D = D_arg;
    D.n_lds = 0;
    if (guard && step_skipped(D, step, first_step)) return;
    const int waves = blockDim.x >> 6;
    apply_phase(M, D, step, uniform(blockIdx.x * waves + (threadIdx.x >> 6)), gridDim.x * waves);
}

__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(5))) void publish_kernel(DevMatrix M, DevState D_arg, int step, int guard,
                                                      int first_step, int n_units) {
    DevState D = D_arg;
    D.n_lds = 0;
    if (guard && step_skipped(D, step, first_step)) return;
    const int waves = blockDim.x >> 6;
    publish_phase(M, D, step, uniform(blockIdx.x * waves + (threadIdx.x >> 6)), gridDim.x * waves, n_units);
}

// ---------------------------------------------------------------------------
// persistent kernel
// ---------------------------------------------------------------------------

// Device-wide barrier.  Workgroups arrive at one of 8 group counters
// (blockIdx mod 8, each on its own cache line); the last arrival of a group
// arrives at the top counter, and the last of those advances the generation
// word that all others wait for.  Waiting is bounded by wall-clock time so
// that a fault elsewhere ends in an error flag instead of a hang.
// Everything the phases exchange is written with atomics or device-coherent
// stores, so no cache write-back is needed.  With `invalidate`, each
// workgroup invalidates its caches after the barrier so that its next
// gathers of the snapshot cannot hit lines cached before the publish.
// Always inlined: as a call it makes the caller spill its DevState argument
// to scratch and lose a wave of occupancy in the persistent kernel.
__device__ __forceinline__ bool grid_barrier(const DevState &D, unsigned nblocks, bool invalidate) {
    __shared__ int ok_sh;
    mem_wait();
    __syncthreads();
    if (threadIdx.x == 0) {
        int ok = 1;
        unsigned *top = D.barrier + kBarrierTop;
        unsigned *gen = D.barrier + kBarrierGen;
        const unsigned x = blockIdx.x & 7;
        unsigned *grp = D.barrier + kBarrierGroup + 32 * x;
        const unsigned per = nblocks / 8 + ((nblocks & 7) > x ? 1u : 0u);
        const unsigned groups = nblocks < 8 ? nblocks : 8;
        const unsigned g0 = coherent_load(gen);
        bool released = false;
        if (__hip_atomic_fetch_add(grp, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == per - 1) {
            coherent_store(grp, 0u);
            mem_wait();
            if (__hip_atomic_fetch_add(top, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == groups - 1) {
                coherent_store(top, 0u);
                mem_wait();
                __hip_atomic_fetch_add(gen, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                released = true;
            }
        }
        if (!released) {
            const long long t0 = wall_clock64();
            while (coherent_load(gen) == g0) {
                __builtin_amdgcn_s_sleep(1);
                if (coherent_load(&D.global[kGlobalError])) {
                    ok = 0;
                    break;
                }
                if (wall_clock64() - t0 > kWaitTimeoutTicks) {
                    atomic_or_i(&D.global[kGlobalError], 1);
                    ok = 0;
                    break;
                }
            }
        }
        if (invalidate) __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "agent");
        ok_sh = ok;
    }
    __syncthreads();
    return ok_sh != 0;
}

// Steps [first_step, first_step + max_steps) in one persistent launch
// (MEGAKERNEL).  Every workgroup walks the work of a phase with a grid
// stride, all meet at a barrier, and all read the same status words, so all
// take the same decision to go on: the run ends after a step in which no
// unit moved a bound.  Phases of a step: sweep; apply of the split rows when
// the sweep queued any; publish.
template <int kThreads, bool kLds>
__global__ __launch_bounds__(kThreads) __attribute__((amdgpu_waves_per_eu(4))) void mega_kernel(DevMatrix M, DevState D_arg, int first_step, int max_steps,
                                                        int n_units) {
    // kLds: a launch of one unit that reads binary columns from LDS; without
    // it n_lds is a constant 0, and the LDS reads compile out (with it n_codes)
    DevState D = D_arg;
    if constexpr (kLds) D.n_codes = 0;
    else D.n_lds = 0;
    const unsigned nblocks = gridDim.x;
    const int waves = blockDim.x >> 6;
    const int wave = uniform(blockIdx.x * waves + (threadIdx.x >> 6));
    const int nwaves = gridDim.x * waves;
    const int n_slots = M.replicas ? D.n_active : n_units;  // replicas: positions in the launch's list
    for (int step = first_step; step < first_step + max_steps; step++) {
        int *st = status_row(D, step);
        UnitStep one{};
        if (n_slots == 1) {
            const int u1 = M.replicas ? uniform(D.active[0]) : 0;
            one = unit_step(M, D, u1, step);
            if (D.n_lds > 0) {
                // the unit's binary codes as published by the previous step
                // (the waves of this workgroup that read the LDS in the
                // previous step are past its barriers)
                const uint4 *src = reinterpret_cast<const uint4 *>(unit_view(M, D, u1).SB);
                uint4 *dst = reinterpret_cast<uint4 *>(dyn_lds);
                for (int i = threadIdx.x; i < D.n_lds / 64; i += blockDim.x) dst[i] = src[i];
                __syncthreads();
            }
        }
        sweep_phase(M, D, step, wave, nwaves, n_units, dyn_lds, one);
        if (!grid_barrier(D, nblocks, false)) return;
        if (coherent_load(&st[kStatusApply]) > 0) {
            apply_phase(M, D, step, wave, nwaves);
            if (!grid_barrier(D, nblocks, false)) return;
        }
        publish_phase(M, D, step, wave, nwaves, n_units);
        if (!grid_barrier(D, nblocks, true)) return;
        if (!coherent_load(&st[kStatusChanged])) break;
    }
}

template __global__ void mega_kernel<256, false>(DevMatrix, DevState, int, int, int);
template __global__ void mega_kernel<512, false>(DevMatrix, DevState, int, int, int);
template __global__ void mega_kernel<1024, false>(DevMatrix, DevState, int, int, int);
template __global__ void mega_kernel<256, true>(DevMatrix, DevState, int, int, int);
template __global__ void mega_kernel<512, true>(DevMatrix, DevState, int, int, int);
template __global__ void mega_kernel<1024, true>(DevMatrix, DevState, int, int, int);

// ---------------------------------------------------------------------------
// double-buffered rounds of one bound vector (gdp_device.h, RoundPlan)
// ---------------------------------------------------------------------------

// The bitmap of the columns that round `step` moves.  Three take turns: round
// s reads the one of round s - 1 while it writes its own and clears that of
// round s + 1.
__device__ __forceinline__ unsigned *moved_bitmap(const RoundPlan &R, int step) {
    const int k = step % 3;
    return k == 0 ? R.bm[0] : (k == 1 ? R.bm[1] : R.bm[2]);
}

// The columns that the round before `step` moved, copied to LDS by the whole
// workgroup, if the round has n_items enough for it; else every row counts as
// moved.  Eight loads a thread are in flight (one at a time, 64 KB took 8 us).
// Every thread calls it; ends with a barrier.
template <int kMode, bool kTest>
__device__ __forceinline__ MovedBits load_moved_bits(const DevMatrix &M, const RoundPlan &R, int step, int n_items,
                                                     unsigned *words) {
    if constexpr (!kTest) {
        __syncthreads();
        return MovedBits{nullptr, 0u};
    }
    if (step == 1 || n_items < kMinTestItems) {
        __syncthreads();
        return MovedBits{nullptr, 0u};
    }
    constexpr int kFlight = 8;
    const long long *bm = reinterpret_cast<const long long *>(moved_bitmap(R, step - 1));
    long long *out = reinterpret_cast<long long *>(words);
    const int n = R.bit_words / 2, have = (M.nwords + 1) / 2;  // (the bitmaps are a multiple of 8 bytes)
    const int stride = static_cast<int>(blockDim.x);
    for (int w0 = threadIdx.x; w0 < n; w0 += kFlight * stride) {
        long long v[kFlight];
#pragma unroll
        for (int q = 0; q < kFlight; q++) {
            const int w = w0 + q * stride;
            v[q] = 0;
            if (w < n && w < have) v[q] = kMode == kWideCoherent ? coherent_load(&bm[w]) : bm[w];
        }
#pragma unroll
        for (int q = 0; q < kFlight; q++) {
            const int w = w0 + q * stride;
            if (w >= n) break;
            for (int x = w + n; x < have; x += n) v[q] |= kMode == kWideCoherent ? coherent_load(&bm[x]) : bm[x];
            out[w] = v[q];
        }
    }
    __syncthreads();
    return MovedBits{words, static_cast<unsigned>(R.bit_words - 1)};
}

// The state of round `step`: records read from block (step - 1) & 1,
// candidates and moved-column bits into the other parity's arrays.
__device__ __forceinline__ DevState round_view(const DevMatrix &M, const DevState &D, const RoundPlan &R, int step) {
    const bool odd = step & 1;
    char *nxt = odd ? R.block[1] : R.block[0];
    DevState V = D;
    V.S16 = reinterpret_cast<unsigned *>(odd ? R.block[0] : R.block[1]);
    V.AI = reinterpret_cast<int2 *>(nxt);
    V.AF = reinterpret_cast<double2 *>(nxt + M.snap_offF);
    V.AX = odd ? R.AX[1] : R.AX[0];
    V.bm = moved_bitmap(R, step);
    V.n_lds = 0;
    return V;
}

// The accumulator view of a parity (as read after its round).
__device__ __forceinline__ DevState block_view(const DevMatrix &M, const DevState &D, const RoundPlan &R, int parity) {
    char *block = parity ? R.block[1] : R.block[0];
    DevState V = D;
    V.AI = reinterpret_cast<int2 *>(block);
    V.AF = reinterpret_cast<double2 *>(block + M.snap_offF);
    V.AX = parity ? R.AX[1] : R.AX[0];
    return V;
}

// Folds the columns that round step - 1 moved into the block of round `step`
// and clears the bitmap of the next round (without kTest its own).  Returns whether one of the lane's columns is
// crossed.  Each wave takes `chunk` words of the bitmap at a time (one lane
// each) and works through the nonzero ones two at a time, a half-wave per
// word.
// With kUnits (a batch), only words of the units in the run, run[u] != 0, are
// folded: a unit that has crossed keeps the block of its last round as it is.
template <bool kUnits, bool kTest>
__device__ __forceinline__ bool carry_moved(const DevMatrix &M, const DevState &D, const RoundPlan &R, int step,
                                            int wave, int nwaves, const int *run) {
    const DevState C = block_view(M, D, R, (step - 1) & 1);
    const DevState N = block_view(M, D, R, step & 1);
    unsigned *bm = moved_bitmap(R, step - 1);
    unsigned *next_bm = moved_bitmap(R, step + 1);
    const int lane = threadIdx.x & 63;
    const int half = lane >> 5, b = lane & 31;
    int chunk = (M.nwords + nwaves - 1) / nwaves;
    chunk = chunk < 2 ? 2 : (chunk > 64 ? 64 : chunk);
    bool crossed = false;
    for (int w0 = (nwaves - 1 - wave) * chunk; w0 < M.nwords; w0 += nwaves * chunk) {
        const int w = w0 + lane;
        unsigned bits = 0u;
        if (lane < chunk && w < M.nwords) {
            bits = coherent_load(&bm[w]);
            if constexpr (kTest) {
                if (coherent_load(&next_bm[w]) != 0u) coherent_store(&next_bm[w], 0u);
            } else if (bits) {  // nobody else reads it
                coherent_store(&bm[w], 0u);
            }
        }
        unsigned long long pending = __ballot(bits != 0u);
        while (pending) {
            const int t0 = __ffsll(static_cast<long long>(pending)) - 1;
            pending &= pending - 1;
            int t1 = -1;
            if (pending) {
                t1 = __ffsll(static_cast<long long>(pending)) - 1;
                pending &= pending - 1;
            }
            const int t = half ? t1 : t0;
            const unsigned wb = __shfl(bits, t < 0 ? 0 : t, 64);
            if (t < 0 || !((wb >> b) & 1u)) continue;
            const int id = (w0 + t) * 32 + b;
            int unit = 0;
            if constexpr (kUnits) {
                unit = M.word_unit[w0 + t];
                if (!run[unit]) continue;
            }
            const AccRaw raw = acc_load(M, C, id);
            double l, u;
            acc_resolve(M, C, id, raw, l, u);
            if (eps_gt(l, u)) {
                crossed = true;
                if constexpr (kUnits) atomic_max_i(&D.units[unit].infeasible, step - 1);
            }
            if (id < M.n_int) {
                atomic_max_i(&N.AI[id].x, static_cast<int>(static_cast<unsigned long long>(raw.w) & 0xffffffffull));
                atomic_min_i(&N.AI[id].y, static_cast<int>(static_cast<unsigned long long>(raw.w) >> 32));
            } else {
                atomic_max_d(&N.AF[id - M.n_int].x, raw.fl);
                atomic_min_d(&N.AF[id - M.n_int].y, raw.fu);
            }
        }
    }
    return crossed;
}

// Lists the items of the rounds: the segments of the split rows, then the
// bins' rows from wide to narrow.
__global__ __launch_bounds__(256) void plan_rounds_kernel(DevMatrix M, RoundBins B, int4 *items) {
    const int n = B.item0[kPlanBins];
    for (int it = blockIdx.x * blockDim.x + threadIdx.x; it < n; it += gridDim.x * blockDim.x) {
        int4 d = make_int4(0, 0, 0, 0);
        if (it < B.n_segs) {
            const int lr = M.part_row[it];
            d = make_int4(kItemSeg, lr, it - M.seg_rows[lr].y, 1);
        } else {
#pragma unroll
            for (int q = 0; q < kPlanBins; q++)
                if (it >= B.item0[q] && it < B.item0[q + 1]) {
                    const int first = B.row0[q] + (it - B.item0[q]) * B.rows_per_item[q];
                    d = make_int4(kItemGroup | (B.logg[q] << 4) | (B.logk[q] << 8), first,
                                  min(B.rows_per_item[q], B.row0[q + 1] - first), 0);
                }
        }
        items[it] = d;
    }
}

// Item `it` of a round.  Returns the lane's accepted candidates.
template <int kMode, bool kTest>
__device__ __forceinline__ int round_item(const DevMatrix &M, const DevState &V, const RoundPlan &R, int it, int step,
                                          int *st, const MovedBits &B) {
    int4 d = R.items[uniform(it)];
    d.x = uniform(d.x);
    d.y = uniform(d.y);
    d.z = uniform(d.z);
    if ((d.x & 15) == kItemSeg) {
        seg_item<kMode, kTest>(M, V, V, 0, d.y, d.z, 1, st, step, B);
        return 0;
    }
    const int logg = (d.x >> 4) & 15;
    const Sink S = make_sink(V);
    switch ((d.x >> 8) & 15) {
        case 0: return group_item<1, kMode, kTest>(M, S, d.y, d.z, logg, nullptr, B);
        case 1: return group_item<2, kMode, kTest>(M, S, d.y, d.z, logg, nullptr, B);
        default: return group_item<4, kMode, kTest>(M, S, d.y, d.z, logg, nullptr, B);
    }
}

// Resets the state words, the status ring, the global words and the
// barrier's arrival slots for a run (one workgroup).  `fail`: the error word of
// a failed wait is set from the start.
__global__ __launch_bounds__(256) void reset_rounds_kernel(DevState D, RoundPlan R, int fail) {
    const int tid = threadIdx.x;
    for (int u = tid; u < R.n_units; u += 256) {
        UnitState s = {};
        s.start = 1;
        s.markall = 1;
        s.max_rounds = R.max_rounds;
        s.mark_limit = R.mark_limit;
        D.units[u] = s;
    }
    for (int k = tid; k < kStatusRows * kStatusWords; k += 256) D.status[k] = 0;
    for (int k = tid; k < kGlobalWords; k += 256) D.global[k] = k == kGlobalError ? fail : 0;
    for (int k = tid; k < 2 * kMoveLanes * R.n_units; k += 256)
        D.moved[moved_index(k / (2 * kMoveLanes), k & 1, (k >> 1) % kMoveLanes)] = 0;
    for (int k = tid; k < 2 * kMaxGatherBlocks * R.slot_words; k += 256) R.slots[k] = 0ull;
}

// Loads the caller's vectors into both blocks and flags crossed bounds and
// bounds outside a column's storage class (the storage classes of the
// original matrix: n16, n_bin of the arguments).  kUnits: a batch.  The exact
// integer accumulators are clean unless some run of this state has used them;
// `first` (a new state, or one that was another problem's before) cleans them
// (both of every integer column: 9.6M of them 47 us of a call of 544).
template <bool kUnits>
__global__ __launch_bounds__(256) void load_rounds_kernel(DevMatrix M, DevState D, RoundPlan R, int n16, int n_bin,
                                                          int first) {
    const int used = D.persist[kPersistAx];  // (of a new state: anything)
    const bool ax = (first | used) != 0;
    const int tid = blockIdx.x * blockDim.x + threadIdx.x;
    const int stride = gridDim.x * blockDim.x;
    const DevState A = block_view(M, D, R, 0), B = block_view(M, D, R, 1);
    for (int id = tid; id < M.n; id += stride) {
        const int j = M.perm[id];
        int unit = 0;
        double l = 0.0, u = 0.0;
        if (!kUnits || j >= 0) {  // a batch has padding ids
            if constexpr (kUnits) unit = M.word_unit[id >> 5];
            l = R.lbs[j];
            u = R.ubs[j];
        }
        if (eps_gt(l, u)) atomic_or_i(&D.units[unit].crossed, 1);
        if (id < M.n_int) {
            const double lim = id < n16 ? 32767.0 : 2147483647.0;
            const double lo_lim = id < n_bin ? 0.0 : -lim, hi_lim = id < n_bin ? 1.0 : lim;
            const bool fits = l >= lo_lim && l <= hi_lim && u >= lo_lim && u <= hi_lim && floor(l) == l &&
                              floor(u) == u;
            if (!fits && !eps_gt(l, u)) {
                atomic_or_i(&D.units[unit].envelope, 1);
                if constexpr (kUnits) atomic_or_i(&D.global[kGlobalEnvelope], 1);
            }
            const int2 v = make_int2(fits ? static_cast<int>(l) : 0, fits ? static_cast<int>(u) : 0);
            A.AI[id] = v;
            B.AI[id] = v;
            if (ax) A.AX[id] = B.AX[id] = make_double2(-INFINITY, INFINITY);
        } else {
            A.AF[id - M.n_int] = make_double2(l, u);
            B.AF[id - M.n_int] = make_double2(l, u);
        }
    }
    if (tid == 0) A.AF[M.n - M.n_int] = B.AF[M.n - M.n_int] = make_double2(0.0, 0.0);  // the padding entries' column
    for (int w = tid; w < (M.nwords + 1) / 2 * 2; w += stride) {
        R.bm[0][w] = 0u;
        R.bm[1][w] = 0u;
        R.bm[2][w] = 0u;
    }
    for (int q = tid; q < M.n_seg_rows; q += stride) D.seg_count[q] = 0u;
}

template __global__ void load_rounds_kernel<false>(DevMatrix, DevState, RoundPlan, int, int, int);
template __global__ void load_rounds_kernel<true>(DevMatrix, DevState, RoundPlan, int, int, int);

// Whether a round moved a bound, for the launches: the round's number in any
// of kMoveLanes words, each on its own line, by parity (the last rounds of
// each parity, so that no round has to clear them).  Writers look first: a
// store that every workgroup sends to one line costs about 50 ns each.
__device__ __forceinline__ void note_round_moved(const DevState &D, int step, int unit = 0) {
    int *w = &D.moved[moved_index(unit, step & 1, blockIdx.x % kMoveLanes)];
    if (coherent_load(w) != step) coherent_store(w, step);
}
__device__ __forceinline__ bool round_moved(const DevState &D, int step) {
    const int lane = threadIdx.x & 63;
    const int w = lane < kMoveLanes ? coherent_load(&D.moved[moved_index(0, step & 1, lane)]) : 0;
    return __any(w == step);
}

// One round as one launch.  The launch first checks on the device whether
// the run goes on (input usable, not infeasible, the previous round moved a
// bound); the first workgroup tells the host: its word becomes `step` when
// the round runs, else kRoundsOver.
template <bool kTest>
__global__ __launch_bounds__(kTest ? 512 : 256) __attribute__((amdgpu_waves_per_eu(kTest ? 4 : 5))) void round_kernel(
    DevMatrix M, DevState D, RoundPlan R, int step) {
    __shared__ int any_moved;
    const long long *p = reinterpret_cast<const long long *>(&D.units[0]);
    const long long w0 = coherent_load(p), w2 = coherent_load(p + 2);
    const bool runs = round_runs(step, static_cast<int>(w0 >> 32), w2 != 0) && (step == 1 || round_moved(D, step - 1));
    if (blockIdx.x == 0 && threadIdx.x == 0)
        __hip_atomic_store(D.host_word, runs ? step : kRoundsOver, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
    if (!runs) return;
    if (threadIdx.x == 0) any_moved = 0;
    const MovedBits B = load_moved_bits<kWide, kTest>(M, R, step, R.n_items, dyn_lds);
    const int waves = blockDim.x >> 6;
    const int wave = uniform(blockIdx.x * waves + (threadIdx.x >> 6));
    const int nwaves = gridDim.x * waves;
    int *st = status_row(D, step);
    const DevState V = round_view(M, D, R, step);
    if (step > 1 && carry_moved<false, kTest>(M, D, R, step, wave, nwaves, nullptr)) atomic_max_i(&D.units[0].infeasible, step - 1);
    int moved = 0;
    for (int it = wave; it < R.n_items; it += nwaves) moved |= round_item<kWide, kTest>(M, V, R, it, step, st, B);
    if (__any(moved != 0) && (threadIdx.x & 63) == 0) any_moved = 1;
    __syncthreads();
    if (threadIdx.x == 0 && any_moved) note_round_moved(D, step);
}

// The candidates of the split rows whose gate passed in the round.
__global__ __launch_bounds__(256) void round_apply_kernel(DevMatrix M, DevState D, RoundPlan R, int step) {
    const int count = coherent_load(&status_row(D, step)[kStatusApply]);
    const int waves = blockDim.x >> 6;
    const DevState V = round_view(M, D, R, step);
    int moved = 0, u;
    for (int t = blockIdx.x * waves + (threadIdx.x >> 6); t < count; t += gridDim.x * waves)
        moved |= apply_split_task<kWide>(M, V, coherent_load(&D.apply_tasks[t]), u);
    if (__any(moved != 0) && (threadIdx.x & 63) == 0) note_round_moved(D, step);
}

// Grid barrier by gathering: every workgroup stores its arrival (sequence
// number and flags) into a slot of its own, and the first wave of every
// workgroup polls all slots, so that a barrier is one store and one load
// deep and hands every workgroup the union of all flags.  Two sets of slots
// take turns: a set is written again only after everybody has left the
// barrier between.  Waiting is bounded as in grid_barrier.
// wg_flags (LDS, zero at first): the workgroup's flags, two words in turn.
__device__ __forceinline__ bool gather_barrier(const DevState &D, const RoundPlan &R, unsigned seq, unsigned flags,
                                               unsigned *wg_flags, unsigned &all_flags) {
    __shared__ unsigned result[2];
    mem_wait();
    if (flags) atomicOr(&wg_flags[seq & 1], flags);
    __syncthreads();
    if (threadIdx.x < 64) {
        unsigned long long *slots = R.slots + (seq & 1) * kMaxGatherBlocks;
        const int nb = gridDim.x;
        if (threadIdx.x == 0)
            coherent_store(&slots[blockIdx.x], (static_cast<unsigned long long>(seq) << 32) | wg_flags[seq & 1]);
        unsigned got = 0u;
        bool ok = true;
        const long long t0 = wall_clock64();
        for (int base = 0; base < nb && ok; base += 64) {
            const int k = base + static_cast<int>(threadIdx.x);
            while (true) {
                const unsigned long long v =
                    k < nb ? coherent_load(&slots[k]) : (static_cast<unsigned long long>(seq) << 32);
                if (!__any(static_cast<unsigned>(v >> 32) != seq)) {
                    got |= static_cast<unsigned>(v);
                    break;
                }
                if (wall_clock64() - t0 > kWaitTimeoutTicks || coherent_load(&D.global[kGlobalError])) {
                    ok = false;
                    break;
                }
            }
        }
#pragma unroll
        for (int h = 1; h < 64; h <<= 1) got |= static_cast<unsigned>(__shfl_xor(static_cast<int>(got), h, 64));
        if (threadIdx.x == 0) {
            if (!ok) atomic_or_i(&D.global[kGlobalError], 1);
            wg_flags[(seq + 1) & 1] = 0u;
            result[0] = got;
            result[1] = ok ? 1u : 0u;
        }
    }
    __syncthreads();
    all_flags = result[0];
    return result[1] != 0u;
}

// Rounds 1 .. max_rounds in one persistent launch.  Bounds are gathered with
// device-coherent loads (nothing is invalidated between the rounds, so the
// matrix stays in the caches); one barrier per round, and a second one in
// rounds in which a split row passed its gate.
template <bool kTest>
__global__ __launch_bounds__(1024) void rounds_kernel(DevMatrix M, DevState D, RoundPlan R) {
    constexpr unsigned kMoved = 1u, kCrossed = 2u;
    const long long w2 = coherent_load(reinterpret_cast<const long long *>(&D.units[0]) + 2);
    if (w2 != 0) return;  // crossed or outside the envelope
    const int waves = blockDim.x >> 6;
    const int wave = uniform(blockIdx.x * waves + (threadIdx.x >> 6));
    const int nwaves = gridDim.x * waves;
    __shared__ unsigned wg_flags[2];
    if (threadIdx.x < 2) wg_flags[threadIdx.x] = 0u;
    __syncthreads();
    unsigned seq = 0, all = 0;
    int last = 0, infeasible = 0;
    bool ok = true;
    for (int step = 1; ok && step <= R.max_rounds; step++) {
        int *st = status_row(D, step);
        const DevState V = round_view(M, D, R, step);
        const MovedBits B = load_moved_bits<kWideCoherent, kTest>(M, R, step, R.n_items, dyn_lds);
        unsigned flags = 0u;
        if (step > 1 && carry_moved<false, kTest>(M, D, R, step, wave, nwaves, nullptr)) flags |= kCrossed;
        for (int it = wave; it < R.n_items; it += nwaves)
            if (round_item<kWideCoherent, kTest>(M, V, R, it, step, st, B)) flags |= kMoved;
        ok = gather_barrier(D, R, ++seq, flags, wg_flags, all);
        unsigned seen = all;
        if (ok && M.n_seg_parts > 0) {
            const int count = coherent_load(&st[kStatusApply]);
            if (count > 0) {
                flags = 0u;
                int u;
                for (int t = wave; t < count; t += nwaves)
                    if (apply_split_task<kWideCoherent>(M, V, coherent_load(&D.apply_tasks[t]), u)) flags |= kMoved;
                ok = gather_barrier(D, R, ++seq, flags, wg_flags, all);
                seen |= all;
            }
        }
        if (!ok) break;
        if (seen & kCrossed) {
            infeasible = step - 1;
            break;
        }
        if (!(seen & kMoved)) break;
        last = step;
    }
    if (blockIdx.x == 0 && threadIdx.x == 0) {
        D.units[0].infeasible = infeasible;
        D.moved[moved_index(0, last & 1, 0)] = last;
    }
}

// The gather barrier with a bit per unit of a batch: a workgroup's arrival is
// R.slot_words words, each the sequence number and the bits of 31 units (bit
// 31: a crossed unit among them), so that every word shows by itself that it
// has arrived.  All waves poll, 64 workgroups' words of one kind each.
// own / all (LDS, 2 x kMaxSlotWords, zero at first): the workgroup's bits and
// the union, two sets in turn.
__device__ __forceinline__ bool gather_units(const DevState &D, const RoundPlan &R, unsigned seq,
                                             unsigned (*own)[kMaxSlotWords], unsigned (*all)[kMaxSlotWords],
                                             int *wg_ok) {
    const int set = seq & 1;
    mem_wait();
    __syncthreads();
    unsigned long long *slots = R.slots + static_cast<size_t>(set) * kMaxGatherBlocks * R.slot_words;
    const int tid = threadIdx.x, lane = tid & 63, nb = gridDim.x;
    if (tid < R.slot_words)
        coherent_store(&slots[tid * kMaxGatherBlocks + blockIdx.x],
                       (static_cast<unsigned long long>(seq) << 32) | own[set][tid]);
    if (tid < kMaxSlotWords) {
        own[set ^ 1][tid] = 0u;
        all[set ^ 1][tid] = 0u;
    }
    const int groups = (nb + 63) / 64;
    const long long t0 = wall_clock64();
    for (int c = uniform(tid >> 6); c < groups * R.slot_words; c += blockDim.x >> 6) {
        const int word = c / groups, k = (c - word * groups) * 64 + lane;
        unsigned got = 0u;
        while (true) {
            const unsigned long long v = k < nb ? coherent_load(&slots[word * kMaxGatherBlocks + k])
                                                : (static_cast<unsigned long long>(seq) << 32);
            if (!__any(static_cast<unsigned>(v >> 32) != seq)) {
                got = static_cast<unsigned>(v);
                break;
            }
            if (wall_clock64() - t0 > kWaitTimeoutTicks || coherent_load(&D.global[kGlobalError])) {
                if (lane == 0) {
                    atomic_or_i(&D.global[kGlobalError], 1);
                    *wg_ok = 0;
                }
                break;
            }
        }
#pragma unroll
        for (int h = 1; h < 64; h <<= 1) got |= static_cast<unsigned>(__shfl_xor(static_cast<int>(got), h, 64));
        if (lane == 0 && got) atomicOr(&all[set][word], got);
    }
    __syncthreads();
    return *wg_ok != 0;
}

// The running totals of the items of the instances in the run, by one wave.
__device__ __forceinline__ void run_totals(int n_units, const int *run, const int *first, int *upto) {
    const int lane = threadIdx.x & 63;
    int before = 0;
    for (int u0 = 0; u0 < n_units; u0 += 64) {
        const int u = u0 + lane;
        int inc = run[u] ? first[u + 1] - first[u] : 0;
#pragma unroll
        for (int h = 1; h < 64; h <<= 1) {
            const int x = __shfl_up(inc, h, 64);
            if (lane >= h) inc += x;
        }
        upto[u] = before + inc;
        before += __shfl(inc, 63, 64);
    }
}
// The instance whose item is the t-th of the round: one LDS read and a ballot
// per 64 instances.
__device__ __forceinline__ int run_unit(int n_units, const int *upto, int t) {
    int u = 0;
    for (int u0 = 0; u0 < n_units; u0 += 64)
        u += __popcll(__ballot(upto[u0 + static_cast<int>(threadIdx.x & 63)] <= t));
    return uniform(u);
}

// The rounds of a batch in one persistent launch: the instances side by side
// in the two blocks, each round over the items of the instances that moved a
// bound in the round before.  Every workgroup learns the moved and crossed
// instances from the barrier and keeps its own list of them, with the running
// totals of their items, in LDS.
// Bound by the bounds' gathers while most instances run, by the barrier and
// one pass's chain of loads, butterfly and divisions (8 us) in the tail.  64
// instances of 42,000 entries, 58 rounds: 17 us a round (three phases: 47).
template <bool kTest>
__global__ __launch_bounds__(1024) void batch_rounds_kernel(DevMatrix M, DevState D, RoundPlan R) {
    __shared__ int run[kMaxRoundUnits];      // the instance takes part in the round
    __shared__ int last[kMaxRoundUnits];     // its last round that moved a bound
    __shared__ int first[kMaxRoundUnits + 1];  // its first item
    __shared__ int upto[kMaxRoundUnits];     // items of the instances in the run up to and with this one
    __shared__ unsigned own[2][kMaxSlotWords], all[2][kMaxSlotWords];
    __shared__ int wg_ok;
    const int tid = threadIdx.x, lane = tid & 63;
    const int waves = blockDim.x >> 6;
    const int wave = uniform(blockIdx.x * waves + (tid >> 6));
    const int nwaves = gridDim.x * waves;
    const int n_units = R.n_units;
    for (int u = tid; u < kMaxRoundUnits; u += blockDim.x) {
        // neither crossed nor outside the envelope
        run[u] = u < n_units && coherent_load(reinterpret_cast<const long long *>(&D.units[u]) + 2) == 0;
        last[u] = 0;
    }
    for (int u = tid; u <= n_units; u += blockDim.x) first[u] = R.unit_item[u];
    if (tid < kMaxSlotWords) own[0][tid] = own[1][tid] = all[0][tid] = all[1][tid] = 0u;
    if (tid == 0) wg_ok = 1;
    __syncthreads();
    unsigned seq = 0;
    for (int step = 1; step <= R.max_rounds; step++) {
        if (tid < 64) run_totals(n_units, run, first, upto);
        __syncthreads();
        const int total = upto[(n_units - 1) | 63];
        if (total == 0) break;
        const MovedBits B = load_moved_bits<kWideCoherent, kTest>(M, R, step, total, dyn_lds);
        int *st = status_row(D, step);
        const DevState V = round_view(M, D, R, step);
        const int set = (seq + 1) & 1;
        if (step > 1 && carry_moved<true, kTest>(M, D, R, step, wave, nwaves, run))
            for (int k = 0; k < R.slot_words; k++) atomicOr(&own[set][k], 1u << 31);
        for (int t = wave; t < total; t += nwaves) {
            const int u = run_unit(n_units, upto, t);
            const int it = uniform(first[u + 1] - upto[u]) + t;
            const int moved = round_item<kWideCoherent, kTest>(M, V, R, it, step, st, B);
            if (__any(moved != 0) && lane == 0) atomicOr(&own[set][u / 31], 1u << (u % 31));
        }
        if (!gather_units(D, R, ++seq, own, all, &wg_ok)) break;
        unsigned *seen = all[seq & 1];
        bool crossed = false;
        if (M.n_seg_parts > 0) {
            const int count = coherent_load(&st[kStatusApply]);
            if (count > 0) {
                // (the bits of the round go on into the second barrier)
                const int set2 = (seq + 1) & 1;
                if (tid < R.slot_words) atomicOr(&own[set2][tid], seen[tid]);
                for (int t = wave; t < count; t += nwaves) {
                    const int task = coherent_load(&D.apply_tasks[t]);
                    int u;
                    const int moved = apply_split_task<kWideCoherent>(M, V, task, u);
                    u = uniform(M.seg_rows[M.part_row[uniform(task)]].w);
                    if (__any(moved != 0) && lane == 0) atomicOr(&own[set2][u / 31], 1u << (u % 31));
                }
                if (!gather_units(D, R, ++seq, own, all, &wg_ok)) break;
                seen = all[seq & 1];
            }
        }
        for (int k = 0; k < R.slot_words; k++) crossed |= (seen[k] >> 31) != 0;
        for (int u = tid; u < n_units; u += blockDim.x) {
            if (!run[u]) continue;
            // (a workgroup ahead may already report crossings of this round)
            if (crossed && coherent_load(&D.units[u].infeasible) == step - 1)
                run[u] = 0;
            else if ((seen[u / 31] >> (u % 31)) & 1u)
                last[u] = step;
            else
                run[u] = 0;
        }
        __syncthreads();
    }
    if (blockIdx.x == 0)
        for (int u = tid; u < n_units; u += blockDim.x) D.units[u].changed[last[u] & 1] = last[u];
}

// The rounds of a batch as launches.  Before round `step`, one workgroup finds
// the instances that take part in it, notes the last rounds that moved a
// bound, and tells the host how far the run is.
__global__ __launch_bounds__(kMaxRoundUnits) void batch_plan_kernel(DevMatrix M, DevState D, RoundPlan R, int step) {
    __shared__ int run[kMaxRoundUnits], first[kMaxRoundUnits + 1], upto[kMaxRoundUnits];
    const int u = threadIdx.x;
    int in = 0;
    if (u < R.n_units) {
        first[u] = R.unit_item[u];
        if (u == R.n_units - 1) first[u + 1] = R.unit_item[u + 1];
        const UnitState &s = D.units[u];
        if (step == 1) {
            in = s.crossed == 0 && s.envelope == 0;
        } else if (R.run[u] && s.infeasible == 0) {
            for (int j = 0; j < kMoveLanes; j++) in |= D.moved[moved_index(u, (step - 1) & 1, j)] == step - 1;
            if (in) D.units[u].changed[(step - 1) & 1] = step - 1;
        }
        R.run[u] = in;
    }
    run[u] = in;
    __syncthreads();
    if (u < 64) run_totals(R.n_units, run, first, upto);
    __syncthreads();
    if (u < R.n_units) R.upto[u] = upto[u];
    if (u == 0)
        __hip_atomic_store(D.host_word, upto[R.n_units - 1] > 0 ? step : kRoundsOver, __ATOMIC_RELAXED,
                           __HIP_MEMORY_SCOPE_SYSTEM);
}

// Round `step` of a batch; bounds as in batch_rounds_kernel, the kernel
// boundaries in the barrier's place.  64 instances of 42,000 entries: 16 us a
// round with its plan (three phases: 42).
template <bool kTest>
__global__ __launch_bounds__(kTest ? 512 : 256) __attribute__((amdgpu_waves_per_eu(kTest ? 4 : 5))) void batch_round_kernel(
    DevMatrix M, DevState D, RoundPlan R, int step) {
    __shared__ int run[kMaxRoundUnits], first[kMaxRoundUnits + 1], upto[kMaxRoundUnits];
    __shared__ unsigned moved_units[kMaxRoundUnits / 32];
    const int tid = threadIdx.x;
    const int n_units = R.n_units;
    const int total = R.upto[n_units - 1];
    if (total == 0) return;
    if (tid < kMaxRoundUnits) {
        run[tid] = tid < n_units ? R.run[tid] : 0;
        upto[tid] = tid < n_units ? R.upto[tid] : total;
    }
    if (tid < n_units) first[tid + 1] = R.unit_item[tid + 1];
    if (tid < kMaxRoundUnits / 32) moved_units[tid] = 0u;
    const MovedBits B = load_moved_bits<kWide, kTest>(M, R, step, total, dyn_lds);
    const int waves = blockDim.x >> 6;
    const int wave = uniform(blockIdx.x * waves + (tid >> 6));
    const int nwaves = gridDim.x * waves;
    int *st = status_row(D, step);
    const DevState V = round_view(M, D, R, step);
    if (step > 1) carry_moved<true, kTest>(M, D, R, step, wave, nwaves, run);
    for (int t = wave; t < total; t += nwaves) {
        const int u = run_unit(n_units, upto, t);
        const int it = uniform(first[u + 1] - upto[u]) + t;
        const int moved = round_item<kWide, kTest>(M, V, R, it, step, st, B);
        if (__any(moved != 0) && (tid & 63) == 0) atomicOr(&moved_units[u >> 5], 1u << (u & 31));
    }
    __syncthreads();
    if (tid < n_units && ((moved_units[tid >> 5] >> (tid & 31)) & 1u)) note_round_moved(D, step, tid);
}

// The candidates of the batch's split rows whose gate passed in the round.
__global__ __launch_bounds__(256) void batch_apply_kernel(DevMatrix M, DevState D, RoundPlan R, int step) {
    const int count = coherent_load(&status_row(D, step)[kStatusApply]);
    const DevState V = round_view(M, D, R, step);
    for (int t = blockIdx.x * 4 + (threadIdx.x >> 6); t < count; t += gridDim.x * 4) {
        const int task = uniform(coherent_load(&D.apply_tasks[t]));
        int u;
        const int moved = apply_split_task<kWide>(M, V, task, u);
        if (__any(moved != 0) && (threadIdx.x & 63) == 0)
            note_round_moved(D, step, M.seg_rows[M.part_row[task]].w);
    }
}

template __global__ void round_kernel<false>(DevMatrix, DevState, RoundPlan, int);
template __global__ void round_kernel<true>(DevMatrix, DevState, RoundPlan, int);
template __global__ void rounds_kernel<false>(DevMatrix, DevState, RoundPlan);
template __global__ void rounds_kernel<true>(DevMatrix, DevState, RoundPlan);
template __global__ void batch_round_kernel<false>(DevMatrix, DevState, RoundPlan, int);
template __global__ void batch_round_kernel<true>(DevMatrix, DevState, RoundPlan, int);
template __global__ void batch_rounds_kernel<false>(DevMatrix, DevState, RoundPlan);
template __global__ void batch_rounds_kernel<true>(DevMatrix, DevState, RoundPlan);

// Writes the final bounds of a batch to the caller's vectors (not when some
// input was outside its envelope or a wait failed), finds crossed bounds of the instances' last
// rounds, and the last workgroup to finish writes the outcomes to pinned host
// memory.
__global__ __launch_bounds__(256) void unpack_batch_rounds_kernel(DevMatrix M, DevState D, RoundPlan R) {
    if (D.global[kGlobalEnvelope] == 0 && D.global[kGlobalError] == 0) {
        const DevState A = block_view(M, D, R, 0), B = block_view(M, D, R, 1);
        const int stride = gridDim.x * blockDim.x;
        for (int id = blockIdx.x * blockDim.x + threadIdx.x; id < M.n; id += stride) {
            const int j = M.perm[id];
            if (j < 0) continue;
            const int unit = M.word_unit[id >> 5];
            const int c0 = D.units[unit].changed[0], c1 = D.units[unit].changed[1];
            const int last = c0 > c1 ? c0 : c1;
            const bool odd = last & 1;
            double l, u;
            if (id < M.n_int) {
                const int2 a = odd ? B.AI[id] : A.AI[id];
                l = static_cast<double>(a.x);
                u = static_cast<double>(a.y);
                if (a.x == kAiHigh || a.y == kAiLow) {
                    const double2 x = odd ? B.AX[id] : A.AX[id];
                    l = x.x > l ? x.x : l;
                    u = x.y < u ? x.y : u;
                }
            } else {
                const double2 a = odd ? B.AF[id - M.n_int] : A.AF[id - M.n_int];
                l = a.x;
                u = a.y;
            }
            if (last > 0 && eps_gt(l, u)) atomic_max_i(&D.units[unit].infeasible, last);
            R.lbs[j] = l;
            R.ubs[j] = u;
        }
    }
    __shared__ int final_wg;
    mem_wait();
    __syncthreads();
    if (threadIdx.x == 0)
        final_wg = atomic_add_i(&D.global[kGlobalTicket], 1) == static_cast<int>(gridDim.x) - 1;
    __syncthreads();
    if (!final_wg) return;
    for (int u = threadIdx.x; u < R.n_units; u += blockDim.x) {
        UnitState s = D.units[u];
        s.infeasible = coherent_load(&D.units[u].infeasible);
        s.error = coherent_load(&D.global[kGlobalError]);
        R.host_state[u] = s;
    }
}

// Writes the final bounds to the caller's vectors (not when the input was
// outside the envelope or a wait failed), finds crossed bounds of the last round, and the last
// workgroup to finish writes the outcome to pinned host memory.
__global__ __launch_bounds__(256) void unpack_rounds_kernel(DevMatrix M, DevState D, RoundPlan R) {
    const long long *p = reinterpret_cast<const long long *>(&D.units[0]);
    const int infeasible = static_cast<int>(coherent_load(p) >> 32);
    const long long w2 = coherent_load(p + 2);
    const int error = coherent_load(&D.global[kGlobalError]);
    // the last round that moved a bound
    const int lane = threadIdx.x & 63;
    int last = lane < 2 * kMoveLanes ? coherent_load(&D.moved[moved_index(0, lane & 1, lane >> 1)]) : 0;
#pragma unroll
    for (int h = 1; h < 64; h <<= 1) {
        const int o = __shfl_xor(last, h, 64);
        last = o > last ? o : last;
    }
    last = uniform(infeasible ? infeasible : last);
    const DevState V = block_view(M, D, R, last & 1);
    if ((w2 >> 32) == 0 && error == 0) {
        const int stride = gridDim.x * blockDim.x;
        bool crossed = false;
        for (int id = blockIdx.x * blockDim.x + threadIdx.x; id < M.n; id += stride) {
            const int j = M.perm[id];
            double l, u;
            if (id < M.n_int) {
                const int2 a = V.AI[id];
                l = static_cast<double>(a.x);
                u = static_cast<double>(a.y);
                if (a.x == kAiHigh || a.y == kAiLow) {
                    const double2 x = V.AX[id];
                    l = x.x > l ? x.x : l;
                    u = x.y < u ? x.y : u;
                }
            } else {
                const double2 a = V.AF[id - M.n_int];
                l = a.x;
                u = a.y;
            }
            crossed |= eps_gt(l, u);
            R.lbs[j] = l;
            R.ubs[j] = u;
        }
        if (last > 0 && __any(crossed) && (threadIdx.x & 63) == 0) atomic_max_i(&D.units[0].infeasible, last);
    }
    mem_wait();
    __syncthreads();
    if (threadIdx.x == 0 &&
        atomic_add_i(&D.global[kGlobalTicket], 1) == static_cast<int>(gridDim.x) - 1) {
        UnitState s = D.units[0];
        s.infeasible = coherent_load(&D.units[0].infeasible);
        s.changed[last & 1] = last;
        s.error = coherent_load(&D.global[kGlobalError]);
        *R.host_state = s;
    }
}

// ---------------------------------------------------------------------------
// loading and reading bound vectors
// ---------------------------------------------------------------------------

// Resets the state words of unit q.x (q as in unit_reset_kernel), by one wave.
__device__ __forceinline__ void reset_unit(const DevState &D, const int4 q, int start_step) {
    const int lane = threadIdx.x & 63;
    if (lane == 0) {
        UnitState s = {};
        s.start = start_step;
        s.markall = q.z ? start_step : 0;
        s.max_rounds = q.w;
        s.mark_limit = q.y;
        D.units[q.x] = s;
    }
    static_assert(kMoveSlots * kMoveLanes == 64 && 2 * kCountWords <= 64, "a lane per counter");
    D.moved[moved_index(q.x, lane / kMoveLanes, lane % kMoveLanes)] = 0;
    if (lane < 2 * kCountWords)
        D.wl_cnt[static_cast<size_t>(q.x) * 2 * kCountWords + lane] = 0ull;
}

__device__ __forceinline__ void clear_run_words(const DevState &D, int tid, int stride, int epoch, int fail) {
    if (tid == 0) D.persist[kPersistEpoch] = epoch;
    for (int k = tid; k < kStatusRows * kStatusWords; k += stride) D.status[k] = 0;
    for (int k = tid; k < kGlobalWords; k += stride) D.global[k] = k == kGlobalError ? fail : 0;
    for (int k = tid; k < kBarrierWords; k += stride) D.barrier[k] = 0u;
}

// unit_reset_kernel and the launch tables for a single vector, all from the
// arguments (no copy to the device): the listed unit and the vector's pointers.
__global__ __launch_bounds__(256) void reset_one_kernel(DevState D, int4 q, int start_step, int clear_status, int epoch, int fail, int *list,
                                                        double **lbp, double **ubp, double *lbs, double *ubs) {
    if (threadIdx.x < 64) reset_unit(D, q, start_step);
    if (threadIdx.x == 0) {
        list[0] = q.x;
        lbp[0] = lbs;
        ubp[0] = ubs;
    }
    if (clear_status) clear_run_words(D, threadIdx.x, blockDim.x, epoch, fail);
}

// The state words of the listed units and the error word, to pinned host
// memory.
__global__ __launch_bounds__(256) void report_kernel(DevState D, int n_list, const int *list, UnitState *out) {
    for (int k = blockIdx.x * blockDim.x + threadIdx.x; k < n_list; k += gridDim.x * blockDim.x) {
        UnitState s = D.units[list[k]];
        s.error = D.global[kGlobalError];
        out[k] = s;
    }
}

// Resets the state words of the listed units, params[k] = {unit, mark
// limit, all rows in round 1, round cap}: round 1 in `start_step`, every row
// processed in that step unless marks come from changed-column hints.  With
// `clear_status`, also clears the step-status ring, the global words (`fail`:
// the error word is set from the start) and the barrier and starts the marks'
// epoch.
__global__ void unit_reset_kernel(DevState D, int n_list, const int4 *params, int start_step, int clear_status,
                                  int epoch, int fail) {
    const int tid = blockIdx.x * blockDim.x + threadIdx.x;
    const int stride = gridDim.x * blockDim.x;
    for (int k = tid >> 6; k < n_list; k += stride >> 6) reset_unit(D, params[k], start_step);
    if (clear_status) clear_run_words(D, tid, stride, epoch, fail);
}

// The passes over all columns of many vectors (load, unpack).  Workgroup j of
// the ones with per_unit workgroups a vector: from 64 vectors on a vector's
// workgroups lie on one XCD (workgroups go round the 8 XCDs), because the
// storage classes are gathered from interleaved columns: every line of the
// caller's vectors is touched once per class, and only one L2 then reads or
// merges it.  Calls pass(k, b) for vector k, workgroup b of it.
template <typename Pass>
__device__ __forceinline__ void for_vectors(int n_vectors, int per_unit, const Pass &pass) {
    if (n_vectors >= kVectorsByXcd) {
        const int xcd = blockIdx.x & 7, on_xcd = (n_vectors - xcd + 7) / 8;
        for (int j = blockIdx.x >> 3; j < on_xcd * per_unit; j += gridDim.x >> 3)
            pass(j / per_unit * 8 + xcd, j % per_unit);
    } else {
        for (int j = blockIdx.x; j < n_vectors * per_unit; j += gridDim.x) pass(j / per_unit, j % per_unit);
    }
}

// Bits 0 .. 15 of x in the even bits.
__device__ __forceinline__ unsigned spread16(unsigned x) {
    x &= 0xffffu;
    x = (x | x << 8) & 0x00ff00ffu;
    x = (x | x << 4) & 0x0f0f0f0fu;
    x = (x | x << 2) & 0x33333333u;
    return (x | x << 1) & 0x55555555u;
}

// Loads the bound vectors of the listed units (caller's column order: unit
// k's bounds at lbp[k], ubp[k]; blocks mode: one concatenated vector) into
// snapshot and accumulator, clears their bitmaps and split-row counters, and
// flags crossed input bounds and bounds outside a column's storage class.
// With a reference (replicas), every unit notes the columns in which it
// differs from it and takes over its segment partials.
// The exact integer accumulators are clean unless some run of this state has
// used them, and row marks of earlier runs are of earlier epochs; `all` (a
// state that was another problem's before) sets both.
// Bound by the memory: 16 bytes read and 12 (int16 columns) or 32 (FP64)
// written per column.  A thread has four columns in flight.  256 vectors of
// 100,000 columns: 0.92 GB in 300 us (591 us with one column in flight, the
// vectors over all XCDs, marks and exact accumulators cleared each time).
__global__ __launch_bounds__(256) void load_kernel(DevMatrix M, DevState D, int n_list, const int *list,
                                                   const double *const *lbp, const double *const *ubp,
                                                   ReferenceView ref, int per_unit, int all) {
    const bool ax = all || D.persist[kPersistAx] != 0;
    const int lane = threadIdx.x & 63;
    // blocks mode: one pass over all columns
    for_vectors(M.replicas ? n_list : 1, per_unit, [&](int k, int b) {
        const int tid = b * 256 + static_cast<int>(threadIdx.x), stride = per_unit * 256;
        const int u = list[k];
        const DevState V = unit_view(M, D, u);
        const double *lbs = lbp[M.replicas ? k : 0];
        const double *ubs = ubp[M.replicas ? k : 0];
        for (int i0 = tid - lane; i0 < M.n; i0 += 4 * stride) {
            int col[4];
            double low[4], up[4];
#pragma unroll
            for (int q = 0; q < 4; q++) {
                const int id = i0 + q * stride + lane;
                col[q] = id < M.n ? M.perm[id] : -1;
            }
#pragma unroll
            for (int q = 0; q < 4; q++) {
                low[q] = up[q] = 0.0;
                if (col[q] >= 0) {
                    low[q] = lbs[col[q]];
                    up[q] = ubs[col[q]];
                }
            }
#pragma unroll
            for (int q = 0; q < 4; q++) {
                const int first = i0 + q * stride, id = first + lane;
                if (first >= M.n) break;
                const double l = low[q], uu = up[q];
                const int cu = M.replicas ? u : M.word_unit[(id < M.n ? id : first) >> 5];
                if (eps_gt(l, uu)) atomic_or_i(&D.units[cu].crossed, 1);
                if (ref.parts != nullptr) {
                    const bool differs =
                        id < M.n && (__double_as_longlong(l) != __double_as_longlong(ref.lbs[id]) ||
                                     __double_as_longlong(uu) != __double_as_longlong(ref.ubs[id]));
                    const unsigned long long both = __ballot(differs);
                    if ((lane & 31) == 0 && id < M.n) {
                        const unsigned w = static_cast<unsigned>(lane ? both >> 32 : both);
                        ref.diff[static_cast<size_t>(k) * M.nwords + (id >> 5)] = w;
                        if (w) atomic_add_i(&ref.n_diff[k], 1);
                    }
                }
                if (first < M.n_bin) {
                    // 2-bit codes of the wave's binary columns, padding bits zero
                    const unsigned long long at1 = __ballot(id < M.n_bin && l >= 1.0);
                    const unsigned long long at0 = __ballot(id < M.n_bin && uu < 1.0);
                    if (lane < 4)
                        V.SB[first / 16 + lane] = spread16(static_cast<unsigned>(at1 >> (16 * lane))) |
                                                  spread16(static_cast<unsigned>(at0 >> (16 * lane))) << 1;
                }
                if (id >= M.n) continue;
                if (id < M.n_int) {
                    const double lim = id < M.n16 ? 32767.0 : 2147483647.0;
                    const double lo_lim = id < M.n_bin ? 0.0 : -lim, hi_lim = id < M.n_bin ? 1.0 : lim;
                    const bool fits = l >= lo_lim && l <= hi_lim && uu >= lo_lim && uu <= hi_lim && floor(l) == l &&
                                      floor(uu) == uu;
                    // crossed input bounds make the vector infeasible, whatever
                    // the column's storage class
                    if (!fits && !eps_gt(l, uu)) {
                        atomic_or_i(&D.units[cu].envelope, 1);
                        atomic_or_i(&D.global[kGlobalEnvelope], 1);
                    }
                    const int il = fits ? static_cast<int>(l) : 0, iu = fits ? static_cast<int>(uu) : 0;
                    V.AI[id] = make_int2(il, iu);
                    if (ax) V.AX[id] = make_double2(-INFINITY, INFINITY);
                    if (id < M.n16) V.S16[id] = pack16(il, iu);
                    else V.S32[id - M.n16] = make_int2(il, iu);
                } else {
                    V.AF[id - M.n_int] = make_double2(l, uu);
                    V.SF[id - M.n_int] = make_double2(l, uu);
                }
            }
        }
        if (tid == 0) V.SF[M.n - M.n_int] = make_double2(0.0, 0.0);  // the padding entries' column
        for (int w = tid; w < M.nwords; w += stride) V.bm[w] = 0u;
        for (int q = tid; q < M.n_seg_rows; q += stride) V.seg_count[q] = 0u;
        for (int q = tid; q < M.n_seg_parts; q += stride) {
            if (ref.parts != nullptr) {
                SegPart part = ref.parts[q];
                part.stamp = ref.start;
                V.seg_parts[q] = part;
            } else {
                V.seg_parts[q].stamp = 0;
            }
        }
        if (all) {
            for (int r = tid; r < M.m; r += stride) V.marks[r] = 0;
            for (int q = tid; q < M.n_seg_parts; q += stride) V.seg_marks[q] = 0;
        }
    });
}

// The exact integer accumulators of a new run state, of every unit.
__global__ __launch_bounds__(256) void clean_ax_kernel(DevState D, long long count) {
    for (long long i = blockIdx.x * 256LL + threadIdx.x; i < count; i += gridDim.x * 256LL)
        D.AX[i] = make_double2(-INFINITY, INFINITY);
}

// The bitwise majority of up to three vectors (the first one where all
// differ), column by column: a lower and an upper bound of one vector or of
// two, whichever.  Any mixture is a valid reference.
__device__ __forceinline__ double majority(double a, double b, double c) {
    const long long x = __double_as_longlong(a), y = __double_as_longlong(b), z = __double_as_longlong(c);
    return x != y && y == z ? b : a;
}

// The reference vector (by internal id) and its snapshot block (records as
// load_kernel writes them).  Values outside a column's class leave a wrong record: a unit with
// the same value there is refused, one with another drops the segment.
__global__ __launch_bounds__(256) void load_reference_kernel(DevMatrix M, DevState V, ReferenceVectors R, double *lbs,
                                                             double *ubs) {
    for (int id = blockIdx.x * blockDim.x + threadIdx.x; id < M.n; id += gridDim.x * blockDim.x) {
        const int j = M.perm[id];
        double l = R.lb[0][j], u = R.ub[0][j];
        if (R.n == 3) {
            l = majority(l, R.lb[1][j], R.lb[2][j]);
            u = majority(u, R.ub[1][j], R.ub[2][j]);
        }
        lbs[id] = l;
        ubs[id] = u;
        if (id < M.n_int) {
            const bool fits = fits_int32(l) && fits_int32(u);
            const int il = fits ? static_cast<int>(l) : 0, iu = fits ? static_cast<int>(u) : 0;
            if (id < M.n16) V.S16[id] = pack16(il, iu);
            else V.S32[id - M.n16] = make_int2(il, iu);
        } else {
            V.SF[id - M.n_int] = make_double2(l, u);
        }
    }
    if (blockIdx.x == 0 && threadIdx.x == 0) V.SF[M.n - M.n_int] = make_double2(0.0, 0.0);
}

// The segment partials of a reference vector, one wave per segment.
__global__ __launch_bounds__(256) void reference_parts_kernel(DevMatrix M, DevState V_arg, SegPart *parts) {
    constexpr int K = kSegLen / 64;
    DevState V = V_arg;
    V.n_lds = 0;
    const int lane = threadIdx.x & 63;
    const int waves = gridDim.x * (blockDim.x >> 6);
    for (int q = uniform(blockIdx.x * (blockDim.x >> 6) + (threadIdx.x >> 6)); q < M.n_seg_parts; q += waves) {
        const int4 info = M.seg_rows[M.part_row[q]];
        int start, len;
        row_extent(M, info.x, start, len);
        const int s0 = (q - info.y) * kSegLen;
        LaneEntries<K, kRecords> E;
        E.load(M, V, start + s0, lane * K, len - s0);
        E.template reduce<true>(64);
        if (lane == 0) {
            SegPart p;
            p.smin = E.tmin;
            p.smax = E.tmax;
            p.dmax = E.dmax;
            p.infs = E.infs;
            p.stamp = 0;
            parts[q] = p;
        }
    }
}

// Drops the copied partials of the segments that hold a column in which the
// unit differs from the reference; all of them where so many words differ
// that walking the columns would cost more than the segments.  A wave looks
// at 64 words, and its lanes take the entries of a differing column.
__global__ __launch_bounds__(256) void drop_parts_kernel(DevMatrix M, DevState D, int n_list, const int *list,
                                                         ReferenceView ref, int limit) {
    const int lane = threadIdx.x & 63;
    const int waves = gridDim.x * (blockDim.x >> 6);
    const int wave = uniform(blockIdx.x * (blockDim.x >> 6) + (threadIdx.x >> 6));
    for (int k = blockIdx.y; k < n_list; k += gridDim.y) {
        const DevState V = unit_view(M, D, uniform(list[k]));
        if (ref.n_diff[k] > limit) {
            for (int q = wave * 64 + lane; q < M.n_seg_parts; q += waves * 64) V.seg_parts[q].stamp = 0;
            continue;
        }
        for (int w0 = wave * 64; w0 < M.nwords; w0 += waves * 64) {
            const int w = w0 + lane;
            const unsigned mine = w < M.nwords ? ref.diff[static_cast<size_t>(k) * M.nwords + w] : 0u;
            unsigned long long pending = __ballot(mine != 0u);
            while (pending) {
                const int t = __ffsll(static_cast<long long>(pending)) - 1;
                pending &= pending - 1;
                unsigned bits = static_cast<unsigned>(__shfl(static_cast<int>(mine), t, 64));
                while (bits) {
                    const int id = (w0 + t) * 32 + __ffs(static_cast<int>(bits)) - 1;
                    bits &= bits - 1;
                    for (int q = M.col_ptr[id] + lane; q < M.col_ptr[id + 1]; q += 64) {
                        const int part = M.col_seg[q];
                        if (part >= 0) V.seg_parts[part].stamp = 0;
                    }
                }
            }
        }
    }
}

// Computes the segment partials that hinted units do not have yet (no
// reference, or dropped): a step of marked rows recomputes only listed
// segments.  Those that the hints have listed are left to the first step: a
// dropped segment mostly is one, because it holds a column in which the unit
// differs.  Each wave looks at `chunk` segments of a unit; units that process
// every row in their first step compute theirs there.  256 vectors, 2784 segments:
// 160 us with the listed segments and four a wave, 17 without and 16 a wave.
__global__ __launch_bounds__(256) void fill_parts_kernel(DevMatrix M, DevState D_arg, int n_list, const int *list,
                                                         int start_step, int chunk) {
    DevState D = D_arg;
    D.n_lds = 0;
    const int lane = threadIdx.x & 63;
    // workgroups go round the 8 XCDs: a unit's keep to one, unit after unit, so
    // that an L2 holds the snapshots in work
    const int listed = static_cast<int>(mark_stamp(start_step, true) + static_cast<unsigned>(D.persist[kPersistEpoch]));
    const int wg_parts = (blockDim.x >> 6) * chunk;
    const int per_unit = (M.n_seg_parts + wg_parts - 1) / wg_parts;
    const int xcd = blockIdx.x & 7, on_xcd = (n_list - xcd + 7) / 8;
    for (int j = blockIdx.x >> 3; j < on_xcd * per_unit; j += gridDim.x >> 3) {
        const int k = j / per_unit * 8 + xcd;
        const int u = uniform(list[k]);
        if (coherent_load(&D.units[u].markall) == start_step) continue;
        const DevState V = unit_view(M, D, u);
        {
            const int p0 = uniform((j % per_unit) * wg_parts + (threadIdx.x >> 6) * chunk);
            const int p = p0 + lane;
            unsigned long long todo = __ballot(lane < chunk && p < M.n_seg_parts && V.seg_parts[p].stamp == 0 &&
                                               V.seg_marks[p] != listed);
            while (todo) {
                const int part = uniform(p0 + __ffsll(static_cast<long long>(todo)) - 1);
                todo &= todo - 1;
                const int4 info = M.seg_rows[M.part_row[part]];
                int start, len;
                row_extent(M, info.x, start, len);
                segment_partial<kRecords>(M, V, info.y, part - info.y, start, len, start_step);
            }
        }
    }
}

// Marks the rows of hinted columns (caller's column indices; unit k's hints
// at hints[hint_ptr[k] .. hint_ptr[k + 1])) for the listed units' first step:
// the bound vector differs from a propagated fixpoint only in these columns.
__global__ __launch_bounds__(256) void hint_kernel(DevMatrix M, DevState D, int n_list, const int *list,
                                                   const int *hint_ptr, const int *hints, const int *inv_perm,
                                                   int start_step) {
    // a wave per hinted column, its lanes over the column's entries
    const int lane = threadIdx.x & 63;
    const int waves = gridDim.x * (blockDim.x >> 6);
    const int wave = uniform(blockIdx.x * (blockDim.x >> 6) + (threadIdx.x >> 6));
    for (int k = blockIdx.y; k < n_list; k += gridDim.y) {
        const int u = uniform(list[k]);
        const DevState V = unit_view(M, D, u);
        for (int h = hint_ptr[k] + wave; h < hint_ptr[k + 1]; h += waves) {
            const int id = inv_perm[hints[h]];
            const int end = M.col_ptr[id + 1];
            for (int q0 = M.col_ptr[id]; q0 < end; q0 += 64) {
                const int q = q0 + lane;
                const bool in[1] = {q < end};
                const int row[1] = {in[0] ? M.col_rows[q] : 0};
                const int code[1] = {in[0] ? M.col_seg[q] : -1};
                mark_entries<true>(M, V, u, in, row, code, start_step);
            }
        }
    }
}

// Writes the accumulated bounds of the listed units back to the caller's
// column order.  Nothing when a wait of the run failed or, with `checked`, a
// loaded vector left the envelope: the run is an error and leaves the vectors
// alone.  256 vectors of
// 100,000 columns: 174 us (336 with one column in flight, over all XCDs and
// with the exact accumulators read for every column).
// With kDiff (a server's finished requests) it also lists the columns in which
// a vector differs, bit for bit, from the one at L.lb[k], L.ub[k] (null: not
// asked for): the differing lanes of a wave take their places from one atomic.
// A pass of its own over vectors and bases took three times the unpack.
template <bool kDiff>
__global__ __launch_bounds__(256) void unpack_kernel(DevMatrix M, DevState D, int n_list, const int *list,
                                                     double *const *lbp, double *const *ubp, int per_unit,
                                                     int checked, ChangeLists L) {
    if (D.global[kGlobalError] != 0 || (checked && D.global[kGlobalEnvelope] != 0)) return;
    // blocks mode: one pass over all columns
    for_vectors(M.replicas ? n_list : 1, per_unit, [&](int k, int b) {
        const int tid = b * 256 + static_cast<int>(threadIdx.x), stride = per_unit * 256;
        const DevState V = unit_view(M, D, list[k]);
        double *lbs = lbp[M.replicas ? k : 0];
        double *ubs = ubp[M.replicas ? k : 0];
        const int lane = static_cast<int>(threadIdx.x & 63);
        const double *base_l = nullptr, *base_u = nullptr;
        if constexpr (kDiff) {
            base_l = L.lb[k];
            base_u = L.ub[k];
        }
        for (int w0 = tid - lane; w0 < M.n; w0 += 4 * stride) {
            const int i0 = w0 + lane;
            int col[4];
            int2 ai[4];
            double2 af[4];
#pragma unroll
            for (int q = 0; q < 4; q++) {
                const int id = i0 + q * stride;
                col[q] = id < M.n ? M.perm[id] : -1;
                if (id < M.n_int) ai[q] = V.AI[id];
                else if (id < M.n) af[q] = V.AF[id - M.n_int];
            }
#pragma unroll
            for (int q = 0; q < 4; q++) {
                const int id = i0 + q * stride;
                if (!kDiff && col[q] < 0) continue;
                double l = 0.0, u = 0.0;
                if (col[q] < 0) {
                } else if (id < M.n_int) {
                    l = static_cast<double>(ai[q].x);
                    u = static_cast<double>(ai[q].y);
                    if (ai[q].x == kAiHigh || ai[q].y == kAiLow) {
                        const double2 x = V.AX[id];
                        l = x.x > l ? x.x : l;
                        u = x.y < u ? x.y : u;
                    }
                } else {
                    l = af[q].x;
                    u = af[q].y;
                }
                if (col[q] >= 0) {
                    lbs[col[q]] = l;
                    ubs[col[q]] = u;
                }
                if constexpr (kDiff) {
                    if (base_l == nullptr) continue;
                    const bool differs = col[q] >= 0 &&
                                         (__double_as_longlong(l) != __double_as_longlong(base_l[col[q]]) ||
                                          __double_as_longlong(u) != __double_as_longlong(base_u[col[q]]));
                    const unsigned long long all = __ballot(differs);
                    if (all == 0ull) continue;
                    int at = 0;
                    if (lane == 0) at = atomic_add_i(&L.cnt[k], __popcll(all));
                    at = __shfl(at, 0, 64) + __popcll(all & ((1ull << lane) - 1ull));
                    if (differs && at < L.cap) {
                        const size_t to = static_cast<size_t>(k) * L.cap + at;
                        L.cols[to] = col[q];
                        L.vl[to] = l;
                        L.vu[to] = u;
                    }
                }
            }
        }
    });
}

template __global__ void unpack_kernel<false>(DevMatrix, DevState, int, const int *, double *const *, double *const *,
                                              int, int, ChangeLists);
template __global__ void unpack_kernel<true>(DevMatrix, DevState, int, const int *, double *const *, double *const *,
                                             int, int, ChangeLists);

// Writes the changed columns of delta requests into their bound vectors:
// vector k gets lbs[cols[h]] = lv[h], ubs[cols[h]] = uv[h] for h in
// [ptr[k], ptr[k + 1]) (caller's column order).
__global__ __launch_bounds__(256) void delta_kernel(int n_list, double *const *lbp, double *const *ubp,
                                                    const int *ptr, const int *cols, const double *lv,
                                                    const double *uv) {
    for (int k = blockIdx.y; k < n_list; k += gridDim.y)
        for (int h = ptr[k] + blockIdx.x * blockDim.x + threadIdx.x; h < ptr[k + 1]; h += gridDim.x * blockDim.x) {
            lbp[k][cols[h]] = lv[h];
            ubp[k][cols[h]] = uv[h];
        }
}

// Copies `count` bound-vector pairs of n2 doubles: ptrs[k] to ptrs[count + k]
// (16-byte accesses; n2 is even).  Grid: x over elements, y over pairs.
__global__ __launch_bounds__(256) void copy_pairs_kernel(long long n2, int count, double *const *ptrs) {
    const long long h = n2 / 2;
    for (int k = blockIdx.y; k < count; k += gridDim.y) {
        const double2 *src = reinterpret_cast<const double2 *>(ptrs[k]);
        double2 *dst = reinterpret_cast<double2 *>(ptrs[count + k]);
        for (long long i = blockIdx.x * static_cast<long long>(blockDim.x) + threadIdx.x; i < h;
             i += static_cast<long long>(gridDim.x) * blockDim.x)
            dst[i] = src[i];
    }
}

// Progress measure of one round (src/progressMeasureMethods/progress_function.h:45-116,
// :152-195): for every column the finite progress of its bounds between the
// weakest bounds (wl, wu) and the limit bounds (ll, lu), and the bounds that
// became finite since the previous round (pl, pu, then overwritten with this
// round's).  Bounds in the caller's column order.  Each workgroup writes the
// sums of its columns to fin_part / inf_part[blockIdx.x] in a fixed order.
__global__ __launch_bounds__(256) void measure_kernel(int n, const double *lb, const double *ub, const double *wl,
                                                      const double *wu, const double *ll, const double *lu,
                                                      double *pl, double *pu, double *fin_part, int *inf_part) {
    __shared__ double sf[4];
    __shared__ int si[4];
    double f = 0.0;
    int k = 0;
    for (int j = blockIdx.x * blockDim.x + threadIdx.x; j < n; j += gridDim.x * blockDim.x) {
        const double l = lb[j], u = ub[j], a = wl[j], b = wu[j], c = ll[j], d = lu[j];
        double v = 0.0;
        if (eps_gt(a, -kInf) && eps_gt(l, -kInf) && eps_ge(l, a) && !(fabs(c - a) <= kEps)) v += (l - a) / (c - a);
        if (eps_lt(b, kInf) && eps_lt(u, kInf) && eps_le(u, b) && !(fabs(b - d) <= kEps)) v += (b - u) / (b - d);
        f += v;
        k += (is_neg_inf(pl[j]) && eps_gt(l, -kInf)) ? 1 : 0;
        k += (is_pos_inf(pu[j]) && eps_lt(u, kInf)) ? 1 : 0;
        pl[j] = l;
        pu[j] = u;
    }
    for (int h = 32; h >= 1; h >>= 1) {
        f += shfl_xor_d(f, h);
        k += __shfl_xor(k, h, 64);
    }
    const int wave = threadIdx.x >> 6;
    if ((threadIdx.x & 63) == 0) {
        sf[wave] = f;
        si[wave] = k;
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        fin_part[blockIdx.x] = (sf[0] + sf[1]) + (sf[2] + sf[3]);
        inf_part[blockIdx.x] = si[0] + si[1] + si[2] + si[3];
    }
}

// Sums the workgroup partials of measure_kernel in index order into
// fin[0], inf[0] (one wave).
__global__ __launch_bounds__(64) void measure_total_kernel(int parts, const double *fin_part, const int *inf_part,
                                                           double *fin, int *inf) {
    double f = 0.0;
    int k = 0;
    for (int q = threadIdx.x; q < parts; q += 64) {
        f += fin_part[q];
        k += inf_part[q];
    }
    for (int h = 32; h >= 1; h >>= 1) {
        f += shfl_xor_d(f, h);
        k += __shfl_xor(k, h, 64);
    }
    if (threadIdx.x == 0) {
        fin[0] = f;
        inf[0] = k;
    }
}


// Packs the changed columns listed for nd vectors (vector k's cnt[k] entries
// at [k * cap, ...), none when cnt[k] > cap) into consecutive positions of
// pinned host memory: vector k's count into cnt_out[k], its start into off[k],
// the total into off[nd].  One workgroup per vector; each sums the counts
// before its own.
__global__ __launch_bounds__(256) void compact_changes_kernel(int nd, int cap, const int *cnt, const int *cols,
                                                              const double *vl, const double *vu, int *cnt_out, int *off,
                                                              int *kcols, double *kl, double *ku) {
    __shared__ int part[256];
    for (int k = blockIdx.x; k < nd; k += gridDim.x) {
        int sum = 0;
        for (int j = threadIdx.x; j < k; j += blockDim.x) {
            const int c = cnt[j];
            sum += c <= cap ? c : 0;
        }
        part[threadIdx.x] = sum;
        __syncthreads();
        for (int h = 128; h > 0; h >>= 1) {
            if (static_cast<int>(threadIdx.x) < h) part[threadIdx.x] += part[threadIdx.x + h];
            __syncthreads();
        }
        const int o = part[0];
        const int c = cnt[k] <= cap ? cnt[k] : 0;
        if (threadIdx.x == 0) {
            cnt_out[k] = cnt[k];
            off[k] = o;
            if (k == nd - 1) off[nd] = o + c;
        }
        const size_t src = static_cast<size_t>(k) * cap;
        for (int q = threadIdx.x; q < c; q += blockDim.x) {
            kcols[o + q] = cols[src + q];
            kl[o + q] = vl[src + q];
            ku[o + q] = vu[src + q];
        }
        __syncthreads();
    }
}

// ---------------------------------------------------------------------------
// problem layout on the device (single instance): the passes over the
// nonzeros.  The host orders the rows (tree-width bins), pads them and
// relabels the columns; these kernels move the entries.
// ---------------------------------------------------------------------------

// Row r of the layout takes the entries col_in / val_in [src_start[r],
// src_start[r] + len), len from the padded row starts row_ptr_out, of
// instance row_inst[r] (instance 0 when row_inst is null), whose columns are
// global columns inst_col_off[i] .. inst_col_off[i + 1] - 1.  Each entry goes
// to its padded place as (internal id | integer flag, coefficient) and counts
// one for its column in col_cnt (by internal id).  Padding entries are left
// as written before (zeros).  A column index outside the instance's range
// sets *bad and the entry is skipped.  One wave per row, grid-stride.
__global__ __launch_bounds__(256) void layout_rows_kernel(int mp, const long long *src_start, const int *row_inst,
                                                          const int *inst_col_off, const int *col_in,
                                                          const double *val_in, const int *row_ptr_out,
                                                          const int *internal, const int *vartype, int *col_out,
                                                          double *val_out, int *col_cnt, int *bad) {
    const int lane = threadIdx.x & 63;
    const int waves = gridDim.x * (blockDim.x >> 6);
    for (int r = blockIdx.x * (blockDim.x >> 6) + (threadIdx.x >> 6); r < mp; r += waves) {
        const long long k0 = src_start[r];
        const int a = row_ptr_out[r], b = row_ptr_out[r + 1];
        const int dst = a & ~(kRowAlign - 1);
        const int len = (b & ~(kRowAlign - 1)) - dst - (a & (kRowAlign - 1));
        const int inst = row_inst ? row_inst[r] : 0;
        const int base = inst_col_off[inst], lim = inst_col_off[inst + 1] - base;
        for (int e = lane; e < len; e += 64) {
            const int j = col_in[k0 + e];
            if (j < 0 || j >= lim) {
                atomic_or_i(bad, 1);
                continue;
            }
            const int g = base + j;
            const int id = internal[g];
            col_out[dst + e] = id | (vartype[g] == kVarContinuous ? 0 : kIntFlag);
            val_out[dst + e] = val_in[k0 + e];
            atomic_add_i(&col_cnt[id], 1);
        }
    }
}

// Column-to-row index: every entry of layout row r appends r to its column's
// list (fill[] starts at col_ptr[]) and, for split rows (row_part[r] >= 0),
// the entry's segment, else -1 - the row's class.  The order inside a
// column's list is not fixed; the lists are used as sets (marking).  One wave
// per row.
__device__ __forceinline__ int row_code(int len) {
    if (len > kSegLen) return -2;  // class 1
    const int log_width = len <= 1 ? 0 : 32 - __clz(len - 1);
    return -1 - (10 - log_width);
}

__global__ __launch_bounds__(256) void layout_csc_kernel(int mp, const int *row_ptr_out, const int *col_out,
                                                         const int *row_part, int *fill, int *col_rows,
                                                         int *col_seg) {
    const int lane = threadIdx.x & 63;
    const int waves = gridDim.x * (blockDim.x >> 6);
    for (int r = blockIdx.x * (blockDim.x >> 6) + (threadIdx.x >> 6); r < mp; r += waves) {
        const int a = row_ptr_out[r], b = row_ptr_out[r + 1];
        const int st = a & ~(kRowAlign - 1);
        const int len = (b & ~(kRowAlign - 1)) - st - (a & (kRowAlign - 1));
        const int part = row_part[r];
        for (int e = lane; e < len; e += 64) {
            const int id = col_out[st + e] & kIdMask;
            const int slot = atomic_add_i(&fill[id], 1);
            col_rows[slot] = r;
            col_seg[slot] = part >= 0 ? part + e / kSegLen : row_code(len);
        }
    }
}

// Rows of at most 64 entries (the tail of the layout: rows are ordered by
// decreasing tree width), 64 rows per wave.  Lane t holds the start, length,
// source position and instance of row r0 + t; the wave walks the padded
// entries of its rows 64 at a time, and each lane finds the row of its entry
// by a binary search over the starts the lanes hold.  The padding entries
// (zeroed beforehand) are skipped.  Same results as the kernels above.
struct ShortRows {
    int nrows, st, len, inst, S0, S1;
    long long k0;
};

__device__ __forceinline__ ShortRows short_rows(int r0, int mp, const int *row_ptr_out, const long long *src_start,
                                                const int *row_inst) {
    const int lane = threadIdx.x & 63;
    ShortRows R;
    R.nrows = min(64, mp - r0);
    const int r = r0 + min(lane, R.nrows - 1);
    const int a = row_ptr_out[r], b = row_ptr_out[r + 1];
    R.st = a & ~(kRowAlign - 1);
    R.len = (b & ~(kRowAlign - 1)) - R.st - (a & (kRowAlign - 1));
    R.k0 = src_start ? src_start[r] : 0;
    R.inst = row_inst ? row_inst[r] : 0;
    R.S0 = __shfl(R.st, 0, 64);
    R.S1 = __shfl(b & ~(kRowAlign - 1), R.nrows - 1, 64);
    return R;
}

// Lane of the row holding padded entry e (S0 <= e): the largest j < nrows
// with start_j <= e.  Every lane of the wave takes part.
__device__ __forceinline__ int short_row_of(const ShortRows &R, int e) {
    int lo = 0;
    for (int step = 32; step > 0; step >>= 1) {
        const int j = lo + step;
        const int sj = __shfl(R.st, j < R.nrows ? j : R.nrows - 1, 64);
        if (j < R.nrows && sj <= e) lo = j;
    }
    return lo;
}

__global__ __launch_bounds__(256) void layout_rows_short_kernel(int r_begin, int mp, const long long *src_start,
                                                                const int *row_inst, const int *inst_col_off,
                                                                const int *col_in, const double *val_in,
                                                                const int *row_ptr_out, const int *internal,
                                                                const int *vartype, int *col_out, double *val_out,
                                                                int *col_cnt, int *bad) {
    const int lane = threadIdx.x & 63;
    const int waves = gridDim.x * (blockDim.x >> 6);
    for (int r0 = r_begin + 64 * (blockIdx.x * (blockDim.x >> 6) + (threadIdx.x >> 6)); r0 < mp; r0 += 64 * waves) {
        const ShortRows R = short_rows(r0, mp, row_ptr_out, src_start, row_inst);
        for (int base = R.S0; base < R.S1; base += 64) {
            const int e = base + lane;
            const int j = short_row_of(R, e);
            const int rs = __shfl(R.st, j, 64), rl = __shfl(R.len, j, 64), inst = __shfl(R.inst, j, 64);
            const long long k0 = __shfl(R.k0, j, 64);
            const int k = e - rs;
            if (e >= R.S1 || k >= rl) continue;
            const int cbase = inst_col_off[inst], lim = inst_col_off[inst + 1] - cbase;
            const int c = col_in[k0 + k];
            if (c < 0 || c >= lim) {
                atomic_or_i(bad, 1);
                continue;
            }
            const int g = cbase + c;
            const int id = internal[g];
            col_out[e] = id | (vartype[g] == kVarContinuous ? 0 : kIntFlag);
            val_out[e] = val_in[k0 + k];
            atomic_add_i(&col_cnt[id], 1);
        }
    }
}

// Column-to-row index entries of the short rows (never split).
__global__ __launch_bounds__(256) void layout_csc_short_kernel(int r_begin, int mp, const int *row_ptr_out,
                                                               const int *col_out, int *fill, int *col_rows,
                                                               int *col_seg) {
    const int lane = threadIdx.x & 63;
    const int waves = gridDim.x * (blockDim.x >> 6);
    for (int r0 = r_begin + 64 * (blockIdx.x * (blockDim.x >> 6) + (threadIdx.x >> 6)); r0 < mp; r0 += 64 * waves) {
        const ShortRows R = short_rows(r0, mp, row_ptr_out, nullptr, nullptr);
        for (int base = R.S0; base < R.S1; base += 64) {
            const int e = base + lane;
            const int j = short_row_of(R, e);
            const int rs = __shfl(R.st, j, 64), rl = __shfl(R.len, j, 64);
            if (e >= R.S1 || e - rs >= rl) continue;
            const int id = col_out[e] & kIdMask;
            const int slot = atomic_add_i(&fill[id], 1);
            col_rows[slot] = r0 + j;
            col_seg[slot] = row_code(rl);
        }
    }
}

}  // namespace gdp
