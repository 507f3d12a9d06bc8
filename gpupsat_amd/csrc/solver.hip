// solver.hip -- CDCL on the device: one wavefront solves one job (an instance, or an
// instance plus a cube of assumed literals); a persistent grid pulls jobs from a
// device work queue until it is empty.
//
// Reference path restated in wave-parallel form (src/SATSolver/SATSolver.cu:67-218):
//   decide -> propagate -> on conflict analyse, learn, backjump -> restart.
// Strategy surfaces of the reference and where they live here:
//   BCPStrategy       (src/BCPStrategy/WatchedClausesList.cu:46-309): two watched literals,
//                     per-literal watch lists; a wave walks a list 64 entries at a time
//                     and finds units / conflicts with ballots.
//   ConflictAnalysis  (src/ConflictAnalysis/GraphAnalyzer.cu:31-138): 1-UIP over the trail
//                     (the reference's decision-scheme analysis is kept in the CPU oracle).
//   ClauseLearning    (src/ClauseLearning/LearntClausesManager.cu:16-41): learned clauses are
//                     appended to a per-job arena and watched; the DB is reduced at restarts.
//   DecisionStrategy  (src/DecisionStrategy/VSIDS.cu:77-140, src/SATSolver/DecisionMaker.cu:45-55):
//                     VSIDS with phase saving, or the reference's last-free-var/positive rule.
//   Restarts          (src/Restarts/GeometricRestartsManager.cu:3-31): geometric schedule.
//   JobsQueue         (src/SATSolver/JobsQueue.cu:10-32): atomic queue head; every cube of an
//                     instance must be refuted before the instance is UNSAT.
#include "common.hpp"
#include "gpsat_internal.hpp"
#include "solver.hpp"

namespace gpsat {

namespace {

__device__ __forceinline__ int32_t prefix_count(uint64_t m)
{
    return (int32_t)__builtin_amdgcn_mbcnt_hi((uint32_t)(m >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)m, 0u));
}

__device__ __forceinline__ int32_t popc64(uint64_t m) { return __builtin_popcountll(m); }
__device__ __forceinline__ int32_t ctz64(uint64_t m) { return __builtin_ctzll(m); }

__device__ __forceinline__ int32_t wave_inclusive_scan(int32_t x)
{
#pragma unroll
    for (int s = 1; s < 64; s <<= 1) {
        int32_t y = __shfl_up(x, s);
        if (lane_id() >= s) x += y;
    }
    return x;
}

// Max over the 64 lanes in every lane, by DPP and the permlane swaps as wave_or32 (a shuffle
// tree of 64-bit keys is 12 LDS round trips; this is none).
__device__ __forceinline__ uint32_t wave_max_u32(uint32_t x)
{
    x = max(x, (uint32_t)__builtin_amdgcn_update_dpp(0u, x, 0xB1, 0xF, 0xF, true));
    x = max(x, (uint32_t)__builtin_amdgcn_update_dpp(0u, x, 0x4E, 0xF, 0xF, true));
    x = max(x, (uint32_t)__builtin_amdgcn_update_dpp(0u, x, 0x124, 0xF, 0xF, true));
    x = max(x, (uint32_t)__builtin_amdgcn_update_dpp(0u, x, 0x128, 0xF, 0xF, true));
    const auto r = __builtin_amdgcn_permlane16_swap(x, x, false, false);
    x = max(r[0], r[1]);
    const auto q = __builtin_amdgcn_permlane32_swap(x, x, false, false);
    return max(q[0], q[1]);
}

__device__ __forceinline__ int32_t uni(int32_t x) { return __builtin_amdgcn_readfirstlane(x); }
__device__ __forceinline__ uint32_t uniu(uint32_t x) { return (uint32_t)__builtin_amdgcn_readfirstlane((int)x); }

// A 64-bit value of lane 0 in every lane.  Values that steer the search must reach it through
// readfirstlane: a shuffle's result counts as divergent, and one divergent exit of the search
// loop turns all of its scalar state and branches into vector registers and exec masks.
__device__ __forceinline__ uint64_t lane0_u64(uint64_t x)
{
    return (uint64_t)uniu((uint32_t)x) | (uint64_t)uniu((uint32_t)(x >> 32)) << 32;
}

__device__ __forceinline__ int32_t load_status(int32_t* p)
{
    return uni(__hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT));
}

template <class I> struct Vec;
template <> struct Vec<uint16_t> {
    typedef uint16_t x2 __attribute__((ext_vector_type(2)));
    typedef uint16_t x4 __attribute__((ext_vector_type(4)));
};
template <> struct Vec<uint32_t> {
    typedef uint32_t x2 __attribute__((ext_vector_type(2)));
    typedef uint32_t x4 __attribute__((ext_vector_type(4)));
};

// A literal's watch header: where its original-clause list starts and how long its two lists
// are, in one LDS read.  With 16-bit ids both lengths share a word (original low, learned
// high), so that one atomic add appends to either list.
template <class I> struct Hdr;
template <> struct Hdr<uint16_t> {
    typedef uint2 type;
    static __device__ __forceinline__ int32_t no(const type& h) { return (int32_t)(h.y & 0xffffu); }
    static __device__ __forceinline__ int32_t nl(const type& h) { return (int32_t)(h.y >> 16); }
    static __device__ __forceinline__ int32_t add_o(type* h) { return (int32_t)(atomicAdd(&h->y, 1u) & 0xffffu); }
    static __device__ __forceinline__ int32_t add_l(type* h) { return (int32_t)(atomicAdd(&h->y, 0x10000u) >> 16); }
    static __device__ __forceinline__ void sub_o(type* h) { atomicSub(&h->y, 1u); }
    static __device__ __forceinline__ void sub_l(type* h) { atomicSub(&h->y, 0x10000u); }
    static __device__ __forceinline__ void set(type* h, int32_t no, int32_t nl) { h->y = (uint32_t)no | (uint32_t)nl << 16; }
    static __device__ __forceinline__ void set_l0(type* h) { h->y &= 0xffffu; }
};
template <> struct Hdr<uint32_t> {
    struct type {
        uint32_t x, y, z;
    };
    static __device__ __forceinline__ int32_t no(const type& h) { return (int32_t)h.y; }
    static __device__ __forceinline__ int32_t nl(const type& h) { return (int32_t)h.z; }
    static __device__ __forceinline__ int32_t add_o(type* h) { return (int32_t)atomicAdd(&h->y, 1u); }
    static __device__ __forceinline__ int32_t add_l(type* h) { return (int32_t)atomicAdd(&h->z, 1u); }
    static __device__ __forceinline__ void sub_o(type* h) { atomicSub(&h->y, 1u); }
    static __device__ __forceinline__ void sub_l(type* h) { atomicSub(&h->z, 1u); }
    static __device__ __forceinline__ void set(type* h, int32_t no, int32_t nl)
    {
        h->y = (uint32_t)no;
        h->z = (uint32_t)nl;
    }
    static __device__ __forceinline__ void set_l0(type* h) { h->z = 0u; }
};

// One wavefront's search.  kMode: see k_solve.  I: the type of literal codes, clause ids,
// levels and positions.  ALL3: every original clause has three literals.
//
// The search is one long chain of dependent steps, run by one wavefront at a time at about 5
// cycles an instruction, 64 a trip to LDS, 20 a branch and 15-20 each time a scalar is made from
// vector lanes or used by them after a compare (measured on one wavefront).  Before this layout a
// propagated literal took 2,800 cycles in about 400 instructions, whether 1 or 8,192 wavefronts
// ran.  So:
//  * 16-bit ids, so that what a step reads is one record: a literal's header (list start and
//    both lengths), a clause's record (its watches and literals), a variable's level and
//    reason; the per-job state shrinks enough to hold the watch structures in LDS.  With 32-bit
//    ids (kShared: formulas whose watch structures are in HBM at any size) a wavefront keeps a
//    clause's two watches (or one unwatched literal of three) only and reads its literals from the
//    batch's arrays, which all wavefronts share: 16 bytes per 3-literal clause (20 in a mixed
//    formula) instead of the 52 of records and literals of its own, with which 8,192 wavefronts
//    had room for 0.42 M clauses instead of 0.7 M, and 1,024 cubes of 66,000 clauses over 2,000
//    variables took 73.7 ms instead of 46.6.
//  * both watch lists of a literal are walked in one pass of the wavefront, one entry per lane,
//    and the next literal's header and entries are fetched while the current one is processed
//    (a queued literal's negation is false, so nothing moves a watch to its lists meanwhile).
//  * what a lane decides is computed from value codes (false 0, unassigned 1, true 2) by vector
//    arithmetic; only a unit, a conflict or an open learned clause leaves the straight line.
//  * reductions run on DPP and ballots, not on LDS shuffles.
template <int kMode, class I, bool ALL3>
struct Search {
    typedef typename Vec<I>::x2 I2;
    typedef typename Vec<I>::x4 I4;
    typedef Hdr<I> H;
    typedef typename H::type HT;
    static constexpr bool kShared = sizeof(I) == 4;
    static constexpr I kNone = (I)~(I)0;
    static constexpr I kDrop = (I)((I)1 << (8 * sizeof(I) - 1));   // a literal dropped by minimization

    // instance (uniform)
    int32_t n, m, inst;
    // per-var / per-literal state
    HT* hdr;             // [2n]
    I4* vi;              // [n] of an assigned var: level, reason clause (kNone: a decision or a
                         // level-0 fact), trail index, nonzero at level 0 or while the analysis
                         // has the var in its clause
    float* act;          // [n]
    int32_t* lstamp;     // [n+2] level stamps for LBD
    I* trail;            // [n]
    I* tlim;             // [n+2] trail index where each level starts
    I* lbuf;             // [n+1] clause being learned
    uint8_t* lv;         // [2n+1] literal value: 0 false, 1 unassigned, 2 true; [2n] is always false
    int8_t* phase;       // [n]
    uint8_t* mark;       // [64] scratch of the analysis, zero between its steps
    // watch structures
    I* Wo;               // original-clause watch lists (capacity = occurrences)
    I4* rec;             // [m] ALL3: the three literals in order and the unwatched one; else the
                         // two watches, first literal / 4 in olits, length
    I2* wrec;            // [m] in its place with kShared: the two watches, or
    I* urec;             // [m] (ALL3) the unwatched literal
    I* Wl;               // learned-clause watch lists, slack slots per literal (index of the clause)
    I4* lrec;            // [learnt_cap] the two watches (kNone: detached), first literal / 8 in larena, length
    I* llbd;             // [learnt_cap]
    I* remap;            // [learnt_cap] scratch of reduce_db
    uint8_t* lused;      // [learnt_cap] used by an analysis since the last reduction
    I* olits;            // original literals (not ALL3), each clause filled up to a multiple of 4
                         // with the always-false literal
    const I* lits;       // kShared: the instance's literals and clause offsets in the batch
    const int32_t* coff;
    I* larena;           // learned literals, likewise to a multiple of 8
    int32_t slack, learnt_cap, larena_cap;
    // search state (uniform)
    int32_t dl, tsize, qhead;
    int32_t nlearnt, larena_used, larena_top;   // clauses held, their literals, next free literal / 8
    float inc;
    int32_t stamp;
    bool dups;               // some original clause names a variable twice
    bool shortl;             // no watch list can outgrow the wavefront
    int32_t base_trail;      // trail entries of the formula's unit clauses
    int32_t setup_inst;      // instance whose watch lists are built (-1: none)
    bool setup_ok;
    bool ran;                // the current job set up its instance (its per-var state is valid)
    int64_t conf_reported;   // conflicts of the current job already added to its instance pool
    uint64_t ph_t;           // telemetry: tick at which the current phase began
    int32_t ph_cur;          // telemetry: the current phase (Phase)
    unsigned long long* ph_out;  // telemetry: this job's JS_PH_* counters (null: off)
    int32_t* bumps;          // the instance's slice of var_bumps (null: off)
    int64_t conflicts, decisions, props, learned, restarts;
    int32_t levelmax;

    // Orders this wavefront's accesses across its lanes.  What one wavefront issues to an address,
    // loads, stores and atomics, takes effect there in the order it was issued, in LDS as in its HBM
    // slice (all go through one CU's path to memory; the wavefront scope of the memory model needs
    // no wait either), and no other wavefront touches the slice during a job.  So only the compiler
    // has to be held.  msync also waits for what is outstanding: the steps that rewrite whole arrays
    // (set-up, reductions, a new learned clause) use it, where it is not measurable; none needs it.
    static __device__ __forceinline__ void lsync() { wave_sync(); }
    static __device__ __forceinline__ void msync()
    {
        if (kMode != 1) __builtin_amdgcn_s_waitcnt(0);
        wave_sync();
    }
    static __device__ __forceinline__ bool lane0() { return lane_id() == 0; }

    // ---- layout: state part, watch part, learned literals (see solve_layout)
    __device__ __forceinline__ void carve(char* s, char* w, char* ar, const SolveArgs& a)
    {
        const SolveLayout& L = a.lay;
        hdr = (HT*)(s + L.hdr);
        vi = (I4*)(s + L.vi);
        act = (float*)(s + L.act);
        lstamp = (int32_t*)(s + L.lstamp);
        trail = (I*)(s + L.trail);
        tlim = (I*)(s + L.tlim);
        lbuf = (I*)(s + L.lbuf);
        lv = (uint8_t*)(s + L.lv);
        phase = (int8_t*)(s + L.phase);
        mark = (uint8_t*)(s + L.mark);
        rec = (I4*)(w + L.rec);
        wrec = (I2*)(w + L.rec);
        urec = (I*)(w + L.rec);
        lrec = (I4*)(w + L.lrec);
        Wo = (I*)(w + L.wo);
        Wl = (I*)(w + L.wl);
        llbd = (I*)(w + L.llbd);
        remap = (I*)(w + L.remap);
        lused = (uint8_t*)(w + L.lused);
        olits = (I*)(w + L.olits);
        larena = (I*)ar;
    }

    // Values of both literals of var v in one store (v's literals are adjacent bytes).
    __device__ __forceinline__ void set_value(int32_t u) { *(uint16_t*)(lv + (u & ~1)) = (u & 1) ? 0x0200u : 0x0002u; }
    __device__ __forceinline__ void clear_value(int32_t u) { *(uint16_t*)(lv + (u & ~1)) = 0x0101u; }

    // Uniform assignment of literal u with reason clause r.  One lane stores: 64 lanes storing the
    // same 1- or 2-byte value to one address are served one after another.
    __device__ __forceinline__ void assign(int32_t u, I r)
    {
        if (lane0()) {
            set_value(u);
            I4 x;
            x.x = (I)dl;
            x.y = r;
            x.z = (I)tsize;
            x.w = dl == 0 ? (I)1 : (I)0;
            vi[u >> 1] = x;
            trail[tsize] = (I)u;
        }
        tsize++;
        lsync();
    }

    __device__ __forceinline__ uint32_t value(int32_t u) const { return (uint32_t)lv[u]; }

    // Assigns the units of one step in lane order (mask um: lanes whose clause id is unit on
    // their literal u, all unassigned before the step).  A literal met again is skipped; the
    // complement of one assigned here is a conflict in that lane's clause.
    __device__ __forceinline__ void assign_units(uint64_t um, int32_t u, int32_t id, int32_t& confl)
    {
        int j = ctz64(um);
        int32_t x = readlane(u, j);
        assign(x, (I)readlane(id, j));
        um &= um - 1;
        uint64_t comp = 0;
        while (um) {
            um &= ~ballot(u == x);
            comp |= ballot(u == (x ^ 1));
            j = ctz64(um);
            if (um && ((comp >> j) & 1)) {
                confl = readlane(id, j);
                um = 0;
            }
            if (um) {
                x = readlane(u, j);
                assign(x, (I)readlane(id, j));
                um &= um - 1;
            }
        }
    }

    // The literals k .. k+3 of a clause of len literals at q; past its end, the false literals it
    // is filled up with (FILLED), or its last literal again.
    template <bool FILLED>
    static __device__ __forceinline__ I4 four(const I* q, int32_t k, int32_t len)
    {
        if constexpr (FILLED) return *(const I4*)(q + k);
        I4 y;
        y.x = q[k];
        y.y = q[min(k + 1, len - 1)];
        y.z = q[min(k + 2, len - 1)];
        y.w = q[min(k + 3, len - 1)];
        return y;
    }

    // The first literal of a clause (its literals at q) that is neither `other` nor false, kNone
    // if none: W literals per round trip.
    template <int W, bool FILLED>
    __device__ __forceinline__ uint32_t find_watch(const I* q, int32_t len, uint32_t other) const
    {
        uint32_t rep = kNone;
        for (int32_t k = 0; k < len && rep == (uint32_t)kNone; k += W) {
            uint32_t x[W], v[W];
#pragma unroll
            for (int t = 0; t < W; t += 4) {
                const I4 y = four<FILLED>(q, FILLED ? k + t : min(k + t, len - 1), len);
                x[t] = y.x;
                x[t + 1] = y.y;
                x[t + 2] = y.z;
                x[t + 3] = y.w;
            }
#pragma unroll
            for (int t = 0; t < W; t++) v[t] = lv[x[t]];
#pragma unroll
            for (int t = W - 1; t >= 0; t--) rep = min(v[t], x[t] ^ other) != 0u ? x[t] : rep;
        }
        return rep;
    }

    // Original clause e's record; its watches only (x and y) with kShared and not ALL3.
    __device__ __forceinline__ I4 record(uint32_t e) const
    {
        if constexpr (!kShared) return rec[e];
        I4 r = {};
        if constexpr (ALL3) {
            const I* q = lits + 3 * e;
            r.x = q[0];
            r.y = q[1];
            r.z = q[2];
            r.w = urec[e];
        } else {
            const I2 w = wrec[e];
            r.x = w.x;
            r.y = w.y;
        }
        return r;
    }

    __device__ __forceinline__ void set_unwatched(uint32_t e, uint32_t u)
    {
        if constexpr (kShared) urec[e] = (I)u;
        else rec[e].w = (I)u;
    }

    __device__ __forceinline__ void set_watches(uint32_t e, uint32_t x, uint32_t y)
    {
        I2 w;
        w.x = (I)x;
        w.y = (I)y;
        if constexpr (kShared) wrec[e] = w;
        else *(I2*)&rec[e] = w;
    }

    // Where the literals of original clause c with record r are (not ALL3).
    __device__ __forceinline__ const I* original_lits(uint32_t c, I4 r, int32_t& len) const
    {
        if constexpr (kShared) {
            const int32_t b = coff[c];
            len = coff[c + 1] - b;
            return lits + b;
        }
        len = (int32_t)r.w;
        return olits + 4 * (uint32_t)r.z;
    }

    // One step of an original-clause list of the false literal fl (start ws), 64 entries from i0,
    // of which lanes `in` hold one (e) and its record (r).  Moves watches, compacts the list in
    // place from `keep` on, assigns units in lane order and reports the first conflict.
    __device__ __forceinline__ void step_original(uint32_t fl, uint32_t ws, int32_t i0, int32_t& keep, bool in,
                                                  uint32_t e, I4 r, int32_t& confl)
    {
        uint32_t other, rep;
        bool open, move;
        if (ALL3) {
            // the unwatched literal is the only candidate
            rep = r.w;
            other = (uint32_t)r.x + r.y + r.z - fl - rep;
            open = in && confl < 0 && value(other) != 2;
            move = open && rep != other && value(rep) != 0;
        } else {
            other = (uint32_t)r.x + r.y - fl;
            open = in && confl < 0 && value(other) != 2;
            rep = kNone;
            if constexpr (kShared) {
                if (open) {
                    int32_t len;
                    const I* q = original_lits(e, r, len);
                    if (len > 2) rep = find_watch<4, false>(q, len, other);
                }
            } else if (open && r.w > 2) {
                rep = find_watch<4, true>(olits + 4 * (uint32_t)r.z, r.w, other);
            }
            move = rep != (uint32_t)kNone;
        }
        const bool no = open && !move && value(other) == 0, unit = open && !move && !no;
        const uint64_t mm = ballot(move);
        if (move) {
            const uint32_t at = (uint32_t)hdr[rep].x + H::add_o(&hdr[rep]);
            H::sub_o(&hdr[fl]);
            Wo[at] = (I)e;
            if (ALL3) {
                set_unwatched(e, fl);
            } else {
                set_watches(e, other, rep);
            }
        }
        const uint64_t km = ballot(in) & ~mm;
        if ((mm || keep != i0) && in && !move) Wo[ws + keep + prefix_count(km)] = (I)e;
        keep += popc64(km);
        lsync();
        const uint64_t cm = ballot(no), um = ballot(unit);
        if (cm) confl = readlane(e, ctz64(cm));
        else if (um) assign_units(um, other, e, confl);
    }

    // One step of a learned-clause list of fl (start base), as above; other, vo: the entry's
    // other watch and its value, read after the last assignment.  A clause with no room in its
    // new list is detached: it stops propagating, but may still be a reason.
    __device__ __forceinline__ void step_learned(uint32_t fl, uint32_t base, int32_t i0, int32_t& keep, bool in,
                                                 uint32_t e, I4 r, uint32_t other, uint32_t vo, int32_t& confl)
    {
        const bool active = in && confl < 0;
        const bool dead = active && r.x == kNone;
        const bool open = active && !dead && vo != 2;
        uint32_t rep = kNone;
        uint64_t om = ballot(open);
        if ((om & (om - 1)) == 0) {
            // one open clause: its literals across the lanes
            if (om) {
                const int j = ctz64(om);
                const I* q = larena + 8 * readlane(r.z, j);
                const int32_t len = readlane(r.w, j);
                const uint32_t oj = readlane(other, j);
                for (int32_t k = 0; om && k < len; k += kWave) {
                    const uint32_t x = q[min(k + (int32_t)lane_id(), len - 1)];
                    const uint64_t hit = ballot(min(value(x), x ^ oj) != 0u);
                    if (hit) {
                        const uint32_t f = readlane(x, ctz64(hit));
                        rep = lane_id() == j ? f : rep;
                        om = 0;
                    }
                }
            }
        } else if (open) {
            rep = find_watch<8, true>(larena + 8 * (uint32_t)r.z, r.w, other);
        }
        const bool move = rep != (uint32_t)kNone;
        const bool no = open && !move && vo == 0, unit = open && !move && vo != 0;
        const bool drop = move || dead;
        if (drop) H::sub_l(&hdr[fl]);
        if (move) {
            const int32_t pos = H::add_l(&hdr[rep]);
            I2 w;
            w.x = (I)other;
            w.y = (I)rep;
            if (pos < slack) {
                Wl[rep * slack + pos] = (I)e;
            } else {
                H::sub_l(&hdr[rep]);
                w.x = w.y = kNone;
            }
            *(I2*)&lrec[e] = w;
        }
        const uint64_t dm = ballot(drop), km = ballot(in) & ~dm;
        if ((dm || keep != i0) && in && !drop) Wl[base + keep + prefix_count(km)] = (I)e;
        keep += popc64(km);
        lsync();
        const uint64_t cm = ballot(no), um = ballot(unit);
        if (cm) confl = m + readlane(e, ctz64(cm));
        else if (um) assign_units(um, other, e + m, confl);
    }

    // A learned entry's other watch; a detached clause (and a lane without an entry) gives the
    // always-false literal, so that it counts as open.
    __device__ __forceinline__ uint32_t learned_other(I4 r, uint32_t fl) const
    {
        return min((uint32_t)r.x + r.y - fl, 2u * (uint32_t)n);
    }

    // Propagation for lists of any length: 64 entries per step.
    __device__ __forceinline__ int32_t propagate_long()
    {
        const uint32_t lane = lane_id();
        int32_t confl = -1;
        while (confl < 0 && qhead < tsize) {
            const uint32_t fl = uniu(trail[qhead]) ^ 1u;
            qhead++;
            props++;
            const HT h = hdr[fl];
            const uint32_t ws = uniu(h.x), lb = fl * (uint32_t)slack;
            const int32_t co = uni(H::no(h)), cl = uni(H::nl(h));
            int32_t keep = 0;
            for (int32_t i0 = 0; i0 < co; i0 += kWave) {
                const uint32_t e = Wo[ws + min(i0 + (int32_t)lane, co - 1)];
                step_original(fl, ws, i0, keep, i0 + (int32_t)lane < co, e, record(e), confl);
            }
            keep = 0;
            for (int32_t i0 = 0; i0 < cl; i0 += kWave) {
                const uint32_t e = Wl[lb + min(i0 + (int32_t)lane, cl - 1)];
                const I4 r = lrec[e];
                const uint32_t other = learned_other(r, fl);
                step_learned(fl, lb, i0, keep, i0 + (int32_t)lane < cl, e, r, other, value(other), confl);
            }
        }
        return confl;
    }

    // Keeps a wave-uniform value in a vector register: what is computed from it stays on the
    // vector side, where the loads that need it are.
    static __device__ __forceinline__ uint32_t vec(uint32_t x)
    {
        asm("" : "+v"(x));
        return x;
    }

    // This lane's entry of the list of k <= 64 at W[start] (lanes past it: any).  With kShared the
    // lists, in HBM, are read no further than they go.  (The place is one 32-bit sum: an offset from
    // a pointer to the list's start cost pigeonhole formulas in placement 2 2%.)
    static __device__ __forceinline__ uint32_t entry(const I* W, uint32_t start, int32_t k)
    {
        const uint32_t lane = lane_id();
        return W[start + (kShared ? min(lane, (uint32_t)max(k - 1, 0)) : lane)];
    }

    __device__ __forceinline__ int32_t propagate()
    {
        if (!shortl) return propagate_long();
        if (qhead >= tsize) return -1;
        const uint32_t lane = lane_id();
        const uint32_t top = 2u * (uint32_t)n;   // (a lane without an entry reads clause 0, which need not hold fl)
        int32_t confl = -1;
        // the current literal (its negation fl), its lists (ws, co original entries; lb, cl
        // learned) and their entries
        do {
            uint32_t fl = vec(trail[qhead]) ^ 1u;
            HT h = hdr[fl];
            uint32_t lb = fl * (uint32_t)slack;
            bool fetched;
            uint32_t eo = entry(Wo, h.x, H::no(h)), el = entry(Wl, lb, H::nl(h));
            for (;;) {
                qhead++;
                props++;
                const uint32_t ws = h.x;
                const bool ino = lane < (uint32_t)H::no(h), inl = lane < (uint32_t)H::nl(h);
                eo = ino ? eo : 0u;
                el = inl ? el : 0u;
                uint32_t fln = vec(trail[qhead]) ^ 1u;   // the next one, if one is queued
                const I4 ro = record(eo), rl = lrec[el];
                HT hn = hdr[fln];
                uint32_t lbn = fln * (uint32_t)slack;
                uint32_t other, rep, vo, vq = 0;
                if (ALL3) {
                    rep = ro.w;
                    other = min((uint32_t)ro.x + ro.y + ro.z - fl - rep, top);
                    vq = value(rep);
                    if (dups) vq = rep == other ? 0u : vq;
                } else {
                    other = min((uint32_t)ro.x + ro.y - fl, top);
                }
                vo = value(other);
                const uint32_t lother = learned_other(rl, fl);
                uint32_t vl = value(lother);
                uint32_t eon = entry(Wo, hn.x, H::no(hn)), eln = entry(Wl, lbn, H::nl(hn));
                vo = ino ? vo : 2u;
                vl = inl ? vl : 2u;
                // (decisions are single compares: a ballot of one goes straight to scalar
                // registers, a ballot of a conjunction takes two vector operations more)
                uint64_t ev;
                if (ALL3) {
                    const uint64_t mm = ballot((2u - vo) * vq != 0u);
                    if (mm) {
                        if ((mm >> lane) & 1) {
                            const uint32_t at = (uint32_t)hdr[rep].x + H::add_o(&hdr[rep]);
                            H::sub_o(&hdr[fl]);
                            Wo[at] = (I)eo;
                            set_unwatched(eo, fl);
                        } else if (ino) {
                            Wo[ws + lane - prefix_count(mm)] = (I)eo;
                        }
                        lsync();
                    }
                    // a unit or falsified clause (vo < 2, vq false), or a learned clause not satisfied
                    ev = ballot(min(vq | (vo & 2u), vl & 2u) == 0u);
                } else {
                    ev = ballot(min(vo, vl) < 2u);
                }
                int32_t queued = tsize;
                if (ev) {
                    if (ALL3) {
                        const uint64_t cm = ballot((vq | vo) == 0u), um = ballot((vq << 2 | vo) == 1u);
                        if (cm) confl = readlane(eo, ctz64(cm));
                        else if (um) assign_units(um, other, eo, confl);
                    } else if (ballot(vo < 2u)) {
                        int32_t keep = 0;
                        step_original(fl, ws, 0, keep, ino, eo, ro, confl);
                    }
                    if (confl < 0) {
                        if (tsize != queued) {
                            vl = value(lother);
                            vl = inl ? vl : 2u;
                            if (qhead >= queued) {
                                // the first of the new ones is next: fetch its lists meanwhile
                                fln = vec(trail[qhead]) ^ 1u;
                                hn = hdr[fln];
                                lbn = fln * (uint32_t)slack;
                                eon = entry(Wo, hn.x, H::no(hn));
                                eln = entry(Wl, lbn, H::nl(hn));
                                queued = tsize;
                            }
                        }
                        if (ballot(vl < 2u)) {
                            int32_t keep = 0;
                            step_learned(fl, lb, 0, keep, inl, el, rl, lother, vl, confl);
                        }
                    }
                }
                fetched = qhead < queued;
                if (confl >= 0 || !fetched) break;
                fl = fln;
                h = hn;
                lb = lbn;
                eo = eon;
                el = eln;
            }
        } while (confl < 0 && qhead < tsize);
        return confl;
    }

    __device__ __forceinline__ void backtrack(int32_t b, bool save_phase)
    {
        if (dl <= b) return;
        const int32_t start = uni((int32_t)tlim[b + 1]);
        for (int32_t t = start + lane_id(); t < tsize; t += kWave) {
            const int32_t u = trail[t];
            clear_value(u);
            if (save_phase) phase[u >> 1] = (int8_t)(u & 1);
        }
        lsync();
        tsize = start;
        qhead = start;
        dl = b;
    }

    __device__ __forceinline__ void bump_activity(int32_t v)
    {
        if (kMode == 4) act[v] += inc;
        else __hip_atomic_fetch_add(&act[v], inc, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WAVEFRONT);
        if (bumps) atomicAdd(&bumps[v], 1);
    }

    // Where the literals of clause c (uniform) are; ALL3 originals keep theirs in the record.
    __device__ __forceinline__ const I* clause_lits(int32_t c, int32_t& len) const
    {
        if (c < m) {
            if constexpr (kShared) {
                const int32_t b = uni(coff[c]);
                len = uni(coff[c + 1]) - b;
                return lits + b;
            }
            const I4 r = rec[c];
            len = uni((int32_t)r.w);
            return olits + 4 * uni((int32_t)r.z);
        }
        const I4 r = lrec[c - m];
        len = uni((int32_t)r.w);
        return larena + 8 * uni((int32_t)r.z);
    }

    // Whether every literal of reason clause r is in the clause being learned (as the literal it
    // is the reason of is) or a level-0 fact.
    __device__ __forceinline__ bool implied(int32_t r) const
    {
        if (ALL3 && r < m) {
            const I4 x = record(r);
            return min(min((uint32_t)vi[x.x >> 1].w, (uint32_t)vi[x.y >> 1].w), (uint32_t)vi[x.z >> 1].w) != 0u;
        }
        if (kShared && r < m) {
            int32_t len;
            const I* q = original_lits(r, I4{}, len);
            return all_in_clause<false>(q, len);
        }
        const I4 x = r < m ? rec[r] : lrec[r - m];
        return all_in_clause<true>(r < m ? olits + 4 * (int32_t)x.z : larena + 8 * (int32_t)x.z, x.w);
    }

    template <bool FILLED>
    __device__ __forceinline__ bool all_in_clause(const I* q, int32_t len) const
    {
        uint32_t all = 1;
        for (int32_t k = 0; k < len && all; k += 4) {
            const I4 y = four<FILLED>(q, k, len);
            const int32_t a = y.x >> 1, b = k + 1 < len ? y.y >> 1 : a, c = k + 2 < len ? y.z >> 1 : a,
                          d = k + 3 < len ? y.w >> 1 : a;
            all = min(min((uint32_t)vi[a].w, (uint32_t)vi[b].w), min((uint32_t)vi[c].w, (uint32_t)vi[d].w));
        }
        return all != 0u;
    }

    // Takes the literals q of lanes `take` (below the current level, not yet in it) into the
    // clause being learned, in lane order.
    __device__ __forceinline__ void take_lower(uint64_t take, int32_t q, int32_t& nl)
    {
        if ((take >> lane_id()) & 1) {
            vi[q >> 1].w = 1;
            bump_activity(q >> 1);
            lbuf[nl + prefix_count(take)] = (I)q;
        }
        nl += popc64(take);
        lsync();
    }

    // Of the lanes `m64`, the first of each variable (clauses that name one twice).
    __device__ __forceinline__ uint64_t first_of_var(uint64_t m64, int32_t v) const
    {
        uint64_t keep = 0;
        while (m64) {
            const int j = ctz64(m64);
            keep |= 1ull << j;
            m64 &= ~ballot(v == readlane(v, j));
        }
        return keep;
    }

    // The resolution steps of analyze() when the current level's part of the trail fits the
    // wavefront: lane i stands for trail entry tsize-1-i, a scalar mask holds the entries still to
    // resolve, and the current level's literals never touch memory flags.  Returns the clause's
    // length (-1: no literal of the current level, an internal error) and the asserting literal's
    // negation p.
    __device__ __forceinline__ int32_t resolve(int32_t confl, int32_t& p)
    {
        const int lane = lane_id();
        const uint32_t end = (uint32_t)tsize - 1u;
        const int32_t tl = trail[max((int32_t)end - lane, 0)];
        const int32_t rs = vi[tl >> 1].y;
        const uint32_t seg = (uint32_t)tsize - uniu(tlim[dl]);   // entries of the current level (<= 64)
        uint64_t todo = 0, ever = 0, past = 0;
        int32_t nl = 1, c = confl, j = 0;
        do {
            if (ALL3 && c < m) {
                const I4 r = record(c);
                const int32_t q = lane == 0 ? r.x : lane == 1 ? r.y : r.z;
                const I4 x = vi[q >> 1];
                const uint32_t ra = end - (uint32_t)vi[r.x >> 1].z, rb = end - (uint32_t)vi[r.y >> 1].z,
                               rc = end - (uint32_t)vi[r.z >> 1].z;
                todo |= ballot((uint32_t)lane == ra) | ballot((uint32_t)lane == rb) | ballot((uint32_t)lane == rc);
                // lanes past the clause, and those of the current level, are not lower
                const uint32_t in = min((uint32_t)(lane < 3 ? 1 : 0), end - (uint32_t)x.z < seg ? 0u : 1u);
                uint64_t low = ballot(((uint32_t)x.w ^ 1u) * in == 1u);
                if (low) {
                    if (dups) low = first_of_var(low, q >> 1);
                    take_lower(low, q, nl);
                }
            } else {
                int32_t len;
                const I* cl = clause_lits(c, len);
                if (c >= m && lane == 0) lused[c - m] = 1;
                for (int32_t k0 = 0; k0 < len; k0 += kWave) {
                    const int32_t k = k0 + lane;
                    // every lane reads (lanes past the clause re-read its last literal)
                    const int32_t q = cl[min(k, len - 1)];
                    const I4 x = vi[q >> 1];
                    const uint32_t rq = end - (uint32_t)x.z;
                    const bool cur = rq < seg;
                    if (cur) mark[rq] = 1;
                    uint64_t low = ballot(k < len && !cur && x.w == 0);
                    if (low) {
                        if (dups && c < m) low = first_of_var(low, q >> 1);
                        take_lower(low, q, nl);
                    }
                }
                lsync();
                todo |= ballot(mark[lane] != 0);
                mark[lane] = 0;
                lsync();
            }
            todo &= ~0ull >> (64u - seg);
            ever |= todo;
            todo &= ~past;
            j = ctz64(todo);
            past |= todo & (~todo + 1);
            past |= past - 1;
            todo &= todo - 1;
            c = readlane(rs, j);
        } while (todo);
        p = readlane(tl, j);
        if ((ever >> lane) & 1) bump_activity(tl >> 1);
        return ever ? nl : -1;
    }

    // The same for a current level of any length: flags on every literal met, the trail walked
    // back 64 entries at a time.
    __device__ __forceinline__ int32_t resolve_long(int32_t confl, int32_t& p)
    {
        const int lane = lane_id();
        int32_t nl = 1, pathc = 0, c = confl;
        int32_t wb = tsize - 1, off = 0;
        int32_t tl = trail[max(wb - lane, 0)];
        p = -1;
        do {
            int32_t len = 3;
            const I* cl = nullptr;
            I4 r3 = {};
            if (ALL3 && c < m) r3 = record(c);
            else cl = clause_lits(c, len);
            if (c >= m && lane == 0) lused[c - m] = 1;
            for (int32_t k0 = 0; k0 < len; k0 += kWave) {
                const int32_t k = k0 + lane;
                int32_t q;
                if (ALL3 && c < m) q = lane == 0 ? r3.x : lane == 1 ? r3.y : r3.z;
                else q = cl[min(k, len - 1)];
                const I4 x = vi[q >> 1];
                uint64_t met = ballot(k < len && q != p && x.w == 0);
                if (dups && c < m) met = first_of_var(met, q >> 1);
                const uint64_t low = met & ~ballot((int32_t)x.x == dl);
                if (((met & ~low) >> lane) & 1) {
                    vi[q >> 1].w = 1;
                    bump_activity(q >> 1);
                }
                pathc += popc64(met & ~low);
                take_lower(low, q, nl);
            }
            // the next literal met of the current level, walking back
            uint64_t hm = ballot(lane >= off && wb - lane >= 0 && vi[tl >> 1].w != 0);
            while (hm == 0 && wb >= kWave) {
                wb -= kWave;
                off = 0;
                tl = trail[max(wb - lane, 0)];
                hm = ballot(wb - lane >= 0 && vi[tl >> 1].w != 0);
            }
            const int j = hm ? ctz64(hm) : 0;
            off = j + 1;
            p = readlane(tl, j);
            c = uni((int32_t)vi[p >> 1].y);
            if (lane == 0) vi[p >> 1].w = 0;
            lsync();
            pathc--;
        } while (pathc > 0 && c != (int32_t)kNone);
        return pathc > 0 ? -1 : nl;
    }

    // 1-UIP.  Leaves the learned clause in lbuf[0..len) with the asserting literal first and
    // a literal of the backjump level second.
    __device__ __forceinline__ int32_t analyze(int32_t confl, int32_t& bt, int32_t& lbd)
    {
        const int lane = lane_id();
        int32_t p;
        int32_t nl = tsize - uni((int32_t)tlim[dl]) <= kWave ? resolve(confl, p) : resolve_long(confl, p);
        if (lane == 0) lbuf[0] = (I)(p ^ 1);
        lsync();
        // Local minimization: a literal whose reason's other literals are all in the clause (or at
        // level 0) is implied by the rest and dropped.  First every literal is tested against the
        // clause as learned (drops are marked, the vars' flags untouched), then the clause is
        // compacted, so the result does not depend on lane order.  Dropping several at once is
        // sound: resolving them out in reverse trail order only meets literals that stay in the
        // clause or are resolved out earlier.
        for (int32_t k = 1 + lane; k < nl; k += kWave) {
            const int32_t q = lbuf[k];
            const int32_t r = vi[q >> 1].y;
            if (r != (int32_t)kNone && implied(r)) lbuf[k] = (I)(q | kDrop);
        }
        lsync();
        // compaction, the vars' flags, backjump level = highest level among the other literals (the
        // first literal of that level), LBD = distinct levels
        stamp++;
        int32_t kept = 1, distinct = 0, best = -1, bi = 0;
        for (int32_t k0 = 1; k0 < nl; k0 += kWave) {
            const int32_t k = k0 + lane;
            const bool in = k < nl;
            const int32_t x = lbuf[min(k, nl - 1)];
            const int32_t q = x & (int32_t)(I)~kDrop;
            const int32_t lvl = vi[q >> 1].x;
            if (in) vi[q >> 1].w = 0;
            const bool keep = in && !(x & (int32_t)kDrop);
            const uint64_t km = ballot(keep);
            bool first = false;
            if (keep) first = atomicExch(&lstamp[lvl], stamp) != stamp;
            lsync();
            if (keep) lbuf[kept + prefix_count(km)] = (I)q;
            distinct += popc64(ballot(first));
            if (km) {
                const int32_t top = (int32_t)uniu(wave_max_u32(keep ? (uint32_t)lvl + 1u : 0u)) - 1;
                if (top > best) {
                    best = top;
                    bi = kept + popc64(km & ((1ull << ctz64(ballot(keep && lvl == top))) - 1ull));
                }
            }
            kept += popc64(km);
            lsync();
        }
        nl = kept;
        lbd = distinct + 1;
        bt = 0;
        if (nl > 1) {
            bt = best;
            const I t1 = lbuf[1], tb = lbuf[bi];
            lsync();
            if (lane0()) {
                lbuf[1] = tb;
                lbuf[bi] = t1;
            }
        }
        lsync();
        return nl;
    }

    __device__ __forceinline__ bool room(int32_t len) const
    {
        return nlearnt < learnt_cap && larena_used + len <= larena_cap;
    }

    // Append lbuf[0..len) as a learned clause, not yet watched.  Returns its index.
    __device__ __forceinline__ int32_t store_learned(int32_t len, int32_t lbd)
    {
        const int32_t id = nlearnt;
        const int32_t full = (len + 7) & ~7;
        for (int32_t k = lane_id(); k < full; k += kWave)
            larena[8 * larena_top + k] = k < len ? lbuf[k] : (I)(2 * n);
        if (lane0()) {
            I4 r;
            r.x = r.y = kNone;
            r.z = (I)larena_top;
            r.w = (I)len;
            lrec[id] = r;
            llbd[id] = (I)lbd;
            lused[id] = 0;
        }
        nlearnt++;
        larena_used += len;
        larena_top += full >> 3;
        learned++;
        msync();
        return id;
    }

    // Watch learned clause i on literals x and y (uniform); without room in both lists it stays
    // detached.
    __device__ __forceinline__ void watch_learned(int32_t i, int32_t x, int32_t y)
    {
        const HT hx = hdr[x], hy = hdr[y];
        const int32_t px = uni(H::nl(hx)), py = uni(H::nl(hy)) + (x == y ? 1 : 0);
        if (px < slack && py < slack) {
            if (lane0()) {
                I2 w;
                w.x = (I)x;
                w.y = (I)y;
                *(I2*)&lrec[i] = w;
                Wl[x * slack + px] = (I)i;
                Wl[y * slack + py] = (I)i;
                (void)H::add_l(&hdr[x]);
                (void)H::add_l(&hdr[y]);
            }
        }
        lsync();
    }

    // At level 0: attach learned clause i.  A clause satisfied at level 0 is dropped, a clause
    // with one non-false literal asserts it, a falsified clause means the job is UNSAT (returns
    // false).
    __device__ __forceinline__ bool attach_level0(int32_t i)
    {
        const int lane = lane_id();
        const I4 r = lrec[i];
        const int32_t st = 8 * uni((int32_t)r.z), len = uni((int32_t)r.w);
        int32_t nf0 = -1, nf1 = -1;
        bool sat = false;
        for (int32_t k0 = 0; k0 < len && nf1 < 0 && !sat; k0 += kWave) {
            const int32_t k = k0 + lane;
            const int32_t q = larena[st + min(k, len - 1)];
            const uint32_t v = k < len ? value(q) : 0u;
            if (ballot(v == 2)) sat = true;
            uint64_t um = ballot(v == 1);
            while (um && nf1 < 0) {
                const int j = ctz64(um);
                um &= um - 1;
                const int32_t x = uni(readlane(q, j));
                if (nf0 < 0) nf0 = x;
                else nf1 = x;
            }
        }
        bool ok = true;
        if (!sat) {
            if (nf0 < 0) ok = false;
            else if (nf1 < 0) assign(nf0, kNone);
            else watch_learned(i, nf0, nf1);
        }
        msync();
        return ok;
    }

    // Reduce the learned DB at the current level.  Survivors: reasons of assigned literals
    // (always), glue clauses (LBD <= 3) and, in mode 0, clauses used since the last
    // reduction; mode 2 keeps the reasons only.  Clause ids are renumbered, reasons are
    // remapped and the learned watch lists are rebuilt from the watch pairs, which keeps
    // the two-watched-literal invariant at any level.
    __device__ __forceinline__ void reduce_db(int mode)
    {
        const int lane = lane_id();
        for (int32_t i = lane; i < nlearnt; i += kWave) remap[i] = 0;
        msync();
        for (int32_t t = lane; t < tsize; t += kWave) {
            const I4 x = vi[trail[t] >> 1];
            // level-0 reasons are never read
            if (x.y != kNone && (int32_t)x.y >= m && x.x > 0) remap[(int32_t)x.y - m] = 1;
        }
        msync();
        int32_t ns = 0;
        for (int32_t i0 = 0; i0 < nlearnt; i0 += kWave) {
            const int32_t i = i0 + lane;
            const bool in = i < nlearnt;
            const int32_t ic = min(i, nlearnt - 1);
            const I4 r = lrec[ic];
            const I lbd = llbd[ic];
            const bool used = lused[ic] != 0, locked = remap[ic] != 0;
            const bool del = r.x == kNone;
            const bool wanted = mode == 0 ? (lbd <= 3 || used) : false;
            const bool keep = in && (locked || (!del && wanted));
            const uint64_t km = ballot(keep);
            msync();
            const int32_t ni = ns + prefix_count(km);
            if (in) remap[i] = keep ? (I)ni : kNone;
            if (keep) {
                lrec[ni] = r;
                llbd[ni] = lbd;
                lused[ni] = 0;
            }
            ns += popc64(km);
            msync();
        }
        // compact literals (forward copy; a destination never lies above its source)
        int32_t top = 0, used = 0;
        for (int32_t i = 0; i < ns; i++) {
            const I4 r = lrec[i];
            const int32_t st = uni((int32_t)r.z), len = uni((int32_t)r.w);
            const int32_t full = (len + 7) & ~7;
            if (st != top) {
                for (int32_t k0 = 0; k0 < full; k0 += kWave) {
                    const int32_t k = k0 + lane;
                    const I x = larena[8 * st + min(k, full - 1)];
                    msync();
                    if (k < full) larena[8 * top + k] = x;
                    msync();
                }
                if (lane0()) lrec[i].z = (I)top;
            }
            top += full >> 3;
            used += len;
        }
        for (int32_t t = lane; t < tsize; t += kWave) {
            const int32_t v = trail[t] >> 1;
            const I r = vi[v].y;
            if (r != kNone && (int32_t)r >= m) {
                const I x = remap[(int32_t)r - m];
                vi[v].y = x != kNone ? (I)(m + x) : kNone;
            }
        }
        for (int32_t l = lane; l < 2 * n; l += kWave) H::set_l0(&hdr[l]);
        msync();
        for (int32_t i = lane; i < ns; i += kWave) {
            const I2 w = *(const I2*)&lrec[i];
            if (w.x == kNone) continue;
            const int32_t wl[2] = {(int32_t)w.x, (int32_t)w.y};
            for (int h = 0; h < 2; h++) {
                const int32_t pos = H::add_l(&hdr[wl[h]]);
                if (pos < slack) {
                    Wl[wl[h] * slack + pos] = (I)i;
                } else {
                    H::sub_l(&hdr[wl[h]]);
                    I2 none;
                    none.x = none.y = kNone;
                    *(I2*)&lrec[i] = none;
                }
            }
        }
        nlearnt = ns;
        larena_used = used;
        larena_top = top;
        msync();
    }

    // The branching variable (-1: none free): highest activity, then the lower var (VSIDS), or
    // the highest free var (the reference's last free var).
    __device__ __forceinline__ int32_t pick_branch(int mode)
    {
        uint32_t best = 0;
        int32_t bv = 0;
        // With the state in HBM a trip takes about 0.6 us, so eight variables of each lane are read
        // at once, assigned or not (n = 20,000, 1,024 wavefronts: a decision 0.19 ms one by one, 0.05
        // eight at a time).
        constexpr int kAtOnce = kMode == 4 ? 8 : 1;
        for (int32_t v0 = lane_id(); v0 < n; v0 += kAtOnce * kWave) {
            uint32_t val[kAtOnce];
            float score[kAtOnce];
#pragma unroll
            for (int u = 0; u < kAtOnce; u++) {
                const int32_t v = min(v0 + u * kWave, n - 1);
                val[u] = lv[2 * v];
                if (kMode == 4) score[u] = act[v];
            }
#pragma unroll
            for (int u = 0; u < kAtOnce; u++) {
                const int32_t v = v0 + u * kWave;
                if (val[u] == 1 && v < n) {
                    // non-negative floats order as integers
                    const float a = kMode == 4 ? score[u] : act[v];
                    const uint32_t key = mode == 1 ? (uint32_t)v + 1u : (__float_as_uint(a) | 0x80000000u);
                    if (key > best) {
                        best = key;
                        bv = v;
                    }
                }
            }
        }
        const uint32_t top = uniu(wave_max_u32(best));
        if (top == 0) return -1;
        const uint64_t tie = ballot(best == top);
        const int j = ctz64(tie);
        if ((tie & (tie - 1)) == 0) return uni(readlane(bv, j));
        return (int32_t)~uniu(wave_max_u32(best == top ? ~(uint32_t)bv : 0u));
    }

    __device__ __forceinline__ void rescale_activity()
    {
        for (int32_t v = lane_id(); v < n; v += kWave) act[v] *= 1e-30f;
        inc *= 1e-30f;
        lsync();
    }

    // Build the per-instance part of a job: watch lists of the original clauses and the
    // formula's unit clauses at level 0.  Returns false if the formula is falsified there.
    __device__ __forceinline__ bool setup_instance(const SolveArgs& a, int32_t ins)
    {
        const int lane = lane_id();
        const SolveOptsDev& o = a.o;
        const InstMeta mi = a.meta[ins];
        inst = ins;
        n = uni(mi.n);
        m = uni(mi.m);
        const int32_t* lits = a.lits + mi.lit_base;
        const int32_t* coff = a.coff + mi.coff_base;
        // (without clauses the lanes that have no list entry read their own first record instead)
        if constexpr (kShared) {
        this->lits = m ? (const I*)lits : (const I*)urec;
        this->coff = coff;
        }
        const int32_t n2 = 2 * n;
        const int64_t vb = a.var_base[ins];
        slack = o.watch_slack;
        learnt_cap = o.learnt_cap;
        larena_cap = o.larena_cap;
        dl = 0;
        tsize = 0;
        qhead = 0;
        nlearnt = 0;
        larena_used = 0;
        larena_top = 0;
        inc = 1.0f;
        stamp = 0;
        for (int32_t v = lane; v < n; v += kWave) {
            act[v] = a.act_init ? a.act_init[vb + v] : 0.0f;
            phase[v] = a.phase_init ? a.phase_init[vb + v] : (int8_t)o.phase_init;
        }
        for (int32_t v = lane; v < n + 2; v += kWave) lstamp[v] = 0;
        for (int32_t t = lane; t < n + 1; t += kWave) trail[t] = 0;   // entries past the end are read ahead
        if (lane == 0) lv[n2] = 0;
        mark[lane] = 0;
        for (int32_t l = lane; l < n2; l += kWave) {
            lv[l] = 1;
            hdr[l].x = 0u;
            H::set(&hdr[l], 0, 0);
        }
        msync();
        // occurrence counts give the capacity of every original-clause watch list
        const int32_t L = uni(coff[m]);
        for (int32_t k = lane; k < L; k += kWave) atomicAdd(&hdr[lits[k]].x, 1u);
        msync();
        int32_t carry = 0;
        bool longl = slack > kWave;
        for (int32_t l0 = 0; l0 < n2; l0 += kWave) {
            const int32_t l = l0 + lane;
            const int32_t x = l < n2 ? (int32_t)hdr[min(l, n2 - 1)].x : 0;
            longl |= x > kWave;
            const int32_t s = wave_inclusive_scan(x);
            if (l < n2) hdr[l].x = (uint32_t)(carry + s - x);
            carry += readlane(s, 63);
        }
        msync();
        // watch the first two distinct literals of every clause; units and empty clauses at level 0
        bool unsat = false, twice = false;
        int32_t top = 0;
        for (int32_t c0 = 0; c0 < m && !unsat; c0 += kWave) {
            const int32_t c = c0 + lane;
            int32_t len = -1, l0 = -1, l1 = -1;
            int32_t b = 0, full = 0;
            if (c < m) {
                b = ALL3 ? 3 * c : coff[c];
                full = ALL3 ? 3 : coff[c + 1] - b;
                len = full;
            }
            int32_t start = 0;
            if (!ALL3 && !kShared) {
                const int32_t quads = (full + 3) >> 2;
                const int32_t s = wave_inclusive_scan(quads);
                start = top + s - quads;
                top += readlane(s, 63);
            }
            if (len >= 1) {
                l0 = lits[b];
                // the two watches are distinct literals; a clause repeating one literal is a unit
                if (ALL3) {
                    const int32_t y = lits[b + 1], z = lits[b + 2];
                    const int32_t rest = y != l0 ? z : y;
                    if (y != l0) l1 = y;
                    else if (z != l0) l1 = z;
                    twice |= (y >> 1) == (l0 >> 1) || (z >> 1) == (l0 >> 1) || (y >> 1) == (z >> 1);
                    if (kShared) {
                        set_unwatched(c, rest);
                    } else {
                        I4 r;
                        r.x = (I)l0;
                        r.y = (I)y;
                        r.z = (I)z;
                        r.w = (I)rest;
                        rec[c] = r;
                    }
                } else {
                    for (int32_t k = 0; k < full; k++) {
                        const int32_t q = lits[b + k];
                        if (!kShared) olits[4 * start + k] = (I)q;
                        if (l1 < 0 && q != l0) l1 = q;
                        if (full <= 8)
                            for (int32_t j = 0; j < k; j++) twice |= (lits[b + j] >> 1) == (q >> 1);
                    }
                    if (kShared) {
                        set_watches(c, l0, l1);
                    } else {
                        for (int32_t k = full; k & 3; k++) olits[4 * start + k] = (I)n2;
                        I4 r;
                        r.x = (I)l0;
                        r.y = (I)l1;
                        r.z = (I)start;
                        r.w = (I)full;
                        rec[c] = r;
                    }
                }
                if (l1 >= 0) {
                    len = 2;
                    Wo[(int32_t)hdr[l0].x + H::add_o(&hdr[l0])] = (I)c;
                    Wo[(int32_t)hdr[l1].x + H::add_o(&hdr[l1])] = (I)c;
                } else {
                    len = 1;
                }
            }
            if (ballot(len == 0)) unsat = true;
            uint64_t um = ballot(len == 1);
            if (!ALL3) {
                // a longer clause's variables, a lane each: its stamp shows one met before
                uint64_t big = ballot(full > 8);
                while (big) {
                    const int j = ctz64(big);
                    big &= big - 1;
                    const int32_t e = uni(readlane(full, j)), at = uni(readlane(b, j));
                    for (int32_t k = lane; k < e; k += kWave)
                        twice |= atomicExch(&lstamp[lits[at + k] >> 1], c0 + j + 1) == c0 + j + 1;
                    lsync();
                }
            }
            while (um && !unsat) {
                const int j = ctz64(um);
                um &= um - 1;
                const int32_t u = uni(readlane(l0, j));
                const uint32_t val = uniu(value(u));
                if (val == 0) unsat = true;
                else if (val == 1) assign(u, kNone);
            }
        }
        if (m == 0) {
            if (kShared && ALL3) {
                set_unwatched(0, 0);
            } else if (kShared) {
                set_watches(0, 0, 0);
            } else {
                I4 none;
                none.x = none.y = none.z = none.w = 0;
                rec[0] = none;
            }
        }
        dups = ballot(twice) != 0;
        // (a list longer than a wavefront or a watch_slack above 64 makes the instance take
        // propagate_long: 2,000 x n=120 at a slack of 100 137 ms, at 16 76)
        shortl = ballot(longl) == 0;
        if (!ALL3)
            for (int32_t v = lane; v < n + 2; v += kWave) lstamp[v] = 0;
        base_trail = tsize;
        msync();
        return !unsat;
    }

    // Next cube of the instance already set up on this wavefront: undo everything above the
    // formula's unit clauses and forget the learned clauses (they may rest on the previous
    // cube).  Every remaining watch pair is repaired by propagating the units again from the
    // start of the trail.  Activities and saved phases carry over.
    __device__ __forceinline__ void reset_instance()
    {
        const int lane = lane_id();
        for (int32_t t = base_trail + lane; t < tsize; t += kWave) clear_value(trail[t]);
        for (int32_t l = lane; l < 2 * n; l += kWave) H::set_l0(&hdr[l]);
        msync();
        tsize = base_trail;
        qhead = 0;
        dl = 0;
        nlearnt = 0;
        larena_used = 0;
        larena_top = 0;
    }

    // Telemetry: charge the time since the last switch to the current phase and enter
    // `next`.  The counters are the job's JS_PH_* fields, added to without waiting.
    __device__ __forceinline__ void enter(int32_t next)
    {
        if (!ph_out) return;
        const uint64_t now = wall_clock64();
        if (lane0()) atomicAdd(&ph_out[ph_cur], (unsigned long long)(now - ph_t));
        ph_t = now;
        ph_cur = next;
    }

    // Adds the conflicts of this job not yet reported to its instance's pool; returns the
    // pool's new total (wave-uniform).
    __device__ __forceinline__ int64_t report_conflicts(const SolveArgs& a, int32_t ins)
    {
        unsigned long long tot = 0;
        const unsigned long long delta = (unsigned long long)(conflicts - conf_reported);
        if (lane0()) tot = atomicAdd(&a.inst_conf[ins], delta) + delta;
        conf_reported = conflicts;
        return (int64_t)lane0_u64(tot);
    }

    // Testing aid: append the job's held learned clauses and its level-0 literals (as unit
    // clauses) to the dump as one block [inst, slots, then per clause its literals and -1].  The
    // block's space is reserved only if all of it fits, so the dump stays parseable.
    __device__ __forceinline__ void dump_learned(const SolveArgs& a, int32_t ins)
    {
        const int lane = lane_id();
        const int32_t n0 = dl > 0 ? uni((int32_t)tlim[1]) : tsize;   // level-0 part of the trail
        const int64_t slots = (int64_t)larena_used + nlearnt + 2 * (int64_t)n0;
        const unsigned long long total = (unsigned long long)(slots + 2);
        long long base = -1;
        if (lane == 0) {
            atomicAdd(a.learned_need, total);
            unsigned long long old = __hip_atomic_load(a.learned_pos, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            while (old + total <= (unsigned long long)a.learned_cap) {
                const unsigned long long prev = atomicCAS(a.learned_pos, old, old + total);
                if (prev == old) {
                    base = (long long)old;
                    break;
                }
                old = prev;
            }
        }
        base = (long long)lane0_u64((uint64_t)base);
        if (base < 0) return;
        int32_t* out = a.learned_out + base;
        if (lane == 0) {
            out[0] = ins;
            out[1] = (int32_t)slots;
        }
        int64_t p = 2;
        for (int32_t i = 0; i < nlearnt; i++) {
            const I4 r = lrec[i];
            const int32_t st = 8 * uni((int32_t)r.z), len = uni((int32_t)r.w);
            for (int32_t k = lane; k < len; k += kWave) out[p + k] = (int32_t)larena[st + k];
            if (lane == 0) out[p + len] = -1;
            p += len + 1;
        }
        for (int32_t t = lane; t < n0; t += kWave) {
            out[p + 2 * t] = (int32_t)trail[t];
            out[p + 2 * t + 1] = -1;
        }
    }

    // Returns the job verdict: 0 SAT, 1 UNSAT, 2 UNDEF (budget), 3 skipped (instance decided).
    // deadline: wall-clock tick after which the job stops as UNDEF (0: none).
    __device__ __forceinline__ int32_t run_job(const SolveArgs& a, const JobDesc& jd, int64_t max_conflicts,
                                               uint64_t deadline)
    {
        const SolveOptsDev& o = a.o;
        ran = false;
        conf_reported = 0;
        if (load_status(&a.inst_status[jd.inst]) != 2) return 3;
        if (o.inst_conflicts > 0 &&
            (int64_t)__atomic_load_n(&a.inst_conf[jd.inst], __ATOMIC_RELAXED) >= o.inst_conflicts)
            return 2;
        const uint64_t t_start = wall_clock64();
        ph_t = t_start;
        ph_cur = PH_SETUP;
        bumps = a.var_bumps ? a.var_bumps + a.var_base[jd.inst] : nullptr;
        if (setup_inst == jd.inst) {
            reset_instance();
        } else {
            setup_ok = setup_instance(a, jd.inst);
            setup_inst = jd.inst;
        }
        ran = true;
        if (!setup_ok) return 1;
        bool unsat = false;
        // the cube's literals are facts of this job
        for (int32_t k = 0; k < jd.cube_len && !unsat; k++) {
            const int32_t u = uni(a.cube_lits[jd.cube_off + k]);
            const uint32_t val = uniu(value(u));
            if (val == 0) unsat = true;
            else if (val == 1) assign(u, kNone);
        }
        if (unsat) return 1;

        int32_t restart_thr = o.restart_first, restart_cnt = 0;
        const float decay_inv = 1.0f / o.var_decay;
        for (;;) {
            enter(PH_BCP);
            const int32_t confl = propagate();
            if (confl >= 0) {
                // a conflict among the formula's units and the cube counts as none of the search's
                if (dl == 0 && decisions == 0) return 1;
                enter(PH_ANALYZE);
                conflicts++;
                restart_cnt++;
                if (dl == 0) return 1;
                int32_t bt, lbd;
                const int32_t nl = analyze(confl, bt, lbd);
                if (nl < 0) return 4;
                enter(PH_BACKTRACK);
                const int32_t first = uni((int32_t)lbuf[0]);
                if (nl == 1) {
                    backtrack(0, o.decision_mode == 0);
                    assign(first, kNone);
                } else {
                    backtrack(bt, o.decision_mode == 0);
                    enter(PH_ANALYZE);
                    if (!room(nl)) {
                        reduce_db(0);
                        if (!room(nl)) reduce_db(2);
                    }
                    const bool fits = room(nl);
                    if (!fits) {
                        // every held clause is a reason: restart, then add the clause at level 0
                        backtrack(0, o.decision_mode == 0);
                        restarts++;
                        restart_cnt = 0;
                        reduce_db(2);
                    }
                    const int32_t id = store_learned(nl, lbd);
                    if (fits) {
                        watch_learned(id, first, uni((int32_t)lbuf[1]));
                        assign(first, (I)(m + id));
                    } else if (!attach_level0(id)) {
                        return 1;
                    }
                }
                inc *= decay_inv;
                if (inc > 1e30f) rescale_activity();
                if (max_conflicts > 0 && conflicts >= max_conflicts) return 2;
                if ((conflicts & 63) == 0) {
                    const uint64_t now = wall_clock64();
                    if (o.max_ticks > 0 && (int64_t)(now - t_start) > o.max_ticks) return 2;
                    if (deadline && now > deadline) return 2;
                    if (o.inst_conflicts > 0 && report_conflicts(a, jd.inst) >= o.inst_conflicts) return 2;
                }
            } else {
                if (restart_cnt >= restart_thr) {
                    enter(PH_BACKTRACK);
                    restart_thr = (int32_t)((float)restart_thr * o.restart_factor);
                    restart_cnt = 0;
                    backtrack(0, o.decision_mode == 0);
                    restarts++;
                    if (load_status(&a.inst_status[jd.inst]) != 2) return 3;
                    if (nlearnt * 2 >= learnt_cap || larena_used * 2 >= larena_cap) reduce_db(0);
                    continue;
                }
                enter(PH_DECIDE);
                const int32_t v = pick_branch(o.decision_mode);
                if (v < 0) return 0;
                decisions++;
                if (o.max_decisions > 0 && decisions > o.max_decisions) return 2;
                if ((decisions & 1023) == 0) {
                    if (load_status(&a.inst_status[jd.inst]) != 2) return 3;
                    const uint64_t now = wall_clock64();
                    if (o.max_ticks > 0 && (int64_t)(now - t_start) > o.max_ticks) return 2;
                    if (deadline && now > deadline) return 2;
                }
                dl++;
                if (dl > levelmax) levelmax = dl;
                if (lane0()) tlim[dl] = (I)tsize;
                const int32_t ph = o.decision_mode == 1 ? 1 : uni((int32_t)phase[v]);
                assign(2 * v + ph, kNone);
            }
        }
    }
};

}  // namespace

// kMode: where a job's state sits -- 1 all in LDS; 2 the per-var state in LDS, the watch
// structures and the learned literals in this wavefront's slice of the HBM workspace; 3 the
// per-var state and the watch structures (read on every propagation step) in LDS, the learned
// literals in HBM; 4 everything in the HBM slice (formulas whose per-var state does not fit a
// workgroup's LDS).
template <int kMode, class I, bool ALL3>
__global__ __launch_bounds__(kWave) __attribute__((amdgpu_waves_per_eu(solve_waves_per_eu(kMode), solve_waves_per_eu(kMode))))
void k_solve(SolveArgs a)
{
    extern __shared__ __align__(16) char smem_all[];
    const int lane = lane_id();
    // (a workgroup is one wavefront, so wslot is 0; with the LDS region's place known at compile time
    // placement 2 took 1.5-2.5% longer, pigeonhole formulas 137.8 instead of 134.7 ms)
    const int wslot = __builtin_amdgcn_readfirstlane((int)(threadIdx.x / kWave));
    const int64_t gwave = (int64_t)blockIdx.x * (blockDim.x / kWave) + wslot;
    char* smem = smem_all + (uint32_t)wslot * (uint32_t)a.lds_per_wave;
    char* slice = (char*)(a.ws + gwave * a.ws_ints_per_wave);
    Search<kMode, I, ALL3> J;
    if (kMode == 4) J.carve(slice, slice + a.lay.state_bytes, slice + a.lay.state_bytes + a.lay.watch_bytes, a);
    else if (kMode == 2) J.carve(smem, slice, slice + a.lay.watch_bytes, a);
    else if (kMode == 3) J.carve(smem, smem + a.lay.state_bytes, slice, a);
    else J.carve(smem, smem + a.lay.state_bytes, smem + a.lay.state_bytes + a.lay.watch_bytes, a);
    J.setup_inst = -1;
    J.setup_ok = false;
    J.n = 0;
    J.dl = J.tsize = 0;
    int32_t n_jobs = a.n_jobs;
    const int32_t* order = nullptr;
    int64_t budget = a.o.max_conflicts;
    if (a.epoch) {
        const int32_t e = uni(*a.epoch);
        n_jobs = uni(a.n_active[e & 1]);
        order = a.active + (int64_t)(e & 1) * a.n_jobs;
        budget = a.epoch_budget[e];
    }
    // the whole-solve deadline counts from the first wavefront's start (kept across epochs)
    uint64_t deadline = 0;
    if (a.o.deadline_ticks > 0) {
        unsigned long long t0 = 0;
        if (lane == 0) {
            const unsigned long long now = wall_clock64();
            const unsigned long long old = atomicCAS(a.t_start, 0ull, now);
            t0 = old ? old : now;
        }
        t0 = lane0_u64(t0);
        deadline = (uint64_t)t0 + (uint64_t)a.o.deadline_ticks;
    }
    int32_t j = 0, j_end = 0;
    for (;;) {
        if (j >= j_end) {
            // grab the next chunk of consecutive jobs (cubes of one instance are adjacent)
            int32_t k = 0;
            if (lane == 0) k = atomicAdd(a.queue_head, 1);
            k = uni(k);
            j = k * a.chunk;
            if (j >= n_jobs) break;
            j_end = min(j + a.chunk, n_jobs);
        }
        const JobDesc jd = a.jobs[order ? order[j] : j];
        j++;
        const uint64_t t_job = wall_clock64();
        // past the deadline a job is not started: UNDEF
        J.ran = false;
        J.conflicts = J.decisions = J.props = J.learned = J.restarts = 0;
        J.levelmax = 0;
        J.ph_out = (a.o.telemetry && a.job_stats)
                       ? (unsigned long long*)(a.job_stats + (int64_t)jd.order * JS_COUNT + JS_PH_SETUP) : nullptr;
        J.ph_t = t_job;
        J.ph_cur = PH_SETUP;
        // in epoch mode the epoch's budget replaces the per-job one, bounded by what is left
        // of opts.max_conflicts after the job's earlier epochs (a spent job is UNDEF)
        int64_t job_budget = budget;
        if (a.epoch && a.o.max_conflicts > 0 && a.job_stats) {
            const int64_t left = a.o.max_conflicts - a.job_stats[(int64_t)jd.order * JS_COUNT + JS_CONFLICTS];
            job_budget = min(budget, left);
        }
        const bool spent = a.epoch && a.o.max_conflicts > 0 && a.job_stats && job_budget <= 0;
        const int32_t st = ((deadline && t_job > deadline) || spent) ? 2 : J.run_job(a, jd, job_budget, deadline);
        J.enter(PH_SETUP);   // charge the last phase
        const uint64_t job_ticks = wall_clock64() - t_job;
        J.msync();
        const int32_t inst = jd.inst;
        if (a.o.inst_conflicts > 0 && J.ran) (void)J.report_conflicts(a, inst);
        if (a.learned_out && J.ran && J.setup_ok) J.dump_learned(a, inst);
        if (st == 0) {
            int32_t won = 0;
            if (lane == 0) won = atomicCAS(&a.inst_status[inst], 2, 0) == 2;
            won = uni(won);
            if (won) {
                const InstMeta mi = a.meta[inst];
                const int32_t W = words_per_row(mi.n);
                for (int32_t w = lane; w < W; w += kWave) {
                    uint32_t x = 0;
                    for (int b = 0; b < 32; b++) {
                        const int32_t l = 32 * w + b;
                        if (l < 2 * mi.n && J.lv[l] == 2) x |= 1u << b;
                    }
                    a.model_rows[mi.word_base + w] = x;
                }
            }
        } else if (st == 1) {
            if (lane == 0) {
                const int32_t r = atomicAdd(&a.inst_refuted[inst], 1) + 1;
                if (r == a.inst_ncubes[inst]) atomicCAS(&a.inst_status[inst], 2, 1);
            }
        } else if (st == 2) {
            if (lane == 0) atomicAdd(&a.inst_undef[inst], 1);
            if (a.act_store && J.ran) {
                // a job stopped at an epoch boundary restarts next epoch from these
                const int64_t vb = a.var_base[inst];
                for (int32_t v = lane; v < J.n; v += kWave) {
                    a.act_store[vb + v] = J.act[v];
                    a.phase_store[vb + v] = J.phase[v];
                }
            }
        }
        if (a.job_stats && lane == 0) {
            int64_t* s = a.job_stats + (int64_t)jd.order * JS_COUNT;
            // counters add up over the epochs a job runs in
            s[JS_STATUS] = st;
            s[JS_CONFLICTS] += J.conflicts;
            s[JS_DECISIONS] += J.decisions;
            s[JS_PROPS] += J.props;
            s[JS_LEARNED] += J.learned;
            s[JS_RESTARTS] += J.restarts;
            s[JS_LEVELMAX] = max(s[JS_LEVELMAX], (int64_t)J.levelmax);
            s[JS_TICKS] += (int64_t)job_ticks;
        }
        J.msync();
    }
}

// Restart epochs.  begin: empty the queue and the next job list.  end: every job of
// this epoch stopped by the budget whose instance is still open goes to the next list;
// then the epoch counter advances and the number of open jobs is published.
__global__ void k_epoch_begin(int32_t* queue_head, const int32_t* epoch, int32_t* n_active)
{
    if (threadIdx.x == 0) {
        *queue_head = 0;
        n_active[(*epoch + 1) & 1] = 0;
    }
}

__global__ void k_epoch_end(SolveArgs a, int32_t* active, int32_t* n_active)
{
    const int32_t e = *a.epoch;
    const int32_t n = n_active[e & 1];
    const int32_t* cur = active + (int64_t)(e & 1) * a.n_jobs;
    int32_t* next = active + (int64_t)((e + 1) & 1) * a.n_jobs;
    for (int32_t k = blockIdx.x * blockDim.x + threadIdx.x; k < n; k += gridDim.x * blockDim.x) {
        const int32_t job = cur[k];
        const JobDesc jd = a.jobs[job];
        const int64_t* js = a.job_stats + (int64_t)jd.order * JS_COUNT;
        const bool spent = a.o.max_conflicts > 0 && js[JS_CONFLICTS] >= a.o.max_conflicts;
        if (js[JS_STATUS] == 2 && !spent && a.inst_status[jd.inst] == 2) next[atomicAdd(&n_active[(e + 1) & 1], 1)] = job;
    }
}

__global__ void k_epoch_advance(int32_t* epoch, const int32_t* n_active, int32_t* remaining)
{
    if (threadIdx.x == 0) {
        const int32_t e = *epoch;
        *remaining = n_active[(e + 1) & 1];
        *epoch = e + 1;
    }
}

hipError_t launch_epoch_begin(const SolveArgs& a, hipStream_t st)
{
    hipLaunchKernelGGL(k_epoch_begin, dim3(1), dim3(64), 0, st, a.queue_head, a.epoch, (int32_t*)a.n_active);
    return hipGetLastError();
}

hipError_t launch_epoch_end(const SolveArgs& a, int32_t* remaining, hipStream_t st)
{
    hipLaunchKernelGGL(k_epoch_end, dim3(std::max(1, std::min(1024, (a.n_jobs + 255) / 256))), dim3(256), 0, st, a,
                       (int32_t*)a.active, (int32_t*)a.n_active);
    hipLaunchKernelGGL(k_epoch_advance, dim3(1), dim3(64), 0, st, (int32_t*)a.epoch, a.n_active, remaining);
    return hipGetLastError();
}

// Byte offsets of a job's arrays for instances of up to max_n variables, max_m clauses and max_L
// literals, with ids of id_bytes bytes.
SolveLayout solve_layout(int32_t max_n, int32_t max_m, int64_t max_L, bool all3, int id_bytes, const SolveOptsDev& o)
{
    SolveLayout L{};
    const int64_t n = max_n, I = id_bytes;
    int64_t at = 0;
    const auto take = [&](int64_t bytes) {
        const int64_t p = at;
        at = (at + bytes + 15) & ~(int64_t)15;
        return p;
    };
    L.id_bytes = id_bytes;
    L.lv = take(2 * n + 1);   // at the region's start: its address needs no addition
    L.hdr = take(2 * n * (id_bytes == 2 ? 8 : 12));
    L.vi = take(n * 4 * I);
    L.act = take(n * 4);
    L.lstamp = take((n + 2) * 4);
    L.trail = take((n + 1) * I);
    L.tlim = take((n + 2) * I);
    L.lbuf = take((n + 1) * I);
    L.phase = take(n);
    L.mark = take(64);
    L.state_bytes = at;
    at = 0;
    // a list is read by all 64 lanes, and clause 0 also where there is none
    L.rec = take((int64_t)(max_m + 1) * (id_bytes == 2 ? 4 : all3 ? 1 : 2) * I);
    L.lrec = take((int64_t)o.learnt_cap * 4 * I);
    L.wo = take((max_L + 64) * I);
    L.wl = take((2 * n * o.watch_slack + 64) * I);
    L.llbd = take(o.learnt_cap * I);
    L.remap = take(o.learnt_cap * I);
    L.lused = take(o.learnt_cap);
    L.olits = take(all3 || id_bytes == 4 ? 0 : (max_L + 3 * (int64_t)max_m) * I);
    L.watch_bytes = at;
    L.arena_bytes = ((int64_t)o.larena_cap + 7 * (int64_t)o.learnt_cap) * I;
    L.arena_bytes = (L.arena_bytes + 15) & ~(int64_t)15;
    return L;
}

// 16-bit ids hold every literal (with a mark bit), clause id (with a none value), clause start in
// units of 4 literals, clause length (max_len: the longest; literals may repeat, so n does not
// bound it) and list length of these sizes.
bool solve_ids16(int32_t max_n, int32_t max_m, int64_t max_L, int64_t max_len, const SolveOptsDev& o)
{
    return max_n < 16000 && max_len <= UINT16_MAX && (int64_t)max_m + o.learnt_cap < 65000 && max_L + 3 * (int64_t)max_m < 4 * 65000 &&
           max_L < 65000 * 4 && (int64_t)o.larena_cap + 7 * (int64_t)o.learnt_cap < 8 * 65000 && o.watch_slack < 65000;
}

template <bool ALL3>
static void launch_mode(const SolveArgs& a, int mode, dim3 grid, dim3 block, size_t lds, hipStream_t st)
{
    if (mode == 1) hipLaunchKernelGGL((k_solve<1, uint16_t, ALL3>), grid, block, lds, st, a);
    else if (mode == 3) hipLaunchKernelGGL((k_solve<3, uint16_t, ALL3>), grid, block, lds, st, a);
    else hipLaunchKernelGGL((k_solve<2, uint16_t, ALL3>), grid, block, lds, st, a);
}

hipError_t launch_solve(const SolveArgs& a, int clause_mem, int waves, size_t lds_bytes, hipStream_t st)
{
    if ((size_t)a.lds_per_wave != lds_bytes) return hipErrorInvalidValue;
    const dim3 grid(waves), block(kWave);   // a workgroup per wavefront
    const size_t lds = lds_bytes;
    const bool ids16 = a.lay.id_bytes == 2;
    if (clause_mem == 4 && a.all3)
        hipLaunchKernelGGL((k_solve<4, uint32_t, true>), grid, block, 0, st, a);
    else if (clause_mem == 4)
        hipLaunchKernelGGL((k_solve<4, uint32_t, false>), grid, block, 0, st, a);
    else if (!ids16 && a.all3)
        hipLaunchKernelGGL((k_solve<2, uint32_t, true>), grid, block, lds, st, a);
    else if (!ids16)
        hipLaunchKernelGGL((k_solve<2, uint32_t, false>), grid, block, lds, st, a);
    else if (a.all3)
        launch_mode<true>(a, clause_mem, grid, block, lds, st);
    else
        launch_mode<false>(a, clause_mem, grid, block, lds, st);
    return hipGetLastError();
}

}  // namespace gpsat
