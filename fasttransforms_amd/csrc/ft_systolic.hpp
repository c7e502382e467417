// ft_systolic.hpp -- band-systolic rotation engine for the whole-matrix
// executors (ft_execute_{sph,tri,disk}_{hi2lo,lo2hi}, drivers.c:58-110,
// 314-326, 414-430).
//
// What is computed (src/rotations/rotations_default.c:31-71): every column
// applies a chain of rotation sequences; sequence j rotates the row pairs
// (e, e+1) of its class rows e = top(j) .. 0 (hi2lo) or 0 .. top(j) (lo2hi).
// Consecutive sequences of a chain differ by one in top(j), and every column
// of a class applies a suffix (hi2lo) or prefix (lo2hi) of one common list of
// sequences k = 0 .. K-1.
//
// How it maps onto the GPU:
//
//  * Lanes are sequences.  A wave runs one band: FTAMD_SYS_LANES*S
//    consecutive sequences, S per lane, for the 8 columns of a chain (4 rows
//    of 16 lanes, 2 columns per lane).  Each lane holds, per sequence and
//    column, the row its sequence carries; every step every sequence rotates
//    (carried, fresh) and emits the other row to the next sequence: inside a
//    lane in the same step, from lane to lane by a DPP row shift one step
//    later.  Rows enter the band as a stream at lane 0 of each row (rows
//    R .. 0 for hi2lo, 0 .. R for lo2hi) and leave it at lane 15, S+1 steps
//    per lane later.  Steps where a sequence has no rotation (before its rows
//    arrive, after its last row, or for a column that does not apply it) use
//    the identity (s, c) = (0, 1), which passes the stream through with the
//    same delay; so the whole band is one uniform loop, and the table of a
//    band is laid out step-major ([step][lane][slot]) with identities in the
//    gaps.
//  * s and c are per lane (each lane is a different sequence): no broadcast;
//    the 4 rows of a wave read the same 16 lanes' entries.
//  * A chain runs its bands as waves of one workgroup; band b+1 reads band
//    b's output stream through an LDS ring as it is produced, so a chain's
//    bands overlap and the chain's latency is about one band's stream plus
//    (S+1)*LANES steps per band.  The first band reads A; rows that leave the
//    chain are stored to A once per 8-step block by the band that emits them.
//  * A long chain runs in parts of at most a set number of bands, each part
//    on its own workgroup: the last band of a part stores every row it emits
//    to A and publishes a progress counter, and the first band of the next
//    part reads those rows back from A as they are published.  This spreads a
//    long chain's waves over several CUs and lifts the bound of 16 bands (one
//    workgroup's waves) per chain.
//  * Workgroups are persistent (about one per CU).  The host deals the parts
//    to slots, per XCD, and a workgroup takes its XCD's slots in order; a
//    slot's parts stream through the workgroup's waves one after another.
//    The parts of one chain run in increasing slots of one XCD, so a waiting
//    part only ever waits on a slot that a running workgroup holds or has
//    finished, and the rows they hand over stay in that XCD's L2.
//
// Arithmetic: the reference's rotation in fused form, x' = fma(c, x, s*y),
// y' = fma(c, y, -(s*x)) (src/rotations/rotations_AVX512F.c:4-15).  With
// x = the fresh row and y = the carried one this is both the hi2lo rotation of
// rows (e, e+1) and the transposed lo2hi rotation of (e+1, e), so one loop
// serves both directions.  Compiled with -ffp-contract=off.
#pragma once

#include <hip/hip_runtime.h>

#include "ft_hip_abi.h"

namespace ftsys {

constexpr int kLanes = FTAMD_SYS_LANES;
constexpr int kRows = 4;
constexpr int kCols = 2;
constexpr int kWaves = FTAMD_SYS_WAVES;
// ring slots between two bands (a multiple of kU):
// 64 lets a band run up to 64 rows ahead of the next (64 KB of LDS per
// workgroup; 3-9 % faster than 32 at n = 1024, 80 no better)
constexpr int kZ = 64;
constexpr int kU = FTAMD_SYS_UNROLL;   // steps per loop iteration
constexpr int kDin = 2;                // input positions read ahead
constexpr int kChunk = 16;             // rows of another part fetched per lane-parallel load


template <typename T> using Pair = T __attribute__((ext_vector_type(2)));

// The launch's records never change while it runs: read through the constant
// address space, so that wave-uniform reads are scalar loads.
typedef __attribute__((address_space(4))) FtamdSysBand ConstBand;
typedef __attribute__((address_space(4))) FtamdSysChain ConstChain;
typedef __attribute__((address_space(4))) FtamdSysItem ConstItem;
typedef __attribute__((address_space(4))) int ConstInt;

__device__ __forceinline__ int uniform(int v) { return __builtin_amdgcn_readfirstlane(v); }

template <typename T> __device__ __forceinline__ T lds_ld(const T *p) {
    return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
}
template <typename T> __device__ __forceinline__ void lds_st(T *p, T v) {
    __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
}

// Lanes 1..15 of every row of 16 take src of the lane before; lane 0 of each
// row keeps old (DPP row_shr:1 without bound control).
template <typename T> __device__ __forceinline__ T shift_in(T old, T src) {
    return __builtin_amdgcn_update_dpp(old, src, 0x111, 0xf, 0xf, false);
}

template <typename T> __device__ __forceinline__ T fmaT(T a, T b, T c);
template <> __device__ __forceinline__ double fmaT<double>(double a, double b, double c) { return __builtin_fma(a, b, c); }
template <> __device__ __forceinline__ float fmaT<float>(float a, float b, float c) { return __builtin_fmaf(a, b, c); }

template <typename T, int S, bool ROWMASK>
struct Engine {
    static constexpr int B = kLanes * S;  // sequences per band
    // a row that enters lane 0 at step p leaves lane 15 at step p + kOutDelay:
    // S+1 steps per lane (the lane's S sequences pass it on within a step,
    // the DPP shift to the next lane takes a step)
    static constexpr int kOutDelay = (S + 1) * (kLanes - 1) + S;
    // steps the table entries are read out of LDS ahead of their use
    static constexpr int kAhead = 2;
    // what a band has besides its neighbours' rings: rows from A all along (a
    // chain's first band), rows to A all along (its last), either
    static constexpr int kInner = 0, kFirst = 1, kLast = 2, kBoth = 3;

    // table bytes of one step (all 16 lanes) and steps per 1 KB LDS-DMA load
    static constexpr int kStepBytes = kLanes * S * 2 * (int)sizeof(T);
    static constexpr int kSPD = 1024 / kStepBytes;
    // steps of table entries staged ahead in LDS (4 DMA blocks)
    static constexpr int kD = 4 * kSPD;
    static_assert(kZ % kU == 0 && kZ >= 2 * kChunk, "ring of whole blocks, two fetch chunks deep");
    static_assert(kSPD >= 1 && kU % kSPD == 0 && kD <= FTAMD_SYS_PREFETCH,
                  "DMA blocks must tile the unroll and the tables' spare steps");
    // a block's table slots are at most one wrap of the LDS ring, and its
    // DMAs use the compile-time offsets 0, 2, 4, 6 (kSPD 2) or 0, 4 (kSPD 4)
    static_assert(kD >= kU && kD % kU == 0 && (kSPD == 2 || kSPD == 4),
                  "table staging supports 2 or 4 steps per DMA and a ring of whole blocks");


    struct Shared {
        // table entries of the next kD steps of each wave, written by LDS DMA
        // (first in the block: the DMA's LDS address is taken from M0)
        // step-major; within a step slot-major for FP64 ([slot][lane]: a
        // lane's 16-byte pair next to the next lane's, so a 128-bit read of
        // 8 lanes spans all banks once) and lane-major for FP32 ([lane][slot]:
        // a lane's S pairs in one 128-bit read); the tables are laid out
        // the same way (FTAMD_SYS_SLOT_MAJOR)
        Pair<T> scr[kWaves][kD][kLanes * S];
        Pair<T> ring[kWaves][kZ][kRows];  // ring g: input stream of the band wave g runs (a row's two columns)
        // per wave, published together after every block: the ring slots of
        // ring g it has read, and those of ring g+1 it has written (exclusive ends)
        struct Published {
            int freed, avail;
        } pub[kWaves + 2];                 // wave g's at index g + 1
        Pair<T> ident[kD][kLanes * S];     // (0, 1): what a masked sequence reads in place of scr
        unsigned spare[64];                // where fillers go
        int abort_flag;
        int slot;                          // the workgroup's current slot (ticket)
    };

    // The table entries of one lane for one step: S (s, c) pairs, one for each
    // of MC columns or one for both.
    template <int MC> struct SC {
        Pair<T> p[S][MC];
    };

    // A wave whose wait expires raises the workgroup's abort flag (every
    // other wait then ends too) and reports the error once its loop is left.
    __device__ static void fail(Shared &sh) { lds_st(&sh.abort_flag, 1); }


    // Waits until *ctr >= need (seen: the last value read), at most `limit`
    // polls.
    __device__ static bool wait_ge(Shared &sh, int *ctr, int need, int &seen, int limit) {
        for (int it = 1;; ++it) {
            seen = uniform(lds_ld(ctr));
            if (seen >= need) return true;
            if (it >= limit || uniform(lds_ld(&sh.abort_flag))) return false;
            // far behind (a band waiting for the chain's fill): poll rarely,
            // so waiting waves leave the issue slots to the working ones
            if (need - seen > 2 * kU) __builtin_amdgcn_s_sleep(4);
            else __builtin_amdgcn_s_sleep(1);
        }
    }

    // Table entries reach the waves by LDS DMA (global_load_lds_dwordx4: 64
    // lanes x 16 bytes, the kSPD steps of one block, straight into the
    // wave's LDS ring, no registers in flight), issued by hand with hand
    // counted waits: in this loop the compiler's own wait insertion loses
    // count and would drain every load at every step, defeating the
    // prefetch.  Each block's DMA is the only vector-memory instruction the
    // loop issues besides the first band's matrix fetches (which only add
    // to the count), so a block is in LDS once at most as many DMAs as were
    // issued after it are outstanding.
    // `after` is a value the caller computed from the entries last read out
    // of the block being refilled: tying it to the DMA keeps the DMA after
    // those reads have returned.
    __device__ static void dma_block(Shared &sh, int w, const char *tab_band, int step, unsigned lane16, T after) {
        const int slot = step % kD;
        const unsigned lds = (unsigned)(uintptr_t)&sh.scr[w][slot][0];
        const char *src = tab_band + (long long)uniform(step) * kStepBytes;
        // M0 (the DMA's LDS address) needs one wait state before the DMA
        // reads it; nothing else in this kernel uses M0.
        asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2"
                     :
                     : "s"(uniform((int)lds)), "v"(lane16), "s"(src), "v"(after)
                     : "memory");
    }
    // The same in the loop, with the step split into a uniform base and a
    // compile-time part K: the instruction's immediate offset is added to both
    // the global and the LDS address, so M0 stays at the base slot for a whole
    // block of steps (set_m0) and offset:K*bytes selects step base+K on both
    // sides.
    __device__ static void set_m0(unsigned lds_base) { asm volatile("s_mov_b32 m0, %0" : : "s"(lds_base) : "memory"); }
    template <int K>
    __device__ static void dma_block_at(const char *src_base, unsigned lane16, T after) {
        asm volatile("global_load_lds_dwordx4 %0, %1 offset:%3"
                     :
                     : "v"(lane16), "s"(src_base), "v"(after), "n"(K * kStepBytes)
                     : "memory");
    }
    // A DMA of a dword a lane from the start of a table to nowhere in particular.
    __device__ static void dma_filler(Shared &sh, const char *tab, unsigned lane16) {
        asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dword %1, %2"
                     :
                     : "s"(uniform((int)lds_addr(sh.spare))), "v"(lane16), "s"(tab)
                     : "memory");
    }
    // Called before the first read of a block, kAhead steps before its first
    // step, when the two blocks after it have been requested and the third
    // not yet.
    // `Extra`: other vector memory operations issued since the block that may
    // stay outstanding with them.
    template <int Extra = 0>
    __device__ static void wait_block() {
        asm volatile("s_waitcnt vmcnt(%0)" ::"n"(kD / kSPD - 2 + Extra) : "memory");
    }
    // Lane 15 of each row of 16 (the row's last sequence), DPP row_newbcast:15,
    // into the lanes 4b .. 4b+3 of each row (bank b) of `keep`.
    template <int B> __device__ static T row_end(T keep, T v) {
        return __builtin_amdgcn_update_dpp(keep, v, 0x15f, 0xf, 1 << B, false);
    }
    __device__ static unsigned lds_addr(const void *p) { return (unsigned)(uintptr_t)p; }
    template <typename V> using Lds = __attribute__((address_space(3))) V;
    template <typename V> __device__ static Lds<V> *lds_at(unsigned addr) { return (Lds<V> *)(uintptr_t)addr; }

    // position of (lane i, slot s) in a step's entries, and of lane i's first
    static constexpr bool kSlotMajor = sizeof(T) == 8;
    static constexpr int kSlotStride = kSlotMajor ? kLanes : 1;
    __device__ static int lane_entry(int i) { return kSlotMajor ? i : i * S; }

    // Progress counters of split chains.  The producing band stores its rows
    // to A with device-scope stores and, once they are complete, publishes
    // how many it has stored with a device-scope store; the consuming band
    // polls the counter with a scalar load that bypasses the scalar cache
    // (GLC), so that polling never waits on the vector-memory counter the
    // table DMAs run on, and then reads the rows with device-scope loads.
    // Both parts run on one XCD, so they meet in one L2.
    __device__ static int poll_prog(const int *p) {
        int v;
        asm volatile("s_load_dword %0, %1, 0x0 glc\n\ts_waitcnt lgkmcnt(0)" : "=s"(v) : "s"(p) : "memory");
        return v;
    }
    __device__ static bool wait_prog(Shared &sh, const int *p, int need, int &seen, int limit) {
        for (int it = 0; seen < need; ++it) {
            if (it >= limit || uniform(lds_ld(&sh.abort_flag))) return false;
            if (it > 0) __builtin_amdgcn_s_sleep(2);
            seen = uniform(poll_prog(p));
        }
        return true;
    }

    // One step in two halves, so that what the next lane and the next step
    // wait for comes first: emit() computes every sequence's outgoing row,
    // carry() its new carried row, after the step's LDS accesses are issued.
    // X0: the fresh rows of the lane's first sequence (the last sequence of
    // the lane before emitted them at the previous step, or the stream at
    // lane 0); Y: carried rows; sequence s > 0 takes as its fresh row what
    // sequence s-1 emits in this step.
    template <int MC> struct Applied {  // a step's (s, c) with its fresh rows
        SC<MC> sc;
        T x[S][kCols];
    };
    template <int MC>
    __device__ static void emit(const T (&Y)[S][kCols], T (&E)[S][kCols], const T (&X0)[kCols], const SC<MC> &sc,
                                Applied<MC> &ap) {
        ap.sc = sc;
#pragma unroll
        for (int s = 0; s < S; ++s)
#pragma unroll
            for (int c = 0; c < kCols; ++c) {
                const Pair<T> e = sc.p[s][c % MC];
                ap.x[s][c] = s == 0 ? X0[c] : E[s - 1][c];
                E[s][c] = fmaT<T>(e.y, Y[s][c], -(e.x * ap.x[s][c]));
            }
    }
    template <int MC> __device__ static void carry(T (&Y)[S][kCols], const Applied<MC> &ap) {
#pragma unroll
        for (int s = 0; s < S; ++s)
#pragma unroll
            for (int c = 0; c < kCols; ++c) {
                const Pair<T> e = ap.sc.p[s][c % MC];
                Y[s][c] = fmaT<T>(e.y, ap.x[s][c], e.x * Y[s][c]);
            }
    }

    // w: the band's index in its chain part; g: the wave (and ring) index in
    // the workgroup.  Ring slots are counted across the chains a workgroup
    // streams: this band's input stream starts at slot in_base of ring g, its
    // output (the next band's input) at out_base of ring g+1, both multiples
    // of kZ; stream position p is in slot off + p (idle()).  END: kFirst a
    // chain's first band, kLast its last, kBoth any; MASK 0: every column
    // applies every sequence of the band; 1: the two columns of a lane row
    // apply the same sequences; 2: per column (a sequence a column does not
    // apply is the identity (0, 1), read from a block of identities in place
    // of the table: no arithmetic); LINK: a band that hands
    // rows to or takes them from another part of its chain (through A).
    // Returns false if a wait expired (abort raised).
    //
    // What bounds it: a step is 16 FP64 operations (S = 2), 4 DPP moves to the
    // next lane and 2 that keep its outputs; an LDS write takes 13 clocks of
    // the CU's LDS input whatever its lane mask (a 128-bit read 4), so
    // outputs are kept in registers and leave a block of 8 at a time: the DPP
    // broadcast of the row's last lane writes one bank of 4 lanes per step
    // under its bank mask, no selects.  A step's outputs are kept a step late,
    // which takes them off the critical path.  Everything
    // that does not happen in every block waits for a step count (t_in, t_out):
    // a block's own work is one compare, its steps, its outputs and one write
    // of the counters.  (sph hi2lo n = 1024, 1024 x 2047 FP64, with the copy
    // of the coefficients before it: 170 -> 142 us; FP32 lo2hi n = 733: 89 ->
    // 67 us, against selects per step, an LDS round trip per wait and the
    // first band's rows through registers; the kernel alone under the
    // profiler 192 -> 153.  A step takes a lone wave about 190
    // clocks, 22 of its instructions on the vector ALU; with four waves on a
    // SIMD the ALU bounds it.)
    template <int MASK, int END, bool LINK>
    __device__ static bool run_band(const FtamdSysLaunch &a, Shared &sh, const ConstChain &ch, const FtamdSysChain &cv,
                                    int w, int g, int lane, int in_base, int out_base) {
        constexpr int kLag = kOutDelay + 1;  // a position's steps from lane 0 to its store
        constexpr int kNever = 0x7fffffff;
        // what follows from the lane is computed here, not once for every
        // instantiation before the loop over the parts (it would not fit the
        // registers)
        asm volatile("" : "+v"(lane));
        const int r = lane >> 4, i = lane & 15;
        const int nb = uniform(ch.nb);
        const ConstBand *band = (const ConstBand *)(uintptr_t)a.bands + (uniform(ch.band0) + w);
        const int R = uniform(band->R);
        const int gbase = uniform(band->gbase);
        const bool first = END == kBoth ? w == 0 : END == kFirst, last = END == kBoth ? w == nb - 1 : END == kLast;
        const int dir = uniform(ch.dir);
        const int Rprev = first ? 0 : uniform(band[-1].R);
        const int off = idle(w);
        // stream positions 0 .. npa-1 come from A, the rest from the previous band
        const int npa = first ? R + 1 : (dir == 0 ? R - Rprev : 0);
        // a part after the first of its chain: its positions from npa_own on
        // are the previous part's output position p - npa_own, published on
        // counter split_in; the last band of a part before the last stores
        // every row it emits and publishes them on counter split_out
        const int split_in = LINK && first ? uniform(ch.split_in) : -1;
        const int split_out = LINK && last ? uniform(ch.split_out) : -1;
        const bool polled = LINK && split_in >= 0;
        const int npa_own = polled && dir == 0 ? R - uniform(band[-1].R) : 0;
        int prog_seen = 0, published = 0, pub = 0;
        // output position p goes to slot p + out_off of the next band's
        // stream; positions beyond ring_hi leave the chain (or the part)
        int ring_hi = -1, out_off = 0;
        if (!last) {
            const int Rnext = uniform(band[1].R);
            const int npa_next = dir == 0 ? Rnext - R : 0;
            ring_hi = min(R, Rnext - npa_next);
            out_off = npa_next + idle(w + 1);
        }
        const long long rstep = uniform(ch.rstep), lda = uniform(ch.lda);
        const int rpar = uniform(ch.rpar);
        const int spin = uniform(a.spin_limit);  // polls before a wait gives up
        T *A = (T *)a.A + ch.aoff;
        // step t takes the table's step t - off (the steps before a later
        // band's table are the spare steps of the band before: identities)
        const char *tab_band = (const char *)a.tab + (band->tab * (long long)sizeof(Pair<T>) - (long long)off * kStepBytes);
        const unsigned lane16 = (unsigned)lane * 16u;

        // ---- table prefetch: steps 0 .. kD-1
#pragma unroll
        for (int d = 0; d < kD; d += kSPD) dma_block(sh, g, tab_band, d, lane16, T(0));

        // class row of stream position p
        auto row_of = [&](int p) { return dir == 0 ? R - p : p; };
        const long long astep = dir == 0 ? -rstep : rstep;  // elements of A from one position to the next

        Pair<T>(*in_ring)[kRows] = sh.ring[g];
        T *out_ring = (T *)sh.ring[last ? g : g + 1];
        int *const avail = &sh.pub[g].avail;       // of the wave before
        int *const freed = &sh.pub[g + 2].freed;   // of the wave after
        const int slots = R + off;                 // the stream's last slot
        bool ok = true;
        // the slots before position 0 pass through as rows of zeros
        if (i < off) in_ring[i][r] = Pair<T>{T(0), T(0)};

        // ---- stream positions from A.  By LDS DMA straight into the ring: a
        // load of one dword a lane covers kRowsDma positions (8 elements each,
        // in the ring's order), so no register waits for it, and the waits on
        // the table DMAs issued after it cover it.
        constexpr int kDw = (int)sizeof(T) / 4;
        constexpr int kRowsDma = 64 / (FTAMD_SYS_COLS * kDw);  // positions of one DMA
        const int de = lane / kDw;                              // the lane's element of the block
        const int dcol = cv.col[de % FTAMD_SYS_COLS], dpos = de / FTAMD_SYS_COLS;
        const char *rows_src = (const char *)(A + ((long long)max(dcol, 0) * lda + rpar + rstep * row_of(dpos))) +
                               4 * (lane % kDw);
        const unsigned in_lds = uniform(lds_addr(in_ring));
        const unsigned long long rows_on = __ballot(dcol >= 0);
        auto dma_rows = [&](int p0) {  // positions p0 .. p0 + kRowsDma - 1 (those below npa)
            unsigned long long on = rows_on;
            if (p0 + kRowsDma > npa) on = __ballot(dcol >= 0 && p0 + dpos < npa);
            unsigned long long save;
            asm volatile("s_mov_b64 %0, exec\n\ts_mov_b32 m0, %1\n\ts_mov_b64 exec, %2\n\t"
                         "global_load_lds_dword %3, off\n\ts_mov_b64 exec, %0"
                         : "=&s"(save)
                         : "s"(in_lds + (unsigned)((p0 + off) % kZ) * (unsigned)sizeof(Pair<T>[kRows])), "s"(on),
                           "v"(rows_src)
                         : "memory");
            rows_src += astep * (kRowsDma * (int)sizeof(T));
        };
        // how far ahead of the step that starts a block its rows are requested
        constexpr int kRowsAhead = 32;
        // A band that takes rows from A all along or stores its rows there
        // issues this many vector memory operations per block after its last
        // table DMA and before the next block's first: the next rows from A,
        // a store of A, or a filler in their place, so that the waits on the
        // table DMAs can leave them outstanding (rows of A take a trip to HBM).
        constexpr int kExtra = (END & kFirst ? kU / kRowsDma : 0) + (END & kLast ? 1 : 0);
        static_assert(kZ >= kRowsAhead + 2 * kU, "slots are read before they are written again");

        // A chain part that takes rows from another part polls for them and
        // reads them with device-scope loads: lane i of each row fetches
        // position p0 + i of a chunk of 16, 16 steps before it is written to
        // the ring, 32 before it is read.
        const int colv[kCols] = {cv.col[2 * r], cv.col[2 * r + 1]};
        auto aptr = [&](int c, int e) -> T * { return A + ((long long)colv[c] * lda + rstep * e + rpar); };
        T chunk[kCols] = {T(0), T(0)};
        auto fetch = [&](int p0, T (&v)[kCols]) -> bool {
            const int p = p0 + i;
            const int need = min(p0 + kChunk - 1, R) - npa_own + 1;
            if (need > 0 && !wait_prog(sh, a.prog + split_in, need, prog_seen, spin)) return false;
#pragma unroll
            for (int c = 0; c < kCols; ++c)
                v[c] = (p <= R && colv[c] >= 0)
                           ? __hip_atomic_load(aptr(c, row_of(p)), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)
                           : T(0);
            return true;
        };
        auto put = [&](int p0, const T (&v)[kCols]) {
            const int p = p0 + i;
            if (p <= R) in_ring[(p + off) % kZ][r] = Pair<T>{v[0], v[1]};
        };

        if (polled) {
            T v[kCols];
            ok = fetch(0, v);
            put(0, v);
            ok = ok && fetch(kChunk, chunk);
        } else {
            // (a band after the first takes at most B positions from A)
            const int n0 = first ? min(npa, kRowsAhead) : npa;
            for (int p = 0; p < n0; p += kRowsDma) dma_rows(p);
        }

        // where the lane reads the entries of sequence s for column c: with
        // MASK 1 column 0 of a row carries the row's mask (column 1's when
        // column 0 is absent)
        constexpr int MC = MASK == 2 ? kCols : 1;
        unsigned sc_at[S][MC];
#pragma unroll
        for (int s = 0; s < S; ++s)
#pragma unroll
            for (int c = 0; c < MC; ++c) {
                const int q = gbase + S * i + s;
                const int k = MASK == 1 && colv[0] < 0 ? 2 * r + 1 : 2 * r + c;
                const bool on = MASK == 0 || (q >= cv.glo[k] && q <= cv.ghi[k]);
                sc_at[s][c] = lds_addr(on ? &sh.scr[g][0][0] : &sh.ident[0][0]) +
                              (unsigned)(lane_entry(i) + s * kSlotStride) * (unsigned)sizeof(Pair<T>);
            }
        auto read_sc = [&](int slot, SC<MC> &sc, unsigned at = 0) {
#pragma unroll
            for (int s = 0; s < S; ++s)
#pragma unroll
                for (int c = 0; c < MC; ++c) {
                    // (MASK 0: one address, the slots by constant offsets)
                    const Lds<Pair<T>> *q = MASK == 0 ? lds_at<Pair<T>>(sc_at[0][0] + at) + s * kSlotStride
                                                   : lds_at<Pair<T>>(sc_at[s][c] + at);
                    sc.p[s][c] = q[slot * kLanes * S];
                }
        };

        // ---- a block's outputs: lane i of each row holds output u =
        // i / 4 + 4 (i % 2) of column (i / 2) % 2
        const int out_u = (i >> 2) + 4 * (i & 1), out_c = (i >> 1) & 1;
        const int ocol = out_c ? colv[1] : colv[0];
        T outv[2][kCols];
#pragma unroll
        for (int c = 0; c < kCols; ++c) outv[0][c] = outv[1][c] = T(0);
        // its row of A in the block that starts at step 0
        T *out_a = A + ((long long)max(ocol, 0) * lda + rpar + rstep * row_of(0) + astep * (out_u - kLag - off));
        const unsigned out_lane = lds_addr(out_ring) + (unsigned)(r * kCols + out_c) * (unsigned)sizeof(T);

        // ---- the events between blocks: input slots the next block reads
        // ahead must be in the ring, slots its outputs go to read by the next
        // band, or (LINK) another part's rows read from A.
        int avail_seen = 0, freed_seen = 0;  // last counter values read (global slots)
        int t_chunk = polled && kChunk <= R ? 0 : kNever;                // next chunk of another part's rows
        auto in_event = [&]() {  // first block that needs more than the slots known to be there
            const int have = max(npa + off, avail_seen - in_base);
            return have > slots ? kNever : have - (kU - 1 + kDin);
        };
        auto out_event = [&]() {  // first block whose outputs need more than the slots known to be free
            const int have = freed_seen - out_base + kZ - out_off;  // positions below this may be written
            return last || have > ring_hi ? kNever : max(have + kLag + off - (kU - 1), kLag);
        };
        int t_in = in_event(), t_out = out_event();
        auto event = [&](int t0) -> bool {
            if (LINK && t0 >= t_chunk) {
                put(t0 + kChunk, chunk);
                if (!fetch(t0 + 2 * kChunk, chunk)) return false;
                t_chunk = t0 + 2 * kChunk <= R ? t0 + kChunk : kNever;
            }
            if (t0 >= t_in) {
                if (!wait_ge(sh, avail, in_base + min(t0 + kU - 1 + kDin, slots) + 1, avail_seen, spin)) return false;
                t_in = in_event();
            }
            if (t0 >= t_out) {
                if (!wait_ge(sh, freed, out_base + min(t0 - kLag - off + kU - 1, ring_hi) + out_off - kZ + 1, freed_seen, spin))
                    return false;
                t_out = out_event();
            }
            return true;
        };

        // ---- input prefetch: slots 0 .. kDin-1, table entries of steps 0 ..
        // kAhead-1; the DMAs of the first rows are waited for here
        Pair<T> inbuf[kDin];
        SC<MC> scn[kAhead];
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        if (ok && min(kDin - 1, slots) >= npa + off)
            ok = wait_ge(sh, avail, in_base + min(kDin - 1, slots) + 1, avail_seen, spin);
        asm volatile("" ::: "memory");
#pragma unroll
        for (int d = 0; d < kDin; ++d) inbuf[d] = in_ring[d][r];
#pragma unroll
        for (int d = 0; d < kAhead; ++d) read_sc(d, scn[d]);

        T Y[S][kCols], E[S][kCols];
        Applied<MC> ap;  // the step before's: Y = 0 * 0 + 0 * Y at first
#pragma unroll
        for (int s = 0; s < S; ++s)
#pragma unroll
            for (int c = 0; c < kCols; ++c) {
                Y[s][c] = E[s][c] = ap.x[s][c] = T(0);
                ap.sc.p[s][c % MC] = Pair<T>{T(0), T(0)};
            }

        const unsigned m0_base = uniform(lds_addr(&sh.scr[g][0][0]));
        const int total = (slots + kLag + kU) & ~(kU - 1);  // the last position is stored in step slots + kLag
        // the last block of the table (identities, as all past the band's
        // steps): FP32 reads two blocks ahead, past the table's end at the last
        // steps, and takes this one there; FP64's one stays inside
        const int t_tab = uniform(band->steps) + FTAMD_SYS_PREFETCH - kU + off;
        static_assert(kD > kU || kLag + kU + kD <= kOutDelay + 1 + FTAMD_SYS_PREFETCH, "table reads past the table");
        const int in_free_end = in_base + span(R, off);
        constexpr unsigned kSlotBytes = sizeof(Pair<T>[kRows]);
        const unsigned in_lane = in_lds + (unsigned)r * (unsigned)sizeof(Pair<T>);
        const unsigned pub_lds = lds_addr(&sh.pub[g + 1]);
        // the blocks whose outputs all go to the next band's ring, or (of a
        // chain's last band) all to A: steps t_same .. t_same + n_same - 1
        const int t_same = (kLag + off + kU - 1) & ~(kU - 1);
        const int n_same = max(0, ((last ? R : ring_hi) + 1 + kLag + off - t_same) & ~(kU - 1));
        const unsigned out_slot0 = (unsigned)(out_off - kLag - off + out_u);  // slot of the lane's output, less t0
        const bool out_on = ocol >= 0;
        int pub_freed = in_base, pub_avail = out_base;
        unsigned pin = in_lane;                        // ring slot of position t0
        asm volatile("" : "+v"(pin));

        // Steps run in blocks of kU.
        for (int t0 = 0, t_event = 0;;) {
            if (t0 >= t_event) {
                if (t0 >= total) break;
                if (!ok || !event(t0)) {
                    fail(sh);
                    atomicOr(a.ctl + FTAMD_SYS_CTL_ERR, FTAMD_ERR_TIMEOUT);
                    return false;
                }
                t_event = min(min(t_in, t_out), LINK ? min(t_chunk, total) : total);
            }
            if (END & kFirst) {
                // the block's share of the rows from A (see kExtra)
                const int p0 = t0 + kRowsAhead;
                if (first && !polled && p0 < npa) {
#pragma unroll
                    for (int q = 0; q < kU; q += kRowsDma) {
                        if (q == 0 || p0 + q < npa) dma_rows(p0 + q);
                        else dma_filler(sh, tab_band, lane16);
                    }
                } else {
#pragma unroll
                    for (int q = 0; q < kU; q += kRowsDma) dma_filler(sh, tab_band, lane16);
                }
            }
            // the addresses of the block's LDS accesses: ring slots of the
            // reads (the last kDin steps read the next block's), table slots,
            // DMA targets
            const unsigned tab0 = kD == kU ? 0u : (unsigned)(t0 % kD) * kStepBytes;
            const unsigned tab1 = kD == kU ? 0u : (unsigned)((t0 + kU) % kD) * kStepBytes;
            set_m0(m0_base + tab0);
            // step t0+kD+K: the DMA of step u, K = u+1-kSPD
            const char *src = tab_band + (long long)(kD > kU ? min(t0 + kD, t_tab) : t0 + kD) * kStepBytes;
            const unsigned pin_next = in_lane + ((unsigned)(t0 + kU) % kZ) * kSlotBytes;
#pragma unroll
            for (int u = 0; u < kU; ++u) {
                // keep each step's instructions together: the entries and
                // rows read for the steps after next then have two steps of
                // issue time to arrive before their first use
                __builtin_amdgcn_sched_barrier(0);
                const Pair<T> in = inbuf[u % kDin];
                inbuf[u % kDin] = u + kDin >= kU ? lds_at<Pair<T>>(pin_next)[(u + kDin - kU) * kRows]
                                                 : lds_at<Pair<T>>(pin)[(u + kDin) * kRows];
                const SC<MC> sc = scn[u % kAhead];
                if ((u + kAhead) % kSPD == 0) {
                    // from the second DMA of the block on, its own are the youngest
                    if (u < kU - kSPD) wait_block<kExtra>();
                    else wait_block();
                }
                read_sc((u + kAhead) % kU, scn[u % kAhead], u + kAhead < kU ? tab0 : tab1);
                // the reads above are issued before the step's arithmetic
                __builtin_amdgcn_sched_barrier(0);
                T X0[kCols];
#pragma unroll
                for (int c = 0; c < kCols; ++c) X0[c] = shift_in(c == 0 ? in.x : in.y, E[S - 1][c]);
                // the last sequence's outputs of the step before
#pragma unroll
                for (int c = 0; c < kCols; ++c) {
                    T &k = outv[u >> 2][c];
                    switch (u & 3) {  // a constant once the loop is unrolled
                        case 0: k = row_end<0>(k, E[S - 1][c]); break;
                        case 1: k = row_end<1>(k, E[S - 1][c]); break;
                        case 2: k = row_end<2>(k, E[S - 1][c]); break;
                        default: k = row_end<3>(k, E[S - 1][c]); break;
                    }
                }
                carry(Y, ap);
                emit(Y, E, X0, sc, ap);
                if (u % kSPD == kSPD - 1) {
                    // u is a constant once the loop is unrolled
                    switch (u + 1 - kSPD) {
                        case 0: dma_block_at<0>(src, lane16, E[S - 1][0]); break;
                        case 2: dma_block_at<2>(src, lane16, E[S - 1][0]); break;
                        case 4: dma_block_at<4>(src, lane16, E[S - 1][0]); break;
                        case 6: dma_block_at<6>(src, lane16, E[S - 1][0]); break;
                        default: break;
                    }
                }
            }
            pin = pin_next;
            // a split part's last band publishes the rows the previous block
            // stored: they are complete once at most this block's DMAs are
            // outstanding (vector memory operations complete in issue order)
            if (LINK && split_out >= 0 && pub > published) {
                asm volatile("s_waitcnt vmcnt(%0)" ::"n"(kU / kSPD) : "memory");
                if (lane == 0) __hip_atomic_store(a.prog + split_out, pub, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                published = pub;
            }
            // the block's outputs, positions po0 .. po0+kU-1: to the next
            // band's ring up to ring_hi, else (leaving the chain or the part)
            // to their rows of A; positions outside [0, R] carry no row
            const T ve = (i & 1) ? outv[1][0] : outv[0][0];
            const T vo = (i & 1) ? outv[1][1] : outv[0][1];
            const T v = out_c ? vo : ve;
            if (!LINK && (unsigned)(t0 - t_same) < (unsigned)n_same) {
                if (END & kLast && last) {
                    if (out_on) *out_a = v;
                } else {
                    *lds_at<T>(out_lane + ((unsigned)t0 + out_slot0) % kZ * kSlotBytes) = v;
                    pub_avail = out_base + (t0 + kU - kLag - off) + out_off;
                    if (END & kLast) dma_filler(sh, tab_band, lane16);
                }
            } else {
                const int po0 = t0 - kLag - off, po = po0 + out_u;
                if (po0 + kU > 0) {
                    if (po >= 0 && po <= R) {
                        if (po <= ring_hi) {
                            out_ring[(((po + out_off) & (kZ - 1)) * kRows + r) * kCols + out_c] = v;
                        } else if (out_on) {
                            if (split_out >= 0) __hip_atomic_store(out_a, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                            else *out_a = v;
                        }
                    }
                    if (ring_hi >= 0) pub_avail = max(pub_avail, out_base + min(po0 + kU - 1, ring_hi) + out_off + 1);
                    pub = max(0, min(po0 + kU, R + 1));
                }
                // unless some lane stored a row of A
                if (END & kLast && max(max(po0, ring_hi + 1), 0) > min(po0 + kU - 1, R)) dma_filler(sh, tab_band, lane16);
            }
            out_a += astep * kU;
            t0 += kU;
            // publish what the block read (never beyond this chain's part of
            // the ring) and wrote
            pub_freed = min(in_base + t0, in_free_end);
            asm volatile("s_mov_b64 exec, 1\n\tds_write2_b32 %0, %1, %2 offset1:1\n\ts_mov_b64 exec, -1"
                         :
                         : "v"(pub_lds), "v"(pub_freed), "v"(pub_avail)
                         : "memory");
        }

        if (LINK && split_out >= 0) {
            // every row stored and complete
            asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
            if (lane == 0) __hip_atomic_store(a.prog + split_out, R + 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        }
        return true;
    }

    // Ring slots one band's stream takes: its R + 1 positions from slot `off`
    // on, rounded up to whole rings, so that every stream starts at ring slot 0.
    __device__ static int span(int R, int off) { return (R + off + kZ) / kZ * kZ; }

    // Idle steps (and ring slots) before position 0 of the stream of a part's
    // band w.  A block needs input up to kDin slots past its own; with kDin
    // more idle steps than the band before, that is where a block of the band
    // before ends, and it follows that band by kLag + kU + kDin steps (without,
    // by up to kU - kDin more).
    __device__ static int idle(int w) { return (kDin * w) & (kU - 1); }

    // XCD (accelerator complex die, with its own L2) this workgroup runs on.
    __device__ static int xcd_id(int nxcd) {
        const int id = (int)__builtin_amdgcn_s_getreg((20) | (0 << 6) | ((4 - 1) << 11));  // HW_REG_XCC_ID[3:0]
        return nxcd > 1 ? id % nxcd : 0;
    }

    // A workgroup takes the slots of its XCD in order (tickets), and streams
    // a slot's chain parts (items) one after another through its waves: item
    // k runs its part's bands on waves wave0 .. wave0+nb-1, and every wave
    // takes the items in list order, so a wave starts its band of the next
    // part as soon as it has finished its band of the previous one.  A part
    // that waits on another part waits on an earlier slot of the same XCD,
    // which a running workgroup holds or has finished: the launch completes
    // however many workgroups the hardware runs at once.
    __device__ static void run(const FtamdSysLaunch &a, Shared &sh) {
        {
            T *rp = (T *)&sh.ring[0][0][0];
            for (int x = threadIdx.x; x < kWaves * kZ * kRows * kCols; x += blockDim.x) rp[x] = T(0);
            Pair<T> *id = &sh.ident[0][0];
            for (int x = threadIdx.x; x < kD * kLanes * S; x += blockDim.x) id[x] = Pair<T>{T(0), T(1)};
            if (threadIdx.x < kWaves + 2) sh.pub[threadIdx.x].freed = sh.pub[threadIdx.x].avail = 0;
            if (threadIdx.x == 0) sh.abort_flag = 0;
        }
        const int lane = threadIdx.x & 63;
        const int g = uniform(threadIdx.x >> 6);
        const int x = uniform(xcd_id(a.nxcd));
        const int s0 = uniform(a.xcd_slot[x]), ns = uniform(a.xcd_slot[x + 1]) - s0;
        unsigned *ticket = (unsigned *)(a.ctl + FTAMD_SYS_CTL_TICKET) + x;
        int in_base = 0, out_base = 0;  // where the current part's streams start in rings g and g+1
        for (;;) {
            __syncthreads();
            if (threadIdx.x == 0) sh.slot = (int)atomicAdd(ticket, 1u);
            __syncthreads();
            const int t = uniform(lds_ld(&sh.slot));
            if (t >= ns || uniform(lds_ld(&sh.abort_flag))) break;
            const int slot = s0 + t;
            const ConstInt *slot_items = (const ConstInt *)(uintptr_t)a.slot_items;
            const int it0 = slot_items[slot], it1 = slot_items[slot + 1];
            for (int it = it0; it < it1; ++it) {
                const ConstItem &item = ((const ConstItem *)(uintptr_t)a.items)[it];
                const int chain = uniform(item.chain);
                const ConstChain &ch = ((const ConstChain *)(uintptr_t)a.chains)[chain];
                const int nb = uniform(ch.nb), b0 = uniform(ch.band0);
                const int w = g - uniform(item.wave0);  // this wave's band of the part, if any
                if (w < -1 || w >= nb) continue;
                const ConstBand *bands = (const ConstBand *)(uintptr_t)a.bands + b0;
                if (w >= 0) {
                    switch (uniform(ch.prio)) {
                        case 3: __builtin_amdgcn_s_setprio(3); break;
                        case 2: __builtin_amdgcn_s_setprio(2); break;
                        case 1: __builtin_amdgcn_s_setprio(1); break;
                        default: __builtin_amdgcn_s_setprio(0); break;
                    }
                    // a band needs masks if some column of the chain does
                    // not apply some of its sequences; with ROWMASK one mask
                    // per lane row serves both columns (sph and disk: the two
                    // columns of a row are the cosine and sine columns of one
                    // order, so they apply the same sequences)
                    const int gbase = uniform(bands[w].gbase);
                    const int glast = gbase + uniform(bands[w].nseq) - 1;
                    bool masked = false;
#pragma unroll
                    for (int k = 0; k < FTAMD_SYS_COLS; ++k)
                        masked |= ch.col[k] >= 0 && (ch.glo[k] > gbase || ch.ghi[k] < glast);
                    // the kinds of bands run their own instantiations, so
                    // that each carries only its own code
                    const bool link = (w == 0 && uniform(ch.split_in) >= 0) || (w == nb - 1 && uniform(ch.split_out) >= 0);
                    constexpr int MK = ROWMASK ? 1 : 2;
                    const FtamdSysChain &cv = a.chains[chain];
                    const bool f = w == 0, l = w == nb - 1;
                    bool ok;
#define FTAMD_RUN_BAND(mask, end, lk) run_band<mask, end, lk>(a, sh, ch, cv, w, g, lane, in_base, out_base)
                    if (link) ok = FTAMD_RUN_BAND(MK, kBoth, true);
                    else if (masked && f && !l) ok = FTAMD_RUN_BAND(MK, kFirst, false);
                    else if (masked && l && !f) ok = FTAMD_RUN_BAND(MK, kLast, false);
                    else if (masked) ok = FTAMD_RUN_BAND(MK, kBoth, false);
                    else if (f) ok = l ? FTAMD_RUN_BAND(0, kBoth, false) : FTAMD_RUN_BAND(0, kFirst, false);
                    else ok = l ? FTAMD_RUN_BAND(0, kLast, false) : FTAMD_RUN_BAND(0, kInner, false);
#undef FTAMD_RUN_BAND
                    if (!ok) break;
                    const int R = uniform(bands[w].R);
                    in_base += span(R, idle(w));
                }
                if (w + 1 < nb) {
                    const int R = uniform(bands[w + 1].R);
                    out_base += span(R, idle(w + 1));
                }
            }
            __builtin_amdgcn_s_setprio(0);
            __syncthreads();
            if (threadIdx.x == 0 && !lds_ld(&sh.abort_flag)) atomicAdd((unsigned *)(a.ctl + FTAMD_SYS_CTL_COMPLETED), 1u);
        }
        // The last workgroup out checks that every slot ran and resets the
        // tickets, counters and progress words for the next launch (or graph
        // replay).
        __syncthreads();
        if (threadIdx.x == 0) {
            unsigned *done = (unsigned *)(a.ctl + FTAMD_SYS_CTL_DONE);
            unsigned *completed = (unsigned *)(a.ctl + FTAMD_SYS_CTL_COMPLETED);
            const unsigned d = __hip_atomic_fetch_add(done, 1u, __ATOMIC_ACQ_REL, __HIP_MEMORY_SCOPE_AGENT);
            if (d == gridDim.x - 1) {
                if (__hip_atomic_load(completed, __ATOMIC_ACQUIRE, __HIP_MEMORY_SCOPE_AGENT) != (unsigned)a.nslots)
                    atomicOr(a.ctl + FTAMD_SYS_CTL_ERR, FTAMD_ERR_INCOMPLETE);
                for (int k = 0; k < a.nprog; ++k)
                    __hip_atomic_store(a.prog + k, 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                for (int k = 0; k < a.nxcd; ++k)
                    __hip_atomic_store((unsigned *)(a.ctl + FTAMD_SYS_CTL_TICKET) + k, 0u, __ATOMIC_RELAXED,
                                       __HIP_MEMORY_SCOPE_AGENT);
                __hip_atomic_store(completed, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                __hip_atomic_store(done, 0u, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_AGENT);
            }
        }
    }
};

template <typename T, int S, bool ROWMASK>
__global__ void __launch_bounds__(kWaves * 64) sys_kernel(FtamdSysLaunch a) {
    using E = Engine<T, S, ROWMASK>;
    __shared__ typename E::Shared sh;
    E::run(a, sh);
}

}  // namespace ftsys
