// sor_resident.h -- a Poisson solve as one kernel whose tiles stay in registers from sweep to sweep.
//
// sor_rb.h advances the grid S sweeps per launch; at 1024^2 about half of such a launch is the
// kernel boundary, the tile loads and the stores.  Here one workgroup per tile stays on the GPU
// for a whole solve (up to `epochs` epochs of S sweeps): after each epoch it publishes the cells
// of its tile that other tiles hold in their halos and takes its own halo's cells from them.
//
// Exchange.  The cells go through three planes in device memory (epoch e's through plane e % 3)
// whose cells hold a mark -- a signalling NaN, which no arithmetic result is -- until they are
// written: a reader loads its halo cells again until none is marked, so data and "ready" travel
// together, in one trip.  Once all waves of a tile have taken epoch e+1's cells, the tile's own cells
// of epoch e have been read by everyone: each tile that reads them is one whose cells it reads, and
// that one published e+1 after all its waves had taken e.  A wave by itself knows less -- one whose
// rows are all owned takes nothing from above and below, where its rows may be read -- so the cells
// are marked again behind the first barrier of the next epoch's sweeps, which every wave reaches
// after its take.  The plane is used next by the publication at the end of the epoch after that one,
// so the marks are in place before a reader can look for it (the wait before a publication orders
// the tile's own marks before it, and a reader takes that one before it looks for the next).
//
// Coherence.  The 8 XCDs have an L2 each.  Reads are agent-scope loads, which see what the XCD's own
// L2 holds for it and what other XCDs have written through.  Tile rows are dealt to the XCDs in
// contiguous bands, and each workgroup takes the next free tile of the band of the XCD it finds
// itself on (workgroups are dealt to the XCDs round-robin, so every band gets as many as it has
// tiles; if one did not, its neighbours' waits would run out; where whole tile rows leave too many
// CUs empty, an eighth of all tiles takes the place of a band), so most cells are read on the XCD that
// wrote them: these are stored plainly, into that L2; only the rows another band reads are
// written through (agent-scope stores).  Writing every cell through measured 5.9 us per exchange
// at 1024^2 with (5, 16, 4) tiles, this split 3.0; polling flags instead of the data 10.8.
//
// Decision.  As in sor_rb.h one extra workgroup decides (sor_resident_decider): it takes the
// tiles' per-sweep sums of epoch e (marked cells again), decides as sor_rb_decider does, with the
// same sums in the same order, and leaves each tile a decision word.  The tiles read it one epoch
// later, so it costs them nothing; they keep their values of the last two epochs' starts and go
// back to them: a solve ends with the iterate of exactly the first sweep with e < tol
// (src/poisson.c:273).  The values are kept in LDS where the tile is small, else in device memory
// and then only while the last decided update is within kNearTol of ending the solve (keeping them
// always cost 1.0 of 8.2 us per epoch at 1024^2): a solve that ends from further out is run
// again from the kernel's input plane to exactly its last sweep.
//
// Waiting.  All workgroups of the launch must be on the GPU together; the host launches only what
// fits beside the other resident solves of the process.  Every wait is bounded all the same: a
// wave that runs out of polls reports it, waits no more, and the kernel ends; the host then
// repeats the epochs with sor_rb.h's launches from the kernel's input plane, which it never writes.
#pragma once

#include <vector>

#include "sor_rb.h"

namespace cnv {

typedef unsigned long long u64;
constexpr double kNearTol = 4.0;     // an update within this factor of its tolerance may end the solve soon
constexpr int kAgent = 16;           // cache policy bits of buffer accesses: sc1, agent scope

template <typename T> struct Marked;
template <> struct Marked<double> {
    typedef unsigned raw __attribute__((ext_vector_type(4)));
    static __device__ __forceinline__ bool ready(double x) { return (u64)__double_as_longlong(x) != kMark64; }
    static __device__ __forceinline__ double mark() { return __longlong_as_double((long long)kMark64); }
};
template <> struct Marked<float> {
    typedef unsigned raw __attribute__((ext_vector_type(2)));
    static __device__ __forceinline__ bool ready(float x) { return (unsigned)__float_as_int(x) != kMark32; }
    static __device__ __forceinline__ float mark() { return __int_as_float((int)kMark32); }
};

// A pair of cells of the exchange planes: soff (wave-uniform) + voff bytes from the buffer's start.
template <typename T>
__device__ __forceinline__ void exch_load(__amdgpu_buffer_rsrc_t rs, int voff, int soff, T& x0, T& x1) {
    typename Marked<T>::raw d;
    if constexpr (sizeof(T) == 8) d = __builtin_amdgcn_raw_buffer_load_b128(rs, voff, soff, kAgent);
    else d = __builtin_amdgcn_raw_buffer_load_b64(rs, voff, soff, kAgent);
    T x[2];
    __builtin_memcpy(x, &d, sizeof(d));
    x0 = x[0];
    x1 = x[1];
}
template <typename T, int POLICY>
__device__ __forceinline__ void exch_store(__amdgpu_buffer_rsrc_t rs, int voff, int soff, T x0, T x1) {
    const T x[2] = {x0, x1};
    typename Marked<T>::raw d;
    __builtin_memcpy(&d, x, sizeof(d));
    if constexpr (sizeof(T) == 8) __builtin_amdgcn_raw_buffer_store_b128(d, rs, voff, soff, POLICY);
    else __builtin_amdgcn_raw_buffer_store_b64(d, rs, voff, soff, POLICY);
}
__device__ __forceinline__ u64 agent_load(const u64* p) { return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT); }
__device__ __forceinline__ void agent_store(u64* p, u64 x) { __hip_atomic_store(p, x, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT); }
__device__ __forceinline__ void report_abort(const SorResident& r) {
    __hip_atomic_store(r.abort, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ void report_source(const SorResident& r) {
    __hip_atomic_store(r.abort + 1, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ bool gave_up(const SorResident& r) {
    return __builtin_amdgcn_readfirstlane(__hip_atomic_load(r.abort, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)) != 0;
}
// every memory operation this wave has issued is complete
__device__ __forceinline__ void wait_memory() {
    __atomic_signal_fence(__ATOMIC_SEQ_CST);
    __builtin_amdgcn_s_waitcnt(0x0f70);  // vmcnt(0)
    __atomic_signal_fence(__ATOMIC_SEQ_CST);
}

// LDS that lanes of one wave hand to one another: what was written before is read after, and not overwritten sooner
__device__ __forceinline__ void wave_lds() {
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront", "local");
    __builtin_amdgcn_wave_barrier();
}

// a decision word: the number of decided epochs, whether the end is near after the last of them and
// after the one before, what to do, sweeps to redo
enum ResidentCode : unsigned { RES_CONTINUE = 0, RES_END = 1, RES_REDO = 2, RES_RERUN = 3 };
__device__ __forceinline__ u64 res_word(int decided, bool near, bool near_before, unsigned code, int redo) {
    return ((u64)(unsigned)decided << 32) | ((unsigned)near_before << 17) | ((unsigned)near << 16) | (code << 8) |
           (unsigned)redo;
}

typedef double SnapPair __attribute__((ext_vector_type(2)));
// pairs of the two kept epoch starts in LDS
template <typename T, int NW, int RB>
constexpr int kSnapPairs = sizeof(T) == 8 && resident_snap_lds(NW, RB) ? 2 * RB * NW * 64 : 1;

// the largest share of rb rows that has at most `most`
constexpr int chunk_rows(int rb, int most) {
    int rows = rb < most ? rb : most;
    while (rb % rows) --rows;
    return rows;
}

// The rows of a band [row_lo, row_hi) of tile rows that other bands read: below lo or from hi on.
template <typename Tile, typename T>
__device__ __forceinline__ int band_lo(const SorArgs<T>& a, int row_lo) { return row_lo > 0 ? row_lo * Tile::TI + Tile::H : 0; }
template <typename Tile, typename T>
__device__ __forceinline__ int band_hi(const SorArgs<T>& a, int row_hi) {
    return row_hi < a.tiles_i ? row_hi * Tile::TI - Tile::H : a.nr;
}

// One tile's workgroup: tile (ti, tj); grid rows below lo or from hi on are read on other XCDs;
// snap_part: which part of r.snap is its own.
template <typename T, int S, int NW, int RB, bool GS, bool XR, bool NORM, bool ISO = false>
__device__ __forceinline__ void sor_resident_tile(const SorArgs<T>& a, const SorResident& r, const int ti, const int tj,
                                                  const int lo, const int hi, const int snap_part,
                                                  typename SorTile<T, S, NW, RB, GS, XR, NORM>::Shared& sh,
                                                  SnapPair* const snap_lds) {
    typedef SorTile<T, S, NW, RB, GS, XR, NORM, ISO> Tile;
    constexpr int H = Tile::H, TI = Tile::TI, TJ = Tile::TJ;
    constexpr bool kSnap = sizeof(T) == 8;
    constexpr bool kSnapLds = kSnap && resident_snap_lds(NW, RB);
    typedef SnapPair Two;
    constexpr bool kThick = NW * RB >= 96 && H <= RB;

    const int tile = ti * a.tiles_j + tj;
    const SorCtl* P = a.ctl + r.rslot;
    if (P->status != SOR_RUNNING) return;
    const int itmax = r.stop > 0 ? r.stop : P->itmax;
    int k = P->k;
    Tile t;
    t.place(a, ti, tj);
    t.load(a, sor_plane(a, r.src), sh);
    t.fix_odd_edge();
    if constexpr (sizeof(T) == 8) {
        if (!__all(t.f_exact)) report_source(r);
    }
    const bool owns = t.owns_rows();

    // pairs of this lane's columns, and which rows' pairs it takes from or gives to other tiles
    const bool inside = t.gj >= 0 && t.gj < t.nc;
    const bool owncol = t.ownc[0];
    const bool ringcol = owncol && (2 * t.lane < 2 * H || 2 * t.lane >= TJ);
    const int pitch = r.ldx * (int)sizeof(T);
    const int plane = (int)(r.xplane * (long long)sizeof(T));
    const __amdgpu_buffer_rsrc_t rs = __builtin_amdgcn_make_buffer_rsrc(r.exch, 0, 3 * plane, 0x00027000);
    // The rows' masks and addresses are held through the sweeps (worked out anew at every exchange they
    // cost 10% of a sweep at 64^2); where the source term is in LDS their registers are needed, and those of
    // what a tile gives and what it does with what it took are worked out when it does.
    auto row_now = [&]() -> int {
        if constexpr (Tile::RF == RB) return t.row0;
        int row0 = __builtin_amdgcn_readfirstlane(t.row0);
        asm volatile("" : "+s"(row0));
        return row0;
    };
    auto own_row = [&](int row0, int rr) {
        const int li = row0 + rr;
        return li >= H && li < H + TI && t.gi0 + li < t.nr;
    };
    auto takes = [&](int row0, int rr) {
        const int gi = t.gi0 + row0 + rr;
        return gi >= 0 && gi < t.nr && inside && !(own_row(row0, rr) && owncol);
    };
    auto gives = [&](int row0, int rr) {
        const int li = row0 + rr;
        return own_row(row0, rr) && (li < 2 * H || li >= TI ? owncol : ringcol);
    };
    // Columns.  A wave whose rows are all owned takes only S pairs at each end of a row, and gives only
    // the S next to them unless its rows are read from above or below: 10 of 64 lanes.  A memory
    // instruction costs its 16 cycles whatever its lanes do, so such a wave handles kRows rows with
    // one: lane m takes pair m % kPairs of row m / kPairs, and the values change lanes through the
    // wave's part of the half-sweeps' exchange rows (xch[1], which nobody reads between the last
    // half-sweep and the next epoch's first barrier).  1024^2: FP32 0.97 -> 0.91 us per sweep, FP64
    // 1.46 -> 1.45; with two rows a wave the detour costs more than the one instruction saved (3% at
    // 64^2), and so it does on 12 waves in FP64 (2% at 600^2).
    constexpr int kPairs = 2 * S;
    constexpr int kRows = chunk_rows(RB, 64 / kPairs);
    static_assert(kRows * kPairs <= 64 && RB % kRows == 0, "a chunk of rows is one pair a lane");
    typedef T Pair2 __attribute__((ext_vector_type(2)));
    Pair2* const stage = reinterpret_cast<Pair2*>(sh.xch[1][t.wv][0]);  // 64 pairs
    struct Column {  // this lane's pair of a chunk: there is one, and its offset
        bool has;
        int voff;
    };
    // (offsets are worked out when they are used: held through the sweeps they cost registers those need)
    auto lane_now = [&]() -> int {
        int m = threadIdx.x & 63;
        if constexpr (RB > 2) asm volatile("" : "+v"(m));
        return m;
    };
    auto row_offset = [&]() -> int { return (t.gj0 + 2 * lane_now()) * (int)sizeof(T); };
    auto column = [&](bool taken) -> Column {
        const int m = lane_now();
        const int mr = m / kPairs, mj = m - mr * kPairs;
        const int at = taken ? (mj < S ? mj : 64 - kPairs + mj) : (mj < S ? S + mj : 64 - 3 * S + mj);
        const int gj = t.gj0 + 2 * at;
        return Column{mr < kRows && gj >= 0 && gj < t.nc, mr * pitch + gj * (int)sizeof(T)};
    };
    constexpr bool kColumns = RB >= 4 && (sizeof(T) == 4 || NW != 12 || RB > 4);
    bool all_own = kColumns, no_ring = kColumns;  // wave-uniform
#pragma unroll
    for (int rr = 0; rr < RB; ++rr) {
        const int li = t.row0 + rr;
        all_own = all_own && own_row(t.row0, rr);
        no_ring = no_ring && own_row(t.row0, rr) && li >= 2 * H && li < TI;
    }
    auto give = [&](int slot, bool marks) __attribute__((always_inline)) {
        T mk = Marked<T>::mark();
        if constexpr (RB > 2) asm volatile("" : "+v"(mk));
        const int row0 = row_now();
        if (no_ring) {
            const bool through = t.gi0 + row0 < lo || t.gi0 + row0 + RB > hi;
            const Column col = column(false);
#pragma unroll
            for (int c = 0; c < RB; c += kRows) {
                Pair2 d = {mk, mk};
                if (!marks) {
                    // lanes S .. 2S-1 hold the left pairs, 64-2S .. 64-S-1 the right ones
                    const int m = lane_now();
                    const bool at_left = m < 2 * S;
                    const int j = at_left ? m - S : m - 64 + 3 * S;
                    if (j >= (at_left ? 0 : S) && j < kPairs) {
#pragma unroll
                        for (int rr = 0; rr < kRows; ++rr) stage[rr * kPairs + j] = Pair2{t.v[0][c + rr], t.v[1][c + rr]};
                    }
                    wave_lds();
                    d = stage[lane_now()];
                    wave_lds();
                }
                const int soff = slot * plane + (t.gi0 + row0 + c) * pitch;
                if (col.has) {
                    if (through) exch_store<T, kAgent>(rs, col.voff, soff, d.x, d.y);
                    else exch_store<T, 0>(rs, col.voff, soff, d.x, d.y);
                }
            }
            return;
        }
        const int voff = row_offset();
#pragma unroll
        for (int rr = 0; rr < RB; ++rr) {
            const int gi = t.gi0 + row0 + rr;
            if (!gives(row0, rr)) continue;
            const T x0 = marks ? mk : t.v[0][rr], x1 = marks ? mk : t.v[1][rr];
            if (gi < lo || gi >= hi) exch_store<T, kAgent>(rs, voff, slot * plane + gi * pitch, x0, x1);
            else exch_store<T, 0>(rs, voff, slot * plane + gi * pitch, x0, x1);
        }
    };

    bool dead = gave_up(r);  // a batch's kernel goes on to other tiles after a wave has given up
    const u64* dec = r.dec + (size_t)tile * 8;
    // Thick tiles (H <= RB): halo rows are the first H of wave 0 and the last H of wave NW - 1; every
    // wave takes the columns of its owned rows by chunks.  What is under way then needs registers for
    // H rows, and not for all RB beside the values they replace.
    auto take_thick = [&](int slot, int decided) __attribute__((always_inline)) -> u64 {
        u64 word = 0;
        struct {
            T x, y;
        } got[RB / kRows], row[H];
        const bool edge = t.wv == 0 || t.wv == NW - 1;
        for (int spins = 0;; ++spins) {
            bool ok = true;
            if (decided) word = agent_load(dec);
            if (slot >= 0) {
                const Column col = column(true);
                const int m = lane_now() / kPairs;
                const int first = t.gi0 + t.row0;
                if (edge && inside) {
                    const int voff = row_offset();
                    const int at = first + (t.wv == 0 ? 0 : RB - H);
#pragma unroll
                    for (int j = 0; j < H; ++j)
                        if (at + j >= 0 && at + j < t.nr) exch_load<T>(rs, voff, slot * plane + (at + j) * pitch, row[j].x, row[j].y);
                }
#pragma unroll
                for (int c = 0; c < RB / kRows; ++c)
                    if (col.has && own_row(t.row0, c * kRows + m)) exch_load<T>(rs, col.voff, slot * plane + (first + c * kRows) * pitch, got[c].x, got[c].y);
                if (edge && inside) {
                    const int at = t.gi0 + t.row0 + (t.wv == 0 ? 0 : RB - H);
#pragma unroll
                    for (int j = 0; j < H; ++j)
                        if (at + j >= 0 && at + j < t.nr) ok = ok && Marked<T>::ready(row[j].x) && Marked<T>::ready(row[j].y);
                }
#pragma unroll
                for (int c = 0; c < RB / kRows; ++c)
                    if (col.has && own_row(t.row0, c * kRows + m)) ok = ok && Marked<T>::ready(got[c].x) && Marked<T>::ready(got[c].y);
            }
            if (decided) ok = ok && (int)(word >> 32) >= decided;
            if (__all(ok) || dead) break;
            if (spins >= r.spins) {
                dead = true;
                report_abort(r);
            }
        }
        if (slot >= 0) {
            const int row0 = row_now();
            const int first = t.gi0 + row0;
#pragma unroll
            for (int rr = 0; rr < RB; ++rr) {
                const bool in = inside && first + rr >= 0 && first + rr < t.nr;
                if (rr < H) {
                    const bool top = in && t.wv == 0;
                    t.v[0][rr] = top ? row[rr < H ? rr : 0].x : t.v[0][rr];
                    t.v[1][rr] = top ? row[rr < H ? rr : 0].y : t.v[1][rr];
                }
                if (rr >= RB - H) {
                    const bool bottom = in && t.wv == NW - 1;
                    t.v[0][rr] = bottom ? row[rr >= RB - H ? rr - (RB - H) : 0].x : t.v[0][rr];
                    t.v[1][rr] = bottom ? row[rr >= RB - H ? rr - (RB - H) : 0].y : t.v[1][rr];
                }
            }
            const int m = lane_now();
            const int j = m < S ? m : m - 64 + kPairs;
#pragma unroll
            for (int c = 0; c < RB / kRows; ++c) {
                stage[m] = Pair2{got[c].x, got[c].y};
                wave_lds();
                if (inside && !owncol && j >= 0) {
#pragma unroll
                    for (int rr = 0; rr < kRows; ++rr) {
                        if (!own_row(row0, c * kRows + rr)) continue;
                        const Pair2 d = stage[rr * kPairs + j];
                        t.v[0][c * kRows + rr] = d.x;
                        t.v[1][c * kRows + rr] = d.y;
                    }
                }
                wave_lds();
            }
        }
        const unsigned hi32 = __builtin_amdgcn_readfirstlane((unsigned)(word >> 32));
        const unsigned lo32 = __builtin_amdgcn_readfirstlane((unsigned)word);
        return ((u64)hi32 << 32) | lo32;
    };
    // the halo cells of plane `slot` (slot < 0: none) and a decision on `decided` epochs (0: none)
    auto take_thin = [&](int slot, int decided) __attribute__((always_inline)) -> u64 {
        u64 word = 0;
        struct {
            T x, y;
        } got[RB / kRows];
        const Column col = column(true);
        const int voff = row_offset();
        for (int spins = 0;; ++spins) {
            bool ok = true;
            if (decided) word = agent_load(dec);
            if (slot >= 0 && all_own) {
                if (col.has) {
#pragma unroll
                    for (int c = 0; c < RB / kRows; ++c)
                        exch_load<T>(rs, col.voff, slot * plane + (t.gi0 + t.row0 + c * kRows) * pitch, got[c].x, got[c].y);
#pragma unroll
                    for (int c = 0; c < RB / kRows; ++c)
                        ok = ok && Marked<T>::ready(got[c].x) && Marked<T>::ready(got[c].y);
                }
            } else if (slot >= 0) {
#pragma unroll
                for (int rr = 0; rr < RB; ++rr)
                    if (takes(t.row0, rr)) exch_load<T>(rs, voff, slot * plane + (t.gi0 + t.row0 + rr) * pitch, t.v[0][rr], t.v[1][rr]);
#pragma unroll
                for (int rr = 0; rr < RB; ++rr)
                    if (takes(t.row0, rr)) ok = ok && Marked<T>::ready(t.v[0][rr]) && Marked<T>::ready(t.v[1][rr]);
            }
            if (decided) ok = ok && (int)(word >> 32) >= decided;
            if (__all(ok) || dead) break;
            if (spins >= r.spins) {
                dead = true;
                report_abort(r);
            }
        }
        if (slot >= 0 && all_own) {
            const int m = lane_now();
            const int j = m < S ? m : m - 64 + kPairs;
#pragma unroll
            for (int c = 0; c < RB / kRows; ++c) {
                stage[m] = Pair2{got[c].x, got[c].y};
                wave_lds();
                if (inside && !owncol && j >= 0) {
#pragma unroll
                    for (int rr = 0; rr < kRows; ++rr) {
                        const Pair2 d = stage[rr * kPairs + j];
                        t.v[0][c * kRows + rr] = d.x;
                        t.v[1][c * kRows + rr] = d.y;
                    }
                }
                wave_lds();
            }
        }
        const unsigned hi32 = __builtin_amdgcn_readfirstlane((unsigned)(word >> 32));
        const unsigned lo32 = __builtin_amdgcn_readfirstlane((unsigned)word);
        return ((u64)hi32 << 32) | lo32;
    };

    auto take = [&](int slot, int decided) __attribute__((always_inline)) -> u64 {
        if constexpr (kThick) return take_thick(slot, decided);
        else return take_thin(slot, decided);
    };

    // the values at an epoch's start, in two turns (FP64)
    Two* const mem = kSnapLds ? nullptr : reinterpret_cast<Two*>(r.snap) + (size_t)snap_part * 2 * RB * NW * 64;
    auto snap_at = [&](int turn, int rr) -> Two* {
        int m = threadIdx.x;
        asm volatile("" : "+v"(m));
        const int q = (turn * RB + rr) * NW * 64 + m;
        return kSnapLds ? snap_lds + q : mem + q;
    };
    auto keep = [&](int turn) {
        if constexpr (kSnap) {
#pragma unroll
            for (int rr = 0; rr < RB; ++rr) *snap_at(turn, rr) = Two{t.v[0][rr], t.v[1][rr]};
        }
    };
    auto back_to = [&](int turn) {
        if constexpr (kSnap) {
#pragma unroll
            for (int rr = 0; rr < RB; ++rr) {
                const Two d = *snap_at(turn, rr);
                t.v[0][rr] = d.x;
                t.v[1][rr] = d.y;
            }
        }
    };

    // points outside the domain hold 0 (read by the domain boundary only, whose factor is 0)
#pragma unroll
    for (int rr = 0; rr < RB; ++rr) {
        const int gi = t.gi0 + t.row0 + rr;
        const bool row = gi >= 0 && gi < t.nr;
#pragma unroll
        for (int q = 0; q < 2; ++q)
            if (!(row && t.gj + q >= 0 && t.gj + q < t.nc)) t.v[q][rr] = T(0);
    }

    T* const dst = sor_plane(a, r.dst);
    bool tested_prev = false;
    bool near = true;  // the decision on the epoch before the last: keep this epoch's start
    int give_to = 1;  // plane (e + 1) % 3
    for (int e = 0;; ++e) {
        const int budget = itmax - k;
        const int s_run = budget < S ? budget : S;
        const bool last = e + 1 == r.epochs || budget <= S;
        const bool tested = r.stop == 0 && (sizeof(T) == 8 || ((r.launch0 + e) & a.test_mask) == a.test_mask);
        if (kSnapLds || near) keep(e & 1);
        if (!kSnap && tested_prev) t.store(a, dst);  // FP32: what a decision on the last epoch would end with
        if constexpr (ISO && sizeof(T) == 8) t.check(sh);
        t.begin(sh);
        // every wave has taken what epoch e - 1 left: what epoch e - 2 left has been read (plane (e - 1) % 3)
        if (e > 1) give(give_to == 2 ? 0 : give_to + 1, true);
        t.sweeps(sh, s_run, tested, owns);
        k += s_run;
        if (e == 0) {  // a first iterate's wall values (kept +0 by every store) end with the first epoch
#pragma unroll
            for (int rr = 0; rr < RB; ++rr) {
                const int gi = t.gi0 + t.row0 + rr;
                const bool rint = gi >= 1 && gi <= t.nr - 2;
#pragma unroll
                for (int q = 0; q < 2; ++q)
                    if (!(rint && t.colin[q])) t.v[q][rr] = T(0);
            }
        }
        if (!last) {
            wait_memory();  // this tile's marks of earlier epochs come before what it gives now
            give(give_to, false);
        }
        if (tested) {
            __syncthreads();
            double* part = r.part + ((size_t)(e & 3) * r.ntiles + tile) * kResidentRows;
            const int nupd = Tile::kLastOnly ? 1 : s_run;
            t.reduce(sh, nupd, [&](int row, double sum) {
                agent_store(reinterpret_cast<u64*>(part + (row < nupd ? row : Tile::SE)), (u64)__double_as_longlong(sum));
            });
        }
        u64 word = take(last ? -1 : give_to, tested_prev ? e : 0);
        near = e == 0 || (word >> ((int)(word >> 32) == e ? 16 : 17) & 1);
        int ended = e - 1;  // the epoch a decision that ends the solve is about
        unsigned code = tested_prev && (int)(word >> 32) == e ? (unsigned)(word >> 8) & 255 : RES_CONTINUE;
        if (code == RES_CONTINUE && last && tested) {
            word = take(-1, e + 1);
            ended = e;
            code = (int)(word >> 32) == e + 1 ? (unsigned)(word >> 8) & 255 : RES_CONTINUE;
        }
        if (code == RES_REDO) {
            back_to(ended & 1);
            t.begin(sh);
            const int n = (int)(word & 255);
            for (int s = 0; s < n; ++s) t.template sweep<false>(sh, 0, false, s < n - 1);
        } else if (code == RES_END && ended < e) {
            if (!kSnap) return;  // stored when epoch e began
            back_to(e & 1);
        } else if (code == RES_RERUN) {
            return;
        }
        if (code != RES_CONTINUE || last) break;
        give_to = give_to == 2 ? 0 : give_to + 1;
        tested_prev = tested;
    }
    t.store(a, dst);
}

// The decisions on a solve's epochs, one after the other; the state of the solve.
template <typename T, int S, int NW, int RB, bool NORM>
struct ResidentDecider {
    static constexpr bool kNorm = sizeof(T) == 4 || NORM;
    static constexpr bool kLastOnly = sizeof(T) == 4;
    static constexpr int SE = kLastOnly ? 1 : S;
    static constexpr int nq = SE + (kNorm ? 1 : 0);
    // whether the tiles of this kernel keep their values at the start of every epoch, and, else, of
    // this epoch and the next (what the decisions on the epochs two and one before said)
    static constexpr bool kAlways = sizeof(T) == 4 || resident_snap_lds(NW, RB);
    bool kept = true, kept_next = true;
    int itmax, k, status, launches, rb_n = 0;
    double tol, rtol, e_last, n_last;
    int e = 0, k_prev, sd;
    bool last, tested;
    unsigned code;

    // false: the solve of slot rslot has ended before, and slot wslot says so too
    __device__ __forceinline__ bool begin(SorCtl* ctl, const SorResident& r, const bool writes) {
        const SorCtl* p = ctl + r.rslot;
        itmax = p->itmax;
        k = p->k;
        status = p->status;
        launches = p->launches;
        tol = p->tol;
        rtol = p->rtol;
        e_last = p->e_last;
        n_last = p->n_last;
        if (status == SOR_RUNNING) return true;
        if (writes) ctl[r.wslot] = *p;
        return false;
    }
    __device__ __forceinline__ void end(SorCtl* ctl, const SorResident& r) const {
        SorCtl* p = ctl + r.wslot;
        p->k = k;
        p->parity = r.dst;
        p->status = status;
        p->s_done = 0;
        p->launches = launches;
        p->itmax = itmax;
        p->rb_src = 0;
        p->rb_n = rb_n;
        p->e_last = e_last;
        p->tol = tol;
        p->rtol = rtol;
        p->n_last = n_last;
    }
    __device__ __forceinline__ void epoch(const SorResident& r, const int test_mask) {
        k_prev = k;
        const int budget = itmax - k_prev;
        sd = budget < S ? budget : S;
        last = e + 1 == r.epochs || budget <= S;
        tested = sizeof(T) == 8 || ((r.launch0 + e) & test_mask) == test_mask;
        code = RES_CONTINUE;
        k = k_prev + sd;
        launches += 1;
    }
    // the sums of one tile's epoch, marked again
    __device__ __forceinline__ void sums(const SorResident& r, const int tile, double (&x)[nq], bool& dead) const {
        const int nupd = kLastOnly ? 1 : sd;
        u64* pp = reinterpret_cast<u64*>(r.part + ((size_t)(e & 3) * r.ntiles + tile) * kResidentRows);
        for (int spins = 0;; ++spins) {
            bool ok = true;
#pragma unroll
            for (int i = 0; i < nq; ++i) x[i] = __longlong_as_double((long long)agent_load(pp + i));
#pragma unroll
            for (int i = 0; i < nq; ++i)
                if (i < nupd || i >= SE) ok = ok && Marked<double>::ready(x[i]);
            if (ok || dead) break;
            if (spins >= r.spins) {
                dead = true;
                report_abort(r);
            }
        }
#pragma unroll
        for (int i = 0; i < nq; ++i) {
            if (i >= nupd && i < SE) x[i] = 0.0;  // no such sweep in a budget's last epoch
            agent_store(pp + i, kMark64);
        }
    }
    // the decision on the epoch with the sums tot (as sor_rb_decider's): the tiles' word
    __device__ __forceinline__ u64 decide(const double (&tot)[nq]) {
        const double ntot = kNorm ? tot[nq - 1] : 0.0;
        int s_conv = -1, s_fold = -1, s_bad = -1, redo = 0;
#pragma unroll
        for (int i = 0; i < SE; ++i) {
            const int s = kLastOnly ? sd - 1 : i;
            if (s < sd && s_conv < 0 && s_fold < 0 && s_bad < 0) {
                if (!(tot[i] <= DBL_MAX)) s_bad = s;
                else if (tot[i] < tol) s_conv = s;
                else if (rtol > 0.0 && tot[i] < rtol * ntot) s_fold = s;
            }
        }
        if (kNorm && s_conv < 0 && s_fold < 0 && s_bad < 0 && !(ntot <= DBL_MAX)) s_bad = sd - 1;
        const bool inner = s_conv >= 0 && s_conv < sd - 1;
        const int s_rep = inner ? s_conv : sd - 1;  // reported sweep
#pragma unroll
        for (int i = 0; i < SE; ++i)
            if ((kLastOnly ? sd - 1 : i) == s_rep) e_last = tot[i];
        n_last = ntot;
        if (inner) {
            code = RES_REDO;
            redo = s_conv + 1;
            k = k_prev + redo;
            status = SOR_CONVERGED;
        } else if (s_conv >= 0 || s_fold >= 0 || s_bad >= 0) {
            code = RES_END;
            status = s_conv >= 0 ? SOR_CONVERGED : (s_fold >= 0 ? SOR_FOLD : SOR_DIVERGED);
        }
        if (!kAlways && code != RES_CONTINUE) {
            // the end of this epoch is the next one's start (the tile's own values, if last)
            if (code == RES_END && !last && !kept_next) {
                code = RES_REDO;
                redo = sd;
            }
            if (code == RES_REDO && !kept) {
                code = RES_RERUN;
                rb_n = kNotStored;
            }
        }
        const bool near = e_last < kNearTol * tol || (rtol > 0.0 && e_last < kNearTol * rtol * ntot);
        const u64 word = res_word(e + 1, near, kept_next, code, redo);
        kept = kept_next;
        kept_next = near;
        return word;
    }
    __device__ __forceinline__ bool ended() {
        if (code == RES_CONTINUE && k >= itmax) status = SOR_FAILED;
        return code != RES_CONTINUE || last;
    }
};

// The deciding workgroup: after each tested epoch the decision of sor_rb_decider on its sums, left
// in every tile's word; at the end the solve's state in slot wslot.
template <typename T, int S, int NW, int RB, bool NORM>
__device__ __forceinline__ void sor_resident_decider(const SorArgs<T>& a, const SorResident& r) {
    typedef ResidentDecider<T, S, NW, RB, NORM> Decider;
    constexpr int nq = Decider::nq;
    constexpr int NT = NW * 64;
    __shared__ double lw[NW][nq];
    const int tid = threadIdx.x, lane = tid & 63;
    const int wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    if (r.stop > 0) return;  // the slot holds the solve's end already
    Decider d;
    if (!d.begin(a.ctl, r, tid == 0)) return;
    const int nwp = min(NW, (r.ntiles + 63) >> 6);  // waves holding partials
    bool dead = false;
    for (;; ++d.e) {
        d.epoch(r, a.test_mask);
        if (d.tested) {
            double pv[nq], tot[nq];
#pragma unroll
            for (int i = 0; i < nq; ++i) pv[i] = 0.0;
            for (int t = tid; t < r.ntiles; t += NT) {
                double x[nq];
                d.sums(r, t, x, dead);
#pragma unroll
                for (int i = 0; i < nq; ++i) pv[i] += x[i];
            }
            if (wv < nwp) {
                wave_sum_n(pv);
                if (lane == 0) {
#pragma unroll
                    for (int i = 0; i < nq; ++i) lw[wv][i] = pv[i];
                }
            }
            wait_memory();  // the marks come before the decision that lets a tile write there again
            __syncthreads();
#pragma unroll
            for (int i = 0; i < nq; ++i) {
                tot[i] = 0.0;
                for (int j = 0; j < nwp; ++j) tot[i] += lw[j][i];
            }
            const u64 word = d.decide(tot);
            for (int t = tid; t < r.ntiles; t += NT) agent_store(r.dec + (size_t)t * 8, word);
            __syncthreads();  // lw is read before the next epoch's sums replace it
        }
        if (d.ended()) break;
    }
    if (tid == 0) d.end(a.ctl, r);
}

// The same by one wave, with the same sums in the same order.
template <typename T, int S, int NW, int RB>
__device__ __forceinline__ void sor_resident_wave_decider(const SorArgs<T>& a, const SorResident& r) {
    typedef ResidentDecider<T, S, NW, RB, false> Decider;
    constexpr int nq = Decider::nq;
    const int lane = threadIdx.x & 63;
    if (r.stop > 0) return;
    Decider d;
    if (!d.begin(a.ctl, r, lane == 0)) return;
    bool dead = gave_up(r);
    for (;; ++d.e) {
        d.epoch(r, a.test_mask);
        if (d.tested) {
            double tot[nq];
#pragma unroll
            for (int i = 0; i < nq; ++i) tot[i] = 0.0;
            for (int t0 = 0; t0 < r.ntiles; t0 += 64) {
                double x[nq];
#pragma unroll
                for (int i = 0; i < nq; ++i) x[i] = 0.0;
                if (t0 + lane < r.ntiles) d.sums(r, t0 + lane, x, dead);
                wave_sum_n(x);
#pragma unroll
                for (int i = 0; i < nq; ++i) tot[i] += x[i];
            }
            wait_memory();
            const u64 word = d.decide(tot);
            for (int t = lane; t < r.ntiles; t += 64) agent_store(r.dec + (size_t)t * 8, word);
        }
        if (d.ended()) break;
    }
    if (lane == 0) d.end(a.ctl, r);
}

template <typename T, int S, int NW, int RB, bool GS, bool XR, bool NORM, bool ISO>
__global__ void __launch_bounds__(NW * 64) sor_resident_kernel(SorArgs<T> a, SorResident r) {
    // the next free tile of this XCD's band; the first workgroup that finds none decides
    typedef SorTile<T, S, NW, RB, GS, XR, NORM> Tile;
    __shared__ typename Tile::Shared sh;
    __shared__ SnapPair snap_lds[kSnapPairs<T, NW, RB>];
    __shared__ int place;
    const int band = __builtin_amdgcn_s_getreg(20 | (3 << 11)) & (kBands - 1);  // hwreg XCC_ID
    // its tiles: those of a band of tile rows, or (runs) an eighth of all tiles, row after row
    int first = band_start(band, r.runs ? r.ntiles : a.tiles_i), end = band_start(band + 1, r.runs ? r.ntiles : a.tiles_i);
    int lo = band_lo<Tile>(a, first), hi = band_hi<Tile>(a, end);
    if (!r.runs) {
        first *= a.tiles_j;
        end *= a.tiles_j;
    }
    if (threadIdx.x == 0) {
        int at = atomicAdd(r.claim + band * kClaimStride, 1);
        if (at >= end - first) at = atomicAdd(r.claim + kBands * kClaimStride, 1) == 0 ? -1 : -2;
        place = at;
    }
    __syncthreads();
    const int at = __builtin_amdgcn_readfirstlane(place);
    if (at >= 0) {
        const int tile = first + at;
        const int ti = tile / a.tiles_j, tj = tile - ti * a.tiles_j;
        if (r.runs) {  // TI and TJ >= H: only the 8 tiles around it read its cells
            const int l = tj > 0, g = tj < a.tiles_j - 1;
            const bool beside = (l && tile == first) || (g && tile + 1 == end);
            const bool above = ti > 0 && tile - a.tiles_j - l < first;
            const bool below = ti < a.tiles_i - 1 && tile + a.tiles_j + g >= end;
            lo = beside ? a.nr : (above ? ti * Tile::TI + Tile::H : 0);
            hi = below ? (ti + 1) * Tile::TI - Tile::H : a.nr;
        }
        sor_resident_tile<T, S, NW, RB, GS, XR, NORM, ISO>(a, r, ti, tj, lo, hi, tile, sh, snap_lds);
    } else if (at == -1) {
        sor_resident_decider<T, S, NW, RB, NORM>(a, r);
    }
}

// Many solves in one launch, a workgroup per CU.  Each XCD has a queue of tiles, solve after solve, and
// its workgroups take the next one whenever they have finished a tile, so a solve whose tiles find
// no place yet waits for the ones before it while those run on.  The queues hold the solves in one
// order, so the first unfinished solve always has its tiles next in line on every XCD it spans
// (never more of them on one than that has workgroups): some solve can always run.  The waves of
// the deciding workgroups take the solves in the same order.
template <typename T, int S, int NW, int RB, bool GS>
__global__ void __launch_bounds__(NW * 64) sor_resident_batch_kernel(const SorArgs<T>* __restrict__ args,
                                                                     const SorResident* __restrict__ res,
                                                                     ResidentQueues q) {
    typedef SorTile<T, S, NW, RB, GS, true, false> Tile;
    __shared__ typename Tile::Shared sh;
    __shared__ SnapPair snap_lds[kSnapPairs<T, NW, RB>];
    __shared__ int place;
    const int xcc = __builtin_amdgcn_s_getreg(20 | (3 << 11)) & (kBands - 1);  // hwreg XCC_ID
    if (threadIdx.x == 0) place = atomicAdd(q.counters + xcc * kClaimStride, 1);
    __syncthreads();
    if (__builtin_amdgcn_readfirstlane(place) * kBands + xcc < q.deciders) {
        while (true) {
            int c = 0;
            if ((threadIdx.x & 63) == 0) c = atomicAdd(q.counters + 2 * kBands * kClaimStride, 1);
            c = __builtin_amdgcn_readfirstlane(c);
            if (c >= q.count) return;
            const int i = q.order[c];
            sor_resident_wave_decider<T, S, NW, RB>(args[i], res[i]);
        }
    }
    while (true) {
        __syncthreads();
        if (threadIdx.x == 0) place = atomicAdd(q.counters + (kBands + xcc) * kClaimStride, 1);
        __syncthreads();
        const int at = q.start[xcc] + __builtin_amdgcn_readfirstlane(place);
        if (at >= q.start[xcc + 1]) return;
        const ResidentJob j = q.jobs[at];
        const SorArgs<T>& a = args[j.inst];
        const int ti = j.tile / a.tiles_j, tj = j.tile % a.tiles_j;
        const int lo = band_lo<Tile>(a, j.row_lo), hi = band_hi<Tile>(a, j.row_hi);
        if constexpr (sizeof(T) == 8) {
            if (!a.exact_rcp) {
                sor_resident_tile<T, S, NW, RB, GS, false, false>(a, res[j.inst], ti, tj, lo, hi, blockIdx.x, sh,
                                                                  snap_lds);
                continue;
            }
        }
        sor_resident_tile<T, S, NW, RB, GS, true, false, RB == 8>(a, res[j.inst], ti, tj, lo, hi, blockIdx.x,
                                                                  sh, snap_lds);
    }
}

template <typename T, int S, int NW, int RB>
inline int sor_resident_launch_shape(const SorArgs<T>& a, const SorResident& r, bool gs, hipStream_t st) {
    const dim3 grid(r.blocks), block(NW * 64);
    const bool xr = sizeof(T) == 4 || a.exact_rcp;
    if constexpr (sizeof(T) == 8) {
        if (!gs) {
            constexpr bool kScaled = NW * RB < 96;  // the short form beside the general one: not in thick tiles
            if (kScaled && a.scaled == 1) {
                if (a.norm) hipLaunchKernelGGL((sor_resident_kernel<T, S, NW, RB, false, true, true, kScaled>), grid, block, 0, st, a, r);
                else hipLaunchKernelGGL((sor_resident_kernel<T, S, NW, RB, false, true, false, kScaled>), grid, block, 0, st, a, r);
                return hipGetLastError() == hipSuccess ? 0 : 1;
            }
            if (a.norm) {
                if (xr) hipLaunchKernelGGL((sor_resident_kernel<T, S, NW, RB, false, true, true, false>), grid, block, 0, st, a, r);
                else hipLaunchKernelGGL((sor_resident_kernel<T, S, NW, RB, false, false, true, false>), grid, block, 0, st, a, r);
                return hipGetLastError() == hipSuccess ? 0 : 1;
            }
        }
    }
    if (gs && xr) hipLaunchKernelGGL((sor_resident_kernel<T, S, NW, RB, true, true, false, false>), grid, block, 0, st, a, r);
    else if (xr) hipLaunchKernelGGL((sor_resident_kernel<T, S, NW, RB, false, true, false, false>), grid, block, 0, st, a, r);
    else if constexpr (sizeof(T) == 8) {
        if (gs) hipLaunchKernelGGL((sor_resident_kernel<T, S, NW, RB, true, false, false, false>), grid, block, 0, st, a, r);
        else hipLaunchKernelGGL((sor_resident_kernel<T, S, NW, RB, false, false, false, false>), grid, block, 0, st, a, r);
    }
    return hipGetLastError() == hipSuccess ? 0 : 1;
}

// The shapes compiled as resident kernels, and those for FP64 only.
#define CNV_RESIDENT_SHAPES(X) \
    X(6, 16, 2)                \
    X(5, 16, 2)                \
    X(4, 16, 2)                \
    X(6, 12, 4)                \
    X(6, 16, 4)                \
    X(5, 16, 4)                \
    X(5, 12, 8)                \
    X(5, 12, 10)
#define CNV_RESIDENT_SHAPES_FP64(X) \
    X(3, 12, 14)

template <typename T>
inline int sor_resident_dispatch(const SorArgs<T>& a, const SorResident& r, TileShape sh, bool gs, hipStream_t st) {
#define CNV_RESIDENT_CASE(s_, nw_, rb_) \
    if (sh.s == s_ && sh.nw == nw_ && sh.rb == rb_) return sor_resident_launch_shape<T, s_, nw_, rb_>(a, r, gs, st);
    CNV_RESIDENT_SHAPES(CNV_RESIDENT_CASE)
    if constexpr (sizeof(T) == 8) {
        CNV_RESIDENT_SHAPES_FP64(CNV_RESIDENT_CASE)
    }
#undef CNV_RESIDENT_CASE
    return 2;
}

// The shapes of batched resident solves and the time of one sweep (us, a full GPU).  FP32 tiles of
// 128 x 128 points (8 rows a wave) fit the registers where dx = dy, FP64 ones do not.
struct ResidentBatchShape {
    TileShape shape;
    double us;
};
template <typename T>
inline const std::vector<ResidentBatchShape>& resident_batch_shapes() {
    static const std::vector<ResidentBatchShape> f64 = {{{5, 16, 2}, 1.12}, {{5, 16, 4}, 1.60}};
    static const std::vector<ResidentBatchShape> f32 = {{{5, 16, 2}, 0.86}, {{5, 16, 4}, 1.17}, {{5, 16, 8}, 1.73}};
    return sizeof(T) == 8 ? f64 : f32;
}

template <typename T, int RB>
inline void sor_resident_batch_launch_rb(const SorArgs<T>* args, const SorResident* res, const ResidentQueues& q,
                                         int blocks, bool gs, hipStream_t st) {
    const dim3 grid(blocks), block(16 * 64);
    if (gs) hipLaunchKernelGGL((sor_resident_batch_kernel<T, 5, 16, RB, true>), grid, block, 0, st, args, res, q);
    else hipLaunchKernelGGL((sor_resident_batch_kernel<T, 5, 16, RB, false>), grid, block, 0, st, args, res, q);
}
template <typename T>
inline int sor_resident_batch_launch(const SorArgs<T>* args, const SorResident* res, const ResidentQueues& q,
                                     TileShape sh, int blocks, bool gs, hipStream_t st) {
    if (sh.rb == 2) sor_resident_batch_launch_rb<T, 2>(args, res, q, blocks, gs, st);
    else if (sh.rb == 4) sor_resident_batch_launch_rb<T, 4>(args, res, q, blocks, gs, st);
    else if constexpr (sizeof(T) == 4) sor_resident_batch_launch_rb<T, 8>(args, res, q, blocks, gs, st);
    return hipGetLastError() == hipSuccess ? 0 : 1;
}

}  // namespace cnv
