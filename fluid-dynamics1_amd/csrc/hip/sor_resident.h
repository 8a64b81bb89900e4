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
// together, in one trip.  After a tile has taken epoch e+1's cells, its own cells of epoch e have
// been read by everyone (the tiles that published e+1 had taken e before), and it marks them
// again; the plane's next use is two epochs later, so the marks are in place before a reader can
// look for it (the wait before a publication orders the tile's own marks before it).
//
// Coherence.  The 8 XCDs have an L2 each.  Reads are agent-scope loads, which see what the XCD's own
// L2 holds for it and what other XCDs have written through.  Tile rows are dealt to the XCDs in
// contiguous bands, and each workgroup takes the next free tile of the band of the XCD it finds
// itself on (workgroups are dealt to the XCDs round-robin, so every band gets as many as it has
// tiles; if one did not, its neighbours' waits would run out), so most cells are read on the XCD that
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

#include "sor_rb.h"

namespace cnv {

typedef unsigned long long u64;
constexpr double kNearTol = 4.0;     // an update within this factor of its tolerance may end the solve soon
constexpr int kSpinLimit = 1 << 20;  // polls of one wait (about 0.1 s)
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
// every memory operation this wave has issued is complete
__device__ __forceinline__ void wait_memory() {
    __atomic_signal_fence(__ATOMIC_SEQ_CST);
    __builtin_amdgcn_s_waitcnt(0x0f70);  // vmcnt(0)
    __atomic_signal_fence(__ATOMIC_SEQ_CST);
}

// a decision word: the number of decided epochs, whether the end is near after the last of them and
// after the one before, what to do, sweeps to redo
enum ResidentCode : unsigned { RES_CONTINUE = 0, RES_END = 1, RES_REDO = 2, RES_RERUN = 3 };
__device__ __forceinline__ u64 res_word(int decided, bool near, bool near_before, unsigned code, int redo) {
    return ((u64)(unsigned)decided << 32) | ((unsigned)near_before << 17) | ((unsigned)near << 16) | (code << 8) |
           (unsigned)redo;
}

// One tile's workgroup: tile (ti, tj), in the band `band` of tile rows [row_lo, row_hi).
template <typename T, int S, int NW, int RB, bool GS, bool XR, bool NORM>
__device__ __forceinline__ void sor_resident_tile(const SorArgs<T>& a, const SorResident& r, const int ti, const int tj,
                                                  const int row_lo, const int row_hi) {
    typedef SorTile<T, S, NW, RB, GS, XR, NORM> Tile;
    constexpr int H = Tile::H, TI = Tile::TI, TJ = Tile::TJ;
    constexpr bool kSnap = sizeof(T) == 8;
    constexpr bool kSnapLds = kSnap && resident_snap_lds(NW, RB);
    typedef double Two __attribute__((ext_vector_type(2)));
    __shared__ typename Tile::Shared sh;
    __shared__ Two snap_lds[kSnapLds ? 2 * RB * NW * 64 : 1];

    const int tile = ti * a.tiles_j + tj;
    const SorCtl* P = a.ctl + r.rslot;
    if (P->status != SOR_RUNNING) return;
    const int itmax = r.stop > 0 ? r.stop : P->itmax;
    int k = P->k;
    Tile t;
    t.place(a, ti, tj);
    t.load(a, sor_plane(a, r.src));
    t.fix_odd_edge();
    const bool owns = t.owns_rows();

    // pairs of this lane's columns, and which rows' pairs it takes from or gives to other tiles
    const bool inside = t.gj >= 0 && t.gj < t.nc;
    const bool owncol = t.ownc[0];
    const bool ringcol = owncol && (2 * t.lane < 2 * H || 2 * t.lane >= TJ);
    const int voff = t.gj * (int)sizeof(T);
    const int pitch = r.ldx * (int)sizeof(T);
    const int plane = (int)(r.xplane * (long long)sizeof(T));
    const __amdgpu_buffer_rsrc_t rs = __builtin_amdgcn_make_buffer_rsrc(r.exch, 0, 3 * plane, 0x00027000);
    auto own_row = [&](int rr) {
        const int li = t.row0 + rr;
        return li >= H && li < H + TI && t.gi0 + li < t.nr;
    };
    auto takes = [&](int rr) {
        const int gi = t.gi0 + t.row0 + rr;
        return gi >= 0 && gi < t.nr && inside && !(own_row(rr) && owncol);
    };
    auto gives = [&](int rr) {
        const int li = t.row0 + rr;
        return own_row(rr) && (li < 2 * H || li >= TI ? owncol : ringcol);
    };
    const int lo = row_lo > 0 ? row_lo * TI + H : 0;  // rows another band reads: below lo or from hi on
    const int hi = row_hi < a.tiles_i ? row_hi * TI - H : t.nr;
    auto give = [&](int slot, bool marks) {
#pragma unroll
        for (int rr = 0; rr < RB; ++rr) {
            const int gi = t.gi0 + t.row0 + rr;
            if (!gives(rr)) continue;
            const T x0 = marks ? Marked<T>::mark() : t.v[0][rr], x1 = marks ? Marked<T>::mark() : t.v[1][rr];
            if (gi < lo || gi >= hi) exch_store<T, kAgent>(rs, voff, slot * plane + gi * pitch, x0, x1);
            else exch_store<T, 0>(rs, voff, slot * plane + gi * pitch, x0, x1);
        }
    };

    bool dead = false;
    const u64* dec = r.dec + (size_t)tile * 8;
    // the halo cells of plane `slot` (slot < 0: none) and a decision on `decided` epochs (0: none)
    auto take = [&](int slot, int decided) -> u64 {
        u64 word = 0;
        for (int spins = 0;; ++spins) {
            bool ok = true;
            if (decided) word = agent_load(dec);
            if (slot >= 0) {
#pragma unroll
                for (int rr = 0; rr < RB; ++rr)
                    if (takes(rr)) exch_load<T>(rs, voff, slot * plane + (t.gi0 + t.row0 + rr) * pitch, t.v[0][rr], t.v[1][rr]);
#pragma unroll
                for (int rr = 0; rr < RB; ++rr)
                    if (takes(rr)) ok = ok && Marked<T>::ready(t.v[0][rr]) && Marked<T>::ready(t.v[1][rr]);
            }
            if (decided) ok = ok && (int)(word >> 32) >= decided;
            if (__all(ok) || dead) break;
            if (spins >= kSpinLimit) {
                dead = true;
                report_abort(r);
            }
        }
        const unsigned hi32 = __builtin_amdgcn_readfirstlane((unsigned)(word >> 32));
        const unsigned lo32 = __builtin_amdgcn_readfirstlane((unsigned)word);
        return ((u64)hi32 << 32) | lo32;
    };

    // the values at an epoch's start, in two turns (FP64)
    Two* const mem = kSnapLds ? nullptr : reinterpret_cast<Two*>(r.snap) + (size_t)tile * 2 * RB * NW * 64;
    auto snap_at = [&](int turn, int rr) -> Two* {
        const int q = (turn * RB + rr) * NW * 64 + (int)threadIdx.x;
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
    int give_to = 1, mark_in = 0;  // planes (e + 1) % 3 and e % 3
    for (int e = 0;; ++e) {
        const int budget = itmax - k;
        const int s_run = budget < S ? budget : S;
        const bool last = e + 1 == r.epochs || budget <= S;
        const bool tested = r.stop == 0 && (sizeof(T) == 8 || ((r.launch0 + e) & a.test_mask) == a.test_mask);
        if (kSnapLds || near) keep(e & 1);
        if (!kSnap && tested_prev) t.store(a, dst);  // FP32: what a decision on the last epoch would end with
        t.begin(sh);
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
        if (e > 0) give(mark_in, true);
        mark_in = give_to;
        give_to = give_to == 2 ? 0 : give_to + 1;
        tested_prev = tested;
    }
    t.store(a, dst);
}

// The deciding workgroup: after each tested epoch the decision of sor_rb_decider on its sums, left
// in every tile's word; at the end the solve's state in slot wslot.
template <typename T, int S, int NW, int RB, bool NORM>
__device__ __forceinline__ void sor_resident_decider(const SorArgs<T>& a, const SorResident& r) {
    constexpr bool kNorm = sizeof(T) == 4 || NORM;
    constexpr bool kLastOnly = sizeof(T) == 4;
    constexpr int SE = kLastOnly ? 1 : S;
    constexpr int nq = SE + (kNorm ? 1 : 0);
    constexpr int NT = NW * 64;
    __shared__ double lw[NW][nq];
    const SorCtl P = a.ctl[r.rslot];
    const int tid = threadIdx.x, lane = tid & 63;
    const int wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    if (r.stop > 0) return;  // the slot holds the solve's end already
    if (P.status != SOR_RUNNING) {
        if (tid == 0) a.ctl[r.wslot] = P;
        return;
    }
    // whether the tiles of this kernel keep their values at the start of every epoch, and, else, of
    // this epoch and the next (what the decisions on the epochs two and one before said)
    constexpr bool kAlways = sizeof(T) == 4 || resident_snap_lds(NW, RB);
    bool kept = true, kept_next = true;
    const int nwp = min(NW, (r.ntiles + 63) >> 6);  // waves holding partials
    SorCtl next = P;
    next.s_done = 0;
    next.parity = r.dst;
    next.rb_n = 0;
    bool dead = false;
    for (int e = 0;; ++e) {
        const int k_prev = next.k;
        const int budget = P.itmax - k_prev;
        const int sd = budget < S ? budget : S;
        const bool last = e + 1 == r.epochs || budget <= S;
        const bool tested = sizeof(T) == 8 || ((r.launch0 + e) & a.test_mask) == a.test_mask;
        unsigned code = RES_CONTINUE;
        int redo = 0;
        next.k = k_prev + sd;
        next.launches += 1;
        if (tested) {
            const int nupd = kLastOnly ? 1 : sd;
            double pv[nq];
#pragma unroll
            for (int i = 0; i < nq; ++i) pv[i] = 0.0;
            for (int t = tid; t < r.ntiles; t += NT) {
                u64* pp = reinterpret_cast<u64*>(r.part + ((size_t)(e & 3) * r.ntiles + t) * kResidentRows);
                double x[nq];
                for (int spins = 0;; ++spins) {
                    bool ok = true;
#pragma unroll
                    for (int i = 0; i < nq; ++i) x[i] = __longlong_as_double((long long)agent_load(pp + i));
#pragma unroll
                    for (int i = 0; i < nq; ++i)
                        if (i < nupd || i >= SE) ok = ok && Marked<double>::ready(x[i]);
                    if (ok || dead) break;
                    if (spins >= kSpinLimit) {
                        dead = true;
                        report_abort(r);
                    }
                }
#pragma unroll
                for (int i = 0; i < nq; ++i) {
                    if (i < nupd || i >= SE) pv[i] += x[i];
                    agent_store(pp + i, kMark64);
                }
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
            double etot[SE], ntot = 0.0;
#pragma unroll
            for (int s = 0; s < SE; ++s) {
                etot[s] = 0.0;
                for (int j = 0; j < nwp; ++j) etot[s] += lw[j][s];
            }
            if (kNorm)
                for (int j = 0; j < nwp; ++j) ntot += lw[j][nq - 1];
            int s_conv = -1, s_fold = -1, s_bad = -1;
#pragma unroll
            for (int i = 0; i < SE; ++i) {
                const int s = kLastOnly ? sd - 1 : i;
                if (s < sd && s_conv < 0 && s_fold < 0 && s_bad < 0) {
                    if (!(etot[i] <= DBL_MAX)) s_bad = s;
                    else if (etot[i] < P.tol) s_conv = s;
                    else if (P.rtol > 0.0 && etot[i] < P.rtol * ntot) s_fold = s;
                }
            }
            if (kNorm && s_conv < 0 && s_fold < 0 && s_bad < 0 && !(ntot <= DBL_MAX)) s_bad = sd - 1;
            const bool inner = s_conv >= 0 && s_conv < sd - 1;
            const int s_rep = inner ? s_conv : sd - 1;  // reported sweep
#pragma unroll
            for (int i = 0; i < SE; ++i)
                if ((kLastOnly ? sd - 1 : i) == s_rep) next.e_last = etot[i];
            next.n_last = ntot;
            if (inner) {
                code = RES_REDO;
                redo = s_conv + 1;
                next.k = k_prev + redo;
                next.status = SOR_CONVERGED;
            } else if (s_conv >= 0 || s_fold >= 0 || s_bad >= 0) {
                code = RES_END;
                next.status = s_conv >= 0 ? SOR_CONVERGED : (s_fold >= 0 ? SOR_FOLD : SOR_DIVERGED);
            }
            if (!kAlways && code != RES_CONTINUE) {
                // the end of this epoch is the next one's start (the tile's own values, if last)
                if (code == RES_END && !last && !kept_next) {
                    code = RES_REDO;
                    redo = sd;
                }
                if (code == RES_REDO && !kept) {
                    code = RES_RERUN;
                    next.rb_n = kNotStored;
                }
            }
            const bool near = next.e_last < kNearTol * P.tol || (P.rtol > 0.0 && next.e_last < kNearTol * P.rtol * ntot);
            const u64 word = res_word(e + 1, near, kept_next, code, redo);
            kept = kept_next;
            kept_next = near;
            for (int t = tid; t < r.ntiles; t += NT) agent_store(r.dec + (size_t)t * 8, word);
            __syncthreads();  // lw is read before the next epoch's sums replace it
        }
        if (code == RES_CONTINUE && next.k >= P.itmax) next.status = SOR_FAILED;
        if (code != RES_CONTINUE || last) break;
    }
    if (tid == 0) a.ctl[r.wslot] = next;
}

template <typename T, int S, int NW, int RB, bool GS, bool XR, bool NORM>
__global__ void __launch_bounds__(NW * 64) sor_resident_kernel(SorArgs<T> a, SorResident r) {
    // the next free tile of this XCD's band; the first workgroup that finds none decides
    __shared__ int place;
    const int band = __builtin_amdgcn_s_getreg(20 | (3 << 11)) & (kBands - 1);  // hwreg XCC_ID
    const int row_lo = band_start(band, a.tiles_i), row_hi = band_start(band + 1, a.tiles_i);
    const int tiles = (row_hi - row_lo) * a.tiles_j;
    if (threadIdx.x == 0) {
        int at = atomicAdd(r.claim + band * kClaimStride, 1);
        if (at >= tiles) at = atomicAdd(r.claim + kBands * kClaimStride, 1) == 0 ? -1 : -2;
        place = at;
    }
    __syncthreads();
    const int at = __builtin_amdgcn_readfirstlane(place);
    if (at >= 0) {
        const int ti = row_lo + at / a.tiles_j;
        sor_resident_tile<T, S, NW, RB, GS, XR, NORM>(a, r, ti, at % a.tiles_j, row_lo, row_hi);
    } else if (at == -1) {
        sor_resident_decider<T, S, NW, RB, NORM>(a, r);
    }
}

template <typename T, int S, int NW, int RB>
inline int sor_resident_launch_shape(const SorArgs<T>& a, const SorResident& r, bool gs, hipStream_t st) {
    const dim3 grid(r.blocks), block(NW * 64);
    const bool xr = sizeof(T) == 4 || a.exact_rcp;
    if constexpr (sizeof(T) == 8) {
        if (a.norm && !gs) {
            if (xr) hipLaunchKernelGGL((sor_resident_kernel<T, S, NW, RB, false, true, true>), grid, block, 0, st, a, r);
            else hipLaunchKernelGGL((sor_resident_kernel<T, S, NW, RB, false, false, true>), grid, block, 0, st, a, r);
            return hipGetLastError() == hipSuccess ? 0 : 1;
        }
    }
    if (gs && xr) hipLaunchKernelGGL((sor_resident_kernel<T, S, NW, RB, true, true, false>), grid, block, 0, st, a, r);
    else if (xr) hipLaunchKernelGGL((sor_resident_kernel<T, S, NW, RB, false, true, false>), grid, block, 0, st, a, r);
    else if constexpr (sizeof(T) == 8) {
        if (gs) hipLaunchKernelGGL((sor_resident_kernel<T, S, NW, RB, true, false, false>), grid, block, 0, st, a, r);
        else hipLaunchKernelGGL((sor_resident_kernel<T, S, NW, RB, false, false, false>), grid, block, 0, st, a, r);
    }
    return hipGetLastError() == hipSuccess ? 0 : 1;
}

// The shapes compiled as resident kernels.
#define CNV_RESIDENT_SHAPES(X) \
    X(6, 16, 2)                \
    X(5, 16, 2)                \
    X(4, 16, 2)                \
    X(6, 12, 4)                \
    X(6, 16, 4)                \
    X(5, 16, 4)

template <typename T>
inline int sor_resident_dispatch(const SorArgs<T>& a, const SorResident& r, TileShape sh, bool gs, hipStream_t st) {
#define CNV_RESIDENT_CASE(s_, nw_, rb_) \
    if (sh.s == s_ && sh.nw == nw_ && sh.rb == rb_) return sor_resident_launch_shape<T, s_, nw_, rb_>(a, r, gs, st);
    CNV_RESIDENT_SHAPES(CNV_RESIDENT_CASE)
#undef CNV_RESIDENT_CASE
    return 2;
}

}  // namespace cnv
