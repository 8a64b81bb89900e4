// sor_rb.h -- red-black SOR sweeps for the 5-point Poisson stencil, register-blocked and
// temporally blocked.
//
// One launch advances the whole grid by up to S full sweeps (red half-sweep, then black),
// computing exactly what S successive global sweeps compute, point for point:
//   * each workgroup owns a TI x TJ tile and loads it with a halo of H = 2S cells (one cell per
//     half-sweep) into registers; after half-sweep h the points of the extended tile at distance
//     > h from its edge hold exactly what h+1 global half-sweeps produce (their four neighbours
//     were exact after half-sweep h-1); after 2S half-sweeps the owned tile is exact and is
//     written to the other buffer (ping-pong);
//   * the extended tile is 128 columns wide: lane m of every wave holds columns 2m and 2m+1,
//     and wave w holds RB consecutive rows.  A point's N/S neighbours are in the same lane's
//     registers (rows r+-1), one of its E/W neighbours is the lane's other column and the other
//     comes from lane m+-1 through a DPP wave shift; only the first and last row of each wave
//     are exchanged through LDS, once per half-sweep;
//   * every point of a row is computed, so the sweep is straight-line code with no selects.  A
//     point outside the valid rectangle takes a wrong (finite) value, which only points outside
//     the valid rectangle ever read.  Domain-boundary points must keep psi = 0: their relaxation
//     factor is 0 instead of beta, which leaves them at +-0, and the final store writes +0 there.
//     Points outside the domain have factor 0 too and start from a copy of the nearest data
//     (the tile loads are clamped into the plane): finite, and read only by the boundary and by
//     other points outside;
//   * the L1 norms are accumulated per lane with a 0/1 weight per row (owned rows only) and a
//     per-column ownership mask, written to LDS once per sweep and reduced once per launch
//     (FP32 planes: in the launch's last sweep only).
// Point update (src/poisson.c:268 SOR, src/poisson.c:205 Gauss-Seidel), same association:
//   u = beta*(dy*dy*(N+S) + dx*dx*(E+W) - dx*dx*dy*dy*f) / (2*(dx*dx+dy*dy)) + (1-beta)*u0
// where u0 (the value before this sweep) is the point's current value in either colouring.
// In FP64 the division by the constant B = 2*(dx*dx+dy*dy) is q0 = x*RN(1/B),
// q = fma(fma(-q0, B, x), RN(1/B), q0): Markstein's correction step, which returns the
// correctly rounded quotient RN(x/B) -- the same double as x/B -- for finite x.  When B is a
// power of two (dx = dy = 2^-k), 1/B is exact and x*(1/B) is already RN(x/B): one multiply (XR).
// The L1 norm of each sweep's update (src/poisson.c:34-60; sqrt(pow(d,2)) == |d|) is summed
// over owned points per workgroup in a fixed order into partial[L&1][s][tile] (FP32 planes: the
// last sweep's only, into s = 0).  The next launch decides on them in one extra workgroup beside
// its sweeping ones (the decider), so that neither the partials' latency nor the reduction delays
// any sweep: the decider of launch L+1 reduces launch L's partials in a fixed order and writes
// state slot (L+1)&1 (SorCtl), which launch L+2's workgroups and the host read; the sweepers of
// launch L+1 read slot L&1 only, complete before they started, and sweep speculatively:
//   * a launch whose slot is terminal returns after its tile load (its decider copies the slot
//     forward);
//   * if launch L's sweeps ended the solve, launch L+1's speculative sweeps are discarded;
//   * if sweep s < S-1 of launch L reached e < tol, launch L's output is discarded too: launch
//     L+2 redoes s+1 sweeps from launch L's input plane, which FP64 keeps intact by rotating
//     through three planes, so the final iterate is exactly the one of the first sweep with
//     e < tol (src/poisson.c:273); FP32 planes, a preconditioner, test the last sweep of a
//     launch only, and only of the launches with (L & test_mask) == test_mask (the others sum
//     nothing, leave no partials, and their decider carries the state forward), and rotate
//     through two;
//   * the sweep budget itmax is honoured exactly (src/poisson.c:234);
//   * a non-finite L1 update (or iterate norm) ends the solve with SOR_DIVERGED;
//   * relative rule: with rtol > 0 the solve also stops ("fold") once the update norm of a sweep
//     fell below rtol times the iterate's own L1 norm after that launch's last sweep (measured
//     once per launch) -- the resolution limit of an FP32 defect-correction inner solve, or the
//     relative tolerance of the adjoint problem's FP64 solves (NORM).
#pragma once

#include <float.h>

#include <type_traits>

#include "cnv_device.h"

namespace cnv {

__device__ inline int sor_tile_of_block(int b, int ntiles) {
    // Workgroups are dispatched round-robin over the 8 XCDs of an MI355X.  Give each XCD a
    // contiguous band of tiles so that the halo rows two neighbouring tiles share are fetched
    // into the same L2.
    if ((ntiles & 7) == 0) {
        const int per = ntiles >> 3;
        return (b & 7) * per + (b >> 3);
    }
    return b;
}

__device__ inline double sor_div(double x, double B, double rB) {
    const double q0 = x * rB;
    const double r = __fma_rn(-q0, B, x);
    return __fma_rn(r, rB, q0);
}
// FP32 planes (defect correction): no bit-parity requirement, one multiply by RN(1/B)
__device__ inline float sor_div(float x, float, float rB) { return x * rB; }

// Two consecutive elements of a row, aligned to one element: rows of any pitch are accessed in
// pairs, one multi-dword access each (the hardware needs dword alignment only).
template <typename T> struct PairOf;
template <> struct PairOf<double> { typedef double type __attribute__((ext_vector_type(2), aligned(8))); };
template <> struct PairOf<float> { typedef float type __attribute__((ext_vector_type(2), aligned(4))); };

// The pair at byte offset boff of a row: the row pointer is wave-uniform and the lane's offset a
// 32-bit value, so the address is a scalar base plus a vector offset with no 64-bit lane arithmetic.
template <typename T>
__device__ inline typename PairOf<T>::type load_pair(const T* __restrict__ row, unsigned boff) {
    return *reinterpret_cast<const typename PairOf<T>::type*>(reinterpret_cast<const char*>(row) + boff);
}
// The pair (x0, x1) at byte offset boff of a row when both, else x0 alone.  FP32 tiles are stored
// non-temporally, FP64 tiles with ordinary stores: each measured 0.8% (FP32) and 2.5% (FP64)
// faster per 1024^2 step than the other kind (the FP64 tile read back by the next launch then
// comes from nearer).
template <typename T>
__device__ inline void store_pair(T* __restrict__ row, unsigned boff, bool both, T x0, T x1) {
    typedef typename PairOf<T>::type P;
    constexpr bool kNT = sizeof(T) == 4;
    T* p = reinterpret_cast<T*>(reinterpret_cast<char*>(row) + boff);
    if (both) {
        P d;
        d.x = x0;
        d.y = x1;
        if (kNT) __builtin_nontemporal_store(d, reinterpret_cast<P*>(p));
        else *reinterpret_cast<P*>(p) = d;
    } else {
        if (kNT) __builtin_nontemporal_store(x0, p);
        else *p = x0;
    }
}

// Lane i receives the value of the lane the DPP control CTRL names, e.g. lane i+1's
// (wave_shl:1) or lane i-1's (wave_shr:1); a lane without a source (63 / 0 there) reads 0
// (bound_ctrl), so no old value has to be materialised.
template <int CTRL>
__device__ inline double dpp_shift(double x) {
    const int lo = __builtin_amdgcn_update_dpp(0, __double2loint(x), CTRL, 0xf, 0xf, true);
    const int hi = __builtin_amdgcn_update_dpp(0, __double2hiint(x), CTRL, 0xf, 0xf, true);
    return __hiloint2double(hi, lo);
}
template <int CTRL>
__device__ inline float dpp_shift(float x) {
    return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(x), CTRL, 0xf, 0xf, true));
}
constexpr int kDppFromNext = 0x130;  // wave_shl:1
constexpr int kDppFromPrev = 0x138;  // wave_shr:1

// One step of a wave reduction of N values: x[i] += the lane value that CTRL selects.
template <int CTRL, int N>
__device__ inline void dpp_accumulate(double (&x)[N]) {
    double y[N];
#pragma unroll
    for (int i = 0; i < N; ++i) y[i] = dpp_shift<CTRL>(x[i]);
#pragma unroll
    for (int i = 0; i < N; ++i) x[i] += y[i];
}
// Sums over the 64 lanes of a wave of N independent values, returned to every lane, in a fixed
// association (the same in every workgroup): pairs and quads (quad_perm [1,0,3,2] and
// [2,3,0,1]), the four quads of each 16-lane row (row_shr 4 and 8: lane 15 of a row holds the
// row's sum), then the rows (row_bcast 15: lane 63 gets rows 3 + 2, lane 31 rows 1 + 0;
// row_bcast 31: lane 63 gets all four); lane 63's value is broadcast.  Cross-lane moves only, no
// LDS round trips; each step is applied to all N values before the next, so that their chains
// interleave (no idle cycles between a value's update and its next cross-lane read).
template <int N>
__device__ inline void wave_sum_n(double (&x)[N]) {
    dpp_accumulate<0xb1>(x);
    dpp_accumulate<0x4e>(x);
    dpp_accumulate<0x114>(x);
    dpp_accumulate<0x118>(x);
    dpp_accumulate<0x142>(x);
    dpp_accumulate<0x143>(x);
#pragma unroll
    for (int i = 0; i < N; ++i) {
        const int lo = __builtin_amdgcn_readlane(__double2loint(x[i]), 63);
        const int hi = __builtin_amdgcn_readlane(__double2hiint(x[i]), 63);
        x[i] = __hiloint2double(hi, lo);
    }
}
__device__ inline double wave_sum(double x) {
    double v[1] = {x};
    wave_sum_n(v);
    return v[0];
}

// Plane idx of a solve's iterate planes (FP64: 0, 1, 2; FP32: 0, 1 -- psi2 is not used).
template <typename T>
__device__ inline T* sor_plane(const SorArgs<T>& a, int idx) {
    if constexpr (SorPlanes<T>::value == 2) return (idx & 1) ? a.psi1 : a.psi0;
    else return idx == 0 ? a.psi0 : (idx == 1 ? a.psi1 : a.psi2);
}

// Values at which a scaled tile's arithmetic is exact (SorTile): 0 or of a magnitude in [2^-200, 2^900).
constexpr unsigned kSmallHi = (1023u - 200) << 21, kRangeHi = 1100u << 21;  // of the high word, its sign shifted out
__device__ __forceinline__ bool in_range(double x) { return ((unsigned)__double2hiint(x) << 1) - kSmallHi < kRangeHi; }

// A tile's LDS: the waves' first and last rows, and one column per thread of per-lane sums.
template <typename T, int NW, int SE, bool kNorm, int FL = 0>
struct SorShared {
    T xch[2][NW][2][64];  // [half-sweep parity][wave][first/last row][lane]
    T fcl[FL > 0 ? FL * 2 * NW * 64 : 1];  // the source term of the rows that registers do not hold
    double lred[SE][NW * 64];  // this launch's per-lane L1 update sums, one row per summed sweep
    double lnrm[kNorm ? NW * 64 : 1];  // the per-lane iterate norm after the last sweep
    int exact[NW];             // scaled tiles: the wave's values are in range
};

// A workgroup's tile in registers (NW waves of 64 lanes): wave w holds rows [w*RB, w*RB + RB) of the
// extended tile, lane m columns 2m and 2m+1.
// ISO: dx = dy.  FP32: the two stencil coefficients of a point are one number and held once.  FP64 (a
// "scaled" tile): c1 = c2 = B/4 is a power of two 2^-m, so that factor can be taken out of the update:
//   ((c1*(N+S) + c1*(E+W)) - c3*f) * beta / B  ==  (((N+S) + (E+W)) - (c3*f)/c1) * beta / 4
// with every rounding in the same place of a number 2^m times as large: the same bits in 7
// operations a point instead of 10, as long as no result is subnormal or infinite on either side.
// That holds for a pass of up to 12 half-sweeps from values that are 0 or in [2^-200, 2^900) in
// magnitude (in_range): they are multiples of 2^-252; sums of multiples are multiples; a product with
// beta or 1-beta (1/64 to 16) is rounded to a multiple of a number at most 2^58 times smaller.  So
// what is not 0 stays above 2^-948, 2^-m (at least 2^-61) times that is a normal number, and
// nothing grows by more than 2^6 in a half-sweep.  Where a tile has other values (the front of a
// first iterate, whose cells fall off twofold from one to the next), it takes the general form, in a
// rolled loop.  A tile whose source term has other values (the front of a vorticity that spreads from
// the walls: below 2^-200 from step 16 on at 1024^2) would do so at every epoch, and all tiles wait for
// it: it says so, and the solve's next kernels, and the next solve's, are the general form's, until
// the source is in range again (1024^2 from rest, steps from 17 on: 1.62 -> 1.45 us a sweep).
// Resident, us per sweep: 64^2 0.765 -> 0.728, 256^2 0.860 -> 0.832, 1024^2 1.445 -> 1.323; the check is
// about 20 of an epoch's 600 instructions.
template <typename T, int S, int NW, int RB, bool GS, bool XR, bool NORM, bool ISO = false>
struct SorTile {
    static constexpr int H = 2 * S;
    static constexpr int EJ = 128;  // extended tile columns; lane m holds columns 2m, 2m+1
    static constexpr int TJ = EJ - 2 * H;
    static constexpr int EI = NW * RB;  // extended tile rows; wave w holds rows [w*RB, w*RB+RB)
    static constexpr int TI = EI - 2 * H;
    static_assert(TI > 0 && TJ > 0, "halo larger than the tile");
    static_assert(RB % 2 == 0, "even row blocks keep each wave's colour pattern static");
    // the iterate's L1 norm is needed by the relative stopping rule (rtol): always on FP32
    // planes, on request (NORM) for FP64.  It is measured once per launch, after its last sweep.
    static constexpr bool kNorm = sizeof(T) == 4 || NORM;
    // FP32 planes (the inner solves of defect correction) are a preconditioner with no bit-parity
    // requirement: their stopping rule is applied to a launch's last sweep only (and only on the
    // launches the test mask selects), so the other sweeps skip the L1 update (a solve runs at
    // most (test_mask + 1) * S - 1 sweeps past the first sweep that met the rule).  FP64 applies
    // it to every sweep, as src/poisson.c:272-278 does.
    static constexpr bool kLastOnly = sizeof(T) == 4;
    static constexpr int SE = kLastOnly ? 1 : S;  // L1 update sums per launch
    typedef typename std::conditional<sizeof(T) == 4, float, double>::type Acc;
    typedef typename PairOf<T>::type Pair;

    // Thick FP64 tiles (resident solves of large grids) have no registers for a relaxation factor per
    // point: the rows' share of it, and of the norms' weights, is a bit mask, from which every row's
    // factor comes as a scalar; the columns' share, 0 on the domain boundary, is in the lane's
    // reciprocal.  The thickest keep the source term of only RF rows of a wave, the others' in LDS.
    static constexpr bool kMasks = sizeof(T) == 8 && NW * RB >= 96;
    static constexpr int RF = kMasks && RB > 10 ? 5 : RB;
    static_assert(!(ISO && kMasks), "no scaled thick tiles: both forms of their update do not fit the registers");

    typedef SorShared<T, NW, SE, kNorm, RB - RF> Shared;

    T v[2][RB];   // v[q][r]: value at (row0 + r, 2*lane + q)
    T fc[2][RF];  // FP64: c3*f (the hoisted c3*f product of the update); FP32: -be*c3*f
    T be[2][kMasks ? 1 : RB];  // FP64: bcoef at interior points, 0 on the domain boundary and outside it
    T cn[2][RB];  // FP32: be*c1 and be*c2, the relaxation folded into the stencil coefficients
    T ce[2][ISO ? 1 : RB];
    Acc w[kMasks ? 1 : RB];  // 1 for owned rows inside the domain, else 0 (wave-uniform)
    unsigned inner, owned;   // kMasks: bit r for an interior, an owned row r
    T bcoef, rBc[2];         // kMasks: the relaxation factor; rB, 0 on the domain boundary's columns
    bool f_exact;            // this lane's source terms are in range (a scaled tile's, or one that could be)
    T c1, c2, B, rB, omb;
    int gi0, gj0, gj, lane, wv, row0, nr, nc;
    unsigned bld;
    bool colin[2], ownc[2];

    __device__ __forceinline__ void place(const SorArgs<T>& a, int ti, int tj) {
        gi0 = ti * TI - H;  // even, so the colour of local (li, lj) is (li + lj) & 1
        gj0 = tj * TJ - H;
        nr = a.nr;
        nc = a.nc;
        lane = threadIdx.x & 63;
        wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);  // wave-uniform (SGPR)
        row0 = wv * RB;  // even: the colour of (row0 + r, 2m + q) is (r + q) & 1
        // Column facts of the lane's pair (gj, gj+1), gj even: q = 0 -> column gj, q = 1 -> gj+1.
        gj = gj0 + 2 * lane;
#pragma unroll
        for (int q = 0; q < 2; ++q) {
            colin[q] = gj + q >= 1 && gj + q <= nc - 2;
            ownc[q] = 2 * lane + q >= H && 2 * lane + q < H + TJ && gj + q < nc;  // ownc[1] implies ownc[0]
        }
        // Every load reads a pair inside the data: rows clamped into [0, nr), the pair's first column
        // into [0, nc-2].  So no lane needs a select on what it loads: a point outside the domain may
        // start from any finite value (it is read only by points outside the domain and by the domain
        // boundary, whose relaxation factor is 0), and each domain-boundary point is read from its own
        // position (+-0 there).  With nc odd, the lane of column nc-1 reads the pair (nc-2, nc-1) and
        // takes its second element (fixed after the loads); its column nc is outside.
        bld = (unsigned)(gj < 0 ? 0 : (gj > nc - 2 ? nc - 2 : gj)) * sizeof(T);
    }
    __device__ __forceinline__ const T* row_of(const SorArgs<T>& a, const T* plane, int gi) const {  // wave-uniform row pointer
        return plane + (gi < 0 ? 0 : (gi >= nr ? nr - 1 : gi)) * (long long)a.ld;
    }

    // the tile's values from plane src, its source term and its coefficients
    __device__ __forceinline__ void load(const SorArgs<T>& a, const T* __restrict__ src, Shared& sh) {
#pragma clang fp contract(off)
        // relaxation factor of an updated point: FP64 beta (1 for Gauss-Seidel), applied before the
        // division; FP32 beta/B (1/B), which folds the division in.  Per column, 0 off the interior
        // columns; per point, also 0 on the boundary rows and outside the domain.
        if constexpr (sizeof(T) == 8) bcoef = GS ? T(1) : a.beta;
        else bcoef = GS ? a.rB : a.beta * a.rB;
        const T c3s = a.negate ? -a.c3 : a.c3;  // f = -src folded in: c3*(-x) == (-c3)*x exactly
        T bcol[2], cncol[2], cecol[2];
        inner = owned = 0;
        f_exact = true;
#pragma unroll
        for (int q = 0; q < 2; ++q) {
            rBc[q] = colin[q] ? a.rB : T(0);
            bcol[q] = colin[q] ? bcoef : T(0);
            cncol[q] = colin[q] ? bcoef * a.c1 : T(0);
            cecol[q] = colin[q] ? bcoef * a.c2 : T(0);
        }
#pragma unroll
        for (int r = 0; r < RB; ++r) {
            const int li = row0 + r;
            const int gi = gi0 + li;
            const bool rint = gi >= 1 && gi <= nr - 2;
            const bool own = li >= H && li < H + TI && gi < nr;
            if constexpr (kMasks) {
                inner |= (unsigned)rint << r;
                owned |= (unsigned)own << r;
            } else {
                w[r] = own ? Acc(1) : Acc(0);
            }
            const Pair d = load_pair(row_of(a, src, gi), bld);
            const Pair f = load_pair(row_of(a, a.src_f, gi), bld);
            v[0][r] = d.x;
            v[1][r] = d.y;
#pragma unroll
            for (int q = 0; q < 2; ++q) {
                // a non-interior point's source is not read by the reference: 0, whatever it holds
                const bool inter = rint && colin[q];
                const T fq = q ? f.y : f.x;
                if constexpr (sizeof(T) == 8) {
                    // scaled: (c3*f)/c1
                    const T fr = inter ? (ISO ? (c3s * fq) * (T(1) / a.c1) : c3s * fq) : T(0);
                    if constexpr (ISO) f_exact = f_exact && (in_range(fr) || fr == T(0));
                    else if (XR && !GS && !kMasks && a.scaled == 2) {
                        const T fs = fr * (T(1) / a.c1);
                        f_exact = f_exact && (in_range(fs) || fs == T(0));
                    }
                    if (r < RF) fc[q][r < RF ? r : 0] = fr;
                    else sh.fcl[(r < RF ? 0 : (r - RF) * 2 + q) * NW * 64 + threadIdx.x] = fr;
                    if constexpr (!kMasks) be[q][r] = rint ? bcol[q] : T(0);
                } else {
                    fc[q][r < RF ? r : 0] = inter ? bcoef * -(c3s * fq) : T(0);
                    cn[q][r] = rint ? cncol[q] : T(0);
                    if constexpr (!ISO) ce[q][r] = rint ? cecol[q] : T(0);
                }
            }
        }
        c1 = a.c1;
        c2 = a.c2;
        B = a.B;
        rB = a.rB;
        omb = a.omb;
    }
    __device__ __forceinline__ void load_values(const SorArgs<T>& a, const T* __restrict__ src) {
#pragma unroll
        for (int r = 0; r < RB; ++r) {
            const Pair d = load_pair(row_of(a, src, gi0 + row0 + r), bld);
            v[0][r] = d.x;
            v[1][r] = d.y;
        }
    }
    __device__ __forceinline__ void fix_odd_edge() {
        if (nc & 1) {  // wave-uniform: the lane of column nc-1 read the pair (nc-2, nc-1)
            if (gj == nc - 1) {
#pragma unroll
                for (int r = 0; r < RB; ++r) v[0][r] = v[1][r];
            }
        }
    }
    __device__ __forceinline__ bool owns_rows() const {  // wave-uniform: the wave holds an owned row
        bool owns = kMasks && owned != 0;
        if constexpr (!kMasks) {
#pragma unroll
            for (int r = 0; r < RB; ++r) owns = owns || w[r] != Acc(0);
        }
        return owns;
    }

    // half-sweep 0 updates colour 0 and reads its neighbours' colour-1 boundary rows: colour 1
    // sits in column q = (r + 1) & 1 of row r
    __device__ __forceinline__ void begin(Shared& sh) {
        sh.xch[1][wv][0][lane] = v[1][0];
        sh.xch[1][wv][1][lane] = v[(RB - 1 + 1) & 1][RB - 1];
        __syncthreads();
    }
    // sweep s (red half-sweep, then black) of a pass; with_norm: also sum the iterate's norm
    // (FP32: and the update, which only the last sweep sums); kL1: sum the L1 norms at all, which
    // a wave holding no owned row skips (its sums are 0); more: another sweep follows, which needs
    // the other waves' boundary rows
    // kScaled: the short form of a scaled tile's update
    template <bool kL1, bool kScaled = false>
    __device__ __forceinline__ void sweep(Shared& sh, const int s, const bool with_norm, const bool more) {
#pragma clang fp contract(off)
        const int tid = threadIdx.x;
        Acc acc[2] = {Acc(0), Acc(0)}, nrm[2] = {Acc(0), Acc(0)};
#pragma unroll
        for (int c = 0; c < 2; ++c) {
            // LDS offsets reach 64 KB: the source terms beyond have a base of their own
            constexpr int kNear = 65536 / (NW * 64 * (int)sizeof(T)) - 1;
            unsigned at0 = tid, at1 = tid + kNear * NW * 64;
            if constexpr (RF < RB) asm volatile("" : "+v"(at0), "+v"(at1));
            unsigned in_now = kMasks ? inner : 0, own_now = kMasks ? owned : 0;
            if constexpr (kMasks) asm volatile("" : "+s"(in_now), "+s"(own_now));  // the rows' scalars are not kept
            // boundary rows of the neighbouring waves (colour 1-c, written by half-sweep h-1)
            const T sb = sh.xch[c ^ 1][wv > 0 ? wv - 1 : 0][1][lane];
            const T nb = sh.xch[c ^ 1][wv < NW - 1 ? wv + 1 : NW - 1][0][lane];
            // rows 1..RB-2 first: they do not wait for the LDS reads of sb / nb
#pragma unroll
            for (int rr = 0; rr < RB; ++rr) {
                const int r = rr < RB - 2 ? rr + 1 : (rr == RB - 2 ? 0 : RB - 1);
                const int q = (c + r) & 1;  // column of colour c in row r (compile-time)
                const T old = v[q][r];
                const T up = (r < RB - 1) ? v[q][r + 1] : nb;
                const T dn = (r > 0) ? v[q][r - 1] : sb;
                // E + W: the lane's other column plus the neighbouring lane's nearer column
                const T own = v[q ^ 1][r];
                const T far = q ? dpp_shift<kDppFromNext>(v[0][r]) : dpp_shift<kDppFromPrev>(v[1][r]);
                T cand;
                if constexpr (sizeof(T) == 8) {
                    // the reference's association: ((c1*(N+S) + c2*(E+W)) - c3*f), times beta,
                    // divided by B, plus (1-beta)*u0; + is commutative, so E/W order is free
                    const int j2 = r < RF ? 0 : (r - RF) * 2 + q;  // compile-time
                    const bool far_f = j2 >= kNear;
                    if constexpr (kScaled) {
                        const T z = be[q][kMasks ? 0 : r] * (((up + dn) + (own + far)) - fc[q][r]);
                        cand = __fma_rn(z, T(0.25), omb * old);
                    } else {
                        const T x = c1 * (up + dn) + c2 * (own + far) -
                                    (r < RF ? (ISO ? c1 : T(1)) * fc[q][r < RF ? r : 0]
                                            : sh.fcl[far_f ? at1 + (j2 - kNear) * NW * 64 : at0 + j2 * NW * 64]);
                        const T y = (kMasks ? (in_now >> r & 1 ? bcoef : T(0)) : be[q][kMasks ? 0 : r]) * x;
                        const T rq = kMasks ? rBc[q] : rB;
                        const T qt = XR ? y * rq : sor_div(y, B, rq);
                        cand = GS ? qt : qt + omb * old;
                    }
                    if constexpr (!kMasks) v[q][r] = cand;
                    if constexpr (kL1) {
                        const T wr = kMasks ? (own_now >> r & 1 ? T(1) : T(0)) : w[kMasks ? 0 : r];
                        acc[q] = __fma_rn(wr, fabs(cand - old), acc[q]);
                        if (kNorm && with_norm) nrm[q] = __fma_rn(wr, fabs(cand), nrm[q]);
                    }
                    // into the old value's register, once the sum is done with that: the compiler
                    // otherwise holds every row twice and moves all of them at the end of a sweep
                    // (no lane exchange of this value follows before the next barrier)
                    if constexpr (kMasks) asm volatile("v_mov_b64 %0, %2" : "+v"(v[q][r]), "+v"(acc[q]) : "v"(cand));
                } else {
                    // relaxation and 1/B folded into cn, ce and fc (0 where the point is fixed)
                    const T x = __fmaf_rn(cn[q][r], up + dn, __fmaf_rn(ISO ? cn[q][r] : ce[q][ISO ? 0 : r], own + far, fc[q][r < RF ? r : 0]));
                    cand = GS ? x : __fmaf_rn(omb, old, x);
                    v[q][r] = cand;
                    if (kL1 && with_norm) {
                        acc[q] = __fmaf_rn(w[r], fabsf(cand - old), acc[q]);
                        nrm[q] = __fmaf_rn(w[r], fabsf(cand), nrm[q]);
                    }
                }
            }
            if (c == 0 || more) {
                sh.xch[c][wv][0][lane] = v[c & 1][0];
                sh.xch[c][wv][1][lane] = v[(c + RB - 1) & 1][RB - 1];
                __syncthreads();
            }
        }
        // per-lane sums of this sweep, owned columns only; reduced once after the last sweep
        if (!kLastOnly || with_norm)
            sh.lred[kLastOnly ? 0 : s][tid] = (double)((ownc[0] ? acc[0] : Acc(0)) + (ownc[1] ? acc[1] : Acc(0)));
        if (kNorm && with_norm)
            sh.lnrm[tid] = (double)((ownc[0] ? nrm[0] : Acc(0)) + (ownc[1] ? nrm[1] : Acc(0)));
    }
    // scaled tiles, before begin() and after it: whether the short form gives the same bits, the same
    // for every wave of the workgroup (they read one another's rows)
    __device__ __forceinline__ void check(Shared& sh) const {
        bool ok = f_exact;
#pragma unroll
        for (int r = 0; r < RB; ++r)
#pragma unroll
            for (int q = 0; q < 2; ++q) ok = ok && in_range(v[q][r]);
        if (!__all(ok)) {  // some are 0: in boundary tiles, and in a first iterate
            ok = f_exact;
#pragma unroll
            for (int r = 0; r < RB; ++r)
#pragma unroll
                for (int q = 0; q < 2; ++q) ok = ok && (in_range(v[q][r]) || v[q][r] == T(0));
        }
        const bool all = __all(ok);
        if (lane == 0) sh.exact[wv] = all;
    }
    __device__ __forceinline__ bool checked(const Shared& sh) const { return __all(sh.exact[lane < NW ? lane : 0] != 0); }
    // s_run sweeps of a launch or epoch, with the L1 sums its stopping test needs (tested)
    __device__ __forceinline__ void sweeps(Shared& sh, const int s_run, const bool tested, const bool owns) {
        constexpr bool kShort = ISO && sizeof(T) == 8;
        const bool general = kShort && !checked(sh);
        // the common full pass, unrolled: the values stay in their registers from sweep to sweep (a
        // rolled loop makes the compiler rotate them through copies at every iteration); not for the
        // FP64 shapes whose unrolled pass no longer fits the register budget of their wave count.
        // A rollback or a budget-limited last launch takes the loop, which sums the FP64 norm in
        // every sweep (the last one's stays).
        // The waves that hold only halo rows (a quarter of them at 1024^2) run it without the FP64
        // L1 sums, two of the point update's 14 instructions.
        constexpr bool kUnroll = sizeof(T) == 4 || (S * RB <= 40 && NW != 12 && !(kNorm && S * RB > 20));
        if (kUnroll && s_run == S && !general) {
            // FP32: an untested launch skips the last sweep's sums.  Small shapes get a pass of their
            // own without them (6.10 against 6.29 us per launch at 1024^2 with (5, 16, 4)); large ones
            // branch on the uniform flag in the last sweep, since a second unrolled pass of their
            // size made the kernel slower (the batched (8, 8, 10) FP32 sweep 4.05 -> 4.7 us)
            constexpr bool kSplit = sizeof(T) == 4 && S * RB <= 24;
            if (kSplit && !tested) {
#pragma unroll
                for (int s = 0; s < S; ++s) sweep<false, kShort>(sh, s, false, s < S - 1);
            } else if (owns || sizeof(T) == 4) {
#pragma unroll
                for (int s = 0; s < S; ++s) sweep<true, kShort>(sh, s, s == S - 1 && (kSplit || tested), s < S - 1);
            } else {
#pragma unroll
                for (int s = 0; s < S; ++s) sweep<false, kShort>(sh, s, s == S - 1, s < S - 1);
            }
        } else if (!kUnroll && kShort && !general) {
            for (int s = 0; s < s_run; ++s) sweep<true, kShort>(sh, s, kNorm, s < s_run - 1);
        } else {
            for (int s = 0; s < s_run; ++s)
                sweep<true>(sh, s, kLastOnly ? tested && s == s_run - 1 : kNorm, s < s_run - 1);
        }
    }
    // the owned tile to plane dst; domain-boundary points hold +-0: store +0
    __device__ __forceinline__ void store(const SorArgs<T>& a, T* __restrict__ dst) const {
        int gj = this->gj;
        if constexpr (kMasks) {  // not kept from the loads on
            int m = threadIdx.x & 63;
            asm volatile("" : "+v"(m));
            gj = gj0 + 2 * m;
        }
#pragma unroll
        for (int r = 0; r < RB; ++r) {
            const int li = row0 + r;
            const int gi = gi0 + li;
            if (li >= H && li < H + TI && gi < nr) {  // owned row (wave-uniform)
                const bool rint = gi >= 1 && gi <= nr - 2;
                // owned columns lie inside the row: 0 <= gj < nc
                if (ownc[0])
                    store_pair(dst + gi * (long long)a.ld, (unsigned)gj * sizeof(T), ownc[1], (rint && colin[0]) ? v[0][r] : T(0),
                               (rint && colin[1]) ? v[1][r] : T(0));
            }
        }
    }
    // this wave's rows of the tile's per-sweep sums (the per-lane sums in lred, the norm in lnrm;
    // wave w reduces rows w, w + NW, ..., each in a fixed order), handed to put(row, sum) by lane 0;
    // row i < nupd is an update sum, row nupd the norm
    template <typename Put>
    __device__ __forceinline__ void reduce(const Shared& sh, const int nupd, Put put) const {
        const int nrows = nupd + (kNorm ? 1 : 0);
        for (int row = wv; row < nrows; row += NW) {
            const double* col = row < nupd ? sh.lred[row] : sh.lnrm;
            // the NW lane sums of this column, pairwise (depth log2 NW, not a chain of NW adds)
            double t[NW];
#pragma unroll
            for (int j = 0; j < NW; ++j) t[j] = col[lane + 64 * j];
#pragma unroll
            for (int d = 1; d < NW; d *= 2)
#pragma unroll
                for (int j = 0; j + d < NW; j += 2 * d) t[j] += t[j + d];
            const double acc = wave_sum(t[0]);
            if (lane == 0) put(row, acc);
        }
    }
};

// One sweeping workgroup's launch on tile `tile` of the solve described by `a` (NW*64 threads).
// It reads the state slot the previous launch's decider wrote: RUNNING -- sweep on from plane
// L % NB (the previous launch's output) into plane (L+1) % NB, as many sweeps as the budget
// leaves, and leave this tile's per-sweep L1 sums for the next launch's decider; ROLLBACK -- the
// solve converged inside the launch before last: redo rb_n sweeps from plane rb_src into plane
// `parity`, which then holds the final iterate; anything else -- the solve has ended: return.
template <typename T, int S, int NW, int RB, bool GS, bool XR, bool NORM>
__device__ __forceinline__ void sor_rb_sweeper(const SorArgs<T>& a, const int L, const int tile) {
    typedef SorTile<T, S, NW, RB, GS, XR, NORM> Tile;
    constexpr int NB = SorPlanes<T>::value;
    __shared__ typename Tile::Shared sh;
    const SorCtl* prev = a.ctl + ((L + 1) & 1);
    const int ntiles = a.tiles_i * a.tiles_j;
    const int ti = tile / a.tiles_j;
    const int tj = tile - ti * a.tiles_j;
    Tile t;
    t.place(a, ti, tj);
    // Speculative tile load for the common case (sweep on from the previous launch's output),
    // issued before the state slot is read so that both are in flight together.
    t.load(a, sor_plane(a, L % NB), sh);

    // what this launch does: the state after launch L-2 and the sweeps launch L-1 performed
    const int pstatus = prev->status;
    bool rollback = false;
    int s_run = 0;
    T* __restrict__ dst = nullptr;
    if (pstatus == SOR_RUNNING) {
        const int budget = prev->itmax - (prev->k + prev->s_done);
        s_run = budget < S ? budget : S;
        dst = sor_plane(a, (L + 1) % NB);
    } else if (pstatus == SOR_ROLLBACK) {
        rollback = true;
        s_run = prev->rb_n;
        dst = sor_plane(a, prev->parity);
    }
    if (s_run <= 0) return;  // the solve has ended, or its budget is spent
    // FP32: whether this launch's last sweep is tested (FP64: every sweep of every launch)
    const bool tested = sizeof(T) == 8 || (L & a.test_mask) == a.test_mask;
    // the converged launch's input replaces the speculatively loaded tile
    if (rollback) t.load_values(a, sor_plane(a, prev->rb_src));
    t.fix_odd_edge();
    const bool owns = t.owns_rows();
    t.begin(sh);
    t.sweeps(sh, s_run, tested, owns);

    // every wave's lane sums are in LDS; the stores below do not wait for this barrier's peers,
    // so the reducing waves start as soon as their own stores are issued
    if (!rollback && tested) __syncthreads();
    t.store(a, dst);
    if (rollback || !tested) return;  // the final iterate, or an untested launch: no partials

    // this tile's per-sweep partials for the next launch's decider (FP32: the last sweep's update)
    double* part = a.partial + (L & 1) * ((size_t)kMaxSweepsPerLaunch * ntiles * 2);
    const int nupd = Tile::kLastOnly ? 1 : s_run;
    t.reduce(sh, nupd, [&](int row, double sum) {
        part[row < nupd ? ((size_t)row * ntiles + tile) * 2 : (size_t)tile * 2 + 1] = sum;
    });
}

// The deciding workgroup of launch L (NW*64 threads): decides on launch L-1's sweeps from their
// per-tile partial sums (src/poisson.c:272-278) and writes state slot L&1, which launch L+1's
// workgroups and the host read.  Every sum runs in one fixed order: thread t adds the partials of
// tiles t, t + NT, ... in that order, each wave reduces its threads' sums with DPP moves, and lane
// i adds the per-wave totals of quantity i in wave order.
template <typename T, int S, int NW, bool NORM>
__device__ __forceinline__ void sor_rb_decider(const SorArgs<T>& a, const int L) {
    constexpr int NB = SorPlanes<T>::value;
    constexpr bool kNorm = sizeof(T) == 4 || NORM;
    constexpr bool kLastOnly = sizeof(T) == 4;
    constexpr int SE = kLastOnly ? 1 : S;
    constexpr int nq = SE + (kNorm ? 1 : 0);  // reduced quantities: SE updates (and the norm)
    __shared__ double lw[NW][nq];             // per-wave totals

    const SorCtl* prev = a.ctl + ((L + 1) & 1);
    SorCtl* mine = a.ctl + (L & 1);
    const int tid = threadIdx.x;
    const int lane = threadIdx.x & 63;
    const int wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int ntiles = a.tiles_i * a.tiles_j;
    // FP32: launch L-1 left partials only if it was a tested launch
    const bool tested = sizeof(T) == 8 || ((L - 1) & a.test_mask) == a.test_mask;

    // the previous launch's per-tile partials (all S rows are read, before the slot is known, so
    // that these loads are in flight together with it; only the first sd are used).  Layout per
    // tile: [s][tile][0] the L1 update of sweep s (FP32: [0][tile][0], the launch's last sweep),
    // [0][tile][1] the iterate's norm after the last sweep.
    const size_t pstride = (size_t)kMaxSweepsPerLaunch * ntiles * 2;
    double pv[nq];
#pragma unroll
    for (int i = 0; i < nq; ++i) pv[i] = 0.0;
    if (tested) {
        const double* pp = a.partial + ((L + 1) & 1) * pstride;
        constexpr int NT = NW * 64;
        if (ntiles <= NT) {  // one tile per thread at most (1024^2: 240 tiles)
            if (tid < ntiles) {
#pragma unroll
                for (int s = 0; s < SE; ++s) pv[s] = pp[((size_t)s * ntiles + tid) * 2];
                if (kNorm) pv[nq - 1] = pp[(size_t)tid * 2 + 1];
            }
        } else {
            // several tiles per thread: U at a time, all loads issued before the sums, so that
            // the round trips overlap instead of following one another (same order)
            constexpr int U = 4;
            for (int t0 = tid; t0 < ntiles; t0 += U * NT) {
                double x[U][nq];
#pragma unroll
                for (int u = 0; u < U; ++u) {
                    const int t = t0 + u * NT;
                    const int tc = t < ntiles ? t : 0;  // in range; its value is discarded
#pragma unroll
                    for (int s = 0; s < SE; ++s) x[u][s] = pp[((size_t)s * ntiles + tc) * 2];
                    if (kNorm) x[u][nq - 1] = pp[(size_t)tc * 2 + 1];
                }
#pragma unroll
                for (int u = 0; u < U; ++u) {
                    if (t0 + u * NT < ntiles) {
#pragma unroll
                        for (int i = 0; i < nq; ++i) pv[i] += x[u][i];
                    }
                }
            }
        }
    }
    const SorCtl P = *prev;
    if (P.status != SOR_RUNNING) {
        // ended: carry the state forward; a rollback is being done by this launch's sweepers,
        // after which plane P.parity holds the final iterate
        if (tid == 0) {
            SorCtl next = P;
            if (P.status == SOR_ROLLBACK) {
                next.status = SOR_CONVERGED;
                next.launches += 1;
            }
            next.s_done = 0;
            *mine = next;
        }
        return;
    }
    const int sd = P.s_done;  // sweeps the previous launch performed (0: none, e.g. launch 0)
    if (!tested) {
        // an untested launch: its sweeps are accepted, the solve runs on unless its budget is spent
        if (tid == 0) {
            SorCtl next = P;
            next.parity = L % NB;
            next.k = P.k + sd;
            if (next.k >= P.itmax) next.status = SOR_FAILED;
            const int budget = P.itmax - next.k;
            next.s_done = next.status == SOR_RUNNING ? (budget < S ? (budget > 0 ? budget : 0) : S) : 0;
            if (next.status == SOR_RUNNING && next.s_done > 0) next.launches = P.launches + 1;
            *mine = next;
        }
        return;
    }
    const int nwp = min(NW, (ntiles + 63) >> 6);  // waves holding partials
    if (sd > 0 && wv < nwp) {
        wave_sum_n(pv);
        if (lane == 0) {
#pragma unroll
            for (int i = 0; i < nq; ++i) lw[wv][i] = pv[i];
        }
    }
    __syncthreads();
    if (wv != 0) return;
    // lane i of wave 0 sums the per-wave totals of quantity i in wave order; broadcast
    double etot[SE];
    double ntot = 0.0;
    {
        double e = 0.0;
        if (sd > 0 && (lane < (kLastOnly ? 1 : sd) || (kNorm && lane == nq - 1))) {
            for (int j = 0; j < nwp; ++j) e += lw[j][lane];
        }
        const int lo = __double2loint(e), hi = __double2hiint(e);
#pragma unroll
        for (int s = 0; s < SE; ++s)
            etot[s] = __hiloint2double(__builtin_amdgcn_readlane(hi, s), __builtin_amdgcn_readlane(lo, s));
        if (kNorm)
            ntot = __hiloint2double(__builtin_amdgcn_readlane(hi, nq - 1), __builtin_amdgcn_readlane(lo, nq - 1));
    }
    const int k_prev = P.k, itmax = P.itmax;
    const double tol = P.tol, rtol = P.rtol;
    SorCtl next = P;
    next.parity = L % NB;  // where the previous launch left its output
    next.status = SOR_RUNNING;
    if (sd > 0) {
        // the first sweep s < sd with e < tol (converged) or, failing that, below rtol times the
        // iterate's norm after the launch (fold); static indices keep etot in registers.  Sum i
        // belongs to sweep i (FP32: to the last sweep, sd - 1, so there is never a rollback).
        // A sum that is NaN or +infinity (sums of |delta| are never negative) ends the solve as
        // diverged at that sweep: no later sweep can bring a non-finite iterate below tol, and the
        // reference's loop would spend its whole budget before failing (src/poisson.c:280-284).
        int s_conv = -1, s_fold = -1, s_bad = -1;
#pragma unroll
        for (int i = 0; i < SE; ++i) {
            const int s = kLastOnly ? sd - 1 : i;
            if (s < sd && s_conv < 0 && s_fold < 0 && s_bad < 0) {
                if (!(etot[i] <= DBL_MAX)) s_bad = s;
                else if (etot[i] < tol) s_conv = s;
                else if (rtol > 0.0 && etot[i] < rtol * ntot) s_fold = s;
            }
        }
        if (kNorm && s_conv < 0 && s_fold < 0 && s_bad < 0 && !(ntot <= DBL_MAX)) s_bad = sd - 1;
        const int s_rep = (s_conv >= 0 && s_conv < sd - 1) ? s_conv : sd - 1;  // reported sweep
        double e_rep = 0.0;
#pragma unroll
        for (int i = 0; i < SE; ++i) {
            if ((kLastOnly ? sd - 1 : i) == s_rep) e_rep = etot[i];
        }
        next.e_last = e_rep;
        next.n_last = ntot;
        if (s_conv >= 0 && s_conv < sd - 1) {
            // converged inside the previous launch: the next launch redoes s_conv+1 sweeps from
            // that launch's input (plane (L-1) % NB, untouched since), into plane L % NB (its
            // output, no longer needed); that iterate is the final one (src/poisson.c:273)
            next.status = SOR_ROLLBACK;
            next.k = k_prev + s_conv + 1;
            next.rb_src = (L + NB - 1) % NB;
            next.rb_n = s_conv + 1;
        } else {
            next.k = k_prev + sd;
            if (s_conv >= 0) next.status = SOR_CONVERGED;
            else if (s_fold >= 0) next.status = SOR_FOLD;
            else if (s_bad >= 0) next.status = SOR_DIVERGED;
            else if (next.k >= itmax) next.status = SOR_FAILED;
        }
    } else if (itmax <= k_prev) {
        next.status = SOR_FAILED;
    }
    // the sweeps this launch's sweepers perform (they computed the same from the slot they read)
    const int budget = itmax - (k_prev + sd);
    next.s_done = next.status == SOR_RUNNING ? (budget < S ? (budget > 0 ? budget : 0) : S) : 0;
    if (next.status == SOR_RUNNING && next.s_done > 0) next.launches = P.launches + 1;
    if (lane == 0) *mine = next;
}

template <typename T, int S, int NW, int RB, bool GS, bool XR, bool NORM = false>
__global__ void __launch_bounds__(NW * 64) sor_rb_kernel(SorArgs<T> a) {
    const int ntiles = a.tiles_i * a.tiles_j;
    if ((int)blockIdx.x == ntiles) sor_rb_decider<T, S, NW, NORM>(a, a.launch);
    else sor_rb_sweeper<T, S, NW, RB, GS, XR, NORM>(a, a.launch, sor_tile_of_block(blockIdx.x, ntiles));
}

// Batched form: workgroup b runs tile map[b].tile of solve map[b].inst (inst < 0: padding; tile
// == the solve's tile count: its decider).  All solves of a batch share the launch index L.  The
// solve's arguments are read in place from global memory: a private copy would be indexed by the
// plane number and live in scratch memory.
template <typename T, int S, int NW, int RB, bool GS, bool XR>
__global__ void __launch_bounds__(NW * 64) sor_rb_batch_kernel(const SorArgs<T>* __restrict__ args,
                                                               const SorBlock* __restrict__ map, int L) {
    const SorBlock m = map[blockIdx.x];
    if (m.inst < 0) return;
    const SorArgs<T>& a = args[m.inst];
    if (m.tile == a.tiles_i * a.tiles_j) sor_rb_decider<T, S, NW, false>(a, L);
    else sor_rb_sweeper<T, S, NW, RB, GS, XR, false>(a, L, m.tile);
}

template <typename T, int S, int NW, int RB>
inline int sor_launch_shape(const SorArgs<T>& a, bool gs, hipStream_t st) {
    const int ntiles = a.tiles_i * a.tiles_j;
    const dim3 grid(ntiles + 1), block(NW * 64);  // the tiles' sweepers and one decider
    // FP32 always multiplies by RN(1/B); FP64 does when 1/B is exact
    const bool xr = sizeof(T) == 4 || a.exact_rcp;
    if constexpr (sizeof(T) == 8) {
        if (a.norm && !gs) {  // FP64 with the iterate norm (relative stopping rule)
            if (xr) hipLaunchKernelGGL((sor_rb_kernel<T, S, NW, RB, false, true, true>), grid, block, 0, st, a);
            else hipLaunchKernelGGL((sor_rb_kernel<T, S, NW, RB, false, false, true>), grid, block, 0, st, a);
            return hipGetLastError() == hipSuccess ? 0 : 1;
        }
    }
    if (gs && xr) hipLaunchKernelGGL((sor_rb_kernel<T, S, NW, RB, true, true>), grid, block, 0, st, a);
    else if (gs) hipLaunchKernelGGL((sor_rb_kernel<T, S, NW, RB, true, false>), grid, block, 0, st, a);
    else if (xr) hipLaunchKernelGGL((sor_rb_kernel<T, S, NW, RB, false, true>), grid, block, 0, st, a);
    else hipLaunchKernelGGL((sor_rb_kernel<T, S, NW, RB, false, false>), grid, block, 0, st, a);
    return hipGetLastError() == hipSuccess ? 0 : 1;
}

// The launch shapes compiled in, TileShape {s, nw, rb}: S sweeps per launch, nw waves of rb rows;
// the tile owns (nw*rb - 4s) rows x (128 - 4s) columns.  The default is the first of (5, 4, 6),
// (5, 8, 4), (6, 16, 4), (5, 16, 4) whose tiles fit the device's CUs one per CU: on a small
// grid the GPU is otherwise idle, so thin tiles (more halo, shorter workgroups) win -- per sweep
// at 256^2 FP64 1.50 us with (5, 4, 6) (192 workgroups of 4 waves) against 2.21 us with
// (5, 16, 4) (18 workgroups); at 1024^2 (5, 16, 4) gives 240 workgroups of 16 waves (four per
// SIMD), 1.72x halo redundancy.  The others serve the batched autotuner and the sweep tests.
#define CNV_SOR_SHAPES(X) \
    X(1, 4, 10)           \
    X(2, 4, 10)           \
    X(4, 8, 8)            \
    X(6, 8, 8)            \
    X(8, 8, 10)           \
    X(4, 16, 4)           \
    X(5, 16, 4)           \
    X(6, 16, 4)           \
    X(5, 12, 6)           \
    X(5, 8, 4)            \
    X(5, 8, 8)            \
    X(4, 8, 4)            \
    X(5, 4, 6)

template <typename T>
inline int sor_dispatch(const SorArgs<T>& a, TileShape sh, bool gs, hipStream_t st) {
#define CNV_SOR_CASE(s_, nw_, rb_) \
    if (sh.s == s_ && sh.nw == nw_ && sh.rb == rb_) return sor_launch_shape<T, s_, nw_, rb_>(a, gs, st);
    CNV_SOR_SHAPES(CNV_SOR_CASE)
#undef CNV_SOR_CASE
    return 2;
}

// Batched launch: FP64 uses the corrected division (exact for every B), FP32 the multiply.
template <typename T, int S, int NW, int RB>
inline int sor_batch_launch_shape(const SorArgs<T>* args, const SorBlock* map, int nblocks, int L, bool gs,
                                  hipStream_t st) {
    constexpr bool XR = sizeof(T) == 4;
    const dim3 grid(nblocks), block(NW * 64);
    if (gs) hipLaunchKernelGGL((sor_rb_batch_kernel<T, S, NW, RB, true, XR>), grid, block, 0, st, args, map, L);
    else hipLaunchKernelGGL((sor_rb_batch_kernel<T, S, NW, RB, false, XR>), grid, block, 0, st, args, map, L);
    return hipGetLastError() == hipSuccess ? 0 : 1;
}

template <typename T>
inline int sor_batch_dispatch(const SorArgs<T>* args, const SorBlock* map, int nblocks, int L, TileShape sh,
                              bool gs, hipStream_t st) {
#define CNV_SOR_CASE(s_, nw_, rb_) \
    if (sh.s == s_ && sh.nw == nw_ && sh.rb == rb_) return sor_batch_launch_shape<T, s_, nw_, rb_>(args, map, nblocks, L, gs, st);
    CNV_SOR_SHAPES(CNV_SOR_CASE)
#undef CNV_SOR_CASE
    return 2;
}

}  // namespace cnv
