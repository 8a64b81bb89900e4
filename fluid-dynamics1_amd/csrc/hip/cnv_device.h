// cnv_device.h -- structures shared by the gfx950 kernels and the host side of libcnv.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

namespace cnv {

constexpr int kStencilWidth = 7;  // every Diff1/Diff2 row fits a 7-column window
constexpr int kBlock = 256;       // threads per workgroup (4 wave64)

// Device-side state of one Poisson solve, kept in two slots.  SOR launch L (launch index passed
// by the host, counted from 0 per solve) has one deciding workgroup, which reads slot (L-1)&1 and
// the previous launch's per-tile partial sums and writes slot L&1; its sweeping workgroups read
// slot (L-1)&1 only (the state after launch L-2, and how many sweeps launch L-1 did).  The init
// kernels write slot 1 for launch 0.
enum SorStatus : int {
    SOR_RUNNING = 0,
    SOR_CONVERGED = 1,  // a sweep's L1 update fell below tol
    SOR_FAILED = 2,     // itmax sweeps without convergence
    SOR_FOLD = 4,       // defect correction: the FP32 iterate reached its resolution (rtol)
    SOR_DIVERGED = 8,   // a sweep's L1 update (or the iterate's norm) was NaN or infinite
    SOR_ROLLBACK = 16   // converged inside a launch before its last sweep: the next launch redoes
                        // rb_n sweeps from plane rb_src into plane `parity` (not terminal yet)
};

struct SorCtl {
    int k;              // sweeps accepted before the launch that wrote the slot
    int parity;         // terminal states (and ROLLBACK): the plane holding the final iterate
    int status;         // SorStatus after deciding on the previous launch
    int s_done;         // sweeps the writing launch performs itself (0: none)
    int launches;       // launches that did work (diagnostic)
    int itmax;          // sweep budget of this solve
    int rb_src;         // ROLLBACK: the plane to sweep from (the input of the converged launch)
    int rb_n;           // ROLLBACK: sweeps to redo
    double e_last;      // L1 update of the last accepted sweep
    double tol;         // stop when a sweep's L1 update < tol
    double rtol;        // stop ("fold") when the L1 update < rtol * L1 norm of the iterate (0: never)
    double n_last;      // L1 norm of the iterate after the last accepted sweep (FP32 planes)
};
static_assert(sizeof(SorCtl) == 64, "one state slot per 64 bytes");

// Iterate planes a solve rotates through: launch L reads plane L % NB and writes (L+1) % NB.
// FP64 three, so that the input of the launch before last is still intact when the decision on
// it arrives (a rollback redoes sweeps from it); FP32 two (its stopping rule looks at each
// launch's last sweep only, so it never rolls back).
template <typename T>
struct SorPlanes {
    static constexpr int value = sizeof(T) == 8 ? 3 : 2;
};
// Launches per stopping test of a one-cavity context's FP32 inner solves (SorArgs::test_mask + 1):
// only the launches with L % 4 == 3 test their last sweep; a batch tests every launch.
constexpr int kFp32TestEvery = 4;

// The planes of an FP64 solve, for the kernels that read its final iterate (plane fin->parity).
struct Planes {
    const double* p[3];
};

// Continuity diagnostic: max/min as order-preserving unsigned keys (exact, order independent),
// and the largest |u| or |v| of the stored velocities (a NaN orders above +infinity), which the
// blow-up check reads.
struct Diag {
    unsigned long long kmax;
    unsigned long long kmin;
    unsigned long long kspd;
};

__host__ __device__ inline unsigned long long dkey(double x) {
    unsigned long long b = __builtin_bit_cast(unsigned long long, x);
    return (b >> 63) ? ~b : (b | 0x8000000000000000ull);
}
__host__ __device__ inline double dkey_inv(unsigned long long k) {
    unsigned long long b = (k >> 63) ? (k & 0x7fffffffffffffffull) : ~k;
    return __builtin_bit_cast(double, b);
}

// Per-row stencil tables: row r of an operator has its nonzeros inside columns
// [start[r], start[r] + 7); coef[r*7 + m] multiplies column start[r] + m (zero-padded).
struct Stencils {
    const int* start;
    const double* d1x;  // Diff1(n, order, dx)
    const double* d1y;  // Diff1(n, order, dy)
    const double* d2x;  // Diff2(n, order, dx)
    const double* d2y;  // Diff2(n, order, dy)
    const float* f1x;   // the same tables rounded to FP32 (defect-correction transport)
    const float* f1y;
    const float* f2x;
    const float* f2y;
};

struct WallBC {
    double u1, u2, u3, u4, v1, v2, v3, v4;
};

// SOR launch arguments (one instance per precision).
template <typename T>
struct SorArgs {
    const T* src_f;      // source term: w (plain path, negate = 1) or the FP32 residual
    T* psi0;             // iterate planes (psi2: FP64 only)
    T* psi1;
    T* psi2;
    double* partial;     // [2][kMaxSweepsPerLaunch][ntiles][2]: per-tile L1 update and
                         // iterate norm, double-buffered by launch parity
    SorCtl* ctl;         // the solve's two state slots
    int launch;          // launch index within the solve
    int nr, nc, ld, tiles_i, tiles_j;  // rows (i, y) and columns (j, x) of the grid
    int negate;          // 1: f = -src (the reference's invsig before the solve)
    T c1, c2, c3, B, beta, omb;  // dy*dy, dx*dx, dx*dx*dy*dy, 2*(dx*dx+dy*dy), beta, 1-beta
    T rB;                // RN(1/B)
    int exact_rcp;       // 1: 1/B is exact (B a power of two), so x*rB == RN(x/B)
    int scaled;          // FP64: c1 = c2 = B/4 a power of two, relaxation factors of ordinary size (SorTile); 2: and
                         // the general form all the same
    int norm;            // FP64: also sum the iterate's L1 norm (needed when rtol > 0)
    int test_mask;       // FP32: the stopping rule is tested on the last sweep of the launches
                         // with (launch & test_mask) == test_mask only (test_mask + 1, a power
                         // of two, launches per test); the others sum nothing, leave no
                         // partials, and their decision carries the state forward.  FP64
                         // tests every sweep (0)
};

// A resident solve (sor_resident.h): its exchange planes, decision words and place on the XCDs.
constexpr unsigned long long kMark64 = 0x7ff4c0de0badc0deull;  // signalling NaNs: not an arithmetic result
constexpr unsigned kMark32 = 0x7fa5c0deu;
constexpr int kResidentRows = 16;  // doubles per tile and epoch of partial sums (128 bytes)
constexpr int kClaimStride = 32;   // ints between two XCDs' counters (128 bytes)
constexpr int kBands = 8;          // XCDs of an MI355X, each with a band of tile rows
struct SorResident {
    void* exch;                // three planes of nr rows, pitch ldx, marked where nothing was given yet
    long long xplane;          // elements of one plane
    double* part;              // [4][ntiles][kResidentRows], marked
    unsigned long long* dec;   // [ntiles][8]: each tile's decision word
    double* snap;              // FP64 tiles too large for LDS: two copies of each extended tile
    int* abort;                // set by a wave that gave up waiting; [1]: by a tile of a scaled grid whose source
                               // term is out of the short form's range
    int ldx, ntiles;
    int blocks;                // workgroups of a launch
    int runs;                  // an XCD's tiles are an eighth of all, row after row (0: a band of whole tile rows)
    int epochs, launch0;       // epochs at most; index of the first one within the solve
    int stop;                  // > 0: run to exactly this many sweeps of the solve, without tests
    int spins;                 // polls of one wait before it is given up
    int src, dst;              // planes of the input and of the result
    int rslot, wslot;          // state slots read and written
    int* claim;                // [9][kClaimStride]: tiles taken on each XCD; the deciding workgroup
};
__host__ __device__ inline int band_start(int band, int tiles_i) { return band * tiles_i / kBands; }
constexpr int kNotStored = -1;  // SorCtl::rb_n: the solve has ended, its iterate is not in plane `parity` yet
// FP64 tiles whose two copies fit in LDS
constexpr bool resident_snap_lds(int nw, int rb) { return nw * rb <= 32; }
// Batched resident solves: a tile of a solve, in the band of its tile rows [row_lo, row_hi).
struct ResidentJob {
    int inst, tile, row_lo, row_hi;
};
// The tiles each XCD takes, in order, and the solves in the same order (sor_resident_batch_kernel).
struct ResidentQueues {
    const ResidentJob* jobs;
    int start[kBands + 1];     // XCD x takes jobs [start[x], start[x + 1])
    const int* order;
    int count;                 // solves
    int deciders;              // workgroups that decide: the first on each of XCDs 0, 1, ..., then the second
    int* counters;             // [2 * kBands + 1][kClaimStride], zeroed: workgroups arrived and jobs taken on
                               // each XCD, solves taken by the deciders
};
constexpr int kQueueCounters = (2 * kBands + 1) * kClaimStride;
// What one reset writes before a resident launch: marks over the exchange planes, marks over the
// partial sums, zeros over the decision words and tile counters (in that order from base) and in the two flags at abort.
struct ResidentReset {
    unsigned long long* base;    // nullptr: nothing to reset
    long long exch, part, zero;  // 64-bit words
    unsigned long long mark;     // of the exchange planes
    int* abort;
};

// The start of a Poisson solve, made by the transport launch before it (psi0 == nullptr: none).
struct SolveInit {
    double* psi0;     // zeroed unless keep (the refined form's accumulator, kept by a warm start)
    SorCtl* ctl;      // both slots
    Diag* diag;
    int* budget;      // refined form: the solve's sweep budget
    double tol;
    int itmax, keep;
    ResidentReset rr;
};

// Batched SOR launch: workgroup -> (solve, tile); inst < 0 marks padding workgroups, tile ==
// the solve's tile count its deciding workgroup.
struct SorBlock {
    int inst;
    int tile;
};

// ---- host launch wrappers (defined in the .hip files) ---------------------------------
// SOR launch shape: s sweeps per launch, nw waves per workgroup holding rb rows each; the
// workgroup's tile owns (nw*rb - 4s) rows x (128 - 4s) columns.
struct TileShape { int s, nw, rb; };
constexpr int kMaxSweepsPerLaunch = 8;
inline int tile_cols(const TileShape& t) { return 128 - 4 * t.s; }
inline int tile_rows(const TileShape& t) { return t.nw * t.rb - 4 * t.s; }



int sor_fp64_launch(const SorArgs<double>& a, TileShape shape, bool gs, hipStream_t st);
int sor_fp32_launch(const SorArgs<float>& a, TileShape shape, bool gs, hipStream_t st);
int sor_fp64_resident(const SorArgs<double>& a, const SorResident& r, TileShape shape, bool gs, hipStream_t st);
int sor_fp32_resident(const SorArgs<float>& a, const SorResident& r, TileShape shape, bool gs, hipStream_t st);
bool sor_resident_supported(TileShape shape);
int resident_reset_launch(const ResidentReset& rr, hipStream_t st);
bool sor_shape_supported(TileShape shape);

int wall_vorticity_launch(double* w, const double* u, const double* v, int n, int ld,
                          const Stencils& s, const WallBC& bc, hipStream_t st);
int transport_fp64_launch(const double* w_in, double* w_out, const double* u, const double* v,
                          int n, int ld, const Stencils& s, const WallBC& bc, double rRe,
                          double dt, hipStream_t st, const SolveInit& si = SolveInit{});
int transport_fp32_launch(const double* w_in, double* w_out, const double* u, const double* v,
                          int n, int ld, const Stencils& s, const WallBC& bc, double rRe,
                          double dt, hipStream_t st, const SolveInit& si = SolveInit{});
int diag_reset_launch(Diag* diag, hipStream_t st);
// zero = 0 keeps psi0 (warm start) and only resets the state slots and the diagnostic
int poisson_init_launch(double* psi0, SorCtl* ctl, Diag* diag, int n, int ld, double tol,
                        int itmax, hipStream_t st, int zero = 1, const ResidentReset& rr = ResidentReset{});
// warm start: psi0 <- psi.p[fin->parity] (the previous solve's final iterate)
int warm_start_launch(double* psi0, const Planes& psi, const SorCtl* fin, int n, int ld, hipStream_t st);
int velocity_launch(const Planes& psi, const SorCtl* fin, double* u, double* v, int n, int ld,
                    const Stencils& s, hipStream_t st);
int continuity_launch(const double* u, const double* v, Diag* diag, int n, int ld,
                      const Stencils& s, hipStream_t st);
int euler_launch(double* w, const double* dwdx, const double* dwdy, const double* d2x,
                 const double* d2y, const double* u, const double* v, double rRe, double dt,
                 long long count, hipStream_t st);
int add_launch(const double* a, const double* b, double* out, long long count, int sub,
               hipStream_t st);
int copy_launch(double* dst, const double* src, long long count, hipStream_t st);
int snapshot_launch(const double* w, const Planes& psi, const double* u, const double* v, const SorCtl* fin,
                    double* dst, long long count, hipStream_t st);

// defect correction
// refined-form velocities from psi with FP32 stencils
int velocity_fp32_launch(const double* psi, double* u, double* v, int n, int ld, const Stencils& s,
                         hipStream_t st);
// go != nullptr: do nothing unless *go (the inner solve before was added to psi)
int dc_residual_launch(const double* w, const double* psi, float* r32, int n, int ld, double c1,
                       double c2, double c3, double B, hipStream_t st, const int* go = nullptr);
// psi += e and *budget -= the inner solve's sweeps, if that solve (slot fin) has ended; *go says so
int dc_correct_launch(double* psi, const float* e0, const float* e1, const SorCtl* fin, const int* abort,
                      int* budget, int* go, int n, int ld, hipStream_t st);
// the inner solve's sweep budget: *budget, or itmax without one
int dc_inner_init_launch(float* e0, SorCtl* ctl, int n, int ld, double rtol, double tol, int itmax, hipStream_t st,
                         const int* budget = nullptr, const ResidentReset& rr = ResidentReset{},
                         const int* go = nullptr);

}  // namespace cnv
