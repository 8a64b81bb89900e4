// resident.hip -- host side of the resident solves (sor_resident.h): which contexts use them, when
// they may run, and the launches of one solve.
//
// All workgroups of a resident kernel wait for one another, so they have to be on the GPU
// together.  A kernel's share is counted in CUs per XCD, one a workgroup, and a solve runs resident only while
// the shares of the process's running solves fit on the device (else it runs as launches, at
// once); kernels of other kinds end by themselves and only delay it.  What remains -- another
// process's resident kernel -- is left to the bounded waits: the solve goes on as launches and the
// context uses those from then on.
#include <hip/hip_runtime.h>
#include <limits.h>
#include <stdlib.h>
#include <string.h>

#include <algorithm>
#include <atomic>

#include "cnv.h"
#include "cnv_device.h"
#include "ctx.h"

using namespace cnv;

namespace {

constexpr int kMaxDevices = 64;
// epochs of one launch: at 1024^2 about 16 ms, after which other work gets its turn.  A multiple
// of 64, the longest test cadence of FP32 inner solves, and of 30, so that launches of 5 or 6 sweeps
// that take over between two kernels go on in step with those from the solve's start.
constexpr int kEpochs = 1920;

// Polls of a wait.  A poll of a tile's halo takes 0.24 us at 256^2, 0.9 at 1024^2, 1.65 at 2048^2 (FP32 0.84 to 1.5):
// a wait is given up after 0.25 to 1.7 s.
constexpr int kSpins = 1 << 20;

std::atomic<int> g_units[kMaxDevices];  // CUs per XCD in use by resident solves

// The shapes in order of speed; a solve takes the first whose tiles fit on the GPU together (FP32 inner
// solves and the adjoint's among those with the launches' sweeps an epoch).  us per FP64 sweep:
//   n       64     257    384    513    700    900    1024
//   6,16,2  0.755  0.917  0.938  -
//   5,16,2  0.817  0.972  1.012  1.037  -
//   4,16,2  0.866  1.019  1.028  1.044  -      (600^2 1.14, 660^2 1.22 as eighths of all tiles)
//   6,12,4  1.142  1.294  1.314  1.306  1.350  -
//   6,16,4  1.202  1.372  1.388  1.405  1.445  1.471  -
//   5,16,4  1.272  1.479  1.475  1.493  1.486  1.526  1.459
// and with the short update (powers of two) 0.728 at 64^2, 1.323 at 1024^2;
// so thin tiles first: an epoch's sweeps cost as much as the rows of its tile.  As launches of
// sor_rb.h the default shapes took 1.27 us at 64^2, 1.34 at 257^2 and 2.0 at 1024^2.  Larger grids
// (us per FP64 sweep; "launches" the (5, 16, 4) ones, all that these grids had before; an FP32
// sweep at 1100^2 1.22 against 1.65, at 1600^2 1.77 against 2.55):
//   n        1100  1400  1600  1900  2048
//   5,12,8   2.35  2.38  -
//   5,12,10  3.04  3.07  3.05  -
//   3,12,14  5.12  5.16  5.14  5.16  4.90
//   launches 4.09  4.09  6.56  7.62  8.74
// Their tiles fill the register files; 12 waves of up to 168 registers a lane run them 20-25% faster
// than 8 waves of 256, which leave a SIMD two waves to hide an FP64 operation behind.  Beyond 2072^2
// or so (14 x 18 tiles of 156 x 116 points) the grid does not fit in the registers.
constexpr TileShape kShapes[] = {{6, 16, 2}, {5, 16, 2}, {4, 16, 2}, {6, 12, 4}, {6, 16, 4}, {5, 16, 4},
                                 {5, 12, 8}, {5, 12, 10}, {3, 12, 14}};

// Workgroups per XCD of a resident solve with tiles of shape sh (0: they do not fit together).
int resident_slots(int n, TileShape sh, int per_xcd, SorResident* r) {
    const int ti = (n + tile_rows(sh) - 1) / tile_rows(sh), tj = (n + tile_cols(sh) - 1) / tile_cols(sh);
    r->ntiles = ti * tj;
    // An XCD's tiles are whole tile rows where they fit so; else an eighth of all tiles, whose cells are
    // written through more often: up to 2 more neighbours' tiles are on other XCDs.
    for (r->runs = 0; r->runs < 2; ++r->runs) {
        if (r->runs && (tile_rows(sh) < 2 * sh.s || tile_cols(sh) < 2 * sh.s)) break;  // halos of one tile only
        // every XCD gets as many workgroups as the largest share has tiles, or one of them one more:
        // a workgroup without a tile decides
        int most = 0;
        for (int b = 0; b < kBands; ++b)
            most = std::max(most, r->runs ? band_start(b + 1, r->ntiles) - band_start(b, r->ntiles)
                                          : (band_start(b + 1, ti) - band_start(b, ti)) * tj);
        r->blocks = kBands * most + (r->ntiles == kBands * most);
        const int slots = (r->blocks + kBands - 1) / kBands;
        if (slots <= per_xcd) return slots;  // a workgroup, of 12 or 16 waves, a CU
    }
    return 0;
}

int cus_per_xcd(int dev) {
    int cus = 0;
    if (hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess) return 0;
    return cus / kBands;
}

int launch_resident(const SorArgs<double>& a, const SorResident& r, TileShape sh, bool gs, hipStream_t st) {
    return sor_fp64_resident(a, r, sh, gs, st);
}
int launch_resident(const SorArgs<float>& a, const SorResident& r, TileShape sh, bool gs, hipStream_t st) {
    return sor_fp32_resident(a, r, sh, gs, st);
}

}  // namespace

bool resident_plan(int n, bool fp64, int dev, TileShape base, bool named, bool in_step, ResidentPlan* p) {
    const int per_xcd = dev < kMaxDevices ? cus_per_xcd(dev) : 0;
    if (per_xcd < 8) return false;
    *p = ResidentPlan{};
    SorResident& r = p->r;
    int slots = 0;
    if (named) {
        p->shape = base;
        if (sor_resident_supported(base)) slots = resident_slots(n, base, per_xcd, &r);
    } else {
        for (const TileShape& sh : kShapes) {
            if (in_step && sh.s != base.s) continue;
            p->shape = sh;
            slots = resident_slots(n, sh, per_xcd, &r);
            if (slots) break;
        }
    }
    if (!slots) return false;
    p->units = slots;
    resident_layout(n, fp64, p->shape, p);
    p->launch_s = base.s;
    return true;
}

int resident_polls(int dflt) {
    const char* s = getenv("CNV_RESIDENT_POLLS");
    char* end = nullptr;
    const long v = s ? strtol(s, &end, 10) : -1;
    return s && end != s && !*end && v >= 0 && v <= INT_MAX ? (int)v : dflt;
}

void resident_layout(int n, bool fp64, TileShape sh, ResidentPlan* p) {
    SorResident& r = p->r;
    p->shape = sh;
    p->fp64 = fp64;
    p->tiles_i = (n + tile_rows(sh) - 1) / tile_rows(sh);
    p->tiles_j = (n + tile_cols(sh) - 1) / tile_cols(sh);
    r.ntiles = p->tiles_i * p->tiles_j;
    // exchange rows start on 128-byte lines: rows of two bands share none
    r.ldx = (n + 1 + 31) / 32 * 32;
    r.xplane = (long long)r.ldx * n;
    p->launch_s = sh.s;
    r.epochs = kEpochs;
    r.spins = resident_polls(kSpins);
    ResidentReset& rr = p->reset;
    rr.exch = 3 * r.xplane / (fp64 ? 1 : 2);
    rr.part = 4LL * r.ntiles * kResidentRows;
    rr.zero = 8LL * r.ntiles + (kBands + 1) * kClaimStride / 2;  // decision words, counters
    rr.mark = fp64 ? kMark64 : ((unsigned long long)kMark32 << 32 | kMark32);
    p->words = rr.exch + rr.part + rr.zero;
    p->snap = fp64 && !resident_snap_lds(sh.nw, sh.rb) ? 2LL * r.ntiles * sh.nw * sh.rb * 128 : 0;
}

void resident_bind(ResidentPlan* p, unsigned long long* words, double* snap, SorCtl* ctl) {
    ResidentReset& rr = p->reset;
    rr.base = words;
    rr.abort = reinterpret_cast<int*>(ctl + 2);
    SorResident& r = p->r;
    r.exch = words;
    r.part = reinterpret_cast<double*>(words + rr.exch);
    r.dec = words + rr.exch + rr.part;
    r.claim = reinterpret_cast<int*>(r.dec + 8LL * r.ntiles);
    r.snap = snap;
    r.abort = rr.abort;
}

int resident_setup(cnv_ctx* c, Resident use) {
    const bool named = c->p.sweeps_per_launch > 0 || c->p.tile_waves > 0 || c->p.wave_rows > 0;
    ResidentPlan p;
    const bool fp64 = c->p.precision == CNV_PREC_FP64;
    if (use == Resident::none ||
        !resident_plan(c->n, fp64, c->p.device, c->shape, named, !fp64 || use == Resident::in_step, &p))
        return CNV_OK;
    if (hipMalloc(&c->d_res, sizeof(*c->d_res) * p.words) != hipSuccess ||
        (p.snap && hipMalloc(&c->d_res_snap, sizeof(double) * p.snap) != hipSuccess)) {
        (void)hipGetLastError();  // no room for them: the solves run as launches
        if (c->d_res) (void)hipFree(c->d_res);
        c->d_res = nullptr;
        c->d_res_snap = nullptr;
        return CNV_OK;
    }
    resident_bind(&p, c->d_res, c->d_res_snap, c->ctl);
    c->res = p;
    c->res_on = true;
    return CNV_OK;
}

bool resident_enter(int dev, int units) {
    if (dev < 0 || dev >= kMaxDevices) return false;
    std::atomic<int>& used = g_units[dev];
    if (used.fetch_add(units) + units <= cus_per_xcd(dev)) return true;
    used.fetch_sub(units);
    return false;
}
void resident_leave(int dev, int units) { g_units[dev].fetch_sub(units); }

template <typename T>
int resident_chunks(cnv_ctx* c, const ResidentPlan& p, SorArgs<T> a, bool gs, int itmax, hipStream_t st, SorCtl* h,
                    SorCtl* fin, int* fin_slot, int* resume, bool* gave_up, bool* src_out, Behind* behind) {
    constexpr int NB = SorPlanes<T>::value;
    SorResident r = p.r;
    a.tiles_i = p.tiles_i;
    a.tiles_j = p.tiles_j;
    r.launch0 = 0;
    r.stop = 0;
    r.src = 0;
    r.rslot = 0;
    *resume = -1;
    *gave_up = false;
    const long long most = (long long)itmax / p.shape.s + 2LL * kEpochs;  // epochs of a whole budget
    while (r.launch0 <= most) {
        r.dst = (r.src + 1) % NB;
        r.wslot = r.rslot ^ 1;
        if (a.scaled) a.scaled = *src_out ? 2 : 1;
        LAUNCH(c, launch_resident(a, r, p.shape, gs, st));
        const bool first = r.launch0 == 0 && r.stop == 0 && behind && behind->queue;
        if (first) behind->queued = true;
        int rc = first && !behind->read ? behind->queue(c, behind->arg) : CNV_OK;
        if (rc) return rc;
        HIPC(c, hipMemcpyAsync(h, a.ctl, 4 * sizeof(SorCtl), hipMemcpyDeviceToHost, st));
        if (first && behind->read) {
            HIPC(c, hipEventRecord(behind->read, st));
            if ((rc = behind->queue(c, behind->arg))) return rc;
            HIPC(c, hipEventSynchronize(behind->read));
        } else {
            HIPC(c, hipStreamSynchronize(st));
        }
        int flags[2];
        memcpy(flags, h + 2, sizeof(flags));
        const bool aborted = flags[0];
        *src_out = flags[1];
        const SorCtl s = h[r.wslot];
        if (aborted || (s.status == SOR_DIVERGED && p.shape.s != p.launch_s)) {
            *gave_up = aborted;
            // both slots as the chunk found them; FP32 planes: into plane 0, where launch 0 reads
            HIPC(c, hipMemcpyAsync(a.ctl + r.wslot, a.ctl + r.rslot, sizeof(SorCtl), hipMemcpyDeviceToDevice, st));
            if (NB == 2 && r.src == 1)
                HIPC(c, hipMemcpyAsync(a.psi0, a.psi1, sizeof(T) * (size_t)a.nr * a.ld, hipMemcpyDeviceToDevice, st));
            *resume = NB == 2 ? 0 : r.src;
            return CNV_OK;
        }
        if (sor_done(s.status)) {
            if (s.rb_n != kNotStored || r.stop > 0) {
                *fin = s;
                *fin_slot = r.wslot;
                if (behind) behind->counts = first;
                return CNV_OK;
            }
            r.stop = s.k;  // once more, to exactly the sweep the solve ended with
        } else {
            r.src = r.dst;
            r.rslot = r.wslot;
            r.launch0 += kEpochs;
        }
        LAUNCH(c, resident_reset_launch(p.reset, st));
    }
    return cnv_fail(c, CNV_ERR_HIP, "SOR state did not terminate after %d epochs", r.launch0);
}
template int resident_chunks<double>(cnv_ctx*, const ResidentPlan&, SorArgs<double>, bool, int, hipStream_t, SorCtl*,
                                     SorCtl*, int*, int*, bool*, bool*, Behind*);

template <typename T>
int run_sor_resident(cnv_ctx* c, const SorArgs<T>& a, SorCtl* final_ctl, bool* ran, Behind* behind) {
    const int dev = c->p.device;
    // with other resident solves running that leave too few CUs, this one runs as launches
    *ran = c->res_on && c->res.fp64 == (sizeof(T) == 8) && resident_enter(dev, c->res.units);
    if (!*ran) return CNV_OK;
    int resume = -1;
    bool gave_up = false;
    int rc = resident_chunks<T>(c, c->res, a, c->p.poisson_type == 1, c->p.itmax, c->stream, c->h_ctl, final_ctl,
                                      &c->fin_slot, &resume, &gave_up, &c->src_out, behind);
    // a failed call may leave its kernel running, which holds its place until it has ended
    if (rc) (void)hipStreamSynchronize(c->stream);
    resident_leave(dev, c->res.units);
    if (rc) return rc;
    if (gave_up) c->res_on = false;
    if (resume >= 0 && (rc = run_sor_launches<T>(c, a, final_ctl, resume))) return rc;
    // captured launches read a solve's end from slot 1, whichever call made it
    if (c->p.use_graph && c->fin_slot != 1) {
        HIPC(c, hipMemcpyAsync(c->ctl + 1, c->ctl, sizeof(SorCtl), hipMemcpyDeviceToDevice, c->stream));
        c->fin_slot = 1;
    }
    return CNV_OK;
}
template int run_sor_resident<double>(cnv_ctx*, const SorArgs<double>&, SorCtl*, bool*, Behind*);
template int run_sor_resident<float>(cnv_ctx*, const SorArgs<float>&, SorCtl*, bool*, Behind*);
