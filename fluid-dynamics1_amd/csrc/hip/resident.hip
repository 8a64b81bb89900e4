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
// of 64, the longest test cadence of FP32 inner solves.
constexpr int kEpochs = 1984;

std::atomic<int> g_units[kMaxDevices];  // CUs per XCD in use by resident solves

// The shapes in order of speed; a solve takes the first whose tiles fit on the GPU together (an FP32
// inner solve among those with the launches' sweeps, its test cadence).  us per FP64 sweep:
//   n       64     257    384    513    700    900    1024
//   6,16,2  0.755  0.917  0.938  -
//   5,16,2  0.817  0.972  1.012  1.037  -
//   4,16,2  0.866  1.019  1.028  1.044  -
//   6,12,4  1.142  1.294  1.314  1.306  1.350  -
//   6,16,4  1.202  1.372  1.388  1.405  1.445  1.471  -
//   5,16,4  1.272  1.479  1.475  1.493  1.486  1.526  1.459
// so thin tiles first: an epoch's sweeps cost as much as the rows of its tile.  As launches of
// sor_rb.h the default shapes took 1.27 us at 64^2, 1.34 at 257^2 and 2.0 at 1024^2.
constexpr TileShape kShapes[] = {{6, 16, 2}, {5, 16, 2}, {4, 16, 2}, {6, 12, 4}, {6, 16, 4}, {5, 16, 4}};

}  // namespace

// Workgroups per XCD of a resident solve with tiles of shape sh (0: they do not fit together).
static int resident_slots(int n, TileShape sh, int per_xcd, SorResident* r) {
    const int ti = (n + tile_rows(sh) - 1) / tile_rows(sh), tj = (n + tile_cols(sh) - 1) / tile_cols(sh);
    // every XCD gets as many workgroups as the largest band has tiles, or one of them one more: a
    // workgroup without a tile decides
    int most = 0;
    for (int b = 0; b < kBands; ++b) most = std::max(most, (band_start(b + 1, ti) - band_start(b, ti)) * tj);
    r->ntiles = ti * tj;
    r->blocks = kBands * most + (r->ntiles == kBands * most);
    const int slots = (r->blocks + kBands - 1) / kBands;
    // a workgroup of 16 waves (or of 8 with two tile copies in LDS) fills a CU; two of 4 waves fit
    return slots <= (sh.nw > 4 ? per_xcd : 2 * per_xcd) ? slots : 0;
}

int resident_setup(cnv_ctx* c) {
    const int dev = c->p.device;
    int cus = 0;
    if (dev >= kMaxDevices || hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess ||
        cus < 8 * kBands)
        return CNV_OK;
    const int per_xcd = cus / kBands;
    const bool fp64 = c->p.precision == CNV_PREC_FP64;
    SorResident& r = c->res;
    int slots = 0;
    const bool named = c->p.sweeps_per_launch > 0 || c->p.tile_waves > 0 || c->p.wave_rows > 0;
    if (named) {
        c->res_shape = c->shape;
        if (sor_resident_supported(c->shape)) slots = resident_slots(c->n, c->shape, per_xcd, &r);
    } else {
        for (const TileShape& sh : kShapes) {
            if (!fp64 && sh.s != c->shape.s) continue;
            c->res_shape = sh;
            slots = resident_slots(c->n, sh, per_xcd, &r);
            if (slots) break;
        }
    }
    if (!slots) return CNV_OK;
    const TileShape sh = c->res_shape;
    c->res_tiles_i = (c->n + tile_rows(sh) - 1) / tile_rows(sh);
    c->res_tiles_j = (c->n + tile_cols(sh) - 1) / tile_cols(sh);
    c->res_units = std::min(slots, per_xcd);
    // exchange rows start on 128-byte lines: rows of two bands share none
    r.ldx = (c->n + 1 + 31) / 32 * 32;
    r.xplane = (long long)r.ldx * c->n;
    ResidentReset& rr = c->res_reset;
    rr.exch = 3 * r.xplane / (fp64 ? 1 : 2);
    rr.part = 4LL * r.ntiles * kResidentRows;
    const long long words = 8LL * r.ntiles;  // decision words
    rr.zero = words + (kBands + 1) * kClaimStride / 2;
    rr.mark = fp64 ? kMark64 : ((unsigned long long)kMark32 << 32 | kMark32);
    rr.abort = reinterpret_cast<int*>(c->ctl + 2);
    HIPC(c, hipMalloc(&c->d_res, sizeof(*c->d_res) * (rr.exch + rr.part + rr.zero)));
    rr.base = c->d_res;
    r.exch = c->d_res;
    r.part = reinterpret_cast<double*>(c->d_res + rr.exch);
    r.dec = c->d_res + rr.exch + rr.part;
    r.claim = reinterpret_cast<int*>(r.dec + words);
    r.abort = rr.abort;
    if (fp64 && !resident_snap_lds(sh.nw, sh.rb)) {
        HIPC(c, hipMalloc(&c->d_res_snap, sizeof(double) * 2 * (size_t)r.ntiles * sh.nw * sh.rb * 128));
        r.snap = c->d_res_snap;
    }
    r.epochs = kEpochs;
    c->res_on = true;
    return CNV_OK;
}

static int resident_launch(cnv_ctx* c, SorArgs<double> a, const SorResident& r, bool gs) {
    a.tiles_i = c->res_tiles_i;
    a.tiles_j = c->res_tiles_j;
    return sor_fp64_resident(a, r, c->res_shape, gs, c->stream);
}
static int resident_launch(cnv_ctx* c, SorArgs<float> a, const SorResident& r, bool gs) {
    a.tiles_i = c->res_tiles_i;
    a.tiles_j = c->res_tiles_j;
    return sor_fp32_resident(a, r, c->res_shape, gs, c->stream);
}

// The chunks of a solve; *resume < 0 when it has ended, else the launch index to go on from (a
// wave of the last chunk gave up waiting: its input is where that launch reads).
template <typename T>
static int resident_chunks(cnv_ctx* c, const SorArgs<T>& a, SorCtl* final_ctl, int* resume) {
    constexpr int NB = SorPlanes<T>::value;
    const bool gs = c->p.poisson_type == 1;
    SorResident r = c->res;
    r.launch0 = 0;
    r.stop = 0;
    r.src = 0;
    r.rslot = 0;
    *resume = -1;
    const long long most = (long long)c->p.itmax / c->res_shape.s + 2LL * kEpochs;  // epochs of a whole budget
    while (r.launch0 <= most) {
        r.dst = (r.src + 1) % NB;
        r.wslot = r.rslot ^ 1;
        LAUNCH(c, resident_launch(c, a, r, gs));
        HIPC(c, hipMemcpyAsync(c->h_ctl, c->ctl, 3 * sizeof(SorCtl), hipMemcpyDeviceToHost, c->stream));
        HIPC(c, hipStreamSynchronize(c->stream));
        int aborted = 0;
        memcpy(&aborted, &c->h_ctl[2], sizeof(aborted));
        if (aborted) {
            // both slots as the chunk found them; FP32 planes: into plane 0, where launch 0 reads
            HIPC(c, hipMemcpyAsync(c->ctl + r.wslot, c->ctl + r.rslot, sizeof(SorCtl), hipMemcpyDeviceToDevice, c->stream));
            if (NB == 2 && r.src == 1)
                HIPC(c, hipMemcpyAsync(a.psi0, a.psi1, sizeof(T) * c->cells, hipMemcpyDeviceToDevice, c->stream));
            *resume = NB == 2 ? 0 : r.src;
            return CNV_OK;
        }
        const SorCtl st = c->h_ctl[r.wslot];
        if (sor_done(st.status) && st.rb_n == kNotStored && r.stop == 0) {
            r.stop = st.k;  // once more, to exactly the sweep the solve ended with
            LAUNCH(c, resident_reset_launch(c->res_reset, c->stream));
            continue;
        }
        if (sor_done(st.status)) {
            *final_ctl = st;
            c->fin_slot = r.wslot;
            return CNV_OK;
        }
        LAUNCH(c, resident_reset_launch(c->res_reset, c->stream));
        r.src = r.dst;
        r.rslot = r.wslot;
        r.launch0 += kEpochs;
    }
    return cnv_fail(c, CNV_ERR_HIP, "SOR state did not terminate after %d epochs", r.launch0);
}

template <typename T>
int run_sor_resident(cnv_ctx* c, const SorArgs<T>& a, SorCtl* final_ctl, bool* ran) {
    *ran = false;
    if (!c->res_on) return CNV_OK;
    int cus = 0;
    if (hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, c->p.device) != hipSuccess) return CNV_OK;
    std::atomic<int>& used = g_units[c->p.device];
    if (used.fetch_add(c->res_units) + c->res_units > cus / kBands) {
        used.fetch_sub(c->res_units);
        return CNV_OK;  // other resident solves are running: this one runs as launches
    }
    *ran = true;
    int resume = -1;
    const int rc = resident_chunks<T>(c, a, final_ctl, &resume);
    // a failed call may leave its kernel running, which holds its place until it has ended
    if (rc) (void)hipStreamSynchronize(c->stream);
    used.fetch_sub(c->res_units);
    if (rc || resume < 0) return rc;
    c->res_on = false;
    return run_sor_launches<T>(c, a, final_ctl, resume);
}
template int run_sor_resident<double>(cnv_ctx*, const SorArgs<double>&, SorCtl*, bool*);
template int run_sor_resident<float>(cnv_ctx*, const SorArgs<float>&, SorCtl*, bool*);
