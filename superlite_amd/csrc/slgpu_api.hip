// C ABI of libslgpu.so (include/slgpu.h): context, uploads, per-iteration entry points.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstdio>
#include <cstring>
#include <initializer_list>
#include <mutex>
#include <string>
#include <vector>

#include "slgpu_device.h"
#include "slgpu_internal.h"
#include "slgpu_sample.h"

using namespace slgpu;

// Device memory of slgpu_opacity_build_noalloc: the staging of the per-call ion populations
// (oc and ginv, 2 * nion * nc doubles), so that entry point needs no allocation.  Each GPU
// holds its own copy until the process ends; every call on a GPU shares it (calls that
// overlap on one GPU race).  Host code never uses the array's name as an address: its
// device address is resolved once per device at slgpu_create (hipGetSymbolAddress) and
// kept in g_scratch_ptr.
constexpr size_t SLGPU_SCRATCH_BYTES = (size_t)4 << 20;
static __device__ __align__(256) unsigned char scratch[SLGPU_SCRATCH_BYTES];

namespace {

thread_local std::string g_err;

constexpr int SCRATCH_MAX_DEVICES = 64;
std::mutex g_scratch_mu;
void *g_scratch_ptr[SCRATCH_MAX_DEVICES] = {};

// device address of `scratch` on the current device, resolved on first use per device
hipError_t scratch_address(void **out)
{
    int dev = 0;
    hipError_t e = hipGetDevice(&dev);
    if (e != hipSuccess) return e;
    if (dev < 0 || dev >= SCRATCH_MAX_DEVICES) return hipErrorInvalidDevice;
    std::lock_guard<std::mutex> lk(g_scratch_mu);
    if (!g_scratch_ptr[dev]) {
        void *p = nullptr;
        e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
        if (e != hipSuccess) return e;
        g_scratch_ptr[dev] = p;
    }
    *out = g_scratch_ptr[dev];
    return hipSuccess;
}

int fail(int code, const std::string &msg)
{
    g_err = msg;
    return code;
}

#define HIPCHK(call)                                                                    \
    do {                                                                                \
        hipError_t e_ = (call);                                                         \
        if (e_ != hipSuccess)                                                           \
            return fail(SLGPU_EHIP, std::string(#call) + ": " + hipGetErrorString(e_)); \
    } while (0)

template <class T>
int dalloc(slgpu_ctx *c, T **p, size_t n)
{
    void *q = nullptr;
    if (n == 0) n = 1;
    hipError_t e = hipMalloc(&q, n * sizeof(T));
    if (e != hipSuccess) return fail(SLGPU_ENOMEM, std::string("hipMalloc: ") + hipGetErrorString(e));
    (void)hipMemsetAsync(q, 0, n * sizeof(T), c->stream);
    c->allocations.push_back(q);
    *p = (T *)q;
    return 0;
}

// one allocation for several arrays, one directly behind the other (multiples of 4 bytes; 8-byte
// elements before 4-byte ones)
int dparts(slgpu_ctx *c, std::initializer_list<std::pair<void **, size_t>> parts)
{
    size_t n = 0;
    for (const auto &x : parts) n += x.second;
    char *p = nullptr;
    const int rc = dalloc(c, &p, n);
    if (rc) return rc;
    for (const auto &x : parts) {
        *x.first = p;
        p += x.second;
    }
    return 0;
}

void dfree(slgpu_ctx *c, void *p)
{
    if (!p) return;
    auto it = std::find(c->allocations.begin(), c->allocations.end(), p);
    if (it != c->allocations.end()) c->allocations.erase(it);
    hipFree(p);
}

struct PhaseTimer {
    slgpu_ctx *c;
    int slot;
    PhaseTimer(slgpu_ctx *c_, int s) : c(c_), slot(s) { hipEventRecord(c->ev[2 * s], c->stream); }
    // the phase ends when its outputs are on the host
    int stop(Outputs &out)
    {
        hipError_t e = out.finish(c->ev[2 * slot + 1]);
        if (e != hipSuccess) return fail(SLGPU_EHIP, std::string("device: ") + hipGetErrorString(e));
        float ms = 0.f;
        hipEventElapsedTime(&ms, c->ev[2 * slot], c->ev[2 * slot + 1]);
        c->t_ms[slot] += ms + out.tail_ms();
        return 0;
    }
};

// SOURCE/sourcenumbers.f90:83-145 with one rank, in_srcepwr = 1, tot_esurf = 0
int64_t source_numbers(const std::vector<double> &emit, int64_t nstot, std::vector<int> &nvol)
{
    const int nc = (int)emit.size();
    double etot = 0.0;
    int64_t ncactive = 0;
    for (double e : emit) {
        etot += std::pow(e, 1.0);
        if (e > 0.0) ncactive++;
    }
    nvol.assign(nc, 0);
    if (ncactive == 0) return -1;
    const int64_t nsavail = nstot;
    const double invn = 1.0 / (double)nsavail;
    const double einv = etot == 0.0 ? 0.0 : 1.0 / etot;
    double edone = 0.0;
    int64_t ndone = 0;
    for (int l = 0; l < nc; ++l) {
        const double en = std::pow(emit[l], 1.0);
        if (en == 0.0) continue;
        int64_t n = std::max<int64_t>(1, (int64_t)(en * (double)nsavail * einv));
        if (edone * einv > (double)ndone * invn) n = n + 1;
        nvol[l] = (int)n;
        edone += en;
        ndone += n;
    }
    int64_t s = 0;
    for (int v : nvol) s += v;
    int64_t nextra = nstot - s;
    if (nextra > nc) return -2;       // sourcenumbers.f90:130-131
    const int64_t nsmean = nstot / ncactive;
    while (nextra != 0) {
        for (int l = 0; l < nc; ++l) {
            if (nextra == 0) break;
            if (nvol[l] < nsmean) continue;
            const int sg = nextra > 0 ? 1 : -1;
            nvol[l] += sg;
            nextra -= sg;
        }
    }
    s = 0;
    for (int v : nvol) s += v;
    return s;
}

}  // namespace

extern "C" {

const char *slgpu_last_error_message(void) { return g_err.c_str(); }

int slgpu_create(const slgpu_config *cfg, slgpu_ctx **out)
{
    if (!cfg || !out) return fail(SLGPU_EINVAL, "null argument");
    if (cfg->nx < 1 || cfg->nx > 8192) return fail(SLGPU_EINVAL, "nx must be in 1..8192");
    if (cfg->ng < 2 || cfg->ng > 32767) return fail(SLGPU_EINVAL, "ng must be in 2..32767 (groupmod.f:38)");
    if (cfg->nep < 1 || cfg->nep > 1024 || cfg->nepg < 1)
        return fail(SLGPU_EINVAL, "nep must be in 1..1024 and nepg >= 1");
    if (cfg->npartmax < 1 || cfg->npartmax > (int64_t)1 << 31)
        return fail(SLGPU_EINVAL, "npartmax must be in 1..2^31");
    if (cfg->precision != SLGPU_FP64 && cfg->precision != SLGPU_MIXED)
        return fail(SLGPU_EINVAL, "precision must be SLGPU_FP64 or SLGPU_MIXED");
    if ((cfg->ampfact != 0 && cfg->ampfact != 1) || (cfg->thm_aniso != 0 && cfg->thm_aniso != 1))
        return fail(SLGPU_EINVAL, "ampfact and thm_aniso must be 0 or 1");
    int ndev = 0;
    if (hipGetDeviceCount(&ndev) != hipSuccess || ndev < 1)
        return fail(SLGPU_EHIP, "no HIP device visible");
    void *scr = nullptr;
    {
        hipError_t e = scratch_address(&scr);
        if (e != hipSuccess)
            return fail(SLGPU_EHIP, std::string("hipGetSymbolAddress(scratch): ") + hipGetErrorString(e));
    }
    slgpu_ctx *c = new slgpu_ctx();
    c->scratch = scr;
    c->cfg = *cfg;
    c->nx = cfg->nx;
    c->ng = cfg->ng;
    Dev &d = c->d;
    std::memset(&d, 0, sizeof(d));
    d.nx = cfg->nx;
    d.ng = cfg->ng;
    d.nep = cfg->nep;
    d.nepg = cfg->nepg;
    d.tauddmc = cfg->tauddmc;
    d.taulump = cfg->taulump;
    d.puretran = cfg->puretran;
    d.precision = cfg->precision;
    d.ampfact = cfg->ampfact != 0;
    d.thm_aniso = cfg->thm_aniso != 0;
    d.max_steps = cfg->max_steps > 0 ? cfg->max_steps : ((int64_t)1 << 26);
    d.seed = cfg->seed;
    if (hipStreamCreateWithFlags(&c->stream, hipStreamNonBlocking) != hipSuccess) {
        delete c;
        return fail(SLGPU_EHIP, "hipStreamCreate failed");
    }
    for (int k = 0; k < 24; ++k) hipEventCreate(&c->ev[k]);
    const size_t nc = c->nx, ng = c->ng, cg = nc * ng, np = cfg->npartmax;
    int rc = 0;
    rc |= dalloc(c, (double **)&d.xarr, nc + 1);
    rc |= dalloc(c, (double **)&d.vxarr, nc + 1);
    rc |= dalloc(c, (double **)&d.divv, nc);
    rc |= dalloc(c, (double **)&d.vol, nc);
    rc |= dalloc(c, (double **)&d.dvdr, nc);
    rc |= dalloc(c, (double **)&d.c3divv, nc);
    rc |= dalloc(c, (double **)&d.wl, ng + 1);
    rc |= dalloc(c, (double **)&d.wlinv, ng + 1);
    rc |= dalloc(c, (double **)&d.gff, 81 * 41);
    rc |= dalloc(c, &d.hckt, nc);
    rc |= dalloc(c, &d.hlparr, nc);
    rc |= dalloc(c, &d.ffB, (size_t)nc * FF_NU);
    rc |= dalloc(c, &d.ffclamp, nc);
    rc |= dalloc(c, &d.ffC, (size_t)nc * FF_NU);
    rc |= dalloc(c, &d.tempinv, nc);
    // what crosses the bus together lies together, in the order of the transfers
    rc |= dparts(c, {{(void **)&d.temp, nc * 8}, {(void **)&d.mass, nc * 8}, {(void **)&d.natomfr, 30 * nc * 8},
                     {(void **)&d.natom_in, nc * 8}, {(void **)&d.vol_in, nc * 8},
                     {(void **)&d.nelec_in, nc * 8}, {(void **)&d.el_z, 30 * 4}});
    rc |= dparts(c, {{(void **)&d.sig, nc * 8}, {(void **)&d.capgrey, nc * 8}, {(void **)&d.capross, nc * 8}});
    rc |= dalloc(c, &d.capT, cg);
    rc |= dalloc(c, &d.cap64, cg);
    rc |= dalloc(c, &d.cap32, cg);
    rc |= dalloc(c, &d.emiss, cg);
    d.capem32 = d.cap32;
    d.capemgrey = d.capgrey;
    d.nlte = 0;
    rc |= dalloc(c, &d.specarr, cg);
    rc |= dparts(c, {{(void **)&d.opaclump, 11 * nc * 8}, {(void **)&d.emitprob, (size_t)cfg->nep * nc * 8}});
    rc |= dalloc(c, &d.emitcum, cg);
    rc |= dparts(c, {{(void **)&d.emit, nc * 8}, {(void **)&d.radtemp, nc * 8}});
    rc |= dalloc(c, &d.srccum, cg);
    rc |= dalloc(c, &d.srctot, nc);
    rc |= dalloc(c, &d.cell, nc);
    rc |= dalloc(c, &d.gcapT, cg);
    rc |= dalloc(c, &d.gmpart, (size_t)2 * ((ng + 63) / 64) * nc);
    rc |= dalloc(c, &d.ctpart, (size_t)2 * ((ng + 1023) / 1024) * nc);
    rc |= dalloc(c, &d.cprob, nc);
    rc |= dalloc(c, &d.gprob, cg);
    rc |= dalloc(c, &d.gshort, cg);
    rc |= dalloc(c, &d.cshort, nc);
    rc |= dalloc(c, &d.geo, nc);
    rc |= dalloc(c, &d.gorder, cg);
    rc |= dalloc(c, &d.cumL, cg);
    rc |= dalloc(c, &d.cumR, cg);
    rc |= dalloc(c, &d.cumD, cg);
    rc |= dalloc(c, &d.cumS, cg);
    rc |= dalloc(c, &d.btab, (size_t)NTAB * nc * BT_K);
    rc |= dalloc(c, (int64_t **)&d.pstart, nc + 1);
    rc |= dalloc(c, &d.px, np);
    rc |= dalloc(c, &d.pmu, np);
    rc |= dalloc(c, &d.pwl, np);
    rc |= dalloc(c, &d.pe, np);
    rc |= dalloc(c, &d.pstat, np);
    rc |= dalloc(c, &d.pig, np);
    rc |= dalloc(c, &d.perr, np);
    rc |= dalloc(c, &d.pnstep, np);
    rc |= dalloc(c, &d.pix, np);
    rc |= dparts(c, {{(void **)&d.tally, nc * 8}, {(void **)&d.eamp, nc * 8}, {(void **)&d.tot, 8 * 8},
                     {(void **)&d.ct, 10 * 8}, {(void **)&d.queue, 8}});
    // grd_jrad gets one atomic per event; on small grids every lane hits a few hot
    // (cell, group) entries, so blocks add into one of R replicas (R from a 256 MiB budget,
    // 1..32) that a reduction folds into replica 0 after the transport
    {
        const size_t budget = (size_t)256 << 20;
        size_t r = budget / (cg * sizeof(double));
        d.jrad_copies = (int)(r < 1 ? 1 : (r > 32 ? 32 : r));
    }
    rc |= dalloc(c, &d.jrad, (size_t)d.jrad_copies * cg);
    rc |= dparts(c, {{(void **)&d.lum, ng * 8}, {(void **)&d.dev, ng * 8}, {(void **)&d.num, ng * 4}});
    rc |= dalloc(c, &d.flags, 1);
    rc |= dalloc(c, &d.eos_ni, 30);
    rc |= dalloc(c, &d.eos_e, 30 * 31);
    rc |= dalloc(c, &d.eos_q, 30 * 31);
    rc |= dalloc(c, &d.eos_g1, 30 * 31);
    rc |= dalloc(c, &d.eos_amass, 30);
    rc |= dalloc(c, &d.eos_sahac2, nc);
    rc |= dparts(c, {{(void **)&c->eos_temp, nc * 8}, {(void **)&c->eos_mass, nc * 8},
                     {(void **)&c->eos_massfr, 30 * nc * 8}, {(void **)&c->eos_nelec, nc * 8},
                     {(void **)&c->eos_natom, nc * 8}, {(void **)&c->eos_natomfr, 30 * nc * 8},
                     {(void **)&c->eos_niter, nc * 4}});
    if (!rc) {
        // inputs of a call: 35 per-cell numbers and two per ion; what does not fit goes straight from the
        // caller's memory.  Outputs: up to 20 bytes per (cell, group) and some hundred per cell, or the
        // particles' 49 bytes each (10^6 of them on 4 x 16 groups: 434 ms through a ring sized by the
        // grid alone, 2.8 ms so).
        const hipError_t e = c->io.create(std::min((size_t)4 << 20, nc * 167 * 8 + 4096),
                                          std::max(20 * cg + 200 * 8 * nc, 49 * np));
        if (e != hipSuccess) rc = fail(SLGPU_ENOMEM, std::string("hipHostMalloc: ") + hipGetErrorString(e));
    }
    if (rc) {
        std::string m = g_err;
        slgpu_destroy(c);
        return fail(SLGPU_ENOMEM, m);
    }
    hipStreamSynchronize(c->stream);
    *out = c;
    return 0;
}

int slgpu_destroy(slgpu_ctx *c)
{
    if (!c) return 0;
    if (c->stream) hipStreamSynchronize(c->stream);
    for (void *p : c->allocations) hipFree(p);
    c->allocations.clear();
    c->io.destroy();
    for (int k = 0; k < 24; ++k) hipEventDestroy(c->ev[k]);
    if (c->stream) hipStreamDestroy(c->stream);
    delete c;
    return 0;
}

void *slgpu_stream(slgpu_ctx *c) { return c ? (void *)c->stream : nullptr; }

int slgpu_set_grid(slgpu_ctx *c, const double *xarr, const double *vxarr, const double *divv,
                   const double *vol, const double *rcell)
{
    if (!c || !xarr || !vxarr || !divv || !vol || !rcell) return fail(SLGPU_EINVAL, "null argument");
    const int nx = c->nx;
    for (int i = 0; i < nx; ++i)
        if (!(xarr[i + 1] > xarr[i])) return fail(SLGPU_EINVAL, "grd_xarr must increase");
    for (int i = 0; i < nx; ++i)
        if (!(vol[i] > 0.0)) return fail(SLGPU_EINVAL, "grd_vol must be positive");
    c->h_xarr.assign(xarr, xarr + nx + 1);
    c->h_vxarr.assign(vxarr, vxarr + nx + 1);
    c->h_divv.assign(divv, divv + nx);
    c->h_vol.assign(vol, vol + nx);
    c->h_rcell.assign(rcell, rcell + nx);
    HIPCHK(hipMemcpyAsync((void *)c->d.xarr, xarr, (nx + 1) * 8, hipMemcpyHostToDevice, c->stream));
    HIPCHK(hipMemcpyAsync((void *)c->d.vxarr, vxarr, (nx + 1) * 8, hipMemcpyHostToDevice, c->stream));
    HIPCHK(hipMemcpyAsync((void *)c->d.divv, divv, nx * 8, hipMemcpyHostToDevice, c->stream));
    HIPCHK(hipMemcpyAsync((void *)c->d.vol, vol, nx * 8, hipMemcpyHostToDevice, c->stream));
    // per-cell constants of the transport, with the kernels' own expression order (one
    // IEEE operation each, so the values are the ones the step would compute)
    std::vector<double> dvdr(nx), c3(nx);
    for (int i = 0; i < nx; ++i) {
        dvdr[i] = (vxarr[i + 1] - vxarr[i]) / (xarr[i + 1] - xarr[i]);
        c3[i] = (3.0 * PC_C) / divv[i];
    }
    HIPCHK(hipMemcpyAsync((void *)c->d.dvdr, dvdr.data(), nx * 8, hipMemcpyHostToDevice, c->stream));
    HIPCHK(hipMemcpyAsync((void *)c->d.c3divv, c3.data(), nx * 8, hipMemcpyHostToDevice, c->stream));
    HIPCHK(hipStreamSynchronize(c->stream));
    c->have_grid = true;
    return 0;
}

static int upload_lines(slgpu_ctx *c);
static int build_lines64(slgpu_ctx *c);
static int build_bfxs(slgpu_ctx *c);

int slgpu_set_groups(slgpu_ctx *c, const double *wl)
{
    if (!c || !wl) return fail(SLGPU_EINVAL, "null argument");
    const int ng = c->ng;
    for (int g = 0; g < ng; ++g)
        if (!(wl[g + 1] > wl[g]) || !(wl[g] > 0.0)) return fail(SLGPU_EINVAL, "grp_wl must be positive and increasing");
    c->h_wl.assign(wl, wl + ng + 1);
    std::vector<double> inv(ng + 1);
    for (int g = 0; g <= ng; ++g) inv[g] = 1.0 / wl[g];     // groupmod.f:50-51
    HIPCHK(hipMemcpyAsync((void *)c->d.wl, wl, (ng + 1) * 8, hipMemcpyHostToDevice, c->stream));
    HIPCHK(hipMemcpyAsync((void *)c->d.wlinv, inv.data(), (ng + 1) * 8, hipMemcpyHostToDevice, c->stream));
    HIPCHK(hipStreamSynchronize(c->stream));
    c->have_groups = true;
    int rc = 0;
    if (c->have_lines && c->have_ions) rc = upload_lines(c);
    if (!rc && c->have_bf && c->have_ions) rc = build_bfxs(c);
    return rc;
}

int slgpu_set_ions(slgpu_ctx *c, int nion, const int *ion_iz, const int *ion_ii)
{
    if (!c || nion < 0 || (nion > 0 && (!ion_iz || !ion_ii))) return fail(SLGPU_EINVAL, "bad ion list");
    for (int k = 0; k < nion; ++k) {
        if (ion_iz[k] < 1 || ion_iz[k] > 30 || ion_ii[k] < 1 || ion_ii[k] > ion_iz[k])
            return fail(SLGPU_EINVAL, "ion (iz, ii) out of range");
        if (k > 0 && (ion_iz[k] < ion_iz[k - 1] || (ion_iz[k] == ion_iz[k - 1] && ion_ii[k] <= ion_ii[k - 1])))
            return fail(SLGPU_EINVAL, "ion list must be ascending in (iz, ii)");
    }
    c->nion = nion;
    c->d.nion = nion;
    c->h_ion_iz.assign(ion_iz, ion_iz + nion);
    c->h_ion_ii.assign(ion_ii, ion_ii + nion);
    dfree(c, c->d.ion_z);
    dfree(c, c->d.ion_i);
    dfree(c, c->eos_oc);
    dfree(c, c->stage);
    dfree(c, c->vjp_out);
    dfree(c, c->eos_vjp);
    dfree(c, c->d.ocg);
    dfree(c, c->d.ocT);
    dfree(c, c->d.ginvT);
    dfree(c, c->d.goc);
    dfree(c, (void *)c->d.bfxs);
    dfree(c, c->d.bfmask);
    const size_t nc = c->nx;
    int rc = 0;
    rc |= dalloc(c, &c->d.ocg, (size_t)std::max(nion, 1) * nc);
    rc |= dalloc(c, &c->d.ginvT, (size_t)std::max(nion, 1) * nc);
    rc |= dalloc(c, &c->d.goc, vjp_acc_doubles(nion, nc));
    rc |= dalloc(c, &c->d.ocT, (size_t)(nion + 30) * nc);     // tail: ff coordinates per element
    rc |= dalloc(c, (double **)&c->d.bfxs, (size_t)std::max(nion, 1) * c->ng);
    rc |= dalloc(c, &c->d.bfmask, (size_t)(std::max(nion, 1) + 31) / 32 * c->ng);
    rc |= dalloc(c, &c->d.ion_z, std::max(nion, 1));
    rc |= dalloc(c, &c->d.ion_i, std::max(nion, 1));
    c->eos_oc = c->stage = c->vjp_out = c->eos_vjp = nullptr;
    const size_t ni = std::max(nion, 1);
    rc |= dparts(c, {{(void **)&c->eos_oc, ni * nc * 8}, {(void **)&c->eos_ginv, ni * nc * 8}});
    rc |= dalloc(c, &c->stage, 2 * ni * nc);
    rc |= dalloc(c, &c->vjp_out, (33 + ni) * nc);
    rc |= dalloc(c, &c->eos_vjp, (64 + ni) * nc);
    if (rc) return rc;
    c->d.ffW = c->d.goc + (size_t)GACC_COPIES * std::max(nion, 1) * nc;
    c->d.gcell = c->d.ffW + (size_t)GACC_COPIES * FF_NU * nc;
    c->d.gfr = c->d.gcell + 2 * nc;
    if (nion > 0) {
        HIPCHK(hipMemcpyAsync(c->d.ion_z, ion_iz, nion * sizeof(int), hipMemcpyHostToDevice, c->stream));
        HIPCHK(hipMemcpyAsync(c->d.ion_i, ion_ii, nion * sizeof(int), hipMemcpyHostToDevice, c->stream));
        HIPCHK(hipStreamSynchronize(c->stream));
    }
    c->have_ions = true;
    c->have_eos = false;
    if (c->have_lines && c->have_groups) rc = upload_lines(c);
    if (!rc && c->have_bf && c->have_groups) rc = build_bfxs(c);
    return rc;
}

int slgpu_set_lines(slgpu_ctx *c, int64_t nline, const float *wl0, const float *gxs,
                    const float *chilw, const int16_t *iz, const int16_t *ii)
{
    if (!c || nline < 0 || (nline > 0 && (!wl0 || !gxs || !chilw || !iz || !ii)))
        return fail(SLGPU_EINVAL, "bad line list");
    if (nline > ((int64_t)1 << 31) - 1) return fail(SLGPU_EINVAL, "too many lines");
    for (int64_t l = 1; l < nline; ++l)
        if (wl0[l] < wl0[l - 1]) return fail(SLGPU_EINVAL, "line list must be sorted by wl0 (bbxsmod.f:126-179)");
    c->nline = nline;
    c->h_wl0.assign(wl0, wl0 + nline);
    c->h_gxs.assign(gxs, gxs + nline);
    c->h_chilw.assign(chilw, chilw + nline);
    c->h_liz.assign(iz, iz + nline);
    c->h_lii.assign(ii, ii + nline);
    c->have_lines = true;
    if (c->have_groups && c->have_ions) return upload_lines(c);
    return 0;
}

// Lines of group g (1-based) are those with wlsub(g) <= wl0 < wlsub(g+1), the
// pointer walk of physical_opacity.f:118-125 on a sorted list; lines outside the grid and
// lines of ions without populations are dropped (they add nothing, physical_opacity.f:146).
static int upload_lines(slgpu_ctx *c)
{
    const int ng = c->ng;
    int lut[31][32];
    for (auto &r : lut)
        for (int &v : r) v = -1;
    for (int k = 0; k < c->nion; ++k) lut[c->h_ion_iz[k]][c->h_ion_ii[k]] = k;
    std::vector<LineRec> recs;
    recs.reserve(c->nline);
    std::vector<int> cnt(ng + 2, 0);
    int g = 1;
    for (int64_t l = 0; l < c->nline; ++l) {
        const double w = (double)c->h_wl0[l] * PC_ANG;
        if (w < c->h_wl[0] || !(w < c->h_wl[ng])) continue;
        while (g < ng && !(c->h_wl[g] > w)) ++g;      // wlsub(g) <= w < wlsub(g+1)
        const int zi = c->h_liz[l], ii = c->h_lii[l];
        const int k = (zi >= 1 && zi <= 30 && ii >= 1 && ii <= 31) ? lut[zi][ii] : -1;
        if (k < 0) continue;
        recs.push_back(LineRec{c->h_gxs[l], c->h_chilw[l], k, 0});
        cnt[g]++;
    }
    std::vector<int> gstart(ng + 2, 0);
    for (int q = 1; q <= ng; ++q) gstart[q + 1] = gstart[q] + cnt[q];
    c->nline_used = (int64_t)recs.size();
    // the backward's copy: each group's lines ordered by ion (stable), so a run of one ion's
    // lines shares its population and its gradient accumulator
    std::vector<LineRec> recs_ion(recs);
    for (int q = 1; q <= ng; ++q)
        std::stable_sort(recs_ion.begin() + gstart[q], recs_ion.begin() + gstart[q + 1],
                         [](const LineRec &a, const LineRec &b) { return a.ion < b.ion; });
    // pad of an ion-ordered record: the lines left in its run of one ion within its group
    // (itself included), so the backward walks a run as a counted loop
    for (int q = 1; q <= ng; ++q)
        for (int l = gstart[q + 1] - 1; l >= gstart[q]; --l)
            recs_ion[l].pad = (l + 1 < gstart[q + 1] && recs_ion[l + 1].ion == recs_ion[l].ion)
                                  ? recs_ion[l + 1].pad + 1 : 1;
    dfree(c, (void *)c->d.lines);
    dfree(c, (void *)c->d.lines_ion);
    dfree(c, (void *)c->d.gstart);
    dfree(c, c->d.lines64);
    c->d.lines64 = nullptr;
    c->d.line_step = 0.0;
    int rc = 0;
    rc |= dalloc(c, (LineRec **)&c->d.lines, recs.size());
    rc |= dalloc(c, (LineRec **)&c->d.lines_ion, recs.size());
    rc |= dalloc(c, (int **)&c->d.gstart, ng + 2);
    if (rc) return rc;
    if (!recs.empty()) {
        HIPCHK(hipMemcpyAsync((void *)c->d.lines, recs.data(), recs.size() * sizeof(LineRec),
                              hipMemcpyHostToDevice, c->stream));
        HIPCHK(hipMemcpyAsync((void *)c->d.lines_ion, recs_ion.data(), recs_ion.size() * sizeof(LineRec),
                              hipMemcpyHostToDevice, c->stream));
    }
    HIPCHK(hipMemcpyAsync((void *)c->d.gstart, gstart.data(), (ng + 2) * sizeof(int),
                          hipMemcpyHostToDevice, c->stream));
    // largest lower level, and whether every line suits the exponential tables
    double top = 0.0;
    bool plain = true;
    for (const LineRec &q : recs) {
        plain = plain && q.chilw >= 0.0f && std::isfinite(q.chilw) && std::isfinite(q.gxs);
        top = std::max(top, (double)q.chilw);
    }
    c->line_top = plain && !recs.empty() ? std::max(top, 1.0) : 0.0;
    if (c->cfg.precision == SLGPU_FP64 || c->have_nlte) rc = build_lines64(c);
    HIPCHK(hipStreamSynchronize(c->stream));
    return rc;
}

// The FP64 line sums' records and tables (FP64 builds and NLTE builds).  The step is the largest
// lower level over the table's range, rounded up to a multiple of 1/16 so that every split is exact;
// lists with negative or non-finite records keep exp() per line.
static int build_lines64(slgpu_ctx *c)
{
    if (!(c->line_top > 0.0) || c->d.line_step > 0.0) return 0;
    const double step = std::ceil(c->line_top / (EXP_K1 * EXP_K2 - 1) * 16.0) / 16.0;
    if (step > 1e6) return 0;
    int rc = dalloc(c, &c->d.lines64, c->nline_used);
    if (!rc && !c->d.etab) rc = dalloc(c, &c->d.etab, (size_t)EXP_ROWS * c->nx);
    if (rc) return rc;
    c->d.line_step = step;
    launch_lines64(c, c->nline_used);
    HIPCHK(hipGetLastError());
    return 0;
}

static int build_bfxs(slgpu_ctx *c)
{
    float *d1 = nullptr, *d2 = nullptr;
    int *diz = nullptr, *dii = nullptr;
    int rc = 0;
    rc |= dalloc(c, &d1, c->h_ph1.size());
    rc |= dalloc(c, &d2, c->h_ph2.size());
    rc |= dalloc(c, &diz, std::max(c->nion, 1));
    rc |= dalloc(c, &dii, std::max(c->nion, 1));
    if (rc) return rc;
    HIPCHK(hipMemcpyAsync(d1, c->h_ph1.data(), c->h_ph1.size() * 4, hipMemcpyHostToDevice, c->stream));
    HIPCHK(hipMemcpyAsync(d2, c->h_ph2.data(), c->h_ph2.size() * 4, hipMemcpyHostToDevice, c->stream));
    if (c->nion > 0) {
        HIPCHK(hipMemcpyAsync(diz, c->h_ion_iz.data(), c->nion * 4, hipMemcpyHostToDevice, c->stream));
        HIPCHK(hipMemcpyAsync(dii, c->h_ion_ii.data(), c->nion * 4, hipMemcpyHostToDevice, c->stream));
    }
    launch_bfxs(c, d1, d2, diz, dii);
    HIPCHK(hipGetLastError());
    HIPCHK(hipStreamSynchronize(c->stream));
    dfree(c, d1); dfree(c, d2); dfree(c, diz); dfree(c, dii);
    return 0;
}

int slgpu_set_bf_tables(slgpu_ctx *c, const float *ph1, const float *ph2)
{
    if (!c || !ph1 || !ph2) return fail(SLGPU_EINVAL, "null argument");
    c->h_ph1.assign(ph1, ph1 + 6 * 7 * 30 * 30);
    c->h_ph2.assign(ph2, ph2 + 7 * 30 * 30);
    c->have_bf = true;
    if (c->have_groups && c->have_ions) return build_bfxs(c);
    return 0;
}

int slgpu_set_ff_table(slgpu_ctx *c, const double *gff)
{
    if (!c || !gff) return fail(SLGPU_EINVAL, "null argument");
    HIPCHK(hipMemcpyAsync((void *)c->d.gff, gff, 81 * 41 * 8, hipMemcpyHostToDevice, c->stream));
    HIPCHK(hipStreamSynchronize(c->stream));
    c->have_ff = true;
    return 0;
}

}  // extern "C"

namespace {

// The opacity build (O2-O8) with the per-call staging of the ion populations oc and ginv
// (2 * nion * nc doubles) at `stage`: the context's for slgpu_opacity_build, the
// library's static scratch array for slgpu_opacity_build_noalloc.
// the NLTE part of a build (physical_opacity_nlte): per-call inputs and extra outputs
struct NlteCall {
    const double *radtemp, *ndens;
    float *out_capemit;
    double *out_capemitgrey, *out_npop;
};

int opacity_build_impl(slgpu_ctx *c, const slgpu_gas *gas, int flags, double *out_cap64,
                       float *out_cap32, double *out_sig, double *out_capgrey,
                       double *out_capross, float *out_emiss, double *stage,
                       const NlteCall *nlc = nullptr)
{
    const int nc = c->nx, ng = c->ng, nion = c->nion;
    // present elements (ff adds exactly zero for the others, physical_opacity.f:240-241)
    int nel = 0, elz[30] = {};
    for (int z = 1; z <= 30; ++z) {
        bool any = false;
        for (int i = 0; i < nc && !any; ++i) any = gas->natomfr[(size_t)i * 30 + z - 1] != 0.0;
        if (any) elz[nel++] = z;
    }
    c->d.nel = nel;
    c->hckt_max = 0.0;
    for (int i = 0; i < nc; ++i) c->hckt_max = std::max(c->hckt_max, PC_H * PC_C / (PC_KB * gas->temp[i]));
    PhaseTimer tm(c, 0);
    // per-call host inputs (small: nc and nion*nc doubles)
    double *dn = c->d.natom_in, *dv = c->d.vol_in, *de = c->d.nelec_in;   // kept for the backward
    double *doc = stage, *dgi = stage + (size_t)std::max(nion, 1) * nc;
    Inputs in(c->io, c->stream);
    in.add(c->d.temp, gas->temp, nc * 8);
    in.add(c->d.mass, gas->mass, nc * 8, true);
    in.add(c->d.natomfr, gas->natomfr, (size_t)nc * 30 * 8, true);
    in.add(dn, gas->natom, nc * 8, true);
    in.add(dv, gas->vol, nc * 8, true);
    in.add(de, gas->nelec, nc * 8, true);
    in.add(c->d.el_z, elz, sizeof(elz), true);
    if (nion > 0) {
        in.add(doc, gas->oc, (size_t)nion * nc * 8);
        in.add(dgi, gas->ginv, (size_t)nion * nc * 8, true);
    }
    if (nlc) {
        in.add(c->nl.radtemp, nlc->radtemp, nc * 8);
        in.add(c->nl.ndens, nlc->ndens, (size_t)2 * nc * 8, true);
        HIPCHK(hipMemsetAsync(c->nl.flag, 0, sizeof(int), c->stream));
    }
    HIPCHK(in.send());
    hipEventRecord(c->ev[22], c->stream);
    launch_cell_prep(c, dn, dv, de, doc, dgi, flags);
    hipEventRecord(c->ev[10], c->stream);
    if (nlc) launch_opacity_nlte(c, flags, ff_prefactor(), rgg_scratch(c));
    else launch_opacity(c, flags);
    hipEventRecord(c->ev[11], c->stream);
    if (nlc) {
        launch_cell_tables(c);
        launch_nlte_means(c);
    } else {
        launch_opacity_finish(c);
    }
    hipEventRecord(c->ev[23], c->stream);
    HIPCHK(hipGetLastError());
    const size_t cg = (size_t)nc * ng;
    Outputs out(c->io, c->stream);
    int flag = 0;
    if (nlc) {
        out.add(&flag, c->nl.flag, sizeof(int));
        out.add(nlc->out_capemit, c->nl.capemit32, cg * 4);
        out.add(nlc->out_capemitgrey, c->nl.capemitgrey, nc * 8);
        out.add(nlc->out_npop, c->nl.pop, (size_t)nc * c->nl.n * 8);
    }
    out.add(out_cap64, c->d.cap64, cg * 8);
    out.add(out_cap32, c->d.cap32, cg * 4);
    out.add(out_emiss, c->d.emiss, cg * 4);
    out.add(out_sig, c->d.sig, nc * 8);
    out.add(out_capgrey, c->d.capgrey, nc * 8, true);
    out.add(out_capross, c->d.capross, nc * 8, true);
    out.start();
    int rc = tm.stop(out);
    if (!rc && flag) {
        c->have_opacity = false;            // the device opacity is partly overwritten
        c->have_prep = false;
        return fail(SLGPU_EINVAL, "nlte opacity: rate matrix numerically singular");
    }
    float kms = 0.f;
    hipEventElapsedTime(&kms, c->ev[10], c->ev[11]);
    c->t_ms[5] += kms;
    hipEventElapsedTime(&kms, c->ev[22], c->ev[23]);
    c->t_ms[11] += kms;
    c->opac_flags = flags;
    // the emission opacity the DDMC prep and the samplers read (gridmod.f:41,56 grd_capemit,
    // grd_capemitgrey; the absorption opacity in LTE)
    c->d.nlte = nlc ? 1 : 0;
    c->d.capem32 = nlc ? c->nl.capemit32 : c->d.cap32;
    c->d.capemgrey = nlc ? c->nl.capemitgrey : c->d.capgrey;
    c->have_prep = false;
    if (rc) {
        c->have_opacity = false;
        return rc;
    }
    c->have_opacity = true;
    return 0;
}

int check_opacity_inputs(slgpu_ctx *c, const slgpu_gas *gas)
{
    if (!c || !gas || !gas->temp || !gas->natom || !gas->vol || !gas->mass || !gas->nelec ||
        !gas->natomfr || (c->nion > 0 && (!gas->oc || !gas->ginv)))
        return fail(SLGPU_EINVAL, "null gas state");
    if (!(c->have_groups && c->have_lines && c->have_bf && c->have_ff && c->have_ions))
        return fail(SLGPU_EORDER, "groups, lines, ions and bf/ff tables must be set first");
    for (int i = 0; i < c->nx; ++i)
        if (!(gas->temp[i] > 0.0)) return fail(SLGPU_EINVAL, "gas_temp must be positive (gas_update.f:71-72)");
    return 0;
}

}  // namespace

extern "C" {

int slgpu_opacity_build(slgpu_ctx *c, const slgpu_gas *gas, int flags, double *out_cap64,
                        float *out_cap32, double *out_sig, double *out_capgrey,
                        double *out_capross, float *out_emiss)
{
    int rc = check_opacity_inputs(c, gas);
    if (rc) return rc;
    return opacity_build_impl(c, gas, flags, out_cap64, out_cap32, out_sig, out_capgrey,
                              out_capross, out_emiss, c->stage);
}

int slgpu_opacity_build_noalloc(slgpu_ctx *c, const slgpu_gas *gas, int flags,
                                double *out_cap64, float *out_cap32, double *out_sig,
                                double *out_capgrey, double *out_capross, float *out_emiss)
{
    int rc = check_opacity_inputs(c, gas);
    if (rc) return rc;
    const size_t need = (size_t)2 * std::max(c->nion, 1) * c->nx * sizeof(double);
    if (need > SLGPU_SCRATCH_BYTES)
        return fail(SLGPU_EINVAL, "opacity_build_noalloc: 2*nion*nc doubles exceed the " +
                                      std::to_string(SLGPU_SCRATCH_BYTES) + "-byte scratch array");
    double *stage = (double *)c->scratch;
    if (!stage) return fail(SLGPU_EORDER, "scratch array address not resolved at slgpu_create");
    return opacity_build_impl(c, gas, flags, out_cap64, out_cap32, out_sig, out_capgrey,
                              out_capross, out_emiss, stage);
}

int slgpu_set_nlte_data(slgpu_ctx *c, int nlev, int nlin, int ncoll, const double *glev,
                        const int *llw, const int *lup, const double *wl0, const double *f,
                        const double *gl, const double *gu, const double *aul, const double *bul,
                        const double *blu, const int *llw_coll, const int *lup_coll,
                        const double *coll_c, const double *dele, const int *lev_pi,
                        const double *pi_c, const double *rr_c, const double *dele_pi)
{
    if (!c || !glev || !llw || !lup || !wl0 || !f || !gl || !gu || !aul || !bul || !blu ||
        (ncoll > 0 && (!llw_coll || !lup_coll || !coll_c || !dele)) || !lev_pi || !pi_c ||
        !rr_c || !dele_pi)
        return fail(SLGPU_EINVAL, "null argument");
    if (!(c->have_groups && c->have_ions)) return fail(SLGPU_EORDER, "groups and ions must be set first");
    if (nlev < 2 || nlev > 1024 || nlin < 1 || ncoll < 0)
        return fail(SLGPU_EINVAL, "nlte data: need 2 <= nlev <= 1024, nlin >= 1, ncoll >= 0");
    // distinct level pairs (the reference's rate coefficients are set per pair, so a repeated
    // radiative pair would keep only its last line, a repeated collision pair would add)
    std::vector<char> seen((size_t)nlev * nlev, 0), seenc((size_t)nlev * nlev, 0), seenl(nlev, 0);
    for (int k = 0; k < nlin; ++k) {
        if (llw[k] < 1 || lup[k] > nlev || !(llw[k] < lup[k]))
            return fail(SLGPU_EINVAL, "nlte data: radiative lines need 1 <= llw < lup <= nlev");
        char &v = seen[(size_t)(llw[k] - 1) * nlev + lup[k] - 1];
        if (v) return fail(SLGPU_EINVAL, "nlte data: repeated radiative level pair");
        v = 1;
    }
    for (int k = 0; k < ncoll; ++k) {
        if (llw_coll[k] < 1 || lup_coll[k] > nlev || !(llw_coll[k] < lup_coll[k]))
            return fail(SLGPU_EINVAL, "nlte data: collision lines need 1 <= llw < lup <= nlev");
        char &v = seenc[(size_t)(llw_coll[k] - 1) * nlev + lup_coll[k] - 1];
        if (v) return fail(SLGPU_EINVAL, "nlte data: repeated collision level pair");
        v = 1;
    }
    for (int k = 0; k < nlev; ++k) {
        if (lev_pi[k] < 1 || lev_pi[k] > nlev || seenl[lev_pi[k] - 1])
            return fail(SLGPU_EINVAL, "nlte data: lev_pi must list every level once");
        seenl[lev_pi[k] - 1] = 1;
    }
    const int ng = c->ng, nc = c->nx;
    // group of each line: the first grp_wl edge above wl0 (physical_opacity_nlte.f:166-172),
    // 0 outside the grid; and the lines of each group in file order
    std::vector<int> igs(nlin), cnt(ng + 2, 0);
    for (int k = 0; k < nlin; ++k) {
        const double w = wl0[k] * PC_ANG;
        int g = 0;
        while (g <= ng && !(c->h_wl[g] > w)) ++g;
        igs[k] = (g >= 1 && g <= ng) ? g : 0;
        if (igs[k]) cnt[igs[k]]++;
    }
    std::vector<int> hstart(ng + 2, 0);
    for (int g = 1; g <= ng; ++g) hstart[g + 1] = hstart[g] + cnt[g];
    std::vector<int> fill(hstart);
    std::vector<HLine> hline(std::max(hstart[ng + 1], 1));
    for (int k = 0; k < nlin; ++k)
        if (igs[k]) hline[fill[igs[k]]++] = {f[k], gl[k], gu[k], aul[k], wl0[k], llw[k] - 1, lup[k] - 1};
    int kH = -1;
    for (int k = 0; k < c->nion; ++k)
        if (c->h_ion_iz[k] == 1 && c->h_ion_ii[k] == 1) kH = k;
    NlteDev &q = c->nl;
    if (c->have_nlte) {
        void *ps[] = {q.glev, q.aul, q.bul, q.blu, q.cc, q.dele, q.pic, q.rrc,
                      q.delepi, q.llw, q.lup, q.igs, q.cl, q.cu, q.levpi, q.hstart, q.hline, q.radtemp,
                      q.A, q.pop, q.popT, q.flag, q.capemitT, q.emissT,
                      q.capemit32, q.capemitgrey};
        for (void *p : ps) dfree(c, p);
        c->have_nlte = false;
        if (c->d.nlte) {            // the last build's emission opacity is gone with them
            c->d.nlte = 0;
            c->d.capem32 = c->d.cap32;
            c->d.capemgrey = c->d.capgrey;
            c->have_opacity = false;
            c->have_prep = false;
        }
    }
    q = NlteDev();
    q.n = nlev; q.nlin = nlin; q.ncoll = ncoll; q.kH = kH;
    const int nc1 = std::max(ncoll, 1);
    int rc = 0;
    rc |= dalloc(c, &q.glev, nlev);
    rc |= dalloc(c, &q.aul, nlin); rc |= dalloc(c, &q.bul, nlin); rc |= dalloc(c, &q.blu, nlin);
    rc |= dalloc(c, &q.cc, (size_t)4 * nc1); rc |= dalloc(c, &q.dele, nc1);
    rc |= dalloc(c, &q.pic, (size_t)4 * nlev); rc |= dalloc(c, &q.rrc, (size_t)4 * nlev);
    rc |= dalloc(c, &q.delepi, nlev);
    rc |= dalloc(c, &q.llw, nlin); rc |= dalloc(c, &q.lup, nlin); rc |= dalloc(c, &q.igs, nlin);
    rc |= dalloc(c, &q.cl, nc1); rc |= dalloc(c, &q.cu, nc1); rc |= dalloc(c, &q.levpi, nlev);
    rc |= dalloc(c, &q.hstart, ng + 2); rc |= dalloc(c, &q.hline, hline.size());
    rc |= dparts(c, {{(void **)&q.radtemp, (size_t)nc * 8}, {(void **)&q.ndens, (size_t)2 * nc * 8}});
    if (!nlte_in_lds(nlev)) rc |= dalloc(c, &q.A, (size_t)nc * nlev * (nlev + 1));
    rc |= dalloc(c, &q.pop, (size_t)nc * nlev); rc |= dalloc(c, &q.popT, (size_t)nc * nlev);
    rc |= dalloc(c, &q.flag, 1);
    rc |= dalloc(c, &q.capemitT, (size_t)nc * ng); rc |= dalloc(c, &q.emissT, (size_t)nc * ng);
    rc |= dalloc(c, &q.capemit32, (size_t)nc * ng); rc |= dalloc(c, &q.capemitgrey, nc);
    if (rc) return rc;
    auto up = [&](void *dst, const void *src, size_t bytes) {
        return hipMemcpyAsync(dst, src, bytes, hipMemcpyHostToDevice, c->stream);
    };
    HIPCHK(up(q.glev, glev, nlev * 8));
    HIPCHK(up(q.aul, aul, nlin * 8)); HIPCHK(up(q.bul, bul, nlin * 8)); HIPCHK(up(q.blu, blu, nlin * 8));
    if (ncoll > 0) {
        HIPCHK(up(q.cc, coll_c, (size_t)4 * ncoll * 8)); HIPCHK(up(q.dele, dele, ncoll * 8));
        HIPCHK(up(q.cl, llw_coll, ncoll * 4)); HIPCHK(up(q.cu, lup_coll, ncoll * 4));
    }
    HIPCHK(up(q.pic, pi_c, (size_t)4 * nlev * 8)); HIPCHK(up(q.rrc, rr_c, (size_t)4 * nlev * 8));
    HIPCHK(up(q.delepi, dele_pi, nlev * 8));
    HIPCHK(up(q.llw, llw, nlin * 4)); HIPCHK(up(q.lup, lup, nlin * 4)); HIPCHK(up(q.igs, igs.data(), nlin * 4));
    HIPCHK(up(q.levpi, lev_pi, nlev * 4));
    HIPCHK(up(q.hstart, hstart.data(), (ng + 2) * 4)); HIPCHK(up(q.hline, hline.data(), hline.size() * sizeof(HLine)));
    HIPCHK(hipStreamSynchronize(c->stream));
    c->have_nlte = true;
    rc = build_lines64(c);          // NLTE builds take the FP64 line sums in both precision forms
    HIPCHK(hipStreamSynchronize(c->stream));
    return rc;
}

int slgpu_opacity_build_nlte(slgpu_ctx *c, const slgpu_gas *gas, const double *radtemp,
                             const double *ndens, int flags, double *out_cap64, float *out_cap32,
                             float *out_capemit, double *out_sig, double *out_capgrey,
                             double *out_capemitgrey, double *out_capross, float *out_emiss,
                             double *out_npop)
{
    int rc = check_opacity_inputs(c, gas);
    if (rc) return rc;
    if (!c->have_nlte) return fail(SLGPU_EORDER, "NLTE data must be set first");
    if (!radtemp || !ndens) return fail(SLGPU_EINVAL, "null argument");
    if (!(flags & SLGPU_NOBB))
        for (int i = 0; i < c->nx; ++i) {
            if (gas->mass[i] <= 0.0) continue;
            if (!(radtemp[i] > 0.0) || !(ndens[2 * (size_t)i] > 0.0) || !(ndens[2 * (size_t)i + 1] >= 0.0))
                return fail(SLGPU_EINVAL, "nlte opacity: radtemp and the H I density must be positive "
                                          "and the H II density non-negative in every massive cell");
        }
    NlteCall nlc{radtemp, ndens, out_capemit, out_capemitgrey, out_npop};
    return opacity_build_impl(c, gas, flags, out_cap64, out_cap32, out_sig, out_capgrey,
                              out_capross, out_emiss, c->stage, &nlc);
}

int slgpu_nlte_rad_est(slgpu_ctx *c, double *radtemp, double *out_jrad)
{
    if (!c || !radtemp) return fail(SLGPU_EINVAL, "null argument");
    if (!c->have_transport) return fail(SLGPU_EORDER, "slgpu_transport must run first");
    const int nc = c->nx, ng = c->ng;
    for (int i = 0; i < nc; ++i)
        if (!(radtemp[i] > 0.0)) return fail(SLGPU_EINVAL, "grd_radtemp must be positive");
    if (!c->est) {
        int rc = dalloc(c, &c->est, (size_t)nc * (ng + 1));
        if (rc) return rc;
    }
    double *drt = c->est, *dj = out_jrad ? c->est + nc : nullptr;
    Inputs in(c->io, c->stream);
    in.add(drt, radtemp, nc * 8);
    HIPCHK(in.send());
    launch_nlte_rad_est(c, drt, dj);
    HIPCHK(hipGetLastError());
    Outputs out(c->io, c->stream);
    out.add(radtemp, drt, nc * 8);
    out.add(out_jrad, dj, (size_t)nc * ng * 8, true);
    out.start();
    HIPCHK(out.finish(c->ev[1]));
    return 0;
}

int slgpu_ddmc_prep(slgpu_ctx *c, const double *radtemp, double lbol, double *out_opaclump,
                    double *out_emitprob, double *out_emit, double *out_sthermal)
{
    if (!c || !radtemp) return fail(SLGPU_EINVAL, "null argument");
    if (!c->have_opacity || !c->have_grid) return fail(SLGPU_EORDER, "opacity and grid must be set first");
    const int nc = c->nx;
    for (int i = 0; i < nc; ++i)
        if (!(radtemp[i] > 0.0)) return fail(SLGPU_EINVAL, "grd_radtemp must be positive");
    // SOURCE/sourceenergy.f90:23-50 (surface-like thermal source)
    std::vector<double> emit(nc);
    double s = 0.0;
    for (int i = 0; i < nc; ++i) {
        const double t2 = radtemp[i] * radtemp[i];
        emit[i] = PC_PI * PC_C * (c->h_rcell[i] * c->h_rcell[i]) * PC_ACOEF * (t2 * t2);
        s += emit[i];
    }
    double st = 0.0;
    for (int i = 0; i < nc; ++i) { emit[i] = emit[i] / s * lbol; st += emit[i]; }
    PhaseTimer tm(c, 1);
    Inputs in(c->io, c->stream);
    in.add(c->d.emit, emit.data(), nc * 8);
    in.add(c->d.radtemp, radtemp, nc * 8, true);
    HIPCHK(in.send());
    launch_ddmc_tables(c);
    launch_ddmc_probs(c);
    HIPCHK(hipGetLastError());
    Outputs out(c->io, c->stream);
    out.add(out_opaclump, c->d.opaclump, (size_t)11 * nc * 8);
    out.add(out_emitprob, c->d.emitprob, (size_t)c->cfg.nep * nc * 8, true);
    out.start();
    int rc = tm.stop(out);
    if (rc) return rc;
    if (out_emit) std::memcpy(out_emit, emit.data(), nc * 8);
    if (out_sthermal) *out_sthermal = st;
    c->h_emit_cache = emit;
    c->have_prep = true;
    return 0;
}

int slgpu_sources(slgpu_ctx *c, int64_t nstot, uint32_t iteration, int *out_nvol,
                  int64_t *out_nnew)
{
    if (!c) return fail(SLGPU_EINVAL, "null context");
    if (!c->have_prep) return fail(SLGPU_EORDER, "slgpu_ddmc_prep must run first");
    if (nstot < 1) return fail(SLGPU_EINVAL, "nstot must be positive");
    std::vector<int> nvol;
    int64_t nnew = source_numbers(c->h_emit_cache, nstot, nvol);
    if (nnew == -1) return fail(SLGPU_EINVAL, "sourcenumbers: no cell emits");
    if (nnew == -2) return fail(SLGPU_EINVAL, "sourcenumbers: nextra>grd_ncell (sourcenumbers.f90:130-131)");
    if (nnew > c->cfg.npartmax) return fail(SLGPU_EINVAL, "vacancies: nnew>npartmax (vacancies.f90:21)");
    std::vector<int64_t> pstart(c->nx + 1, 0);
    for (int i = 0; i < c->nx; ++i) pstart[i + 1] = pstart[i] + nvol[i];
    PhaseTimer tm(c, 2);
    Inputs in(c->io, c->stream);
    in.add((void *)c->d.pstart, pstart.data(), (c->nx + 1) * 8);
    HIPCHK(in.send());
    HIPCHK(hipMemsetAsync(c->d.flags, 0, 4, c->stream));
    c->d.npart = nnew;
    launch_sources(c, iteration);
    HIPCHK(hipGetLastError());
    int flag = 0;
    Outputs out(c->io, c->stream);
    out.add(&flag, c->d.flags, 4);
    out.start();
    int rc = tm.stop(out);
    if (rc) return rc;
    if (flag) return fail(SLGPU_EINVAL, "interior_source: position rejection did not terminate");
    if (out_nvol) std::memcpy(out_nvol, nvol.data(), c->nx * sizeof(int));
    if (out_nnew) *out_nnew = nnew;
    c->have_sources = true;
    c->have_transport = false;
    return 0;
}

int slgpu_transport(slgpu_ctx *c, uint32_t iteration, double *out_tally, double *out_jrad,
                    double *out_eamp, double *out_totals, int64_t *out_counters)
{
    if (!c) return fail(SLGPU_EINVAL, "null context");
    if (!c->have_sources) return fail(SLGPU_EORDER, "slgpu_sources must run first");
    const int nc = c->nx, ng = c->ng;
    PhaseTimer tm(c, 3);
    // particle_advance.f90:65-67: zero the tallies
    HIPCHK(hipMemsetAsync(c->d.tally, 0, (size_t)2 * nc * 8 + (8 + 10 + 1) * 8, c->stream));   // to the queue
    HIPCHK(hipMemsetAsync(c->d.jrad, 0, (size_t)c->d.jrad_copies * nc * ng * 8, c->stream));
    hipEventRecord(c->ev[12], c->stream);
    launch_transport(c, iteration);
    hipEventRecord(c->ev[13], c->stream);
    launch_jrad_reduce(c);
    HIPCHK(hipGetLastError());
    double tot[8];
    unsigned long long ct[10];
    Outputs out(c->io, c->stream);
    out.add(out_jrad, c->d.jrad, (size_t)nc * ng * 8);
    out.add(out_tally, c->d.tally, nc * 8);
    out.add(out_eamp, c->d.eamp, nc * 8, true);
    out.add(tot, c->d.tot, 8 * 8, true);
    out.add(ct, c->d.ct, 10 * 8, true);
    out.start();
    int rc = tm.stop(out);
    if (rc) return rc;
    float kms = 0.f;
    hipEventElapsedTime(&kms, c->ev[12], c->ev[13]);
    c->t_ms[6] += kms;
    tot[2] = -tot[0];     // tot_sflux = -sum e(flux) (particle_advance.f90:283)
    if (out_totals)
        for (int k = 0; k < 7; ++k) out_totals[k] = tot[k];
    if (out_counters)
        for (int k = 0; k < 10; ++k) out_counters[k] = (int64_t)ct[k];
    c->have_transport = true;
    if (ct[7] > 0 && c->cfg.errorfatal)
        return fail(SLGPU_ETRANSPORT, "particle_advance: fatal transport error (" + std::to_string(ct[7]) + " particles)");
    return 0;
}

int slgpu_fluxtally(slgpu_ctx *c, double *out_luminos, double *out_lumdev, int *out_lumnum)
{
    if (!c) return fail(SLGPU_EINVAL, "null context");
    if (!c->have_transport) return fail(SLGPU_EORDER, "slgpu_transport must run first");
    const int ng = c->ng;
    PhaseTimer tm(c, 4);
    HIPCHK(hipMemsetAsync(c->d.lum, 0, (size_t)ng * 20, c->stream));       // lum, dev and num
    launch_fluxtally(c);
    HIPCHK(hipGetLastError());
    Outputs out(c->io, c->stream);
    out.add(out_luminos, c->d.lum, ng * 8);
    out.add(out_lumdev, c->d.dev, ng * 8, true);
    out.add(out_lumnum, c->d.num, ng * 4, true);
    out.start();
    return tm.stop(out);
}

int slgpu_get_particles(slgpu_ctx *c, int64_t n, uint8_t *stat, double *x, double *mu,
                        double *wl, double *e, int *ig, int64_t *nstep, int *err)
{
    if (!c) return fail(SLGPU_EINVAL, "null context");
    if (n < 0 || n > c->d.npart) return fail(SLGPU_EINVAL, "n exceeds the particle count");
    Outputs out(c->io, c->stream);
    out.add(x, c->d.px, n * 8);
    out.add(mu, c->d.pmu, n * 8);
    out.add(wl, c->d.pwl, n * 8);
    out.add(e, c->d.pe, n * 8);
    out.add(nstep, c->d.pnstep, n * 8);
    out.add(ig, c->d.pig, n * 4);
    out.add(err, c->d.perr, n * 4);
    out.add(stat, c->d.pstat, n);
    out.start();
    HIPCHK(out.finish(c->ev[5]));
    return 0;
}

namespace {
// the VJP with its three input gradients on the host (copied in) or, with dev, already on the
// context's device (read in place)
int opacity_vjp_impl(slgpu_ctx *c, bool dev, const double *grad_cap64, const double *grad_capgrey,
                     const double *grad_capross, double *out_grad_temp, double *out_grad_natom,
                     double *out_grad_nelec, double *out_grad_natomfr, double *out_grad_oc)
{
    if (!c) return fail(SLGPU_EINVAL, "null context");
    if (!c->have_opacity) return fail(SLGPU_EORDER, "slgpu_opacity_build must run first");
    if (c->d.nlte) return fail(SLGPU_EORDER, "opacity backward: the last build was NLTE; the backward covers the LTE build");
    const int nc = c->nx, ng = c->ng, nion = c->nion;
    if ((size_t)(nion + c->d.nel) * 64 * sizeof(double) > 65536)
        return fail(SLGPU_EINVAL, "opacity backward: ions + elements exceed 128 per cell");
    PhaseTimer tm(c, 7);
    const size_t cg = (size_t)nc * ng;
    double *dgc = nullptr, *dgp = nullptr, *dgr = nullptr;
    if (!dev) {
        if (!c->vjp_in) {
            int rc = dalloc(c, &c->vjp_in, cg + 2 * (size_t)nc);
            if (rc) return rc;
        }
        if (grad_cap64) dgc = c->vjp_in + 2 * (size_t)nc;
        if (grad_capgrey) dgp = c->vjp_in;
        if (grad_capross) dgr = c->vjp_in + nc;
    }
    Inputs in(c->io, c->stream);
    if (dgp) in.add(dgp, grad_capgrey, nc * 8);
    if (dgr) in.add(dgr, grad_capross, nc * 8, true);
    if (dgc) in.add(dgc, grad_cap64, cg * 8, true);
    HIPCHK(in.send());
    const double *igc = dev ? grad_cap64 : dgc, *igp = dev ? grad_capgrey : dgp, *igr = dev ? grad_capross : dgr;
    double *gT = c->vjp_out, *gn = gT + nc, *ge = gT + 2 * nc, *gf = gT + 3 * nc, *go = gT + 33 * (size_t)nc;
    hipEventRecord(c->ev[20], c->stream);
    launch_opacity_vjp(c, c->opac_flags, igc, igp, igr, gT, gn, ge, gf, go, ff_prefactor(),
                       rgg_scratch(c));
    hipEventRecord(c->ev[21], c->stream);
    HIPCHK(hipGetLastError());
    Outputs out(c->io, c->stream);
    out.add(out_grad_temp, gT, nc * 8);
    out.add(out_grad_natom, gn, nc * 8, true);
    out.add(out_grad_nelec, ge, nc * 8, true);
    out.add(out_grad_natomfr, gf, (size_t)30 * nc * 8, true);
    out.add(out_grad_oc, go, (size_t)nion * nc * 8, true);
    out.start();
    const int rc = tm.stop(out);
    if (!rc) {
        float kms = 0.f;
        hipEventElapsedTime(&kms, c->ev[20], c->ev[21]);
        c->t_ms[10] += kms;
    }
    return rc;
}
}  // namespace

int slgpu_opacity_vjp(slgpu_ctx *c, const double *grad_cap64, const double *grad_capgrey,
                      const double *grad_capross, double *out_grad_temp, double *out_grad_natom,
                      double *out_grad_nelec, double *out_grad_natomfr, double *out_grad_oc)
{
    return opacity_vjp_impl(c, false, grad_cap64, grad_capgrey, grad_capross, out_grad_temp,
                            out_grad_natom, out_grad_nelec, out_grad_natomfr, out_grad_oc);
}

int slgpu_opacity_vjp_dev(slgpu_ctx *c, const double *d_grad_cap64, const double *d_grad_capgrey,
                          const double *d_grad_capross, double *out_grad_temp, double *out_grad_natom,
                          double *out_grad_nelec, double *out_grad_natomfr, double *out_grad_oc)
{
    return opacity_vjp_impl(c, true, d_grad_cap64, d_grad_capgrey, d_grad_capross, out_grad_temp,
                            out_grad_natom, out_grad_nelec, out_grad_natomfr, out_grad_oc);
}

int slgpu_opacity_outputs_dev(slgpu_ctx *c, double *d_cap64, double *d_capgrey, double *d_capross)
{
    if (!c) return fail(SLGPU_EINVAL, "null context");
    if (!c->have_opacity) return fail(SLGPU_EORDER, "an opacity build must run first");
    const size_t nc = c->nx, cg = nc * c->ng;
    if (d_cap64) HIPCHK(hipMemcpyAsync(d_cap64, c->d.cap64, cg * 8, hipMemcpyDeviceToDevice, c->stream));
    if (d_capgrey) HIPCHK(hipMemcpyAsync(d_capgrey, c->d.capgrey, nc * 8, hipMemcpyDeviceToDevice, c->stream));
    if (d_capross) HIPCHK(hipMemcpyAsync(d_capross, c->d.capross, nc * 8, hipMemcpyDeviceToDevice, c->stream));
    HIPCHK(hipStreamSynchronize(c->stream));
    return 0;
}

int slgpu_set_unstaged(slgpu_ctx *c, int on)
{
    if (!c) return fail(SLGPU_EINVAL, "null context");
    if (on != 0 && on != 1) return fail(SLGPU_EINVAL, "on must be 0 or 1");
    c->force_unstaged = on;
    return SLGPU_OK;
}

int slgpu_sample_groups(slgpu_ctx *c, int table, int direct, int64_t n, const double *r,
                        const int *cell, int *out_group)
{
    if (!c) return fail(SLGPU_EINVAL, "null context");
    if (!c->have_prep) return fail(SLGPU_EORDER, "slgpu_ddmc_prep must run first");
    if (table < 0 || table >= NTAB) return fail(SLGPU_EINVAL, "table must be in 0..4");
    if (n < 0 || (n > 0 && (!r || !cell || !out_group))) return fail(SLGPU_EINVAL, "bad sample arrays");
    if (n == 0) return 0;
    for (int64_t k = 0; k < n; ++k)
        if (!(r[k] > 0.0 && r[k] <= 1.0)) return fail(SLGPU_EINVAL, "draws must lie in (0, 1]");
    double *dr = nullptr;
    int *dc = nullptr, *dg = nullptr;
    if (hipMalloc(&dr, n * 8) != hipSuccess || hipMalloc(&dc, n * 4) != hipSuccess ||
        hipMalloc(&dg, n * 4) != hipSuccess) {
        hipFree(dr); hipFree(dc); hipFree(dg);
        return fail(SLGPU_ENOMEM, "sample buffers");
    }
    int rc = 0;
    if (hipMemcpyAsync(dr, r, n * 8, hipMemcpyHostToDevice, c->stream) != hipSuccess ||
        hipMemcpyAsync(dc, cell, n * 4, hipMemcpyHostToDevice, c->stream) != hipSuccess) rc = 1;
    if (!rc) {
        launch_sample_groups(c, table, direct, n, dr, dc, dg);
        if (hipGetLastError() != hipSuccess ||
            hipMemcpyAsync(out_group, dg, n * 4, hipMemcpyDeviceToHost, c->stream) != hipSuccess ||
            hipStreamSynchronize(c->stream) != hipSuccess) rc = 1;
    }
    hipFree(dr); hipFree(dc); hipFree(dg);
    return rc ? fail(SLGPU_EHIP, "sample_groups: device error") : 0;
}

int slgpu_set_eos_data(slgpu_ctx *c, const int *ni, const double *e, const double *q,
                       const double *g1, const double *amass)
{
    if (!c || !ni || !e || !q || !g1 || !amass) return fail(SLGPU_EINVAL, "null argument");
    for (int iz = 1; iz <= 30; ++iz) {
        const int n = ni[iz - 1];
        if (n < 1 || n > iz + 1) return fail(SLGPU_EINVAL, "ni(iz) must be in 1..iz+1 (ionsmod.f:102)");
        if (!(amass[iz - 1] > 0.0)) return fail(SLGPU_EINVAL, "element masses must be positive");
        for (int ii = 1; ii <= n; ++ii)
            if (!(q[(iz - 1) * 31 + ii - 1] > 0.0))
                return fail(SLGPU_EINVAL, "partition functions must be positive for every stage");
    }
    HIPCHK(hipMemcpyAsync(c->d.eos_ni, ni, 30 * sizeof(int), hipMemcpyHostToDevice, c->stream));
    HIPCHK(hipMemcpyAsync(c->d.eos_e, e, 30 * 31 * 8, hipMemcpyHostToDevice, c->stream));
    HIPCHK(hipMemcpyAsync(c->d.eos_q, q, 30 * 31 * 8, hipMemcpyHostToDevice, c->stream));
    HIPCHK(hipMemcpyAsync(c->d.eos_g1, g1, 30 * 31 * 8, hipMemcpyHostToDevice, c->stream));
    HIPCHK(hipMemcpyAsync(c->d.eos_amass, amass, 30 * 8, hipMemcpyHostToDevice, c->stream));
    HIPCHK(hipStreamSynchronize(c->stream));
    c->have_eos_data = true;
    c->have_eos = false;
    return 0;
}

int slgpu_eos(slgpu_ctx *c, const double *temp, const double *mass, const double *massfr,
              double acc, double *nelec, double *out_natom, double *out_natomfr, double *out_oc,
              double *out_ginv, int *out_niter)
{
    if (!c || !temp || !mass || !massfr || !nelec) return fail(SLGPU_EINVAL, "null argument");
    if (!(c->have_grid && c->have_ions && c->have_eos_data))
        return fail(SLGPU_EORDER, "grid, ions and EOS data must be set first");
    const int nc = c->nx, nion = c->nion;
    for (int i = 0; i < nc; ++i) {
        if (mass[i] <= 0.0) continue;
        if (!(temp[i] > 0.0) || !(nelec[i] > 0.0))
            return fail(SLGPU_EINVAL, "temperatures and start electron fractions must be positive");
        double s = 0.0;
        for (int l = 0; l < 30; ++l) {
            if (massfr[(size_t)i * 30 + l] < 0.0) return fail(SLGPU_EINVAL, "massfr2natomfr: negative mass fractions");
            s += massfr[(size_t)i * 30 + l];
        }
        if (!(s > 0.0)) return fail(SLGPU_EINVAL, "massfr2natomfr: all mass fractions zero");
    }
    if (!(acc > 0.0)) acc = 1e-8;                            // ionsmod.f:183
    PhaseTimer tm(c, 8);
    HIPCHK(hipMemsetAsync(c->d.flags, 0, 4, c->stream));
    Inputs in(c->io, c->stream);
    in.add(c->eos_temp, temp, nc * 8);
    in.add(c->eos_mass, mass, nc * 8, true);
    in.add(c->eos_massfr, massfr, (size_t)30 * nc * 8, true);
    in.add(c->eos_nelec, nelec, nc * 8, true);
    HIPCHK(in.send());
    launch_eos(c, c->eos_temp, c->eos_mass, c->eos_massfr, acc, c->eos_nelec, c->eos_natom,
               c->eos_natomfr, c->eos_oc, c->eos_ginv, c->eos_niter);
    HIPCHK(hipGetLastError());
    int flag = 0;
    Outputs out(c->io, c->stream);
    out.add(&flag, c->d.flags, 4);
    out.add(nelec, c->eos_nelec, nc * 8);
    out.add(out_natom, c->eos_natom, nc * 8, true);
    out.add(out_natomfr, c->eos_natomfr, (size_t)30 * nc * 8, true);
    out.add(out_niter, c->eos_niter, nc * sizeof(int), true);
    out.add(out_oc, c->eos_oc, (size_t)nion * nc * 8);
    out.add(out_ginv, c->eos_ginv, (size_t)nion * nc * 8, true);
    out.start();
    int rc = tm.stop(out);
    if (rc) return rc;
    if (flag) {
        c->have_eos = false;
        return fail(SLGPU_EINVAL, "ions_solve_eos: nelec <= 0 or invalid Saha normalisation (ionsmod.f:291,338-349)");
    }
    c->have_eos = true;
    return 0;
}

int slgpu_eos_nlte_ndens(slgpu_ctx *c, double *out_ndens)
{
    if (!c || !out_ndens) return fail(SLGPU_EINVAL, "null argument");
    if (!c->have_eos) return fail(SLGPU_EORDER, "slgpu_eos must run first");
    const int nc = c->nx;
    if (!c->ndens) {
        int rc = dalloc(c, &c->ndens, (size_t)2 * nc);
        if (rc) return rc;
    }
    launch_eos_ndens(c, c->eos_temp, c->eos_mass, c->eos_natom, c->eos_natomfr, c->ndens);
    HIPCHK(hipGetLastError());
    Outputs out(c->io, c->stream);
    out.add(out_ndens, c->ndens, (size_t)2 * nc * 8);
    out.start();
    HIPCHK(out.finish(c->ev[17]));
    return 0;
}

int slgpu_eos_vjp(slgpu_ctx *c, const double *grad_natom, const double *grad_natomfr,
                  const double *grad_nelec, const double *grad_oc, double *out_grad_temp,
                  double *out_grad_mass, double *out_grad_massfr)
{
    if (!c) return fail(SLGPU_EINVAL, "null context");
    if (!c->have_eos) return fail(SLGPU_EORDER, "slgpu_eos must run first");
    const int nc = c->nx, nion = c->nion;
    PhaseTimer tm(c, 9);
    double *buf = c->eos_vjp;
    const size_t nin = (size_t)nc * (2 + 30 + std::max(nion, 1));
    double *gna = buf, *gne = buf + nc, *gfr = buf + 2 * (size_t)nc, *goc = buf + 32 * (size_t)nc;
    double *oT = buf + nin, *om = oT + nc, *omf = om + nc;
    if (!(grad_natom && grad_nelec && grad_natomfr && grad_oc))     // gradients not given are zero
        HIPCHK(hipMemsetAsync(buf, 0, nin * 8, c->stream));
    Inputs in(c->io, c->stream);
    if (grad_natom) in.add(gna, grad_natom, nc * 8);
    if (grad_nelec) in.add(gne, grad_nelec, nc * 8, true);
    if (grad_natomfr) in.add(gfr, grad_natomfr, (size_t)30 * nc * 8, true);
    if (grad_oc) in.add(goc, grad_oc, (size_t)nion * nc * 8, true);
    HIPCHK(in.send());
    launch_eos_vjp(c, c->eos_temp, c->eos_mass, c->eos_massfr, c->eos_nelec, c->eos_natom,
                   c->eos_natomfr, c->eos_oc, gna, gfr, gne, goc, oT, om, omf);
    HIPCHK(hipGetLastError());
    Outputs out(c->io, c->stream);
    out.add(out_grad_temp, oT, nc * 8);
    out.add(out_grad_mass, om, nc * 8, true);
    out.add(out_grad_massfr, omf, (size_t)30 * nc * 8, true);
    out.start();
    return tm.stop(out);
}

int slgpu_timers(slgpu_ctx *c, double *ms, int n, int reset)
{
    if (!c) return fail(SLGPU_EINVAL, "null context");
    for (int k = 0; k < n && k < 12; ++k) ms[k] = c->t_ms[k];
    if (reset)
        for (double &t : c->t_ms) t = 0.0;
    return 0;
}

}  // extern "C"
