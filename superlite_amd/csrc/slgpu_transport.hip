// Source sampling, 1D-spherical IMC/DDMC particle transport and the flux tally on gfx950.
//
//   k_sources    SOURCE/interior_source.f90:57-168 + source_transformdirection.f90:23-46
//   k_transport  particle_advance.f90:140-294 with TRANSPORT1/transport11.f90:86-489
//                (one IMC event) and TRANSPORT1/diffusion11.f90:91-631 (one DDMC event)
//   k_fluxtally  fluxtally.f:30-54
//
// Transport is a persistent kernel over SoA particle arrays: a lane runs one particle to
// escape or death, then takes the next from a global counter, so lanes stay busy until
// the pool is drained; every particle is capped at max_steps events.  The event count of
// SuperLite's random walk (no census: a particle leaves only by escaping or dying) is
// dominated by effective scatters, so the group samplers they call are the exact bucket
// maps of slgpu_sample.h: one table load for most draws instead of nested searches.
// Per-particle randomness is a Philox-4x32-10 stream keyed on (seed, iteration) and
// counted on (particle, step, phase, draw within the step), so trajectories do not depend
// on the schedule, and every lane of a pass computes its step's first block together.
//
// Tallies: the per-cell energy tally lives in LDS (nc doubles) per block and is flushed
// with FP64 atomics at the end; a particle's consecutive events in one cell are merged in
// registers before the LDS atomic.  Each event adds to grd_jrad with one FP64 atomic into
// one of its replicas (block-indexed), which k_jrad_reduce folds together afterwards.
#include "slgpu_device.h"
#include "slgpu_internal.h"
#include "slgpu_sample.h"

// No fused multiply-add contraction in this file: the reference evaluates each product and
// sum separately, and a contraction can turn an exact cancellation into a negative
// rounding residue (the grazing shell-crossing root sqrt(x_l^2 - (1-mu^2)x^2) at x = x_l
// becomes the square root of -ulp, a NaN path length).
#pragma clang fp contract(off)

namespace slgpu {

#define CAPT(ig, ic) ((double)d.cap32[(size_t)((ic) - 1) * ng + ((ig) - 1)])
#define XA(i) (d.xarr[(i) - 1])
#define VXA(i) (d.vxarr[(i) - 1])
#define DXX(i) (d.xarr[(i)] - d.xarr[(i) - 1])
#define DX3X(i) (d.xarr[(i)] * d.xarr[(i)] * d.xarr[(i)] - d.xarr[(i) - 1] * d.xarr[(i) - 1] * d.xarr[(i) - 1])
#define SIGT(ic) (d.sig[(ic) - 1])
#define OPL(k, ic) (d.opaclump[(size_t)((ic) - 1) * 11 + ((k) - 1)])
#define WLG(ig) (d.wl[(ig) - 1])
#define WLI(ig) (d.wlinv[(ig) - 1])
#define DIVV(ix) (d.divv[(ix) - 1])
#define TINV(ic) (d.tempinv[(ic) - 1])

// ---------------------------------------------------------------------------
__global__ __launch_bounds__(256) void k_sources(Dev d, uint32_t iteration)
{
    const int64_t p = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (p >= d.npart) return;
    const int ng = d.ng, nx = d.nx;
    // owning cell: particles are numbered cell by cell (interior_source.f90:60-88)
    int lo = 0, hi = nx;
    while (hi - lo > 1) {
        int mid = (lo + hi) >> 1;
        if (d.pstart[mid] <= p) lo = mid; else hi = mid;
    }
    const int i = lo + 1;
    const int64_t nemit = d.pstart[i] - d.pstart[i - 1];
    Philox rng;
    rng.init(d.seed, iteration, (uint32_t)p, 0u);
    double r1 = rng.draw();
    const double *cum = d.srccum + (size_t)(i - 1) * ng;
    int iig = first_above(cum, 0, ng, r1) + 1;
    if (iig > ng) iig = ng;
    r1 = rng.draw();
    const double wl0 = 1.0 / ((1.0 - r1) * WLI(iig) + r1 * WLI(iig + 1));
    const double ep0 = d.emit[i - 1] / (double)nemit;
    r1 = rng.draw();
    const double mu0 = sqrt(r1);
    r1 = rng.draw();       // azimuth (om), unused in 1D spherical transport
    const int l1 = i - 1 < 1 ? 1 : i - 1, l2 = i + 1 > nx ? nx : i + 1;
    double uul = 0.5 * (d.emit[l1 - 1] + d.emit[i - 1]);
    double uur = 0.5 * (d.emit[l2 - 1] + d.emit[i - 1]);
    const double uumax = uul > uur ? uul : uur;
    uul = uul / uumax;
    uur = uur / uumax;
    const double third = (double)(1.0f / 3.0f);   // single-precision 1.0/3.0 of the reference
    const double xl = XA(i), xr = XA(i + 1);
    const double xl3 = xl * xl * xl, xr3 = xr * xr * xr;
    double r2 = 1.0, r3 = 0.0, x0 = xl;
    int guard = 0;
    while (r2 > r3 && guard < (1 << 20)) {
        r1 = rng.draw();
        x0 = pow(r1 * xr3 + (1.0 - r1) * xl3, third);
        r3 = (x0 - xl) / DXX(i);
        r3 = r3 * uur + (1.0 - r3) * uul;
        r2 = rng.draw();
        ++guard;
    }
    int ix = binsrch(x0, d.xarr, nx + 1, false);
    ix = ix < 1 ? i : ix;
    const double h1 = XA(ix), h2 = XA(ix + 1);
    const double vx = (VXA(ix) * (h2 - x0) + VXA(ix + 1) * (x0 - h1)) / (h2 - h1);
    const double cmffact = 1.0 + mu0 * vx * CINV;
    double mu = (mu0 + vx * CINV) / cmffact;
    mu = mu > 1.0 ? 1.0 : (mu < -1.0 ? -1.0 : mu);
    d.px[p] = x0;
    d.pmu[p] = mu;
    d.pe[p] = ep0;
    d.pwl[p] = wl0;
    if (guard >= (1 << 20)) atomicOr(d.flags, 1);
}

// ---------------------------------------------------------------------------
struct Ptcl {
    double x, mu, e, wl, vx;
    int ix, ig, itype, stat, idist;
    // for a DDMC particle: NF_VALID | BT_LUMP of its current (group, cell) when the step that
    // put it there knew them, so its next step needs no opacity load to pick its thresholds
    uint32_t nflag;
};
constexpr uint32_t NF_VALID = 1u;
// A DDMC -> IMC conversion (diffusion11.f90:329-355, 402-423, 515-538, 587-618) is recorded
// in nflag and completed at the particle's next pass, an IMC pass, where most lanes are
// such conversions: bits 1-3 the kind, bit 4 set when the step's draw 2 was still unused.
// The adiabatic factor of the converting step and that draw wait in the block's LDS.
enum { PEND_SCAT = 1, PEND_LEFT = 2, PEND_RIGHT = 3, PEND_DOP = 4 };
constexpr uint32_t NF_PEND = 7u << 1;
constexpr uint32_t NF_R2FREE = 1u << 4;
constexpr uint32_t NF_FULL = 1u << 5;      // this DDMC step needs diffusion11, not the short step

// TRANSPORT1/transport11.f90:86-489 (trn_noampfact = .true.)
// Arithmetic of the precision form.  SLGPU_MIXED evaluates the sampled path lengths and
// event times (-ln r), the adiabatic factor and the r^3-uniform position in FP32; the
// shell-crossing quadratic, the Newton-Raphson Doppler distance, the DDMC thresholds,
// positions, energies and every tally stay FP64.
template <bool M> __device__ __forceinline__ double p_log(double x)
{
    if constexpr (M) return (double)__logf((float)x);
    else return log(x);
}
// -ln(r)/k: a sampled path length for opacity k (transport11.f90:112-125)
template <bool M> __device__ __forceinline__ double p_path(double r, double k)
{
    if constexpr (M) return -(double)__logf((float)r) / k;
    else return -log(r) / k;
}
// exp(-divv*t/3): the DDMC adiabatic factor (diffusion11.f90:623-629).  A particle takes
// ~1e4-1e5 of these factors, so a systematic last-bit error in an FP32 factor near 1
// compounds into a percent-level energy bias.  The precision form therefore evaluates the
// loss fraction d = 1 - exp(-a) in FP32 to FP32 *relative* accuracy (series for small a)
// and forms the factor 1 - d in FP64.
template <bool M> __device__ __forceinline__ double p_adiabatic(double divv, double t)
{
    if constexpr (M) {
        const float a = (float)(divv * t) * (1.0f / 3.0f);
        const float d = a < 0.03f
                            ? a * (1.0f - a * (0.5f - a * (1.0f / 6.0f - a * (1.0f / 24.0f))))
                            : 1.0f - expf(-a);
        return 1.0 - (double)d;
    } else {
        // most steps lose less than 2^-5, where the series' remainder a^8/8! is under 2^-55: eight
        // operations instead of exp()'s forty
        const double a = divv * t * (1.0 / 3.0);
        if (!(fabs(a) <= 0x1p-5)) return exp(-divv * t / 3);
        double f = -1.0 / 5040.0;
        f = fma(f, a, 1.0 / 720.0);
        f = fma(f, a, -1.0 / 120.0);
        f = fma(f, a, 1.0 / 24.0);
        f = fma(f, a, -1.0 / 6.0);
        f = fma(f, a, 0.5);
        f = fma(f, a, -1.0);
        return fma(f, a, 1.0);
    }
}
// r^3-uniform radius in [xl, xr]: (r*xr^3 + (1-r)*xl^3)**(1.0/3.0) with the reference's
// single-precision exponent e = (1.0/3.0 in single) = (1 + 2^-25)/3 (diffusion11.f90:336,597).
// Radii cubed (~1e47 cm^3) overflow FP32, so the precision form takes the FP32 root of the
// normalised b = r + (1-r)*(xl/xr)^3 and multiplies by xr^(3e) = xr * exp(2^-25 * ln xr).
// That last factor (~1 + 1.1e-6 at supernova radii) is what carries the outermost draws past
// xr into the caller's clamp, as in the FP64 form; dropping it moves ~0.1% of the
// conversions in thin shells off the face and biased the step count by +0.75%.
template <bool M> __device__ __forceinline__ double p_shell_root(double r1, double xl, double xr)
{
    if constexpr (M) {
        const double q = xl / xr;
        const double dl = 0x1p-25 * (double)__logf((float)xr);
        const double xr3e = xr * (1.0 + dl * (1.0 + 0.5 * dl));
        return xr3e * (double)powf((float)(r1 + (1.0 - r1) * (q * q * q)), 1.0f / 3.0f);
    } else {
        return pow(r1 * (xr * xr * xr) + (1.0 - r1) * (xl * xl * xl), (double)(1.0f / 3.0f));
    }
}

// transport11.f90:259-285: the experimental anisotropic Thomson cosine for draw r1.  The
// second cube root has a negative base for r1 below ~0.957, where the real power is NaN;
// every range test then fails and the isotropic cosine is taken, as in the reference.
__device__ __forceinline__ double thomson_aniso_mu(double r1)
{
    const double q = sqrt(1.0 + 16.0 * ((r1 - 0.5) * (r1 - 0.5)));
    const double mutemp = pow(4.0 * r1 - 2.0 + q, 1.0 / 3.0) - pow(q - (4.0 - 2.0 * r1), 1.0 / 3.0);
    const double muhelp = mutemp;
    const double B = 2 * mutemp * muhelp;
    const double C = mutemp * mutemp + muhelp * muhelp - 1;
    const double munew1 = (-B + sqrt(B * B - 4 * C)) / 2;
    const double munew2 = (-B - sqrt(B * B - 4 * C)) / 2;
    const bool ok1 = munew1 <= 1 && munew1 >= -1, ok2 = munew2 <= 1 && munew2 >= -1;
    if (ok1 && ok2) return r1 < 0.5 ? munew1 : munew2;
    if (ok1) return munew1;
    if (ok2) return munew2;
    return 1.0 - 2.0 * r1;
}

// What an IMC pass reads of its cell and group, requested together at the top of the pass, the
// cell's part as one record (nine arrays took as many address computations and requests):
// the conversion that most passes begin with and the event then wait for one round trip
// instead of one at each branch.
struct ImcIn {
    CellGeo g;
    double wi0, wi1;                                   // WLI(ig), WLI(ig+1)
    float cp, cpup, cpdn;                              // gas_cap of the group and of its two neighbours
};

__device__ __forceinline__ void imc_request(const Dev &d, const Ptcl &p, ImcIn &q)
{
    const int ng = d.ng, ix = p.ix, ig = p.ig;
    const float *row = d.cap32 + (size_t)(ix - 1) * ng;
    q.cp = row[ig - 1];
    q.cpup = row[ig < ng ? ig : ig - 1];
    q.cpdn = row[ig > 1 ? ig - 2 : ig - 1];
    q.wi0 = WLI(ig); q.wi1 = WLI(ig + 1);
    q.g = d.geo[ix - 1];
}

// the smallest double whose quotient by c is at least 0.1
constexpr double NEWTON_DV = 0x1.656165a400000p+31;
static_assert(NEWTON_DV / PC_C >= 0.1 && 0x1.656165a3fffffp+31 / PC_C < 0.1, "NEWTON_DV");

// BT_THIN and BT_LUMP of a group of opacity cp in the cell (group_flags of slgpu_sample.h)
__device__ __forceinline__ uint32_t cell_flags(const Dev &d, const CellGeo &q, double cp)
{
    const double dx = q.xr - q.xl;
    if (d.puretran || (q.sg + cp) * dx < d.tauddmc) return BT_THIN;
    return cp * dx >= d.taulump && q.nlump > 0 ? BT_LUMP : 0u;
}

template <bool M, bool X>
__device__ int transport11(const Dev &d, Ptcl &p, StepRng &s, const ImcIn &q, double &erd, double &jrd,
                           double &eamp, double &evelo)
{
    const int ng = d.ng, nx = d.nx;
    int ix = p.ix, ig = p.ig;
    double x = p.x, mu = p.mu, e = p.e, wl = p.wl, vx = p.vx;
    int ic = ix;
    double r1, r2, db, dcol, dthm, ddop, dd;
    int ixnext;
    erd = 0.0; jrd = 0.0; eamp = 0.0;
    double elabfact = 1.0 - mu * vx * CINV;
    const double elabfactold = elabfact;
    const double xl = q.g.xl, xr = q.g.xr;
    const double far = q.g.far;
    if (ix == 1 || mu >= -sqrt(1.0 - (xl / x) * (xl / x))) {
        db = fabs(sqrt(xr * xr - (1.0 - mu * mu) * x * x) - mu * x);
        ixnext = ix + 1;
    } else {
        db = fabs(sqrt(xl * xl - (1.0 - mu * mu) * x * x) + mu * x);
        ixnext = ix - 1;
    }
    // the neighbour cell, for an event at the face
    const int nb = ixnext < 1 ? 1 : (ixnext > nx ? nx : ixnext);
    const CellGeo &gn = d.geo[nb - 1];
    const double cap_nb = CAPT(ig, nb), sig_nb = gn.sg, dx_nb = gn.xr - gn.xl;
    if (db != db) return 1;
    const double sg = q.g.sg, cp = (double)q.cp;
    const double dvdr = q.g.dvdr;
    if (sg > 0.0) { r1 = s.draw(); dthm = p_path<M>(r1, elabfact * sg); }
    else dthm = far;
    if (cp <= 0.0) dcol = far;
    else { r1 = s.draw(); dcol = p_path<M>(r1, elabfact * cp); }
    const double vhelp = q.g.vhelp;
    if (fabs(vx - vhelp) >= NEWTON_DV) {                      // / c >= 0.1
        // Newton-Raphson Doppler distance (transport11.f90:159-199)
        const double epstol = 1e-3;
        int it = 0;
        double shelp = db;
        double xhelp = sqrt(x * x + shelp * shelp + 2.0 * shelp * x * mu);
        double muhelp = (mu * x + shelp) / xhelp;
        double phi = dvdr * mu * x - PC_C * (1 - wl * q.wi1) + vhelp * muhelp + dvdr * shelp;
        double dphi = dvdr + vhelp * (1 - muhelp * muhelp) / xhelp;
        ddop = shelp - phi / dphi;
        while ((fabs(ddop - shelp) > ddop * epstol) && it < 100) {
            it = it + 1;
            shelp = ddop;
            xhelp = sqrt(x * x + shelp * shelp + 2.0 * shelp * x * mu);
            muhelp = (mu * x + shelp) / xhelp;
            if (dvdr > 0 && ig < ng)
                phi = dvdr * mu * x - PC_C * (1 - wl * q.wi1) + vhelp * muhelp + dvdr * shelp;
            else if (dvdr < 0 && ig > 1)
                phi = dvdr * mu * x - PC_C * (1 - wl * q.wi0) + vhelp * muhelp + dvdr * shelp;
            else { ddop = far; break; }
            dphi = dvdr + vhelp * (1 - muhelp * muhelp) / xhelp;
            ddop = shelp - phi / dphi;
        }
        if (ddop <= 0.0 || it == 100) ddop = far;
    } else {
        if (dvdr > 0 && ig < ng) ddop = q.g.c3 * (elabfact - wl * q.wi1);
        else if (dvdr < 0 && ig > 1) ddop = q.g.c3 * (elabfact - wl * q.wi0);
        else ddop = far;
        if (ddop < 0.0) ddop = far;
    }
    // minloc over [dcol, dthm, ddop, db]
    int idist = 1;
    dd = dcol;
    if (dthm < dd) { dd = dthm; idist = 2; }
    if (ddop < dd) { dd = ddop; idist = 3; }
    if (db < dd) { dd = db; idist = 4; }
    p.idist = idist;
    if (dcol != dcol || dthm != dthm || ddop != ddop) return 3;
    if (dd < 0.0) return 4;
    const double xold = x;
    x = sqrt(x * x + dd * dd + 2.0 * dd * x * mu);
    vx = (q.g.vl * (xr - x) + q.g.vr * (x - xl)) / (xr - xl);
    if (x == 0.0) mu = 1.0;
    else mu = (xold * mu + dd) / x;
    erd = e * elabfact * elabfact * dd * CINV;
    jrd = PC_C * erd;
    elabfact = 1.0 - mu * vx * CINV;
    int ret = 0;
    if (x < XA(1)) {
        x = XA(1);
        vx = VXA(1);
        ix = 1;
        r1 = s.draw();
        mu = 1.0 - r1;
        goto done;
    }
    if (dd == dthm || dd == dcol) {
        r1 = s.draw();
        if (X && dd == dthm && d.thm_aniso) mu = thomson_aniso_mu(r1);
        else mu = 1.0 - 2.0 * r1;
        mu = (mu + vx * CINV) / (1.0 + vx * mu * CINV);
    } else if (dd == db) {
        if (mu >= 0.0 && ix == nx) { p.stat = 1; goto done; }
    }
    if (dd == dthm) {
        wl = wl * (1.0 - mu * vx * CINV) / elabfact;
        const double help = elabfact / (1.0 - mu * vx * CINV);
        evelo = evelo + e * (1.0 - help);
        e = e * help;
    } else if (dd == dcol) {
        r1 = s.draw();                 // unused draw (transport11.f90:313)
        const double help = elabfact / (1.0 - mu * vx * CINV);
        evelo = evelo + e * (1.0 - help);
        e = e * help;
        if (ng != 1) {
            r1 = s.draw();
            const uint32_t ent = bt_row(d, TAB_E, ic)[bt_key(r1)];
            uint32_t fl = ent & (BT_THIN | BT_LUMP);
            if (ent & BT_PURE) {
                ig = (int)(ent & 0x7fffu);
            } else {
                double cg;
                ig = emitgroup_range(d, r1, q.g.em, ic, (int)(ent & 0x7fffu), (int)((ent >> 15) & 0x7fffu), cg);
                fl = cell_flags(d, q.g, cg);
            }
            if (!(fl & BT_THIN)) {
                p.itype = 2;
                p.nflag = NF_VALID | (fl & BT_LUMP);
            }
        }
        if (p.itype == 2) {
            evelo = evelo + e * vx * mu * CINV;
            e = e * (1.0 - vx * mu * CINV);
        } else {
            r1 = s.draw();
            wl = 1.0 / ((1.0 - r1) * WLI(ig) + r1 * WLI(ig + 1));
            wl = wl * (1.0 - vx * mu * CINV);
        }
    } else if (dd == db && ixnext > ix && ix == nx) {
        // outer boundary reached with a rounding-negative cosine: escapes (the reference
        // would index the non-existent cell nx+1 here)
        p.stat = 1;
        goto done;
    } else if (dd == db && ixnext > ix) {
        const int l = ix + 1;
        if ((sig_nb + cap_nb) * dx_nb < d.tauddmc || d.puretran) {
            x = xr;
            vx = q.g.vr;
            ix = ix + 1;
        } else {
            mu = (mu - vx * CINV) / (1.0 - vx * mu * CINV);
            double help = (cap_nb + sig_nb) * dx_nb;
            help = 4.0 / (3.0 * help + 6.0 * PC_DEXT);
            r1 = s.draw();
            if (r1 < help * (1.0 + 1.5 * fabs(mu))) {
                p.itype = 2;
                p.nflag = NF_VALID | lump_flag(d, cap_nb, dx_nb, l);
                evelo = evelo + e * (1.0 - elabfact);
                e = e * elabfact;
                wl = wl / elabfact;
                ix = ix + 1;
            } else {
                r1 = s.draw();
                r2 = s.draw();
                mu = -(r1 > r2 ? r1 : r2);
                mu = (mu + vx * CINV) / (1.0 + vx * mu * CINV);
                x = xr;
                vx = q.g.vr;
            }
        }
    } else if (dd == db) {
        const int l = ix - 1;
        if ((sig_nb + cap_nb) * dx_nb < d.tauddmc || d.puretran) {
            x = xl;
            vx = q.g.vl;
            ix = ix - 1;
        } else {
            mu = (mu - vx * CINV) / (1.0 - vx * mu * CINV);
            if (X && d.ampfact && mu < 0.0) {
                // amplification factor (transport11.f90:410-421)
                double h = 1.0 / fabs(mu);
                h = h < 100.0 ? h : 100.0;
                evelo = evelo - e * 2.0 * (0.55 * h - 1.25 * fabs(mu)) * vx * CINV;
                eamp = e * 2.0 * 0.55 * (h - 2.0 > 0.0 ? h - 2.0 : 0.0) * vx * CINV;
                h = h < 2.0 ? h : 2.0;
                e = e * (1.0 + 2.0 * (0.55 * h - 1.25 * fabs(mu)) * vx * CINV);
            }
            double help = (cap_nb + sig_nb) * dx_nb;
            help = 4.0 / (3.0 * help + 6.0 * PC_DEXT);
            r1 = s.draw();
            if (r1 < help * (1.0 + 1.5 * fabs(mu))) {
                p.itype = 2;
                p.nflag = NF_VALID | lump_flag(d, cap_nb, dx_nb, l);
                evelo = evelo + e * (1.0 - elabfact);
                e = e * elabfact;
                wl = wl / elabfact;
                ix = ix - 1;
            } else {
                r1 = s.draw();
                r2 = s.draw();
                mu = r1 > r2 ? r1 : r2;
                mu = (mu + vx * CINV) / (1.0 + vx * mu * CINV);
                x = xl;
                vx = q.g.vl;
            }
        }
    } else if (dd == ddop) {
        double cnew = (double)q.cp;
        if (dvdr > 0) {
            if (ig < ng) {
                ig = ig + 1;
                cnew = (double)q.cpup;
                wl = (WLG(ig) + 1e-6 * (WLG(ig + 1) - WLG(ig))) * elabfactold;
            } else {
                r1 = s.draw();
                wl = 1.0 / (r1 * WLI(ng + 1) + (1.0 - r1) * WLI(ng));
                wl = wl * elabfact;
            }
        } else if (dvdr < 0) {
            if (ig > 1) {
                wl = (WLG(ig) + 1e-6 * (WLG(ig - 1) - WLG(ig))) * elabfactold;
                ig = ig - 1;
                cnew = (double)q.cpdn;
            } else {
                r1 = s.draw();
                wl = 1.0 / (r1 * WLI(1) + (1.0 - r1) * WLI(2));
                wl = wl * elabfact;
            }
        }
        if (((sg + cnew) * (xr - xl) >= d.tauddmc) && !d.puretran) {
            p.itype = 2;
            p.nflag = NF_VALID | lump_flag(d, cnew, xr - xl, ic);
            evelo = evelo + e * vx * mu * CINV;
            e = e * elabfact;
            wl = wl / elabfact;
        }
    } else {
        ret = 17;
    }
done:
    p.x = x; p.mu = mu; p.e = e; p.wl = wl; p.vx = vx;
    p.ix = ix; p.ig = ig;
    return ret;
}

// resolved leakage opacity through the left (side<0) / right face (diffusion11.f90:204-239)
__device__ __forceinline__ double resleak_t(const Dev &d, int ix, int g, int side)
{
    const int ng = d.ng, ic = ix;
    if (side < 0) {
        const int l = ix - 1;
        if ((CAPT(g, l) + SIGT(l)) * DXX(ix - 1) < d.tauddmc) {
            double mfp = (CAPT(g, ic) + SIGT(ic)) * DXX(ix);
            double ppl = 4.0 / (3.0 * mfp + 6.0 * PC_DEXT);
            return 1.5 * ppl * (XA(ix) * XA(ix)) / DX3X(ix);
        }
        double mfp = (SIGT(ic) + CAPT(g, ic)) * DXX(ix) + (SIGT(l) + CAPT(g, l)) * DXX(ix - 1);
        return 2.0 * (XA(ix) * XA(ix)) / (mfp * DX3X(ix));
    }
    if (ix == d.nx) {
        double mfp = (CAPT(g, ic) + SIGT(ic)) * DXX(ix);
        double ppr = 4.0 / (3.0 * mfp + 6.0 * PC_DEXT);
        return 1.5 * ppr * (XA(ix + 1) * XA(ix + 1)) / DX3X(ix);
    }
    const int l = ix + 1;
    if ((CAPT(g, l) + SIGT(l)) * DXX(ix + 1) < d.tauddmc) {
        double mfp = (CAPT(g, ic) + SIGT(ic)) * DXX(ix);
        double ppr = 4.0 / (3.0 * mfp + 6.0 * PC_DEXT);
        return 1.5 * ppr * (XA(ix + 1) * XA(ix + 1)) / DX3X(ix);
    }
    double mfp = (SIGT(ic) + CAPT(g, ic)) * DXX(ix) + (SIGT(l) + CAPT(g, l)) * DXX(ix + 1);
    return 2.0 * (XA(ix + 1) * XA(ix + 1)) / (mfp * DX3X(ix));
}

// uniform position in the shell with the single-precision 1/3 exponent, clamped (:336-339)
template <bool M>
__device__ __forceinline__ double shell_position(double xl, double xr, double r1)
{
    double x = p_shell_root<M>(r1, xl, xr);
    x = x > xr ? xr : x;
    x = x < xl ? xl : x;
    return x;
}

// diffusion11.f90:243-283: the denominator and event thresholds of one DDMC step
__device__ __forceinline__ DdmcProb ddmc_prob(double opl, double opr, double emitlump,
                                              double caplump, double doplump)
{
    double denom = opl + opr + (1.0 - emitlump) * caplump + doplump;
    denom = 1.0 / denom;
    const double pl = opl * denom, pr = opr * denom, pdop = doplump * denom;
    DdmcProb q;
    q.denom = denom;
    q.t1 = 0.0 + pdop;
    q.t2 = 0.0 + pdop + pl;
    q.t3 = 0.0 + pdop + (pl + pr);
    return q;
}

// The per-event constants of diffusion11.f90:95-152 and 204-239 depend only on the cell
// and, for an unlumped group, on the group; they are evaluated once per iteration here,
// one thread per (group, cell), and the step loads them.
// The short step's form of the thresholds.  The event draw is (m + 0.5) 2^-42 with a 42-bit m
// whose upper 32 bits are a generator word w.  With T = floor(t 2^32), w < T gives draw < t and
// w > T gives draw > t, exactly; w == T leaves the step to the full FP64 test.  A denominator
// that is not a number (no threshold means anything then) sends every step there.
__device__ __forceinline__ uint32_t word_threshold(double t)
{
    if (!(t > 0.0)) return 0u;
    return t >= 1.0 ? 0xFFFFFFFFu : (uint32_t)(t * 4294967296.0);
}

__global__ __launch_bounds__(256) void k_ddmc_probs(Dev d)
{
    const int ng = d.ng;
    const int ig = blockIdx.x * 256 + threadIdx.x + 1, ic = blockIdx.y + 1, ix = ic;
    if (ig > ng) return;
    const CellDDMC cc = d.cell[ic - 1];
    const double cp = CAPT(ig, ic);
    // diffusion11.f90:175-182: grd_cap(ig)*capgreyinv in LTE, grd_capemit(ig)*capemitgreyinv in NLTE
    const double ce = (double)d.capem32[(size_t)(ic - 1) * ng + ig - 1];
    const double emitlump = specint0(TINV(ic), d.wlinv, ig) * cc.emgreyinv * ce;
    const double sa = d.specarr[(size_t)(ic - 1) * ng + ig - 1];
    double doplump;
    if (ig != ng && DIVV(ix) >= 0)
        doplump = dopspeccalc(TINV(ic), d.wlinv, ig) * DIVV(ix) / (sa * 3 * PC_C);
    else if (ig != 1 && DIVV(ix) < 0)
        doplump = -1 * dopspeccalc(TINV(ic), d.wlinv, ig - 1) * DIVV(ix) / (sa * 3 * PC_C);
    else
        doplump = 0.0;
    const double opl = (ix == 1) ? 0.0 : resleak_t(d, ix, ig, -1);
    const double opr = resleak_t(d, ix, ig, +1);
    const DdmcProb q = ddmc_prob(opl, opr, emitlump, cp, doplump);
    d.gprob[(size_t)(ic - 1) * ng + ig - 1] = q;
    ShortProb sp;
    sp.denom = q.t3 == q.t3 ? q.denom : q.t3;
    sp.w3 = word_threshold(q.t3);
    // the Doppler shift of an unlumped particle: the threshold's upper 30 bits and the flags of the
    // group it leads to
    const int to = DIVV(ix) >= 0 ? (ig + 1 > ng ? ng : ig + 1) : (ig < 2 ? 1 : ig - 1);
    sp.w1 = (word_threshold(q.t1) & ~3u) | (group_flags(d, to, ic) >> 29 & 3u);
    d.gshort[(size_t)(ic - 1) * ng + ig - 1] = sp;
    if (ig == 1) {
        const DdmcProb c = ddmc_prob(OPL(1, ic), OPL(2, ic), cc.emitlump, cc.caplump, cc.doplump);
        d.cprob[ic - 1] = c;
        ShortCell sc;
        sc.denom = c.t3 == c.t3 ? c.denom : c.t3;
        sc.divv = DIVV(ic);
        sc.w1 = word_threshold(c.t1);
        sc.w2 = word_threshold(c.t2);
        sc.w3 = word_threshold(c.t3);
        sc.pad = 0;
        d.cshort[ic - 1] = sc;
    }
}

void launch_ddmc_probs(slgpu_ctx *c)
{
    hipLaunchKernelGGL(k_ddmc_probs, dim3((c->ng + 255) / 256, c->nx), dim3(256), 0, c->stream,
                       c->d);
}

// TRANSPORT1/diffusion11.f90:91-631 — one DDMC event.  Every cell constant is evaluated for
// the current cell.  The four events (Doppler, left leak, right leak, effective scatter,
// :283-620) run through ONE code path: the event selects the sampling table, the
// destination cell and the IMC-conversion rule by data, while the random draws keep the
// reference's order per event.  That keeps the lanes of a wave on the same instructions.
enum { EV_DOP = 0, EV_LEFT = 1, EV_RIGHT = 2, EV_SCAT = 3 };

template <bool M>
__device__ int diffusion11(const Dev &d, Ptcl &p, StepRng &s, double &erd, double &jrd,
                           double &evelo, double &pend_f, double &pend_r2)
{
    const int ng = d.ng, nx = d.nx;
    int ix = p.ix, ig = p.ig;
    const int ic = ix;
    double x = p.x, mu = p.mu, e = p.e, wl = p.wl, vx = p.vx;
    double r1;
    erd = 0.0; jrd = 0.0;
    const double dist = DXX(ix);
    const int nlump = d.cell[ic - 1].nlump;
    // The step's first three draws.  Draw 2 samples the group of every effective scatter
    // (and of lumped events), so with the flags the previous step left, the thresholds and
    // that draw's bucket entry are requested together: one memory round trip per step
    // instead of opacity -> thresholds -> entry.  Draws are counted on (step, index), so
    // drawing early does not change any value.
    const double rt = s.draw(), rev = s.draw(), r2 = s.draw();
    const bool known = (p.nflag & NF_VALID) != 0;
    uint32_t lump;                                             // BT_LUMP of (ig, ic)
    if (known) {
        lump = p.nflag & BT_LUMP;
    } else {
        const double cp = CAPT(ig, ic);
        if ((SIGT(ic) + cp) * dist < d.tauddmc) return 100;
        lump = (cp * dist >= d.taulump && nlump > 0) ? BT_LUMP : 0u;
    }
    const int glump = lump ? nlump : 0;                        // :156-160
    // the cell's lumped thresholds or the group's own
    const DdmcProb q = lump ? d.cprob[ic - 1] : d.gprob[(size_t)(ic - 1) * ng + (ig - 1)];
    const int tscat = lump ? TAB_S : TAB_E;
    const uint32_t escat = known ? bt_row(d, tscat, ic)[bt_key(r2)] : 0u;
    const double denom = q.denom;
    const double ddmct = fabs(p_log<M>(rt) * denom * CINV);
    erd = e * ddmct;
    jrd = PC_C * erd;
    int ev;
    if (rev >= 0.0 && rev < q.t1) ev = EV_DOP;
    else if (rev >= q.t1 && rev < q.t2) ev = EV_LEFT;
    else if (rev >= q.t2 && rev < q.t3) ev = EV_RIGHT;
    else ev = EV_SCAT;
    // keep the entry's load ahead of the branches that use it
    asm volatile("" ::"v"(escat));
    p.idist = ev == EV_LEFT ? -3 : (ev == EV_RIGHT ? -4 : (ev == EV_SCAT ? -2 : p.idist));
    // draws after the first three continue the step's sequence; draw 2 is taken by the
    // first consumer that needs a fourth number in the reference's order
    bool r2_free = true;
    auto next = [&]() -> double {
        if (r2_free) { r2_free = false; return r2; }
        return s.draw();
    };
    int ret = 0;
    bool adiabatic = true;
    uint32_t nflag = NF_VALID | lump;                          // particle stays in (ig, ic)
    if (ev == EV_LEFT && ix == 1) {
        adiabatic = false;                                     // :362-365 returns
    } else if (ev == EV_SCAT && glump == ng) {
        ret = 102;                                             // :552-556
        adiabatic = false;
    } else {
        const bool flux = (ev == EV_RIGHT && ix == nx);        // :438-478
        if (flux) {
            p.stat = 1;
            const double ra = next(), rb = next();
            mu = ra > rb ? ra : rb;
        }
        // group sampling: lumped particles draw from the cell's table of this event,
        // unlumped effective scatters from the emission probabilities (emitgroup)
        int iiig = ig, fl = -1;
        if (glump > 0 || ev == EV_SCAT) {
            const bool pre = known && r2_free && ev == EV_SCAT;
            r1 = next();
            const int t = glump == 0 ? TAB_E
                        : (ev == EV_LEFT ? TAB_L : (ev == EV_RIGHT ? TAB_R : (ev == EV_DOP ? TAB_D : TAB_S)));
            const uint32_t ent = pre ? escat : bt_row(d, t, ic)[bt_key(r1)];
            iiig = sample_entry(d, t, ic, nlump, r1, ent, fl);
        }
        if (flux) {
            ig = iiig;
            r1 = next();
            wl = 1.0 / (r1 * WLI(ig + 1) + (1.0 - r1) * WLI(ig));
            x = XA(nx + 1);
            vx = VXA(nx + 1);
            mu = (mu + vx * CINV) / (1.0 + vx * mu * CINV);
            mu = mu > 1.0 ? 1.0 : mu;
            const double help = 1.0 / (1.0 - mu * vx * CINV);
            evelo = evelo + e * (1.0 - help);
            wl = wl / help;
            e = e * help;
            adiabatic = false;
        } else {
            // destination group and the cell whose optical depth decides IMC conversion
            int ig2 = iiig, lc = ic;
            if (ev == EV_DOP) {
                if (DIVV(ix) >= 0) { ig2 = iiig + 1; wl = WLG(ig2); ig2 = ig2 > ng ? ng : ig2; }
                else { ig2 = iiig - 1; wl = WLG(ig2 + 1); ig2 = ig2 < 1 ? 1 : ig2; }
            } else if (ev == EV_LEFT) {
                lc = ix - 1;
            } else if (ev == EV_RIGHT) {
                lc = ix + 1;
            }
            if (fl < 0) fl = (int)group_flags(d, ig2, lc);
            nflag = NF_VALID | ((uint32_t)fl & BT_LUMP);
            if (fl & (int)BT_THIN) {
                // conversion to IMC: recorded here, sampled by imc_entry at the next pass
                p.itype = 1;
                const uint32_t kind = ev == EV_SCAT ? PEND_SCAT
                                    : (ev == EV_LEFT ? PEND_LEFT : (ev == EV_RIGHT ? PEND_RIGHT : PEND_DOP));
                nflag = (kind << 1) | (r2_free ? NF_R2FREE : 0u) | ((uint32_t)fl & BT_LUMP);
                if (r2_free) pend_r2 = r2;
            }
            ig = ig2;
            if (ev == EV_LEFT) ix = ix - 1;
            else if (ev == EV_RIGHT) ix = ix + 1;
        }
    }
    p.nflag = nflag;
    if (adiabatic) {
        if (nflag & NF_PEND) {
            // after the conversion's frame change, at the next pass (its position lies in
            // the shell, so the inner-boundary test below never fires for it)
            pend_f = p_adiabatic<M>(DIVV(ix), ddmct);
        } else if (x < XA(1)) {
            p.stat = 2;                                        // :623-626
        } else {
            const double f = p_adiabatic<M>(DIVV(ix), ddmct);
            evelo = evelo + e * (1.0 - f);
            e = e * f;
        }
    }
    p.x = x; p.mu = mu; p.e = e; p.wl = wl; p.vx = vx;
    p.ix = ix; p.ig = ig;
    return ret;
}

// The recorded DDMC -> IMC conversion of step `step` (diffusion11.f90:329-355, 402-423,
// 515-538, 587-618): the new wavelength, direction and position, the frame change, then the
// step's adiabatic factor f, in the reference's order.  Its draws are that step's: draw 2 when
// it was still unused (r2), then draws 3.. (block 1 of the step).
template <bool M>
__device__ void imc_entry(const Dev &d, Ptcl &p, const StepRng &s, const ImcIn &q, uint32_t step,
                          double &evelo, double f, double r2)
{
    const uint32_t kind = (p.nflag & NF_PEND) >> 1;
    bool r2_free = (p.nflag & NF_R2FREE) != 0;
    uint32_t o[4];
    Philox::block(s.pid, step, StepRng::PHASE, 1u, s.k0, s.k1, o);
    uint32_t j = 0;
    auto next = [&]() -> double {
        if (r2_free) { r2_free = false; return r2; }
        const double u = Philox::u42(j == 0 ? o[0] : (j == 1 ? o[1] : o[2]), (o[3] >> (10u * j)) & 0x3FFu);
        ++j;
        return u;
    };
    double x, mu, vx, e = p.e, wl = p.wl;
    const bool face = kind == PEND_LEFT || kind == PEND_RIGHT;
    if (kind == PEND_SCAT) {
        const double r1 = next();
        wl = 1.0 / ((1.0 - r1) * q.wi0 + r1 * q.wi1);
    } else if (face) {
        const double r1 = next();
        wl = 1.0 / (r1 * q.wi1 + (1.0 - r1) * q.wi0);
    }
    const double ra = next(), rb = next();
    if (face) {
        x = kind == PEND_LEFT ? q.g.xr : q.g.xl;                  // the face crossed into cell ix
        vx = kind == PEND_LEFT ? q.g.vr : q.g.vl;
        mu = ra > rb ? ra : rb;
        if (kind == PEND_LEFT) mu = -mu;
    } else {
        mu = 1.0 - 2.0 * ra;
        x = shell_position<M>(q.g.xl, q.g.xr, rb);
        vx = (q.g.vl * (q.g.xr - x) + q.g.vr * (x - q.g.xl)) / (q.g.xr - q.g.xl);
    }
    mu = (mu + vx * CINV) / (1.0 + vx * mu * CINV);
    const double help = 1.0 / (1.0 - vx * mu * CINV);
    evelo = evelo + e * (1.0 - help);
    e = e * help;
    wl = wl * (1.0 - vx * mu * CINV);
    evelo = evelo + e * (1.0 - f);
    e = e * f;
    p.x = x; p.mu = mu; p.vx = vx; p.e = e; p.wl = wl;
    p.nflag = NF_VALID | (p.nflag & BT_LUMP);
}

// Block totals in LDS, indexed like Dev::tot and Dev::ct.  Whatever changes once per
// particle or pass (its start, its end, conversions, the rare warnings and amplification
// energies) is added here at once; only evelo, summed per step, stays in a register, which
// keeps the persistent lane state small.  The DDMC step count is the particles' total steps
// minus the IMC steps.
struct BlockTotals {
    double tot[7];                 // eout, evelo, -, estart, edead, esrc, eamp
    unsigned long long ct[9];      // nact, nimc, total steps (then nddmc), nmax, nswap,
                                   // nflux, ndead, nerr, nwarn
};

__device__ __forceinline__ void flush_totals(const Dev &d, BlockTotals &b, double evelo)
{
    const double ev = wave_sum(evelo);
    if ((threadIdx.x & 63) == 0 && ev != 0.0) atomicAdd(&b.tot[1], ev);
    __syncthreads();
    if (threadIdx.x < 7) {
        const double v = b.tot[threadIdx.x];
        if (v != 0.0) atomicAdd(&d.tot[threadIdx.x], v);
    } else if (threadIdx.x >= 64 && threadIdx.x < 64 + 9) {
        const int q = threadIdx.x - 64;
        unsigned long long v = b.ct[q];
        if (q == 2) v -= b.ct[1];                                // DDMC steps
        if (q == 3) atomicMax(&d.ct[3], v);
        else if (v) atomicAdd(&d.ct[q], v);
    }
}

// Occupancy target per precision (waves per SIMD), measured on c2: the precision form runs
// best at 4 (VGPRs capped at 128), the FP64 form at 3 (capped at 168); the compiler's own
// choice (2 and 3) is 6-11% slower.
#ifndef SLGPU_WAVES_MIXED
#define SLGPU_WAVES_MIXED 4
#endif
#ifndef SLGPU_WAVES_FP64
#define SLGPU_WAVES_FP64 3
#endif
// A wave runs short DDMC steps while at least this many eighths of its lanes take them: 2, 3
// and 4 are within 4% of each other on c2 and c1, 5 and 6 are 10-40% slower (the lanes that
// wait for a full or an IMC pass wait too long for company of their own kind).
#ifndef SLGPU_RUN_EIGHTHS
#define SLGPU_RUN_EIGHTHS 3
#endif

// What a lane's particle carries that the short step does not touch waits in LDS between
// its full and IMC passes.
struct Cold {
    double x[256], mu[256], wl[256], vx[256];
    double pend_f[256], pend_r2[256];          // a recorded conversion
};

__device__ __forceinline__ void cold_load(Ptcl &p, const Cold &s)
{
    const int t = threadIdx.x;
    p.x = s.x[t]; p.mu = s.mu[t]; p.wl = s.wl[t]; p.vx = s.vx[t];
}
__device__ __forceinline__ void cold_store(const Ptcl &p, Cold &s)
{
    const int t = threadIdx.x;
    s.x[t] = p.x; s.mu[t] = p.mu; s.wl[t] = p.wl; s.vx[t] = p.vx;
}

// The short DDMC step: one event of diffusion11.f90:243-620 that needs no more than a pure
// bucket entry: an effective scatter, or a lumped particle's leak or Doppler shift inside the
// mesh; the group, the cell and the optical-depth flags of the destination all come from the
// entry.  These are 93% of the DDMC steps of the c2 workload.  A lane runs them back to back.
// Per step it waits for one round trip to memory: a lumped particle's event follows from the
// cell's thresholds (held in registers while the cell stays), so its entry comes from the
// right table at once; an unlumped one requests its threshold and the effective-scatter entry
// together.  The logarithm and the next step's Philox block are computed while they travel.
// Any other step is left untouched for diffusion11 (NF_FULL).  The draws, the arithmetic and
// the order of the sums are diffusion11's.  least: the lanes below which the wave leaves.
// An unlumped particle's Doppler shift samples no group: its threshold and the flags of the group it
// leads to come with the record of its group.
// What bounds it is instruction issue: four waves of a SIMD share it, and a lane alone is held up by
// dependent instructions and branches more than by the round trip.  So the tables' addresses stay in
// scalar registers, conditions are combined instead of branched on, and the generator's ten rounds
// are unrolled (in a loop of five trips they cost 15% of the transport).  Requesting the entry of the
// step after next as well, which is known to follow a pure effective scatter, halves the round
// trips but adds a generator block and an entry per step: 5% slower.
// Against a full diffusion11 pass per DDMC step, c2 (400 x 10^4) at 2^20 particles went from 3.69 to
// 2.87 s in the precision form and from 4.69 to 3.75 s in FP64; the leaner loop together with
// CellGeo and the unlumped Doppler shift took c2 at 2^17 particles from 1.03-1.09 to 0.90-0.98 s,
// FP64 (154 x 6000, 10^5 particles) from 0.35-0.38 to 0.31-0.34 s.
template <bool M>
__device__ __forceinline__ void short_run(const Dev &d, Ptcl &p, uint32_t pid, uint32_t k0, uint32_t k1,
                                          int64_t &istep, double &evelo, int &run_ic, double &run_e,
                                          double *s_tally, double *jrad, Cold &cold, BlockTotals &bt,
                                          int least)
{
    const uint32_t ng = d.ng, nx = d.nx;
    // in registers for the whole run, not fetched again from the kernel's arguments
#define GLOBAL_CONST __attribute__((address_space(1))) const
    GLOBAL_CONST uint32_t *btab = (GLOBAL_CONST uint32_t *)d.btab;
    GLOBAL_CONST ShortProb *gshort = (GLOBAL_CONST ShortProb *)d.gshort;
    GLOBAL_CONST ShortCell *cshort = (GLOBAL_CONST ShortCell *)d.cshort;
    asm volatile("" : "+s"(btab), "+s"(gshort), "+s"(cshort));
    auto cell = [&](uint32_t ic) {
        GLOBAL_CONST ShortCell *q = cshort + ic;
        return ShortCell{q->denom, q->divv, q->w1, q->w2, q->w3, 0u};
    };
    uint32_t o[4];
    Philox::block(pid, (uint32_t)(istep + 1), StepRng::PHASE, 0u, k0, k1, o);
    ShortCell c = cell(p.ix - 1), cn = c;                    // of the particle's cell, of the next
    uint32_t wlg = 0;                                          // group edge a Doppler shift left wl at
    bool go = true, open;
    uint32_t t, ent, w3, w1;
    double denom;
    auto request = [&]() {
        const uint32_t ic = p.ix, w = o[1];
        const bool lump = (p.nflag & BT_LUMP) != 0;
        const uint32_t tl = w > c.w3 ? TAB_S : (w < c.w1 ? TAB_D : (w < c.w2 ? TAB_L : TAB_R));
        t = lump ? tl : (uint32_t)TAB_E;
        ent = btab[((t * nx + (ic - 1)) << BT_BITS) + (o[2] >> (32 - BT_BITS))];
        // undecided, or a face of the mesh: not a short step
        open = lump & ((w == c.w1) | (w == c.w2) | (w == c.w3) | ((t == TAB_L) & (ic == 1)) |
                                  ((t == TAB_R) & (ic == nx)));
        denom = c.denom;
        w3 = w1 = 0u;
        if (!lump) {
            GLOBAL_CONST ShortProb *q = gshort + ((ic - 1) * ng + (p.ig - 1));
            denom = q->denom;
            w3 = q->w3;
            w1 = q->w1;
        }
        if ((t <= TAB_R) & !open) cn = cell(t == TAB_L ? ic - 2 : ic);
    };
    request();
    do {
        const double lrt = p_log<M>(Philox::u42(o[0], o[3] & 0x3FFu));
        const uint32_t w = o[1], r2_hi = o[2], r2_lo = o[3] >> 20;
        Philox::block<10>(pid, (uint32_t)(istep + 2), StepRng::PHASE, 0u, k0, k1, o);
        asm volatile("" : "+v"(o[0]), "+v"(o[1]), "+v"(o[2]), "+v"(o[3]));     // before the wait
        __builtin_amdgcn_sched_barrier(0);
        // an unlumped particle's Doppler shift samples no group
        const bool shift = (w & ~3u) < (w1 & ~3u);
        ent = shift ? BT_PURE | (w1 & 3u) << 29 | (uint32_t)p.ig : ent;
        t = shift ? (uint32_t)TAB_D : t;
        if (((ent & BT_PURE) != 0u) & !open & (denom == denom) & ((t != TAB_E) | (w > w3))) {
            const uint32_t ic = p.ix;
            const double ddmct = fabs(lrt * denom * CINV);
            const double erd = p.e * ddmct, jrd = PC_C * erd;
            if (jrd != 0.0) atomicAdd(jrad + ((ic - 1) * ng + (p.ig - 1)), jrd);
            run_e += erd;
            uint32_t g = ent & 0x7fffu, kind = PEND_SCAT;
            if (t == TAB_D) {
                kind = PEND_DOP;
                wlg = c.divv >= 0 ? g + 1 : g;
                g = c.divv >= 0 ? (g + 1 > ng ? ng : g + 1) : (g < 2 ? 1 : g - 1);
            } else if (t <= TAB_R) {
                kind = t == TAB_L ? PEND_LEFT : PEND_RIGHT;
                atomicAdd(&s_tally[ic - 1], run_e);
                run_e = 0.0;
                p.ix = t == TAB_L ? ic - 1 : ic + 1;
                c = cn;
            }
            p.ig = g;
            ++istep;
            const double f = p_adiabatic<M>(c.divv, ddmct);
            if (ent & BT_THIN) {                               // conversion, at the next pass
                p.itype = 1;
                p.nflag = (kind << 1) | (ent & BT_LUMP);
                cold.pend_f[threadIdx.x] = f;
                if (shift) {                                   // whose third draw is still unused
                    p.nflag |= NF_R2FREE;
                    cold.pend_r2[threadIdx.x] = Philox::u42(r2_hi, r2_lo & 0x3FFu);
                }
                atomicAdd(&bt.ct[4], 1ull);
                go = false;
            } else {
                p.nflag = NF_VALID | (ent & BT_LUMP);
                evelo = evelo + p.e * (1.0 - f);
                p.e = p.e * f;
            }
        } else {
            p.nflag |= NF_FULL;
            go = false;
        }
        // max_steps belongs to the full step; leave when too few of the wave's lanes remain
        go = go && istep + 1 < d.max_steps;
        if (__popcll(__ballot(go)) < least) go = false;
        if (go) request();
    } while (go);
    run_ic = p.ix;
    if (wlg) cold.wl[threadIdx.x] = d.wl[wlg - 1];
}

// particle_advance.f90:140-294 as a persistent kernel: each lane takes the next particle
// from a global counter, runs it event by event to escape or death (145-202 on start,
// 271-292 at the end), then takes another, so lanes stay busy until the pool is empty.
// Lanes that leave the loop drop out of the votes; a pass always runs the kind of at
// least one remaining lane, so every particle advances.  lanes: how many lanes of a wave take
// particles.  A pool smaller than the lanes resident on the chip is spread over all waves: its
// time is the longest walk's, and a step costs a lane 1.9 us with one neighbour in its wave
// against 3 us with 31 (8192 particles on c2: 1.34 s in full waves, 0.59 s spread).
// X: the amplification factor or anisotropic Thomson scattering is on; without them the kernel
// holds 5 KB less code and needs no scratch memory (36 bytes per lane otherwise).
template <bool M, bool X>
__global__ __launch_bounds__(256)
__attribute__((amdgpu_waves_per_eu(M ? SLGPU_WAVES_MIXED : SLGPU_WAVES_FP64, 8)))
void k_transport(Dev d, uint32_t iteration, int lanes)
{
    extern __shared__ double s_tally[];
    const int ng = d.ng, nx = d.nx;
    __shared__ BlockTotals bt;
    __shared__ Cold cold;
    for (int k = threadIdx.x; k < nx; k += blockDim.x) s_tally[k] = 0.0;
    if (threadIdx.x < 7) bt.tot[threadIdx.x] = 0.0;
    if (threadIdx.x < 9) bt.ct[threadIdx.x] = 0;
    __syncthreads();
    double evelo = 0.0;
    int run_ic = -1;
    double run_e = 0.0;
    double *jrad = d.jrad + (size_t)(blockIdx.x % d.jrad_copies) * nx * ng;
    Ptcl p;
    StepRng s;
    s.key(d.seed, iteration);
    uint32_t ip = 0;
    int64_t istep = 0;
    bool have = false;
    for (;;) {
        if (!have) {
            if ((int)(threadIdx.x & 63) >= lanes) break;
            const int64_t next = (int64_t)atomicAdd(d.queue, 1ull);
            if (next >= d.npart) break;
            ip = (uint32_t)next;
            p.x = d.px[ip]; p.mu = d.pmu[ip]; p.e = d.pe[ip]; p.wl = d.pwl[ip];
            atomicAdd(&bt.tot[5], p.e);
            atomicAdd(&bt.ct[0], 1ull);
            p.ix = binsrch(p.x, d.xarr, nx + 1, false);
            p.ig = binsrch(p.wl, d.wl, ng + 1, false);
            if (p.ix < 1 || p.ig < 1) {                        // NaN position or wavelength
                atomicAdd(&bt.ct[7], 1ull); atomicAdd(&bt.ct[6], 1ull);
                atomicAdd(&bt.tot[4], p.e);
                d.pstat[ip] = 2; d.perr[ip] = 1; d.pnstep[ip] = 0;
                continue;
            }
            const double tau = (SIGT(p.ix) + CAPT(p.ig, p.ix)) * DXX(p.ix);
            p.itype = (d.puretran || tau < d.tauddmc) ? 1 : 2;
            const double h1 = XA(p.ix), h2 = XA(p.ix + 1);
            p.vx = (VXA(p.ix) * (h2 - p.x) + VXA(p.ix + 1) * (p.x - h1)) / (h2 - h1);
            if (p.itype == 1) {
                const double labfact = 1.0 - p.vx * p.mu / PC_C;
                p.wl = p.wl * labfact;
                p.e = p.e / labfact;
            }
            atomicAdd(&bt.tot[3], p.e);
            p.nflag = 0;
            cold_store(p, cold);
            istep = 0;
            have = true;
        }
        // The wave runs one kind of step per pass: short DDMC steps while they are enough of
        // its lanes, else one IMC event or one full DDMC event, whichever more lanes wait for.
        // The other lanes wait a pass, so each pass executes one body.
        const bool imc = p.itype == 1 || d.puretran;
        const bool quick = !imc && (p.nflag & (NF_VALID | NF_FULL)) == NF_VALID && istep + 1 < d.max_steps;
        const int n_imc = __popcll(__ballot(imc)), n_quick = __popcll(__ballot(quick));
        const int live = __popcll(__ballot(1)), n_full = live - n_imc - n_quick;
        const int least = (SLGPU_RUN_EIGHTHS * live + 7) / 8;
        if (n_quick >= least) {
            if (quick) {
                if (p.ix != run_ic) {
                    if (run_ic > 0) atomicAdd(&s_tally[run_ic - 1], run_e);
                    run_ic = p.ix; run_e = 0.0;
                }
                short_run<M>(d, p, ip, s.k0, s.k1, istep, evelo, run_ic, run_e, s_tally, jrad, cold, bt, least);
            }
            continue;
        }
        if (quick || imc != (n_imc >= n_full)) continue;
        istep++;
        cold_load(p, cold);
        p.stat = 0;
        p.idist = 0;
        s.init(ip);
        ImcIn q;
        if (imc) imc_request(d, p, q);
        if (imc && (p.nflag & NF_PEND))
            imc_entry<M>(d, p, s, q, (uint32_t)(istep - 1), evelo, cold.pend_f[threadIdx.x], cold.pend_r2[threadIdx.x]);
        s.begin_step((uint32_t)istep);
        const int icold = p.ix, igold = p.ig;
        double erd, jrd;
        int ierr;
        if (imc) {
            double ea;
            atomicAdd(&bt.ct[1], 1ull);
            ierr = transport11<M, X>(d, p, s, q, erd, jrd, ea, evelo);
            if (ea != 0.0) {                                   // particle_advance.f90:216-217
                atomicAdd(&d.eamp[icold - 1], ea);
                atomicAdd(&bt.tot[6], ea);
            }
            if (p.itype != 1) atomicAdd(&bt.ct[4], 1ull);
        } else {
            ierr = diffusion11<M>(d, p, s, erd, jrd, evelo, cold.pend_f[threadIdx.x], cold.pend_r2[threadIdx.x]);
            if (p.itype == 1) atomicAdd(&bt.ct[4], 1ull);
        }
        // grd_jrad: one FP64 atomic per event into the block's replica (the group changes on
        // almost every step, so merging a particle's events would save no atomics); the
        // energy tally merges a particle's consecutive events in one cell before its LDS atomic
        if (jrd != 0.0) atomicAdd(&jrad[(size_t)(icold - 1) * ng + igold - 1], jrd);
        if (icold != run_ic) {
            if (run_ic > 0) atomicAdd(&s_tally[run_ic - 1], run_e);
            run_ic = icold; run_e = 0.0;
        }
        run_e += erd;
        if (p.itype == 1 && p.stat == 0 && !(p.nflag & NF_PEND)) {   // particle_advance.f90:234-250
            if (p.x > XA(p.ix + 1) || p.x < XA(p.ix) || p.x != p.x) {
                if (ierr == 0) ierr = -99;
            }
        }
        if (ierr < 0) atomicAdd(&bt.ct[8], 1ull);
        if (ierr == 0 && p.stat == 0 && istep >= d.max_steps) ierr = 200;
        if (ierr > 0) { atomicAdd(&bt.ct[7], 1ull); p.stat = 2; }
        if (p.stat != 0) {
            if (p.nflag & NF_PEND) {                           // stopped by max_steps right after
                imc_request(d, p, q);
                imc_entry<M>(d, p, s, q, (uint32_t)istep, evelo, cold.pend_f[threadIdx.x], cold.pend_r2[threadIdx.x]);
            }
            atomicMax(&bt.ct[3], (unsigned long long)istep);
            atomicAdd(&bt.ct[2], (unsigned long long)istep);
            if (p.stat == 2) { atomicAdd(&bt.ct[6], 1ull); atomicAdd(&bt.tot[4], p.e); }
            else { atomicAdd(&bt.ct[5], 1ull); atomicAdd(&bt.tot[0], p.e); }
            d.pstat[ip] = (uint8_t)p.stat;
            d.px[ip] = p.x; d.pmu[ip] = p.mu; d.pwl[ip] = p.wl; d.pe[ip] = p.e;
            d.pig[ip] = p.ig; d.pix[ip] = p.ix;
            d.pnstep[ip] = istep;
            d.perr[ip] = ierr > 0 ? ierr : 0;
            have = false;
        } else {
            cold_store(p, cold);
            // inside the innermost face every DDMC step ends the particle (diffusion11.f90:623-626)
            if (p.itype == 2 && p.x < XA(1)) p.nflag |= NF_FULL;
        }
    }
    if (run_ic > 0) atomicAdd(&s_tally[run_ic - 1], run_e);
    __syncthreads();
    for (int k = threadIdx.x; k < nx; k += blockDim.x)
        if (s_tally[k] != 0.0) atomicAdd(&d.tally[k], s_tally[k]);
    flush_totals(d, bt, evelo);
}

// fluxtally.f:30-54 (flux grid == group grid; polar/azimuth bins are single)
__global__ __launch_bounds__(256) void k_fluxtally(Dev d)
{
    const int64_t p = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (p >= d.npart) return;
    if (d.pstat[p] != 1) return;
    const int ig = binsrch(d.pwl[p], d.wl, d.ng + 1, false);
    if (ig < 1) return;                  // NaN wavelength: not binned
    const double e = d.pe[p];
    atomicAdd(&d.lum[ig - 1], e);
    atomicAdd(&d.dev[ig - 1], e * e);
    atomicAdd(&d.num[ig - 1], 1);
}

// The same for group grids whose edges and bins fit a block's LDS: particles outnumber the bins a
// thousandfold at 2^20 x 1000, and their atomics on a bin follow each other.  A block bins its share
// in LDS, searching the edges there, and adds its nonzero bins to the tally.
// 2^20 particles on 1000 groups: 0.50 ms with every particle's atomics on the tally, 0.09 ms so;
// 16384 on 250: 24 us, under 10 us so.
constexpr int FLUX_THREADS = 1024, FLUX_GROUPS = 2300;     // 28 bytes a group, 64 KB of LDS
__global__ __launch_bounds__(FLUX_THREADS) void k_fluxtally_lds(Dev d)
{
    extern __shared__ double s_edge[];
    const int ng = d.ng;
    double *lum = s_edge + ng + 1, *dev = lum + ng;
    int *num = (int *)(dev + ng);
    for (int g = threadIdx.x; g <= ng; g += FLUX_THREADS) s_edge[g] = d.wl[g];
    for (int g = threadIdx.x; g < ng; g += FLUX_THREADS) { lum[g] = 0.0; dev[g] = 0.0; num[g] = 0; }
    __syncthreads();
    for (int64_t p = (int64_t)blockIdx.x * FLUX_THREADS + threadIdx.x; p < d.npart; p += (int64_t)gridDim.x * FLUX_THREADS) {
        const int stat = d.pstat[p];
        const double wl = d.pwl[p], e = d.pe[p];
        if (stat != 1) continue;
        const int ig = binsrch(wl, s_edge, ng + 1, false);
        if (ig < 1) continue;            // NaN wavelength: not binned
        atomicAdd(&lum[ig - 1], e);
        atomicAdd(&dev[ig - 1], e * e);
        atomicAdd(&num[ig - 1], 1);
    }
    __syncthreads();
    for (int g = threadIdx.x; g < ng; g += FLUX_THREADS) {
        if (num[g] == 0) continue;
        atomicAdd(&d.lum[g], lum[g]);
        atomicAdd(&d.dev[g], dev[g]);
        atomicAdd(&d.num[g], num[g]);
    }
}

void launch_sources(slgpu_ctx *c, uint32_t iteration)
{
    int64_t n = c->d.npart;
    if (n == 0) return;
    hipLaunchKernelGGL(k_sources, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, c->stream,
                       c->d, iteration);
}

// the transport's per-cell record, from what was set last
__global__ __launch_bounds__(256) void k_cell_geo(Dev d)
{
    const int i = blockIdx.x * 256 + threadIdx.x;
    if (i >= d.nx) return;
    CellGeo g;
    g.xl = d.xarr[i]; g.xr = d.xarr[i + 1];
    g.vl = d.vxarr[i]; g.vr = d.vxarr[i + 1];
    g.sg = d.sig[i]; g.dvdr = d.dvdr[i]; g.c3 = d.c3divv[i];
    g.em = d.capemgrey[i];
    g.far = 2.0 * fabs(sqrt(g.xr * g.xr - g.xl * g.xl));
    g.vhelp = g.vl - g.dvdr * g.xl;
    g.nlump = d.cell[i].nlump;
    g.pad[0] = g.pad[1] = g.pad[2] = 0;
    d.geo[i] = g;
    d.cshort[i].divv = d.divv[i];
}

void launch_transport(slgpu_ctx *c, uint32_t iteration)
{
    hipLaunchKernelGGL(k_cell_geo, dim3((c->nx + 255) / 256), dim3(256), 0, c->stream, c->d);
    int dev = 0, ncu = 256;
    (void)hipGetDevice(&dev);
    (void)hipDeviceGetAttribute(&ncu, hipDeviceAttributeMultiprocessorCount, dev);
    const int64_t resident = (int64_t)ncu * 4 * (c->d.precision == SLGPU_MIXED ? SLGPU_WAVES_MIXED : SLGPU_WAVES_FP64);
    // Pure IMC: half waves at least.  Its passes cost a wave as much for 1 to 8 lanes as for 64, and less
    // for 16 to 32 (20 x 300, 3000 steps each, FP64: 300 particles 22 ms alone, 21 by 8, 15 by 16, 13 by
    // 32 and 14 by 64; 3000 21, 23, 16, 14 and 17; precision form alike).
    const int64_t share = std::max<int64_t>(c->d.puretran ? 32 : 1, (c->d.npart + resident - 1) / resident);
    const int lanes = share > 64 ? 64 : (int)share;
    // no more blocks than take particles: an empty pool's 2048 cost 90 us of queue and flush
    const int64_t blocks = std::max<int64_t>(1, std::min<int64_t>((int64_t)ncu * 8, (c->d.npart + 4 * lanes - 1) / (4 * lanes)));
    const bool extra = c->d.ampfact || c->d.thm_aniso;
    auto kernel = c->d.precision == SLGPU_MIXED ? (extra ? k_transport<true, true> : k_transport<true, false>)
                                                : (extra ? k_transport<false, true> : k_transport<false, false>);
    hipLaunchKernelGGL(kernel, dim3((unsigned)blocks), dim3(256), c->nx * sizeof(double), c->stream, c->d,
                       iteration, lanes);
}

// the transport's group samplers at arbitrary (r, cell), table path or direct search
__global__ __launch_bounds__(256) void k_sample_groups(Dev d, int t, int direct, int64_t n,
                                                       const double *r, const int *cell, int *out)
{
    const int64_t k = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (k >= n) return;
    const int ic = cell[k];
    if (ic < 1 || ic > d.nx) { out[k] = -1; return; }
    const int nlump = d.cell[ic - 1].nlump;
    if (t != TAB_E) {
        const LumpRow L = lump_row(d, t, ic, nlump);
        if (nlump == 0 || L.cnt == 0) { out[k] = 0; return; }
        if (direct) { out[k] = lump_group(d, L, ic, first_above(L.cum, 0, L.cnt, r[k])); return; }
    } else if (direct) {
        out[k] = emitgroup_direct(d, r[k], ic);
        return;
    }
    int thin;
    out[k] = sample_group(d, t, ic, nlump, r[k], thin);
}

void launch_sample_groups(slgpu_ctx *c, int t, int direct, int64_t n, const double *r,
                          const int *cell, int *out)
{
    hipLaunchKernelGGL(k_sample_groups, dim3((unsigned)((n + 255) / 256)), dim3(256), 0,
                       c->stream, c->d, t, direct, n, r, cell, out);
}

// fold the grd_jrad replicas into replica 0 (fixed order per element)
__global__ __launch_bounds__(256) void k_jrad_reduce(Dev d)
{
    const size_t n = (size_t)d.nx * d.ng;
    for (size_t k = (size_t)blockIdx.x * blockDim.x + threadIdx.x; k < n;
         k += (size_t)gridDim.x * blockDim.x) {
        double s = d.jrad[k];
        for (int r = 1; r < d.jrad_copies; ++r) s += d.jrad[(size_t)r * n + k];
        d.jrad[k] = s;
    }
}

void launch_jrad_reduce(slgpu_ctx *c)
{
    if (c->d.jrad_copies <= 1) return;
    const size_t n = (size_t)c->nx * c->ng;
    size_t blocks = (n + 255) / 256;
    if (blocks > 8192) blocks = 8192;
    hipLaunchKernelGGL(k_jrad_reduce, dim3((unsigned)blocks), dim3(256), 0, c->stream, c->d);
}

void launch_fluxtally(slgpu_ctx *c)
{
    int64_t n = c->d.npart;
    if (n == 0) return;
    if (c->ng <= FLUX_GROUPS) {
        // a block's rounds over its particles take about 1.3 us each, and the bins it flushes 3 ng
        // atomics of 0.16 ns: the sum is least at this count
        const double least = sqrt(2.7 * (double)n / c->ng);
        const int64_t most = std::min<int64_t>(256, (n + FLUX_THREADS - 1) / FLUX_THREADS);
        const unsigned blocks = (unsigned)std::max<int64_t>(1, std::min<int64_t>(most, (int64_t)ceil(least)));
        hipLaunchKernelGGL(k_fluxtally_lds, dim3(blocks), dim3(FLUX_THREADS), (size_t)28 * c->ng + 8, c->stream, c->d);
        return;
    }
    hipLaunchKernelGGL(k_fluxtally, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, c->stream,
                       c->d);
}

}  // namespace slgpu
