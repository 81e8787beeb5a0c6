// Internal state of an slgpu context and the kernel launchers shared between the
// translation units of libslgpu.so.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <string>
#include <vector>

#include "../../include/slgpu.h"
#include "slgpu_device.h"
#include "slgpu_hostio.h"

namespace slgpu {

// One packed line record (the bb_xs fields the binning needs), 16 bytes.
struct LineRec {
    float gxs;      // g*f*(pi e^2/m_e c)
    float chilw;    // lower-level energy [1/cm]
    int ion;        // index into the population list
    int pad;        // in the ion-ordered copy: lines left in this record's ion run
};

// A line of the FP64 line sums, in ion order within its group: its lower level split over the
// rows of the cell's exponential tables, chi = (EXP_K2 k1 + k2) step + r (k_opacity64).
struct Line64 {
    double gxs, r;
    uint32_t k1, k2;    // byte offsets of the rows k1 and EXP_K1 + k2, 512 bytes a row
    uint32_t ion;       // 512 times the ion index, plus 1 on the last line of its run
    float chi;
};
constexpr int EXP_K1 = 32, EXP_K2 = 32, EXP_ROWS = EXP_K1 + EXP_K2;

// What an IMC event reads of its cell: faces, their velocities, sigma_T, dv/dr, 3c/divv,
// capgrey (capemitgrey in NLTE), the longest chord, v - dv/dr r at the inner face and the
// number of lumped groups.
struct CellGeo {
    double xl, xr, vl, vr, sg, dvdr, c3, em, far, vhelp;
    int nlump, pad[3];
};

// Per-cell DDMC constants (diffusion11.f90:95-152), evaluated once per iteration.
struct CellDDMC {
    double emgreyinv;   // 1/capgrey (LTE) or 1/capemitgrey (NLTE), nan -> 0
    double speclump, emitlump, caplump, doplump;
    int nlump;
    int pad;
};

// Event thresholds of one DDMC step in a cell (lumped) or a (cell, group) (unlumped),
// diffusion11.f90:243-283: 1/denominator and the cumulative Doppler / left / right
// probabilities the event draw is compared against.
struct DdmcProb {
    double denom, t1, t2, t3;
};

// The same for the transport's short step: the event thresholds as 32-bit words compared with
// a generator word (k_ddmc_probs), half the bytes of the FP64 record per random gather.
struct ShortProb {              // an unlumped (cell, group): scatter above w3, Doppler shift below w1
    double denom;
    uint32_t w3, w1;            // w1: its upper 30 bits; below, BT_LUMP and BT_THIN of the shift's group
};
struct ShortCell {              // a cell's lumped step, and its divv
    double denom, divv;
    uint32_t w1, w2, w3, pad;
};

// Everything the kernels read or write, passed to kernels by value.
struct Dev {
    int nx, ng, nep, nepg, nion, nel;
    double tauddmc, taulump;
    int puretran, precision;
    int ampfact, thm_aniso;     // !in_trn_noamp, in_thm_aniso
    int64_t max_steps;
    uint32_t seed;
    // mesh (nx+1 / nx)
    const double *xarr, *vxarr, *divv, *vol;
    const double *dvdr, *c3divv;  // nx: (v_{i+1}-v_i)/dx_i and 3c/divv_i (transport11.f90:130,145-149)
    // groups (ng+1)
    const double *wl, *wlinv;
    // lines
    const LineRec *lines;
    const LineRec *lines_ion;   // the same records, sorted by ion within each group (backward)
    Line64 *lines64;            // the records of the FP64 line sums, in lines_ion's order
    double *etab;               // EXP_ROWS*nc: the cells' exponential tables, cell fastest
    double line_step;           // the tables' fine step [1/cm]; 0: no tables (see build_lines64)
    const int *gstart;          // ng+2: lines of group g (1-based) are [gstart[g], gstart[g+1])
    // tables
    double *bfxs;               // ng*nion, xs(ig, k)*1e-18 (Mb -> cm^2)
    uint32_t *bfmask;           // ng*((nion+31)/32): which of a group's bfxs are not zero
    const double *gff;          // 81*41 Fortran order
    // per-iteration gas state (cell-fastest, [k*nc + i])
    double *hckt, *hlparr, *ocg, *ocT, *sig, *tempinv, *temp, *mass, *natomfr;
    double *ffB;                          // FF_NU*nx, cell fastest: per cell, the sum over the unclamped elements
                                          // of z^2 natomfr times g_ff interpolated in gamma^2, at
                                          // each u node (physical_opacity.f:228-243)
    uint32_t *ffclamp;                    // nx: bit k set when element k's gamma^2 coordinate lies
                                          // past the table, where g_ff is clamped to >= 1 per group
    double *ffC;                          // FF_NU*nx: as ffB, with the g_ff rows' difference in
                                          // gamma^2 (the backward's slope of g_ff in rgg)
    double *ctpart;                       // 2*((ng+1023)/1024)*nx: the means' per-slice partial sums
    double *gmpart;                       // 2*((ng+63)/64)*nx: the means backward's per-tile
                                          // partial sums of dL/dT and dL/dsig
    int *el_z;                  // nel present elements (ascending iz)
    // opacity products
    double *capT;               // ng*nc cell-fastest scratch
    double *cap64;              // nc*ng group-fastest
    float *cap32, *emiss;       // nc*ng group-fastest (gas_cap, gas_emiss)
    double *capgrey, *capross;
    // emission opacity of the DDMC prep and the emission samplers: grd_capemit and
    // grd_capemitgrey after an NLTE build (nlte = 1), cap32 and capgrey after an LTE one
    const float *capem32;
    const double *capemgrey;
    int nlte;
    // DDMC prep
    double *specarr;            // nc*ng  specintv(tempinv(ic)) group-fastest
    double *opaclump;           // 11*nc
    double *emitprob;           // nep*nc
    double *emitcum;            // nc*ng  cumulative emission probability inside each bin
    double *emit;               // nc
    double *radtemp;            // nc
    double *srccum;             // nc*ng  cumulative normalised Planck at T_rad
    double *srctot;             // nc     its total before normalisation
    CellDDMC *cell;             // nc
    DdmcProb *cprob;            // nc     lumped-group step of each cell
    DdmcProb *gprob;            // nc*ng  unlumped step of each (cell, group), group-fastest
    ShortProb *gshort;          // nc*ng  the short step's form of gprob
    CellGeo *geo;
    ShortCell *cshort;          // nc     and of cprob
    int *gorder;                // nc*ng  lumped groups ascending, then unlumped ascending
    double *cumL, *cumR, *cumD, *cumS;   // nc*ng cumulative lumped sampling weights
    uint32_t *btab;             // 5*nc*BT_K bucket maps of the cumL/R/D/S rows and emitgroup
    // particles (SoA)
    int64_t npart;
    const int64_t *pstart;      // nc+1
    double *px, *pmu, *pwl, *pe;
    uint8_t *pstat;
    int *pig, *pix, *perr;
    int64_t *pnstep;
    // tallies
    // inputs of the last opacity build kept for its backward, and the backward's scratch
    double *natom_in, *vol_in, *nelec_in; // nc
    double *ginvT;                        // nion*nc (ion-major)
    double *gcapT;                        // ng*nc cell-fastest dL/dcap after the means
    // the backward's accumulators, one allocation in this order (vjp_acc_doubles)
    double *goc;                          // GACC_COPIES*nion*nc ion-major
    double *ffW;                          // GACC_COPIES*FF_NU*nc: sum over groups of G*help spread
                                          // onto the two u nodes of each group
    double *gcell;                        // 2*nc: dL/dhckt, dL/dhlparr
    double *gfr;                          // 30*nc element-major
    double *tally, *jrad, *tot;           // nc, jrad_copies*nc*ng, 8
    double *eamp;                         // nc grd_eamp
    int jrad_copies;                      // replicas of grd_jrad that spread atomic traffic
    unsigned long long *ct;               // 10
    unsigned long long *queue;            // work counter of the persistent transport
    double *lum, *dev;                    // ng
    int *num;                             // ng
    int *flags;                           // bad input flags raised by kernels
    // LTE EOS: the host's ion data (ionsmod.f ion_el) and the state of the last solve
    int *ion_z, *ion_i;                   // nion: the ion list of slgpu_set_ions on the device
    int *eos_ni;                          // 30
    double *eos_e, *eos_q, *eos_g1;       // 30*31 [iz-1][ii-1]
    double *eos_amass;                    // 30
    double *eos_sahac2;                   // nc: Saha constant of the last evaluation (0: not solved)
};

// NLTE hydrogen (physical_opacity_nlte.f): the species data of slgpu_set_nlte_data, the
// per-call inputs and the work arrays, passed by value to the NLTE kernels only.
// One NLTE line, in the order of its group; a wave reads it as one uniform record.
struct HLine {
    double f, gl, gu, aul, wl0;
    int lw, lu;                                 // level indices from 0
};

// What the (cell, group) kernel of an NLTE build needs beside Dev.
struct NlteOut {
    const int *hstart;
    const HLine *hline;
    const double *popT, *ndens;                 // (n, nc), (nc, 2)
    double *capemitT, *emissT;                  // (ng, nc)
};

struct NlteDev {
    int n = 0, nlin = 0, ncoll = 0, kH = -1;    // levels, lines, collision lines, H I ion index
    double *glev, *aul, *bul, *blu;             // nlev / nlin
    double *cc, *dele;                          // 4*ncoll, ncoll
    double *pic, *rrc, *delepi;                 // 4*nlev, 4*nlev, nlev
    int *llw, *lup, *igs;                       // nlin (igs: group of the line, 0 outside)
    int *cl, *cu, *levpi;                       // ncoll, ncoll, nlev
    int *hstart;                                // ng+2 offsets
    HLine *hline;                               // the lines by group, in file order
    double *radtemp, *ndens;                    // nc, 2*nc (H I, H II per cell)
    double *A;                                  // nc*n*(n+1), where the matrix does not fit LDS
    double *pop, *popT;                         // nc*n, and its transpose
    int *flag;                                  // 1
    double *capemitT, *emissT;                  // (ng, nc) cell-fastest
    float *capemit32;                           // (nc, ng)
    double *capemitgrey;                        // nc
};

inline __host__ __device__ NlteOut nlte_out(const NlteDev &q)
{
    return {q.hstart, q.hline, q.popT, q.ndens, q.capemitT, q.emissT};
}

constexpr int GACC_COPIES = 8;          // copies of the backward's most contended accumulators
inline size_t vjp_acc_doubles(int nion, size_t nc)
{
    return ((size_t)GACC_COPIES * ((nion > 1 ? nion : 1) + FF_NU) + 2 + 30) * nc;
}

struct Timer {
    hipEvent_t a, b;
    bool armed = false;
};

}  // namespace slgpu

struct slgpu_ctx {
    slgpu_config cfg;
    slgpu::Dev d;
    hipStream_t stream = nullptr;
    int ng = 0, nx = 0, nion = 0;
    bool have_grid = false, have_groups = false, have_lines = false, have_bf = false,
         have_ff = false, have_ions = false, have_opacity = false, have_prep = false,
         have_sources = false, have_transport = false;
    int force_unstaged = 0;                // slgpu_set_unstaged: opacity and backward unstaged
    int64_t nline = 0, nline_used = 0;
    std::vector<double> h_xarr, h_vxarr, h_divv, h_vol, h_rcell, h_wl;
    std::vector<int> h_ion_iz, h_ion_ii;
    std::vector<float> h_ph1, h_ph2;
    std::vector<float> h_wl0;
    std::vector<int16_t> h_liz, h_lii;
    std::vector<float> h_gxs, h_chilw;
    std::vector<double> h_emit_cache;
    double line_top = 0.0;      // largest lower level of the used lines [1/cm]; 0: no tables
    double hckt_max = 0.0;      // largest hc/kT of the last build's cells
    double etab_step = 0.0;     // line_step that Dev::etab was filled with for the last build's cells; 0: not
    int opac_flags = 0;         // flags of the last opacity build (its backward uses them)
    std::vector<void *> allocations;
    bool have_eos_data = false, have_eos = false;
    // inputs and outputs of the last slgpu_eos, kept on the device for slgpu_eos_vjp
    double *eos_temp = nullptr, *eos_mass = nullptr, *eos_massfr = nullptr, *eos_nelec = nullptr,
           *eos_natom = nullptr, *eos_natomfr = nullptr, *eos_oc = nullptr, *eos_ginv = nullptr;
    int *eos_niter = nullptr;
    double *stage = nullptr;    // ion populations of an opacity build (oc, ginv)
    double *vjp_out = nullptr, *vjp_in = nullptr, *eos_vjp = nullptr;   // backward's workspaces
    double *est = nullptr, *ndens = nullptr;        // slgpu_nlte_rad_est, slgpu_eos_nlte_ndens
    slgpu::HostIO io;
    slgpu::NlteDev nl;          // NLTE species data and work arrays (slgpu_set_nlte_data)
    bool have_nlte = false;
    void *scratch = nullptr;    // device address of the library's static scratch array on this context's GPU
    double t_ms[12] = {0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0};
    hipEvent_t ev[24];
};

namespace slgpu {
// launchers (each enqueues on ctx->stream)
void launch_bfxs(slgpu_ctx *c, const float *d_ph1, const float *d_ph2, const int *d_iz,
                 const int *d_ii);
void launch_cell_prep(slgpu_ctx *c, const double *d_natom, const double *d_vol,
                      const double *d_nelec, const double *d_oc, const double *d_ginv,
                      int flags);
void launch_lines64(slgpu_ctx *c, int64_t n);
void launch_exp_table(slgpu_ctx *c);
int line_degree(const slgpu_ctx *c);
void launch_eos_ndens(slgpu_ctx *c, const double *temp, const double *mass, const double *natom,
                      const double *natomfr, double *ndens);
void launch_nlte_rad_est(slgpu_ctx *c, double *radtemp, double *jrad);
void launch_opacity(slgpu_ctx *c, int flags);
void launch_opacity_finish(slgpu_ctx *c);
void launch_cell_tables(slgpu_ctx *c);
void launch_opacity_nlte(slgpu_ctx *c, int flags, double ffc1, const double *rgg);
void launch_nlte_means(slgpu_ctx *c);
bool nlte_in_lds(int n);
bool launch_opacity64_nlte(slgpu_ctx *c, int flags, double ffc1, const double *rgg);
double ff_prefactor();
const double *rgg_scratch(slgpu_ctx *c);
void launch_opacity_vjp(slgpu_ctx *c, int flags, const double *gc, const double *gp,
                        const double *gr, double *gT, double *gnat, double *gne, double *gfr,
                        double *goc, double ffc1, const double *rgg);
void launch_ddmc_tables(slgpu_ctx *c);
void launch_ddmc_probs(slgpu_ctx *c);
void launch_sources(slgpu_ctx *c, uint32_t iteration);
void launch_transport(slgpu_ctx *c, uint32_t iteration);
void launch_fluxtally(slgpu_ctx *c);
void launch_jrad_reduce(slgpu_ctx *c);
void launch_sample_groups(slgpu_ctx *c, int t, int direct, int64_t n, const double *r,
                          const int *cell, int *out);
void launch_eos(slgpu_ctx *c, const double *temp, const double *mass, const double *massfr,
                double acc, double *nelec, double *natom, double *natomfr, double *oc,
                double *ginv, int *niter);
void launch_eos_vjp(slgpu_ctx *c, const double *temp, const double *mass, const double *massfr,
                    const double *nelec, const double *natom, const double *natomfr,
                    const double *oc, const double *g_natom, const double *g_fr,
                    const double *g_ne, const double *g_oc, double *out_T, double *out_mass,
                    double *out_mf);

// ---------------------------------------------------------------------------
// The FP64 line sums.  exp(-chi h), with h = hc/kT of the cell, is the product of two entries of
// the cell's tables and a short polynomial: chi = (K2 k1 + k2) step + r, |r| <= step/2, splits
// exactly (step has few bits, chi is single), so
//   exp(-chi h) = E1[k1] E2[k2] P(-r h),   E1[k1] = exp(-K2 k1 step h),  E2[k2] = exp(-k2 step h).
// The tables (64 entries per cell, k_exp_table) stand in LDS as rows of the block's 64 cells; k1, k2, r
// and gxs are the same for the whole wave and come as scalars.  That is 10 FP64 operations
// and two LDS rows per line and cell, against about 50 for exp() and the reference's product;
// its error is that of the table entries and their products (2-3 units in the last place; exp()
// takes the product chi h rounded, an error of chi h / 2 units, more from chi h = 5 on).  P is the
// Taylor polynomial of degree DEG; the launch picks the smallest whose remainder, relative to the
// exponential at the largest |r h|, stays under 2^-53 (line_degree).
template <int DEG> __device__ __forceinline__ double exp_poly(double x)
{
    constexpr double inv[13] = {1.0, 1.0, 1.0 / 2, 1.0 / 6, 1.0 / 24, 1.0 / 120, 1.0 / 720, 1.0 / 5040,
                                1.0 / 40320, 1.0 / 362880, 1.0 / 3628800, 1.0 / 39916800, 1.0 / 479001600};
    double p = inv[DEG];
    #pragma unroll
    for (int k = DEG - 1; k >= 0; --k) p = fma(p, x, inv[k]);
    return p;
}

// The tile of a block: blocks go round-robin over the 8 XCDs, so XCD q takes the q-th eighth of the
// tiles in order.  Consecutive tiles (the cell blocks of one group block) then run on one XCD and
// read that group block's lines from its L2 once.
__device__ __forceinline__ uint32_t xcd_tile()
{
    const uint32_t n = gridDim.x, b = blockIdx.x, q = b & 7u, per = n >> 3, rest = n & 7u;
    return q * per + (q < rest ? q : rest) + (b >> 3);
}

// Bring lines [a, b) (the first 512) into L2: a wave reads them one trip after the other with scalar
// loads, each of which would otherwise wait for HBM.  One 4-byte read per 128-byte line; the
// caller consumes the result once it has waited for something else.
__device__ __forceinline__ uint32_t touch_lines(const Line64 *lines, int a, int b, int lane)
{
    const int l0 = a + lane * 4, l1 = l0 + 256;
    const uint32_t v0 = l0 < b ? lines[l0].k1 : 0u, v1 = l1 < b ? lines[l1].k1 : 0u;
    return v0 | v1;
}

// one row's entry of the lane, from the lane's column and a byte offset
__device__ __forceinline__ double row_at(const double *column, uint32_t offset)
{
    return *reinterpret_cast<const double *>(reinterpret_cast<const char *>(column) + offset);
}

// the entries of a line's cell tables times its polynomial; e_lane: the lane's column of the tables
template <int DEG>
__device__ __forceinline__ double line_exp(const Line64 &q, const double *e_lane, double nh)
{
    return row_at(e_lane, q.k1) * row_at(e_lane, q.k2) * exp_poly<DEG>(q.r * nh);
}

// The NLTE species' lines of group g in cell ic (physical_opacity_nlte.f:304-345): absorption with
// stimulated emission from the populations and emission, bnu the group centre's Planck function
__device__ __forceinline__ void nlte_lines(const NlteOut &q, int g, int ic, int nc, double phi, double bnu,
                                           double &cap, double &cape, double &em)
{
#pragma clang fp contract(off)
    const double fconst = PC_PI * (PC_E * PC_E) / (PC_ME * PC_C);
    const double nd = q.ndens[2 * (size_t)ic], *pop = q.popT + ic;
    for (int h = q.hstart[g]; h < q.hstart[g + 1]; ++h) {
        const HLine r = q.hline[h];                     // uniform: scalar loads
        const double npl = pop[(size_t)r.lw * nc] * nd;
        const double npu = pop[(size_t)r.lu * nc] * nd;
        cap += npl * fconst * r.f * phi * (1.0 - (npu * r.gl / (npl * r.gu)));
        const double emithelp = npu * r.aul * phi * PC_H * PC_C / (4.0 * PC_PI * (r.wl0 * PC_ANG));
        cape += emithelp / bnu;
        em += emithelp;
    }
}

// physical_opacity.f:228-243: sum over elements of g_ff(u, gamma^2) z^2 natomfr for cell ic at
// the u coordinate (iu, du). The bilinear g_ff is linear in the table rows of u, so the
// elements whose gamma^2 coordinate lies inside the table are folded into the cell's row
// ffB (built each opacity build by k_ff_table), leaving two loads per (cell, group). Elements
// past the table (bit set in ffclamp) keep the per-group evaluation with g_ff >= 1.
__device__ inline double ff_gaunt_sum(const Dev &d, int ic, int iu, double du,
                                      const double *__restrict__ rgg_tab)
{
    const int nc = d.nx;
    const double *B = d.ffB + ic;                 // node-major: B[j * nc]
    double s = (1.0 - du) * B[(size_t)(iu - 1) * nc] + du * B[(size_t)iu * nc];
    for (uint32_t m = d.ffclamp[ic]; m != 0u; m &= m - 1u) {
        const int k = __builtin_ctz(m);
        const int z = d.el_z[k];
        const double rgg = rgg_tab[(size_t)k * nc + ic];
        int igg = (int)floor(rgg);
        igg = igg < 1 ? 1 : (igg > FF_NGG - 1 ? FF_NGG - 1 : igg);
        const double dgg = rgg - igg;
        const double *T = d.gff;
        double gff = (1.0 - du) * (1.0 - dgg) * T[(igg - 1) * FF_NU + (iu - 1)] +
                     du * (1.0 - dgg) * T[(igg - 1) * FF_NU + iu] +
                     (1.0 - du) * dgg * T[igg * FF_NU + (iu - 1)] +
                     du * dgg * T[igg * FF_NU + iu];
        gff = gff > 1.0 ? gff : 1.0;
        s += gff * (double)(z * z) * d.natomfr[(size_t)ic * 30 + (z - 1)];
    }
    return s;
}

}  // namespace slgpu
