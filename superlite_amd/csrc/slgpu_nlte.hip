// NLTE hydrogen opacity on gfx950 (GAS/physical_opacity_nlte.f:3-708 with nlte_nelem = 1).
//
//   k_nlte_pop     one block per massive cell: the H I rate coefficients (radiative with J
//                  at the group centre, :160-184; electron-impact excitation, :189-222), the
//                  photoionisation and recombination rates (:226-253), the rate matrix
//                  (:255-266), its LU with partial pivoting (LAPACK dgetf2's unblocked
//                  algorithm) and the two substitutions of dgetrs; the normalised level
//                  populations
//   k_opacity_nlte (k_opacity64 with its NLTE form where the cells' exponential tables hold)
//                  one thread per (cell, group), 64 cells x 4 groups per block: the H lines
//                  of the group in the file's order (NLTE absorption with stimulated emission
//                  from the populations, :304-345), the other elements' lines in LTE
//                  (:349-401), bf (:413-452) and ff (:458-511), each added to cap, capemit and
//                  emiss as the reference adds them
//   k_nlte_finish  transpose to the (nc, ng) outputs; k_nlte_means the Planck mean of capemit
//                  (opacity_planckmean.f:22)
//   k_nlte_rad_est the radiation temperature and intensity estimates after the transport
//                  (nltemod.f:231-260)
//
// The reference inverts the rate matrix (dgetrf + dgetri) and multiplies; the populations
// here solve the same system with the same factorisation.  The arithmetic is FP64 in both
// precision forms, without fused multiply-add contraction except where the factorisation
// writes it explicitly (as the oracle does).
#include <float.h>

#include <type_traits>

#include "slgpu_device.h"
#include "slgpu_internal.h"

#pragma clang fp contract(off)

namespace slgpu {

constexpr double KB_EV = PC_KB / PC_EV;
constexpr int NLTE_THREADS = 512;

__device__ __forceinline__ double lane_value(double v, int lane)
{
    const long long u = __double_as_longlong(v);
    const unsigned lo = __builtin_amdgcn_readlane((int)(unsigned)u, lane);
    const unsigned hi = __builtin_amdgcn_readlane((int)(u >> 32), lane);
    return __longlong_as_double((long long)(((unsigned long long)hi << 32) | lo));
}

// largest value of a wave, in every lane (NaN lanes do not count)
__device__ __forceinline__ double wave_max(double v)
{
    auto with = [](double x, auto ctrl) {
        const long long u = __double_as_longlong(x);
        const unsigned lo = __builtin_amdgcn_update_dpp(0, (int)(unsigned)u, decltype(ctrl)::value, 0xf, 0xf, false);
        const unsigned hi = __builtin_amdgcn_update_dpp(0, (int)(u >> 32), decltype(ctrl)::value, 0xf, 0xf, false);
        return fmax(x, __longlong_as_double((long long)(((unsigned long long)hi << 32) | lo)));
    };
    v = with(v, std::integral_constant<int, 0x121>());   // row_ror 1, 2, 4, 8: the 16 lanes of a row
    v = with(v, std::integral_constant<int, 0x122>());
    v = with(v, std::integral_constant<int, 0x124>());
    v = with(v, std::integral_constant<int, 0x128>());
    return fmax(fmax(lane_value(v, 0), lane_value(v, 16)), fmax(lane_value(v, 32), lane_value(v, 48)));
}

// One block per massive cell: rates, rate matrix, LU with partial pivoting and the populations.
// NCH > 0: the matrix (n x n, column-major, the right-hand side as column n) lives in LDS and a lane
// holds the rows lane + 64 c, c < NCH; NCH = 0: it lives in the cell's slot of q.A.
//
// The factorisation is n dependent steps of one barrier each, so it is bound by their latency.  Every
// wave finds the pivot of column j for itself (a wave maximum and a ballot), and swaps row jp into
// place while it updates its columns, so that a step needs no barrier of its own for the search, the
// swap or the scaling; the right-hand side takes the steps with the columns, so no row permutation
// is kept and L is not stored.  Each element sees the operations of dgetf2 and dgetrs in their order.
// 400 cells of 100 levels: 0.29 ms with the rates, two blocks of 82 KB on a CU; 2.87 ms as two
// kernels on a matrix in memory, five barriers a step and the substitutions in one thread.
template <int NCH>
__global__ __launch_bounds__(NLTE_THREADS) void k_nlte_pop(Dev d, NlteDev q)
{
    extern __shared__ __align__(16) double s_mem[];
    const int i = blockIdx.x, n = q.n, t = threadIdx.x;
    const int lane = t & 63, wave = __builtin_amdgcn_readfirstlane(t >> 6);
    constexpr int NW = NLTE_THREADS / 64;
    double *pop = q.pop + (size_t)i * n, *popT = q.popT + i;
    if (!(d.mass[i] > 0.0)) {                             // uniform per block: no populations
        for (int k = t; k < n; k += NLTE_THREADS) {
            pop[k] = 0.0;
            popT[(size_t)k * d.nx] = 0.0;
        }
        return;
    }
    double *a = NCH > 0 ? s_mem : q.A + (size_t)i * n * (n + 1);
    double *diag = NCH > 0 ? s_mem + n * (n + 1) : s_mem;  // photoionisation rates, then the pivots
    double *b = a + (size_t)n * n;
    for (int k = t; k < n * n; k += NLTE_THREADS) a[k] = 0.0;
    for (int k = t; k < n; k += NLTE_THREADS) b[k] = k == 0 ? 1.0 : 0.0;
    __syncthreads();
    const double T = d.temp[i], tempinv = 1.0 / T;
    // radiative: rc(llw, lup) = Blu J, rc(lup, llw) = Aul + Bul J; the level pairs are
    // distinct (slgpu_set_nlte_data checks), so the assignments do not race.  The rate matrix holds
    // rc(ll, l) in row l, column ll: rc is stored by rows
    for (int il = t; il < q.nlin; il += NLTE_THREADS) {
        const int g = q.igs[il];
        if (g < 1) continue;
        const double wlm = 0.5 * (d.wl[g] + d.wl[g - 1]);
        const double jnu = (wlm * wlm / PC_C) * planck(wlm, T);
        const int lw = q.llw[il] - 1, lu = q.lup[il] - 1;
        a[(size_t)lw * n + lu] = q.blu[il] * jnu;
        a[(size_t)lu * n + lw] = q.aul[il] + q.bul[il] * jnu;
    }
    __syncthreads();
    // electron-impact excitation and de-excitation (distinct pairs as well)
    const double tp = pow(tempinv, 1.5), kp = pow(KB_EV, 1.5);
    for (int il = t; il < q.ncoll; il += NLTE_THREADS) {
        const double x = q.dele[il] * tempinv / KB_EV;
        const double lx = log(x);
        const double *c = q.cc + 4 * (size_t)il;
        double f = c[0] + c[1] * lx + c[2] * (lx * lx) + c[3] * (lx * lx * lx);
        f = exp(f);
        const double gamma = 1.58e-5 * (f / x) * exp(-1.0 * x) * tp / kp;
        const int lw = q.cl[il], lu = q.cu[il];
        const double gamma_d = q.glev[lw - 1] * gamma * exp(x) / q.glev[lu - 1];
        const double clu = gamma * d.nelec_in[i] * d.natom_in[i] / d.vol_in[i];
        const double cul = gamma_d * d.nelec_in[i] * d.natom_in[i] / d.vol_in[i];
        double *up = a + (size_t)(lw - 1) * n + (lu - 1), *down = a + (size_t)(lu - 1) * n + (lw - 1);
        *up = *up + clu;
        *down = *down + cul;
    }
    // photoionisation and radiative recombination (each level once)
    for (int ll = t; ll < n; ll += NLTE_THREADS) {
        const int l = q.levpi[ll];
        const double xpi = q.delepi[ll] * tempinv / KB_EV;
        const double lp = log(xpi);
        const double *cp = q.pic + 4 * (size_t)ll, *cr = q.rrc + 4 * (size_t)ll;
        double fpi = cp[0] + cp[1] * lp + cp[2] * (lp * lp) + cp[3] * (lp * lp * lp);
        fpi = exp(fpi);
        diag[l - 1] = (fpi / xpi) * exp(-1.0 * xpi) * tp / kp;
        const double xrr = KB_EV * q.radtemp[i];
        const double lr = log(xrr);
        double frr = cr[0] + cr[1] * lr + cr[2] * (lr * lr) + cr[3] * (lr * lr * lr);
        frr = exp(frr);
        if (l > 1) b[l - 1] = -1.0 * frr * q.ndens[2 * (size_t)i + 1] / q.ndens[2 * (size_t)i];
    }
    __syncthreads();
    // the rate matrix in place: row 1 all ones; on the diagonal of row l > 1 -sum_k rc(l, k) -
    // gamma_PI(l), the sum in index order as the Fortran sum takes it
    for (int r = t; r < n; r += NLTE_THREADS) {
        if (r > 0) {
            double sum = 0.0;
            for (int k = 0; k < n; ++k) sum += a[(size_t)r * n + k];
            double v = -1.0 * sum;
            a[(size_t)r * n + r] = v - diag[r];
        }
        a[(size_t)r * n] = 1.0;
    }
    __syncthreads();
    const int nch = NCH > 0 ? NCH : (n + 63) / 64;
    constexpr int NC = NCH > 0 ? NCH : 1;
    for (int j = 0; j < n; ++j) {
        const double *cj = a + (size_t)j * n;
        // idamax over rows j..n-1: the first largest |a|
        double v[NC], best = -1.0;
        if constexpr (NCH > 0) {
            #pragma unroll
            for (int c = 0; c < NCH; ++c) {
                const int r = lane + 64 * c;
                v[c] = r >= j && r < n ? cj[r] : __builtin_nan("");
                best = fmax(best, fabs(v[c]));
            }
        } else {
            for (int r = lane; r < n; r += 64)
                if (r >= j) best = fmax(best, fabs(cj[r]));
        }
        best = wave_max(best);
        int jp = j;
        if constexpr (NCH > 0) {
            #pragma unroll
            for (int c = NCH - 1; c >= 0; --c) {
                const uint64_t m = __ballot(fabs(v[c]) == best);
                if (m) jp = 64 * c + __builtin_ctzll(m);
            }
        } else {
            for (int c = nch - 1; c >= 0; --c) {
                const int r = lane + 64 * c;
                const uint64_t m = __ballot(r >= j && r < n && fabs(cj[r]) == best);
                if (m) jp = 64 * c + __builtin_ctzll(m);
            }
        }
        const double ajj = cj[j], piv = cj[jp];
        if (!(piv != 0.0)) {                              // the same in every wave
            if (t == 0) atomicOr(q.flag, 1);
            return;
        }
        if (t == 0) diag[j] = piv;
        const bool recip = fabs(piv) >= DBL_MIN;
        const double rcp = 1.0 / piv;
        auto scaled = [&](double x) { return recip ? x * rcp : x / piv; };
        if constexpr (NCH > 0) {
            double l[NCH];
            #pragma unroll
            for (int c = 0; c < NCH; ++c) l[c] = -scaled(lane + 64 * c == jp ? ajj : v[c]);
            constexpr int KB = 4;                         // columns whose reads are in flight together
            for (int k0 = j + 1 + wave; k0 <= n; k0 += KB * NW) {
                double ajk[KB], u[KB], o[KB][NCH];
                #pragma unroll
                for (int m = 0; m < KB; ++m) {
                    const int k = k0 + m * NW;
                    const double *ck = a + (k <= n ? k : n) * n;
                    ajk[m] = ck[j];
                    u[m] = ck[jp];
                    #pragma unroll
                    for (int c = 0; c < NCH; ++c) {
                        const int r = lane + 64 * c;
                        o[m][c] = ck[r < n ? r : n - 1];
                    }
                }
                #pragma unroll
                for (int m = 0; m < KB; ++m) {
                    const int k = k0 + m * NW;
                    if (k > n) break;
                    double *ck = a + k * n;
                    #pragma unroll
                    for (int c = 0; c < NCH; ++c) {
                        const int r = lane + 64 * c;
                        const double old = r == jp ? ajk[m] : o[m][c];
                        const double w = u[m] != 0.0 ? fma(l[c], u[m], old) : old;
                        if (r >= j && r < n) ck[r] = r == j ? u[m] : w;
                    }
                }
            }
        } else {
            for (int k = j + 1 + wave; k <= n; k += NW) {
                double *ck = a + (size_t)k * n;
                const double ajk = ck[j], u = ck[jp];
                for (int r = lane; r < n; r += 64) {
                    if (r < j) continue;
                    const double old = r == jp ? ajk : ck[r];
                    const double l = -scaled(r == jp ? ajj : cj[r]);
                    ck[r] = r == j ? u : (u != 0.0 ? fma(l, u, old) : old);
                }
            }
        }
        __syncthreads();
    }
    // back substitution, column by column
    if constexpr (NCH > 0) {
        if (wave != 0) return;
        double x[NCH];
        #pragma unroll
        for (int c = 0; c < NCH; ++c) x[c] = lane + 64 * c < n ? b[lane + 64 * c] : 0.0;
        #pragma unroll
        for (int c = NCH - 1; c >= 0; --c)
            for (int k = n - 1 < 64 * c + 63 ? n - 1 : 64 * c + 63; k >= 64 * c; --k) {
                const double bk = lane_value(x[c], k & 63);
                if (bk != 0.0) {
                    const double xk = bk / diag[k];
                    #pragma unroll
                    for (int e = 0; e <= c; ++e) {
                        const int r = lane + 64 * e;
                        x[e] = r < k ? fma(-xk, a[k * n + (r < k ? r : 0)], x[e]) : (r == k ? xk : x[e]);
                    }
                }
            }
        #pragma unroll
        for (int c = 0; c < NCH; ++c) {
            const int r = lane + 64 * c;
            if (r < n) {
                pop[r] = x[c];
                popT[(size_t)r * d.nx] = x[c];
            }
        }
    } else {
        for (int k = n - 1; k >= 0; --k) {
            if (t == 0 && b[k] != 0.0) b[k] = b[k] / diag[k];
            __syncthreads();
            const double xk = b[k];
            if (xk != 0.0)
                for (int r = t; r < k; r += NLTE_THREADS) b[r] = fma(-xk, a[(size_t)k * n + r], b[r]);
            __syncthreads();
        }
        for (int r = t; r < n; r += NLTE_THREADS) {
            pop[r] = b[r];
            popT[(size_t)r * d.nx] = b[r];
        }
    }
}

__global__ __launch_bounds__(256) void k_opacity_nlte(Dev d, NlteDev q, int flags, double ffc1,
                                                      const double *__restrict__ rgg_tab)
{
    const int nc = d.nx, ng = d.ng;
    const int lane = threadIdx.x & 63;
    const int i = blockIdx.x * 64 + lane;
    const int g = __builtin_amdgcn_readfirstlane(blockIdx.y * 4 + (threadIdx.x >> 6)) + 1;
    if (g > ng) return;
    const bool act = i < nc;
    const int ic = act ? i : nc - 1;
    const bool massive = act && d.mass[ic] > 0.0;
    const double T = d.temp[ic], hckt = d.hckt[ic];
    const double wlo = d.wl[g - 1], whi = d.wl[g];
    double cap = 0.0, cape = 0.0, em = 0.0;
    if (!(flags & SLGPU_NOBB)) {
        const double wl = 0.5 * (wlo + whi);
        const double dwl = whi - wlo;
        const double phi = wl * wl / (dwl * PC_C);
        const double bnu = (wl * wl / PC_C) * planck(wl, T);
        if (massive) nlte_lines(nlte_out(q), g, ic, nc, phi, bnu, cap, cape, em);
        const double wlinv = 1.0 / wl;
        const double expfac = 1.0 - exp(-hckt * wlinv);
        const double *ocg = d.ocg + ic;
        for (int l = d.gstart[g]; l < d.gstart[g + 1]; ++l) {
            const LineRec r = d.lines[l];                   // uniform: scalar loads
            if (r.ion == q.kH) continue;                    // H I is the NLTE species
            const double o = ocg[(size_t)r.ion * nc];
            if (!(o > 0.0) || !massive) continue;
            const double caphelp = phi * (double)r.gxs * o * exp(-(double)r.chilw * hckt) * expfac;
            cap += caphelp;
            cape += caphelp;
            em += caphelp * bnu;
        }
    }
    const double bnul = (wlo * wlo / PC_C) * planck(wlo, T);     // bf and ff: left edge
    if (!(flags & SLGPU_NOBF) && massive) {
        const double *xs = d.bfxs + (size_t)(g - 1) * d.nion;
        for (int k = 0; k < d.nion; ++k) {
            const double x = xs[k];
            if (x != 0.0) {
                const double v = x * d.ocT[(size_t)k * nc + ic];
                cap += v;
                cape += v;
                em += v * bnul;
            }
        }
    }
    if (!(flags & SLGPU_NOFF) && massive) {
        const double wl = wlo;
        const double u = hckt * (1.0 / wl);
        const double ru = 10.0 * (log10(u) + 4.0) + 1.0;
        int iu = (int)floor(ru);
        iu = iu < 1 ? 1 : (iu > FF_NU - 1 ? FF_NU - 1 : iu);
        const double du = ru - iu;
        const double help = ffc1 * sqrt(hckt) * (1.0 - exp(-u)) * (wl * wl * wl) * d.hlparr[ic];
        const double v = help * ff_gaunt_sum(d, ic, iu, du, rgg_tab);
        cap += v;
        cape += v;
        em += v * bnul;
    }
    if (act) {
        const size_t o = (size_t)(g - 1) * nc + i;
        d.capT[o] = massive ? cap : 0.0;
        q.capemitT[o] = massive ? cape : 0.0;
        q.emissT[o] = massive ? em : 0.0;
    }
}

// (ng, nc) cell-fastest -> (nc, ng) group-fastest for cap, capemit and emiss
__global__ __launch_bounds__(256) void k_nlte_finish(Dev d, NlteDev q, int want64)
{
    __shared__ double t0[32][33], t1[32][33], t2[32][33];
    const int nc = d.nx, ng = d.ng;
    const int g0 = blockIdx.x * 32, i0 = blockIdx.y * 32;
    const int tx = threadIdx.x & 31, ty = threadIdx.x >> 5;
    for (int r = ty; r < 32; r += 8) {
        const int g = g0 + r, i = i0 + tx;
        const bool in = g < ng && i < nc;
        const size_t o = (size_t)g * nc + i;
        t0[r][tx] = in ? d.capT[o] : 0.0;
        t1[r][tx] = in ? q.capemitT[o] : 0.0;
        t2[r][tx] = in ? q.emissT[o] : 0.0;
    }
    __syncthreads();
    for (int r = ty; r < 32; r += 8) {
        const int i = i0 + r, g = g0 + tx;
        if (i < nc && g < ng) {
            const size_t o = (size_t)i * ng + g;
            if (want64) d.cap64[o] = t0[tx][r];
            d.cap32[o] = (float)t0[tx][r];
            q.capemit32[o] = (float)t1[tx][r];
            d.emiss[o] = (float)t2[tx][r];
        }
    }
}

// Planck mean of the FP32 capemit with the specarr of k_cell_tables, in its reduction order
__global__ __launch_bounds__(256) void k_nlte_means(Dev d, NlteDev q)
{
    __shared__ double sh[4];
    const int i = blockIdx.x, ng = d.ng;
    double pe = 0.0;
    for (int g = threadIdx.x + 1; g <= ng; g += 256)
        pe += (double)q.capemit32[(size_t)i * ng + g - 1] * d.specarr[(size_t)i * ng + g - 1];
    pe = block_sum256(pe, sh);
    if (threadIdx.x == 0) q.capemitgrey[i] = pe;
}

// nlte_rad_est (nltemod.f:231-260) after the transport: the radiation temperature estimate
// (tally/(a V))^(1/4) from the census energy tally, damped by one half, and the group-centre
// intensity wlm^2 B(wlm, radtemp)/c at the new radiation temperature; one block per cell
__global__ __launch_bounds__(256) void k_nlte_rad_est(Dev d, double *radtemp, double *jrad)
{
    __shared__ double s_tr;
    const int i = blockIdx.x, ng = d.ng;
    if (threadIdx.x == 0) {
        const double trad = pow(d.tally[i] / (PC_ACOEF * d.vol[i]), 0.25);
        const double r = radtemp[i];
        const double rn = r + 0.5 * (trad - r);
        radtemp[i] = rn;
        s_tr = rn;
    }
    __syncthreads();
    if (!jrad) return;
    const double tr = s_tr;
    for (int g = threadIdx.x + 1; g <= ng; g += 256) {
        const double wlm = 0.5 * (d.wl[g] + d.wl[g - 1]);
        jrad[(size_t)i * ng + g - 1] = wlm * wlm * planck(wlm, tr) / PC_C;
    }
}

void launch_nlte_rad_est(slgpu_ctx *c, double *radtemp, double *jrad)
{
    hipLaunchKernelGGL(k_nlte_rad_est, dim3(c->nx), dim3(256), 0, c->stream, c->d, radtemp, jrad);
}

// The matrix, its right-hand side and the pivots fit the CU's 160 KiB of LDS up to 142 levels; larger
// atoms keep them in memory, where every column update waits on L2.
bool nlte_in_lds(int n) { return ((size_t)n * (n + 2) + 2) * sizeof(double) <= 163840; }

static void launch_nlte_pop(slgpu_ctx *c)
{
    const NlteDev &q = c->nl;
    const dim3 grid(c->nx), block(NLTE_THREADS);
    if (!nlte_in_lds(q.n)) {
        hipLaunchKernelGGL((k_nlte_pop<0>), grid, block, q.n * sizeof(double), c->stream, c->d, q);
        return;
    }
    const size_t lds = (size_t)q.n * (q.n + 2) * sizeof(double);
    if (q.n <= 64) hipLaunchKernelGGL((k_nlte_pop<1>), grid, block, lds, c->stream, c->d, q);
    else if (q.n <= 128) hipLaunchKernelGGL((k_nlte_pop<2>), grid, block, lds, c->stream, c->d, q);
    else hipLaunchKernelGGL((k_nlte_pop<3>), grid, block, lds, c->stream, c->d, q);
}

void launch_opacity_nlte(slgpu_ctx *c, int flags, double ffc1, const double *rgg)
{
    const NlteDev &q = c->nl;
    if (!(flags & SLGPU_NOBB)) {
        launch_nlte_pop(c);
    }
    if (!launch_opacity64_nlte(c, flags, ffc1, rgg)) {
        dim3 grid((c->nx + 63) / 64, (c->ng + 3) / 4);
        hipLaunchKernelGGL(k_opacity_nlte, grid, dim3(256), 0, c->stream, c->d, q, flags, ffc1, rgg);
    }
    dim3 tg((c->ng + 31) / 32, (c->nx + 31) / 32);
    hipLaunchKernelGGL(k_nlte_finish, tg, dim3(256), 0, c->stream, c->d, q, 1);
}

void launch_nlte_means(slgpu_ctx *c)
{
    hipLaunchKernelGGL(k_nlte_means, dim3(c->nx), dim3(256), 0, c->stream, c->d, c->nl);
}

}  // namespace slgpu
