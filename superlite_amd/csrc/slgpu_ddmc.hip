// DDMC preparation on gfx950: lumped leakage opacities (GRID/leakage_opacity11.f90:30-171),
// binned emission probabilities (GRID/emission_probability.f90:39-62), and the per-cell
// sampling tables that replace the reference's per-event O(ng) linear scans
// (GRID/emitgroup.f:23-51, TRANSPORT1/diffusion11.f90:289-313, 375-398, 447-460,
// 489-511, 571-584; SOURCE/interior_source.f90:96-103) by cumulative rows plus exact
// bucket maps (slgpu_sample.h), so a sampled group usually costs one table load.  Per cell:
// lumped sums and lump order (k_leakage), the rows' terms (k_row_terms), emission bins and source
// totals (k_emitprob), the rows' running sums (k_row_sums), the bucket maps (k_bucket_tables; few
// cells: k_bucket_search).
#include "slgpu_device.h"
#include "slgpu_internal.h"
#include "slgpu_sample.h"

namespace slgpu {

constexpr int NT = 1024;
constexpr int NW = NT / 64;

// inclusive block scan (fixed order) returning the block total through `total`
__device__ __forceinline__ double block_scan(double v, double *sh, double &total)
{
    const int w = threadIdx.x >> 6, lane = threadIdx.x & 63;
    double x = wave_inclusive_scan(v);
    if (lane == 63) sh[w] = x;
    __syncthreads();
    if (w == 0) {
        double t = lane < NW ? sh[lane] : 0.0;
        t = wave_inclusive_scan(t);
        if (lane < NW) sh[lane] = t;
    }
    __syncthreads();
    double off = w > 0 ? sh[w - 1] : 0.0;
    total = sh[NW - 1];
    __syncthreads();
    return x + off;
}

__device__ __forceinline__ int block_scan_int(int v, int *sh, int &total)
{
    const int w = threadIdx.x >> 6, lane = threadIdx.x & 63;
    int x = v;
    #pragma unroll
    for (int off = 1; off < 64; off <<= 1) {
        int t = __shfl_up(x, off, 64);
        if (lane >= off) x += t;
    }
    if (lane == 63) sh[w] = x;
    __syncthreads();
    if (w == 0) {
        int t = lane < NW ? sh[lane] : 0;
        #pragma unroll
        for (int off = 1; off < 64; off <<= 1) {
            int u = __shfl_up(t, off, 64);
            if (lane >= off) t += u;
        }
        if (lane < NW) sh[lane] = t;
    }
    __syncthreads();
    int off = w > 0 ? sh[w - 1] : 0;
    total = sh[NW - 1];
    __syncthreads();
    return x + off;
}

__device__ __forceinline__ double block_sum(double v, double *sh)
{
    double t;
    block_scan(v, sh, t);
    return t;
}

#define CAPC(ig, ic) ((double)d.cap32[(size_t)((ic) - 1) * ng + ((ig) - 1)])
// emission opacity: grd_capemit after an NLTE build, grd_cap after an LTE one
#define CAPE(ig, ic) ((double)d.capem32[(size_t)((ic) - 1) * ng + ((ig) - 1)])
#define XA(i) (d.xarr[(i) - 1])
#define DX(i) (d.xarr[(i)] - d.xarr[(i) - 1])
#define DX3(i) (d.xarr[(i)] * d.xarr[(i)] * d.xarr[(i)] - d.xarr[(i) - 1] * d.xarr[(i) - 1] * d.xarr[(i) - 1])
#define SIGC(ic) (d.sig[(ic) - 1])

// resolved leakage opacity of group g through the left (side<0) or right face of cell ix
// (diffusion11.f90:204-239, 383-395, 455-457, 496-508)
__device__ __forceinline__ double resleak(const Dev &d, int ix, int g, int side)
{
    const int ng = d.ng, ic = ix;
    if (side < 0) {
        const int l = ix - 1;
        if ((CAPC(g, l) + SIGC(l)) * DX(ix - 1) < d.tauddmc) {
            double mfp = (CAPC(g, ic) + SIGC(ic)) * DX(ix);
            double ppl = 4.0 / (3.0 * mfp + 6.0 * PC_DEXT);
            return 1.5 * ppl * (XA(ix) * XA(ix)) / DX3(ix);
        }
        double mfp = (SIGC(ic) + CAPC(g, ic)) * DX(ix) + (SIGC(l) + CAPC(g, l)) * DX(ix - 1);
        return 2.0 * (XA(ix) * XA(ix)) / (mfp * DX3(ix));
    }
    if (ix == d.nx) {
        double mfp = (CAPC(g, ic) + SIGC(ic)) * DX(ix);
        double ppr = 4.0 / (3.0 * mfp + 6.0 * PC_DEXT);
        return 1.5 * ppr * (XA(ix + 1) * XA(ix + 1)) / DX3(ix);
    }
    const int l = ix + 1;
    if ((CAPC(g, l) + SIGC(l)) * DX(ix + 1) < d.tauddmc) {
        double mfp = (CAPC(g, ic) + SIGC(ic)) * DX(ix);
        double ppr = 4.0 / (3.0 * mfp + 6.0 * PC_DEXT);
        return 1.5 * ppr * (XA(ix + 1) * XA(ix + 1)) / DX3(ix);
    }
    double mfp = (SIGC(ic) + CAPC(g, ic)) * DX(ix) + (SIGC(l) + CAPC(g, l)) * DX(ix + 1);
    return 2.0 * (XA(ix + 1) * XA(ix + 1)) / (mfp * DX3(ix));
}

// first index of the block's maximum of (v, k) pairs, k = 0 meaning none (the strict '>' of
// an ascending loop): the result is valid on thread 0
__device__ __forceinline__ void block_argmax_first(double &v, int &k, double *s_v, int *s_k)
{
    for (int off = 32; off > 0; off >>= 1) {
        double v2 = __shfl_xor(v, off, 64);
        int k2 = __shfl_xor(k, off, 64);
        if (v2 > v || (v2 == v && k2 != 0 && (k == 0 || k2 < k))) { v = v2; k = k2; }
    }
    const int w = threadIdx.x >> 6;
    if ((threadIdx.x & 63) == 0) { s_v[w] = v; s_k[w] = k; }
    __syncthreads();
    if (threadIdx.x == 0) {
        double bv = 0.0;
        int bk = 0;
        for (int q = 0; q < NW; ++q)
            if (s_v[q] > bv || (s_v[q] == bv && s_k[q] != 0 && (bk == 0 || s_k[q] < bk))) {
                bv = s_v[q]; bk = s_k[q];
            }
        v = bv;
        k = bk;
    }
    __syncthreads();
}

__global__ __launch_bounds__(NT) __attribute__((amdgpu_waves_per_eu(8, 8))) void k_leakage(Dev d)
{
    __shared__ double shd[NW];
    __shared__ int shi[NW];
    __shared__ double s_emax[NW];
    __shared__ int s_imax[NW];
    __shared__ __align__(16) int s_cnt[2][NW];
    const int ng = d.ng, nx = d.nx;
    const int i = blockIdx.x + 1, l = i;
    const int icnb1 = i - 1 < 1 ? 1 : i - 1, icnb2 = i + 1 > nx ? nx : i + 1;
    const double dist = DX(i);
    const double tinv = d.tempinv[l - 1];
    const double sg = SIGC(l);
    const double *spec = d.specarr + (size_t)(l - 1) * ng;
    const double divv = d.divv[l - 1];
    // pass 1: speclump and the lump size (leakage_opacity11.f90:52-59)
    double sl = 0.0;
    int nl = 0;
    for (int g = threadIdx.x + 1; g <= ng; g += NT) {
        const double c = CAPC(g, l);
        if (c * dist >= d.taulump && (sg + c) * dist >= d.tauddmc) { sl += spec[g - 1]; nl++; }
    }
    sl = block_sum(sl, shd);
    int nlump;
    block_scan_int(nl, shi, nlump);
    const double speclump = sl > 0.0 ? 1.0 / sl : 0.0;
    // pass 2: caplump, capemitlump (NLTE), igemitmax, doplump, leakage opacities (:61-168)
    double caplump = 0.0, capemitlump = 0.0, doplump = 0.0, o1 = 0.0, o2 = 0.0, emax = 0.0, emax2 = 0.0;
    int imax = 0, imax2 = 0;
    const double dvol = 3.0 * d.vol[l - 1] / PC_PI4;
    for (int g = threadIdx.x + 1; g <= ng; g += NT) {
        const double c = CAPC(g, l);
        const bool lump = !(c * dist < d.taulump) && !((sg + c) * dist < d.tauddmc);
        if (lump) {
            const double h = spec[g - 1] * c;
            caplump += h;
            if (h > emax) { emax = h; imax = g; }
            if (d.nlte) {
                const double he = spec[g - 1] * CAPE(g, l);
                capemitlump += he;
                if (he > emax2) { emax2 = he; imax2 = g; }
            }
            const double specval = spec[g - 1];
            bool lh = (i == 1) ? true : ((CAPC(g, icnb1) + SIGC(icnb1)) * DX(i - 1) < d.tauddmc);
            if (lh) {
                double help = (c + sg) * DX(i);
                double ppl = 4.0 / (3.0 * help + 6.0 * PC_DEXT);
                o1 += (specval * speclump) * 1.5 * ppl * (XA(i) * XA(i)) / dvol;
            } else {
                double help = (sg + c) * DX(i) + (SIGC(icnb1) + CAPC(g, icnb1)) * DX(i - 1);
                o1 += (specval * speclump) * 2.0 * (XA(i) * XA(i)) / (help * 3.0 * d.vol[l - 1] / PC_PI4);
            }
            lh = (i == nx) ? true : ((CAPC(g, icnb2) + SIGC(icnb2)) * DX(i + 1) < d.tauddmc);
            if (lh) {
                double help = (c + sg) * DX(i);
                double ppr = 4.0 / (3.0 * help + 6.0 * PC_DEXT);
                o2 += (specval * speclump) * 1.5 * ppr * (XA(i + 1) * XA(i + 1)) / dvol;
            } else {
                double help = (sg + c) * DX(i) + (SIGC(icnb2) + CAPC(g, icnb2)) * DX(i + 1);
                o2 += (specval * speclump) * 2.0 * (XA(i + 1) * XA(i + 1)) / (help * 3.0 * d.vol[l - 1] / PC_PI4);
            }
            if (divv >= 0) {
                if (g <= ng - 1 && !(CAPC(g + 1, l) * dist >= d.taulump))
                    doplump += dopspeccalc(tinv, d.wlinv, g) * divv / (3 * PC_C);
            } else {
                if (g >= 2 && !(CAPC(g - 1, l) * dist >= d.taulump))
                    doplump -= dopspeccalc(tinv, d.wlinv, g - 1) * divv / (3 * PC_C);
            }
        }
    }
    caplump = block_sum(caplump, shd);
    doplump = block_sum(doplump, shd);
    o1 = block_sum(o1, shd);
    o2 = block_sum(o2, shd);
    // igemitmax: first index of the maximum (strict '>' in the reference's ascending loop);
    // in NLTE the capemit loop continues from the cap loop's maximum, so its first maximum
    // wins only where it is strictly larger
    block_argmax_first(emax, imax, s_emax, s_imax);
    if (d.nlte) {
        capemitlump = block_sum(capemitlump, shd);
        block_argmax_first(emax2, imax2, s_emax, s_imax);
        if (emax2 > emax) imax = imax2;
    }
    double *op = d.opaclump + (size_t)(l - 1) * 11;
    const double capgrey = d.capgrey[l - 1];
    // capgreyinv (LTE) or capemitgreyinv (NLTE), diffusion11.f90:98-99
    double cgi = 1.0 / d.capemgrey[l - 1];
    if (!(cgi >= 0.0)) cgi = 0.0;
    const int nl_eff = speclump == 0.0 ? 0 : nlump;
    double c_emitlump, c_caplump, c_doplump;
    if (nl_eff == ng) {
        c_emitlump = 1.0; c_caplump = capgrey; c_doplump = 0.0;
    } else {
        c_caplump = caplump * speclump;
        double el = (d.nlte ? capemitlump : caplump) * cgi;     // diffusion11.f90:136-141
        c_emitlump = el < 1.0 ? el : 1.0;
        c_doplump = doplump * speclump;
    }
    if (threadIdx.x == 0) {
        op[0] = o1; op[1] = o2; op[2] = 0.0; op[3] = 0.0; op[4] = 0.0; op[5] = 0.0;
        op[6] = speclump; op[7] = caplump; op[8] = d.nlte ? capemitlump : 0.0;
        op[9] = (double)imax; op[10] = doplump;
        CellDDMC cc;
        cc.emgreyinv = cgi; cc.speclump = speclump; cc.emitlump = c_emitlump;
        cc.caplump = c_caplump; cc.doplump = c_doplump; cc.nlump = nl_eff; cc.pad = 0;
        d.cell[l - 1] = cc;
    }
    if (nl_eff == 0) return;

    // pass 3: lump order.  Ballots count within a wave, the waves' counts meet in LDS (two sets that
    // take turns, one barrier per 1024 groups), and unlumped places follow from the lumped ones.
    int *gorder = d.gorder + (size_t)(l - 1) * ng;
    const int w = threadIdx.x >> 6, lane = threadIdx.x & 63;
    int base = 0;                                  // lumped groups so far
    for (int g0 = 0; g0 < ng; g0 += NT) {
        const int g = g0 + threadIdx.x + 1;
        bool lump = false;
        if (g <= ng) {
            const double c = CAPC(g, l);
            lump = c * dist >= d.taulump && (sg + c) * dist >= d.tauddmc;
        }
        const unsigned long long m = __ballot(lump);
        int *cnt = s_cnt[(g0 / NT) & 1];
        if (lane == 0) cnt[w] = __popcll(m);
        __syncthreads();
        int before = base + __popcll(m & ((1ull << lane) - 1ull)), total = 0;
        #pragma unroll
        for (int k = 0; k < NW; ++k) {
            const int v = cnt[k];
            before += k < w ? v : 0;
            total += v;
        }
        if (g <= ng) gorder[lump ? before : nl_eff + (g - 1 - before)] = g;
        base += total;
    }
}

// The terms of the running sums, one thread per (cell, position): the four lumped rows', in the order
// k_leakage left, and the source spectrum's (interior_source.f90:69-75).  At the end of k_leakage
// they had its 400 blocks alone, which leave half of the CUs half empty, and its register limit:
// 400 x 10^4, both and the source terms 153 us together, 103 + 49 us so, the preparation 644 -> 625 us.
__global__ __launch_bounds__(256) void k_row_terms(Dev d)
{
    const int ng = d.ng, nx = d.nx;
    const int p = blockIdx.x * 256 + threadIdx.x, i = blockIdx.y + 1, l = i;
    if (p >= ng) return;
    const size_t row = (size_t)(l - 1) * ng;
    d.srccum[row + p] = specintv_g(1.0 / d.radtemp[l - 1], d.wlinv, p + 1);
    const CellDDMC cc = d.cell[l - 1];
    if (cc.nlump == 0) return;
    const int g = d.gorder[row + p];
    const double *spec = d.specarr + row;
    if (p >= cc.nlump) {
        const double d2s = 1.0 / (1.0 - cc.emitlump);
        d.cumS[row + p] = spec[g - 1] * CAPE(g, l) * cc.emgreyinv * d2s;     // diffusion11.f90:574-581
        return;
    }
    // a face or Doppler channel with zero total opacity is never chosen (its event
    // probability is 0); its row is kept finite (all zero) so every row is monotone
    const double o1 = d.opaclump[(size_t)(l - 1) * 11], o2 = d.opaclump[(size_t)(l - 1) * 11 + 1];
    const double hL = o1 > 0.0 ? 1.0 / o1 : 0.0, hR = o2 > 0.0 ? 1.0 / o2 : 0.0;
    const double hD = cc.doplump > 0.0 ? 1.0 / cc.doplump : 0.0;
    const double dist = DX(i), tinv = d.tempinv[l - 1], divv = d.divv[l - 1], speclump = cc.speclump;
    // the Doppler scan runs ascending for redshift, descending for blueshift
    const int gd = divv >= 0 ? g : d.gorder[row + cc.nlump - 1 - p];
    const double sp = spec[g - 1];
    double tD = 0.0;
    d.cumL[row + p] = i > 1 ? sp * resleak(d, i, g, -1) * speclump * hL : 0.0;
    d.cumR[row + p] = sp * resleak(d, i, g, +1) * speclump * hR;
    if (divv >= 0) {
        if (gd != ng && !(CAPC(gd + 1, l) * dist >= d.taulump))
            tD = dopspeccalc(tinv, d.wlinv, gd) * divv / (3 * PC_C) * speclump * hD;
    } else {
        if (gd != 1 && !(CAPC(gd - 1, l) * dist >= d.taulump))
            tD = -(dopspeccalc(tinv, d.wlinv, gd - 1) * divv / (3 * PC_C) * speclump * hD);
    }
    d.cumD[row + p] = tD;
}

// The running sums of the cells' sampling rows (the four lumped rows) and of their source
// spectra, normalised Planck at T_rad (interior_source.f90:69-75, 96-103).  The reference
// accumulates sequentially, and a sequential sum of nonnegative terms is monotone (a parallel
// scan is not, by rounding), which the samplers' searches need.  So each row is one lane's
// chain of additions, 6 clocks each, and the work is to keep everything else off the chain:
//   - an LDS access takes the pipe as long for 1 lane as for 64, so a block takes RS_ROWS rows,
//     one per lane of its first wave (one row per block: 37 ns per value with the chip full);
//   - the other eight waves store the tile before, write the tile after to LDS and request the one
//     after that meanwhile, under barriers that wait for LDS alone (with __syncthreads() a tile
//     took a load's and a store's round trip to memory: the two passes that the source rows had
//     then 0.23 ms instead of 0.16);
//   - the chain's LDS reads run 16 values ahead, in two register sets that take turns.
// The source rows, the longest, start first; their totals come from k_emitprob.  400 x 10^4: 0.85 ms
// for the same chains on global memory, 0.11 ms so (11 ns per value of the longest chain).
constexpr int RS_ROWS = 8, RS_TILE = 256, RS_PITCH = RS_TILE + 2, RS_AHEAD = 16;
constexpr int RS_THREADS = 576, RS_MOVERS = RS_THREADS - 64;
typedef __attribute__((address_space(1))) double *RowPtr;     // not a flat access, which counts as one to LDS too

// A barrier for what the block keeps in LDS.  __syncthreads() also waits for every load and store
// under way to global memory, which the movers' tiles are meant to overlap.
__device__ __forceinline__ void lds_barrier()
{
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}

// s and the running sums of the RS_TILE values of buf from s on, in index order; OUT: the running
// sums replace the values
template <bool OUT>
__device__ __forceinline__ double chain_sum(double *buf, double s)
{
    double v[RS_AHEAD], w[RS_AHEAD];
    #pragma unroll
    for (int k = 0; k < RS_AHEAD; ++k) v[k] = buf[k];
    #pragma unroll 1
    for (int j = 0; j < RS_TILE; j += 2 * RS_AHEAD) {
        #pragma unroll
        for (int k = 0; k < RS_AHEAD; ++k) w[k] = buf[j + RS_AHEAD + k];
        __builtin_amdgcn_sched_barrier(0);
        #pragma unroll
        for (int k = 0; k < RS_AHEAD; ++k) { s = s + v[k]; v[k] = s; }
        #pragma unroll
        for (int k = 0; k < RS_AHEAD; ++k) { if (OUT) buf[j + k] = v[k]; }
        __builtin_amdgcn_sched_barrier(0);
        const int q = j + 2 * RS_AHEAD < RS_TILE ? j + 2 * RS_AHEAD : j;
        #pragma unroll
        for (int k = 0; k < RS_AHEAD; ++k) v[k] = buf[q + k];
        __builtin_amdgcn_sched_barrier(0);
        #pragma unroll
        for (int k = 0; k < RS_AHEAD; ++k) { s = s + w[k]; w[k] = s; }
        #pragma unroll
        for (int k = 0; k < RS_AHEAD; ++k) { if (OUT) buf[j + RS_AHEAD + k] = w[k]; }
        __builtin_amdgcn_sched_barrier(0);
    }
    return s;
}

// For the block's rows r: sums of p[r][0..n[r]) / div[r] in index order, on lane r of the first
// wave; OUT: the running sums replace the row.  nmax: the longest row.
template <bool OUT>
__device__ __forceinline__ double rows_sum(RowPtr const *p, const int *n, const double *div, int nmax,
                                           double (*buf)[RS_ROWS][RS_PITCH])
{
    constexpr int PER = RS_ROWS * RS_TILE / RS_MOVERS;
    const int t = threadIdx.x, lt = t - 64, ntile = (nmax + RS_TILE - 1) / RS_TILE;
    double s = 0.0, v[PER];
    RowPtr row[PER];
    int len[PER];
    double dv[PER];
    if (t >= 64) {
        #pragma unroll
        for (int q = 0; q < PER; ++q) {
            const int e = lt + q * RS_MOVERS, r = e / RS_TILE, k = e % RS_TILE;
            row[q] = p[r] + k;
            len[q] = n[r] - k;
            dv[q] = div[r];
            v[q] = len[q] > 0 ? row[q][0] : 0.0;
        }
    }
    for (int c = -1; c <= ntile; ++c) {
        if (t >= 64) {
            // tile c + 1, requested an iteration ago; then tile c + 2 is
            #pragma unroll
            for (int q = 0; q < PER; ++q) {
                const int e = lt + q * RS_MOVERS, r = e / RS_TILE, k = e % RS_TILE;
                if (c + 1 < ntile) buf[(c + 1) % 3][r][k] = OUT ? v[q] / dv[q] : v[q];
            }
            #pragma unroll
            for (int q = 0; q < PER; ++q) {
                const int o = (c + 2) * RS_TILE;
                v[q] = o < len[q] ? row[q][o] : 0.0;
            }
            #pragma unroll
            for (int q = 0; q < PER; ++q) {
                const int e = lt + q * RS_MOVERS, r = e / RS_TILE, k = e % RS_TILE, o = (c - 1) * RS_TILE;
                if (OUT && c > 0 && o < len[q]) row[q][o] = buf[(c - 1) % 3][r][k];
            }
        } else if (t < RS_ROWS && c >= 0 && c < ntile) {
            s = chain_sum<OUT>(buf[c % 3][t], s);
        }
        lds_barrier();
    }
    return s;
}

__global__ __launch_bounds__(RS_THREADS) void k_row_sums(Dev d)
{
    __shared__ __align__(16) double buf[3][RS_ROWS][RS_PITCH];
    __shared__ RowPtr p[RS_ROWS];
    __shared__ double div[RS_ROWS];
    __shared__ int n[RS_ROWS], s_max;
    const int ng = d.ng, row = (int)blockIdx.y - 1, t = threadIdx.x;
    if (t == 0) s_max = 0;
    __syncthreads();
    if (t < RS_ROWS) {
        const int l = blockIdx.x * RS_ROWS + t, lc = l < d.nx ? l : d.nx - 1;
        const int nl = d.cell[lc].nlump;
        double *base = row < 0 ? d.srccum : (row == 0 ? d.cumL : (row == 1 ? d.cumR : (row == 2 ? d.cumD : d.cumS + nl)));
        int m = row < 0 ? ng : (nl == 0 ? 0 : (row == 3 ? ng - nl : nl));
        if (l >= d.nx) m = 0;
        p[t] = (RowPtr)base + (size_t)lc * ng;
        n[t] = m;
        div[t] = row < 0 ? d.srctot[lc] : 1.0;
        atomicMax(&s_max, m);
    }
    __syncthreads();
    if (s_max == 0) return;
    rows_sum<true>(p, n, div, s_max, buf);
}

// emission_probability.f90:39-62 (grd_capemit, grd_capemitgrey in NLTE) and the in-bin
// cumulative sums emitgroup.f:38-50 walks.  A thread adds up a bin, in order; S: the cell's rows
// pass through LDS both ways, since a wave's bins lie nepg groups apart (400 x 10^4: 87 us with
// the strided global accesses, 53 us so).
// The first blocks add up the source spectra, whose running sums are of the normalised terms: a chain
// as long as k_row_sums' own, which hides behind the bins' blocks here (400 x 10^4: the bins 53 us
// alone and 59 us with them, k_row_sums 162 us with both chains and 111 us with its own).
template <bool S>
__global__ __launch_bounds__(RS_THREADS) void k_emitprob(Dev d)
{
    extern __shared__ __align__(16) double s_spec[];           // ng doubles, then ng floats
    __shared__ double binsum[1024];
    __shared__ double pref[1025];
    __shared__ RowPtr p[RS_ROWS];
    __shared__ int n[RS_ROWS];
    const int ng = d.ng, nep = d.nep, nepg = d.nepg, nsrc = (d.nx + RS_ROWS - 1) / RS_ROWS;
    if ((int)blockIdx.x < nsrc) {
        const int l = blockIdx.x * RS_ROWS + threadIdx.x;
        if (threadIdx.x < RS_ROWS) {
            p[threadIdx.x] = (RowPtr)d.srccum + (size_t)(l < d.nx ? l : d.nx - 1) * ng;
            n[threadIdx.x] = l < d.nx ? ng : 0;
            binsum[threadIdx.x] = 1.0;                         // no divisor
        }
        __syncthreads();
        const double s = rows_sum<false>(p, n, binsum, ng, reinterpret_cast<double (*)[RS_ROWS][RS_PITCH]>(s_spec));
        if (threadIdx.x < RS_ROWS && l < d.nx) d.srctot[l] = s;
        return;
    }
    const int l = blockIdx.x - nsrc + 1;
    const double *spec = d.specarr + (size_t)(l - 1) * ng;
    const float *cap = d.capem32 + (size_t)(l - 1) * ng;
    double *cum = d.emitcum + (size_t)(l - 1) * ng, *out = cum;
    if constexpr (S) {
        float *s_cap = reinterpret_cast<float *>(s_spec + ng);
        for (int g = threadIdx.x; g < ng; g += RS_THREADS) {
            s_spec[g] = spec[g];
            s_cap[g] = cap[g];
        }
        __syncthreads();
        spec = s_spec;
        cap = s_cap;
        out = s_spec;
    }
    for (int b = threadIdx.x; b < nep; b += RS_THREADS) {
        const int g1 = (b + 1) * nepg < ng ? (b + 1) * nepg : ng;
        double s = 0.0;
        for (int g = b * nepg; g < g1; ++g) s = fma(spec[g], (double)cap[g], s);
        binsum[b] = s;
    }
    __syncthreads();
    double *ep = d.emitprob + (size_t)(l - 1) * nep;
    if (threadIdx.x == 0) {
        double help = 0.0;
        pref[0] = 0.0;
        for (int iep = 1; iep <= nep - 1; ++iep) {
            help = help + binsum[iep - 1];
            pref[iep] = help;
        }
    }
    __syncthreads();
    for (int b = threadIdx.x; b < nep; b += RS_THREADS) {
        ep[b] = b < nep - 1 ? pref[b + 1] : d.capemgrey[l - 1];
        const int g1 = (b + 1) * nepg < ng ? (b + 1) * nepg : ng;
        double s = pref[b];
        for (int g = b * nepg; g < g1; ++g) {
            s = fma(spec[g], (double)cap[g], s);
            out[g] = s;
        }
    }
    if constexpr (S) {
        __syncthreads();
        const int n = nep * nepg < ng ? nep * nepg : ng;
        for (int g = threadIdx.x; g < n; g += RS_THREADS) cum[g] = s_spec[g];
    }
}

// first index j in [from, n) with cum[j] > r of a monotone row whose entries before `from` are not:
// steps that double, then a search between the last two
__device__ __forceinline__ int first_above_from(const double *cum, int from, int n, double r)
{
    int lo = from, step = 1;
    while (lo < n && !(cum[lo + step <= n ? lo + step - 1 : n - 1] > r)) {
        lo = lo + step < n ? lo + step : n;
        step <<= 1;
    }
    return lo >= n ? n : first_above(cum, lo, lo + step <= n ? lo + step - 1 : n - 1, r);
}

// inclusive running maximum over the block of both 16-bit halves
__device__ __forceinline__ uint32_t max16(uint32_t a, uint32_t b)
{
    const uint32_t lo = max(a & 0xffffu, b & 0xffffu), hi = max(a >> 16, b >> 16);
    return hi << 16 | lo;
}

__device__ __forceinline__ uint32_t block_scan_max16(uint32_t v, uint32_t *sh)
{
    const int w = threadIdx.x >> 6, lane = threadIdx.x & 63;
    #pragma unroll
    for (int off = 1; off < 64; off <<= 1) {
        const uint32_t u = __shfl_up(v, off, 64);
        if (lane >= off) v = max16(v, u);
    }
    if (lane == 63) sh[w] = v;
    __syncthreads();
    for (int k = 0; k < w; ++k) v = max16(v, sh[k]);
    __syncthreads();
    return v;
}

// place of a bucket's answer in LDS: a thread's stretch of 16 starts on a bank of its own
__device__ __forceinline__ int ans_at(int b) { return b + (b >> 4); }
constexpr size_t BT_ANSWERS = (BT_K + BT_K / 16) * sizeof(uint32_t);

// Exact bucket maps of the five group samplers, one block per (cell, table).
// A lumped row's answers need no search.  The draw at the lower end of bucket b is b/K (K = 2^14),
// that at its upper end the double below (b + 1)/K, and the answer is how many running sums c are
// not above the draw: those with ceil(c K) <= b and with floor(c K) <= b (in the last bucket, whose
// upper end is 1, also c = 1).  c K is exact.  So the last sum of every ceil(c K) writes its count
// there, the last of every floor(c K) likewise, and the answers are running maxima.  A row that does
// not rise throughout (a NaN, see slgpu_sample.h) keeps two searches per bucket.
// The emission table's draws are scaled and rounded first, so it is searched: the row in LDS (S;
// rows past the CU's LDS are searched in global memory), each thread a stretch of 16 buckets,
// whose answers rise, so each search starts from the one before.
// The answers change hands in LDS: the entries are then made in bucket order, where neighbouring lanes
// load the same groups' opacities and store side by side.  400 x 10^4: 640 us with two full
// searches per bucket on global memory, 199 us with searches in LDS that resume, 139 us so;
// the gathers bound it.
template <bool S>
__global__ __launch_bounds__(1024) void k_bucket_tables(Dev d)
{
    extern __shared__ double s_row[];
    constexpr int PER = BT_K / 1024;
    // the emission tables, which take longest, start first
    const int ic = blockIdx.x + 1, t = NTAB - 1 - (int)blockIdx.y, ng = d.ng, nep = d.nep, nepg = d.nepg;
    uint32_t *row = d.btab + ((size_t)t * d.nx + (ic - 1)) * BT_K;
    const bool emit = t == TAB_E;
    const int nlump = d.cell[ic - 1].nlump;
    const LumpRow L = lump_row(d, emit ? TAB_S : t, ic, nlump);
    if (!emit && (nlump == 0 || L.cnt <= 0)) {     // rows of cells without lumping are never sampled
        for (int b = threadIdx.x; b < BT_K; b += 1024) row[b] = 0u;
        return;
    }
    const double *cum = emit ? d.emitcum + (size_t)(ic - 1) * ng : L.cum;
    const double *ep = d.emitprob + (size_t)(ic - 1) * nep;
    const int n = emit ? ng : L.cnt, b0 = threadIdx.x * PER;
    uint32_t *s_ans = reinterpret_cast<uint32_t *>(s_row);
    __shared__ int s_bad;
    __shared__ uint32_t s_max[NW];
    if (threadIdx.x == 0) s_bad = 0;
    if (!emit) {
        #pragma unroll
        for (int k = 0; k < PER; ++k) s_ans[ans_at(threadIdx.x + k * 1024)] = 0u;
    }
    __syncthreads();
    if (emit) {
        // searches that resume need bins whose sums rise, bins that rise and draws that rise
        if (threadIdx.x == 0 && !(d.capemgrey[ic - 1] >= 0.0)) s_bad = 1;
        for (int k = threadIdx.x; k < n; k += 1024) {
            const double v = cum[k];
            if constexpr (S) s_row[k] = v;
            if (!(v >= (k % nepg != 0 ? cum[k - 1] : v))) s_bad = 1;
        }
        for (int k = threadIdx.x; k < nep; k += 1024) {
            const double v = ep[k];
            if constexpr (S) s_row[ng + k] = v;
            if (k < nep - 1 && !(v >= (k > 0 ? ep[k - 1] : v))) s_bad = 1;
        }
        if constexpr (S) {
            cum = s_row;
            ep = s_row + ng;
        }
    } else {
        uint16_t *s_half = reinterpret_cast<uint16_t *>(s_row);      // low half: lower ends, high: upper
        auto bucket = [](double c, bool up) {                          // BT_K: past the last bucket
            const double v = c * (double)BT_K;
            if (!(v > 0.0)) return 0;
            if (v > (double)BT_K) return BT_K;
            const int f = (int)v;
            return up ? f + (v > (double)f) : (f < BT_K ? f : BT_K - 1);
        };
        for (int k = threadIdx.x; k < n; k += 1024) {
            const double v = cum[k], w = k + 1 < n ? cum[k + 1] : INFINITY;
            if (!(v <= w)) s_bad = 1;
            const int cv = bucket(v, true), fv = bucket(v, false);
            if (cv < BT_K && (k + 1 == n || bucket(w, true) != cv)) s_half[2 * ans_at(cv)] = (uint16_t)(k + 1);
            if (fv < BT_K && (k + 1 == n || bucket(w, false) != fv)) s_half[2 * ans_at(fv) + 1] = (uint16_t)(k + 1);
        }
    }
    __syncthreads();
    const bool bad = s_bad != 0;
    uint32_t ans[PER];
    if (emit) {
        // a row that does not rise (a NaN, see slgpu_sample.h; negative line strengths) keeps two
        // searches of the whole row per bucket
        const double cg = d.capemgrey[ic - 1];
        int at = 0;
        #pragma unroll
        for (int k = 0; k < 2 * PER; ++k) {
            const double r1 = (k & 1 ? bt_hi(b0 + k / 2) : bt_lo(b0 + k / 2)) * cg;
            int v;
            if (k == 0 || bad) {
                v = emitgroup_search(d, r1, ep, cum);
            } else {
                // the bin index and the place in the bin resume at the answer before
                int iep = (at - 1) / nepg;
                while (iep < nep - 1 && ep[iep] <= r1) ++iep;
                const int ig = iep * nepg + 1, igp1 = ig + nepg - 1 < ng ? ig + nepg - 1 : ng;
                v = first_above_from(cum, (ig > at ? ig : at) - 1, igp1 - 1, r1) + 1;
            }
            at = v;
            ans[k / 2] = k & 1 ? ans[k / 2] | (uint32_t)v << 15 : (uint32_t)v;
        }
    } else if (bad) {
        #pragma unroll 1
        for (int k = 0; k < PER; ++k) {
            const int b = threadIdx.x + k * 1024;
            const uint32_t lo = (uint32_t)first_above(cum, 0, n, bt_lo(b));
            s_ans[ans_at(b)] = lo | (uint32_t)first_above(cum, 0, n, bt_hi(b)) << 16;
        }
        __syncthreads();
        #pragma unroll
        for (int k = 0; k < PER; ++k) { const uint32_t e = s_ans[ans_at(b0 + k)]; ans[k] = (e & 0xffffu) | e >> 16 << 15; }
    } else {
        uint32_t m = 0u;
        #pragma unroll
        for (int k = 0; k < PER; ++k) { m = max16(m, s_ans[ans_at(b0 + k)]); ans[k] = m; }
        // what the threads before have reached
        uint32_t before = __shfl_up(block_scan_max16(m, s_max), 1, 64);
        if ((threadIdx.x & 63) == 0) {
            before = 0u;
            for (int k = 0; k < (int)(threadIdx.x >> 6); ++k) before = max16(before, s_max[k]);
        }
        #pragma unroll
        for (int k = 0; k < PER; ++k) { const uint32_t e = max16(ans[k], before); ans[k] = (e & 0xffffu) | e >> 16 << 15; }
    }
    __syncthreads();
    #pragma unroll
    for (int k = 0; k < PER; ++k) s_ans[ans_at(b0 + k)] = ans[k];
    __syncthreads();
    // a pure bucket's group and its destination's flags: the cell lc that receives the particle
    // (none past the outer face: it escapes) and the group a Doppler event shifts it to
    const int lc = t == TAB_L ? ic - 1 : (t == TAB_R ? ic + 1 : ic), shift = t != TAB_D ? 0 : (d.divv[ic - 1] >= 0 ? 1 : -1);
    const bool inside = lc >= 1 && lc <= d.nx;
    const int ls = inside ? lc : ic;
    const double dx = d.xarr[ls] - d.xarr[ls - 1], sg = d.sig[ls - 1];
    const bool lumps = d.cell[ls - 1].nlump > 0;
    #pragma unroll
    for (int k = 0; k < PER; ++k) {
        const int b = threadIdx.x + k * 1024;
        uint32_t e = s_ans[ans_at(b)];
        const int lo = (int)(e & 0x7fffu), hi = (int)(e >> 15);
        const bool pure = emit ? lo == hi : (lo < n ? lo : n - 1) == (hi < n ? hi : n - 1);
        const int g = !pure ? 0 : (emit ? lo : lump_group(d, L, ic, lo));
        if (g > 0) {
            int g2 = g + shift;
            g2 = g2 < 1 ? 1 : (g2 > ng ? ng : g2);
            const double cp = cap_of(d, g2, ls);
            const bool thin = d.puretran || (sg + cp) * dx < d.tauddmc;
            e = BT_PURE | (uint32_t)g;
            if (inside) e |= thin ? BT_THIN : (cp * dx >= d.taulump && lumps ? BT_LUMP : 0u);
        }
        row[b] = e;
    }
}

// The same maps by two plain searches per bucket, a thread per (bucket, cell, table): 64 blocks a map where
// k_bucket_tables has one, for meshes whose maps leave most CUs without a block there.  The whole
// preparation, blocks against searches: 2 x 16 groups 62 and 39 us, 20 x 250 72 and 60, 24 x 250 72 and 64,
// 24 x 4000 158 and 153, 32 x 250 72 and 70, 32 x 4000 161 and 167, 64 x 250 75 and 98: up to 24 cells.
constexpr int BT_SEARCH_CELLS = 24;
__global__ __launch_bounds__(256) void k_bucket_search(Dev d)
{
    const int b = blockIdx.x * 256 + threadIdx.x, ic = blockIdx.y + 1, t = blockIdx.z;
    const double rlo = bt_lo(b), rhi = bt_hi(b);
    int lo, hi, g = 0;
    if (t == TAB_E) {
        lo = emitgroup_direct(d, rlo, ic);
        hi = emitgroup_direct(d, rhi, ic);
        if (lo == hi) g = lo;
    } else {
        const int nlump = d.cell[ic - 1].nlump;
        const LumpRow L = lump_row(d, t, ic, nlump);
        if (nlump == 0 || L.cnt <= 0) {
            d.btab[((size_t)t * d.nx + (ic - 1)) * BT_K + b] = 0u;
            return;
        }
        lo = first_above(L.cum, 0, L.cnt, rlo);
        hi = first_above(L.cum, 0, L.cnt, rhi);
        if ((lo < L.cnt ? lo : L.cnt - 1) == (hi < L.cnt ? hi : L.cnt - 1)) g = lump_group(d, L, ic, lo);
    }
    uint32_t e = (uint32_t)hi << 15 | (uint32_t)lo;
    if (g > 0) {
        const int lc = t == TAB_L ? ic - 1 : (t == TAB_R ? ic + 1 : ic);
        int g2 = t != TAB_D ? g : (d.divv[ic - 1] >= 0 ? g + 1 : g - 1);
        g2 = g2 < 1 ? 1 : (g2 > d.ng ? d.ng : g2);
        e = BT_PURE | (uint32_t)g | (lc >= 1 && lc <= d.nx ? group_flags(d, g2, lc) : 0u);
    }
    d.btab[((size_t)t * d.nx + (ic - 1)) * BT_K + b] = e;
}

void launch_ddmc_tables(slgpu_ctx *c)
{
    hipLaunchKernelGGL(k_leakage, dim3(c->nx), dim3(NT), 0, c->stream, c->d);
    hipLaunchKernelGGL(k_row_terms, dim3((c->ng + 255) / 256, c->nx), dim3(256), 0, c->stream, c->d);
    const size_t rows = (size_t)c->ng * (sizeof(double) + sizeof(float));
    const size_t tiles = sizeof(double) * 3 * RS_ROWS * RS_PITCH;
    const unsigned rblocks = (c->nx + RS_ROWS - 1) / RS_ROWS;
    if (rows <= 143000)                            // beside 16 KB of bin sums
        hipLaunchKernelGGL(k_emitprob<true>, dim3(rblocks + c->nx), dim3(RS_THREADS), rows > tiles ? rows : tiles,
                           c->stream, c->d);
    else
        hipLaunchKernelGGL(k_emitprob<false>, dim3(rblocks + c->nx), dim3(RS_THREADS), tiles, c->stream, c->d);
    hipLaunchKernelGGL(k_row_sums, dim3(rblocks, 5), dim3(RS_THREADS), 0, c->stream, c->d);
    const size_t lds = (size_t)(c->ng + c->d.nep) * sizeof(double), answers = BT_ANSWERS;
    if (c->nx <= BT_SEARCH_CELLS)
        hipLaunchKernelGGL(k_bucket_search, dim3(BT_K / 256, c->nx, NTAB), dim3(256), 0, c->stream, c->d);
    else if (lds <= 160000)
        hipLaunchKernelGGL(k_bucket_tables<true>, dim3(c->nx, NTAB), dim3(1024), lds > answers ? lds : answers,
                           c->stream, c->d);
    else
        hipLaunchKernelGGL(k_bucket_tables<false>, dim3(c->nx, NTAB), dim3(1024), answers, c->stream, c->d);
}

}  // namespace slgpu
