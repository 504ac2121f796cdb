// Smooth Cooper-Frye spectra dN / (pT dpT dphi dy) of chosen species on a
// (pT, phi) grid, summed over the surface cells: the reference's
// EmissionFunctionArray::calculate_dN_pTdpTdphidy (src/emissionfunction.cpp:
// 625-844).  (one translation unit: included by iss_hip.hip)
//
// The reference contracts the lab momentum with the lab-frame Milne cell
// (p.u, p.dsigma, p_mu p_nu pi^{mu nu}).  These are Lorentz invariants, so
// here the lab momentum (mT cosh y, pT cos phi, pT sin phi, mT sinh y) is
// boosted into each cell's rest frame and contracted with the resident
// rest-frame cell record, whose dsigma already carries the factor tau.  The
// delta f is the sampler's (shear with the three coefficient choices, bulk
// kinds 1/11/20/21; src/FSSW.cpp:1897-1928); for shear and bulk kind 1 this is
// the reference's smooth-path delta f (src/emissionfunction.cpp:768-776,
// 4156-4186).  As in the reference, delta f is not clamped into [0, 2]; it is
// optionally rescaled to |delta f| <= deltaf_max_ratio (flag_restrict_deltaf,
// :791-799) and negative contributions are optionally dropped
// (use_pos_dN_only, :804-806).
//
// Layout: a per-cell FP64 record of kSpecRec values (the species-independent
// part of the integrand, k_spectra_rec) is read with wave-uniform (scalar)
// loads, so the per-point work is pure VALU.  One wave evaluates 64 output
// points over one contiguous chunk of cells; chunk sums go to
// partial[chunk][species][point] in FP64 and k_spectra_reduce adds them in a
// fixed order (deterministic).  FP64 spectra integrated over eta_s have a kernel
// of their own (k_spectra64) on forms of the lab momentum.
#pragma once

#include "kernels.h"
#include "yield_kernels.h"

namespace issdev {

constexpr int kSpecRec = 36;
enum SpecSlot {
    RS_IT = 0,                          // 1 / T
    RS_MB, RS_MS, RS_MQ,                // mu_B / T, mu_S / T, mu_Q / T
    RS_U0, RS_U1, RS_U2, RS_U3, RS_IU,  // u (t, x, y, z), 1 / (u0 + 1)
    RS_D0, RS_D1, RS_D2, RS_D3,         // rest-frame dsigma_mu (includes tau)
    RS_XX, RS_XY2, RS_XZ2, RS_YY, RS_YZ2,  // rest-frame pi: xx, 2xy, 2xz, yy, 2yz
    RS_SA, RS_SB,                       // shear: omf * W * (SA + SB / E)
    RS_BM2, RS_BE0, RS_BB, RS_BS, RS_BQ, RS_BE2, RS_BM2E,
    // bulk: omf * (BM2 m^2 + (BE0 + B BB + S BS + Q BQ) E + BE2 E^2 + BM2E m^2 / E)
    RS_CHE, RS_SHE,                     // cosh, sinh of the cell's eta_s
    RS_QX, RS_QY, RS_QZ, RS_PQ,         // diffusion: q / D_qmu, n_B / (e + P)
    kSpecUsed
};
static_assert(kSpecUsed <= kSpecRec, "spectra record");

__global__ void k_spectra_rec(const float* __restrict__ cells, const double* __restrict__ coef, int64_t N,
                              int shear, int bulk, int neos, int diff, double* __restrict__ rec) {
    const int64_t i = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
    if (i >= N) return;
    double r[kSpecRec];
    for (int k = 0; k < kSpecRec; k++) r[k] = 0.;
    const double T = cells[F_T * N + i];
    r[RS_IT] = 1. / T;
    r[RS_MB] = cells[F_MUB * N + i] / T;
    r[RS_MS] = cells[F_MUS * N + i] / T;
    r[RS_MQ] = cells[F_MUQ * N + i] / T;
    const double u0 = cells[F_U0 * N + i];
    r[RS_U0] = u0;
    r[RS_U1] = cells[F_U1 * N + i];
    r[RS_U2] = cells[F_U2 * N + i];
    r[RS_U3] = cells[F_U3 * N + i];
    r[RS_IU] = 1. / (u0 + 1.);
    r[RS_D0] = cells[F_DA0 * N + i];
    r[RS_D1] = cells[F_DA1 * N + i];
    r[RS_D2] = cells[F_DA2 * N + i];
    r[RS_D3] = cells[F_DA3 * N + i];
    double c[6];
    for (int k = 0; k < 6; k++) c[k] = coef[k * N + i];
    if (shear) {
        r[RS_XX] = cells[F_PIXX * N + i];
        r[RS_XY2] = 2. * cells[F_PIXY * N + i];
        r[RS_XZ2] = 2. * cells[F_PIXZ * N + i];
        r[RS_YY] = cells[F_PIYY * N + i];
        r[RS_YZ2] = 2. * cells[F_PIYZ * N + i];
        if (neos == 1) r[RS_SB] = 1. / (2. * c[2] * T);
        else if (neos == 0) r[RS_SA] = c[0];
        else r[RS_SA] = 1. / (2. * T * T * (static_cast<double>(cells[F_E * N + i]) + cells[F_P * N + i]));
    }
    if (bulk != BULK_NONE) {
        double Pi = cells[F_PI * N + i];
        if (bulk == BULK_RTA) Pi = Pi / kHbarC;
        if (bulk == BULK_RTA || bulk == BULK_CE) {
            // -c0 Pi (m^2 / (3 T E) - c1 E / T)
            r[RS_BM2E] = -c[0] * Pi / (3. * T);
            r[RS_BE0] = c[0] * c[1] * Pi / T;
        } else if (bulk == BULK_14MOM) {
            r[RS_BM2] = Pi * c[0];
            r[RS_BB] = Pi * c[1];
            r[RS_BE2] = Pi * c[2];
        } else if (bulk == BULK_22MOM) {
            r[RS_BM2] = Pi * c[2];
            r[RS_BB] = Pi * c[3];
            r[RS_BS] = Pi * c[4];
            r[RS_BQ] = Pi * c[5];
            r[RS_BE2] = Pi * (c[1] - c[2]);
        }
    }
    const double eta = cells[F_ETA * N + i];
    r[RS_CHE] = cosh(eta);
    r[RS_SHE] = sinh(eta);
    if (diff) {
        // (src/emissionfunction.cpp:777-786): (1 - s f0) (n_B/(e+P) - B/E) p.q / D_qmu
        const double iq = coef[6 * N + i];
        r[RS_QX] = cells[F_QX * N + i] * iq;
        r[RS_QY] = cells[F_QY * N + i] * iq;
        r[RS_QZ] = cells[F_QZ * N + i] * iq;
        r[RS_PQ] = coef[7 * N + i];
    }
    for (int k = 0; k < kSpecRec; k++) rec[i * kSpecRec + k] = r[k];
}

// Which chemical potentials (over T) are not zero on some cell (NaN counts),
// as bits in *used: one atomic per workgroup, so that few meet on the word.
enum MuUsed { MU_B = 1, MU_S = 2, MU_Q = 4 };
__global__ __launch_bounds__(256) void k_mu_used(const double* __restrict__ rec, int64_t N, int* __restrict__ used) {
    int m = 0;
    for (int64_t i = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x; i < N;
         i += static_cast<int64_t>(gridDim.x) * blockDim.x) {
        const double* v = rec + i * kSpecRec;
        m |= !(v[RS_MB] == 0.) ? MU_B : 0;
        m |= !(v[RS_MS] == 0.) ? MU_S : 0;
        m |= !(v[RS_MQ] == 0.) ? MU_Q : 0;
    }
    const int b = __syncthreads_or(m & MU_B), s = __syncthreads_or(m & MU_S), q = __syncthreads_or(m & MU_Q);
    m = (b ? MU_B : 0) | (s ? MU_S : 0) | (q ? MU_Q : 0);
    if (threadIdx.x == 0 && m) atomicOr(used, m);
}

struct SpectraArgs {
    const double* rec;        // [N][kSpecRec]
    int64_t N;
    int64_t cells_per_chunk;
    SpeciesDev sp;
    const int32_t* species;   // [ns] species indices, one of each set with equal integrands
    int ns;
    const double* pT;         // [npT]
    int npT;
    const double* cphi;       // [nphi]
    const double* sphi;
    int nphi;
    // mode 0: nodes of y - eta_s with weights (cosh, sinh, weight);
    // mode 1: rapidities (cosh, sinh), one output plane per rapidity
    const double* ych;
    const double* ysh;
    const double* yw;
    int ny;
    int mode;
    int positive_only;
    double restrict_ratio;    // <= 0: no rescaling of delta f
    int waves_per_species;
    double* partial;          // [chunks][ns][npts]
    const double* milne;      // [N][kMilneRec] (FP64, mode 0)
};

constexpr double kLog2e = 1.4426950408889634;
constexpr int kSpecPts = 4;   // output points per lane

__device__ __forceinline__ double fexp2(double x) { return exp2(x); }
__device__ __forceinline__ float fexp2(float x) { return __builtin_amdgcn_exp2f(x); }

// per (cell, species) constants of the delta f, in the working type R
template <typename R>
struct SpecCell {
    R xx, xy2, xz2, yy, yz2, sa, sb, cm, be, be2, cme, sg, lo, hi;
    R qx, qy, qz, pq, bq;   // diffusion (zero when off)
    __device__ __forceinline__ void set(const R* k) {
        xx = k[0]; xy2 = k[1]; xz2 = k[2]; yy = k[3]; yz2 = k[4]; sa = k[5]; sb = k[6]; cm = k[7];
        be = k[8]; be2 = k[9]; cme = k[10]; pq = k[11]; qx = k[12]; qy = k[13]; qz = k[14];
    }
};
template <typename R>
__device__ __forceinline__ void spec_cell(const double* v, double m, double B, double S, double Q, R* k) {
    k[0] = static_cast<R>(v[RS_XX]); k[1] = static_cast<R>(v[RS_XY2]); k[2] = static_cast<R>(v[RS_XZ2]);
    k[3] = static_cast<R>(v[RS_YY]); k[4] = static_cast<R>(v[RS_YZ2]);
    k[5] = static_cast<R>(v[RS_SA]); k[6] = static_cast<R>(v[RS_SB]);
    k[7] = static_cast<R>(v[RS_BM2] * m * m);
    k[8] = static_cast<R>(v[RS_BE0] + B * v[RS_BB] + S * v[RS_BS] + Q * v[RS_BQ]);
    k[9] = static_cast<R>(v[RS_BE2]);
    k[10] = static_cast<R>(v[RS_BM2E] * m * m);
    k[11] = static_cast<R>(v[RS_PQ]);
    k[12] = static_cast<R>(v[RS_QX]); k[13] = static_cast<R>(v[RS_QY]); k[14] = static_cast<R>(v[RS_QZ]);
}

// the coefficients of mT in E, l_x, l_y, l_z, p.dsigma and E / T * log2(e) for
// the lab direction (ch, sh) (see the linear forms below)
__device__ __forceinline__ void spec_node(const double* v, double ch, double sh, double* nd) {
    const double u0 = v[RS_U0], u1 = v[RS_U1], u2 = v[RS_U2], u3 = v[RS_U3], iu = v[RS_IU];
    const double a0 = u0 * ch - u3 * sh;
    const double g = sh * u3 * iu - ch;
    const double a1 = u1 * g, a2 = u2 * g, a3 = sh + u3 * g;
    nd[0] = a0;
    nd[1] = a1;
    nd[2] = a2;
    nd[3] = a3;
    nd[4] = a0 * v[RS_D0] + a1 * v[RS_D1] + a2 * v[RS_D2] + a3 * v[RS_D3];
    nd[5] = a0 * v[RS_IT] * kLog2e;
}

// f0 p.dsigma (1 + delta f) from the rest-frame energy E, momentum (lx, ly,
// lz), p.dsigma and x2 = (E - mu) / T * log2(e).  |delta f| is clamped at
// deltaf_max_ratio (lo = -ratio, hi = ratio, or -+inf when off): the
// reference's rescaling df * min(1, ratio / (|df| + 1e-10)) differs from the
// clamp by at most ratio * 1e-10 / |df| in 1 + delta f.
// DF leaves out the terms that are zero: none, a polynomial in the momentum,
// plus a constant over E, or all of them.
enum SpecDf { SDF_NONE = 0, SDF_POLY = 1, SDF_CONST_E = 2, SDF_POLY_E = 3 };
template <typename R, int DF>
__device__ __forceinline__ R spectra_integrand(const SpecCell<R>& c, R E, R lx, R ly, R lz, R pds, R x2,
                                               int positive_only) {
    const R f0 = frcp(fexp2(x2) + c.sg);
    R r = f0 * pds;
    if (DF != SDF_NONE) {
        const R omf = R(1) - c.sg * f0;
        const R lz2 = lz * lz;
        const R W =
            c.xx * (lx * lx - lz2) + c.yy * (ly * ly - lz2) + lx * (c.xy2 * ly + c.xz2 * lz) + c.yz2 * ly * lz;
        const R iE = DF >= SDF_CONST_E ? frcp(E) : R(0);
        const R sab = DF == SDF_POLY_E ? c.sa + c.sb * iE : c.sa;
        R df = W * sab + c.cm + E * (c.be + c.be2 * E);
        if (DF >= SDF_CONST_E) df += c.cme * iE;
        if (DF == SDF_POLY_E) df -= (c.pq - c.bq * iE) * (lx * c.qx + ly * c.qy + lz * c.qz);
        df *= omf;
        df = fmin(fmax(df, c.lo), c.hi);
        r *= R(1) + df;
    }
    if (positive_only && r < R(0)) r = R(0);
    return r;
}

// grid (chunks, ns * waves_per_species), 64 threads, kSpecPts points per lane
// (points base + 64 q).
//
// mode 0: the lab momentum at rapidity eta_cell + (y - eta_s)_k is
// (mT ch_k, px, py, mT sh_k); its rest-frame components are linear in mT with
// per-(cell, k) coefficients and offsets per (cell, point):
//   E = mT a0 + Pe,  l_i = mT a_i + P_i,  p.dsigma = mT dk + Pds,
//   a0 = u0 ch - u3 sh, g = sh u3 / (u0 + 1) - ch, (a1, a2, a3) = (u1 g, u2 g, sh + u3 g),
//   Pe = -(px u1 + py u2), P_i = p_i - Pe u_i / (u0 + 1) (p_z = 0).
// The coefficients are formed in FP64 (ch_k, sh_k of boosted cells are
// differences of large terms), a node per lane, and read from LDS by the wave;
// the per-point work runs in FP32.
template <int DF>
__global__ __launch_bounds__(64) void k_spectra32(SpectraArgs a) {
    __shared__ __align__(16) float s_node[64 * 8];
    const int npts = a.npT * a.nphi;
    const int si = blockIdx.y / a.waves_per_species;
    const int lane = threadIdx.x;
    const int base = (blockIdx.y % a.waves_per_species) * 64 * kSpecPts + lane;
    const int s = a.species[si];
    const double m = a.sp.mass[s];
    const double B = a.sp.B[s], S = a.sp.S[s], Q = a.sp.Q[s];
    double mT[kSpecPts], px[kSpecPts], py[kSpecPts], acc[kSpecPts];
#pragma unroll
    for (int q = 0; q < kSpecPts; q++) {
        const int pt = min(base + 64 * q, npts - 1);
        const double pT = a.pT[pt / a.nphi];
        mT[q] = sqrt(pT * pT + m * m);
        px[q] = pT * a.cphi[pt % a.nphi];
        py[q] = pT * a.sphi[pt % a.nphi];
        acc[q] = 0.;
    }
    SpecCell<float> c;
    c.sg = static_cast<float>(a.sp.sign[s]);
    c.bq = static_cast<float>(B);
    c.hi = a.restrict_ratio > 0. ? static_cast<float>(a.restrict_ratio) : INFINITY;
    c.lo = -c.hi;
    const int64_t l0 = static_cast<int64_t>(blockIdx.x) * a.cells_per_chunk;
    const int64_t l1 = min<int64_t>(a.N, l0 + a.cells_per_chunk);
    for (int64_t l = l0; l < l1; l++) {
        const double* v = a.rec + l * kSpecRec;
        const double u1 = v[RS_U1], u2 = v[RS_U2], u3 = v[RS_U3], iu = v[RS_IU];
        const double d0 = v[RS_D0], d1 = v[RS_D1], d2 = v[RS_D2], d3 = v[RS_D3];
        const double it = v[RS_IT], mu = B * v[RS_MB] + S * v[RS_MS] + Q * v[RS_MQ];
        float k16[16];
        spec_cell(v, m, B, S, Q, k16);
        c.set(k16);
        float mTr[kSpecPts], Pe[kSpecPts], Px[kSpecPts], Py[kSpecPts], Pz[kSpecPts], Pds[kSpecPts], X0[kSpecPts];
        float cell[kSpecPts];
#pragma unroll
        for (int q = 0; q < kSpecPts; q++) {
            const double pe = -(px[q] * u1 + py[q] * u2);
            const double qx = px[q] - pe * iu * u1, qy = py[q] - pe * iu * u2, qz = -pe * iu * u3;
            mTr[q] = static_cast<float>(mT[q]);
            Pe[q] = static_cast<float>(pe);
            Px[q] = static_cast<float>(qx);
            Py[q] = static_cast<float>(qy);
            Pz[q] = static_cast<float>(qz);
            Pds[q] = static_cast<float>(pe * d0 + qx * d1 + qy * d2 + qz * d3);
            X0[q] = static_cast<float>((pe * it - mu) * kLog2e);
            cell[q] = 0.f;
        }
        for (int k0 = 0; k0 < a.ny; k0 += 64) {
            const int nk = min(64, a.ny - k0);
            wave_lds_sync();
            if (lane < nk) {
                const double cy = a.ych[k0 + lane], sy = a.ysh[k0 + lane];
                const double che = v[RS_CHE], she = v[RS_SHE];
                double nd[6];
                spec_node(v, che * cy + she * sy, she * cy + che * sy, nd);
                float* o = s_node + lane * 8;
                for (int t = 0; t < 6; t++) o[t] = static_cast<float>(nd[t]);
                o[6] = static_cast<float>(a.yw[k0 + lane]);
            }
            wave_lds_sync();
            for (int k = 0; k < nk; k++) {
                const float4 n0 = *reinterpret_cast<const float4*>(s_node + k * 8);
                const float4 n1 = *reinterpret_cast<const float4*>(s_node + k * 8 + 4);
#pragma unroll
                for (int q = 0; q < kSpecPts; q++) {
                    const float E = mTr[q] * n0.x + Pe[q];
                    const float lx = mTr[q] * n0.y + Px[q], ly = mTr[q] * n0.z + Py[q], lz = mTr[q] * n0.w + Pz[q];
                    const float pds = mTr[q] * n1.x + Pds[q];
                    const float x2 = mTr[q] * n1.y + X0[q];
                    cell[q] += n1.z * spectra_integrand<float, DF>(c, E, lx, ly, lz, pds, x2, a.positive_only);
                }
            }
        }
#pragma unroll
        for (int q = 0; q < kSpecPts; q++) acc[q] += static_cast<double>(cell[q]);
    }
#pragma unroll
    for (int q = 0; q < kSpecPts; q++) {
        const int pt = base + 64 * q;
        if (pt < npts) a.partial[(static_cast<int64_t>(blockIdx.x) * a.ns + si) * npts + pt] = acc[q];
    }
}

// mode 1 on grids of few (pT, phi) points, where k_spectra_y would leave lanes
// idle: kSpecPts points of any rapidity per lane, each boosted by itself
template <typename R>
__global__ __launch_bounds__(64) void k_spectra_points(SpectraArgs a) {
    const int npl = a.npT * a.nphi;
    const int npts = npl * a.ny;
    const int si = blockIdx.y / a.waves_per_species;
    const int base = (blockIdx.y % a.waves_per_species) * 64 * kSpecPts + threadIdx.x;
    const int s = a.species[si];
    const double m = a.sp.mass[s];
    const double B = a.sp.B[s], S = a.sp.S[s], Q = a.sp.Q[s];
    double px[kSpecPts], py[kSpecPts], p0f[kSpecPts], pzf[kSpecPts];
#pragma unroll
    for (int q = 0; q < kSpecPts; q++) {
        const int pt = min(base + 64 * q, npts - 1);
        const int iphi = pt % a.nphi;
        const int ipt = (pt / a.nphi) % a.npT;
        const double pT = a.pT[ipt];
        const double mT = sqrt(pT * pT + m * m);
        px[q] = pT * a.cphi[iphi];
        py[q] = pT * a.sphi[iphi];
        const int iy = pt / npl;
        p0f[q] = mT * a.ych[iy];
        pzf[q] = mT * a.ysh[iy];
    }
    SpecCell<R> c;
    c.sg = static_cast<R>(a.sp.sign[s]);
    c.bq = static_cast<R>(B);
    const R inf = static_cast<R>(INFINITY);
    c.hi = a.restrict_ratio > 0. ? static_cast<R>(a.restrict_ratio) : inf;
    c.lo = -c.hi;
    const int64_t l0 = static_cast<int64_t>(blockIdx.x) * a.cells_per_chunk;
    const int64_t l1 = min<int64_t>(a.N, l0 + a.cells_per_chunk);
    double acc[kSpecPts];
#pragma unroll
    for (int q = 0; q < kSpecPts; q++) acc[q] = 0.;
    for (int64_t l = l0; l < l1; l++) {
        const double* v = a.rec + l * kSpecRec;
        const double u0 = v[RS_U0], u1 = v[RS_U1], u2 = v[RS_U2], u3 = v[RS_U3], iu = v[RS_IU];
        const double d0 = v[RS_D0], d1 = v[RS_D1], d2 = v[RS_D2], d3 = v[RS_D3];
        const double it = v[RS_IT];
        const double mu = B * v[RS_MB] + S * v[RS_MS] + Q * v[RS_MQ];
        R k16[16];
        spec_cell(v, m, B, S, Q, k16);
        c.set(k16);
#pragma unroll
        for (int q = 0; q < kSpecPts; q++) {
            const double pdu = px[q] * u1 + py[q] * u2 + pzf[q] * u3;
            const double E = u0 * p0f[q] - pdu;
            const double kk = pdu * iu - p0f[q];
            const double lx = px[q] + kk * u1, ly = py[q] + kk * u2, lz = pzf[q] + kk * u3;
            const double pds = E * d0 + lx * d1 + ly * d2 + lz * d3;
            acc[q] += static_cast<double>(spectra_integrand<R, SDF_POLY_E>(
                c, static_cast<R>(E), static_cast<R>(lx), static_cast<R>(ly), static_cast<R>(lz),
                static_cast<R>(pds), static_cast<R>((E * it - mu) * kLog2e), a.positive_only));
        }
    }
#pragma unroll
    for (int q = 0; q < kSpecPts; q++) {
        const int pt = base + 64 * q;
        if (pt < npts) a.partial[(static_cast<int64_t>(blockIdx.x) * a.ns + si) * npts + pt] = acc[q];
    }
}

// mode 1 (one output plane per rapidity), in FP32 or FP64: the same linear
// forms at ch = cosh y, sh = sinh y, summed in FP64 before they are rounded to
// R.  A wave holds kYSets sets of 64 (pT, phi) points for up to kYMax
// rapidities, so a point costs six FMAs instead of the boost's seventeen, the
// offsets are formed once per (cell, set), and the constants of kYCells cells
// are formed at a time, a (cell, rapidity) per lane, instead of by every wave
// in all its lanes.  Vector issue bounds it (42 instructions a point, from 72:
// six FMAs, seven conversions, the rest the integrand).  20 10^3 cells, 5
// species, 3168 points: 490 -> 386 us.
constexpr int kYSets = 2, kYMax = 6, kYCells = 8;
__host__ __device__ constexpr int spec_y_chunks(int ny) { return (ny + kYMax - 1) / kYMax; }
__host__ __device__ constexpr int spec_y_waves(int npl) { return (npl + 64 * kYSets - 1) / (64 * kYSets); }

template <typename R, int DF>
__global__ __launch_bounds__(64) void k_spectra_y(SpectraArgs a) {
    __shared__ __align__(16) double s_node[kYCells][8][6];
    __shared__ __align__(16) R s_cell[kYCells][16];
    const int npl = a.npT * a.nphi;
    const unsigned pw = static_cast<unsigned>(a.ns * a.waves_per_species);
    const int chunk = blockIdx.x / pw, rest = blockIdx.x % pw;  // (one-dimensional: many rapidities)
    const int si = rest / a.waves_per_species, w = rest % a.waves_per_species;
    const int lane = threadIdx.x;
    const int per = (a.ny + spec_y_chunks(a.ny) - 1) / spec_y_chunks(a.ny);
    const int iy0 = w / spec_y_waves(npl) * per, nk = min(per, a.ny - iy0);
    const int pl0 = w % spec_y_waves(npl) * 64 * kYSets;
    const int nset = min(kYSets, (npl - pl0 + 63) / 64);
    const int s = a.species[si];
    const double m = a.sp.mass[s];
    const double B = a.sp.B[s], S = a.sp.S[s], Q = a.sp.Q[s];
    double mT[kYSets], px[kYSets], py[kYSets], acc[kYSets][kYMax];
#pragma unroll
    for (int t = 0; t < kYSets; t++) {
        const int pl = min(pl0 + 64 * t + lane, npl - 1);
        const double pT = a.pT[pl / a.nphi];
        mT[t] = sqrt(pT * pT + m * m);
        px[t] = pT * a.cphi[pl % a.nphi];
        py[t] = pT * a.sphi[pl % a.nphi];
#pragma unroll
        for (int k = 0; k < kYMax; k++) acc[t][k] = 0.;
    }
    SpecCell<R> c;
    c.sg = static_cast<R>(a.sp.sign[s]);
    c.bq = static_cast<R>(B);
    c.hi = a.restrict_ratio > 0. ? static_cast<R>(a.restrict_ratio) : static_cast<R>(INFINITY);
    c.lo = -c.hi;
    const int64_t l0 = static_cast<int64_t>(chunk) * a.cells_per_chunk;
    const int64_t l1 = min<int64_t>(a.N, l0 + a.cells_per_chunk);
    for (int64_t lb = l0; lb < l1; lb += kYCells) {
        const int nc = static_cast<int>(min<int64_t>(kYCells, l1 - lb));
        wave_lds_sync();
        if (lane / 8 < nc) {
            const double* v = a.rec + (lb + lane / 8) * kSpecRec;
            const int k = lane % 8;
            if (k < nk) spec_node(v, a.ych[iy0 + k], a.ysh[iy0 + k], s_node[lane / 8][k]);
            if (k == 7 && DF != SDF_NONE) spec_cell(v, m, B, S, Q, s_cell[lane / 8]);
        }
        wave_lds_sync();
        for (int j = 0; j < nc; j++) {
            const double* v = a.rec + (lb + j) * kSpecRec;
            const double u1 = v[RS_U1], u2 = v[RS_U2], u3 = v[RS_U3], iu = v[RS_IU];
            const double d0 = v[RS_D0], d1 = v[RS_D1], d2 = v[RS_D2], d3 = v[RS_D3];
            const double it = v[RS_IT], mu = B * v[RS_MB] + S * v[RS_MS] + Q * v[RS_MQ];
            if (DF != SDF_NONE) c.set(s_cell[j]);
            double Pe[kYSets], Px[kYSets], Py[kYSets], Pz[kYSets], Pds[kYSets], X0[kYSets];
#pragma unroll
            for (int t = 0; t < kYSets; t++) {
                const double pe = -(px[t] * u1 + py[t] * u2), pu = pe * iu;
                Pe[t] = pe;
                Px[t] = px[t] - pu * u1;
                Py[t] = py[t] - pu * u2;
                Pz[t] = -pu * u3;
                Pds[t] = pe * d0 + Px[t] * d1 + Py[t] * d2 + Pz[t] * d3;
                X0[t] = (pe * it - mu) * kLog2e;
            }
#pragma unroll
            for (int k = 0; k < kYMax; k++) {
                if (k < nk) {
                    const double* nd = s_node[j][k];
                    const double a0 = nd[0], a1 = nd[1], a2 = nd[2], a3 = nd[3], dk = nd[4], ax = nd[5];
#pragma unroll
                    for (int t = 0; t < kYSets; t++)
                        if (t < nset)
                            acc[t][k] += static_cast<double>(spectra_integrand<R, DF>(
                                c, static_cast<R>(mT[t] * a0 + Pe[t]), static_cast<R>(mT[t] * a1 + Px[t]),
                                static_cast<R>(mT[t] * a2 + Py[t]), static_cast<R>(mT[t] * a3 + Pz[t]),
                                static_cast<R>(mT[t] * dk + Pds[t]), static_cast<R>(mT[t] * ax + X0[t]),
                                a.positive_only));
                }
            }
        }
    }
    const int64_t npts = static_cast<int64_t>(npl) * a.ny;
    double* out = a.partial + (static_cast<int64_t>(chunk) * a.ns + si) * npts;
#pragma unroll
    for (int t = 0; t < kYSets; t++) {
        const int pl = pl0 + 64 * t + lane;
#pragma unroll
        for (int k = 0; k < kYMax; k++)
            if (pl < npl && k < nk) out[static_cast<int64_t>(iy0 + k) * npl + pl] = acc[t][k];
    }
}

// ------------------------------------------------------ FP64, integrated over eta_s
// The FP64 spectra of mode 0 are VALU-bound: N cells x n_eta nodes x points
// evaluations of one integrand, so its FP64 instruction count is the time.
// The kernel below evaluates the same sums with about 40 FP64 issue slots a
// point where the rest-frame form takes about 110:
//   * Everything the integrand contracts is linear or quadratic in the lab
//     momentum (mT cosh y, px, py, mT sinh y), and cosh, sinh of
//     y = eta_cell + (y - eta_s)_k are linear in those of the node.  So per
//     cell the record holds E, p.dsigma, q.l as linear forms and
//     sa pi^{mu nu} p_mu p_nu + be2 E^2 (and sb pi^{mu nu} p_mu p_nu) as
//     quadratic forms of (mT cosh y_k, mT sinh y_k, px, py); the whole
//     delta f polynomial is 4 FMAs a point and needs neither E nor l.
//   * The (cell, node) coefficients are formed once per wave, one node per
//     lane, and read back from LDS as broadcasts (they cost about 20 FP64
//     instructions per node and wave when every lane forms them).
//   * 1 / E enters only where the delta f has it (Chapman-Enskog shear, the
//     relaxation-time and Chapman-Enskog bulk, diffusion): DF.
//   * exp2 is a polynomial of degree 11 on [-1/2, 1/2] (relative error 2e-17, 2e-16
//     with its rounding) and an exponent shift, the occupancy a hardware
//     reciprocal with one third-order step (1 ulp).
// Measured at 200,000 cells x 3 species x 720 points x 81 nodes: 98.8 ms
// with the rest-frame form, 38.8 ms with this kernel (9.0e11 points/s).
constexpr int kMilneRec = 48;
enum MilneSlot {
    ML_IT = 0, ML_MB, ML_MS, ML_MQ,    // log2(e) / T and log2(e) mu / T
    ML_E1, ML_E2, ML_U1, ML_U2,        // E = mT (E1 ch + E2 sh) - px U1 - py U2
    ML_D1, ML_D2, ML_DX, ML_DY,        // p.dsigma, likewise (plus signs)
    // quadratic form A = sa pi^{mu nu} p_mu p_nu + be2 E^2 (and B = sb pi pp):
    // mT^2 (11 ch^2 + 12 ch sh + 22 sh^2) + mT px (1X ch + 2X sh) + mT py (1Y ch + 2Y sh)
    // + XX px^2 + XY px py + YY py^2
    ML_A,                              // 11, 12, 22, 1X, 2X, 1Y, 2Y, XX, XY, YY
    ML_B = ML_A + 10,
    ML_Q1 = ML_B + 10, ML_Q2, ML_QX, ML_QY,   // q.l / D_qmu, linear
    ML_PQ, ML_BM2, ML_BE0, ML_BB, ML_BS, ML_BQ, ML_BM2E,
    kMilneUsed
};
static_assert(kMilneUsed <= kMilneRec, "Milne spectra record");

// the record of k_spectra_rec (rest frame) as forms of the lab momentum
// relative to the cell's eta_s; one thread per cell
__global__ void k_spectra_milne(const double* __restrict__ rec, int64_t N, double* __restrict__ out) {
    const int64_t i = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
    if (i >= N) return;
    const double* v = rec + i * kSpecRec;
    double r[kMilneRec];
    for (int k = 0; k < kMilneRec; k++) r[k] = 0.;
    const double u0 = v[RS_U0], u1 = v[RS_U1], u2 = v[RS_U2], u3 = v[RS_U3], iu = v[RS_IU];
    const double che = v[RS_CHE], she = v[RS_SHE];
    r[ML_IT] = v[RS_IT] * kLog2e;
    r[ML_MB] = v[RS_MB] * kLog2e;
    r[ML_MS] = v[RS_MS] * kLog2e;
    r[ML_MQ] = v[RS_MQ] * kLog2e;
    r[ML_E1] = u0 * che - u3 * she;
    r[ML_E2] = u0 * she - u3 * che;
    r[ML_U1] = u1;
    r[ML_U2] = u2;
    // rest-frame momentum l = mT (ch b0 + sh b1) + px b2 + py b3
    const double k1 = she * u3 * iu - che, k2 = che * u3 * iu - she, kx = u1 * iu, ky = u2 * iu;
    const double b[4][3] = {{u1 * k1, u2 * k1, she + u3 * k1},
                            {u1 * k2, u2 * k2, che + u3 * k2},
                            {1. + u1 * kx, u2 * kx, u3 * kx},
                            {u1 * ky, 1. + u2 * ky, u3 * ky}};
    const double e[4] = {r[ML_E1], r[ML_E2], -u1, -u2};
    // a temperature or chemical potential that is not a number, or not finite,
    // makes every point so
    const double poison = 0. * (v[RS_IT] + v[RS_MB] + v[RS_MS] + v[RS_MQ]);
    for (int a = 0; a < 4; a++) {
        r[ML_D1 + a] = e[a] * v[RS_D0] + b[a][0] * v[RS_D1] + b[a][1] * v[RS_D2] + b[a][2] * v[RS_D3] + poison;
        r[ML_Q1 + a] = b[a][0] * v[RS_QX] + b[a][1] * v[RS_QY] + b[a][2] * v[RS_QZ];
    }
    const double xx = v[RS_XX], xy = 0.5 * v[RS_XY2], xz = 0.5 * v[RS_XZ2], yy = v[RS_YY], yz = 0.5 * v[RS_YZ2];
    const double sa = v[RS_SA], sb = v[RS_SB], be2 = v[RS_BE2];
    const int ia[10] = {0, 0, 1, 0, 1, 0, 1, 2, 2, 3}, ib[10] = {0, 1, 1, 2, 2, 3, 3, 2, 3, 3};
#pragma unroll
    for (int t = 0; t < 10; t++) {
        const double* p = b[ia[t]];
        const double* q = b[ib[t]];
        const double w = p[0] * (xx * q[0] + xy * q[1] + xz * q[2]) + p[1] * (xy * q[0] + yy * q[1] + yz * q[2]) +
                         p[2] * (xz * q[0] + yz * q[1] - (xx + yy) * q[2]);
        const double f = ia[t] == ib[t] ? 1. : 2.;
        r[ML_A + t] = f * (sa * w + be2 * e[ia[t]] * e[ib[t]]);
        r[ML_B + t] = f * sb * w;
    }
    r[ML_PQ] = v[RS_PQ];
    r[ML_BM2] = v[RS_BM2];
    r[ML_BE0] = v[RS_BE0];
    r[ML_BB] = v[RS_BB];
    r[ML_BS] = v[RS_BS];
    r[ML_BQ] = v[RS_BQ];
    r[ML_BM2E] = v[RS_BM2E];
    for (int k = 0; k < kMilneRec; k++) out[i * kMilneRec + k] = r[k];
}

// 2^x for every finite x, 0 and infinity beyond the double range: x = n + f, f
// in [-1/2, 1/2] (n saturates at the ends of the integers), 2^f by a polynomial
// fitted at the Chebyshev nodes of the interval
__device__ __forceinline__ double exp2_poly(double x) {
    const double t = __builtin_rint(x);
    const double f = x - t;
    const int n = static_cast<int>(t);
    double p = 4.455446116749247e-10;
    p = fma(p, f, 7.072590211349959e-09);
    p = fma(p, f, 1.0178059415329878e-07);
    p = fma(p, f, 1.3215442559248754e-06);
    p = fma(p, f, 1.5252733836343741e-05);
    p = fma(p, f, 0.00015403530441800403);
    p = fma(p, f, 0.0013333558146411463);
    p = fma(p, f, 0.009618129107606836);
    p = fma(p, f, 0.05550410866482161);
    p = fma(p, f, 0.24022650695910097);
    p = fma(p, f, 0.6931471805599453);
    p = fma(p, f, 1.0);
    return __builtin_amdgcn_ldexp(p, n);
}

// 1 / d for finite normal d: the hardware estimate (about 2^-24) and one
// third-order step, within 1 ulp.  occupancy: 0 for d = infinity as well, whose
// step is not a number and becomes 1.
__device__ __forceinline__ double rcp_step(double d) {
    const double r = __builtin_amdgcn_rcp(d);
    const double e = fma(-d, r, 1.);
    return fma(r, fma(e, e, e), r);
}

__device__ __forceinline__ double occupancy(double d) {
    const double r = __builtin_amdgcn_rcp(d);
    const double e = fmin(fma(-d, r, 1.), 1.);
    return fma(r, fma(e, e, e), r);
}

// Grid (chunks, ns * waves_per_species), one wave per workgroup, kSpecPts
// points per lane (points base + 64 q), nodes in groups of 64.
template <int DF, bool POSITIVE>
__global__ __launch_bounds__(64) void k_spectra64(SpectraArgs a) {
    constexpr int NW = DF == SDF_POLY_E ? 12 : 8;   // doubles per node in LDS
    __shared__ __align__(16) double s_node[64 * NW];
    const int npts = a.npT * a.nphi;
    const int si = blockIdx.y / a.waves_per_species;
    const int lane = threadIdx.x;
    const int base = (blockIdx.y % a.waves_per_species) * 64 * kSpecPts + lane;
    const int s = a.species[si];
    const double m = a.sp.mass[s], m2 = m * m;
    const double B = a.sp.B[s], S = a.sp.S[s], Q = a.sp.Q[s], sg = a.sp.sign[s];
    const double hi = a.restrict_ratio > 0. ? a.restrict_ratio : INFINITY;
    double mT[kSpecPts], px[kSpecPts], py[kSpecPts], acc[kSpecPts];
#pragma unroll
    for (int q = 0; q < kSpecPts; q++) {
        const int pt = min(base + 64 * q, npts - 1);
        const double pT = a.pT[pt / a.nphi];
        mT[q] = sqrt(pT * pT + m2);
        px[q] = pT * a.cphi[pt % a.nphi];
        py[q] = pT * a.sphi[pt % a.nphi];
        acc[q] = 0.;
    }
    const int64_t l0 = static_cast<int64_t>(blockIdx.x) * a.cells_per_chunk;
    const int64_t l1 = min<int64_t>(a.N, l0 + a.cells_per_chunk);
    for (int64_t l = l0; l < l1; l++) {
        const double* v = a.milne + l * kMilneRec;
        const double it = v[ML_IT], mu = B * v[ML_MB] + S * v[ML_MS] + Q * v[ML_MQ];
        const double be = v[ML_BE0] + B * v[ML_BB] + S * v[ML_BS] + Q * v[ML_BQ];
        const double cm = v[ML_BM2] * m2, cme = v[ML_BM2E] * m2, pq = v[ML_PQ];
        double X0[kSpecPts], Pds[kSpecPts], G0[kSpecPts], H0[kSpecPts], Pe[kSpecPts], cell[kSpecPts];
#pragma unroll
        for (int q = 0; q < kSpecPts; q++) {
            Pe[q] = -(px[q] * v[ML_U1] + py[q] * v[ML_U2]);
            X0[q] = fma(Pe[q], it, -mu);
            Pds[q] = px[q] * v[ML_DX] + py[q] * v[ML_DY];
            cell[q] = G0[q] = H0[q] = 0.;
            if (DF != SDF_NONE)
                G0[q] = px[q] * (px[q] * v[ML_A + 7] + py[q] * v[ML_A + 8]) + py[q] * py[q] * v[ML_A + 9] + cm +
                        be * Pe[q];
            if (DF == SDF_POLY_E) {
                const double ql = px[q] * v[ML_QX] + py[q] * v[ML_QY];
                G0[q] -= pq * ql;
                H0[q] = px[q] * (px[q] * v[ML_B + 7] + py[q] * v[ML_B + 8]) + py[q] * py[q] * v[ML_B + 9] + cme +
                        B * ql;
            }
        }
        for (int k0 = 0; k0 < a.ny; k0 += 64) {
            const int nk = min(64, a.ny - k0);
            wave_lds_sync();
            if (lane < nk) {
                const double ch = a.ych[k0 + lane], sh = a.ysh[k0 + lane];
                double* nd = s_node + lane * NW;
                const double a0 = v[ML_E1] * ch + v[ML_E2] * sh;
                nd[0] = DF >= SDF_CONST_E ? a0 : a0 * it;
                nd[1] = v[ML_D1] * ch + v[ML_D2] * sh;
                nd[2] = a.yw[k0 + lane];
                if (DF != SDF_NONE) {
                    nd[3] = ch * (v[ML_A + 0] * ch + v[ML_A + 1] * sh) + v[ML_A + 2] * sh * sh;
                    nd[4] = v[ML_A + 3] * ch + v[ML_A + 4] * sh;
                    nd[5] = v[ML_A + 5] * ch + v[ML_A + 6] * sh;
                    nd[6] = be * a0;
                }
                if (DF == SDF_POLY_E) {
                    const double ql = v[ML_Q1] * ch + v[ML_Q2] * sh;
                    nd[6] -= pq * ql;
                    nd[7] = ch * (v[ML_B + 0] * ch + v[ML_B + 1] * sh) + v[ML_B + 2] * sh * sh;
                    nd[8] = v[ML_B + 3] * ch + v[ML_B + 4] * sh;
                    nd[9] = v[ML_B + 5] * ch + v[ML_B + 6] * sh;
                    nd[10] = B * ql;
                }
            }
            wave_lds_sync();
            for (int k = 0; k < nk; k++) {
                double nd[NW];
#pragma unroll
                for (int t = 0; t < NW; t += 2) {
                    const double2 w = *reinterpret_cast<const double2*>(s_node + k * NW + t);
                    nd[t] = w.x;
                    nd[t + 1] = w.y;
                }
#pragma unroll
                for (int q = 0; q < kSpecPts; q++) {
                    double E = 0., x;
                    if (DF >= SDF_CONST_E) {
                        E = fma(mT[q], nd[0], Pe[q]);
                        x = fma(E, it, -mu);
                    } else {
                        x = fma(mT[q], nd[0], X0[q]);
                    }
                    const double f0 = occupancy(exp2_poly(x) + sg);
                    double r = f0 * fma(mT[q], nd[1], Pds[q]);
                    if (DF != SDF_NONE) {
                        double G = fma(mT[q], fma(mT[q], nd[3], fma(px[q], nd[4], fma(py[q], nd[5], nd[6]))), G0[q]);
                        if (DF == SDF_CONST_E) G = fma(rcp_step(E), cme, G);
                        if (DF == SDF_POLY_E)
                            G = fma(rcp_step(E),
                                    fma(mT[q], fma(mT[q], nd[7], fma(px[q], nd[8], fma(py[q], nd[9], nd[10]))), H0[q]),
                                    G);
                        // |delta f| <= deltaf_max_ratio, as spectra_integrand
                        const double df = fmin(fmax(fma(-sg, f0, 1.) * G, -hi), hi);
                        r = fma(r, df, r);
                    }
                    if (POSITIVE && r < 0.) r = 0.;
                    cell[q] = fma(nd[2], r, cell[q]);
                }
            }
        }
#pragma unroll
        for (int q = 0; q < kSpecPts; q++) acc[q] += cell[q];
    }
#pragma unroll
    for (int q = 0; q < kSpecPts; q++) {
        const int pt = base + 64 * q;
        if (pt < npts) a.partial[(static_cast<int64_t>(blockIdx.x) * a.ns + si) * npts + pt] = acc[q];
    }
}

// g / (2 pi hbar c)^3
__device__ __forceinline__ double spectra_pref(int g) {
    return static_cast<double>(g) / (8. * kPi * kPi * kPi) / (kHbarC * kHbarC * kHbarC);
}

// out[slice][i] = the sum over the slice's chunks (blockIdx.y, `per` chunks
// each), in a fixed order: 64 consecutive outputs per workgroup, its four
// waves take every fourth chunk.  Two launches (slices, then the slices'
// sums) keep the whole chip loading where one thread per output would walk
// all chunks alone (911 chunks x 2160 outputs: 221 us, now 2 x 9 us for 4546 chunks).
// species (npts outputs each): the last sums of species that share none, times
// their prefactors (k_spectra_spread without a launch of its own); null: plain sums.
__global__ __launch_bounds__(256) void k_spectra_reduce(const double* __restrict__ partial, int64_t nchunks,
                                                        int64_t per, int64_t n, const int32_t* __restrict__ species,
                                                        const int* __restrict__ g, int64_t npts,
                                                        double* __restrict__ out) {
    __shared__ double s_sum[4][64];
    const int lane = threadIdx.x % 64, w = threadIdx.x / 64;
    const int64_t i = static_cast<int64_t>(blockIdx.x) * 64 + lane;
    const int64_t t0 = blockIdx.y * per, t1 = min<int64_t>(nchunks, t0 + per);
    double s = 0.;
    if (i < n) {
#pragma unroll 8
        for (int64_t t = t0 + w; t < t1; t += 4) s += partial[t * n + i];
    }
    s_sum[w][lane] = s;
    __syncthreads();
    if (w == 0 && i < n) {
        const double v = (s_sum[0][lane] + s_sum[1][lane]) + (s_sum[2][lane] + s_sum[3][lane]);
        out[blockIdx.y * n + i] = species ? v * spectra_pref(g[species[i / npts]]) : v;
    }
}

// out[s] = g_s / (2 pi hbar c)^3 times the sum of the species it shares its
// integrand with (pick[s], an index into the evaluated species)
__global__ void k_spectra_spread(const double* __restrict__ sum, const int32_t* __restrict__ species,
                                 const int32_t* __restrict__ pick, const int* __restrict__ g, int64_t npts, int64_t n,
                                 double* __restrict__ out) {
    const int64_t i = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const int64_t s = i / npts;
    out[i] = sum[pick[s] * npts + (i - s * npts)] * spectra_pref(g[species[s]]);
}

}  // namespace issdev
