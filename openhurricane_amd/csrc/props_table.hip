// props_table.hip -- mixture thermo, transport and temperature recovery for
// run-time mechanism tables, one cell per lane.
//
// The pair sums of Wilke's rule and of the mixture-averaged diffusivities are
// rewritten so that everything that depends on the pair alone is a table
// entry (PairTab, built once per context):
//   Wilke   phi_i = sum_j P_ij x_j (1 + sqrt(mu_i / mu_j sqrt(W_j / W_i)))^2
//                 = (P x)_i + 2 a_i (P xb)_i + a_i^2 (P xb^2)_i,
//           a = sqrt(mu) W^(-1/4), b = 1 / a
//   D_im    sum_j x_j / D_ij = (T^-0.145 sum_j A_ij x_j + sum_j C_ij x_j /
//           (T R_ij + 1/2)^2) / (T^1.5 / p),  A_ij = C_ij R_ij^-0.145
// (R_ij = 1 / sqrt(ek_i ek_j); all terms positive, so nothing cancels): three
// fused multiply-adds per pair for Wilke, one for the power term, and the
// rational term adds up eight fractions over one common denominator, so that
// eight pairs share one reciprocal.  No logarithm, exponential, square root
// or division is left per pair; the wavefront-per-cell form before evaluated
// an exp, a log, three square roots and four divisions for each.
//
// The row i of the tables is wave-uniform (scalar loads, eight columns of all
// four tables contiguous) and the sum over j is unrolled over the padded
// species count, so x_j, x_j b_j and x_j b_j^2 stay in registers; a_i, read
// once per row, is kept in LDS.
#include "wave_dispatch.hpp"
#include "wave_kernels.hpp"

namespace ohcd {

namespace {

template <int NSP>
__global__ __launch_bounds__(64, NSP <= 32 ? 3 : 1) void props_table_kernel(const PropParams P, const WMech M,
                                                         const PairTab pt) {
    // x, x b and x b^2 in registers up to 16 species; above, x and b, with one
    // more multiplication per pair, so that three wavefronts share a SIMD and hide the
    // scalar loads of the rows (32 species, 262,147 cells: 514 us with x, x b, x b^2
    // at one wavefront, 385 us so)
    constexpr bool kThree = NSP <= 16;
    __shared__ double s_a[NSP][64];
    const int lane = threadIdx.x, ns = M.ns;
    const int64_t c0 = (int64_t)blockIdx.x * 64;
    const bool in = c0 + lane < P.n;
    const int64_t cell = in ? c0 + lane : P.n - 1;  // the last lanes repeat the last cell
    ctab *S = as_ctab(M.sp);
    const double T = P.T[cell], p = P.p[cell];
    const bool transport = P.mu || P.kappa || P.Dk;
    const double sqT = sqrt(T), Tp = exp(-0.145 * log(T));
    double x0[NSP], x1[NSP], x2[kThree ? NSP : 1];
    double wm = 0.0;
#pragma unroll
    for (int j = 0; j < NSP; ++j) {
        x0[j] = j < ns ? P.Y[j * P.ldY + cell] : 0.0;
        wm += x0[j] * S[SP_IW * 64 + j];
    }
    const double rwm = 1.0 / fmax(wm, kVeryTiny);
    double rx = 1.0;
    if (transport) {
        // mole fractions (speciesList.cpp:208-222) and viscosities
        double xt = 0.0;
#pragma unroll
        for (int j = 0; j < NSP; ++j) {
            x0[j] = fmax(0.0, fmin(1.0, x0[j] * rwm * S[SP_IW * 64 + j]));
            if (ns == 1) x0[j] = j == 0 ? 1.0 : 0.0;
            xt += x0[j];
        }
        if (xt != 1.0) rx = 1.0 / xt;
#pragma unroll
        for (int j = 0; j < NSP; ++j) {
            x0[j] *= rx;
            // kineticTheory::mu (kineticTheory.cpp:37-57): Omega22 over one
            // denominator
            const double e1 = fma(T, S[SP_IEK * 64 + j], 0.5), e = e1 * e1;
            const double mu = S[SP_MUC * 64 + j] * sqT * (e * frcp(fma(S[SP_OMC * 64 + j] * Tp, e, 1.0)));
            const double r = frsq(mu);
            s_a[j][lane] = mu * r * S[SP_W4 * 64 + j];
            const double b = r * S[SP_IW4 * 64 + j];
            if constexpr (kThree) {
                x1[j] = x0[j] * b;
                x2[j] = x1[j] * b;
            } else {
                x1[j] = b;
            }
        }
    }
    double cpm = 0.0, ham = 0.0, mum = 0.0, km = 0.0;
    const double dT = T * sqT / p;
    for (int i = 0; i < ns; ++i) {
        const double y = P.Y[i * P.ldY + cell];
        double cp, h;
        species_cp_h(S, i, T, cp, h);
        cpm += cp * y;
        ham += h * y;
        if (P.hk && in) P.hk[i * P.ldD + cell] = h;
        if (!transport) continue;
        const double a = s_a[i][lane];
        ctab *row = as_ctab(pt.t) + (size_t)i * PairTab::kRow;
        double s0 = 0.0, s1 = 0.0, s2 = 0.0, sa = 0.0, sr = 0.0;
#pragma unroll
        for (int jb = 0; jb < NSP / 8; ++jb) {
            ctab *q = row + jb * 32;
            double nu[8], de[8];
#pragma unroll
            for (int e = 0; e < 8; ++e) {
                const int j = jb * 8 + e;
                if constexpr (kThree) {
                    s0 = fma(q[e], x0[j], s0);
                    s1 = fma(q[e], x1[j], s1);
                    s2 = fma(q[e], x2[j], s2);
                } else {
                    const double t = fma(a, x1[j], 1.0);
                    s0 = fma(q[e] * x0[j], t * t, s0);
                }
                sa = fma(q[8 + e], x0[j], sa);
                const double d = fma(T, q[16 + e], 0.5);
                de[e] = d * d;
                nu[e] = q[24 + e] * x0[j];
            }
            // nu_0 / de_0 + ... + nu_7 / de_7 over one denominator
#pragma unroll
            for (int w = 1; w < 8; w *= 2)
#pragma unroll
                for (int e = 0; e < 8; e += 2 * w) {
                    nu[e] = fma(nu[e], de[e + w], nu[e + w] * de[e]);
                    de[e] *= de[e + w];
                }
            sr = fma(nu[0], frcp(de[0]), sr);
        }
        // mole fraction of this row's species, as above
        double x = fmax(0.0, fmin(1.0, y * rwm * S[SP_IW * 64 + i])) * rx;
        if (ns == 1) x = 1.0;
        if (P.mu || P.kappa) {
            const double phi = kThree ? fma(a, fma(a, s2, 2.0 * s1), s0) : s0;
            const double t = x * (a * a * S[SP_SQW * 64 + i]) * frcp(phi);  // x mu / phi
            mum += t;
            km += t * (cp + 1.25 * (kRu * S[SP_IW * 64 + i]));
        }
        if (P.Dk && in) {
            double Dim = x < 1.0 - kVeryTiny ? (1.0 - x) * dT / fma(Tp, sa, sr) : 0.0;
            if (isinf(Dim)) Dim = 0.0;
            P.Dk[i * P.ldD + cell] = Dim;
        }
    }
    if (!in) return;
    if (P.cp) P.cp[cell] = cpm;
    if (P.ha) P.ha[cell] = ham;
    if (P.mu) P.mu[cell] = mum;
    if (P.kappa) P.kappa[cell] = km;
    // perfect gas: cv = cp - Rm, ea = ha - Rm T (thermoList.inl:145-156, :289-298)
    const double Rm = ns == 1 ? kRu * S[SP_IW * 64] : kRu * fmax(wm, kVeryTiny);
    if (P.cv) P.cv[cell] = cpm - Rm;
    if (P.ea) P.ea[cell] = ham - Rm * T;
}

// thermoList::T (thermoList.cpp:504-533) for run-time tables, one lane per
// cell.  The Newton iteration needs h and cp of the mixture at a handful of
// temperatures but the composition never changes, so the NASA-7 coefficients
// are mixed once per range (Y read once, 12 fused multiply-adds per species)
// and an iteration evaluates one polynomial.  That holds where one
// range covers every species: T within [Tmin, Tmax] = [max Tlow, min Thigh] and
// one Tcommon for all; elsewhere (uniform = 0, or a lane outside) the species
// are summed one by one.
__global__ __launch_bounds__(256) void tfromh_table_kernel(const ThParams P, const WMech M,
                                                           const int uniform, const double Tmin,
                                                           const double Tmax) {
    const int64_t cell = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (cell >= P.n) return;
    ctab *S = as_ctab(M.sp);
    const int ns = M.ns;
    const double hstar = P.h[cell];
    const double T0 = P.T[cell], Ttol = T0 * 1.0e-4;
    double lo[6] = {}, hi[6] = {}, wm = 0.0;
#pragma unroll 8
    for (int k = 0; k < ns; ++k) {
        const double y = P.Y[k * P.ldY + cell];
#pragma unroll
        for (int m = 0; m < 6; ++m) {
            lo[m] = fma(y, S[(SP_ALO + m) * 64 + k], lo[m]);
            hi[m] = fma(y, S[(SP_AHI + m) * 64 + k], hi[m]);
        }
        wm = fma(y, S[SP_IW * 64 + k], wm);
    }
    // TEa: F = ha - Rm T, dF/dT = cp - Rm (thermoList.inl:343-370)
    const double Rm = !P.energy ? 0.0 : ns == 1 ? kRu * S[SP_IW * 64] : kRu * fmax(wm, kVeryTiny);
    const double Tc = S[SP_TCOM * 64];
    double Test = T0, Tnew = T0;
    int iter = 0, flag = 1;
    do {
        Test = Tnew;
        double hm, cpm;
        if (uniform && Test >= Tmin && Test <= Tmax) {
            const bool l = Test < Tc;
            double a[6];
#pragma unroll
            for (int m = 0; m < 6; ++m) a[m] = l ? lo[m] : hi[m];
            const double T = Test;
            cpm = (((a[4] * T + a[3]) * T + a[2]) * T + a[1]) * T + a[0];
            hm = ((((a[4] * 0.2 * T + a[3] * 0.25) * T + a[2] * (1.0 / 3.0)) * T + a[1] * 0.5) * T +
                  a[0]) * T + a[5];
        } else {
            hm = cpm = 0.0;
            for (int k = 0; k < ns; ++k) {
                double cp, h;
                species_cp_h(S, k, Test, cp, h);
                const double y = P.Y[k * P.ldY + cell];
                hm += h * y;
                cpm += cp * y;
            }
        }
        if (P.energy) {
            hm -= Rm * Test;
            cpm -= Rm;
        }
        double Tn = Test - (hm - hstar) / cpm;
        if (Tn < P.Tlow) {
            flag = 0;
            Tn = P.Tlow;
        } else if (Tn > P.Thigh) {
            flag = 2;
            Tn = P.Thigh;
        } else {
            flag = 1;
        }
        Tnew = Tn;
        if (iter++ > 100) break;
    } while (fabs(Tnew - Test) > Ttol);
    P.T[cell] = Tnew;
    if (P.iflag) P.iflag[cell] = flag;
}

}  // namespace

hipError_t table_props(const PropParams &p, const WMech &m, const PairTab &pt, hipStream_t s) {
    const dim3 g((unsigned)((p.n + 63) / 64)), b(64);
    if (m.ns <= 16) hipLaunchKernelGGL(props_table_kernel<16>, g, b, 0, s, p, m, pt);
    else if (m.ns <= 24) hipLaunchKernelGGL(props_table_kernel<24>, g, b, 0, s, p, m, pt);
    else if (m.ns <= 32) hipLaunchKernelGGL(props_table_kernel<32>, g, b, 0, s, p, m, pt);
    else if (m.ns <= 48) hipLaunchKernelGGL(props_table_kernel<48>, g, b, 0, s, p, m, pt);
    else if (m.ns <= 56) hipLaunchKernelGGL(props_table_kernel<56>, g, b, 0, s, p, m, pt);
    else hipLaunchKernelGGL(props_table_kernel<64>, g, b, 0, s, p, m, pt);
    return hipGetLastError();
}

hipError_t wave_tfromh(const ThParams &p, const WMech &m, hipStream_t s) {
    hipLaunchKernelGGL(tfromh_table_kernel, dim3((unsigned)((p.n + 255) / 256)), dim3(256), 0, s, p,
                       m, m.uniform_range, m.Tmin, m.Tmax);
    return hipGetLastError();
}

}  // namespace ohcd
