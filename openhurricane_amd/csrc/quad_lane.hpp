// quad_lane.hpp -- four cells per wavefront for compiled mechanisms: the
// integrator of quad_kernels.hpp on a compile-time mechanism M, for calls that
// do not fill the chip with one cell per lane.
//
// One lane per cell gives the best throughput, but a Newton iteration of a
// wavefront then takes 10 us, and a stiff H2-air cell needs 17,000 of them: a
// call of 64 cells and one of 65,536 both take as long as their slowest cell.
// With 16 lanes per cell an iteration is spread over the lanes -- species k and row
// k of the Newton matrix in lane k, reactions r and r + 16 in lane r -- and takes
// about 3.5 us.  Nothing but the concentrations goes through LDS:
//   * a reaction lane evaluates its rate constant, the equilibrium constant from
//     the reaction's own summed NASA-7 coefficients, and the partial derivatives
//     of its net rate;
//   * each of those numbers is broadcast to the row of 16 lanes by one DPP move,
//     and lane k adds it, times the stoichiometric coefficient of species k, to
//     its row of J in registers (which entries exist is known at compile time);
//   * the matrix goes straight into the elimination of quad_solve.
// The bound is the dependent chain of one wavefront per SIMD (8,400 cycles an
// iteration: rates 2,200, elimination and back substitution 2,100, checks and
// step control 4,000), so the kernel takes all registers of a SIMD: with two
// wavefronts per SIMD and half the registers 64 cells took 71 ms for 60.
//
// Measured, one flow step of stiff H2-air, one lane per cell -> here, ms: 64
// cells 150 -> 60, 65,536 172 -> 132 (with the sub-steps of the step before 165 ->
// 80), 98,304 172 -> 170 (165 -> 113), 131,072 172 -> 210 (165 -> 151).
#pragma once

#include "quad_kernels.hpp"

namespace ohcd {

// Whether M fits: a row slot per lane, two reactions per lane, rate laws without
// fall-off, orders 1 and 2, one range of validity and one Tcommon for all fits.
template <class M>
constexpr bool quad_fits() {
    if (M::NS > 15 || M::NR > 32 || !uniform_tcommon<M>()) return false;
    for (int k = 1; k < M::NS; ++k)
        if (M::Tlow[k] != M::Tlow[0] || M::Thigh[k] != M::Thigh[0]) return false;
    for (int r = 0; r < M::NR; ++r) {
        const RxnD d = M::R[r];
        if (d.kind > 1 || d.rev > 1 || d.nf > 3 || d.nb > 3) return false;
        for (int i = 0; i < d.nf; ++i)
            if (d.fo[i] != 1.0 && d.fo[i] != 2.0) return false;
        for (int i = 0; i < d.nb; ++i)
            if (d.bo[i] != 1.0 && d.bo[i] != 2.0) return false;
    }
    return true;
}

// Per-lane constants of M, [field][lane of 16] (reactions: [slot][field][lane]).
template <class M>
struct QuadTab {
    static constexpr int NSLOT = (M::NR + 15) / 16;
    enum { F_A, F_B, F_TA, F_REV, F_SUM, F_BASE, F_EFF, F_NASA = F_EFF + M::NS, F_N = F_NASA + 14 };
    enum { P_W, P_TLO, P_THI, P_LO, P_HI = P_LO + 6, P_N = P_HI + 6 };
    double rx[NSLOT][F_N][16];
    double sp[P_N][16];
    double nu[M::NR][16];          // net coefficient of species lane in reaction r
    int idx[NSLOT][6][16];         // participants (NS: absent, concentration 1)
    unsigned sq[NSLOT][16];        // bit i: order of participant i is 2
};
template <class M>
constexpr QuadTab<M> quad_tab() {
    QuadTab<M> t{};
    using Q = QuadTab<M>;
    for (int r = 0; r < Q::NSLOT * 16; ++r) {
        const int s = r / 16, l = r % 16;
        for (int i = 0; i < 6; ++i) t.idx[s][i][l] = M::NS;
        t.rx[s][Q::F_BASE][l] = 1.0;
        if (r >= M::NR) continue;
        const RxnD d = M::R[r];
        t.rx[s][Q::F_A][l] = d.A;
        t.rx[s][Q::F_B][l] = d.b;
        t.rx[s][Q::F_TA][l] = d.Ta;
        t.rx[s][Q::F_REV][l] = d.rev;
        t.rx[s][Q::F_SUM][l] = d.sumStoi;
        if (d.kind == 1) {
            t.rx[s][Q::F_BASE][l] = 0.0;
            for (int k = 0; k < M::NS; ++k) t.rx[s][Q::F_EFF + k][l] = M::EFF[d.tb][k];
        }
        for (int i = 0; i < d.nf; ++i) {
            t.idx[s][i][l] = d.fi[i];
            if (d.fo[i] == 2.0) t.sq[s][l] |= 1u << i;
        }
        for (int i = 0; i < d.nb; ++i) {
            t.idx[s][3 + i][l] = d.bi[i];
            if (d.bo[i] == 2.0) t.sq[s][l] |= 1u << (3 + i);
        }
        for (int m = 0; m < 7; ++m) {
            double lo = 0.0, hi = 0.0;
            for (int i = 0; i < d.nf; ++i) {
                lo -= d.fnu[i] * M::W[d.fi[i]] * M::alo[d.fi[i]][m];
                hi -= d.fnu[i] * M::W[d.fi[i]] * M::ahi[d.fi[i]][m];
            }
            for (int i = 0; i < d.nb; ++i) {
                lo += d.bnu[i] * M::W[d.bi[i]] * M::alo[d.bi[i]][m];
                hi += d.bnu[i] * M::W[d.bi[i]] * M::ahi[d.bi[i]][m];
            }
            t.rx[s][Q::F_NASA + m][l] = lo;
            t.rx[s][Q::F_NASA + 7 + m][l] = hi;
        }
        for (int i = 0; i < d.nf; ++i) t.nu[r][d.fi[i]] -= d.fnu[i];
        for (int i = 0; i < d.nb; ++i) t.nu[r][d.bi[i]] += d.bnu[i];
    }
    for (int k = 0; k < M::NS; ++k) {
        t.sp[Q::P_W][k] = M::W[k];
        t.sp[Q::P_TLO][k] = M::Tlow[k];
        t.sp[Q::P_THI][k] = M::Thigh[k];
        for (int m = 0; m < 6; ++m) {
            t.sp[Q::P_LO + m][k] = M::alo[k][m] * M::W[k];
            t.sp[Q::P_HI + m][k] = M::ahi[k][m] * M::W[k];
        }
    }
    return t;
}
template <class M>
__device__ constexpr QuadTab<M> kQuadTab = quad_tab<M>();

template <class M, int FLOW>
struct CompiledSys {
    using Params = LaneParams;
    static constexpr int NS = M::NS, kN = NS + 1, S = 1, kWavesPerSimd = 1;
    using T = QuadTab<M>;
    struct Lds : QuadLDS<kN> {
        double rx[T::NSLOT][T::F_N][16], sp[T::P_N][16];
        double conc[4][NS + 1];
    };
    int ns;
    double W[1];
    double nu[M::NR];
    int idx[T::NSLOT][6];
    unsigned sq[T::NSLOT];

    static __device__ __forceinline__ const LaneParams &lane(const Params &p) { return p; }
    __device__ __forceinline__ void init(const Params &, Lds &L) {
        const int c = threadIdx.x & 15;
        const QuadTab<M> &t = kQuadTab<M>;
        ns = NS;
        W[0] = c < NS ? t.sp[T::P_W][c] : 1.0;
        for (int e = threadIdx.x; e < T::NSLOT * T::F_N * 16; e += 64) (&L.rx[0][0][0])[e] = (&t.rx[0][0][0])[e];
        for (int e = threadIdx.x; e < T::P_N * 16; e += 64) (&L.sp[0][0])[e] = (&t.sp[0][0])[e];
        if (c == 0) L.conc[threadIdx.x >> 4][NS] = 1.0;
        sfor<0, M::NR>([&](auto r) { nu[r] = t.nu[r][c]; });
#pragma unroll
        for (int s = 0; s < T::NSLOT; ++s) {
#pragma unroll
            for (int i = 0; i < 6; ++i) idx[s][i] = t.idx[s][i][c];
            sq[s] = t.sq[s][c];
        }
        __syncthreads();
    }

    __device__ __forceinline__ void step(const Params &P, Lds &L, const double (&yk)[1], double Tk,
                                         const double (&y0)[1], double y0T, double h, bool act,
                                         QuadF<1> &o, double (&x)[1], double &xT) {
        constexpr int NSLOT = T::NSLOT;
        const int c = threadIdx.x & 15, g = threadIdx.x >> 4;
        const double ci = fmax(yk[0], 0.0);
        if (c < NS) L.conc[g][c] = ci;
        __builtin_amdgcn_wave_barrier();
        // ---- temperature factors, rate and equilibrium constants ----
        const double Tm = fmax(Tk, kTiny), lnT = log_pos(Tm), invT = frcp(Tk), invTm = frcp(Tm),
                     invRuT = invTm * (1.0 / kRu);
        constexpr double kLnPR = 2.5003366899611787;  // ln(Patm / Ru)
        const double lnX = kLnPR - lnT;
        const bool lo = Tk < M::Tcommon[0];
        const bool out = __any(Tk < tlow_max<M>() || Tk > thigh_min<M>());
        double q[NSLOT], s[NSLOT], gam[NSLOT], df[NSLOT][3], db[NSLOT][3];
#pragma unroll
        for (int m = 0; m < NSLOT; ++m) {
            const double(*R)[16] = L.rx[m];
            double cf[3], cb[3];
#pragma unroll
            for (int i = 0; i < 3; ++i) {
                cf[i] = L.conc[g][idx[m][i]];
                cb[i] = L.conc[g][idx[m][3 + i]];
            }
            const double b = R[T::F_B][c], Ta = R[T::F_TA][c], sum = R[T::F_SUM][c];
            const bool rev = R[T::F_REV][c] != 0.0;
            // third-body concentration (1 without one)
            double Mt = R[T::F_BASE][c];
            sfor<0, NS>([&](auto k) { Mt = fma(R[T::F_EFF + k][c], rbcast<k>(ci), Mt); });
            const double kf = Mt * (R[T::F_A][c] * exp(b * lnT - Ta * invT));
            // G = sum nu_k G_k; inside every fit's range dG/dT = -S
            const double(*a)[16] = R + T::F_NASA + (lo ? 0 : 7);
            const double a0 = a[0][c], a1 = a[1][c], a2 = a[2][c], a3 = a[3][c], a4 = a[4][c];
            const double st = ((((a4 * 0.25) * Tk + a3 * (1.0 / 3.0)) * Tk + a2 * 0.5) * Tk + a1) * Tk +
                              a0 * lnT + a[6][c];
            const double G = ((((a4 * -0.05 * Tk - a3 * (1.0 / 12.0)) * Tk - a2 * (1.0 / 6.0)) * Tk -
                               a1 * 0.5) * Tk + a0 * (1.0 - lnT) - a[6][c]) * Tk + a[5][c];
            double dG = -st;
            if (out) {
                // past a fit's range cp is that of its end (JANAF.cpp:155-212)
                const double Tx = fmin(fmax(Tk, tlow_max<M>()), thigh_min<M>());
                const double cx = (((a4 * Tx + a3) * Tx + a2) * Tx + a1) * Tx,
                             ct = (((a4 * Tk + a3) * Tk + a2) * Tk + a1) * Tk;
                dG += Tx != Tk ? cx - ct : 0.0;
            }
            // 1 / Kc (reactionTypes.cpp:178-241)
            const double rK = rev ? fmin(exp(G * invRuT - sum * lnX), kVeryLarge) : 0.0;
            const double kr = rK < kVeryLarge ? kf * rK : 0.0;
            double dk = (dG - G * invTm) * invRuT;
            if (P.exact_dkp) dk = -dk;
            const double pf0 = sq[m] & 1u ? cf[0] * cf[0] : cf[0], pf1 = sq[m] & 2u ? cf[1] * cf[1] : cf[1],
                         pf2 = sq[m] & 4u ? cf[2] * cf[2] : cf[2], pb0 = sq[m] & 8u ? cb[0] * cb[0] : cb[0],
                         pb1 = sq[m] & 16u ? cb[1] * cb[1] : cb[1],
                         pb2 = sq[m] & 32u ? cb[2] * cb[2] : cb[2];
            const double prf = pf0 * pf1 * pf2, prb = pb0 * pb1 * pb2;
            q[m] = kf * prf - kr * prb;
            df[m][0] = kf * (sq[m] & 1u ? cf[0] + cf[0] : 1.0) * (pf1 * pf2);
            df[m][1] = kf * (sq[m] & 2u ? cf[1] + cf[1] : 1.0) * (pf0 * pf2);
            df[m][2] = kf * (sq[m] & 4u ? cf[2] + cf[2] : 1.0) * (pf0 * pf1);
            db[m][0] = kr * (sq[m] & 8u ? cb[0] + cb[0] : 1.0) * (pb1 * pb2);
            db[m][1] = kr * (sq[m] & 16u ? cb[1] + cb[1] : 1.0) * (pb0 * pb2);
            db[m][2] = kr * (sq[m] & 32u ? cb[2] + cb[2] : 1.0) * (pb0 * pb1);
            gam[m] = q[m] * frcp(fmax(Mt, kTiny));
            const double dkf = kf * invTm * (b + Ta * invTm);
            const double dkr = dkf * rK - kr * (dk - sum * invT);
            s[m] = dkf * prf - (rev ? dkr * prb : 0.0);
            if (bad(s[m])) s[m] = 0.0;
        }
        // ---- species thermo (JANAF.cpp:155-217), molar ----
        double dCp = 0.0;
        o.H[0] = o.C[0] = 0.0;
        if (c < NS) {
            const double Tl = L.sp[T::P_TLO][c], Th = L.sp[T::P_THI][c];
            const double(*a)[16] = L.sp + (lo ? T::P_LO : T::P_HI);
            const double a0 = a[0][c], a1 = a[1][c], a2 = a[2][c], a3 = a[3][c], a4 = a[4][c];
            const double Tx = fmin(fmax(Tk, Tl), Th);
            const double Cp = (((a4 * Tx + a3) * Tx + a2) * Tx + a1) * Tx + a0;
            const double H = ((((a4 * 0.2 * Tx + a3 * 0.25) * Tx + a2 * (1.0 / 3.0)) * Tx + a1 * 0.5) * Tx +
                              a0) * Tx + a[5][c] + Cp * (Tk - Tx);
            dCp = a1 + Tk * (2.0 * a2 + Tk * (3.0 * a3 + 4.0 * a4 * Tk));
            o.H[0] = FLOW == 0 ? H : H - kRu * Tk;
            o.C[0] = FLOW == 0 ? Cp : Cp - kRu;
        }
        // ---- this lane's row of J and omega ----
        double J[NS + 1], w = 0.0, u[M::NTB > 0 ? M::NTB : 1];
        sfor<0, NS + 1>([&](auto j) { J[j] = 0.0; });
        sfor<0, M::NTB>([&](auto t) { u[t] = 0.0; });
        sfor<0, M::NR>([&](auto rc) {
            constexpr int r = rc, m = r / 16, l = r % 16;
            constexpr RxnD d = M::R[r];
            w = fma(nu[r], rbcast<l>(q[m]), w);
            J[NS] = fma(nu[r], rbcast<l>(s[m]), J[NS]);
            sfor<0, d.nf>([&](auto i) {
                constexpr int j = d.fi[i];
                J[j] = fma(nu[r], rbcast<l>(df[m][i]), J[j]);
            });
            if constexpr (d.rev != 0)
                sfor<0, d.nb>([&](auto i) {
                    constexpr int j = d.bi[i];
                    J[j] = fma(-nu[r], rbcast<l>(db[m][i]), J[j]);
                });
            if constexpr (d.kind == 1) u[d.tb] = fma(nu[r], rbcast<l>(gam[m]), u[d.tb]);
        });
        sfor<0, M::NTB>([&](auto t) {
            sfor<0, NS>([&](auto j) {
                constexpr double e = M::EFF[t][j];
                if constexpr (e != 0.0) J[j] = fma(u[t], e, J[j]);
            });
        });
        o.w[0] = w;
        o.rcC = frcp(gsum(yk[0] * o.C[0]));
        o.dT = gsum(w * o.H[0]) * o.rcC;
        o.dcC = gsum(yk[0] * dCp);
        // ---- Newton system ----
        const double b[1] = {c < NS ? -yk[0] + y0[0] + h * w : 0.0};
        const double bT = -Tk + y0T + h * -o.dT;
        auto jac = [&](int, auto j) __attribute__((always_inline)) { return J[j]; };
        auto put = [&]() {
            if (c < NS)
                sfor<0, NS + 1>([&](auto j) { L.J[g * QuadShape<kN>::CST + c * QuadShape<kN>::JS + j] = J[j]; });
        };
        quad_solve<kN>(L, jac, put, h, b, bT, o, act, x, xT);
    }
};

// Integrator launch for small calls (ImplicitEuler, FP64); cells: per wavefront.
template <class M>
hipError_t launch_quad_lane(const LaneParams &p, int grid, hipStream_t s) {
    if constexpr (quad_fits<M>()) {
        if (p.flow == 0)
            hipLaunchKernelGGL((ie_quad_kernel<CompiledSys<M, 0>>), dim3(grid), dim3(64), 0, s, p);
        else
            hipLaunchKernelGGL((ie_quad_kernel<CompiledSys<M, 1>>), dim3(grid), dim3(64), 0, s, p);
        return hipGetLastError();
    } else {
        return hipErrorNotSupported;
    }
}
template <class M>
const void *quad_lane_fn() {
    if constexpr (quad_fits<M>()) return (const void *)&ie_quad_kernel<CompiledSys<M, 0>>;
    else return nullptr;
}

}  // namespace ohcd
