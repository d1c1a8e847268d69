// quad_kernels.hpp -- integrator with four cells per wavefront, 16 lanes each,
// for mechanisms of up to 15 species: on run-time tables (TableSys, here) and on
// compiled mechanisms (CompiledSys, quad_lane.hpp).
//
// Why 16 lanes per cell.  A cell's Newton iteration is one Jacobian evaluation
// and one dense solve, a serial chain whose length is all that a call of few
// cells sees.  gfx950 moves a 64-bit value from one lane to the 16 lanes of its
// row in a single vector instruction (v_mov_b64_dpp row_newbcast), so a matrix
// with row i in lane i of the group is eliminated with one move and one FMA per
// pivot-row element, for four cells at once; one wavefront per cell needs a pair
// of v_readlane per element and leaves 52 lanes idle, one lane per cell runs
// every element of the matrix one after the other.  Reactions are evaluated 16
// at a time in each group.  Above 16 rows a lane holds two rows and the LDS holds
// two wavefronts per SIMD at most: at 33 rows that measured no better than one
// wavefront per cell (440 against 445 ms on 524,288 cells), so those sizes stay
// there.
//
// The elimination order is fixed (lane numbers of DPP broadcasts are
// immediates): Gauss-Jordan without row exchanges on the species block of
// I - h J, the temperature row and column bordered.  Every solution is checked
// against the system itself (componentwise backward error, kQuadBackward);
// a system that fails is factored again with partial pivoting
// (quad_solve_pivoted), so a Newton update is never taken from a solve that
// was not verified.
//
// Control flow is that of ie_lane_kernel with a group of 16 lanes in the place
// of a lane: each group holds one cell, takes the wavefront-wide evaluation and
// solve together with the other three, and refills from the work queue by
// itself.  References as in wave_kernels.hpp.
//
// Measured, one ImplicitEuler flow step of the H2-air tables (9 species, 19
// reactions), one wavefront per cell -> four cells per wavefront: 65,536 cells
// 445 -> 278 ms, 32,768 289 -> 240, 8,192 221 -> 209, 4,096 190 -> 187, but 2,048
// 168 -> 187 and 64 140 -> 151: few cells leave the chip idle either way, and the
// 64-lane reaction loop of one cell is the shorter chain (kQuadTableMin).
#pragma once

#include "wave_kernels.hpp"

namespace ohcd {

// largest ODE size (species + 1) of the four-cell kernels
constexpr int kQuadMaxN = 16;
// smallest call that takes them on a run-time mechanism table
constexpr int64_t kQuadTableMin = 4096;

template <int N>
struct QuadShape {
    static constexpr int NS = N - 1;            // species rows and columns
    static constexpr int S = (NS + 15) / 16;    // row slots of a lane
    static constexpr int JS = N | 1;            // row stride of J in LDS (odd: a lane per row
                                                // reads distinct banks)
    // cell stride: a multiple of 16 bytes that puts neighbouring groups on the
    // two halves of the 64 banks
    static constexpr int CST = (N * JS + 15) / 32 * 32 + 16;
    static constexpr int VS = (N + 1) / 2 * 2 + 2;  // stride of the species vectors
};

template <int N>
struct QuadLDS {
    using Q = QuadShape<N>;
    static_assert(Q::CST >= N * Q::JS && Q::CST % 2 == 0, "cell stride");
    // row i: d(omega_i)/dc_j in columns 0..NS-1, d(omega_i)/dT in column NS
    double __attribute__((aligned(16))) J[4 * Q::CST];
    double c[4][Q::VS], G[4][Q::VS], dG[4][Q::VS], w[4][Q::VS];
    double gam[4][18];
};

// value of lane L of this lane's row of 16
template <int L>
__device__ __forceinline__ double rbcast(double v) {
    const long long x = __builtin_bit_cast(long long, v);
    const long long r = __builtin_amdgcn_update_dpp(0ll, x, 0x150 + L, 0xf, 0xf, true);
    return __builtin_bit_cast(double, r);
}
// sum / maximum over the 16 lanes of a row, in every lane of it
__device__ __forceinline__ double gsum(double v) {
    v += dpp<kDppXor1>(v);
    v += dpp<kDppXor2>(v);
    v += dpp<kDppHalfMirror>(v);
    v += dpp<kDppMirror>(v);
    return v;
}
__device__ __forceinline__ double gmax(double v) {
    v = fmax(v, dpp<kDppXor1>(v));
    v = fmax(v, dpp<kDppXor2>(v));
    v = fmax(v, dpp<kDppHalfMirror>(v));
    v = fmax(v, dpp<kDppMirror>(v));
    return v;
}
// whether any lane of this lane's row of 16 has x
__device__ __forceinline__ bool gany(bool x) {
    return ((__builtin_amdgcn_ballot_w64(x) >> (threadIdx.x & 48u)) & 0xffffull) != 0ull;
}

// What the Newton system needs of one evaluation, besides J in LDS.
template <int S>
struct QuadF {
    double w[S];           // omega of the lane's species
    double H[S], C[S];     // molar enthalpy / heat capacity (internal energy / Cv at constant
                           // volume) of the lane's species, 0 past ns
    double dT, rcC, dcC;   // f_T = -dT; 1 / sum c C; sum c dCp/dT
};

// dy/dt and J of each group's cell at (y, T): species c + 16 s in slot s.
template <int N, int FLOW>
__device__ __forceinline__ void quad_eval(const WMech &M, QuadLDS<N> &L,
                                          const double (&y)[QuadShape<N>::S], double T, int exact,
                                          QuadF<QuadShape<N>::S> &o) {
    using Q = QuadShape<N>;
    constexpr int S = Q::S, NS = Q::NS;
    const int lane = threadIdx.x, c = lane & 15, g = lane >> 4, ns = M.ns;
    double *Jg = L.J + g * Q::CST;
    const TFac tf = tfac(T);
    double dCp[S];
#pragma unroll
    for (int s = 0; s < S; ++s) {
        const int k = c + 16 * s;
        o.H[s] = o.C[s] = dCp[s] = 0.0;
        if (k < ns) {
            double G, dG, Cp, H;
            wthermo(M, k, tf, G, dG, Cp, H, dCp[s]);
            L.c[g][k] = fmax(y[s], 0.0);
            L.G[g][k] = G;
            L.dG[g][k] = dG;
            o.H[s] = FLOW == 0 ? H : H - kRu * T;
            o.C[s] = FLOW == 0 ? Cp : Cp - kRu;
        }
        if (k < NS) L.w[g][k] = 0.0;
    }
    {
        double2 *z = (double2 *)L.J;
        constexpr int NZ = 4 * Q::CST / 2;
#pragma unroll 4
        for (int e = lane; e < NZ; e += 64) z[e] = double2{0.0, 0.0};
    }
    __syncthreads();
    const RxnTab tb = rxn_tab(M);
    for (int base = 0; base < M.nr; base += 16) {
        const int tl = (base & 48) + c, r = base + c;  // lane of the 64-reaction table chunk
        double gam = 0.0;
        WRxn x;
        x.nf = x.nb = 0;
        if (r < M.nr) {
            wreaction<true>(M, base >> 6, tl, tf, L.c[g], L.G[g], L.dG[g], exact, x);
#pragma unroll
            for (int side = 0; side < 2; ++side) {
#pragma unroll
                for (int i = 0; i < kWP; ++i) {
                    const bool has = side == 0 ? i < x.nf : i < x.nb;
                    if (!has) continue;
                    const int a = side == 0 ? x.fi[i] : x.bi[i];
                    const double nu = side == 0 ? -x.fnu[i] : x.bnu[i];
                    lds_add(&L.w[g][a], nu * x.q);
                    double *row = Jg + a * Q::JS;
#pragma unroll
                    for (int j = 0; j < kWP; ++j) {
                        if (j < x.nf) lds_add(&row[x.fi[j]], nu * x.dqf[j]);
                        if (j < x.nb && x.rev != 0) lds_add(&row[x.bi[j]], -nu * x.dqr[j]);
                    }
                    lds_add(&row[NS], nu * x.s);
                }
            }
            gam = x.gam;
        }
        // third-body / fall-off terms sigma_a gam_r eff_rj: columns c + 16 s in
        // this lane, one reaction of the quarter after another, the four cells
        // together (each with its own gam)
        unsigned long long m4 = __builtin_amdgcn_ballot_w64(gam != 0.0);
        if (m4) {
            L.gam[g][c] = gam;
            unsigned m = (unsigned)(m4 | m4 >> 32);
            m = (m | m >> 16) & 0xffffu;
            __builtin_amdgcn_wave_barrier();
            while (m) {
                const int sl = __builtin_ctz(m);
                m &= m - 1u;
                const double gm = L.gam[g][sl];
                double e[S];
#pragma unroll
                for (int s = 0; s < S; ++s) e[s] = lde_col(tb, base + sl, c + 16 * s) * gm;
                // participants of reaction base + sl: the same in every group
                const int nf = __builtin_amdgcn_readlane(x.nf, sl),
                          nb = __builtin_amdgcn_readlane(x.nb, sl);
#pragma unroll
                for (int i = 0; i < kWP; ++i) {
                    if (i < nf) {
                        double *row = Jg + __builtin_amdgcn_readlane(x.fi[i], sl) * Q::JS;
                        const double nu = -rdlane(x.fnu[i], sl);
#pragma unroll
                        for (int s = 0; s < S; ++s)
                            if (c + 16 * s < NS) lds_add(&row[c + 16 * s], nu * e[s]);
                    }
                    if (i < nb) {
                        double *row = Jg + __builtin_amdgcn_readlane(x.bi[i], sl) * Q::JS;
                        const double nu = rdlane(x.bnu[i], sl);
#pragma unroll
                        for (int s = 0; s < S; ++s)
                            if (c + 16 * s < NS) lds_add(&row[c + 16 * s], nu * e[s]);
                    }
                }
            }
        }
    }
    __syncthreads();
    // temperature equation (chemistrySource.cpp:863-907, :993-1054)
    double cC = 0.0, hw = 0.0, dc = 0.0;
#pragma unroll
    for (int s = 0; s < S; ++s) {
        const int k = c + 16 * s;
        o.w[s] = k < NS ? L.w[g][k] : 0.0;
        cC += y[s] * o.C[s];
        hw += o.w[s] * o.H[s];
        dc += y[s] * dCp[s];
    }
    o.rcC = frcp(gsum(cC));
    o.dT = gsum(hw) * o.rcC;
    o.dcC = gsum(dc);
}

// largest accepted componentwise backward error of an unpivoted solve: its
// Newton update is within this relative distance of an exact solve's for the
// rows' own scales, far below the loosest Newton tolerance in use (1e-6)
constexpr double kQuadBackward = 1e-11;

// Partial-pivoting solve of group gg's system in LDS, all 64 lanes, row i in
// lane i (rolled loops: taken only for a system the unpivoted elimination
// could not solve to kQuadBackward).  In: J of the cell, H, C in L.G / L.dG
// [gg], right-hand side in L.c[gg] (temperature last); out: x in L.w[gg].
template <int N>
__device__ __noinline__ void quad_solve_pivoted(QuadLDS<N> &L, int gg, double h, double dT,
                                                double rcC, double JTT) {
    using Q = QuadShape<N>;
    constexpr int NS = Q::NS;
    const int lane = threadIdx.x;
    double *A = L.J + gg * Q::CST;
    const bool row = lane < N;
    double *Ar = A + (row ? lane : 0) * Q::JS;
    if (lane < NS) {  // d(f_T)/dc_lane into row NS
        double v = 0.0;
        for (int i = 0; i < NS; ++i) v -= A[i * Q::JS + lane] * L.G[gg][i];
        A[NS * Q::JS + lane] = (v + L.dG[gg][lane] * dT) * rcC;
    }
    if (lane == 0) A[NS * Q::JS + NS] = JTT;
    __syncthreads();
    if (row)
        for (int j = 0; j < N; ++j) Ar[j] = -h * Ar[j] + (j == lane ? 1.0 : 0.0);
    double b = row ? L.c[gg][lane] : 0.0;
    __syncthreads();
    bool avail = row, nan_col = false;
    int step = N;
    double rpv = 0.0;
    for (int k = 0; k < N; ++k) {
        const double av = avail ? fabs(Ar[k]) : -1.0;
        const double mx = wmax(isnan(av) ? -1.0 : av);
        const unsigned long long hit = __builtin_amdgcn_ballot_w64(avail && av == mx);
        nan_col = nan_col || hit == 0ull;
        const int p = hit ? __builtin_ctzll(hit) : 0;
        const double rp = frcp(A[p * Q::JS + k]), bp = rdlane(b, p);
        if (hit && lane == p) {
            step = k;
            rpv = rp;
            avail = false;
        }
        const double l = avail ? Ar[k] * rp : 0.0;
        if (avail)
            for (int j = k + 1; j < N; ++j) Ar[j] = fma(-l, A[p * Q::JS + j], Ar[j]);
        b = fma(-l, bp, b);
        __syncthreads();
    }
    for (int k = N - 1; k >= 0; --k) {
        const bool own = step == k;
        const unsigned long long om = __builtin_amdgcn_ballot_w64(own);
        const double t = b * rpv;
        const double xk = rdlane(t, om ? __builtin_ctzll(om) : 0);
        if (step < k) b = fma(-Ar[k], xk, b);
        if (own) L.w[gg][k] = t;
    }
    if (nan_col && row) L.w[gg][lane] = __builtin_nan("");
    __syncthreads();
}

// (I - h J) x = b for the four groups' cells: species rows b, x by slot, the
// temperature row bT, xT in every lane of the group.  act: groups whose
// solution is used (the others solve whatever their LDS holds).
// jac(s, j): J of row slot s, column j (NS: d/dT), a compile-time index.
// to_lds(): puts the group's J into L.J for the pivoted solve.
template <int N, class JAC, class PUT>
__device__ __forceinline__ void quad_solve(QuadLDS<N> &L, JAC &&jac, PUT &&to_lds, double h,
                                           const double (&b)[QuadShape<N>::S], double bT,
                                           const QuadF<QuadShape<N>::S> &o, bool act,
                                           double (&x)[QuadShape<N>::S], double &xT) {
    using Q = QuadShape<N>;
    constexpr int S = Q::S, NS = Q::NS;
    const int lane = threadIdx.x, c = lane & 15, g = lane >> 4;
    double a[S][NS], bb[S], u[S], u0[S], jT[S], rpv[S];
#pragma unroll
    for (int s = 0; s < S; ++s) {
        const int i = c + 16 * s;
        const bool ok = i < NS;
        sfor<0, NS>([&](auto j) {
            // -h J, then + 1 on the diagonal: two roundings, as the reference
            // forms I - h J (ImplicitEuler.cpp:186-193)
#pragma clang fp contract(off)
            const double v = NS % 16 == 0 || ok ? -h * jac(s, j) : 0.0;
            const bool dj = s == j / 16 && __builtin_amdgcn_inverse_ballot_w64(
                                               0x0001000100010001ull << (j % 16));
            a[s][j] = s == j / 16 ? v + (dj ? 1.0 : 0.0) : v;
        });
        jT[s] = NS % 16 == 0 || ok ? jac(s, std::integral_constant<int, NS>{}) : 0.0;
        bb[s] = b[s];
        u0[s] = u[s] = -h * jT[s];
        rpv[s] = 0.0;
    }
    // Gauss-Jordan: every row but the pivot's loses its column k, so that no
    // back substitution follows
    sfor<0, NS>([&](auto kc) {
        constexpr int k = kc, sk = k / 16, ck = k % 16;
        const bool own = __builtin_amdgcn_inverse_ballot_w64(0x0001000100010001ull << ck);
        const double rp = rcp_raw(rbcast<ck>(a[sk][k]));
        double m[S];
#pragma unroll
        for (int s = 0; s < S; ++s) m[s] = -a[s][k] * rp;
        m[sk] = own ? 0.0 : m[sk];
        rpv[sk] = own ? rp : rpv[sk];
        sfor<k + 1, NS>([&](auto j) {
            const double t = rbcast<ck>(a[sk][j]);
#pragma unroll
            for (int s = 0; s < S; ++s) a[s][j] = fma(m[s], t, a[s][j]);
        });
        const double tb = rbcast<ck>(bb[sk]), tu = rbcast<ck>(u[sk]);
#pragma unroll
        for (int s = 0; s < S; ++s) {
            bb[s] = fma(m[s], tb, bb[s]);
            u[s] = fma(m[s], tu, u[s]);
        }
    });
    // Bordered temperature row.  Its species part is
    //   (row) . z = rcC (sum_i H_i (h J z)_i - h dT sum_j C_j z_j),
    // and h J z1 = z1 - b, h J z2 = z2 - u for the two species solutions, so the
    // row itself is never formed.
    double x1[S], x2[S], h1 = 0.0, h2 = 0.0, c1 = 0.0, c2 = 0.0, tt = 0.0;
#pragma unroll
    for (int s = 0; s < S; ++s) {
        x1[s] = bb[s] * rpv[s];
        x2[s] = u[s] * rpv[s];
        h1 += o.H[s] * (x1[s] - b[s]);
        h2 += o.H[s] * (x2[s] - u0[s]);
        c1 += o.C[s] * x1[s];
        c2 += o.C[s] * x2[s];
        tt += o.C[s] * o.w[s] + o.H[s] * jT[s];
    }
    const double hdT = h * o.dT;
    const double v1 = o.rcC * (gsum(h1) - hdT * gsum(c1)), v2 = o.rcC * (gsum(h2) - hdT * gsum(c2));
    const double JTT = (o.dcC * o.dT - gsum(tt)) * o.rcC;
    const double ATT = 1.0 - h * JTT;
    xT = (bT - v1) * frcp(ATT - v2);
#pragma unroll
    for (int s = 0; s < S; ++s) x[s] = x1[s] - x2[s] * xT;
    // backward error of the whole system, component by component, from J
    double jx[S], ax[S];
#pragma unroll
    for (int s = 0; s < S; ++s) {
        jx[s] = jT[s] * xT;
        ax[s] = fabs(jx[s]);
    }
    sfor<0, NS>([&](auto j) {
        const double t = rbcast<j % 16>(x[j / 16]);
#pragma unroll
        for (int s = 0; s < S; ++s) {
            const double v = jac(s, j);
            jx[s] = fma(v, t, jx[s]);
            ax[s] = fma(fabs(v), fabs(t), ax[s]);
        }
    });
    bool bad_row = false;
    double hj = 0.0, ha = 0.0, cx = 0.0, ca = 0.0;
#pragma unroll
    for (int s = 0; s < S; ++s) {
        if (NS % 16 == 0 || c + 16 * s < NS) {
            const double r = b[s] - (x[s] - h * jx[s]);
            const double sc = fabs(b[s]) + fabs(x[s]) + h * ax[s];
            bad_row = bad_row || !(fabs(r) <= kQuadBackward * sc);
            hj += o.H[s] * (jx[s] - jT[s] * xT);
            ha += fabs(o.H[s]) * ax[s];
            cx += o.C[s] * x[s];
            ca += o.C[s] * fabs(x[s]);
        }
    }
    {
        const double vx = o.rcC * h * (gsum(hj) - o.dT * gsum(cx));
        const double va = fabs(o.rcC) * h * (gsum(ha) + fabs(o.dT) * gsum(ca));
        const double r = bT - (ATT * xT + vx);
        const double sc = fabs(bT) + fabs(ATT * xT) + va;
        bad_row = bad_row || !(fabs(r) <= kQuadBackward * sc);
    }
    const bool redo = act && gany(bad_row);
    unsigned long long rm = __builtin_amdgcn_ballot_w64(redo);
    if (rm) {
        if (redo) {
            to_lds();
#pragma unroll
            for (int s = 0; s < S; ++s) {
                const int i = c + 16 * s;
                if (i < NS) {
                    L.G[g][i] = o.H[s];
                    L.dG[g][i] = o.C[s];
                    L.c[g][i] = b[s];
                }
            }
            L.c[g][NS] = bT;
        }
        __syncthreads();
        while (rm) {
            const int l0 = __builtin_ctzll(rm), gg = l0 >> 4;
            rm &= ~(0xffffull << (gg * 16));
            quad_solve_pivoted<N>(L, gg, rdlane(h, l0), rdlane(o.dT, l0), rdlane(o.rcC, l0),
                                  rdlane(JTT, l0));
        }
        if (redo) {
#pragma unroll
            for (int s = 0; s < S; ++s) {
                const int i = c + 16 * s;
                x[s] = i < NS ? L.w[g][i] : 0.0;
            }
            xT = L.w[g][NS];
        }
        __syncthreads();
    }
}

// The system of a run-time mechanism table.
template <int N, int FLOW>
struct TableSys {
    using Params = WaveParams;
    static constexpr int kN = N, S = QuadShape<N>::S, kWavesPerSimd = 2;
    using Lds = QuadLDS<N>;
    int ns;
    double W[S];
    static __device__ __forceinline__ const LaneParams &lane(const Params &p) { return p.L; }
    __device__ __forceinline__ void init(const Params &p, Lds &) {
        ns = p.M.ns;
#pragma unroll
        for (int s = 0; s < S; ++s) {
            const int k = (threadIdx.x & 15) + 16 * s;
            W[s] = k < ns ? p.M.sp[SP_W * 64 + k] : 1.0;
        }
    }
    __device__ __forceinline__ void step(const Params &p, Lds &L, const double (&yk)[S], double ykT,
                                         const double (&y0)[S], double y0T, double h, bool act,
                                         QuadF<S> &o, double (&x)[S], double &xT) {
        using Q = QuadShape<N>;
        const int c = threadIdx.x & 15, g = threadIdx.x >> 4;
        quad_eval<N, FLOW>(p.M, L, yk, ykT, p.exact_dkp, o);
        double b[S];
#pragma unroll
        for (int s = 0; s < S; ++s) b[s] = c + 16 * s < ns ? -yk[s] + y0[s] + h * o.w[s] : 0.0;
        const double bT = -ykT + y0T + h * -o.dT;
        const double *J = L.J + g * Q::CST;
        auto jac = [&](int s, auto j) __attribute__((always_inline)) {
            const int i = c + 16 * s;
            return J[(i < Q::NS ? i : 0) * Q::JS + j];
        };
        quad_solve<N>(L, jac, [] {}, h, b, bT, o, act, x, xT);
    }
};

// Persistent integrator: ImplicitEuler (ImplicitEuler.cpp:40-342) under
// chemistrySource::solve / solveUpdate, four cells per wavefront.
template <class SYS>
__global__ __launch_bounds__(64, SYS::kWavesPerSimd) void ie_quad_kernel(
    const typename SYS::Params WP) {
    constexpr int S = SYS::S;
    const LaneParams &P = SYS::lane(WP);
    const int lane = threadIdx.x, c = lane & 15;
    __shared__ typename SYS::Lds L;
    SYS sys;
    sys.init(WP, L);
    const int ns = sys.ns;
    const double(&W)[S] = sys.W;
    enum { PQ_NEED, PQ_NEWTON, PQ_ERR0, PQ_DONE };
    int phase = PQ_NEED;
    const double errg = pow(P.maxsc / P.safe, -1.0 / P.alpha);
    // the group's cell: step start y0, previous step start yl, Newton iterate
    // yk (species by slot, temperature in every lane), and the controller
    double y0[S], yl[S], yk[S], y0T = 1000.0, ylT = 1000.0, ykT = 1000.0;
#pragma unroll
    for (int s = 0; s < S; ++s) y0[s] = yl[s] = yk[s] = 1e-6;
    double t = 0.0, tn = 0.0, dt = 0.0, dtl = 0.0, dtTry = 0.0, left = 0.0, sub = 0.0, dtc = 0.0,
           lts0 = 0.0, lts1 = 0.0, lastErr = 0.0;
    int nstep = 0, ncount = 0, chk = 0, last = 0;
    long long cell = 0, csteps = 0, citer = 0;
    long long c_cells = 0, c_steps = 0, c_att = 0, c_newt = 0, c_rhs = 0, c_maxs = 0, c_fail = 0;
    double dtmin = __builtin_huge_val();

    auto finish_cell = [&]() __attribute__((always_inline)) {
        if (c == 0) {
            P.subDt[cell] = sub;
            if (P.cost) P.cost[cell] = (int)(citer < 0x7fffffffll ? citer : 0x7fffffffll);
        }
        if (P.mode == 0) {
            const double rho = P.rho[cell], rdt = 1.0 / dtc;
#pragma unroll
            for (int s = 0; s < S; ++s) {
                const int k = c + 16 * s;
                if (k < ns) {
                    const double c0 = rho * P.Y[k * P.ldY + cell] / W[s];
                    P.R[k * P.ldR + cell] = (y0[s] - c0) * rdt * W[s];
                }
            }
        } else {
            // ciToYi (chemistrySource.cpp:1222-1240)
            double yy[S], rs = 0.0, ys = 0.0;
#pragma unroll
            for (int s = 0; s < S; ++s) {
                yy[s] = c + 16 * s < ns ? fmax(0.0, y0[s]) : 0.0;
                rs += yy[s] * W[s];
            }
            const double rr = 1.0 / fmax(gsum(rs), kTiny);
#pragma unroll
            for (int s = 0; s < S; ++s) {
                yy[s] = yy[s] * W[s] * rr;
                ys += yy[s];
            }
            ys = gsum(ys);
            const double ri = 1.0 / ys;
#pragma unroll
            for (int s = 0; s < S; ++s)
                if (c + 16 * s < ns)
                    P.Yout[(c + 16 * s) * P.ldY + cell] = ys != 1.0 ? yy[s] * ri : yy[s];
            if (c == 0) P.Tout[cell] = y0T;
        }
        ++c_cells;
        dtmin = fmin(dtmin, sub);
        c_maxs = csteps > c_maxs ? csteps : c_maxs;
        phase = PQ_NEED;
    };
    auto start_attempt = [&]() __attribute__((always_inline)) {
        lts0 = dtl;
        ++c_att;
#pragma unroll
        for (int s = 0; s < S; ++s) yk[s] = y0[s];
        ykT = y0T;
        ncount = 0;
        lastErr = 0.0;
        phase = PQ_NEWTON;
    };
    // loop head of ImplicitEuler::solve(t0, tn, dt0, y); false when the step
    // budget is exhausted (tn then becomes the time reached)
    auto start_step = [&]() __attribute__((always_inline)) -> bool {
        if (nstep >= P.max_steps) {
            tn = t;
            return false;
        }
        dtTry = dt;
        if ((t + dt - tn) * (t + dt) > 0) {
            dt = tn - t;
            last = 1;
        } else if (t + dt == tn) {
            last = 1;
        }
        dtl = dt;
        lts1 = lts0;
        chk = 0;
        start_attempt();
        return true;
    };
    auto start_ode = [&]() __attribute__((always_inline)) {
        tn = left;
        t = 0.0;
        dt = 0.2 * sub;
        last = 0;
        nstep = 0;
        return start_step();
    };
    auto start_cell = [&]() __attribute__((always_inline)) {
        const double T0 = P.T[cell];
        dtc = P.dt[cell] * P.dtFactor;
        const double sub_in = P.subDt[cell];
        if (T0 < P.Tthr) {
            if (c == 0) {
                P.subDt[cell] = dtc;
                if (P.cost) P.cost[cell] = 0;
            }
            if (P.mode == 0) {
#pragma unroll
                for (int s = 0; s < S; ++s)
                    if (c + 16 * s < ns) P.R[(c + 16 * s) * P.ldR + cell] = 0.0;
            }
            return;  // stays PQ_NEED
        }
        const double rho = P.rho[cell];
#pragma unroll
        for (int s = 0; s < S; ++s) {
            const int k = c + 16 * s;
            yl[s] = y0[s] = k < ns ? rho * P.Y[k * P.ldY + cell] / W[s] : 0.0;
        }
        ylT = y0T = T0;
        sub = fmin(dtc, fmin(sub_in > 0.0 ? sub_in : dtc, P.dt_max));
        left = dtc;
        csteps = 0;
        citer = 0;
        start_ode();
    };
    // checkNewY and the step-size control of adaptiveSolve, then the loops of
    // ImplicitEuler::solve and chemistrySource::solve
    auto attempt_done = [&](double error) __attribute__((always_inline)) {
        enum { A_RETRY, A_FAIL, A_NEXT, A_ODE_END };
        int action;
        // error^-alpha, wherever a branch below needs it
        const double pw = exp(-P.alpha * log_pos(error));
        const bool ok = !((ykT - y0T) > P.Talpha * y0T);
        if (!ok) dtl *= P.Tbeta;
        if (!ok && chk < 100) {
            ++chk;
            action = dtl <= kVeryTiny ? A_FAIL : A_RETRY;
        } else if (error > 1.0) {
            dtl *= fmax(P.safe * pw, P.minsc);
            action = dtl <= kVeryTiny ? A_FAIL : A_RETRY;
        } else {
            t += dtl;
#pragma unroll
            for (int s = 0; s < S; ++s) {
                yl[s] = y0[s];
                y0[s] = yk[s];
            }
            ylT = y0T;
            y0T = ykT;
            if (error > errg) dt = fmin(fmax(P.safe * pw, P.minsc), P.maxsc) * dtl;
            else dt = fmax(P.safe * P.maxsc * dtl, dtl);
            ++c_steps;
            ++csteps;
            if ((t - tn) * tn >= 0) {
                if (nstep > 0 && last) sub = fmin(dtTry, tn);
                action = A_ODE_END;
            } else {
                ++nstep;
                action = A_NEXT;
            }
        }
        if (action == A_RETRY) {
            start_attempt();
        } else if (action == A_NEXT) {
            if (!start_step()) action = A_ODE_END;
        }
        if (action == A_ODE_END) {
            // while (leftTime > 0): ODE solves of the remaining interval
            left -= tn;
            if (left > 0.0) start_ode();
            else finish_cell();
        } else if (action == A_FAIL) {
            ++c_fail;
            finish_cell();
        }
    };

    for (;;) {
        // ---- groups without a cell take the next ones (one atomic per wavefront) ----
        for (;;) {
            const unsigned long long need = __builtin_amdgcn_ballot_w64(phase == PQ_NEED && c == 0);
            if (need == 0ull) break;
            unsigned long long base = 0;
            if (lane == 0) base = atomicAdd(P.counter, (unsigned long long)__popcll(need));
            base = __shfl(base, 0);
            if (phase == PQ_NEED) {
                const unsigned long long mine =
                    base + (unsigned long long)__popcll(need & ((1ull << (lane & 48)) - 1ull));
                if (mine >= (unsigned long long)P.n) {
                    phase = PQ_DONE;
                } else {
                    cell = P.order ? (long long)P.order[mine] : (long long)mine;
                    start_cell();
                }
            }
        }
        if (!__any(phase != PQ_DONE)) break;
        // ---- f and J at the Newton iterates, and the Newton systems ----
        QuadF<S> o;
        double x[S], xT;
        sys.step(WP, L, yk, ykT, y0, y0T, dtl, phase == PQ_NEWTON, o, x, xT);
        // ---- Newton update, its norm and the error estimate: straight-line for
        // all groups, so that the two maxima run side by side ----
        const bool newton = phase == PQ_NEWTON, err0 = phase == PQ_ERR0;
        bool bad_x = bad(xT);
#pragma unroll
        for (int s = 0; s < S; ++s) bad_x = bad_x || bad(x[s]);
        bad_x = gany(bad_x);
        const bool upd = newton && !bad_x;
        ykT += upd ? xT : 0.0;
        double m1 = fabs(xT) * frcp(P.atol + P.rtol * fabs(ykT));
        // first step: y - y0 - dt f(y) (ImplicitEuler.cpp:111-120); later the
        // second-difference LTE (ImplicitEuler.cpp:122-139)
        const double e1 = lts0 * frcp(lts0 + lts1), e2 = e1 * lts0 * frcp(lts1);
        const double eT = err0 ? ykT - y0T + dtl * o.dT : e1 * (ykT - y0T) - e2 * (y0T - ylT);
        double m2 = fabs(eT) * frcp(P.atol_inc + P.rtol_inc * fmax(fabs(y0T), fabs(ykT)));
        bool nan_y = isnan(ykT);
#pragma unroll
        for (int s = 0; s < S; ++s) {
            yk[s] += upd ? x[s] : 0.0;
            const double e = err0 ? yk[s] - y0[s] - dtl * o.w[s]
                                  : e1 * (yk[s] - y0[s]) - e2 * (y0[s] - yl[s]);
            if (c + 16 * s < ns) {
                m1 = fmax(m1, fabs(x[s]) * frcp(P.atol + P.rtol * fabs(yk[s])));
                m2 = fmax(m2, fabs(e) * frcp(P.atol_inc + P.rtol_inc * fmax(fabs(y0[s]), fabs(yk[s]))));
                nan_y = nan_y || isnan(yk[s]);
            }
        }
        m1 = gmax(m1);
        m2 = gmax(m2);
        if (gany(nan_y)) m2 = 1.5;  // ImplicitEuler::maxIncrement
        // ---- group-local transitions ----
        bool have = false;
        double aerr = 0.0;
        if (err0) {
            ++c_rhs;
            have = true;
            aerr = m2;
        } else if (newton) {
            // NewtonIteration after the solve (ImplicitEuler.cpp:200-249)
            ++c_newt;
            ++citer;
            if (bad_x || (ncount > 5 && m1 > 2.0 * fmax(lastErr, kTiny))) {
                have = true;
                aerr = 1000.0;
            } else {
                lastErr = m1;
                ++ncount;
                if (isnan(m1)) {
                    have = true;
                    aerr = 1000.0;
                } else if (ncount > 1000) {
                    have = true;
                    aerr = m1;
                } else if (m1 <= 1.0) {
                    if (nstep == 0) {
                        phase = PQ_ERR0;
                    } else {
                        have = true;
                        aerr = m2;
                    }
                }
            }
        }
        if (have) {
            attempt_done(aerr);
        } else if (phase == PQ_NEWTON && citer > P.max_cell_iters) {
            // no legitimate cell gets here; the cap guarantees every wavefront drains
            ++c_fail;
            finish_cell();
        }
    }
    // counters: every lane of a group holds its group's, one atomic per wavefront
    const bool one = c == 0;
    const long long s0 = wave_sum(one ? c_cells : 0), s1 = wave_sum(one ? c_steps : 0),
                    s2 = wave_sum(one ? c_att : 0), s3 = wave_sum(one ? c_newt : 0),
                    s4 = wave_sum(one ? c_rhs : 0), s5 = wave_max(c_maxs),
                    s7 = wave_sum(one ? c_fail : 0);
    const double dmin = wave_min(dtmin);
    if (lane == 0) {
        atomicAdd(&P.stats[0], (unsigned long long)s0);
        atomicAdd(&P.stats[1], (unsigned long long)s1);
        atomicAdd(&P.stats[2], (unsigned long long)s2);
        atomicAdd(&P.stats[3], (unsigned long long)s3);
        atomicAdd(&P.stats[4], (unsigned long long)s4);
        atomicMax(&P.stats[5], (unsigned long long)s5);
        if (dmin < __builtin_huge_val())
            atomicMin(&P.stats[6], (unsigned long long)__double_as_longlong(dmin));
        atomicAdd(&P.stats[7], (unsigned long long)s7);
    }
}

}  // namespace ohcd
