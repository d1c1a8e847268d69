// source_table.hip -- chemistry source terms and their (coupled) diagonal for
// run-time mechanism tables, one cell per lane.
//
// The diagonal needs three numbers per species (omega_k, d(omega_k)/d(c_k) and
// d(omega_k)/dT; a fourth, d(omega_k)/d(c_last), with the last species
// eliminated), not the dense Jacobian.  A block of eight wavefronts holds the
// same 64 cells, concentrations and sums in LDS as [species][cell]; the
// wavefronts share the reactions.  A reaction is wave-uniform, so its rate law
// and orders are scalar branches, only the path it takes is issued, and
// every LDS access is 64 consecutive values.  Eight wavefronts per 64 cells,
// because the sums of one cell (1 KB at 32 species) allow two blocks per CU: four
// wavefronts per SIMD.
//
// Each wavefront evaluates one reaction, then the wavefronts add their terms one
// after another (a barrier between turns), so every sum is taken in one fixed
// order and does not depend on timing.  The turns bound the kernel: a round of
// eight reactions takes about 3.4 us, half of it in turns.
//
// 32 species / 150 reactions, 262,144 cells: 2,141 us with one wavefront per
// cell and the dense Jacobian, 616 us so (four wavefronts per block 705 us).  One
// block takes 65 us whatever the number of cells, against 24 us for a hundred
// cells with a wavefront each, so calls of fewer than kSourceTableMin cells
// stay on the wavefront-per-cell kernel.
#include "wave_dispatch.hpp"
#include "wave_kernels.hpp"

namespace ohcd {

namespace {

constexpr int kWaves = 8;  // wavefronts per block

// One reaction's record (SrcTab) and efficiencies, spread over the lanes: lane
// l holds 32-bit words l and 32 + l and the efficiency of species l.  Fetched
// one turn ahead by three vector loads and read by v_readlane (a mechanism's
// records exceed the scalar cache).
struct Rec {
    unsigned u0, u1;
    double e;
    __device__ __forceinline__ void load(const WMech &M, const SrcTab &t, int r, int lane) {
        const unsigned *p = (const unsigned *)(t.rec + (size_t)r * SrcTab::kRec);
        u0 = p[lane];
        u1 = p[32 + lane];
        e = r >= t.first_tb ? M.eff[(size_t)r * 64 + lane] : 0.0;
    }
    __device__ __forceinline__ unsigned u(int i) const {
        return i < 64 ? __builtin_amdgcn_readlane(u0, i) : __builtin_amdgcn_readlane(u1, i - 32);
    }
    __device__ __forceinline__ float f(int i) const { return __uint_as_float(u(i)); }
    __device__ __forceinline__ double d(int i) const {
        return __hiloint2double((int)u(2 * i + 1), (int)u(2 * i));
    }
    // participant p's row (reactants 0..2, products 3..5; the row past the species for
    // an absent one), as an offset into a [species][64 cells] array
    __device__ __forceinline__ int row(int p) const {
        return (int)(u(SrcTab::kRow + p / 2) >> (16 * (p & 1)) & 0xffffu);
    }
};

struct SrcRxn {
    double q, s, gam, df[kWP], dr[kWP];
};

// Net rate q, dq/dT (with the rate laws' own T terms) s, third-body
// coefficient gam and the partial derivatives by each participant of a
// wave-uniform reaction; formulas and references as wreaction.  c: this lane's
// concentrations, stride 64.
template <bool DIAG>
__device__ __forceinline__ void src_reaction(const WMech &M, const Rec &R, const TFac &tf,
                                             bool lo, const double *c, int exact, SrcRxn &o) {
    const unsigned hdr = R.u(SrcTab::kHdr);
    const int rev = (hdr >> 4) & 3u, kind = (hdr >> 6) & 7u, fot = (hdr >> 9) & 7u;
    // absent participants read the row of ones past the species
    const bool three = hdr & SrcTab::kThree;
    double cf[kWP], cb[kWP];
    cf[0] = c[R.row(0)];
    cf[1] = c[R.row(1)];
    cb[0] = c[R.row(3)];
    cb[1] = c[R.row(4)];
    cf[2] = three ? c[R.row(2)] : 1.0;
    cb[2] = three ? c[R.row(5)] : 1.0;
    const double b = R.d(SrcTab::kArr + 1), Ta = R.d(SrcTab::kArr + 2);
    double Mtb = 0.0;
    if (kind != 0) {
#pragma unroll 8
        for (int k = 0; k < M.ns; ++k) Mtb += rdlane(R.e, k) * c[k * 64];
    }
    const double kA = rarrh(R.d(SrcTab::kArr), b, Ta, tf);
    double kf, k0 = 0.0, kinf = 0.0, Pr = 0.0, F = 1.0;
    FoState fs{1.0, 0.0, 0.0};
    if (kind == 0) {
        kf = kA;
    } else if (kind == 1) {
        kf = Mtb * kA;
    } else {
        double fp[5];
#pragma unroll
        for (int i = 0; i < 5; ++i) fp[i] = R.d(SrcTab::kFop + i);
        k0 = rarrh(R.d(SrcTab::kLow), R.d(SrcTab::kLow + 1), R.d(SrcTab::kLow + 2), tf);
        kinf = kA;
        const double kinfz = kinf != 0 ? kinf : kVeryTiny;
        Pr = k0 / kinfz * Mtb;
        fs = rfo_eval<DIAG>(fot, fp, tf, Pr);
        F = fs.F;
        kf = kind == 2 ? kinf * (Pr / (1.0 + Pr)) * F : k0 * (1.0 / (1.0 + Pr)) * F;
    }
    double kr = 0.0, rK = 0.0, dKc = 0.0;
    if (rev == 1) {
        // reactionTypes::Kp / Kc / DKcDT (reactionTypes.cpp:178-241) from the
        // reaction's summed NASA-7 coefficients: G = sum nu_k G_k and, inside the
        // range of every fit, dG/dT = -S
        const double T = tf.T;
        double g[2], st[2];
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            double a[7];
#pragma unroll
            for (int m = 0; m < 7; ++m) a[m] = R.d(SrcTab::kNasa + 7 * h + m);
            const double s = ((((a[4] * 0.25) * T + a[3] * (1.0 / 3.0)) * T + a[2] * 0.5) * T + a[1]) * T +
                             a[0] * tf.lnT + a[6];
            g[h] = ((((a[4] * -0.05 * T - a[3] * (1.0 / 12.0)) * T - a[2] * (1.0 / 6.0)) * T -
                     a[1] * 0.5) * T + a[0] * (1.0 - tf.lnT) - a[6]) * T + a[5];
            st[h] = -s;
        }
        const double G = lo ? g[0] : g[1];
        double dG = lo ? st[0] : st[1];
        if (__any(T < M.Tmin || T > M.Tmax)) {
            // past a fit's range cp is that of its end, and with it dG/dT
            // (JANAF.cpp:155-212): add sum nu_k (cp_k(clamped T) - cp_k(T))
            for (int p = 0; p < 2 * kWP; ++p) {
                const double nu = R.f(SrcTab::kNu + p);
                if (nu == 0.0) continue;
                const int k = R.row(p) / 64;
                const double *S = M.sp;
                const double Tx = fmin(fmax(T, S[SP_TLOW * 64 + k]), S[SP_THIGH * 64 + k]);
                const int oa = lo ? SP_ALO : SP_AHI;
                double cx = 0.0, ct = 0.0;
                for (int m = 4; m >= 0; --m) {
                    cx = cx * Tx + S[(oa + m) * 64 + k];
                    ct = ct * T + S[(oa + m) * 64 + k];
                }
                dG += Tx != T ? nu * (cx - ct) * S[SP_W * 64 + k] : 0.0;
            }
        }
        double Kp = exp(-G * tf.invRuT);
        if (bad(Kp)) Kp = kRootVeryLarge;
        const double sS = R.f(SrcTab::kSum);
        const bool zero_s = fabs(sS) < kVeryTiny;
        double Xs = 1.0, Kc = Kp;
        if (!zero_s) {
            Xs = xpow(tf, sS);
            Kc = fmin(Kp * Xs, kVeryLarge);
        }
        rK = frcp(fmax(Kc, kVeryTiny));
        kr = Kc > kVeryTiny ? kf * rK : 0.0;
        if (DIAG) {
            double dk = (dG - G * tf.invTm) * tf.invRuT;
            if (exact) dk = -dk;
            double dKp = Kp * dk;
            if (bad(dKp)) dKp = kVeryLarge;
            dKc = dKp;
            if (!zero_s) {
                double v = (dKp + Kp * (-sS) * tf.invT) * Xs;
                if (bad(v)) v = kVeryLarge;
                dKc = v;
            }
        }
    } else if (rev == 2) {
        kr = rarrh(R.d(SrcTab::kRev), R.d(SrcTab::kRev + 1), R.d(SrcTab::kRev + 2), tf);
        if (kind == 1) kr = Mtb * kr;
    }
    double pf[kWP], pb[kWP], df[kWP], db[kWP];
#pragma unroll
    for (int i = 0; i < kWP; ++i) {
        pf[i] = cf[i];
        pb[i] = cb[i];
        df[i] = db[i] = 1.0;
    }
    if (hdr & (0x3fu << kRhSq)) {
#pragma unroll
        for (int i = 0; i < kWP; ++i) {
            if (hdr >> (kRhSq + i) & 1u) {
                pf[i] = cf[i] * cf[i];
                df[i] = cf[i] + cf[i];
            }
            if (hdr >> (kRhSq + kWP + i) & 1u) {
                pb[i] = cb[i] * cb[i];
                db[i] = cb[i] + cb[i];
            }
        }
    }
    if (hdr & kRhPow) {
        auto dpow = [](double x, double ord) {
            if (ord == 1.0) return 1.0;
            if (ord < 1.0) return x > kTiny ? ord * pow_ool(x, ord - 1.0) : 0.0;
            return ord * rpow(x, ord - 1.0);
        };
#pragma unroll
        for (int i = 0; i < kWP; ++i) {  // an absent one has order 1
            const double e = R.f(SrcTab::kOrd + i), g = R.f(SrcTab::kOrd + kWP + i);
            pf[i] = rpow(cf[i], e);
            df[i] = dpow(cf[i], e);
            pb[i] = rpow(cb[i], g);
            db[i] = dpow(cb[i], g);
        }
    }
    const double f01 = pf[0] * pf[1], b01 = pb[0] * pb[1], prf = f01 * pf[2], prb = b01 * pb[2];
    const double q = kf * prf - kr * prb;
    o.q = q;
    if (!DIAG) return;
    const double kf2 = kf * pf[2], kr2 = kr * pb[2];  // (kr = 0 for an irreversible reaction)
    o.df[0] = kf2 * df[0] * pf[1];
    o.df[1] = kf2 * df[1] * pf[0];
    o.df[2] = three ? kf * df[2] * f01 : 0.0;
    o.dr[0] = kr2 * db[0] * pb[1];
    o.dr[1] = kr2 * db[1] * pb[0];
    o.dr[2] = three ? kr * db[2] * b01 : 0.0;
    o.gam = 0.0;
    double dkf, dkr = 0.0, dgdT = 0.0;
    if (kind <= 1) {
        if (kind == 1) o.gam = q * (1.0 / fmax(Mtb, kTiny));
        dkf = rarrh_dkdT(kf, b, Ta, tf);
    } else {
        const double b0 = R.d(SrcTab::kLow + 1), Ta0 = R.d(SrcTab::kLow + 2);
        const double kinfz = kinf != 0 ? kinf : kVeryTiny, k0z = k0 != 0 ? k0 : kVeryTiny;
        const double r1 = 1.0 / (1.0 + Pr), dk0 = rarrh_dkdT(k0, b0, Ta0, tf),
                     dki = rarrh_dkdT(kinf, b, Ta, tf);
        dkf = kind == 2 ? Pr * r1 * F * dki : r1 * F * dk0;
        if (Mtb > kTiny) {
            const double dPr = k0 / kinfz;
            const double g = (kind == 2 ? dPr / (Pr * (1 + Pr)) : -dPr * r1) + fs.gPr * dPr;
            o.gam = bad(g) ? 0.0 : q * g;
            const double dPrdT = Pr * (dk0 / k0z - dki / kinfz);
            dgdT = q * ((kind == 2 ? dPrdT / (Pr * (1 + Pr)) : -dPrdT * r1) + fs.gT + fs.gPr * dPrdT);
        }
    }
    if (rev == 1) dkr = (dkf - kr * dKc) * rK;
    else if (rev == 2) dkr = rarrh_dkdT(kr, R.d(SrcTab::kRev + 1), R.d(SrcTab::kRev + 2), tf);
    double dqdT = dkf * prf - dkr * prb;
    if (bad(dqdT)) dqdT = 0.0;
    if (bad(dgdT)) dgdT = 0.0;
    o.s = dqdT + dgdT;
}

// What one reaction adds to this lane's sums: addresses and terms, formed
// before the wavefront's turn, so that the turn itself -- the part the four
// wavefronts take one after another -- is reads, adds and writes only.
template <bool DIAG, bool LAST>
struct SrcTerms {
    static constexpr int NV = 1 + 2 * DIAG + LAST;  // omega, d/dT, d/dc, d/dc_last
    int o[4];                                       // rows of reactants 0, 1 and products 0, 1
    double v[4][NV];
    bool simple;
};

template <bool DIAG, bool LAST>
__device__ __forceinline__ void src_terms(const WMech &M, const Rec &R, const SrcRxn &x,
                                          SrcTerms<DIAG, LAST> &a) {
    const unsigned hdr = R.u(SrcTab::kHdr);
    a.simple = !(hdr & (SrcTab::kBoth | SrcTab::kThree));
    if (!a.simple) return;
    const int kind = (hdr >> 6) & 7u;
    double dl = 0.0;  // dq / dc of the last species
    if (LAST) {
        const unsigned at = (hdr >> SrcTab::kLast) & 7u;
        dl = at == 0u ? x.df[0] : at == 1u ? x.df[1] : at == 3u ? -x.dr[0] : at == 4u ? -x.dr[1] : 0.0;
        if (kind != 0) dl += x.gam * rdlane(R.e, M.ns - 1);
    }
#pragma unroll
    for (int m = 0; m < 4; ++m) {
        const int p = m < 2 ? m : m + 1;
        const double nu = R.f(SrcTab::kNu + p);
        a.o[m] = R.row(p);
        a.v[m][0] = nu * x.q;
        if (DIAG) {
            double g = m < 2 ? x.df[m] : -x.dr[m - 2];
            if (kind != 0) g = fma(x.gam, R.d(SrcTab::kEff + p), g);
            a.v[m][1] = nu * x.s;
            a.v[m][2] = nu * g;
            if (LAST) a.v[m][3] = nu * dl;
        }
    }
}

// Adds the terms to this lane's sums acc[quantity][row][64 cells]: plain reads
// and writes, all reads first (an FP64 LDS atomic took 110 cycles).  Absent
// participants add zero to the row past the species.
template <bool DIAG, bool LAST, int NR>
__device__ __forceinline__ void src_add(const WMech &M, const Rec &R, const SrcRxn &x,
                                        const SrcTerms<DIAG, LAST> &a, double *acc) {
    constexpr int NV = SrcTerms<DIAG, LAST>::NV;
    if (a.simple) {
        double s[4][NV];
#pragma unroll
        for (int m = 0; m < 4; ++m)
#pragma unroll
            for (int i = 0; i < NV; ++i) s[m][i] = acc[a.o[m] + i * NR];
#pragma unroll
        for (int m = 0; m < 4; ++m)
#pragma unroll
            for (int i = 0; i < NV; ++i) acc[a.o[m] + i * NR] = s[m][i] + a.v[m][i];
        return;
    }
    // a third participant on a side, or a species on both sides (its derivative
    // collects several terms): one participant after another
    const int kind = (R.u(SrcTab::kHdr) >> 6) & 7u;
    for (int p = 0; p < 2 * kWP; ++p) {
        const double nu = R.f(SrcTab::kNu + p);
        if (nu == 0.0) continue;
        const int o = R.row(p);
        auto dq = [&](int row) {
            double v = kind != 0 ? x.gam * rdlane(R.e, row / 64) : 0.0;
#pragma unroll
            for (int j = 0; j < kWP; ++j) {
                if (R.row(j) == row) v += x.df[j];
                if (R.row(kWP + j) == row) v -= x.dr[j];
            }
            return v;
        };
        acc[o] += nu * x.q;
        if (DIAG) {
            acc[o + NR] += nu * x.s;
            acc[o + 2 * NR] += nu * dq(o);
            if (LAST) acc[o + 3 * NR] += nu * dq((M.ns - 1) * 64);
        }
    }
}

template <int NSP, bool DIAG, bool LAST>
__global__ __launch_bounds__(64 * kWaves, 4) void source_table_kernel(const SourceParams P,
                                                                   const WMech M,
                                                                   const SrcTab tab) {
    // [species][cell], and the row for absent participants
    constexpr int NR = (NSP + 1) * 64;
    constexpr int NV = SrcTerms<DIAG, LAST>::NV;
    __shared__ double s_acc[NV * NR], s_c[NR], s_v[kWaves][64];
    double *s_w = s_acc, *s_t = s_acc + NR, *s_d = s_acc + 2 * NR, *s_l = s_acc + 3 * NR;
    const int lane = threadIdx.x & 63, wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6),
              ns = M.ns;
    const int64_t c0 = (int64_t)blockIdx.x * 64;
    const bool in = c0 + lane < P.n;
    const int64_t cell = in ? c0 + lane : P.n - 1;  // the last lanes repeat the last cell
    ctab *S = as_ctab(M.sp);
    const double T = P.T[cell], rho = P.rho[cell];
    double cv = 0.0;
    if (wv == 0) {
        s_c[ns * 64 + lane] = 1.0;
        s_w[ns * 64 + lane] = 0.0;
        if (DIAG) s_d[ns * 64 + lane] = s_t[ns * 64 + lane] = 0.0;
        if (LAST) s_l[ns * 64 + lane] = 0.0;
    }
    for (int k = wv; k < ns; k += kWaves) {
        const double Y = P.Y[k * P.ldY + cell], W = S[SP_W * 64 + k];
        s_c[k * 64 + lane] = fmax(rho * Y / W, 0.0);
        s_w[k * 64 + lane] = 0.0;
        if (DIAG) {
            s_d[k * 64 + lane] = s_t[k * 64 + lane] = 0.0;
            if (LAST) s_l[k * 64 + lane] = 0.0;
            double cp, h;
            species_cp_h(S, k, T, cp, h);
            cv += (cp - kRu / W) * Y;
        }
    }
    if (DIAG) s_v[wv][lane] = cv;
    const TFac tf = tfac(T);
    const bool lo = T < S[SP_TCOM * 64];
    Rec next;
    next.load(M, tab, min(wv, M.nr - 1), lane);
    __syncthreads();
    for (int base = 0; base < M.nr; base += kWaves) {
        const int r = base + wv;
        const Rec R = next;
        next.load(M, tab, min(r + kWaves, M.nr - 1), lane);
        SrcRxn x;
        SrcTerms<DIAG, LAST> a;
        if (r < M.nr) {
            src_reaction<DIAG>(M, R, tf, lo, s_c + lane, P.exact, x);
            src_terms<DIAG, LAST>(M, R, x, a);
        }
        for (int turn = 0; turn < kWaves; ++turn) {
            if (turn == wv && r < M.nr) src_add<DIAG, LAST, NR>(M, R, x, a, s_acc + lane);
            __syncthreads();
        }
    }
    // R_k = omega_k W_k and the diagonal (chemistrySource.cpp:319-480, :1371-1450)
    double b = 0.0, el = 0.0;
    if (DIAG) {
        for (int v = 0; v < kWaves; ++v) b += s_v[v][lane];
        b = 1.0 / (rho * b);
        if (LAST) {
            double cp, h;
            species_cp_h(S, ns - 1, T, cp, h);
            el = h - kRu / S[SP_W * 64 + ns - 1] * T;
        }
    }
    if (!in) return;
    for (int k = wv; k < ns; k += kWaves) {
        const double W = S[SP_W * 64 + k];
        P.R[k * P.ldR + cell] = s_w[k * 64 + lane] * W;
        if (!DIAG || (LAST && k == ns - 1)) continue;
        double cp, h;
        species_cp_h(S, k, T, cp, h);
        const double ea = h - kRu / W * T, dT = s_t[k * 64 + lane] * W * b;
        double D = s_d[k * 64 + lane];
        if (LAST) D += dT * (el - ea) - s_l[k * 64 + lane] * (W / S[SP_W * 64 + ns - 1]);
        else D -= dT * ea;
        P.D[k * P.ldD + cell] = D;
    }
}

template <int NSP>
void launch(const SourceParams &p, const WMech &m, const SrcTab &t, hipStream_t s) {
    const dim3 g((unsigned)((p.n + 63) / 64)), b(64 * kWaves);
    if (!p.D) hipLaunchKernelGGL((source_table_kernel<NSP, false, false>), g, b, 0, s, p, m, t);
    else if (!p.without_last)
        hipLaunchKernelGGL((source_table_kernel<NSP, true, false>), g, b, 0, s, p, m, t);
    else hipLaunchKernelGGL((source_table_kernel<NSP, true, true>), g, b, 0, s, p, m, t);
}

}  // namespace

hipError_t table_source(const SourceParams &p, const WMech &m, const SrcTab &t, hipStream_t s) {
    if (m.ns <= 16) launch<16>(p, m, t, s);
    else if (m.ns <= 24) launch<24>(p, m, t, s);
    else if (m.ns <= 32) launch<32>(p, m, t, s);
    else if (m.ns <= 48) launch<48>(p, m, t, s);
    else launch<56>(p, m, t, s);
    return hipGetLastError();
}

}  // namespace ohcd
