// wave_dispatch.hpp -- host interface of the generic wavefront-per-cell kernels.
#pragma once

#include <hip/hip_runtime.h>

#include "lane_kernels.hpp"

namespace ohcd {

struct WMech;
struct WaveParams;
struct KimParams;
struct LuParams;

// Padded ODE size the generic kernels use for n = ns + 1 unknowns (-1: too large).
int wave_size(int n);
// ImplicitEuler runs the kernel of `cells` cells per wavefront (wave_cells)
hipError_t wave_integrate(const WaveParams &p, int cells, int grid, hipStream_t s);
hipError_t wave_eval(const EvalParams &p, const WMech &m, int exact, hipStream_t s);
hipError_t wave_source(const SourceParams &p, const WMech &m, hipStream_t s);
hipError_t wave_kim(const KimParams &p, const WMech &m, int fp32, hipStream_t s);
// batched dense LU solves of n x n systems, n <= 64
hipError_t wave_lu(const LuParams &p, hipStream_t s);
// the persistent integrator kernel of n unknowns that holds `cells` cells per
// wavefront (its occupancy sizes the grid), and the cells per wavefront of a call
// of `ncells` cells
const void *wave_integrate_fn(int n, int cells);
int wave_cells(int n, int integrator, int prec, int64_t ncells);
// Pair constants of the mixture rules (props_table.hip), row i, columns in
// blocks of eight: [64 rows][8 blocks][4 tables][8], tables P (Wilke), A, R, C
// (diffusion; A and C are zero for i = j).
struct PairTab {
    static constexpr int kRow = 8 * 4 * 8;
    const double *t;
};
// One record per reaction for kernels with a wave-uniform reaction
// (source_table.hip).  32-bit words: the packed header (RH_HDR) with flags, the
// participants' rows (reactants 0..2, products 3..5; species * 64, two to a
// word; the row past the species for an absent one), their signed coefficients
// (0 if absent), orders (1 if absent) and the sum of the coefficients; then
// doubles: the forward, low-pressure and explicit reverse Arrhenius triples, the
// fall-off parameters, the participants' third-body efficiencies and the
// reaction's NASA-7 coefficients sum nu_k W_k a_k (low range, high range).
struct SrcTab {
    enum { kHdr, kRow, kNu = kRow + 3, kOrd = kNu + 6, kSum = kOrd + 6, kWords = 18 };
    enum { kArr = kWords / 2, kLow = kArr + 3, kRev = kLow + 3, kFop = kRev + 3, kEff = kFop + 5,
           kNasa = kEff + 6, kRec = 48 };
    // header flags: a species on both sides, a third participant on a side, and
    // (3 bits) the participant that is the last species (7: none)
    static constexpr unsigned kBoth = 1u << 20, kThree = 1u << 21;
    static constexpr int kLast = 22;
    const double *rec;
    int first_tb;  // first reaction of the table with a third body (they come last)
};
// source terms of run-time tables whose coefficients and orders the packed
// fields hold exactly, with one Tcommon for all species and ns <= 56, for calls
// of at least kSourceTableMin cells (below, one wavefront per cell is faster: the
// two cost the same at about 6,000 cells of 32 or 54 species)
constexpr int64_t kSourceTableMin = 8192;
hipError_t table_source(const SourceParams &p, const WMech &m, const SrcTab &t, hipStream_t s);
// mixture thermo / transport and T from h for run-time tables; wave_props is
// the split-precision form
hipError_t table_props(const PropParams &p, const WMech &m, const PairTab &pt, hipStream_t s);
hipError_t wave_props(const PropParams &p, const WMech &m, hipStream_t s);
hipError_t wave_tfromh(const ThParams &p, const WMech &m, hipStream_t s);

}  // namespace ohcd
