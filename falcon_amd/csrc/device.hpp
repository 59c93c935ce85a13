// Shared declarations between the kernel file and the C-ABI file.
#pragma once
#include <hip/hip_runtime.h>
#include <cstdint>

namespace falcon {

struct Layout;
// Layout::build's ghost tables (donors, targets, entries, and GC_iBlocks when
// the layout keeps them) built on the device (tables.hip); equal to the host
// build bit for bit
void build_ghosts_device(Layout &lay, int nthreads, hipStream_t s);

// Per-block constants, FP64 (3_6/ModBlock.f90:315-317 and the derivative
// coefficient (1./12./dx) of 3_6/ModDerivative.f90:16,22,28).
struct BlockMeta {
    double cr, ct, cp;      // (double)(1.0f/12.0f)/dx
    double dxi, dxj, dxk;
    int flags;              // bit 0: bottom block (inner radial boundary), bit 1: top block
};

// Geometry and background tables on the device, one row per block.
// Radial rows have NI entries, angular rows NJ entries (padded indices).
struct DevTables {
    const BlockMeta *meta;
    // radial (NI per block)
    const double *xi, *rinv, *r2inv, *rho0, *gp, *gq, *g_over_rho0, *xir2, *heat, *cs, *sqrt_rho0;
    const double *rho0_up;  // rho0 times kDivUp
    // theta (NJ per block)
    const double *sint, *sinv, *cot;
};

// x / b for many x and one b: y = 1/b by two Newton steps on the hardware
// reciprocal, then Markstein's correction of x*y by its exact remainder: the
// correctly rounded quotient (P. Markstein, IBM J. Res. Dev. 34, 1990) in 3
// operations per x, where the general division takes 11 (the same steps with
// a rescaling of operands near the ends of the exponent range).  The fix-up gives
// zeros, infinities and NaN as the division does.
// The remainder is exact for |x| >= 2^-969 (2e-292); below, its rounding changes
// the last bit of one quotient in 2^1022 |x|.  Cell lengths and matrix diagonals
// (2^27 and more) divide their dividends as they are: a normal quotient then has
// |x| > 2^-995.  The divisors near 1 of the FP64 stage (density, sin(theta), 5-k)
// and their dividends are multiplied by kDivUp, which is exact for every dividend
// below 2^970 (1e292).
constexpr double kDivUp = 0x1p54;
__device__ __forceinline__ double div_rcp(double b) {
    double r = __builtin_amdgcn_rcp(b);
    r = __builtin_fma(r, __builtin_fma(-b, r, 1.0), r);
    return __builtin_fma(r, __builtin_fma(-b, r, 1.0), r);
}
__device__ __forceinline__ double div_by(double x, double b, double y) {
    const double q = x * y;
    return __builtin_amdgcn_div_fixup(__builtin_fma(__builtin_fma(-b, q, x), y, q), b, x);
}

struct Dims {
    int ni, nj, nk, ng;
    int NI, NJ, NK;
    int nblocks;
    long long P;            // cells per variable per block (NI*NJ*NK)
    // cell layout within one block variable (cell_off): main part strides
    int SJ;                 // nk
    long long SI;           // NJ*nk
    long long M;            // NI*NJ*nk, the first cell of the side part
};

// Offset of padded cell (I, J, K) within one block variable of a state buffer
// (buffers are [block][variable][P cells]).  The P cells are split in two
// parts so that every row a march reads or writes is whole and aligned:
// - main: the interior phi range of every padded (I, J) row, rows of nk
//   values: (I*NJ + J)*nk + (K - ng).  A 16^3 block's rows are 64 (FP32) or
//   128 (FP64) bytes, and a wavefront's four rows are one contiguous span;
// - side: the 2*ng phi ghosts of every row: M + (I*NJ + J)*2*ng + kg, with
//   kg = K below the interior and K - nk above it.
// Rows padded in place (20 values with the interior at 2..17) made every
// store of a wavefront a set of partial 128-byte lines: such stores measured
// 1.56 TB/s on MI355X against 5.9 TB/s for whole aligned rows.
__host__ __device__ inline long long cell_off(const Dims &d, int I, int J, int K) {
    if (K >= d.ng && K < d.ng + d.nk) return ((long long)I * d.NJ + J) * d.nk + (K - d.ng);
    return d.M + ((long long)I * d.NJ + J) * (2 * d.ng) + (K < d.ng ? K : K - d.nk);
}
// inverse of cell_off
__host__ __device__ inline void cell_ijk(const Dims &d, long long c, int &I, int &J, int &K) {
    if (c < d.M) {
        K = (int)(c % d.nk) + d.ng;
        c /= d.nk;
    } else {
        c -= d.M;
        const int kg = (int)(c % (2 * d.ng));
        K = kg < d.ng ? kg : kg + d.nk;
        c /= 2 * d.ng;
    }
    J = (int)(c % d.NJ);
    I = (int)(c / d.NJ);
}
// Dims of a layout of padded blocks (ni, nj, nk, ng)
inline Dims make_dims(int ni, int nj, int nk, int ng, int nblocks) {
    Dims d{};
    d.ni = ni; d.nj = nj; d.nk = nk; d.ng = ng;
    d.NI = ni + 2 * ng; d.NJ = nj + 2 * ng; d.NK = nk + 2 * ng;
    d.nblocks = nblocks;
    d.P = (long long)d.NI * d.NJ * d.NK;
    d.SJ = nk;
    d.SI = (long long)d.NJ * nk;
    d.M = (long long)d.NI * d.NJ * nk;
    return d;
}

// Entries of one kind of the FP32 buffers' ghost fill.  The first n_face fill
// ghosts outside the block along one axis, all that the stage kernel reads; the
// others, ghosts beyond an edge or a corner, are read by the diffusion's
// shifted speed cells only.  Both parts are in the order of src.
struct DevFill {
    const int2 *idx;        // (dst, src): block*8*P + cell of the ghost and of its (base) source cell, variable 0
    int n, n_face;
};
// Ghost-fill tables of the FP32 buffers (device)
struct DevGhosts {
    DevFill weighted;       // trilinear; bit 31 of dst: a Yin-Yang entry
    const double *w;        // 3 weights per weighted entry
    const double *rot;      // 2 rotation coefficients per weighted entry (read for Yin-Yang entries only)
    DevFill lerp;           // interpolated along r only
    const double *lerp_w;   // their r weight
    DevFill copy;           // plain copies (every one: n_face is not used)
    // copies whose ghosts the consuming kernels do not read in place (see pull below)
    DevFill copy_rest;
    // pull[R*27 + (di+1)*9 + (dj+1)*3 + (dk+1)]: the same-level block D whose
    // interior holds all ghosts of block R in direction (di,dj,dk) as plain
    // copies, ghost index g <- D's cell g - (di*ni, dj*nj, dk*nk); -1 where any
    // ghost of that region is filled otherwise.  null: no pull.
    const int32_t *pull;
};

// Ghost-fill table of the FP64 buffers: first the ghosts outside the block
// along one axis (n_face), then those beyond an edge or a corner, both in the
// order of src (see DevFill).
struct DevGhosts64 {
    const int32_t *all;     // every entry's index, in the order of src
    const int32_t *dst;     // block*8*P + cell of the ghost (variable 0); bit 31: a Yin-Yang entry
    const int32_t *src;     // donor*8*P + cell of the interpolation base (variable 0)
    const double *w;        // 3 weights per entry
    const double *rot;      // 2 rotation coefficients per entry (read for Yin-Yang entries only)
    int n, n_face;
};

struct DevBoundary {
    const int32_t *list;    // block*2 + side (0 bottom, 1 top)
    int n;
};

// radial ghosts formed in a fill's launch (none where bnd.n is 0): the mirror
// of the buffer's interior columns, or with src all radial ghosts of src
struct FillTail {
    DevBoundary bnd{nullptr, 0};
    const void *src = nullptr;
};
// dt from the partial minima, formed in a boundary launch (none where partial is null)
struct DtFinal {
    const double *partial = nullptr;
    int n = 0;
    double cfl = 0.0;
    double *dtp = nullptr;
};

// launchers (kernels.hip)
// pull (null: none): the pull table of DevGhosts; ghosts of `in` in the
// directions it lists are read from the neighbour's interior instead.
// tile: (theta, phi) tile edge of the march, 8 or 16; wgs: 0 launches one
// workgroup per tile, n > 0 launches n workgroups that loop over the tiles (a
// persistent launch).  Results depend on neither; the dt partial minima are
// laid out per tile of the diffusion's edge.
// glm (FP64 only; null: off): grad(psi) per interior cell, [block][3][ni*nj*nk],
// subtracted from R(B) before the update (GLM divergence cleaning)
template <typename T, typename TIN, typename TOUT, typename TB>
void launch_stage(const Dims &d, const DevTables &t, const TIN *in, const TB *U, TOUT *out, float *shadow,
                  const double *dtp, double div, hipStream_t s, const int32_t *pull, int tile, int wgs,
                  const double *glm = nullptr);
// GLM divergence cleaning (FP64 path).  psi buffers are [block][P] in the
// cell_off layout.  Speed (once per step): Ch = c_h and c_h / h_LLL of the
// step's state U, [block][2][interior cells].  Stage: psi_out = psi_n +
// dt R(psi)/div from the stage input (state `in`, psi_in) and Ch, and
// G = grad(psi_in);
// diffusion: psi_new = psi + 0.5 dt R_diff(psi) with the speeds of U;
// ghost fill: launch_exchange64, with the state's (psi a scalar: no Yin-Yang
// rotation).
void launch_glm_speed(const Dims &d, const DevTables &t, const double *U, double *Ch, hipStream_t s);
void launch_glm_stage(const Dims &d, const DevTables &t, const double *in, const double *Ch, const double *psi_in,
                      const double *psi_n, double *psi_out, double *G, const double *dtp, double div, hipStream_t s);
void launch_glm_diffusion(const Dims &d, const DevTables &t, const double *U, const double *psi, double *psi_new,
                          const double *dtp, hipStream_t s);
// the FP64 buffers' ghosts and (psi not null) psi's, in one pass over the
// table; faces: only the ghosts outside the block along one axis
void launch_exchange64(const Dims &d, const DevGhosts64 &g, double *state, double *psi, bool faces, hipStream_t s,
                       const FillTail &tail = FillTail{});
// Uold: U^n for the FP32 path, whose diffusion updates U (= out) in place;
// null for the FP64 path (U != out)
template <typename T, typename TIN>
void launch_diffusion(const Dims &d, const DevTables &t, const TIN *in, const double *U, double *out, float *shadow,
                      double *partial, const double *dtp, hipStream_t s, const int32_t *pull, int tile, int wgs,
                      const double *Uold = nullptr);
// workgroups of the stage (kernel 0) or diffusion (1) march of a precision that
// the device holds resident at once: the persistent grid
int march_resident_wgs(int kernel, int precision, int tile);
// radial segments that a one-workgroup-per-tile launch of the stage or
// diffusion march cuts each tile's column into; 1 for a persistent launch
// (wgs > 0).  Results do not depend on it; the dt partial minima are
// one per tile and segment.
int march_segments(const Dims &d, int tile, int wgs);
// every ghost entry of the FP32 buffers
void launch_exchange(const Dims &d, const DevGhosts &g, float *state, hipStream_t s, const FillTail &tail = FillTail{});
// the entries that kernels reading with pull = g.pull still need; faces: only
// the ghosts outside the block along one axis
void launch_exchange_rest(const Dims &d, const DevGhosts &g, float *state, bool faces, hipStream_t s,
                          const FillTail &tail = FillTail{});
template <typename TS>
void launch_boundary(const Dims &d, const DevBoundary &b, TS *state, hipStream_t s, const int32_t *pull = nullptr,
                     const DtFinal &dt = DtFinal{});
// nseg: the radial segments of the diffusion's tiles (march_segments): one
// partial minimum per tile and segment
void launch_dt_partial(const Dims &d, const DevTables &t, const double *U, double *partial, hipStream_t s, int tile,
                       int nseg);
DtFinal dt_final_args(const Dims &d, const double *partial, double *dtp, double cfl, int tile, int nseg);
void launch_dt_final(const Dims &d, const double *partial, double *dtp, double cfl, hipStream_t s, int tile, int nseg);
// nvar variables of one block ([nvar][P], cell_off layout) in Fortran order into pinned host memory
void launch_block_to_host(const Dims &d, const double *src, int nvar, double *dst, hipStream_t s);
void launch_to_f32(const double *src, float *dst, long long n, hipStream_t s);
void launch_set_scalar(double *p, double v, hipStream_t s);
// NaN scan of a padded state (see k_nan_scan): w[0] counts, w[1] first position;
// w starts as {0, ~0}
template <typename TS>
void launch_nan_scan(const Dims &d, const TS *st, unsigned long long *w, hipStream_t s);
// the same scan of psi ([block][P]) as variable 8 (GLM divergence cleaning)
void launch_nan_scan_psi(const Dims &d, const double *psi, unsigned long long *w, hipStream_t s);
// interior difference of two states (see k_state_diff): pass 0 then pass 1 on
// the same 32 words w, whose first 8 and last 8 start at 0 and at ~0
void launch_state_diff(const Dims &d, const double *a, const double *b, double tol, unsigned long long *w, int pass,
                       hipStream_t s);
// one Fourier mode of the synthetic vector potential: B contribution
// a cos(k.x + ph), a = k x (random amplitude)
struct SynthMode {
    double k[3], a[3], ph;
};
// seeded synthetic initial state on the interior (k_synthetic); rng: 6 per
// block, rows: c_p, sqrt(rho0), c_s (NI each) per block; wgmax: one double
// per 256 interior cells
void launch_synthetic(const Dims &d, const double *rng, const int32_t *yin, const double *rows, const SynthMode *modes,
                      int nm, unsigned long long seed, double s_amp, double b_ratio, double *U, double *wgmax,
                      hipStream_t s);
// corner values of the AllCells output for blocks [b0, b0 + nb) (k_allcells)
void launch_allcells(const Dims &d, const double *U, const double *geo, const int32_t *yin, int b0, int nb,
                     double rsun, double *out, hipStream_t s);
// single-operator entry points used by parity tests: R only
template <typename T, typename TIN>
void launch_rhs_only(const Dims &d, const DevTables &t, const TIN *in, double *R, hipStream_t s, int tile, int wgs);
template <typename T>
void launch_diffusion_only(const Dims &d, const DevTables &t, const double *U, double *R, hipStream_t s, int tile,
                           int wgs);

}  // namespace falcon
