// Device kernels of the RK4 hot path for gfx950.
//
// Layout in HBM: every state buffer is [block][var][I][J][K] with the padded
// block (NI,NJ,NK) = (ni+2ng, nj+2ng, nk+2ng) contiguous and K (phi) fastest,
// so a wavefront's loads along phi are contiguous.
//
// Stage and diffusion kernels march each block along r.  A workgroup of 256
// lanes owns a 16x16 (theta, phi) tile of one block (64 lanes an 8x8 one); lane
// (ty, tx) owns one (j, k) column and keeps a register window of all 8 variables
// for the r-stencils (the stage 5 planes; the diffusion 3, with the radial face
// and half slope it carries), while the current r-plane with its 2-cell theta/phi
// halo is staged in LDS for the theta/phi stencils (the stage double-buffered).
// Corner (edge) halo cells are never needed by these stencils, so they are never
// loaded.
//
// Every arithmetic expression keeps the operand order of the reference line it
// restates; with -ffp-contract=off the FP64 instantiation is bit-identical to
// the reference.  The FP32 instantiation (T = float) is the deviation path: the
// stencil arithmetic runs in FP32 while the stage accumulation into the FP64
// state, the ghost interpolation weights and the time step stay FP64.
#include <algorithm>
#include <stdexcept>
#include <type_traits>

#include "device.hpp"

namespace falcon {

// Stage, diffusion and dt kernels take the (theta, phi) tile edge TL as a
// template parameter: 16 (256 lanes, one 16x16 tile per 16^3 block face) or 8
// (64 lanes).  Each cell's arithmetic is the same for either edge, so the
// choice (made by timing both, falcon_autotune) never changes a result.
template <int TL>
constexpr int tile_pl() { return TL + 4; }   // LDS plane edge (tile + 2 halo each side)

// Tile of workgroup w of a one-workgroup-per-tile launch of n tiles.  The
// dispatcher deals workgroups to the 8 XCDs in turn (w mod 8), and each XCD
// has its own L2.  Giving XCD x the contiguous tile range [x*n/8, ...) in
// dispatch order puts phi-adjacent blocks (consecutive ids) on the same XCD at
// the same time, so the halo each reads from the other is an L2 hit: on the
// 50 M-cell shell the FP32 stage reads 68 instead of 134 bytes per cell from
// HBM (stages 1-3) and the FP32 diffusion 158 instead of 220.
__device__ __forceinline__ int xcd_tile(int w, int n) {
    const int q = n >> 3, r = n & 7, x = w & 7, k = w >> 3;
    return x * q + min(x, r) + k;
}

// the lane index of a flat 1-D launch with the workgroups in xcd_tile's order:
// a run of consecutive lanes (the cells of one block) is served by one XCD,
// whose L2 then holds the neighbour planes the run shares.  (The ghost fills take
// shorter runs of workgroups, xcd_run: one contiguous range per XCD measured
// slower.)
__device__ __forceinline__ long long xcd_lane() {
    return (long long)xcd_tile((int)blockIdx.x, (int)gridDim.x) * blockDim.x + threadIdx.x;
}

// psi (the ninth variable of the reference's MHD blocks, 3_6/ModBlock.f90:163)
// is one padded variable per block, [block][P] in the cell_off layout; the
// ghost tables address [block][8][P] state buffers, so an entry's offset o
// maps to (o / 8P) P + o mod 8P.
__device__ __forceinline__ long long psi_off(const Dims &d, long long o) {
    const long long P8 = 8 * d.P, b = o / P8;
    return b * d.P + (o - b * P8);
}

// radial coefficient rows the stage kernel stages in LDS, and the largest padded
// radial extent NI a march accepts (the launchers reject larger blocks)
constexpr int kStageRows = 10;

constexpr int kMaxNI = 132;

// ModDerivative_1st_O4_3D (3_6/ModDerivative.f90:16-19):
// (1./12./dx)*( -f(+2) + 8.*f(+1) - 8.*f(-1) + f(-2) )
// The products with 8 are exact, so each fused multiply-add rounds as the
// reference's product and sum do.
__device__ __forceinline__ double d4(double fm2, double fm1, double fp1, double fp2, double c) {
    return c * (__builtin_fma(-8.0, fm1, __builtin_fma(8.0, fp1, -fp2)) + fm2);
}

// Smallest t with scale*t >= k in T's rounding: t >= flag_from(scale, k) is
// that comparison without its product.
template <typename T>
constexpr T flag_from(T scale, T k) {
    using I = std::conditional_t<sizeof(T) == 8, unsigned long long, unsigned>;
    I t = __builtin_bit_cast(I, (T)(k / scale));
    while (scale * __builtin_bit_cast(T, t) >= k) t--;
    while (!(scale * __builtin_bit_cast(T, t) >= k)) t++;
    return __builtin_bit_cast(T, t);
}

// Half the slope of ModLinReconstruct_minmod (3_6/ModLinReconstruct.f90:37-48)
// for one triple (the faces use only the half).  The reference forms a =
// (ur-ul)/2, b = 2(ur-u), c = 2(u-ul), m1 = max(ab, 0), m2 = max(bc, 0), takes
// the slope 0 unless m1 m2 1e10 - 1e-30 >= 0 and else the smallest of |a|, |b|,
// |c| with a's sign.  Powers of two scale exactly, so with A = 2a, B = b/2, C =
// c/2 the same decisions and values need 16 instead of about 27 operations:
// ab = AB; bc = 4BC, the 4 in the threshold (FP32, whose m1 m2 may be
// denormal there, keeps it in bc); AB > 0 wherever BC > 0.  A NaN neighbour
// below or at the cell gives NaN, as the reference's product with 0 does.
template <typename T>
__device__ __forceinline__ T half_slope(T ul, T u, T ur) {
    constexpr T from = sizeof(T) == 8 ? flag_from<T>(T(4.0e10), T(1.0e-30f)) : flag_from<T>(T(1.0e10), T(1.0e-30f));
    const T A = ur - ul, B = ur - u, C = u - ul;
    T m2 = sizeof(T) == 8 ? B * C : (T(4) * B) * C;
    m2 = sizeof(T) == 8 ? (T)__builtin_fmax((double)m2, 0.0) : (T)__builtin_fmaxf((float)m2, 0.0f);
    const T f = (A * B) * m2 >= from ? T(1) : T(0);
    const T fa = fabs(A) * T(0.25), fb = fabs(B), fc = fabs(C);
    T mn = sizeof(T) == 8 ? (T)__builtin_fmin((double)fa, (double)fb) : (T)__builtin_fminf((float)fa, (float)fb);
    mn = mn < fc ? mn : fc;
    return f * copysign(mn, A);
}

// One face of ModDiffusion_Aritificial_1 (3_6/ModDiffusion.f90:50-59) between
// cell y (value b, half slope hY) and cell x = y+1 (value c, half slope hX):
// phi * num, with num = c - sX/2 - b - sY/2 and phi = max(0, 1 + 2 (num/(c-b)
// - 1)), a NaN taken as 0; the reference's flux is this times -1/2, times the
// sum of the two speeds, times 1/2.  The factor -1/4 is a power of two: it is
// applied once to the sum over the faces (kFluxScale) with the same rounding.
// RCP (FP32 path): the limiter ratio as a product with the hardware reciprocal
// of (c - b), whose 1 ulp error is far below the FP32 storage rounding; 0 and
// +-0 denominators give the same infinities and NaN as the quotient, so the
// NaN -> 0 rule still applies.
constexpr double kFluxScale = 0.25;
template <typename T, bool RCP>
__device__ __forceinline__ T face_flux(T b, T c, T hY, T hX) {
    const T num = ((c - hX) - b) - hY;
    const T q = RCP ? num * (T)__builtin_amdgcn_rcpf((float)(c - b)) : num / (c - b);
    const T x = q - T(1);
    const T ph = sizeof(T) == 8 ? (T)__builtin_fmax(__builtin_fma(2.0, (double)x, 1.0), 0.0)
                                : (T)__builtin_fmaxf(__builtin_fmaf(2.0f, (float)x, 1.0f), 0.0f);
    return ph * num;
}
// the face between b and c of the four cells a, b, c, d
template <typename T, bool RCP = false>
__device__ __forceinline__ T face_flux4(T a, T b, T c, T d) {
    return face_flux<T, RCP>(b, c, half_slope(a, b, c), half_slope(b, c, d));
}

// Shared r-marching skeleton: loads the column window and the halo'd plane.
// With a pull table (the row of block b: entry (di+1)*9+(dj+1)*3+(dk+1) is the
// same-level neighbour whose interior holds this block's ghosts in direction
// (di,dj,dk), or -1), those ghosts are read from the neighbour at the ghost
// index minus (di*ni, dj*nj, dk*nk); the radial ghost planes of the column are
// direction (-1,0,0) / (+1,0,0), the theta/phi halo strips (0,dj,0) / (0,0,dk).
// PULL = false compiles the plain reads (the pull table is ignored).
template <typename T, typename TIN, bool PULL, int TL>
struct Marcher {
    const TIN *blk;
    long long dlo, dhi;     // offset from blk of the column source of the radial ghost
                            // planes below / above the block, plane shift included
    const TIN *hblk;        // halo strip source
    long long P;
    int SI, SJ;             // main-part plane and row pitch (cell_off)
    int ilo, ihi;           // first interior plane, first plane above the interior
    int J, K;           // padded column of this lane
    // addresses are a base that is the same for the whole workgroup (scalar
    // registers) plus this 32-bit lane offset: J*SJ + K, clamped into the block
    // for lanes outside a partial tile
    unsigned coff;
    bool act;
    bool hv;
    unsigned hoff;      // cell_off of the halo point at plane 0 (a valid cell for lanes without one)
    int hsi;            // plane pitch of the halo point's part (main or side)
    int hly, hlx;

    __device__ __forceinline__ void init(const Dims &d, const TIN *in, int b, int j0, int k0, int TJa, int TKa,
                         const int32_t *pull = nullptr) {
        P = d.P;
        SI = (int)d.SI;
        SJ = d.SJ;
        blk = in + (long long)b * 8 * P;
        ilo = d.ng;
        ihi = d.ng + d.ni;
        hblk = blk;
        dlo = dhi = 0;
        if (PULL && pull) {
            const int Dlo = pull[b * 27 + 4], Dhi = pull[b * 27 + 22];
            if (Dlo >= 0) dlo = (long long)(Dlo - b) * 8 * P + (long long)d.ni * SI;
            if (Dhi >= 0) dhi = (long long)(Dhi - b) * 8 * P - (long long)d.ni * SI;
        }
        const int tx = threadIdx.x & (TL - 1), ty = threadIdx.x / TL;
        act = ty < TJa && tx < TKa;
        J = j0 + ty + d.ng;
        K = k0 + tx + d.ng;
        // loads of inactive lanes read the tile's first cell, so every load can be
        // issued without a branch; their values are never used
        coff = (unsigned)(act ? J * SJ + (K - d.ng) : (j0 + d.ng) * SJ + k0);
        const int h = threadIdx.x;
        hv = false; hly = 0; hlx = 0;
        if (h < 4 * TL) {
            int r = h / TL, kk = h % TL;
            hly = r < 2 ? r : TJa + r;
            hlx = kk + 2;
            hv = kk < TKa;
        } else if (h < 8 * TL) {
            int h2 = h - 4 * TL;
            int c = h2 / TL, jj = h2 % TL;
            hlx = c < 2 ? c : TKa + c;
            hly = jj + 2;
            hv = jj < TJa;
        }
        const int HJ = j0 + hly, HK = k0 + hlx;   // padded halo cell
        const bool hmain = HK >= d.ng && HK < d.ng + d.nk;
        hoff = hv ? (unsigned)cell_off(d, 0, HJ, HK) : coff;
        hsi = (!hv || hmain) ? SI : d.NJ * 2 * d.ng;
        if (PULL && pull && hv) {
            const int dj = HJ < d.ng ? -1 : (HJ >= d.ng + d.nj ? 1 : 0);
            const int dk = HK < d.ng ? -1 : (HK >= d.ng + d.nk ? 1 : 0);
            if (dj | dk) {
                const int D = pull[b * 27 + 9 + (dj + 1) * 3 + (dk + 1)];
                if (D >= 0) {
                    // the neighbour's interior cell: always in its main part
                    hblk = in + (long long)D * 8 * P;
                    hoff = (unsigned)cell_off(d, 0, HJ - dj * d.nj, HK - dk * d.nk);
                    hsi = SI;
                }
            }
        }
    }
    // I is the same for every lane of the workgroup, 0 <= I < NI
    __device__ __forceinline__ T col(int v, int I) const {
        const TIN *base = blk + ((long long)v * P + (long long)I * SI);
        if (PULL) base += (I < ilo ? dlo : 0ll) + (I >= ihi ? dhi : 0ll);
        return (T)base[coff];
    }
    // interior planes only
    __device__ __forceinline__ T halo(int v, int I) const {
        const unsigned o = (unsigned)(I * hsi) + hoff;
        return (T)((PULL ? hblk : blk) + (long long)v * P)[o];
    }
};

// ---------------------------------------------------------------- stage

// RHS of ModEquation_Dynamo (3_6/ModEquation.f90:24-162) for one cell, in
// the reference's operation order, computed in T (FP64 on both paths).
// W(v, q): variable v at r-offset q-2 of this lane's column, read from the
// register window `win` of storage type TW (the FP32 path keeps its stage
// values in FP32 and widens them here); L(v,dj,dk): the LDS plane, widened the
// same way.
// RECIP (FP32 path only): the divisions by rho0 and by sin(theta) become
// products with irho0 = 1/rho0 and sinv = 1/sin(theta), the latter applied
// after the phi derivative instead of to each of its four points.  Each is a
// rounding-level change in FP64 (relative 1e-16, far below the FP32 storage
// rounding of the stage values) and removes 14 FP64 divisions per cell.
template <typename T, typename TW, bool RECIP, typename LDSF>
__device__ __forceinline__ void cell_rhs(const TW (&win)[8][5], LDSF L, const T xr[5], const T rho0r[5], const T gpr[5],
                                         const T gqr[5], const T st[5], T rinv, T r2inv, T xir2, T heat, T gor,
                                         T sinv, T cot, T cr, T ct, T cp, T irho0, T rho0_up, T R[8]) {
    auto W = [&](int v, int q) -> T { return (T)win[v][q]; };
    const T rho0c = rho0r[2];
    // Without RECIP the divisors come times kDivUp, and so do the dividends here
    // (div_by); irho0 is 1/rho0_up then.  The density's row is in the tables that way:
    // formed here it took registers (406 against 392 us per launch on 1536 16^3 blocks).
    constexpr T up = RECIP ? T(1) : T(kDivUp);
    const T bst = st[2] * up, yst = RECIP ? T(0) : div_rcp(bst);
    auto over_rho0 = [&](T x) -> T { return RECIP ? x * irho0 : div_by(x * up, rho0_up, irho0); };
    // d4 of f/sin(theta) along phi (sin(theta) is constant along phi)
    auto d4_over_st = [&](T f0, T f1, T f3, T f4) -> T {
        return RECIP ? d4(f0, f1, f3, f4, cp) * sinv
                     : d4(div_by(f0 * up, bst, yst), div_by(f1 * up, bst, yst), div_by(f3 * up, bst, yst),
                          div_by(f4 * up, bst, yst), cp);
    };
    const T vr = W(1, 2), vt = W(2, 2), vp = W(3, 2);
    const T br = W(4, 2), bt = W(5, 2), bp = W(6, 2);

    // Mass conservation (:50-61) with ModSpherical_div (:104-159)
    {
        T w[5];
#pragma unroll
        for (int q = 0; q < 5; q++) w[q] = (rho0r[q] * W(1, q)) * (xr[q] * xr[q]);
        T t1 = d4(w[0], w[1], w[3], w[4], cr) * r2inv;
        T t2 = d4((rho0c * L(2, -2, 0)) * st[0], (rho0c * L(2, -1, 0)) * st[1], (rho0c * L(2, 1, 0)) * st[3],
                  (rho0c * L(2, 2, 0)) * st[4], ct);
        T dd = d4(rho0c * L(3, 0, -2), rho0c * L(3, 0, -1), rho0c * L(3, 0, 1), rho0c * L(3, 0, 2), cp);
        t2 = t2 + dd;
        t2 = t2 * sinv;
        t2 = t2 * rinv;
        R[0] = xir2 * (t1 + t2);
    }
    // A_dot_Grad_f (ModSpherical.f90:241-279) with A = v at the centre
    auto adg = [&](int f) -> T {
        T o = vr * d4(W(f, 0), W(f, 1), W(f, 3), W(f, 4), cr);
        T tmp = vt * d4(L(f, -2, 0), L(f, -1, 0), L(f, 1, 0), L(f, 2, 0), ct);
        o = o + tmp * rinv;
        tmp = (vp * d4(L(f, 0, -2), L(f, 0, -1), L(f, 0, 1), L(f, 0, 2), cp)) * rinv;
        o = o + sinv * tmp;
        return o;
    };
    // Inertial force (:66-74): -A_dot_nabla_B(v,v) (ModSpherical.f90:281-343)
    {
        T a1 = adg(1), a2 = adg(2), a3 = adg(3);
        T tr = (-vt) * vt - vp * vp;
        a1 = a1 + tr * rinv;
        T tt = (-vp) * vp;
        tt = tt * cot;
        tt = tt + vt * vr;
        a2 = a2 + tt * rinv;
        T tp = vp * vt;
        tp = tp * cot;
        tp = tp + vp * vr;
        a3 = a3 + tp * rinv;
        R[1] = -a1; R[2] = -a2; R[3] = -a3;
    }
    // Pressure gradient (:79-92): p1 (:40-46), ModSpherical_Grad_f (:201-239)
    {
        T pr[5];
#pragma unroll
        for (int q = 0; q < 5; q++) pr[q] = gpr[q] * W(0, q) + gqr[q] * W(7, q);
        auto p1L = [&](int dj, int dk) -> T { return gpr[2] * L(0, dj, dk) + gqr[2] * L(7, dj, dk); };
        T t1 = d4(pr[0], pr[1], pr[3], pr[4], cr);
        T t2 = d4(p1L(-2, 0), p1L(-1, 0), p1L(1, 0), p1L(2, 0), ct);
        T t3 = d4(p1L(0, -2), p1L(0, -1), p1L(0, 1), p1L(0, 2), cp);
        T g2 = t2 * rinv;
        T g3 = (t3 * rinv) * sinv;
        R[1] = R[1] - over_rho0(t1);
        R[2] = R[2] - over_rho0(g2);
        R[3] = R[3] - over_rho0(g3);
    }
    // Lorentz force (:97-116): curl(B) (ModSpherical.f90:38-102) x B / rho0
    {
        T o1 = d4(L(6, -2, 0) * st[0], L(6, -1, 0) * st[1], L(6, 1, 0) * st[3], L(6, 2, 0) * st[4], ct) -
               d4(L(5, 0, -2), L(5, 0, -1), L(5, 0, 1), L(5, 0, 2), cp);
        T o2 = d4_over_st(L(4, 0, -2), L(4, 0, -1), L(4, 0, 1), L(4, 0, 2)) -
               d4(W(6, 0) * xr[0], W(6, 1) * xr[1], W(6, 3) * xr[3], W(6, 4) * xr[4], cr);
        T o3 = d4(W(5, 0) * xr[0], W(5, 1) * xr[1], W(5, 3) * xr[3], W(5, 4) * xr[4], cr) -
               d4(L(4, -2, 0), L(4, -1, 0), L(4, 1, 0), L(4, 2, 0), ct);
        o1 = o1 * rinv; o2 = o2 * rinv; o3 = o3 * rinv;
        o1 = o1 * sinv;
        T c1 = o2 * bp - o3 * bt;
        T c2 = o3 * br - o1 * bp;
        T c3 = o1 * bt - o2 * br;
        R[1] = R[1] + over_rho0(c1);
        R[2] = R[2] + over_rho0(c2);
        R[3] = R[3] + over_rho0(c3);
    }
    // Gravity (:121-127)
    R[1] = R[1] - gor * W(0, 2);
    // Entropy advection and heating (:132-151)
    R[7] = -adg(7);
    R[7] = R[7] + heat;
    // Induction (:154-162): curl(v x B), cross product per point (ModSpherical.f90:26-36)
    {
        auto e1L = [&](int dj, int dk) -> T { return L(2, dj, dk) * L(6, dj, dk) - L(3, dj, dk) * L(5, dj, dk); };
        auto e2L = [&](int dj, int dk) -> T { return L(3, dj, dk) * L(4, dj, dk) - L(1, dj, dk) * L(6, dj, dk); };
        auto e3L = [&](int dj, int dk) -> T { return L(1, dj, dk) * L(5, dj, dk) - L(2, dj, dk) * L(4, dj, dk); };
        T e2r[5], e3r[5];
#pragma unroll
        for (int q = 0; q < 5; q++) {
            e2r[q] = W(3, q) * W(4, q) - W(1, q) * W(6, q);
            e3r[q] = W(1, q) * W(5, q) - W(2, q) * W(4, q);
        }
        T o1 = d4(e3L(-2, 0) * st[0], e3L(-1, 0) * st[1], e3L(1, 0) * st[3], e3L(2, 0) * st[4], ct) -
               d4(e2L(0, -2), e2L(0, -1), e2L(0, 1), e2L(0, 2), cp);
        T o2 = d4_over_st(e1L(0, -2), e1L(0, -1), e1L(0, 1), e1L(0, 2)) -
               d4(e3r[0] * xr[0], e3r[1] * xr[1], e3r[3] * xr[3], e3r[4] * xr[4], cr);
        T o3 = d4(e2r[0] * xr[0], e2r[1] * xr[1], e2r[3] * xr[3], e2r[4] * xr[4], cr) -
               d4(e1L(-2, 0), e1L(-1, 0), e1L(1, 0), e1L(2, 0), ct);
        o1 = o1 * rinv; o2 = o2 * rinv; o3 = o3 * rinv;
        o1 = o1 * sinv;
        R[4] = o1; R[5] = o2; R[6] = o3;
    }
}

// T is the storage type of the stage input (the LDS planes and the register
// window); the right-hand side is computed in FP64 for either.  Stage values
// stored in FP32 are the FP32 path's only rounding: FP32 arithmetic on the
// stencils and FP32 copies of the metric and background coefficients were
// each measured to put 1e-6 of error into the 100-step FP32-vs-FP64 state on
// the 50 M-cell shell, FP32 storage alone 5e-7.
// MODE 0: out = U + (dt*R)/div on the interior (3_6/ModAdvance.f90:87-93), the
//         sum formed in FP64 from the base U of type TB (the FP64 state, or for
//         the FP32 path's intermediate stages its FP32 copy: those stage values
//         are stored in FP32 anyway); with SHADOW the same value is also stored
//         rounded to FP32 in `shadow`.
// MODE 1: write R (interior layout [block][var][i][j][k], FP64) for parity tests.
// pull (null: none): ghost cells of `in` in the directions it lists are read
// from the same-level neighbour's interior (Marcher).
// GLM (FP64 only): grad(psi) from `glm` is subtracted from R(B) (GLM
// divergence cleaning); a separate instantiation, so the plain one is unchanged.
// The body is shared by two kernels, k_stage and k_stage_w2 (below).
template <typename T, typename TIN, typename TOUT, typename TB, int MODE, bool SHADOW, int TL, bool PERSIST,
          bool GLM = false>
__device__ __forceinline__ void stage_body(Dims d, DevTables t, const TIN *__restrict__ in,
                                               const TB *__restrict__ U, TOUT *__restrict__ out,
                                               float *__restrict__ shadow, const double *__restrict__ dtp,
                                               double div, const int32_t *__restrict__ pull,
                                               const double *__restrict__ glm, int nseg) {
    constexpr int PL = tile_pl<TL>();
    __shared__ T lds[2][8][PL][PL];
    // LEAN (FP32 storage): the block's radial coefficient rows (xi, rho0, gp,
    // gq, rinv, r2inv, xir2, heat, g/rho0, and 1/rho0) are staged in LDS once
    // per tile, U of the plane is loaded at the top of the plane, and the next
    // plane's loads are issued unconditionally from clamped addresses.  The
    // plane loop then waits on no global load in the middle of its arithmetic
    // (a load issued after the prefetch would wait for the prefetch too), which
    // took the FP32 stage from 2.99 to 2.78 ms per launch on the 50 M-cell
    // shell.  The FP64 instantiation keeps the table loads: with the LDS rows
    // its register demand exceeds two wavefronts per SIMD.
    constexpr bool LEAN = sizeof(T) == 4;
    __shared__ double crow[kStageRows][kMaxNI];
    const int ntk = (d.nk + TL - 1) / TL, tpb = ((d.nj + TL - 1) / TL) * ntk;
    const int ntot = d.nblocks * tpb * nseg;
    // PERSIST: a grid smaller than the tile count (a persistent launch) takes
    // the next tile at a stride of the grid size; otherwise one pass, tile =
    // the workgroup.  A tile's march is cut into nseg radial segments
    // (march_segments), the segments of a tile consecutive.
    for (int tile = PERSIST ? (int)blockIdx.x : xcd_tile(blockIdx.x, ntot); tile < ntot; tile += gridDim.x) {
        const int tcol = tile / nseg, seg = tile - tcol * nseg;
        const int iA = seg * d.ni / nseg, iB = (seg + 1) * d.ni / nseg;
        const int b = tcol / tpb;
        const int trem = tcol - b * tpb;
        const int tj = trem / ntk, tk = trem - tj * ntk;
        const int j0 = tj * TL, k0 = tk * TL;
        const int TJa = min(TL, d.nj - j0), TKa = min(TL, d.nk - k0);
        const int tx = threadIdx.x & (TL - 1), ty = threadIdx.x / TL;

        constexpr bool PULL = sizeof(T) == 4 && MODE == 0;
        Marcher<T, TIN, PULL, TL> m;
        m.init(d, in, b, j0, k0, TJa, TKa, pull);

        const long long rb = (long long)b * d.NI, tb = (long long)b * d.NJ;
        if (LEAN) {
    #pragma unroll
            for (int r = 0; r < 9; r++) {
                const double *src = r == 0 ? t.xi : r == 1 ? t.rho0 : r == 2 ? t.gp : r == 3 ? t.gq : r == 4 ? t.rinv
                                  : r == 5 ? t.r2inv : r == 6 ? t.xir2 : r == 7 ? t.heat : t.g_over_rho0;
                for (int I = threadIdx.x; I < d.NI; I += TL * TL) crow[r][I] = src[rb + I];
            }
            // 1/rho0 for the reciprocal form of the FP32 path's right-hand side
            for (int I = threadIdx.x; I < d.NI; I += TL * TL) crow[9][I] = 1.0 / t.rho0[rb + I];
        }
        const BlockMeta mt = t.meta[b];
        // the right-hand side is computed in FP64 whatever the storage type T:
        // coefficients from the FP64 tables, stage values widened on use
        const double cr = mt.cr, ct = mt.ct, cp = mt.cp;
        // theta rows are read only by active lanes (inactive lanes of a partial
        // tile have J beyond the padded range)
        double st[5];
    #pragma unroll
        for (int q = 0; q < 5; q++) st[q] = m.act ? t.sint[tb + m.J - 2 + q] : 1.0;
        const double sinv = m.act ? t.sinv[tb + m.J] : 1.0, cot = m.act ? t.cot[tb + m.J] : 0.0;
        const double dt = MODE == 0 ? *dtp : 0.0;
        // the FP32 path's reciprocal form (cell_rhs): the stage increment
        // (dt*R)/(5-k) as a product with 1/(5-k)
        constexpr bool RECIP = LEAN;
        const double rdiv = 1.0 / div, ydiv = div_rcp(div);

        T win[8][5];
        T nxt[8], hn[8];
    #pragma unroll
        for (int v = 0; v < 8; v++) {
    #pragma unroll
            for (int q = 0; q < 5; q++) win[v][q] = m.col(v, iA + q);
            hn[v] = m.halo(v, iA + d.ng);
        }
        const long long bbase = (long long)b * 8 * d.P;
        // G ([block][3][interior cells]) at this lane's column; plane i at + i nj nk
        const long long gnn = (long long)d.ni * d.nj * d.nk;
        const double *gcol = GLM ? glm + (b * 3 * gnn + ((long long)(j0 + ty) * d.nk + (k0 + tx))) : nullptr;

        for (int i = iA; i < iB; i++) {
            const int I = i + d.ng;
            const int buf = i & 1;
            // U of this plane, issued first: the plane's arithmetic covers its latency
            TB ub[8];
            if (MODE == 0 && LEAN) {
    #pragma unroll
                for (int v = 0; v < 8; v++) ub[v] = (U + (bbase + (long long)v * d.P + (long long)I * m.SI))[m.coff];
            }
            // stage this plane: own column centre plus halo strips
    #pragma unroll
            for (int v = 0; v < 8; v++) {
                if (m.act) lds[buf][v][ty + 2][tx + 2] = win[v][2];
                if (m.hv) lds[buf][v][m.hly][m.hlx] = hn[v];
            }
            // prefetch the next window plane and the next halo (on the last plane
            // the clamped loads are discarded; FP64 16-edge tiles leave them out, where
            // the 8-edge ones would spill 16 registers for the branch: 50.5 against
            // 48 us per launch on 648 8^3 blocks)
            const int In = min(I + 3, d.NI - 1), Ih = min(I + 1, d.NI - 1);
            const bool more = i + 1 < iB;
    #pragma unroll
            for (int v = 0; v < 8; v++) {
                nxt[v] = (LEAN || TL == 8 || (m.act && more)) ? m.col(v, In) : T(0);
                hn[v] = (LEAN || TL == 8 || (m.hv && more)) ? m.halo(v, Ih) : T(0);
            }
            __syncthreads();
            if (m.act) {
                // coefficient row r at plane I: LDS (FP32 path) or the table itself
                auto coef = [&](int r, int II) -> double {
                    if (LEAN) return crow[r][II];
                    const double *src = r == 0 ? t.xi : r == 1 ? t.rho0 : r == 2 ? t.gp : r == 3 ? t.gq : r == 4 ? t.rinv
                                      : r == 5 ? t.r2inv : r == 6 ? t.xir2 : r == 7 ? t.heat : t.g_over_rho0;
                    return src[rb + II];
                };
                double xr[5], rho0r[5], gpr[5], gqr[5];
    #pragma unroll
                for (int q = 0; q < 5; q++) {
                    xr[q] = coef(0, I - 2 + q);
                    rho0r[q] = coef(1, I - 2 + q);
                    gpr[q] = coef(2, I - 2 + q);
                    gqr[q] = coef(3, I - 2 + q);
                }
                auto L = [&](int v, int dj, int dk) -> double { return (double)lds[buf][v][ty + 2 + dj][tx + 2 + dk]; };
                double R[8];
                cell_rhs<double, T, RECIP>(win, L, xr, rho0r, gpr, gqr, st, coef(4, I), coef(5, I), coef(6, I),
                                           coef(7, I), coef(8, I), sinv, cot, cr, ct, cp,
                                           RECIP ? coef(9, I) : div_rcp(t.rho0_up[rb + I]),
                                           RECIP ? 1.0 : t.rho0_up[rb + I], R);
                if (MODE == 0) {
                    if constexpr (GLM && sizeof(T) == 8) {
                        // ModDivB_GLM (3_6/ModDivB.f90:27-28): R(B) = R(B) - grad(psi)
                        const double *gi = gcol + i * (d.nj * d.nk);
                        R[4] = R[4] - gi[0];
                        R[5] = R[5] - gi[gnn];
                        R[6] = R[6] - gi[2 * gnn];
                    }
                    const long long base = bbase + (long long)I * m.SI;
    #pragma unroll
                    for (int v = 0; v < 8; v++) {
                        const long long q = base + (long long)v * d.P;
                        const double inc = RECIP ? (dt * R[v]) * rdiv : div_by((dt * R[v]) * kDivUp, div, ydiv);
                        const double x = (double)(LEAN ? ub[v] : (U + q)[m.coff]) + inc;
                        (out + q)[m.coff] = (TOUT)x;
                        if (SHADOW) (shadow + q)[m.coff] = (float)x;
                    }
                } else {
                    const long long nn = (long long)d.ni * d.nj * d.nk;
                    const long long base = (long long)b * 8 * nn + ((long long)i * d.nj + (j0 + ty)) * d.nk + (k0 + tx);
    #pragma unroll
                    for (int v = 0; v < 8; v++) ((double *)out)[base + (long long)v * nn] = (double)R[v];
                }
            }
    #pragma unroll
            for (int v = 0; v < 8; v++) {
                win[v][0] = win[v][1]; win[v][1] = win[v][2]; win[v][2] = win[v][3]; win[v][3] = win[v][4];
                win[v][4] = nxt[v];
            }
        }
        if (!PERSIST) break;
        // the next tile's LDS writes wait for this tile's last reads
        if (tile + (int)gridDim.x < ntot) __syncthreads();
    }
}

template <typename T, typename TIN, typename TOUT, typename TB, int MODE, bool SHADOW, int TL, bool PERSIST,
          bool GLM = false>
__global__ void __launch_bounds__(TL * TL) k_stage(Dims d, DevTables t, const TIN *__restrict__ in,
                                               const TB *__restrict__ U, TOUT *__restrict__ out,
                                               float *__restrict__ shadow, const double *__restrict__ dtp,
                                               double div, const int32_t *__restrict__ pull,
                                               const double *__restrict__ glm, int nseg) {
    stage_body<T, TIN, TOUT, TB, MODE, SHADOW, TL, PERSIST, GLM>(d, t, in, U, out, shadow, dtp, div, pull, glm, nseg);
}

// The FP64 step's stage (16-edge tiles, one workgroup per tile) held to two
// wavefronts per SIMD: left to itself the compiler gives it one (3.9 instead of 2.9
// ms on 12288 16^3 blocks); held to two it takes 250 VGPRs without a spill.  392 us on
// 1536 blocks, 1.55 GB at 4.0 TB/s: bound by the latency of its loads at two
// wavefronts per SIMD (62% of their life waiting on a dependency, the SIMD's VALU
// 28% busy).  The other builds either fit two wavefronts already (the FP32 stages)
// or would spill tens of registers.
template <typename T, typename TIN, typename TOUT, typename TB, int MODE, bool SHADOW, int TL, bool PERSIST,
          bool GLM = false>
__global__ void __launch_bounds__(TL * TL) __attribute__((amdgpu_waves_per_eu(2)))
k_stage_w2(Dims d, DevTables t, const TIN *__restrict__ in, const TB *__restrict__ U, TOUT *__restrict__ out,
           float *__restrict__ shadow, const double *__restrict__ dtp, double div,
           const int32_t *__restrict__ pull, const double *__restrict__ glm, int nseg) {
    stage_body<T, TIN, TOUT, TB, MODE, SHADOW, TL, PERSIST, GLM>(d, t, in, U, out, shadow, dtp, div, pull, glm, nseg);
}

// ---------------------------------------------------------------- diffusion

// Radial mirror parities of ModBoundary_Dynamo_primitives (3_6/ModBoundary.f90:
// 16-52) for rho1, vr, vt, vp, br, bt, bp, s1: bottom (inner) and top (outer).
__constant__ double kParBottom[8] = {1.0, -1.0, 1.0, 1.0, -1.0, 1.0, 1.0, 1.0};
__constant__ double kParTop[8] = {1.0, -1.0, 1.0, 1.0, 1.0, -1.0, -1.0, 1.0};

// ModDiffusion_Aritificial_1 (3_6/ModDiffusion.f90:9-150), h = 2, all 8 vars.
// The characteristic speed c of each face is read where the reference reads it:
// the section c(1:ni+1,:,:) (:63) spans the padded transverse range while flux
// spans 1:nj,1:nk, so the speed comes from transverse index (index - ng); same
// for :96 and :130.
// MODE 0: out = U + (0.5*dt)*R (3_6/ModAdvance.f90:104-107); `shadow` (if not
// null) receives the same value in FP32, and the workgroup's min(h/v_wave) of the
// new state (the next step's ModTimeStep_Dynamo input) goes to partial[tile], one
// per tile and radial segment.
// MODE 1: write R.  `in` is the stencil input (the state or its FP32 shadow).
// FP32 path (T = float, MODE 0): U and out are the same buffer, updated in
// place, and Uold is U^n.  The radial ghosts of the input are the mirror of
// U^n that the first stage's boundary call left (the reference applies
// boundaries only to each stage's input), while the interior is the state
// after the fourth stage; at the domain's radial boundary faces the limiter
// therefore divides by the one-step change of the first cell, which FP32
// cannot resolve.  There the face flux is formed in FP64 from U^n (mirrored
// with the parities of ModBoundary_Dynamo_primitives, 3_6/ModBoundary.f90:
// 16-52) and the FP64 state, as the FP64 path forms it.  Elsewhere the FP32
// path's fluxes are computed in FP32: on the 50 M-cell shell FP64 fluxes
// changed the 100-step FP32-vs-FP64 difference only from 5.2e-7 to 5.5e-7
// (largest variable) and cost 0.8 ms per step.

// A plane takes three phases: half slopes of every cell along theta and phi
// (each formed once, where the reference's whole-array reconstruction is read
// by both faces of a cell), then the upper theta and phi face of every cell
// from its own and its neighbour's half slope, then the cell's update with the
// lower faces of its neighbours; the radial face and slope are carried from
// plane to plane.  The halo cells' half slopes (4 tile edges) and the faces on
// the tile's lower edges are spread one variable a lane over the whole
// workgroup: done by the first wavefront for all variables, as before, the
// others waited about a fifth of the plane for it.  FP64 takes the phases in
// two passes of four variables, so that two workgroups fit a CU's LDS.
// Bound by vector instructions and the latency of a plane's chain: on either path
// the SIMD's VALU is 60% busy at two wavefronts (FP64 1.5 GB at 3.3 TB/s, FP32
// 1.6 GB at 4.3 TB/s).  Against one
// pass that recomputed the slopes per face and kept a five-plane window, with
// the general divisions and the edges on the first wavefront: FP64 706 -> 476
// us, FP32 490 -> 360 us on 1536 16^3 blocks; 192 blocks 105 -> 83 and 91 -> 72
// us.  FP64 held to two wavefronts per SIMD spills 28 bytes per lane; with the
// eight variables in one pass 124 bytes (607 us).
template <typename T, typename TIN, int MODE, int TL, bool PERSIST>
__global__ void __launch_bounds__(TL * TL) __attribute__((amdgpu_waves_per_eu(2)))
k_diffusion(Dims d, DevTables t, const TIN *__restrict__ in, const double *U, double *out,
            float *__restrict__ shadow, double *__restrict__ partial, const double *__restrict__ dtp,
            const int32_t *__restrict__ pull, const double *__restrict__ Uold, int nseg) {
    constexpr int PL = tile_pl<TL>(), NL = TL * TL;
    constexpr bool F32 = sizeof(T) == 4;
    // FP32 path in a step: pulled ghosts, boundary faces from U^n, reciprocals
    constexpr bool LEAN = F32 && MODE == 0, PULL = LEAN, BFACE = LEAN;
    // one r-plane with its theta/phi halo; the barriers of a plane order its
    // reuse, so it is not double-buffered
    __shared__ T lds[8][PL][PL];
    // of the pass's variables: half slopes along theta, sj(v, y+1, x) for tile
    // rows y = -1 .. TJa, and phi, sk(v, y, x+1) for tile columns x = -1 .. TKa;
    // face fluxes fj(v, y, x) through the lower theta face of tile cell (y, x)
    // (row TJa: the upper face of the last row), fk(v, y, x) through its lower
    // phi face
    constexpr int NV = F32 ? 8 : 4, NSJ = (TL + 2) * TL, NFJ = (TL + 1) * TL;
    __shared__ T sbuf[2][NV][NSJ];
    __shared__ T fbuf[2][NV][NFJ];
    auto sj = [&](int v, int y, int x) -> T & { return sbuf[0][v % NV][y * TL + x]; };
    auto sk = [&](int v, int y, int x) -> T & { return sbuf[1][v % NV][y * (TL + 2) + x]; };
    auto fj = [&](int v, int y, int x) -> T & { return fbuf[0][v % NV][y * TL + x]; };
    auto fk = [&](int v, int y, int x) -> T & { return fbuf[1][v % NV][y * (TL + 1) + x]; };
    __shared__ double red[4];
    // block read in place of this block's ghosts in direction code c (the
    // pull table's row, -1 where the ghost itself is read)
    __shared__ int pdir[27];
    // the block's radial rows c_s, xi, sqrt(rho0): staged in a step so that no
    // plane waits on a load issued after its prefetch
    __shared__ double drow[3][MODE == 0 ? kMaxNI : 1];
    const int ntk = (d.nk + TL - 1) / TL, tpb = ((d.nj + TL - 1) / TL) * ntk;
    const int ntot = d.nblocks * tpb * nseg;
    // PERSIST: a grid smaller than the tile count (a persistent launch) takes
    // the next tile at a stride of the grid size; otherwise one pass, tile =
    // the workgroup.  nseg: radial segments per tile, as in stage_body; a
    // segment forms its first plane's lower r-face itself and has at least two
    // planes (march_segments), which the FP32 path's boundary faces need.
    for (int tile = PERSIST ? (int)blockIdx.x : xcd_tile(blockIdx.x, ntot); tile < ntot; tile += gridDim.x) {
        const int tcol = tile / nseg, seg = tile - tcol * nseg;
        const int iA = seg * d.ni / nseg, iB = (seg + 1) * d.ni / nseg;
        const int b = tcol / tpb;
        if (PULL && threadIdx.x < 27) pdir[threadIdx.x] = pull ? pull[b * 27 + threadIdx.x] : -1;
        const int trem = tcol - b * tpb;
        const int tj = trem / ntk, tk = trem - tj * ntk;
        const int j0 = tj * TL, k0 = tk * TL;
        const int TJa = min(TL, d.nj - j0), TKa = min(TL, d.nk - k0);
        const int lane = threadIdx.x, tx = lane & (TL - 1), ty = lane / TL;

        Marcher<T, TIN, PULL, TL> m;
        m.init(d, in, b, j0, k0, TJa, TKa, pull);
        const long long rb = (long long)b * d.NI, tb = (long long)b * d.NJ;
        if constexpr (MODE == 0) {
            for (int I = lane; I < d.NI; I += NL) {
                drow[0][I] = t.cs[rb + I];
                drow[1][I] = t.xi[rb + I];
                drow[2][I] = t.sqrt_rho0[rb + I];
            }
        }
        auto cs_at = [&](int I) -> double { return MODE == 0 ? drow[0][MODE == 0 ? I : 0] : t.cs[rb + I]; };
        auto xi_at = [&](int I) -> double { return MODE == 0 ? drow[1][MODE == 0 ? I : 0] : t.xi[rb + I]; };
        const BlockMeta mt = t.meta[b];
        const T dxi = (T)mt.dxi, dxj = (T)mt.dxj, dxk = (T)mt.dxk;
        // the face sums are divided by the cell lengths: products with hardware
        // reciprocals (LEAN), div_by (FP64, the correctly rounded quotient) or
        // plain divisions
        auto recip = [](T x) -> T {
            if constexpr (!F32) return div_rcp(x);
            else return (T)__builtin_amdgcn_rcpf((float)x);
        };
        auto over = [](T f, T x, T y) -> T {
            if constexpr (!F32) return div_by(f, x, y);
            else return LEAN ? f * y : f / x;
        };
        const T ydxi = recip(dxi);
        double hmin = INFINITY;
        const double sint64 = m.act ? t.sint[tb + m.J] : 1.0;
        const T sintc = m.act ? (T)t.sint[tb + m.J] : T(1);
        const double dt = MODE == 0 ? *dtp : 0.0;
        const double dts = (0.5 * kFluxScale) * dt;
        __syncthreads();   // pdir, drow

        // Column (JJ, KK) of variable v from padded plane II, which lies in radial
        // direction di of the block (-1, 0, 1: below, inside, above its interior):
        // address of that plane, and the plane pitch.  A ghost in a direction listed
        // in the pull table is the same-level neighbour's interior cell, translated
        // by n.
        struct Col {
            const TIN *p;
            int pitch;
        };
        auto column = [&](int v, int II, int JJ, int KK, int di) -> Col {
            int B = b, sh = 0;
            if (PULL) {
                const int dj = JJ < d.ng ? -1 : (JJ >= d.ng + d.nj ? 1 : 0);
                const int dk = KK < d.ng ? -1 : (KK >= d.ng + d.nk ? 1 : 0);
                const int D = pdir[(di + 1) * 9 + (dj + 1) * 3 + (dk + 1)];
                if ((di | dj | dk) && D >= 0) {
                    B = D;
                    sh = di * d.ni; JJ -= dj * d.nj; KK -= dk * d.nk;
                }
            }
            Col c;
            c.pitch = (KK >= d.ng && KK < d.ng + d.nk) ? (int)d.SI : d.NJ * 2 * d.ng;
            c.p = in + ((long long)B * 8 + v) * d.P + cell_off(d, 0, JJ, KK) + (long long)(II - sh) * c.pitch;
            return c;
        };
        // |value| of the column's plane; the column steps to the next plane
        auto step = [](Col &c) -> T {
            const T x = fabs((T)*c.p);
            c.p += c.pitch;
            return x;
        };
        // Speeds |v_d| + c_s are read where the reference reads them (transverse
        // index - ng): (I-2, J, K-2) and (I-2, J+1, K-2) for theta, (I-2, J-2, K)
        // and (I-2, J-2, K+1) for phi, (., J-2, K-2) for r.  Inactive lanes read at
        // the tile's first column.
        const int J = m.act ? m.J : j0 + d.ng, K = m.act ? m.K : k0 + d.ng;
        // faces on the tile's lower edges, one (position, variables) a lane:
        // positions 0 .. TL-1 are the theta faces below row 0, TL .. 2TL-1 the phi
        // faces left of column 0; the lane's variables are ev, ev + EV, ...
        constexpr int EV = NL / (2 * TL);
        const int ep = lane & (2 * TL - 1), ev = lane / (2 * TL);
        const bool bj = ep < TL;
        const int bx = bj ? ep : 0, by = bj ? 0 : ep - TL;
        const bool bact = bj ? bx < TKa : by < TJa;
        const int bvar = bj ? 2 : 3;
        const int bJ0 = !bact ? j0 + d.ng : bj ? j0 + d.ng : j0 + by + d.ng - 2,
                  bK0 = !bact ? k0 + d.ng : bj ? k0 + bx + d.ng - 2 : k0 + d.ng;
        const int bJ1 = bj ? bJ0 - 1 : bJ0, bK1 = bj ? bK0 : bK0 - 1;
        Col q20, q2p, q30, q3p, q1, qe0, qe1;
        auto theta_phi_columns = [&](int II, int di) {
            q20 = column(2, II, J, K - 2, di);
            q2p = column(2, II, J + 1, K - 2, di);
            q30 = column(3, II, J - 2, K, di);
            q3p = column(3, II, J - 2, K + 1, di);
            qe0 = column(bvar, II, bJ0, bK0, di);
            qe1 = column(bvar, II, bJ1, bK1, di);
        };
        // planes I - 2 = i of the theta and phi speeds leave the ghost range at i = ng
        theta_phi_columns(iA, iA < d.ng ? -1 : 0);
        // |v_r| of the radial faces' cells at planes I - 1 (first plane), I and I + 1
        q1 = column(1, iA + d.ng - 1, J - 2, K - 2, iA == 0 ? -1 : 0);
        const T v1m = step(q1);
        if (iA == 0) q1 = column(1, d.ng, J - 2, K - 2, 0);
        T v1c = step(q1), v1n;

        // window: this plane and the two above it
        T w0[8], w1[8], w2[8];
        T nxt[8], hn[8];
        // the upper r-face of plane i is the lower r-face of plane i+1: same four
        // values, same speed sum (speed at the upper cell first); carried with the
        // half slope of the cell above
        T fr[8], sr[8];
        // FP32 path: U before the diffusion on the previous plane (the top
        // boundary face reads it after that plane has been updated in place)
        double uprev[8];
        const bool bot = BFACE && (mt.flags & 1), topb = BFACE && (mt.flags & 2);
        const long long bbase = (long long)b * 8 * d.P;
        {
            const T cm = v1m + (T)cs_at(iA + d.ng - 1);
            const T cc = v1c + (T)cs_at(iA + d.ng);
    #pragma unroll
            for (int v = 0; v < 8; v++) {
                const T a = m.col(v, iA), c = m.col(v, iA + 1);
                w0[v] = m.col(v, iA + 2);
                w1[v] = m.col(v, iA + 3);
                w2[v] = m.col(v, iA + 4);
                hn[v] = m.halo(v, iA + d.ng);
                sr[v] = half_slope(c, w0[v], w1[v]);
                fr[v] = face_flux<T, LEAN>(c, w0[v], half_slope(a, c, w0[v]), sr[v]) * (cc + cm);
                if (BFACE && bot && iA == 0) {
                    // lower face of the first cell: ghosts 0 and -1 mirror cells 1 and 2 of U^n
                    const long long q = bbase + (long long)d.ng * m.SI + (long long)v * d.P + m.coff;
                    const double p = kParBottom[v];
                    const double g0 = p * Uold[q], gm1 = p * Uold[q + m.SI];
                    fr[v] = (T)(face_flux4<double>(gm1, g0, U[q], U[q + m.SI]) * (double)(cc + cm));
                }
            }
        }

        for (int i = iA; i < iB; i++) {
            const int I = i + d.ng;
            // U^n of the plane (LEAN; FP64's is the input itself) and |v_d| at the
            // shifted speed cells, issued before the prefetch
            double ucur[8];
            if (LEAN) {
    #pragma unroll
                for (int v = 0; v < 8; v++) ucur[v] = (U + (bbase + (long long)v * d.P + (long long)I * m.SI))[m.coff];
            }
            if (i == d.ng) theta_phi_columns(i, 0);
            if (i == d.ni - 1) q1 = column(1, I + 1, J - 2, K - 2, 1);
            const T a20 = step(q20), a2p = step(q2p), a30 = step(q30), a3p = step(q3p);
            const T ae0 = step(qe0), ae1 = step(qe1);
            v1n = step(q1);
    #pragma unroll
            for (int v = 0; v < 8; v++) {
                if (m.act) lds[v][ty + 2][tx + 2] = w0[v];
                if (m.hv) lds[v][m.hly][m.hlx] = hn[v];
            }
            const int In = min(I + 3, d.NI - 1), Ih = min(I + 1, d.NI - 1);
    #pragma unroll
            for (int v = 0; v < 8; v++) {
                nxt[v] = m.col(v, In);
                hn[v] = m.halo(v, Ih);
            }
            __syncthreads();
            auto Lv = [&](int v, int dj, int dk) -> T { return lds[v][ty + 2 + dj][tx + 2 + dk]; };
            const T csI2 = (T)cs_at(i), csI = (T)cs_at(I), csIp = (T)cs_at(I + 1);
            const T S2 = (a2p + csI2) + (a20 + csI2), S3 = (a3p + csI2) + (a30 + csI2);
            const T Se = (ae0 + csI2) + (ae1 + csI2);
            const T S1 = (v1n + csIp) + (v1c + csI);
            const T xic = (T)xi_at(I);
            const T L2 = dxj * xic;
            const T L3 = (dxk * xic) * sintc;
            const T y2 = recip(L2), y3 = recip(L3);
            const long long base = bbase + (long long)I * m.SI;
            const long long nn = (long long)d.ni * d.nj * d.nk;
            const long long rbase = (long long)b * 8 * nn + ((long long)i * d.nj + (j0 + ty)) * d.nk + (k0 + tx);
            double vv = 0.0, bb2 = 0.0;   // |v|^2 and |B|^2 of the new state, summed in component order
    #pragma unroll
            for (int p0 = 0; p0 < 8; p0 += NV) {
                if (m.act) {
    #pragma unroll
                    for (int v = p0; v < p0 + NV; v++) {
                        sj(v, ty + 1, tx) = half_slope(Lv(v, -1, 0), w0[v], Lv(v, 1, 0));
                        sk(v, ty, tx + 1) = half_slope(Lv(v, 0, -1), w0[v], Lv(v, 0, 1));
                    }
                }
                // halo cells next to the tile: rows -1 and TJa (theta), columns -1 and TKa (phi)
    #pragma unroll
                for (int h = lane; h < 4 * TL * NV; h += NL) {
                    const int v = p0 + h / (4 * TL), q = (h / TL) & 3, x = h & (TL - 1);
                    if (x < (q < 2 ? TKa : TJa)) {
                        const int y = q == 0 ? -1 : (q == 1 ? TJa : x), xx = q < 2 ? x : (q == 2 ? -1 : TKa);
                        const int st = q < 2 ? PL : 1;
                        const T *pc = &lds[v][y + 2][xx + 2];
                        const T sl = half_slope(pc[-st], pc[0], pc[st]);
                        if (q < 2) sj(v, y + 1, x) = sl;
                        else sk(v, x, xx + 1) = sl;
                    }
                }
                __syncthreads();
                if (m.act) {
    #pragma unroll
                    for (int v = p0; v < p0 + NV; v++) {
                        fj(v, ty + 1, tx) = face_flux<T, LEAN>(w0[v], Lv(v, 1, 0), sj(v, ty + 1, tx), sj(v, ty + 2, tx)) * S2;
                        fk(v, ty, tx + 1) = face_flux<T, LEAN>(w0[v], Lv(v, 0, 1), sk(v, ty, tx + 1), sk(v, ty, tx + 2)) * S3;
                    }
                }
                if (bact) {
    #pragma unroll
                    for (int v = p0 + ev; v < p0 + NV; v += EV) {
                        const T *pv = &lds[v][by + 2][bx + 2];
                        const T lo = bj ? pv[-PL] : pv[-1];
                        const T f = face_flux<T, LEAN>(lo, pv[0], bj ? sj(v, 0, bx) : sk(v, by, 0),
                                                       bj ? sj(v, 1, bx) : sk(v, by, 1)) * Se;
                        if (bj) fj(v, 0, bx) = f;
                        else fk(v, by, 0) = f;
                    }
                }
                __syncthreads();
                if (m.act) {
    #pragma unroll
                    for (int v = p0; v < p0 + NV; v++) {
                        const T su = half_slope(w0[v], w1[v], w2[v]);
                        const T f0 = fr[v];
                        T f1 = face_flux<T, LEAN>(w0[v], w1[v], sr[v], su) * S1;
                        sr[v] = su;
                        if (BFACE && topb && i == d.ni - 1) {
                            // upper face of the last cell: ghosts ni+1 and ni+2 mirror cells ni and ni-1 of U^n
                            const long long q = base + (long long)v * d.P + m.coff;
                            const double p = kParTop[v];
                            const double g1 = p * Uold[q], g2 = p * Uold[q - m.SI];
                            f1 = (T)(face_flux4<double>(uprev[v], ucur[v], g1, g2) * (double)S1);
                        }
                        fr[v] = f1;
                        T r = T(0);
                        r = r + over(f1 - f0, dxi, ydxi);
                        r = r + over(fj(v, ty + 1, tx) - fj(v, ty, tx), L2, y2);
                        r = r + over(fk(v, ty, tx + 1) - fk(v, ty, tx), L3, y3);
                        if (MODE == 0) {
                            const long long q = base + (long long)v * d.P;
                            const double x = (LEAN ? ucur[v] : (double)w0[v]) + dts * (double)r;
                            (out + q)[m.coff] = x;
                            if (LEAN) (shadow + q)[m.coff] = (float)x;
                            if (v == 1) vv = x * x;
                            if (v == 2 || v == 3) vv = vv + x * x;
                            if (v == 4) bb2 = x * x;
                            if (v == 5 || v == 6) bb2 = bb2 + x * x;
                        } else {
                            out[rbase + (long long)v * nn] = kFluxScale * (double)r;
                        }
                    }
                }
            }
            if (m.act) {
                if (MODE == 0) {
                    // ModWaveSpeed_Dynamo (3_6/ModWaveSpeed.f90:12-24) on the new state and
                    // h_LLL (3_6/ModBlock.f90:420-422), as k_dt_tile computes them
                    double w = cs_at(I) + sqrt(vv);
                    w = w + sqrt(bb2) / drow[2][I];
                    const double xi = xi_at(I);
                    double h = mt.dxi, h2 = xi * mt.dxj, h3 = (xi * sint64) * mt.dxk;
                    h = h < h2 ? h : h2;
                    h = h < h3 ? h : h3;
                    const double x = h / w;
                    hmin = x < hmin ? x : hmin;
                }
            }
            v1c = v1n;
    #pragma unroll
            for (int v = 0; v < 8; v++) {
                w0[v] = w1[v]; w1[v] = w2[v]; w2[v] = nxt[v];
                if (BFACE) uprev[v] = ucur[v];
            }
        }
        if (MODE == 0 && partial) {
            // min is exact in any order: wavefront shuffle, then across the wavefronts
            for (int off = 32; off > 0; off >>= 1) {
                double o = __shfl_down(hmin, off, 64);
                hmin = o < hmin ? o : hmin;
            }
            if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = hmin;
            __syncthreads();
            if (threadIdx.x == 0) {
                double r = red[0];
                for (int q = 1; q < TL * TL / 64; q++) r = red[q] < r ? red[q] : r;
                partial[tile] = r;
            }
        }
        if (!PERSIST) break;
        // the next tile's LDS writes wait for this tile's last reads
        if (tile + (int)gridDim.x < ntot) __syncthreads();
    }
}

// ---------------------------------------------------------------- exchange

// ModCommunication_SendRecvGC_new (3_6/ModCommunication.f90:678-721) as a
// table-driven gather: trilinear in the fixed term order of ModMath.f90:283-291
// with FP64 weights and FP64 accumulation, then the Yin-Yang rotation of v and B
// (ModYinYang_VecConv_1D, ModYinYang.f90:59-60).  Each ghost has one donor, and
// donors are read only at interior cells (clamped bases touch a donor ghost only
// with an exactly-zero weight), so entries are independent.

// the trilinear sum in the term order of ModMath.f90:283-291
__device__ __forceinline__ double trilinear8(double f000, double f100, double f010, double f001, double f110,
                                             double f011, double f101, double f111, double wi, double wj, double wk) {
    double t = f000 * (1.0 - wi) * (1.0 - wj) * (1.0 - wk);
    t = t + f100 * (wi) * (1.0 - wj) * (1.0 - wk);
    t = t + f010 * (1.0 - wi) * (wj) * (1.0 - wk);
    t = t + f001 * (1.0 - wi) * (1.0 - wj) * (wk);
    t = t + f110 * (wi) * (wj) * (1.0 - wk);
    t = t + f011 * (1.0 - wi) * (wj) * (wk);
    t = t + f101 * (wi) * (1.0 - wj) * (wk);
    t = t + f111 * (wi) * (wj) * (wk);
    return t;
}

// ModYinYang_VecConv_1D (3_6/ModYinYang.f90:59-60) on B and v
__device__ __forceinline__ void yy_rotate(double (&val)[8], double a, double bb) {
    const double b2 = -(a * val[5]) - bb * val[6];
    const double b3 = -(a * val[6]) + bb * val[5];
    val[5] = b2; val[6] = b3;
    const double v2 = -(a * val[2]) - bb * val[3];
    const double v3 = -(a * val[3]) + bb * val[2];
    val[2] = v2; val[3] = v3;
}

// The radial ghosts that go with a fill, formed by workgroups behind those of the
// entries (they read and write other cells: interior and radial-ghost planes,
// where no entry has its target or a loaded corner).  On their own each was a
// launch of 4 to 8 us between kernels.
// mirror: the radial ghosts of a stage buffer, its interior columns alone (the
//   stage kernels read no other ghost of those planes); parities as k_boundary;
// copy: the radial ghosts of `src` (all columns) into the buffer.
template <typename TS>
__device__ __forceinline__ void fill_tail(const Dims &d, const FillTail &tail, TS *st, unsigned id) {
    const bool mirror = tail.src == nullptr;
    const unsigned nk = (unsigned)(mirror ? d.nk : d.NK), nj = (unsigned)(mirror ? d.nj : d.NJ), ng = (unsigned)d.ng;
    if (id >= (unsigned)tail.bnd.n * ng * nj * nk) return;
    unsigned r = id / nk;
    const int k = (int)(id - r * nk) + (mirror ? d.ng : 0);
    const unsigned q = r / nj;
    const int j = (int)(r - q * nj) + (mirror ? d.ng : 0);
    const unsigned e = q / ng;
    const int g = (int)(q - e * ng);
    const int b = tail.bnd.list[e] >> 1, side = tail.bnd.list[e] & 1;
    const int dI = side ? d.ni + d.ng + g : g, sI = side ? d.ni + d.ng - 1 - g : 2 * d.ng - 1 - g;
    const long long base = (long long)b * 8 * d.P, dst = base + cell_off(d, dI, j, k);
    const long long so = mirror ? base + cell_off(d, sI, j, k) : dst;
    const TS *S = mirror ? st : (const TS *)tail.src;
    const unsigned neg = !mirror ? 0u : (side ? 0x62u : 0x12u);   // as k_boundary
    TS x[8];
#pragma unroll
    for (int v = 0; v < 8; v++) x[v] = S[so + (long long)v * d.P];
#pragma unroll
    for (int v = 0; v < 8; v++) st[dst + (long long)v * d.P] = ((neg >> v) & 1u) ? -x[v] : x[v];
}

// Workgroup of a fill in the order of its sources: runs of kXcdRun workgroups
// go to one XCD, whose L2 then holds the lines they share.
constexpr int kXcdRun = 64;
__device__ __forceinline__ int xcd_run(int wg, int n) {
    const int grp = wg / (8 * kXcdRun), r = wg - grp * 8 * kXcdRun;
    return (grp + 1) * 8 * kXcdRun <= n ? grp * 8 * kXcdRun + (r & 7) * kXcdRun + (r >> 3) : wg;
}

// The FP32 buffers' ghosts: workgroups [0, nw) take the weighted entries, the
// next nl the radial lerps, the rest the copies, so the three kinds run
// together instead of in three launches with three tails.
//   weighted: every corner is loaded (a gather that skips the zero-weight ones
//     measures twice the time); a base on an axis's last cell, whose upper
//     corner would be a ghost that this launch fills, is in the table as the
//     cell before it with weight 1.  THIN: blocks with an axis of one cell, where
//     there is no cell before it; the base stands in for its upper corners;
//   lerp: same-panel entries whose theta/phi weights lie within 1e-12 of 0 or
//     1 and whose r weight does not (neighbours across a radial block face,
//     whose radial spacings differ): the two r corners of the weighted sum;
//   copy: same-panel entries whose weights lie within 1e-12 of 0 or 1
//     (same-level neighbours whose cell centres coincide up to rounding), from
//     the nearest donor cell.
// Bound by HBM and, on small layouts, by launch and tail.  Three launches in
// target-list and destination order took 95 us on 1536 16^3 blocks (500 MB),
// 71 us on 528 refined ones, 20 us on 648 8^3 ones; one launch in source order
// 81, 59 and 13 us, its face ghosts alone 52, 42 and 9 us.
template <bool THIN>
__global__ void __launch_bounds__(256) k_exchange_f32(Dims d, DevGhosts g, DevFill copy, int nwe, int nle, int nce,
                                                      float *__restrict__ st, FillTail tail) {
    const int nw = (nwe + 255) / 256, nl = (nle + 255) / 256, nc = (nce + 255) / 256;
    const long long P = d.P;
    // a base cell is interior along phi, so its corners are in the main part
    const int SI = (int)d.SI, SJ = d.SJ;
    int wg = blockIdx.x;
    if (wg < nw) {
        const int e = xcd_run(wg, nw) * 256 + (int)threadIdx.x;
        if (e >= nwe) return;
        const int2 c = g.weighted.idx[e];
        const double wi = g.w[3 * (long long)e], wj = g.w[3 * (long long)e + 1], wk = g.w[3 * (long long)e + 2];
        const int ci = THIN && d.ni == 1 ? 0 : SI, cj = THIN && d.nj == 1 ? 0 : SJ, ck = THIN && d.nk == 1 ? 0 : 1;
        double val[8];
#pragma unroll
        for (int v = 0; v < 8; v++) {
            const float *F = st + c.y + (long long)v * P;
            const double f000 = F[0], f100 = F[ci], f010 = F[cj], f001 = F[ck], f110 = F[ci + cj], f011 = F[cj + ck],
                         f101 = F[ci + ck], f111 = F[ci + cj + ck];
            val[v] = trilinear8(f000, f100, f010, f001, f110, f011, f101, f111, wi, wj, wk);
        }
        if (c.x < 0) yy_rotate(val, g.rot[2 * (long long)e], g.rot[2 * (long long)e + 1]);
#pragma unroll
        for (int v = 0; v < 8; v++) st[(c.x & 0x7fffffff) + (long long)v * P] = (float)val[v];
        return;
    }
    wg -= nw;
    if (wg < nl) {
        const int e = xcd_run(wg, nl) * 256 + (int)threadIdx.x;
        if (e >= nle) return;
        const int2 c = g.lerp.idx[e];
        const double wi = g.lerp_w[e];
        float f0[8], f1[8];
#pragma unroll
        for (int v = 0; v < 8; v++) {
            const float *F = st + c.y + (long long)v * P;
            f0[v] = F[0];
            f1[v] = F[SI];
        }
#pragma unroll
        for (int v = 0; v < 8; v++) st[c.x + (long long)v * P] = (float)((double)f0[v] * (1.0 - wi) + (double)f1[v] * wi);
        return;
    }
    wg -= nl;
    if (wg >= nc) {
        fill_tail(d, tail, st, (unsigned)(wg - nc) * 256u + threadIdx.x);
        return;
    }
    const int e = xcd_run(wg, nc) * 256 + (int)threadIdx.x;
    if (e >= nce) return;
    const int2 c = copy.idx[e];
    float val[8];
#pragma unroll
    for (int v = 0; v < 8; v++) val[v] = st[c.y + (long long)v * P];
#pragma unroll
    for (int v = 0; v < 8; v++) st[c.x + (long long)v * P] = val[v] + 0.0f;
}

// The FP64 buffers' ghosts.  The entries come in the order of their base
// cells, and runs of kXcdRun workgroups (64 to 256 measure alike, one 6% less) go to one XCD: a donor line is
// then used by neighbouring lanes and workgroups (the two phi faces read the
// same line of a row, the Yin-Yang entries the lines of the plain ones) while
// the L1 or that XCD's L2 holds it.  Bound by HBM: 1536 16^3 blocks read 1731
// and wrote 479 MB per fill in target-list order (342 us) for 403 MB of
// donor rows, 383 MB of ghosts and 172 MB of table; sorted, with the Yin-Yang
// entries behind the plain ones, 881 and 464 MB (277 us), in one sequence and
// in runs of workgroups 240 to 250 us, the face ghosts alone 205 us.  A full
// fill takes both parts of the table through `all`, in one sequence (one part
// after the other reads their shared lines twice: 302 us).  Not kept: staging boxes of donor cells in LDS
// (368 us: whole boxes are read where the ghosts need their shells), one
// contiguous range of workgroups per XCD (312 us), non-temporal table loads
// (no change).
//
// SKIP of zero weights: a corner whose weight factor is exactly zero
// contributes f*0 = +-0 to the reference's sum; it is not loaded and its term
// is +0, which leaves every nonzero result bit-identical (60% of the corner
// loads on the production layouts).
// PSI: also psi of GLM divergence cleaning ([block][P]), a scalar.
template <bool PSI>
__global__ void __launch_bounds__(256) k_exchange_f64(Dims d, DevGhosts64 g, const int32_t *__restrict__ all,
                                                      int n, double *__restrict__ st, double *__restrict__ psi,
                                                      FillTail tail) {
    const int nx = (n + 255) / 256;
    if ((int)blockIdx.x >= nx) {
        fill_tail(d, tail, st, (blockIdx.x - (unsigned)nx) * 256u + threadIdx.x);
        return;
    }
    int e = xcd_run(blockIdx.x, nx) * 256 + (int)threadIdx.x;
    if (e >= n) return;
    if (all) e = all[e];
    const long long P = d.P;
    // the base cell is interior along phi, so its corners are in the main part
    const int SI = (int)d.SI, SJ = d.SJ;
    const int dst0 = g.dst[e], src = g.src[e], dst = dst0 & 0x7fffffff;
    const double wi = g.w[3 * (long long)e], wj = g.w[3 * (long long)e + 1], wk = g.w[3 * (long long)e + 2];
    const bool i0 = wi != 1.0, i1 = wi != 0.0, j0 = wj != 1.0, j1 = wj != 0.0, k0 = wk != 1.0, k1 = wk != 0.0;
    // the two phi corners of each (i, j) pair are adjacent: one 16-byte load
    // per pair (the phi neighbour of a clamped base at the last interior cell
    // is read in bounds and dropped with its zero weight)
    auto value = [&](const double *F) -> double {
        auto ld2 = [](const double *p) -> double2 {
            double2 v;
            __builtin_memcpy(&v, p, sizeof(v));
            return v;
        };
        const double2 z = make_double2(0.0, 0.0);
        const double2 a00 = (i0 && j0) ? ld2(F) : z, a10 = (i1 && j0) ? ld2(F + SI) : z;
        const double2 a01 = (i0 && j1) ? ld2(F + SJ) : z, a11 = (i1 && j1) ? ld2(F + SI + SJ) : z;
        return trilinear8(k0 ? a00.x : 0.0, k0 ? a10.x : 0.0, k0 ? a01.x : 0.0, k1 ? a00.y : 0.0, k0 ? a11.x : 0.0,
                          k1 ? a01.y : 0.0, k1 ? a10.y : 0.0, k1 ? a11.y : 0.0, wi, wj, wk);
    };
    double val[8];
#pragma unroll
    for (int v = 0; v < 8; v++) val[v] = value(st + src + (long long)v * P);
    if (dst0 < 0) yy_rotate(val, g.rot[2 * (long long)e], g.rot[2 * (long long)e + 1]);
#pragma unroll
    for (int v = 0; v < 8; v++) st[dst + (long long)v * P] = val[v];
    // psi has the state's cell layout
    if constexpr (PSI) psi[psi_off(d, dst)] = value(psi + psi_off(d, src));
}

// dt = min(1.e20, CFL * min) of the partial minima, by one workgroup
__device__ __forceinline__ void dt_final(const double *__restrict__ partial, int n, double cfl, double *__restrict__ dtp) {
    double mn = INFINITY;
    for (int i = threadIdx.x; i < n; i += blockDim.x) mn = partial[i] < mn ? partial[i] : mn;
    for (int off = 32; off > 0; off >>= 1) {
        double o = __shfl_down(mn, off, 64);
        mn = o < mn ? o : mn;
    }
    __shared__ double red[4];
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = mn;
    __syncthreads();
    if (threadIdx.x == 0) {
        double r = red[0];
        for (int w = 1; w < (int)(blockDim.x >> 6); w++) r = red[w] < r ? red[w] : r;
        // dt = min(1.e20, CFL*min) (3_6/ModTimeStep.f90:254-262)
        double dt = cfl * r;
        const double big = (double)1.0e20f;
        dtp[0] = dt < big ? dt : big;
    }
}

// ---------------------------------------------------------------- boundary

// ModBoundary_Dynamo_primitives (3_6/ModBoundary.f90:10-55): radial mirror of
// the ng ghost planes of top/bottom blocks over all (j,k), parities per variable.
// The mirror source of the theta/phi ghost columns is a ghost cell of the
// block's own interior plane; with a pull table (see Marcher) those in a listed
// direction are read from the same-level neighbour's interior.
template <typename TS>
__global__ void __launch_bounds__(256) k_boundary(Dims d, DevBoundary bl, TS *__restrict__ st,
                                                  const int32_t *__restrict__ pull, DtFinal dt) {
    // a step's first launch: its last workgroup forms dt
    if (dt.partial && blockIdx.x == gridDim.x - 1) {
        dt_final(dt.partial, dt.n, dt.cfl, dt.dtp);
        return;
    }
    const unsigned plane = (unsigned)(d.NJ * d.NK), per = (unsigned)d.ng * plane;
    const unsigned tid = blockIdx.x * 256u + threadIdx.x;
    if (tid >= per * (unsigned)bl.n) return;
    const int e = (int)(tid / per);
    const unsigned rem = tid - (unsigned)e * per;
    const int g = (int)(rem / plane);
    const unsigned jk = rem - (unsigned)g * plane;
    const int b = bl.list[e] >> 1, side = bl.list[e] & 1;
    int dI, sI;
    if (side) { dI = d.ni + d.ng + g; sI = d.ni + d.ng - 1 - g; }
    else { dI = g; sI = 2 * d.ng - 1 - g; }
    // signs: top (+,-,+,+,+,-,-,+), bottom (+,-,+,+,-,+,+,+)
    const unsigned neg = side ? 0x62u : 0x12u;   // bit v set -> negate variable v
    // (J, K) of this thread's cell, enumerated row by row over the padded plane
    const int J = (int)(jk / (unsigned)d.NK), K = (int)(jk - (unsigned)J * (unsigned)d.NK);
    TS *base = st + (long long)b * 8 * d.P;
    const TS *src = base;
    long long soff = cell_off(d, sI, J, K);
    if (pull) {
        const int dj = J < d.ng ? -1 : (J >= d.ng + d.nj ? 1 : 0);
        const int dk = K < d.ng ? -1 : (K >= d.ng + d.nk ? 1 : 0);
        if (dj | dk) {
            const int D = pull[b * 27 + 9 + (dj + 1) * 3 + (dk + 1)];
            if (D >= 0) {
                src = st + (long long)D * 8 * d.P;
                soff = cell_off(d, sI, J - dj * d.nj, K - dk * d.nk);
            }
        }
    }
    const long long doff = cell_off(d, dI, J, K);
#pragma unroll
    for (int v = 0; v < 8; v++) {
        TS x = src[(long long)v * d.P + soff];
        base[(long long)v * d.P + doff] = ((neg >> v) & 1u) ? -x : x;
    }
}

// ---------------------------------------------------------------- dt

// ModWaveSpeed_Dynamo (3_6/ModWaveSpeed.f90:12-24) and minval(h/v_wave) of
// ModTimeStep_Dynamo (3_6/ModTimeStep.f90:27) over one 16x16 (theta,phi) tile
// column of a block, all r.  Used when the state was set from outside; during
// stepping the diffusion kernel produces the same partials.
template <int TL>
__global__ void __launch_bounds__(TL * TL) k_dt_tile(Dims d, DevTables t, const double *__restrict__ U,
                                                     double *__restrict__ partial, int nseg) {
    __shared__ double red[4];
    const int ntk = (d.nk + TL - 1) / TL, tpb = ((d.nj + TL - 1) / TL) * ntk;
    const int tcol = blockIdx.x / nseg, seg = blockIdx.x - tcol * nseg;
    const int iA = seg * d.ni / nseg, iB = (seg + 1) * d.ni / nseg;
    const int b = tcol / tpb;
    const int trem = tcol - b * tpb;
    const int tj = trem / ntk, tk = trem - tj * ntk;
    const int tx = threadIdx.x & (TL - 1), ty = threadIdx.x / TL;
    const int j = tj * TL + ty, k = tk * TL + tx;
    const long long rb = (long long)b * d.NI, tb = (long long)b * d.NJ;
    const BlockMeta mt = t.meta[b];
    const double *Ub = U + (long long)b * 8 * d.P;
    double mn = INFINITY;
    if (j < d.nj && k < d.nk) {
        const int J = j + d.ng, K = k + d.ng;
        const double st = t.sint[tb + J];
        for (int i = iA; i < iB; i++) {
            const int I = i + d.ng;
            const long long q = cell_off(d, I, J, K);
            const double vr = Ub[q + d.P], vt = Ub[q + 2 * d.P], vp = Ub[q + 3 * d.P];
            const double br = Ub[q + 4 * d.P], bt = Ub[q + 5 * d.P], bp = Ub[q + 6 * d.P];
            double w = t.cs[rb + I] + sqrt(vr * vr + vt * vt + vp * vp);
            w = w + sqrt(br * br + bt * bt + bp * bp) / t.sqrt_rho0[rb + I];
            const double xi = t.xi[rb + I];
            double h = mt.dxi, h2 = xi * mt.dxj, h3 = (xi * st) * mt.dxk;
            h = h < h2 ? h : h2;
            h = h < h3 ? h : h3;
            const double x = h / w;
            mn = x < mn ? x : mn;
        }
    }
    for (int off = 32; off > 0; off >>= 1) {
        double o = __shfl_down(mn, off, 64);
        mn = o < mn ? o : mn;
    }
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = mn;
    __syncthreads();
    if (threadIdx.x == 0) {
        double r = red[0];
        for (int q = 1; q < TL * TL / 64; q++) r = red[q] < r ? red[q] : r;
        partial[blockIdx.x] = r;
    }
}

__global__ void __launch_bounds__(256) k_dt_final(DtFinal f) { dt_final(f.partial, f.n, f.cfl, f.dtp); }

__global__ void k_to_f32(const double *__restrict__ s, float *__restrict__ d, long long n) {
    long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    long long stride = (long long)gridDim.x * blockDim.x;
    for (; i < n; i += stride) d[i] = (float)s[i];
}

// One block's variables in the caller's Fortran order [K][J][I] (I fastest),
// from the cell_off layout; dst is pinned host memory, so a read-back is this
// pass and one copy on the host instead of a device copy and a strided host
// loop.  Bound by the stores over the host link: a workgroup takes 64 (J, I)
// rows x 4 K of a variable and turns them in LDS, so that a wavefront stores
// 512 contiguous bytes, with 32-byte pieces of the rows on the (cached) load
// side.  Read-back of 1536 padded 16^3 blocks 107 -> 72 ms, of 128 64x16x48
// blocks with psi 127 -> 65 ms against the strided host loop.
__global__ void __launch_bounds__(256) k_block_to_host(Dims d, const double *__restrict__ src, double *__restrict__ dst) {
    __shared__ double tile[4][65];
    const int n = d.NI * d.NJ, t = threadIdx.x, p0 = blockIdx.x * 64, K0 = blockIdx.y * 4;
    const double *S = src + (long long)blockIdx.z * d.P;
    double *D = dst + (long long)blockIdx.z * d.P;
    {
        const int p = p0 + (t >> 2), K = K0 + (t & 3);
        if (p < n && K < d.NK) {
            const int J = p / d.NI, I = p - J * d.NI;
            tile[t & 3][t >> 2] = S[cell_off(d, I, J, K)];
        }
    }
    __syncthreads();
    const int p = p0 + (t & 63), K = K0 + (t >> 6);
    if (p < n && K < d.NK) D[(long long)K * n + p] = tile[t >> 6][t & 63];
}

__global__ void k_set_scalar(double *__restrict__ p, double v) {
    if (threadIdx.x == 0) p[0] = v;
}

// Interior difference of two states of one layout, one workgroup per (block,
// variable).  PASS 0: w[v] = max|a-b|, w[8+v] = max|b| (as the bit patterns of
// non-negative doubles, which order like the values).  PASS 1: w[16+v] = cells
// with |a-b| > tol*max|b|, w[24+v] = the smallest interior index
// ((b*ni + i)*nj + j)*nk + k holding max|a-b|.
template <int PASS>
__global__ void __launch_bounds__(256) k_state_diff(Dims d, const double *__restrict__ a, const double *__restrict__ b,
                                                    double tol, unsigned long long *__restrict__ w) {
    const int blk = blockIdx.x >> 3, v = blockIdx.x & 7;
    const long long n3 = (long long)d.ni * d.nj * d.nk;
    const long long base = ((long long)blk * 8 + v) * d.P;
    double m0 = 0.0, m1 = 0.0;
    unsigned long long cnt = 0, first = ~0ull;
    const double dmax = PASS == 1 ? __longlong_as_double((long long)w[v]) : 0.0;
    const double lim = PASS == 1 ? tol * __longlong_as_double((long long)w[8 + v]) : 0.0;
    for (long long q = threadIdx.x; q < n3; q += blockDim.x) {
        const int k = (int)(q % d.nk), j = (int)((q / d.nk) % d.nj), i = (int)(q / ((long long)d.nk * d.nj));
        const long long o = base + cell_off(d, i + d.ng, j + d.ng, k + d.ng);
        const double x = fabs(a[o] - b[o]), y = fabs(b[o]);
        if (PASS == 0) {
            m0 = x > m0 ? x : m0;
            m1 = y > m1 ? y : m1;
        } else {
            cnt += x > lim ? 1 : 0;
            if (x == dmax) {
                const unsigned long long id = (unsigned long long)((((long long)blk * d.ni + i) * d.nj + j) * d.nk + k);
                first = id < first ? id : first;
            }
        }
    }
    if (PASS == 0) {
        atomicMax(&w[v], (unsigned long long)__double_as_longlong(m0));
        atomicMax(&w[8 + v], (unsigned long long)__double_as_longlong(m1));
    } else {
        if (cnt) atomicAdd(&w[16 + v], cnt);
        if (first != ~0ull) atomicMin(&w[24 + v], first);
    }
}

// ModCheck_primitive (3_6/ModCheck.f90:12-71) on a padded state of any
// precision: w[0] += NaN count, w[1] = min over NaN cells of the reference's
// scan position ((b*NK + K)*NJ + J)*NI*8 + I*8 + v (blocks in order, then
// phi, theta, r, variable innermost), one workgroup per (block, variable).
template <typename TS>
__global__ void __launch_bounds__(256) k_nan_scan(Dims d, const TS *__restrict__ st, unsigned long long *__restrict__ w) {
    const int blk = blockIdx.x >> 3, v = blockIdx.x & 7;
    const TS *p = st + ((long long)blk * 8 + v) * d.P;
    unsigned long long cnt = 0, first = ~0ull;
    for (long long q = threadIdx.x; q < d.P; q += blockDim.x) {
        const TS x = p[q];
        if (x != x) {
            int I, J, K;
            cell_ijk(d, q, I, J, K);
            // variable innermost, with room for psi (variable 8) after the eight
            const unsigned long long key =
                ((((unsigned long long)blk * d.NK + K) * d.NJ + J) * d.NI + I) * 9ull + (unsigned long long)v;
            cnt++;
            first = key < first ? key : first;
        }
    }
    if (cnt) {
        atomicAdd(&w[0], cnt);
        atomicMin(&w[1], first);
    }
}

// psi of GLM divergence cleaning ([block][P]), as the ninth variable of the
// same scan order
__global__ void __launch_bounds__(256) k_nan_scan_psi(Dims d, const double *__restrict__ psi,
                                                      unsigned long long *__restrict__ w) {
    const int blk = blockIdx.x;
    const double *p = psi + (long long)blk * d.P;
    unsigned long long cnt = 0, first = ~0ull;
    for (long long q = threadIdx.x; q < d.P; q += blockDim.x) {
        const double x = p[q];
        if (x != x) {
            int I, J, K;
            cell_ijk(d, q, I, J, K);
            const unsigned long long key = ((((unsigned long long)blk * d.NK + K) * d.NJ + J) * d.NI + I) * 9ull + 8ull;
            cnt++;
            first = key < first ? key : first;
        }
    }
    if (cnt) {
        atomicAdd(&w[0], cnt);
        atomicMin(&w[1], first);
    }
}

// ---------------------------------------------------------------- launchers

// workgroups of a march over every block with tile edge TL
static inline unsigned tiles(const Dims &d, int TL) {
    return (unsigned)((long long)d.nblocks * ((d.nj + TL - 1) / TL) * ((d.nk + TL - 1) / TL));
}

static void check_tile(int tile) {
    if (tile != 8 && tile != 16) throw std::runtime_error("tile edge must be 8 or 16");
}

// Blocks whose faces fit an 8-edge tile run the 8-edge march also where 16 is
// asked for (one tile per block either way).
static inline int march_edge(const Dims &d, int tile, int wgs) {
    return tile == 16 && wgs == 0 && d.nj <= 8 && d.nk <= 8 ? 8 : tile;
}

// Radial segments per tile.  A march is a serial chain of planes, so a layout
// with few tiles leaves compute units idle or with an uneven last round; cut
// in segments the tiles fill the chip, at the price of the extra planes each
// segment loads.  The rule minimises the time of the busiest of the 256
// compute units: it runs n workgroups (4 of the 64-lane ones count as one), a
// pair of resident workgroups takes 2 x kPair of one alone, and a segment of
// len planes costs len + kFill (its first window and face).  Both constants
// are fits to the stage and diffusion at 1 .. 8 segments over twelve layouts
// of 40 to 12288 blocks (us per launch, one against the chosen number of
// segments; FP64 stage / FP64 diffusion / FP32 stage / FP32 diffusion):
//    40 blocks of  8x6x12    33.0->13.8   82.0->26.7   25.4->12.7   71.8->26.2
//    60 blocks of 16x16x16   68.6->20.2  154.3->39.2   46.7->17.1  141.1->34.0
//   192 blocks of 16x16x16   79.9->56.9  161.4->103.8  49.2->38.8  137.9->91.6
//   528 blocks of 16x16x16  196.1->155.2 358.9->274.2 107.8->98.7  283.2->216.6
//   128 blocks of 64x16x48  521.5->423.8 929.7->705.4 301.0->259.7 608.8->512.0
// From about 768 16^3 blocks on one segment is best (1536 blocks: 399 against
// 406 us for two, FP32 diffusion 490 against 529), and the rule keeps it
// unless more segments are predicted to save 3%.  A segment has at least two
// planes: the FP32 diffusion's radial boundary faces read the neighbouring
// plane of their own segment.
int march_segments(const Dims &d, int tile, int wgs) {
    if (wgs != 0) return 1;
    constexpr double kPair = 0.75, kFill = 1.5;
    const int TL = march_edge(d, tile, wgs);
    const long long cus = TL == 16 ? 256 : 4 * 256, nt = tiles(d, TL);
    int best = 1;
    double cost = 0.0;
    for (int ns = 1; ns <= 8 && (ns == 1 || 2 * ns <= d.ni); ns *= 2) {
        const long long n = (nt * ns + cus - 1) / cus;
        const double rounds = n > 6 ? kPair * (double)(nt * ns) / (double)cus
                                    : (n & 1) ? (double)(n - 1) * kPair + 1.0 : (double)n * kPair;
        const double c = ((d.ni + ns - 1) / ns + kFill) * rounds;
        if (ns == 1 || c < 0.97 * cost) {
            best = ns;
            cost = c;
        }
    }
    return best;
}

static void check_stage_ni(const Dims &d) {
    if (d.NI > kMaxNI) throw std::runtime_error("stage march: more than 128 radial cells per block");
}

// grid of a march: one workgroup per tile (wgs = 0) or wgs workgroups that
// loop over the tiles (a persistent launch), never more than the tiles
static inline dim3 march_grid(const Dims &d, int TL, int wgs, int nseg) {
    if (wgs < 0) throw std::runtime_error("workgroup count < 0");
    const unsigned n = tiles(d, TL) * (unsigned)nseg;
    return dim3(wgs == 0 ? n : std::min<unsigned>(n, (unsigned)wgs));
}

template <typename K>
static int resident(K kernel, int threads) {
    int dev = 0, per_cu = 0;
    hipDeviceProp_t prop;
    if (hipGetDevice(&dev) != hipSuccess || hipGetDeviceProperties(&prop, dev) != hipSuccess ||
        hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, kernel, threads, 0) != hipSuccess)
        throw std::runtime_error("occupancy query failed");
    return std::max(1, per_cu) * prop.multiProcessorCount;
}

// workgroups of one march resident on the device at once (the persistent grid):
// kernel 0 the stage, 1 the diffusion; precision 0 FP64, 1 FP32.  The FP32
// path launches the stage in two builds (stages 1-3 and the final stage with
// its FP64 output and FP32 copy) on one grid size: the smaller of their counts.
int march_resident_wgs(int kernel, int precision, int tile) {
    check_tile(tile);
    if (kernel == 0 && precision == 0)
        return tile == 16 ? resident(k_stage<double, double, double, double, 0, false, 16, true>, 256)
                          : resident(k_stage<double, double, double, double, 0, false, 8, true>, 64);
    if (kernel == 0)
        return tile == 16 ? std::min(resident(k_stage<float, float, float, float, 0, false, 16, true>, 256),
                                     resident(k_stage<float, float, double, double, 0, true, 16, true>, 256))
                          : std::min(resident(k_stage<float, float, float, float, 0, false, 8, true>, 64),
                                     resident(k_stage<float, float, double, double, 0, true, 8, true>, 64));
    if (precision == 0)
        return tile == 16 ? resident(k_diffusion<double, double, 0, 16, true>, 256)
                          : resident(k_diffusion<double, double, 0, 8, true>, 64);
    return tile == 16 ? resident(k_diffusion<float, float, 0, 16, true>, 256)
                      : resident(k_diffusion<float, float, 0, 8, true>, 64);
}

template <int TL, typename T, typename TIN, typename TOUT, typename TB>
static void stage_tl(const Dims &d, const DevTables &t, const TIN *in, const TB *U, TOUT *out, float *shadow,
                     const double *dtp, double div, hipStream_t s, const int32_t *pull, int wgs, const double *glm) {
    const int nseg = march_segments(d, TL, wgs);
    if (sizeof(T) == 8) div *= kDivUp;   // as cell_rhs takes its divisors
    const dim3 g = march_grid(d, TL, wgs, nseg), b(TL * TL);
    if constexpr (sizeof(T) == 8) {
        if (glm) {
            if (shadow) throw std::runtime_error("GLM stage: no FP32 copy");
            if (wgs)
                hipLaunchKernelGGL((k_stage<T, TIN, TOUT, TB, 0, false, TL, true, true>), g, b, 0, s, d, t, in, U, out,
                                   (float *)nullptr, dtp, div, pull, glm, nseg);
            else if (TL == 16)
                hipLaunchKernelGGL((k_stage_w2<T, TIN, TOUT, TB, 0, false, TL, false, true>), g, b, 0, s, d, t, in, U,
                                   out, (float *)nullptr, dtp, div, pull, glm, nseg);
            else
                hipLaunchKernelGGL((k_stage<T, TIN, TOUT, TB, 0, false, TL, false, true>), g, b, 0, s, d, t, in, U, out,
                                   (float *)nullptr, dtp, div, pull, glm, nseg);
            return;
        }
        if (!shadow && !wgs && TL == 16) {
            hipLaunchKernelGGL((k_stage_w2<T, TIN, TOUT, TB, 0, false, TL, false>), g, b, 0, s, d, t, in, U, out,
                               (float *)nullptr, dtp, div, pull, glm, nseg);
            return;
        }
    }
    if (shadow && wgs)
        hipLaunchKernelGGL((k_stage<T, TIN, TOUT, TB, 0, true, TL, true>), g, b, 0, s, d, t, in, U, out, shadow, dtp, div,
                           pull, glm, nseg);
    else if (shadow)
        hipLaunchKernelGGL((k_stage<T, TIN, TOUT, TB, 0, true, TL, false>), g, b, 0, s, d, t, in, U, out, shadow, dtp, div,
                           pull, glm, nseg);
    else if (wgs)
        hipLaunchKernelGGL((k_stage<T, TIN, TOUT, TB, 0, false, TL, true>), g, b, 0, s, d, t, in, U, out,
                           (float *)nullptr, dtp, div, pull, glm, nseg);
    else
        hipLaunchKernelGGL((k_stage<T, TIN, TOUT, TB, 0, false, TL, false>), g, b, 0, s, d, t, in, U, out,
                           (float *)nullptr, dtp, div, pull, glm, nseg);
}

template <typename T, typename TIN, typename TOUT, typename TB>
void launch_stage(const Dims &d, const DevTables &t, const TIN *in, const TB *U, TOUT *out, float *shadow,
                  const double *dtp, double div, hipStream_t s, const int32_t *pull, int tile, int wgs,
                  const double *glm) {
    check_tile(tile);
    check_stage_ni(d);
    if (glm && sizeof(T) != 8) throw std::runtime_error("GLM divergence cleaning runs on the FP64 path only");
    if (march_edge(d, tile, wgs) == 16) stage_tl<16, T>(d, t, in, U, out, shadow, dtp, div, s, pull, wgs, glm);
    else stage_tl<8, T>(d, t, in, U, out, shadow, dtp, div, s, pull, wgs, glm);
}

template <int TL, bool PERSIST, typename T, typename TIN>
static void rhs_tl(const Dims &d, const DevTables &t, const TIN *in, double *R, hipStream_t s, int wgs) {
    hipLaunchKernelGGL((k_stage<T, TIN, double, double, 1, false, TL, PERSIST>), march_grid(d, TL, wgs, 1),
                       dim3(TL * TL), 0, s, d, t, in, (const double *)nullptr, R, (float *)nullptr,
                       (const double *)nullptr, 1.0, (const int32_t *)nullptr, (const double *)nullptr, 1);
}

template <typename T, typename TIN>
void launch_rhs_only(const Dims &d, const DevTables &t, const TIN *in, double *R, hipStream_t s, int tile, int wgs) {
    check_tile(tile);
    check_stage_ni(d);
    if (tile == 16) {
        if (wgs) rhs_tl<16, true, T>(d, t, in, R, s, wgs);
        else rhs_tl<16, false, T>(d, t, in, R, s, wgs);
    } else {
        if (wgs) rhs_tl<8, true, T>(d, t, in, R, s, wgs);
        else rhs_tl<8, false, T>(d, t, in, R, s, wgs);
    }
}

template <int TL, bool PERSIST, int MODE, typename T, typename TIN>
static void diffusion_tl(const Dims &d, const DevTables &t, const TIN *in, const double *U, double *out,
                         float *shadow, double *partial, const double *dtp, hipStream_t s, const int32_t *pull,
                         int wgs, const double *Uold) {
    const int nseg = MODE == 0 ? march_segments(d, TL, wgs) : 1;
    hipLaunchKernelGGL((k_diffusion<T, TIN, MODE, TL, PERSIST>), march_grid(d, TL, wgs, nseg), dim3(TL * TL), 0, s, d,
                       t, in, U, out, shadow, partial, dtp, pull, Uold, nseg);
}

template <int MODE, typename T, typename TIN>
static void diffusion_any(const Dims &d, const DevTables &t, const TIN *in, const double *U, double *out,
                          float *shadow, double *partial, const double *dtp, hipStream_t s, const int32_t *pull,
                          int tile, int wgs, const double *Uold) {
    check_tile(tile);
    if (march_edge(d, tile, wgs) == 16) {
        if (wgs) diffusion_tl<16, true, MODE, T>(d, t, in, U, out, shadow, partial, dtp, s, pull, wgs, Uold);
        else diffusion_tl<16, false, MODE, T>(d, t, in, U, out, shadow, partial, dtp, s, pull, wgs, Uold);
    } else {
        if (wgs) diffusion_tl<8, true, MODE, T>(d, t, in, U, out, shadow, partial, dtp, s, pull, wgs, Uold);
        else diffusion_tl<8, false, MODE, T>(d, t, in, U, out, shadow, partial, dtp, s, pull, wgs, Uold);
    }
}

template <typename T, typename TIN>
void launch_diffusion(const Dims &d, const DevTables &t, const TIN *in, const double *U, double *out, float *shadow,
                      double *partial, const double *dtp, hipStream_t s, const int32_t *pull, int tile, int wgs,
                      const double *Uold) {
    check_stage_ni(d);
    if (sizeof(T) == 4 && (U != out || !Uold || !shadow || d.ni < 2))
        throw std::runtime_error("FP32 diffusion: updates the state in place, needs U^n, the FP32 copy and ni >= 2");
    if (sizeof(T) == 8 && ((const void *)in != (const void *)U || out == U || shadow))
        throw std::runtime_error("FP64 diffusion: updates its input into another buffer");
    diffusion_any<0, T>(d, t, in, U, out, shadow, partial, dtp, s, pull, tile, wgs, Uold);
}

template <typename T>
void launch_diffusion_only(const Dims &d, const DevTables &t, const double *U, double *R, hipStream_t s, int tile,
                           int wgs) {
    diffusion_any<1, T>(d, t, U, U, R, (float *)nullptr, (double *)nullptr, (const double *)nullptr, s,
                        (const int32_t *)nullptr, tile, wgs, (const double *)nullptr);
}

static unsigned tail_wgs(const Dims &d, const FillTail &t) {
    if (t.bnd.n == 0) return 0;
    const long long n = (long long)t.bnd.n * d.ng * (t.src ? (long long)d.NJ * d.NK : (long long)d.nj * d.nk);
    return (unsigned)((n + 255) / 256);
}

static void exchange32(const Dims &d, const DevGhosts &g, const DevFill &copy, bool faces, float *state,
                       hipStream_t s, const FillTail &tail) {
    auto n = [&](const DevFill &f) { return faces ? f.n_face : f.n; };
    const int nw = n(g.weighted), nl = n(g.lerp), nc = n(copy);
    const unsigned wgs = (unsigned)((nw + 255) / 256 + (nl + 255) / 256 + (nc + 255) / 256) + tail_wgs(d, tail);
    if (wgs == 0) return;
    const bool thin = d.ni == 1 || d.nj == 1 || d.nk == 1;
    if (thin) hipLaunchKernelGGL(k_exchange_f32<true>, dim3(wgs), dim3(256), 0, s, d, g, copy, nw, nl, nc, state, tail);
    else hipLaunchKernelGGL(k_exchange_f32<false>, dim3(wgs), dim3(256), 0, s, d, g, copy, nw, nl, nc, state, tail);
}

void launch_exchange(const Dims &d, const DevGhosts &g, float *state, hipStream_t s, const FillTail &tail) {
    exchange32(d, g, g.copy, false, state, s, tail);
}

void launch_exchange_rest(const Dims &d, const DevGhosts &g, float *state, bool faces, hipStream_t s,
                          const FillTail &tail) {
    if (!g.pull) throw std::runtime_error("no pull table: use the full exchange");
    exchange32(d, g, g.copy_rest, faces, state, s, tail);
}

void launch_exchange64(const Dims &d, const DevGhosts64 &g, double *state, double *psi, bool faces, hipStream_t s,
                       const FillTail &tail) {
    const int n = faces ? g.n_face : g.n;
    const unsigned wgs = (unsigned)((n + 255) / 256) + tail_wgs(d, tail);
    if (wgs == 0) return;
    const dim3 grid(wgs), wg(256);
    const int32_t *all = faces ? nullptr : g.all;
    if (psi) hipLaunchKernelGGL(k_exchange_f64<true>, grid, wg, 0, s, d, g, all, n, state, psi, tail);
    else hipLaunchKernelGGL(k_exchange_f64<false>, grid, wg, 0, s, d, g, all, n, state, psi, tail);
}

template <typename TS>
void launch_boundary(const Dims &d, const DevBoundary &b, TS *state, hipStream_t s, const int32_t *pull, const DtFinal &dt) {
    const long long n = (long long)b.n * d.ng * d.NJ * d.NK;
    const unsigned wgs = (unsigned)((n + 255) / 256) + (dt.partial ? 1u : 0u);
    if (wgs) hipLaunchKernelGGL((k_boundary<TS>), dim3(wgs), dim3(256), 0, s, d, b, state, pull, dt);
}

DtFinal dt_final_args(const Dims &d, const double *partial, double *dtp, double cfl, int tile, int nseg) {
    check_tile(tile);
    return DtFinal{partial, (int)(tiles(d, tile) * (unsigned)nseg), cfl, dtp};
}

// the partial minima are laid out as the diffusion with the same tile edge
// leaves them, one per workgroup
void launch_dt_partial(const Dims &d, const DevTables &t, const double *U, double *partial, hipStream_t s, int tile,
                       int nseg) {
    check_tile(tile);
    const dim3 g(tiles(d, tile) * (unsigned)nseg);
    if (march_edge(d, tile, 0) == 16) hipLaunchKernelGGL(k_dt_tile<16>, g, dim3(256), 0, s, d, t, U, partial, nseg);
    else hipLaunchKernelGGL(k_dt_tile<8>, g, dim3(64), 0, s, d, t, U, partial, nseg);
}

void launch_dt_final(const Dims &d, const double *partial, double *dtp, double cfl, hipStream_t s, int tile,
                     int nseg) {
    hipLaunchKernelGGL(k_dt_final, dim3(1), dim3(256), 0, s, dt_final_args(d, partial, dtp, cfl, tile, nseg));
}

void launch_set_scalar(double *p, double v, hipStream_t s) {
    hipLaunchKernelGGL(k_set_scalar, dim3(1), dim3(64), 0, s, p, v);
}

void launch_state_diff(const Dims &d, const double *a, const double *b, double tol, unsigned long long *w, int pass,
                       hipStream_t s) {
    const dim3 grid((unsigned)d.nblocks * 8);
    if (pass == 0) hipLaunchKernelGGL(k_state_diff<0>, grid, dim3(256), 0, s, d, a, b, tol, w);
    else hipLaunchKernelGGL(k_state_diff<1>, grid, dim3(256), 0, s, d, a, b, tol, w);
}

template <typename TS>
void launch_nan_scan(const Dims &d, const TS *st, unsigned long long *w, hipStream_t s) {
    hipLaunchKernelGGL(k_nan_scan<TS>, dim3((unsigned)d.nblocks * 8), dim3(256), 0, s, d, st, w);
}
void launch_nan_scan_psi(const Dims &d, const double *psi, unsigned long long *w, hipStream_t s) {
    hipLaunchKernelGGL(k_nan_scan_psi, dim3((unsigned)d.nblocks), dim3(256), 0, s, d, psi, w);
}
template void launch_nan_scan<double>(const Dims &, const double *, unsigned long long *, hipStream_t);
template void launch_nan_scan<float>(const Dims &, const float *, unsigned long long *, hipStream_t);

void launch_block_to_host(const Dims &d, const double *src, int nvar, double *dst, hipStream_t s) {
    const unsigned n = (unsigned)(d.NI * d.NJ);
    hipLaunchKernelGGL(k_block_to_host, dim3((n + 63) / 64, (unsigned)(d.NK + 3) / 4, (unsigned)nvar), dim3(256), 0, s, d,
                       src, dst);
}

void launch_to_f32(const double *src, float *dst, long long n, hipStream_t s) {
    hipLaunchKernelGGL(k_to_f32, dim3(4096), dim3(256), 0, s, src, dst, n);
}

// ---------------------------------------------------------------- initial state

// Seeded synthetic initial state on the interior of every block (the
// configured runs' initial condition; no reference counterpart beyond
// 3_6/ModInitiation.f90:14-188, which sets other fields): rho1 = v = 0;
// s1 = s_amp * c_p * U(-1,1) with U from a splitmix64 hash of (seed, block,
// cell); B = curl A of a smooth random vector potential, the sum over modes
// of (k x a) cos(k.x + phase) evaluated in global Cartesian coordinates (Yang
// positions and components through the involution (x, y, z) -> (-x, z, y) of
// ModYinYang_CoordConv, 3_6/ModYinYang.f90:8-17), before its scaling.
// rows per block (3 x NI): c_p, sqrt(rho0), c_s.  wgmax[workgroup]: the
// largest |B| / (sqrt(rho0) c_s) of its cells, for the scale.
__device__ __forceinline__ unsigned long long splitmix64(unsigned long long x) {
    x += 0x9E3779B97F4A7C15ull;
    x = (x ^ (x >> 30)) * 0xBF58476D1CE4E5B9ull;
    x = (x ^ (x >> 27)) * 0x94D049BB133111EBull;
    return x ^ (x >> 31);
}

__global__ void __launch_bounds__(256) k_synthetic(Dims d, const double *__restrict__ rng,
                                                   const int32_t *__restrict__ yin, const double *__restrict__ rows,
                                                   const SynthMode *__restrict__ modes, int nm, unsigned long long seed,
                                                   double s_amp, double *__restrict__ U, double *__restrict__ wgmax) {
    __shared__ double red[4];
    const long long n3 = (long long)d.ni * d.nj * d.nk;
    const long long t = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    double ratio = 0.0;
    if (t < (long long)d.nblocks * n3) {
        const int b = (int)(t / n3);
        const long long c = t - (long long)b * n3;
        // Fortran indices, i fastest
        const int i = (int)(c % d.ni) + 1, j = (int)((c / d.ni) % d.nj) + 1, k = (int)(c / ((long long)d.ni * d.nj)) + 1;
        const double *rg = rng + 6 * (long long)b;
        auto centre = [](double lo, double hi, int n, int f) {
            return (lo * (double)((float)(n - f) + 0.5f) + hi * (double)((float)f - 0.5f)) / (double)n;
        };
        const double r = centre(rg[0], rg[1], d.ni, i), th = centre(rg[2], rg[3], d.nj, j);
        const double ph = centre(rg[4], rg[5], d.nk, k);
        const double sth = sin(th), cth = cos(th), sph = sin(ph), cph = cos(ph);
        const bool y = yin[b] != 0;
        const double p0 = r * sth * cph, p1 = r * sth * sph, p2 = r * cth;
        const double x0 = y ? p0 : -p0, x1 = y ? p1 : p2, x2 = y ? p2 : p1;
        double g0 = 0.0, g1 = 0.0, g2 = 0.0;
        for (int m = 0; m < nm; m++) {
            const SynthMode &M = modes[m];
            const double cc = cos(M.k[0] * x0 + M.k[1] * x1 + M.k[2] * x2 + M.ph);
            g0 += M.a[0] * cc; g1 += M.a[1] * cc; g2 += M.a[2] * cc;
        }
        const double l0 = y ? g0 : -g0, l1 = y ? g1 : g2, l2 = y ? g2 : g1;
        const double Br = l0 * (sth * cph) + l1 * (sth * sph) + l2 * cth;
        const double Bt = l0 * (cth * cph) + l1 * (cth * sph) + l2 * (-sth);
        const double Bp = l0 * (-sph) + l1 * cph + l2 * 0.0;
        const int I = i + d.ng - 1;
        const double *rw = rows + 3 * (long long)b * d.NI;
        const double cp = rw[I], srho = rw[d.NI + I], cs = rw[2 * d.NI + I];
        ratio = sqrt(Br * Br + Bt * Bt + Bp * Bp) / srho / cs;
        const unsigned long long id = ((unsigned long long)b << 32) ^ (unsigned long long)((i * 131 + j) * 1031 + k);
        const double u = (double)(splitmix64(seed ^ (id * 0x2545F4914F6CDD1Dull)) >> 11) * (1.0 / 9007199254740992.0);
        const long long q = (long long)b * 8 * d.P + cell_off(d, I, j + d.ng - 1, k + d.ng - 1);
        U[q + 4 * d.P] = Br;
        U[q + 5 * d.P] = Bt;
        U[q + 6 * d.P] = Bp;
        U[q + 7 * d.P] = s_amp * cp * (2.0 * u - 1.0);
    }
    for (int off = 32; off > 0; off >>= 1) {
        const double o = __shfl_down(ratio, off, 64);
        ratio = o > ratio ? o : ratio;
    }
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = ratio;
    __syncthreads();
    if (threadIdx.x == 0) {
        double mx = red[0];
        for (int w = 1; w < (int)(blockDim.x >> 6); w++) mx = red[w] > mx ? red[w] : mx;
        wgmax[blockIdx.x] = mx;
    }
}

// scale = b_ratio / max over the workgroup maxima (0 where the field is 0),
// then B *= scale on every interior cell
__global__ void __launch_bounds__(256) k_synthetic_scale(Dims d, const double *__restrict__ wgmax, int nwg,
                                                         double b_ratio, double *__restrict__ U) {
    __shared__ double sc;
    if (threadIdx.x == 0) {
        double mx = 0.0;
        for (int w = 0; w < nwg; w++) mx = wgmax[w] > mx ? wgmax[w] : mx;
        sc = mx > 0.0 ? b_ratio / mx : 0.0;
    }
    __syncthreads();
    const double scale = sc;
    const long long n3 = (long long)d.ni * d.nj * d.nk;
    for (long long t = (long long)blockIdx.x * blockDim.x + threadIdx.x; t < (long long)d.nblocks * n3;
         t += (long long)gridDim.x * blockDim.x) {
        const int b = (int)(t / n3);
        const long long c = t - (long long)b * n3;
        const int i = (int)(c % d.ni), j = (int)((c / d.ni) % d.nj), k = (int)(c / ((long long)d.ni * d.nj));
        const long long q = (long long)b * 8 * d.P + cell_off(d, i + d.ng, j + d.ng, k + d.ng);
        for (int v = 4; v < 7; v++) U[q + v * d.P] *= scale;
    }
}

void launch_synthetic(const Dims &d, const double *rng, const int32_t *yin, const double *rows, const SynthMode *modes,
                      int nm, unsigned long long seed, double s_amp, double b_ratio, double *U, double *wgmax,
                      hipStream_t s) {
    const long long n = (long long)d.nblocks * d.ni * d.nj * d.nk;
    const int nwg = (int)((n + 255) / 256);
    hipLaunchKernelGGL(k_synthetic, dim3((unsigned)nwg), dim3(256), 0, s, d, rng, yin, rows, modes, nm, seed, s_amp, U,
                       wgmax);
    hipLaunchKernelGGL(k_synthetic_scale, dim3(2048), dim3(256), 0, s, d, wgmax, nwg, b_ratio, U);
}

// ---------------------------------------------------------------- output

// Corner values of ModSave_AllCells (3_6/ModSavePlot.f90:585-640) for blocks
// [b0, b0 + nb): one thread per corner (i, j, k), i fastest, writing the
// line's 12 numbers to out[(b - b0)][corner][12]: the corner's Cartesian
// position in solar radii, then the 9 variables of the reference's state
// averaged over the 8 surrounding cells (ghosts included, summed in the
// reference's order), with v and B turned to Cartesian components; psi is 0
// (the state holds no psi: no term writes it with DivB_option = 0).
// geo per block: face radii xi_F (ni+1), then sin and cos of the theta faces
// (nj+1 each) and of the phi faces (nk+1 each), from the host's libm.
__global__ void __launch_bounds__(256) k_allcells(Dims d, const double *__restrict__ U,
                                                  const double *__restrict__ geo, const int32_t *__restrict__ yin,
                                                  int b0, int nb, double rsun, double *__restrict__ out) {
    const int ci = d.ni + 1, cj = d.nj + 1, ck = d.nk + 1;
    const long long nc = (long long)ci * cj * ck;
    const long long t = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= (long long)nb * nc) return;
    const int lb = (int)(t / nc), b = b0 + lb;
    const long long c = t - (long long)lb * nc;
    const int i = (int)(c % ci) + 1, j = (int)((c / ci) % cj) + 1, k = (int)(c / ((long long)ci * cj)) + 1;
    const long long G = ci + 2 * cj + 2 * ck;
    const double *g = geo + (long long)b * G;
    const double r = g[i - 1];
    const double sth = g[ci + j - 1], cth = g[ci + cj + j - 1];
    const double sph = g[ci + 2 * cj + k - 1], cph = g[ci + 2 * cj + ck + k - 1];
    // padded index of Fortran index f: f + ng - 1
    const int I = i + d.ng - 1, J = j + d.ng - 1, K = k + d.ng - 1;
    auto at = [&](int v, int II, int JJ, int KK) -> double {
        return U[(long long)b * 8 * d.P + (long long)v * d.P + cell_off(d, II, JJ, KK)];
    };
    double o[12];
    const bool y = yin[b] != 0;
    if (y) {
        o[0] = (r * sth) * cph; o[1] = (r * sth) * sph; o[2] = r * cth;
    } else {
        o[0] = -((r * sth) * cph); o[1] = r * cth; o[2] = (r * sth) * sph;
    }
    o[0] = o[0] / rsun; o[1] = o[1] / rsun; o[2] = o[2] / rsun;
    #pragma unroll
    for (int v = 0; v < 8; v++) {
        double s = at(v, I - 1, J - 1, K - 1) + at(v, I, J - 1, K - 1);
        s = s + at(v, I - 1, J, K - 1);
        s = s + at(v, I, J, K - 1);
        s = s + at(v, I - 1, J - 1, K);
        s = s + at(v, I, J - 1, K);
        s = s + at(v, I - 1, J, K);
        s = s + at(v, I, J, K);
        o[3 + v] = 0.125 * s;
    }
    o[11] = 0.0;
    // (vr, vt, vp) and (br, bt, bp) to Cartesian (:614-637); Yang: (-x, z, y)
    #pragma unroll
    for (int q = 0; q < 2; q++) {
        double *w = o + 4 + 3 * q;
        const double x0 = ((w[0] * sth) * cph + (w[1] * cth) * cph) - w[2] * sph;
        const double y0 = ((w[0] * sth) * sph + (w[1] * cth) * sph) + w[2] * cph;
        const double z0 = w[0] * cth - w[1] * sth;
        if (y) { w[0] = x0; w[1] = y0; w[2] = z0; }
        else { w[0] = -x0; w[1] = z0; w[2] = y0; }
    }
    double *dst = out + t * 12;
    #pragma unroll
    for (int q = 0; q < 12; q++) dst[q] = o[q];
}

void launch_allcells(const Dims &d, const double *U, const double *geo, const int32_t *yin, int b0, int nb,
                     double rsun, double *out, hipStream_t s) {
    const long long n = (long long)nb * (d.ni + 1) * (d.nj + 1) * (d.nk + 1);
    if (n <= 0) return;
    hipLaunchKernelGGL(k_allcells, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, s, d, U, geo, yin, b0, nb, rsun,
                       out);
}

// ---------------------------------------------------------------- GLM divergence cleaning


// interior cell c of all blocks (phi fastest): block, interior and padded indices
struct GlmCell {
    int b, i, j, k, I, J, K;
};
__device__ __forceinline__ GlmCell glm_cell(const Dims &d, long long c) {
    const long long nn = (long long)d.ni * d.nj * d.nk;
    GlmCell g;
    g.b = (int)(c / nn);
    long long r = c - (long long)g.b * nn;
    g.k = (int)(r % d.nk);
    r /= d.nk;
    g.j = (int)(r % d.nj);
    g.i = (int)(r / d.nj);
    g.I = g.i + d.ng; g.J = g.j + d.ng; g.K = g.k + d.ng;
    return g;
}

// ModDivB_GLM (3_6/ModDivB.f90:13-38) at one RK stage, one lane per interior
// cell, on the stage input `in` (radial boundaries applied) and psi_in:
//   div B    ModSpherical_div (3_6/ModSpherical.f90:104-159): A_r r^2 along r
//            times 1/r^2, plus (A_t sin(t) along theta + A_p along phi) times
//            1/sin(t), then 1/r;
//   grad psi ModSpherical_Grad_f (:201-239);
//   R(psi) = -c_h^2 div B - (c_h / h_LLL) psi, c_h = v_wave of the step's
//            state (ModWaveSpeed_Dynamo at the step's start), from Ch.
// psi_out = psi_n + dt R(psi) / div (3_6/ModAdvance.f90:88-93), and grad psi
// goes to G ([block][3][interior cells]) for the stage kernel to subtract
// from R(B).  psi_out may be psi_n (the fourth stage): each lane reads psi_n
// at its own cell only.
__global__ void __launch_bounds__(256) k_glm_stage(Dims d, DevTables t, const double *__restrict__ in,
                                                   const double *__restrict__ Ch, const double *__restrict__ psi_in,
                                                   const double *psi_n, double *psi_out, double *__restrict__ G,
                                                   const double *__restrict__ dtp, double div) {
    const long long nn = (long long)d.ni * d.nj * d.nk;
    const long long c = xcd_lane();   // r/theta neighbour planes in one XCD's L2
    if (c >= nn * d.nblocks) return;
    const GlmCell g = glm_cell(d, c);
    const int I = g.I, J = g.J, K = g.K;
    const BlockMeta mt = t.meta[g.b];
    const long long rb = (long long)g.b * d.NI, tb = (long long)g.b * d.NJ;
    const double *S = in + (long long)g.b * 8 * d.P;
    const double *Ps = psi_in + (long long)g.b * d.P;
    // K is interior: the cell and its r and theta neighbours are in the main
    // part (offsets q +- SI, q +- SJ); only the phi neighbours may be ghosts
    const long long q = cell_off(d, I, J, K), SI = d.SI, SJ = d.SJ;
    const long long km2 = cell_off(d, I, J, K - 2), km1 = cell_off(d, I, J, K - 1), kp1 = cell_off(d, I, J, K + 1),
                    kp2 = cell_off(d, I, J, K + 2);
    const double *Br = S + 4 * d.P, *Bt = S + 5 * d.P, *Bp = S + 6 * d.P;
    auto a1 = [&](int di) -> double {
        const double x = t.xi[rb + I + di];
        return Br[q + di * SI] * (x * x);
    };
    auto a2 = [&](int dj) -> double { return Bt[q + dj * SJ] * t.sint[tb + J + dj]; };
    const double rinv = t.rinv[rb + I], sinv = t.sinv[tb + J];
    const double dr = d4(a1(-2), a1(-1), a1(1), a1(2), mt.cr) * t.r2inv[rb + I];
    double d23 = d4(a2(-2), a2(-1), a2(1), a2(2), mt.ct);
    d23 = d23 + d4(Bp[km2], Bp[km1], Bp[kp1], Bp[kp2], mt.cp);
    d23 = d23 * sinv;
    d23 = d23 * rinv;
    const double divb = dr + d23;
    const double g1 = d4(Ps[q - 2 * SI], Ps[q - SI], Ps[q + SI], Ps[q + 2 * SI], mt.cr);
    const double g2 = d4(Ps[q - 2 * SJ], Ps[q - SJ], Ps[q + SJ], Ps[q + 2 * SJ], mt.ct) * rinv;
    double g3 = d4(Ps[km2], Ps[km1], Ps[kp1], Ps[kp2], mt.cp) * rinv;
    g3 = g3 * sinv;
    // c_h and c_h / h_LLL of the step (k_glm_speed)
    const long long gb = (long long)g.b * 3 * nn + ((long long)g.i * d.nj + g.j) * d.nk + g.k;
    const long long cb = (long long)g.b * 2 * nn + ((long long)g.i * d.nj + g.j) * d.nk + g.k;
    const double w = Ch[cb], wh = Ch[cb + nn];
    const double rpsi = -((w * w) * divb) - wh * Ps[q];
    const long long pq = (long long)g.b * d.P + q;
    psi_out[pq] = psi_n[pq] + (*dtp * rpsi) / div;
    G[gb] = g1;
    G[gb + nn] = g2;
    G[gb + 2 * nn] = g3;
}

// c_h = v_wave and c_h / h_LLL of every interior cell of the step's state U
// (ModWaveSpeed_Dynamo, 3_6/ModWaveSpeed.f90:8-27, and h_LLL,
// 3_6/ModBlock.f90:420-422, as k_dt_tile forms them), once per step for the
// four GLM stages: Ch[block][2][interior cells].
__global__ void __launch_bounds__(256) k_glm_speed(Dims d, DevTables t, const double *__restrict__ U,
                                                   double *__restrict__ Ch) {
    const long long nn = (long long)d.ni * d.nj * d.nk;
    const long long c = xcd_lane();   // r/theta neighbour planes in one XCD's L2
    if (c >= nn * d.nblocks) return;
    const GlmCell g = glm_cell(d, c);
    const int I = g.I, J = g.J, K = g.K;
    const BlockMeta mt = t.meta[g.b];
    const long long rb = (long long)g.b * d.NI, tb = (long long)g.b * d.NJ;
    const double *Ub = U + (long long)g.b * 8 * d.P + cell_off(d, I, J, K);
    const double vr = Ub[d.P], vt = Ub[2 * d.P], vp = Ub[3 * d.P];
    const double br = Ub[4 * d.P], bt = Ub[5 * d.P], bp = Ub[6 * d.P];
    double w = t.cs[rb + I] + sqrt(vr * vr + vt * vt + vp * vp);
    w = w + sqrt(br * br + bt * bt + bp * bp) / t.sqrt_rho0[rb + I];
    const double xi = t.xi[rb + I];
    double h = mt.dxi, h2 = xi * mt.dxj, h3 = (xi * t.sint[tb + J]) * mt.dxk;
    h = h < h2 ? h : h2;
    h = h < h3 ? h : h3;
    const long long cb = (long long)g.b * 2 * nn + ((long long)g.i * d.nj + g.j) * d.nk + g.k;
    Ch[cb] = w;
    Ch[cb + nn] = w / h;
}

// The artificial diffusion of psi after the fourth stage
// (3_6/ModDiffusion.f90:9-150, h = 2, the ninth variable; 3_6/ModAdvance.f90:
// 101-108): the faces of k_diffusion's FP64 instantiation, the speeds of the
// state U where the reference reads them (transverse index - ng), and
// psi_new = psi + (0.5 dt) R.
__global__ void __launch_bounds__(256) k_glm_diffusion(Dims d, DevTables t, const double *__restrict__ U,
                                                       const double *__restrict__ psi, double *__restrict__ psi_new,
                                                       const double *__restrict__ dtp) {
    const long long nn = (long long)d.ni * d.nj * d.nk;
    const long long c = xcd_lane();   // r/theta neighbour planes in one XCD's L2
    if (c >= nn * d.nblocks) return;
    const GlmCell g = glm_cell(d, c);
    const int I = g.I, J = g.J, K = g.K;
    const BlockMeta mt = t.meta[g.b];
    const long long rb = (long long)g.b * d.NI, tb = (long long)g.b * d.NJ;
    const double *Sb = U + (long long)g.b * 8 * d.P;
    const double *Pb = psi + (long long)g.b * d.P;
    const double *cs = t.cs + rb;
    // the cell and its r and theta neighbours are in the main part; the phi
    // neighbours and the speed cells at K - 2 may be ghosts
    const long long q = cell_off(d, I, J, K), SI = d.SI, SJ = d.SJ;
    const long long km2 = cell_off(d, I, J, K - 2), km1 = cell_off(d, I, J, K - 1), kp1 = cell_off(d, I, J, K + 1),
                    kp2 = cell_off(d, I, J, K + 2);
    const double *V1 = Sb + d.P, *V2 = Sb + 2 * d.P, *V3 = Sb + 3 * d.P;
    // speed cells (transverse index - ng): (I', J - 2, K - 2), (I - 2, J', K - 2),
    // (I - 2, J - 2, K'); K - 2 lies in the side part below the interior, whose
    // plane and row pitches are NJ 2ng and 2ng
    const long long s1 = cell_off(d, I, J - 2, K - 2), s2 = cell_off(d, I - 2, J, K - 2);
    const bool kmain = K - 2 >= d.ng;
    const long long pI = kmain ? SI : (long long)d.NJ * 2 * d.ng, pJ = kmain ? SJ : 2 * d.ng;
    const double c1m = fabs(V1[s1 - pI]) + cs[I - 1];
    const double c10 = fabs(V1[s1]) + cs[I];
    const double c1p = fabs(V1[s1 + pI]) + cs[I + 1];
    const double p0 = Pb[q];
    // half slopes of the cell and its neighbours along one axis, then its two faces
    auto faces = [&](double m2, double m1, double p1, double p2, double slo, double shi, double &lo, double &hi) {
        const double s0 = half_slope(m1, p0, p1);
        lo = face_flux<double, false>(m1, p0, half_slope(m2, m1, p0), s0) * slo;
        hi = face_flux<double, false>(p0, p1, s0, half_slope(p0, p1, p2)) * shi;
    };
    double f0, f1, fj0, fj1, fk0, fk1;
    faces(Pb[q - 2 * SI], Pb[q - SI], Pb[q + SI], Pb[q + 2 * SI], c10 + c1m, c1p + c10, f0, f1);
    const double csI2 = cs[I - 2];
    const double c2m = fabs(V2[s2 - pJ]) + csI2, c20 = fabs(V2[s2]) + csI2, c2p = fabs(V2[s2 + pJ]) + csI2;
    faces(Pb[q - 2 * SJ], Pb[q - SJ], Pb[q + SJ], Pb[q + 2 * SJ], c20 + c2m, c2p + c20, fj0, fj1);
    const double c3m = fabs(V3[cell_off(d, I - 2, J - 2, K - 1)]) + csI2, c30 = fabs(V3[cell_off(d, I - 2, J - 2, K)]) + csI2,
                 c3p = fabs(V3[cell_off(d, I - 2, J - 2, K + 1)]) + csI2;
    faces(Pb[km2], Pb[km1], Pb[kp1], Pb[kp2], c30 + c3m, c3p + c30, fk0, fk1);
    const double xic = t.xi[rb + I];
    const double L2 = mt.dxj * xic;
    const double L3 = (mt.dxk * xic) * t.sint[tb + J];
    double r = 0.0;
    r = r + (f1 - f0) / mt.dxi;
    r = r + (fj1 - fj0) / L2;
    r = r + (fk1 - fk0) / L3;
    psi_new[(long long)g.b * d.P + q] = p0 + ((0.5 * kFluxScale) * *dtp) * r;
}

static unsigned glm_grid(const Dims &d) {
    const long long n = (long long)d.ni * d.nj * d.nk * d.nblocks;
    return (unsigned)((n + 255) / 256);
}

void launch_glm_speed(const Dims &d, const DevTables &t, const double *U, double *Ch, hipStream_t s) {
    hipLaunchKernelGGL(k_glm_speed, dim3(glm_grid(d)), dim3(256), 0, s, d, t, U, Ch);
}

void launch_glm_stage(const Dims &d, const DevTables &t, const double *in, const double *Ch, const double *psi_in,
                      const double *psi_n, double *psi_out, double *G, const double *dtp, double div, hipStream_t s) {
    if (psi_in == psi_out) throw std::runtime_error("GLM stage: psi_in and psi_out must differ");
    hipLaunchKernelGGL(k_glm_stage, dim3(glm_grid(d)), dim3(256), 0, s, d, t, in, Ch, psi_in, psi_n, psi_out, G, dtp,
                       div);
}

void launch_glm_diffusion(const Dims &d, const DevTables &t, const double *U, const double *psi, double *psi_new,
                          const double *dtp, hipStream_t s) {
    if (psi == psi_new) throw std::runtime_error("GLM diffusion: psi and psi_new must differ");
    hipLaunchKernelGGL(k_glm_diffusion, dim3(glm_grid(d)), dim3(256), 0, s, d, t, U, psi, psi_new, dtp);
}

// explicit instantiations: FP64 path, FP32-deviation path
template void launch_stage<double, double, double, double>(const Dims &, const DevTables &, const double *, const double *, double *, float *, const double *, double, hipStream_t, const int32_t *, int, int, const double *);
template void launch_stage<float, float, float, float>(const Dims &, const DevTables &, const float *, const float *, float *, float *, const double *, double, hipStream_t, const int32_t *, int, int, const double *);
template void launch_stage<float, float, double, double>(const Dims &, const DevTables &, const float *, const double *, double *, float *, const double *, double, hipStream_t, const int32_t *, int, int, const double *);
template void launch_rhs_only<double, double>(const Dims &, const DevTables &, const double *, double *, hipStream_t, int, int);
template void launch_rhs_only<float, double>(const Dims &, const DevTables &, const double *, double *, hipStream_t, int, int);
template void launch_diffusion<double, double>(const Dims &, const DevTables &, const double *, const double *, double *, float *, double *, const double *, hipStream_t, const int32_t *, int, int, const double *);
template void launch_diffusion<float, float>(const Dims &, const DevTables &, const float *, const double *, double *, float *, double *, const double *, hipStream_t, const int32_t *, int, int, const double *);
template void launch_diffusion_only<double>(const Dims &, const DevTables &, const double *, double *, hipStream_t, int, int);
template void launch_diffusion_only<float>(const Dims &, const DevTables &, const double *, double *, hipStream_t, int, int);
template void launch_boundary<double>(const Dims &, const DevBoundary &, double *, hipStream_t, const int32_t *,
                                      const DtFinal &);
template void launch_boundary<float>(const Dims &, const DevBoundary &, float *, hipStream_t, const int32_t *,
                                     const DtFinal &);

}  // namespace falcon
