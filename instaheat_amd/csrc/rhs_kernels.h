// rhs_kernels.h -- the kernels of the right-hand side mk_rhs
// (src/toolbox.c:75-626), each a device body that takes its work-group
// coordinates and its LDS from the caller, and a thin kernel that runs it
// on the hardware's coordinates.  The grouped launches (ihg_group.hip) run
// the same bodies over a table of segments, so a grouped launch computes
// what the per-size launches compute, value for value.
#pragma once

#include <cfloat>
#include <cmath>
#include <type_traits>

#include "fft_kernels.h"
#include "ihg_internal.h"
#include "mem.h"
#include "reduce.h"
#include "rk4_kernels.h"

namespace ihg {

// capply_filter (src/toolbox.c:616-626): in *= filter; out = in / N.
// An output call keeps the filtered spectra of phi (batch 0) and psi (batch
// 2), as mk_ffts_and_filter keeps tmp.phic / tmp.psic (src/toolbox.c:164-
// 171): null pointers keep nothing.
// The mean of phi (its k = 0 mode) goes to *dc instead of the backward
// transform, and the c2r pass adds it (ZShift): so the right-hand side has
// the filtered fluctuations without the rounding of phi, which is of order 1,
// to double precision -- the reference differentiates the kept spectrum, not
// the rounded field.
struct FilterFac {
    const double *__restrict__ filt; // Fx[Nx] | Fy[Ny] | Fz[Mz]
    long plane; // Ny * Mz
    int Nx, Ny, Mz;
    double Nd;
    double2 *keep_phi, *keep_psi;
    double *dc; // mean of the filtered phi per realization, rdc apart
    long rdc;
    __device__ double2 operator()(Blk bk, long line, int n, double2 v) const
    {
        const bool in = line < plane; // padding lines read entry 0
        const long lc = in ? line : 0;
        const long i = (long)n * plane + lc;
        // the mask at (n, j, k) of line j Mz + k: the smallest axis window
        const int j = (int)(lc / Mz), k = (int)(lc - (long)j * Mz);
        const double F = fmin(fmin(filt[n], filt[Nx + j]), filt[Nx + Ny + k]);
        const double2 w = make_double2(v.x * F, v.y * F);
        if (in && bk.y == 0 && keep_phi)
            keep_phi[i] = w;
        if (in && bk.y == 2 && keep_psi)
            keep_psi[i] = w;
        if (bk.y == 0 && line == 0 && n == 0) {
            dc[bk.z * rdc] = w.x / Nd;
            return make_double2(0.0, 0.0);
        }
        return make_double2(w.x / Nd, w.y / Nd);
    }
};

// ---------------------------------------------------------------------------
// The z pass of the right-hand side.  A complex line is a pair of rows A + i
// B of phi (the z derivatives are real operators, so no Hermitian split):
// forward transform, d_z phi and d_zz phi by two backward ones, then with the
// x and y derivatives (k_deriv) assemble_gradient_squared and mk_rho_and_p
// (src/toolbox.c:196-243): block sums of rho and p, p and the part of the
// slope of dphi that needs no mean,
//   A = (1 + 4 psi) lap phi / a^2 - (1 + 2 psi) m^2 phi   (toolbox.c:282-299)
// With GW also the z r2c of the source products: the three gradients are in
// registers at that point, so they are neither written and read again (d_z
// phi is written, for ihg_aux) nor packed with a wasted half line.
//
// GW sources (mk_gw_sources, src/toolbox.c:410-424): only the transverse
// traceless part of d_i phi d_j phi enters the equations, and the projection
// takes delta_ij s to 0 for every s (P is a projector of trace 2 built from
// the full k with k_i k_i = k^2), so one diagonal product, that of axis
// GwAxis::m, is subtracted from the other two: GW_NC = 5 components instead of
// six, (xx - mm, xy, xz, yy - mm, yz) with zz - mm in the place of the one
// that vanishes (two DOPRI853 steps at 256^3 86.0 -> 83.9 ms).  m is the axis
// of the smallest Nyquist wave number, so that a difference is not rounded at
// the size of a much larger product: with m = z on a box resolved more finely
// along z the slopes of h lost a factor of 2.5 (FP32, 4 x 4 x 512 points on a
// cube).  Error of the projected source with FP32 products against six
// components of products of rounded gradients, over white, k^-1 .. k^-3 and
// plane-wave fields, both polarizations (geometric mean per box): 0.87 at 16^3,
// 0.91 at 64^3 and 128^3, 0.94 for spacings of 1 : 2 : 0.5; random fields 0.9 to
// 1.0 on cubes.  The least favourable is a plane wave along m, whose rounding
// enters two components: 1.25 at 64^3 (the other polarization 0.73), 1.8 for
// spacings of 1 : 2 : 0.5.  FP64: below 0.01, from leaving the mean out of the
// transforms.
// Component c of rows A and B is one complex line; its half rows go to W + c M.
//
// A line's T threads are lanes of one wavefront and every wavefront works
// alone (its own LDS lines and its own pair of partial sums), so there is no
// work-group barrier, and the work-group size changes no value: 64 lanes
// spread a small grid over more CUs, 256 share the twiddle table.
//
// Measured at 256^3 with GW: 411 us for the 15 fields' worth of traffic (8 N
// bytes each; 4.9 TB/s), with the FP32 source 401 us for 13, so neither HBM
// alone nor the arithmetic bounds it; the y c2c, z c2r + rho and z r2c passes
// that it replaces moved 31 and took 780 us.  4 values a thread (3 waves a
// SIMD) against 8 (2 waves): 411 against 415 us at 256^3, 278 against 341 us
// for 4 x 128^3, 5.1 against 9.3 us for one 32^3 grid without GW.
// ---------------------------------------------------------------------------

// The axis (0, 1, 2) whose diagonal product is subtracted from the others:
// the one of the smallest Nyquist wave number, z where they are equal.
struct GwAxis {
    int m;
};
inline GwAxis gw_axis(const KGeom &kg)
{
    const double kx = kg.kx1 * kg.Nx, ky = kg.ky1 * kg.Ny, kz = kg.kz1 * kg.Nz;
    GwAxis a{2};
    double least = kz;
    if (kx < least) { a.m = 0; least = kx; }
    if (ky < least) a.m = 1;
    return a;
}

// Line plans of the z pass (512 points: a line in one wavefront)
template <int L> struct ZRhsPlan { using P = typename ZPlanOf<L>::P; };
template <> struct ZRhsPlan<32> { using P = PlanT<4, 4, 4, 2>; };
template <> struct ZRhsPlan<64> { using P = PlanT<4, 4, 4, 4>; };
template <> struct ZRhsPlan<128> { using P = PlanT<4, 4, 4, 4, 2>; };
template <> struct ZRhsPlan<256> { using P = PlanT<4, 4, 4, 4, 4>; };
template <int L> struct ZRhsTile {
    using P = typename ZRhsPlan<L>::P;
    static constexpr int E = P::E, T = L / E, PITCH = Lds<L>::PITCH, LPW = 64 / T;
};

// LDS of the z pass in complex values: the lines, the stage twiddles, and with
// helper wavefronts the three gradients of their 64 E points
template <int L, int WG>
__host__ __device__ constexpr int z_rhs_lines()
{
    return WG / ZRhsTile<L>::T * ZRhsTile<L>::PITCH;
}
template <int L, int WG, bool HELP = false>
__host__ __device__ constexpr int z_rhs_lds()
{
    return z_rhs_lines<L, WG>() + L + (HELP ? 3 * 64 * ZRhsTile<L>::E : 0);
}

// work-groups of the z pass, and its partial sums (one pair a wavefront)
template <int L>
inline unsigned z_rhs_blocks(long nrows, int wg)
{
    const long lines = wg / ZRhsTile<L>::T;
    return (unsigned)((nrows / 2 + lines - 1) / lines);
}

template <class C>
struct ZRhsArgs {
    using R = typename CT<C>::R;
    const double *f;
    double *result;
    const double *phi;     // phi, or after the filter phi - *dc
    const double *dc;      // (NULL: phi itself), rphi and rdc apart
    const double *gx, *gy; // x and y gradients (k_deriv)
    R *g3;                 // GW: all three gradients in the source's type
    C *W;                  // GW: the source components
    long M, N, Ntot, nrows;
    double *rho, *pressure; // output calls (else NULL)
    double *partials;
    double m2;
    double k1, k2;         // 2 pi / (L length), (2 pi / length)^2 / L
    const double2 *tw;
    const C *twc;          // stage twiddles of the source's type
    Ens e;
    long rphi, rdc, rxy, rg, rw; // realization strides of phi, dc, gx / gy, g3, W
    GwAxis ga;
};

// source component K of one point from its gradient
template <int K, class R>
__device__ __forceinline__ R gw_source(R gx, R gy, R gz, int m)
{
    if constexpr (K == 0) {
        const R q = m == 0 ? gz : gx, d = m == 0 ? gx : (m == 1 ? gy : gz);
        return q * q - d * d;
    } else if constexpr (K == 1) {
        return gx * gy;
    } else if constexpr (K == 2) {
        return gx * gz;
    } else if constexpr (K == 3) {
        const R q = m == 1 ? gz : gy, d = m == 0 ? gx : (m == 1 ? gy : gz);
        return q * q - d * d;
    } else {
        return gy * gz;
    }
}

// HELP: all wavefronts of the work-group serve the lines of one; the first does
// the derivatives and the points, then shares the gradients through LDS, and
// the source components are transformed side by side.  On a grid of fewer
// wavefronts than the chip has SIMDs the chain of eight transforms bounds the
// pass (the rule and its figures are at the launch).
template <int L, bool GW, class C, int WG, bool HELP = false>
__device__ __forceinline__ void z_rhs_body(const Blk &bk, double2 *lds,
                                           const ZRhsArgs<C> &a)
{
    static_assert(GW || !HELP, "the sources are what is shared");
    using TL = ZRhsTile<L>;
    using P = typename TL::P;
    using R = typename CT<C>::R;
    constexpr int E = TL::E, T = TL::T, PITCH = TL::PITCH, LPW = TL::LPW;
    constexpr int NW = HELP ? 1 : WG / 64, MZ = L / 2 + 1;
    // The other inputs of a point are loaded ahead of the transforms where
    // too few wavefronts are there to hide their latency (single-wavefront
    // work-groups: 5.1 against 6.0 us at 32^3; the 64- and 128-point lines of
    // the GW pass: 137 against 151 us for 16 x 64^3, 278 against 293 for 4 x
    // 128^3), and at the point elsewhere (256^3 411 against 425 us, 128^3
    // without GW 24 against 28 us): the registers cost a wave a SIMD.
    constexpr bool PRE = HELP || WG == 64 || (GW && (L == 64 || L == 128));
    const int wv = (int)threadIdx.x / 64, lane = (int)threadIdx.x % 64;
    const int w = HELP ? 0 : wv;
    [[maybe_unused]] const int role = __builtin_amdgcn_readfirstlane(wv);
    const int j = lane % T;
    const long wave = (long)bk.x * NW + w, line0 = wave * LPW;
    const long line = line0 + lane / T;
    const bool act = line < a.nrows / 2; // idle lanes work on line 0
    const long ia = (act ? 2 * line : 0) * L; // row A; row B is L further
    double2 *wl = lds + wv * LPW * PITCH, *my = wl + lane / T * PITCH;
    double2 *const ltw = lds + z_rhs_lines<L, WG>();
    // what the sources are made from: FP64 the three gradients; FP32 the
    // components themselves, rounded once from the FP64 gradients (products of
    // gradients rounded to FP32 first: 4 to 7 % more error in the projected
    // source of random fields; this pass 391 us then and 394 now, the
    // right-hand side 1277 and 1278 at 256^3)
    constexpr int NG = sizeof(R) == 4 ? GW_NC : 3;
    [[maybe_unused]] C g[NG][E];
    const double2 *const tw = ltw - L;
    if (!HELP || role == 0) {
    twiddles_to_lds_wave<L>(ltw, a.tw);
    const double *__restrict__ f = a.f + bk.z * a.e.f;
    const double *__restrict__ lx = a.result + bk.z * a.e.f + a.N;
    const double *__restrict__ ly = lx + a.N;
    const double *__restrict__ gxp = a.gx + bk.z * a.rxy;
    const double *__restrict__ gyp = a.gy + bk.z * a.rxy;
    double *__restrict__ outA = a.result + bk.z * a.e.f;
    double *__restrict__ outp = outA + 3 * a.N;

    // the derivatives of phi - phi[0] (see deriv_body)
    const double *__restrict__ phi = a.phi + bk.z * a.rphi;
    const double phi0 = phi[0];
    const double dc = a.dc ? a.dc[bk.z * a.rdc] : 0.0;
    double2 ph[E], lz[E], dz[E];
#pragma unroll
    for (int s = 0; s < E; ++s) {
        const long i = ia + stage1_point<L, P>(j, s);
        ph[s] = make_double2(phi[i], phi[i + L]);
    }
    // the other inputs of the points this thread ends with (rows A and B)
    struct In {
        double2 lx, ly, gx, gy, dph, ps;
    };
    auto load = [&](int s) {
        const long i = ia + last_point<L, P>(j, s);
        return In{make_double2(lx[i], lx[i + L]), make_double2(ly[i], ly[i + L]),
                  make_double2(gxp[i], gxp[i + L]), make_double2(gyp[i], gyp[i + L]),
                  make_double2(f[a.N + i], f[a.N + i + L]),
                  make_double2(f[2 * a.N + i], f[2 * a.N + i + L])};
    };
    In in[PRE ? E : 1];
    if constexpr (PRE) {
#pragma unroll
        for (int s = 0; s < E; ++s) in[s] = load(s);
    }
    {
        double2 spec[E];
        fft_line_wave_regs<L, -1, P>(
            my, j, tw,
            [&](int s, int) {
                return make_double2(ph[s].x - phi0, ph[s].y - phi0);
            },
            [&](int s, int, double2 v) { spec[s] = v; });
        line_sync<true>();
        fft_line_wave_regs<L, +1, P>(
            my, j, tw,
            [&](int s, int n) {
                const double2 v = spec[chain_slot<L, P>(s)];
                const double m = n > L / 2 ? L - n : n, k = -(a.k2 * m * m);
                return make_double2(v.x * k, v.y * k);
            },
            [&](int s, int, double2 v) { lz[s] = v; });
        line_sync<true>();
        fft_line_wave_regs<L, +1, P>(
            my, j, tw,
            [&](int s, int n) {
                const double2 v = spec[chain_slot<L, P>(s)];
                const double k = n > L / 2 ? a.k1 * (n - L)
                                           : (2 * n == L ? 0.0 : a.k1 * n);
                return make_double2(-v.y * k, v.x * k);
            },
            [&](int s, int, double2 v) { dz[s] = v; });
    }
    const double aa = f[a.Ntot - 1];
    const double a2 = aa * aa;
    double srho = 0.0, sp = 0.0;
#pragma unroll
    for (int s = 0; s < E; ++s) {
        const long i = ia + last_point<L, P>(j, s);
        const double2 p = ph[unchain_slot<L, P>(s)];
        if constexpr (!PRE) in[0] = load(s);
        const In &v = in[PRE ? s : 0];
        auto point = [&](long q, double p0, double d_x, double d_y, double d_z,
                         double lap, double dph, double ps) {
            double g = d_x * d_x;
            g += d_y * d_y;
            g += d_z * d_z;
            const double t1 = (0.5 - ps) * dph * dph;
            const double t2 = (0.5 + ps) * g / a2;
            const double V = a.m2 * p0 * p0 / 2.0;
            const double rv = t1 + t2 + V;
            const double pv = t1 - t2 / 3.0 - V;
            const double A = (1.0 + 4.0 * ps) * lap / a2 -
                             (1.0 + 2.0 * ps) * (a.m2 * p0);
            if (act) {
                outA[q] = A;
                outp[q] = pv;
                if (a.rho) {
                    a.rho[q] = rv;
                    a.pressure[q] = pv;
                }
                if constexpr (GW) {
                    R *g3 = a.g3 + bk.z * a.rg;
                    if constexpr (sizeof(R) == 4) {
                        g3[q] = (R)d_x;
                        g3[a.N + q] = (R)d_y;
                    }
                    g3[2 * a.N + q] = (R)d_z;
                }
                srho += rv;
                sp += pv;
            }
        };
        point(i, p.x + dc, v.gx.x, v.gy.x, dz[s].x, v.lx.x + v.ly.x + lz[s].x,
              v.dph.x, v.ps.x);
        point(i + L, p.y + dc, v.gx.y, v.gy.y, dz[s].y, v.lx.y + v.ly.y + lz[s].y,
              v.dph.y, v.ps.y);
        if constexpr (GW && sizeof(R) == 8) {
            g[0][s] = v.gx;
            g[1][s] = v.gy;
            g[2][s] = dz[s];
        } else if constexpr (GW) {
            auto src = [&](auto kc) {
                constexpr int K = decltype(kc)::value;
                g[K][s] = CT<C>::make(
                    (R)gw_source<K>(v.gx.x, v.gy.x, dz[s].x, a.ga.m),
                    (R)gw_source<K>(v.gx.y, v.gy.y, dz[s].y, a.ga.m));
            };
            src(std::integral_constant<int, 0>{});
            src(std::integral_constant<int, 1>{});
            src(std::integral_constant<int, 2>{});
            src(std::integral_constant<int, 3>{});
            src(std::integral_constant<int, 4>{});
        }
    }
    srho = wave_reduce<OpSum>(srho);
    sp = wave_reduce<OpSum>(sp);
    if (lane == 0) {
        double *part = a.partials + bk.z * a.e.p + 2 * wave;
        part[0] = srho;
        part[1] = sp;
    }
    }
    if constexpr (HELP) {
        static_assert(NG * sizeof(C) <= 3 * sizeof(double2), "see z_rhs_lds");
        C *const sh = reinterpret_cast<C *>(ltw + L) + lane;
        if (role == 0) {
#pragma unroll
            for (int s = 0; s < E; ++s)
#pragma unroll
                for (int q = 0; q < NG; ++q) sh[64 * (q * E + s)] = g[q][s];
        }
        lds_barrier();
        if (role != 0) {
#pragma unroll
            for (int s = 0; s < E; ++s)
#pragma unroll
                for (int q = 0; q < NG; ++q) g[q][s] = sh[64 * (q * E + s)];
        }
    }
    if constexpr (GW) {
        C *const cl = reinterpret_cast<C *>(wl); // the wavefront's own lines
        C *const cmy = cl + lane / T * PITCH;
        const long row0 = 2 * line0;
        C *const Wo = a.W + bk.z * a.rw + row0 * MZ;
        // FP64: the LDS table; FP32: its own in global memory
        const C *twc;
        if constexpr (sizeof(R) == 8)
            twc = tw;
        else
            twc = a.twc;
        auto comp = [&](auto kc) {
            constexpr int K = decltype(kc)::value;
            if (HELP && role != K % (WG / 64)) return;
            line_sync<true>(); // earlier LDS reads of these lines are done
            fft_line_impl<L, -1, true, false, P, C, true>(
                cmy, cmy, j, twc,
                [&](int s, int) {
                    const int q = chain_slot<L, P>(s);
                    if constexpr (sizeof(R) == 4)
                        return g[K][q];
                    else
                        return CT<C>::make(
                            gw_source<K>(g[0][q].x, g[1][q].x, g[2][q].x, a.ga.m),
                            gw_source<K>(g[0][q].y, g[1][q].y, g[2][q].y, a.ga.m));
                },
                NoWrite());
            for (int idx = lane; idx < 2 * LPW * MZ; idx += 64) {
                const int r = idx / MZ, k = idx - r * MZ;
                if (row0 + r < a.nrows)
                    Wo[K * a.M + idx] = herm_split<L>(cl + (r >> 1) * PITCH, k, r & 1);
            }
        };
        comp(std::integral_constant<int, 0>{});
        comp(std::integral_constant<int, 1>{});
        comp(std::integral_constant<int, 2>{});
        comp(std::integral_constant<int, 3>{});
        comp(std::integral_constant<int, 4>{});
    }
}

template <int L, bool GW, class C, int WG, bool HELP = false>
__global__ __launch_bounds__(WG) void k_z_rhs(ZRhsArgs<C> a)
{
    __shared__ double2 lds[z_rhs_lds<L, WG, HELP>()];
    z_rhs_body<L, GW, C, WG, HELP>(hw_blk(), lds, a);
}

// The derivative passes of nr realizations of a context: the field they
// differentiate (phi of f, or after the filter the fluctuations that the
// filter's last pass kept) and where the x and y gradients go
struct DerivIO {
    const double *phi;
    const double *dc;
    double *gx, *gy;
    long rphi, rdc, rxy; // realization strides (doubles)
};
DerivIO deriv_io(const ihg_ctx *c, const double *f, int filtered, int nr);
DerivXY deriv_axes(const ihg_ctx *c, const DerivIO &io, double *result, int nr);

// the filter's round trip and last pass
FilterFac filter_fac(const ihg_ctx *c, int output, int nr);
ZShift filter_shift(const ihg_ctx *c, int nr);

// the z pass of nr realizations of a context (no output arrays)
template <class C>
inline ZRhsArgs<C> z_rhs_args(const ihg_ctx *c, const double *f,
                              double *result, const DerivIO &io, int nr)
{
    using R = typename CT<C>::R;
    ZRhsArgs<C> a{};
    a.f = f;
    a.result = result;
    a.phi = io.phi;
    a.dc = io.dc;
    a.gx = io.gx;
    a.gy = io.gy;
    a.rphi = io.rphi;
    a.rdc = io.rdc;
    a.rxy = io.rxy;
    a.g3 = reinterpret_cast<R *>(c->grad3);
    a.W = reinterpret_cast<C *>(c->W);
    a.M = c->M;
    a.N = c->N;
    a.Ntot = c->Ntot;
    a.nrows = (long)c->Nx * c->Ny;
    a.partials = c->partials;
    a.m2 = c->p.mass * c->p.mass;
    a.k1 = c->kg.kz1 / c->Nz;
    a.k2 = c->kg.kz2 / c->Nz;
    a.ga = gw_axis(c->kg);
    a.tw = c->tw;
    if constexpr (sizeof(R) == 4)
        a.twc = c->twf;
    else
        a.twc = c->tw;
    if (nr > 1) {
        a.e = c->ens;
        a.rg = c->ens.g;
        a.rw = c->ens.w * (long)(sizeof(double2) / sizeof(C));
    }
    return a;
}

// rho_mean, pressure_mean (src/toolbox.c:241-242) and da (src/toolbox.c:87)
// of realization r (one thread; EP: the RK4 epilogue of the scale factor)
template <bool EP>
__device__ __forceinline__ void means_store(unsigned r, double rm, double pm,
                                            const double *__restrict__ f,
                                            double *__restrict__ result,
                                            long Ntot,
                                            double *__restrict__ dscal,
                                            const Ens &e, const Rk4Ep &ep)
{
    f += r * e.f;
    result += r * e.f;
    dscal += r * e.s;
    dscal[S_RHO_MEAN] = rm;
    dscal[S_P_MEAN] = pm;
    const double da = f[Ntot - 1] * sqrt(rm / 3.0);
    if constexpr (EP)
        rk4_ep_one(ep.shifted(r * e.f), Ntot - 1, da, result + Ntot - 1);
    else
        result[Ntot - 1] = da;
}

// (one work-group per realization r; sh: MEANS_WG / 64 doubles of LDS)
constexpr int MEANS_WG = 1024;
template <bool EP = false>
__device__ __forceinline__ void means_body(
    unsigned r, double *sh, const double *__restrict__ partials, int nparts,
    long N, const double *__restrict__ f, double *__restrict__ result,
    long Ntot, double *__restrict__ dscal, const Ens &e,
    const Rk4Ep &ep = Rk4Ep{})
{
    partials += r * e.p;
    // (rho, p) pairs as 16-byte loads, four in flight per thread
    const double2 *p2 = reinterpret_cast<const double2 *>(partials);
    double s0 = 0.0, s1 = 0.0;
#pragma unroll 4
    for (int i = threadIdx.x; i < nparts; i += MEANS_WG) {
        const double2 v = p2[i];
        s0 += v.x;
        s1 += v.y;
    }
    s0 = block_reduce<OpSum>(s0, sh, MEANS_WG);
    s1 = block_reduce<OpSum>(s1, sh, MEANS_WG);
    if (threadIdx.x == 0)
        means_store<EP>(r, s0 / N, s1 / N, f, result, Ntot, dscal, e, ep);
}

// The sums of means_body by a work-group of RED_WG threads, bit for bit: a
// thread stands for MEANS_WG / RED_WG of its threads, and the wavefronts' sums
// are added in its order.  sh: 2 MEANS_WG / 64 doubles; every thread gets the
// sums; synchronises.
__device__ __forceinline__ void means_sums(const double *__restrict__ partials,
                                           int nparts, double *sh, double &s0,
                                           double &s1)
{
    constexpr int V = MEANS_WG / RED_WG, NWV = MEANS_WG / 64;
    const double2 *p2 = reinterpret_cast<const double2 *>(partials);
    double a[V], b[V];
#pragma unroll
    for (int v = 0; v < V; ++v) {
        a[v] = b[v] = 0.0;
        for (int i = (int)threadIdx.x + RED_WG * v; i < nparts; i += MEANS_WG) {
            const double2 q = p2[i];
            a[v] += q.x;
            b[v] += q.y;
        }
    }
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
#pragma unroll
    for (int v = 0; v < V; ++v) {
        a[v] = wave_reduce<OpSum>(a[v]);
        b[v] = wave_reduce<OpSum>(b[v]);
        if (lane == 0) {
            sh[w + (RED_WG / 64) * v] = a[v];
            sh[NWV + w + (RED_WG / 64) * v] = b[v];
        }
    }
    __syncthreads();
    s0 = sh[0];
    s1 = sh[NWV];
#pragma unroll
    for (int i = 1; i < NWV; ++i) {
        s0 += sh[i];
        s1 += sh[NWV + i];
    }
}

// update_phi_psi (src/toolbox.c:282-299); the part A of the slope of dphi and
// p were parked in result[0..N) and result[3N..4N) by k_z_rhs
// (work-group bx of gx on realization z; EP: the RK4 epilogue of the four
// blocks' slopes, AHEAD with its loads before the first store; rm, pm: the
// means of rho and p)
template <bool NT, bool EP = false, bool AHEAD = false>
__device__ __forceinline__ void update_phi_psi_body(
    unsigned bx, unsigned gx, unsigned z, const double *__restrict__ f,
    double *__restrict__ result, long N, double rm, double pm, const Ens &e,
    const Rk4Ep &ep0 = Rk4Ep{})
{
    f += z * e.f;
    result += z * e.f;
    [[maybe_unused]] const Rk4Ep ep = EP ? ep0.shifted(z * e.f) : ep0;
    const double hubble = sqrt(rm / 3.0);
    const double h3 = 3.0 * hubble;
    // pairs of points (16-byte loads and stores; N is even and every block
    // starts 16-byte aligned)
    const long stride = (long)gx * RED_WG;
    const double2 *F = reinterpret_cast<const double2 *>(f);
    double2 *Rs = reinterpret_cast<double2 *>(result);
    const long H = N / 2;
    for (long i = (long)bx * RED_WG + threadIdx.x; i < H; i += stride) {
        const double2 dph = ld2<NT>(F + H + i), ps = ld2<NT>(F + 2 * H + i),
                      dps = ld2<NT>(F + 3 * H + i);
        const double2 A = ld2<NT>(Rs + i), pr = ld2<NT>(Rs + 3 * H + i);
        [[maybe_unused]] Rk4In in[4];
        if constexpr (EP && AHEAD) {
#pragma unroll
            for (int q = 0; q < 4; ++q) in[q] = rk4_ep_load<NT>(ep, q * H + i);
        }
        const double2 r1 = make_double2(A.x - (h3 - 4.0 * dps.x) * dph.x,
                                        A.y - (h3 - 4.0 * dps.y) * dph.y);
        const double2 r3 = make_double2(
            0.5 * pr.x + (ps.x - 0.5) * pm - 4.0 * hubble * dps.x,
            0.5 * pr.y + (ps.y - 0.5) * pm - 4.0 * hubble * dps.y);
        if constexpr (EP) {
            auto put = [&](int q, double2 k) {
                if constexpr (AHEAD)
                    rk4_ep_store<NT>(ep, q * H + i, in[q], k, Rs + q * H + i);
                else
                    rk4_ep_pair<NT>(ep, q * H + i, k, Rs + q * H + i);
            };
            put(0, dph);
            put(1, r1);
            put(2, dps);
            put(3, r3);
        } else {
            st2<NT>(Rs + i, dph);
            st2<NT>(Rs + H + i, r1);
            st2<NT>(Rs + 2 * H + i, dps);
            st2<NT>(Rs + 3 * H + i, r3);
        }
    }
}

// the means of realization z from k_means
template <bool NT, bool EP = false>
__device__ __forceinline__ void update_after_means_body(
    unsigned bx, unsigned gx, unsigned z, const double *__restrict__ f,
    double *__restrict__ result, long N, const double *__restrict__ dscal,
    const Ens &e, const Rk4Ep &ep = Rk4Ep{})
{
    const double *d = dscal + z * e.s;
    update_phi_psi_body<NT, EP>(bx, gx, z, f, result, N, d[S_RHO_MEAN],
                                d[S_P_MEAN], e, ep);
}

// ---------------------------------------------------------------------------
// TT projection (mk_gw_sources_tt, src/toolbox.c:363-397) as two linear forms
// of the source components: o0 = sum_c alpha_c S_c, o1 = sum_c beta_c S_c.
// With f = k / k^2 (full k), t1 = sum_ij k_i f_j S_ij, t2 = tr S, s1 = t1 + t2,
// s2 = t1 - t2 and the kept axis pair (p, q) = (x, y) if |kz| > eps, (x, z)
// if |ky| > eps, (y, z) otherwise, the reference computes
//   o0 = S_pp - 2 f_p (sum_j k_j S_pj) + (f_p k_p s1 + s2) / 2
//   o1 = S_pq - f_p (sum_j k_j S_qj) - f_q (sum_j k_j S_pj) + f_p k_q s1 / 2
// alpha_C, beta_C are the derivatives of these with respect to component
// C = 0..5 = (xx, xy, xz, yy, yz, zz); the k = 0 mode projects to 0.
// tt_source_coef<K> gives those of source component K: zz in the place of xx
// (K = 0) where xx is the product subtracted from the others, of yy (K = 3)
// where yy is.
// ---------------------------------------------------------------------------
template <int C, class R>
__device__ __forceinline__ void tt_coef(R kx, R ky, R kz, R inv_ksq,
                                        bool b1, bool zero, R &al, R &be)
{
    const R fx = kx * inv_ksq, fy = ky * inv_ksq, fz = kz * inv_ksq;
    const bool b2 = !b1 && fabs((double)ky) > DBL_EPSILON;
    const bool py = !b1 && !b2; // p = y, else p = x
    const bool qy = b1;         // q = y, else q = z
    const R kp = py ? ky : kx, fp = py ? fy : fx;
    const R kq = qy ? ky : kz, fq = qy ? fy : fz;
    R t1, t2, rowp, rowq, dpp, dpq;
    const R O = 0, I = 1, D = 2;
    if constexpr (C == 0) {
        t1 = kx * fx; t2 = I; rowp = py ? O : kx; rowq = O;
        dpp = py ? O : I; dpq = O;
    } else if constexpr (C == 1) {
        t1 = D * (kx * fy); t2 = O; rowp = py ? kx : ky;
        rowq = qy ? kx : O; dpp = O; dpq = (!py && qy) ? I : O;
    } else if constexpr (C == 2) {
        t1 = D * (kx * fz); t2 = O; rowp = py ? O : kz;
        rowq = qy ? O : kx; dpp = O; dpq = (!py && !qy) ? I : O;
    } else if constexpr (C == 3) {
        t1 = ky * fy; t2 = I; rowp = py ? ky : O; rowq = qy ? ky : O;
        dpp = py ? I : O; dpq = O;
    } else if constexpr (C == 4) {
        t1 = D * (ky * fz); t2 = O; rowp = py ? kz : O;
        rowq = qy ? kz : ky; dpp = O; dpq = py ? I : O;
    } else {
        t1 = kz * fz; t2 = I; rowp = O; rowq = qy ? O : kz;
        dpp = O; dpq = O;
    }
    const R s1 = t1 + t2, s2 = t1 - t2;
    const R half = (R)0.5, two = (R)2.0;
    al = zero ? (R)0 : dpp - two * fp * rowp + half * (fp * kp * s1 + s2);
    be = zero ? (R)0 : dpq - fp * rowq - fq * rowp + half * fp * kq * s1;
}

template <int K, class R>
__device__ __forceinline__ void tt_source_coef(R kx, R ky, R kz, R inv_ksq,
                                               bool b1, bool zero, int m,
                                               R &al, R &be)
{
    if constexpr (K == 0 || K == 3) {
        if (m == (K == 0 ? 0 : 1)) { // uniform
            tt_coef<5>(kx, ky, kz, inv_ksq, b1, zero, al, be);
            return;
        }
    }
    tt_coef<K>(kx, ky, kz, inv_ksq, b1, zero, al, be);
}

// y transform of source component K (its z and x passes are done) with the
// TT accumulation folded into the last Stockham stage; `cur` holds the
// component's first-stage points (loaded ahead).  Two layouts: the
// work-group's threads, lanes over the B lines as the loads are (thread j
// of line `lb`), run the first stage from `cur` into the component's LDS
// buffer, then one work-group barrier; then each wavefront runs the other
// stages on its own lines (thread jw of line `lw`) with wavefront-local
// exchanges.  Components alternate between two LDS buffers: the barrier of
// component K also ends every wavefront's use of the buffer component K + 1
// writes.  kx, kz, b1 (|k_z| > eps) and z0 (ix = iz = 0) are those of line
// lw, inv_ksq the 1/k^2 of its points, m the axis of GwAxis.
template <int L, class P, int K, class C>
__device__ __forceinline__ void tt_component(
    C *lb, C *lw, int j, int jw, const C *__restrict__ tw, const C *cur,
    const KGeom &kg, typename CT<C>::R kx, typename CT<C>::R kz, bool b1,
    bool z0, const typename CT<C>::R *inv_ksq, int m, C *o0, C *o1)
{
    using R = typename CT<C>::R;
    // Register pressure control (empty asm statements, no instructions):
    // an opaque zero offset of the twiddle pointer per component (the
    // pointer itself stays visibly an LDS one) stops the compiler from
    // loading every stage twiddle once and holding it across all the
    // transforms, and pinning the accumulators after each component stops it
    // from deferring the sums (and so keeping every spectrum live).
    int zo = 0;
    asm volatile("" : "+s"(zo));
    const C *twc = tw + zo;
    auto rd = [&](int s, int) { return cur[s]; };
    NoWrite nw;
    stockham_stage<L, P::R0, 1, -1, true, false, P, C, false>(lb, lb, j, twc,
                                                              rd, nw);
    auto acc = [&](int s, int n, C v) {
        // recomputed per component from 1/k^2 alone: an empty asm keeps the
        // compiler from holding every derived coefficient of every point
        // live across the transforms
        R iv = inv_ksq[s];
        asm volatile("" : "+v"(iv));
        const bool zero = z0 && (n == 0);
        R al, be;
        tt_source_coef<K>(kx, (R)kg.kyf(n), kz, iv, b1, zero, m, al, be);
        if constexpr (K == 0) {
            o0[s] = CT<C>::make(al * v.x, al * v.y);
            o1[s] = CT<C>::make(be * v.x, be * v.y);
        } else {
            o0[s] = CT<C>::make(o0[s].x + al * v.x, o0[s].y + al * v.y);
            o1[s] = CT<C>::make(o1[s].x + be * v.x, o1[s].y + be * v.y);
        }
    };
    fft_stages_wave<L, -1, P, 1, C>(lw, jw, twc, acc);
#pragma unroll
    for (int s = 0; s < P::E; ++s)
        asm volatile("" : "+v"(o0[s].x), "+v"(o0[s].y), "+v"(o1[s].x),
                     "+v"(o1[s].y));
}

// Line plans of the fused y pass: few values per thread (radix-4 stages),
// so that the two TT accumulators, 1/k^2 and the transform of every point a
// thread owns stay in registers.
template <int L> struct TTPlan;
template <> struct TTPlan<4>   { using P = PlanT<2, 2, 2>; static constexpr int WG = 256; };
template <> struct TTPlan<8>   { using P = PlanT<4, 4, 2>; static constexpr int WG = 256; };
template <> struct TTPlan<16>  { using P = PlanT<4, 4, 4>; static constexpr int WG = 256; };
template <> struct TTPlan<32>  { using P = PlanT<4, 4, 4, 2>; static constexpr int WG = 256; };
template <> struct TTPlan<64>  { using P = PlanT<4, 4, 4, 4>; static constexpr int WG = 256; };
template <> struct TTPlan<128> { using P = PlanT<4, 4, 4, 4, 2>; static constexpr int WG = 512; };
template <> struct TTPlan<256> { using P = PlanT<4, 4, 4, 4, 4>; static constexpr int WG = 512; };
template <> struct TTPlan<512> { using P = PlanT<8, 8, 4, 4, 4>; static constexpr int WG = 512; };

// LDS of the fused pass in complex values: two lines per tile line and the
// L stage twiddles
template <int L, int WG, class P>
__host__ __device__ constexpr int tt_lds()
{
    return 2 * (WG / (L / P::E)) * Lds<L>::PITCH + L;
}

// update_h at one point (src/toolbox.c:311-346) from the two projected sources
struct HUpdate {
    double a2, h3, pm;
    double2 *r2;
    long Nh1, Nh2, Ndh1, Ndh2; // offsets of the h blocks in complex values
    __device__ __forceinline__ HUpdate(const double *f, double *result, long N,
                                       long Next, long Ntot, const double *dscal)
    {
        const double aa = f[Ntot - 1];
        a2 = aa * aa;
        h3 = 3.0 * sqrt(dscal[S_RHO_MEAN] / 3.0);
        pm = dscal[S_P_MEAN];
        r2 = reinterpret_cast<double2 *>(result);
        Nh1 = 2 * N;
        Nh2 = Nh1 + Next / 2;
        Ndh1 = Nh2 + Next / 2;
        Ndh2 = Ndh1 + Next / 2;
    }
    // AHEAD: what the epilogue reads of the four blocks is loaded first
    template <bool EP, bool AHEAD>
    __device__ __forceinline__ void point(long i, double ksq, double2 h1,
                                          double2 h2, double2 d1, double2 d2,
                                          double2 s0, double2 s1,
                                          const Rk4Ep &ep) const
    {
        const double tmp = -(2.0 * pm + ksq / a2);
        const double2 v1 = make_double2(tmp * h1.x - h3 * d1.x + 2.0 * s0.x / a2,
                                        tmp * h1.y - h3 * d1.y + 2.0 * s0.y / a2);
        const double2 v2 = make_double2(tmp * h2.x - h3 * d2.x + 2.0 * s1.x / a2,
                                        tmp * h2.y - h3 * d2.y + 2.0 * s1.y / a2);
        if constexpr (EP) {
            [[maybe_unused]] Rk4In in[4];
            if constexpr (AHEAD) {
                in[0] = rk4_ep_load<false>(ep, Nh1 + i);
                in[1] = rk4_ep_load<false>(ep, Nh2 + i);
                in[2] = rk4_ep_load<false>(ep, Ndh1 + i);
                in[3] = rk4_ep_load<false>(ep, Ndh2 + i);
            }
            auto put = [&](int q, long at, double2 k) {
                if constexpr (AHEAD)
                    rk4_ep_store<false>(ep, at, in[q], k, r2 + at);
                else
                    rk4_ep_pair<false>(ep, at, k, r2 + at);
            };
            put(0, Nh1 + i, d1);
            put(1, Nh2 + i, d2);
            put(2, Ndh1 + i, v1);
            put(3, Ndh2 + i, v2);
        } else {
            r2[Nh1 + i] = d1;
            r2[Nh2 + i] = d2;
            r2[Ndh1 + i] = v1;
            r2[Ndh2 + i] = v2;
        }
    }
};

// Last pass of the GW sources: y transforms of the components (z and x
// passes done), the TT projection, and update_h (src/toolbox.c:311-346):
//   dh = hdot,  dhdot = -(2 p_mean + k^2/a^2) h - 3 H hdot + 2 S^TT / a^2
// (EP: the RK4 epilogue of the four h blocks' slopes)
template <int L, int WG, class P, class C, bool EP = false>
__device__ __forceinline__ void y_tt_update_h_body(
    const Blk &bk, C *lds, const C *W, long M, const double *__restrict__ f,
    double *__restrict__ result, long N, long Next, long Ntot,
    const KGeom &kg, const double *__restrict__ dscal, const LineSet &ls,
    const C *__restrict__ tw, const Ens &e, long rw, GwAxis ga,
    const Rk4Ep &ep0 = Rk4Ep{})
{
    // realization z of an ensemble (rw: its W stride in units of C)
    W += bk.z * rw;
    f += bk.z * e.f;
    result += bk.z * e.f;
    dscal += bk.z * e.s;
    using R = typename CT<C>::R;
    constexpr int E = P::E, T = L / E, B = WG / T, PITCH = Lds<L>::PITCH;
    const int tid = threadIdx.x, b = tid % B, j = tid / B;
    const long line = (long)tile_x<true>(bk) * B + b;
    const bool act = line < ls.nlines;
    const long lc = act ? line : 0;
    const long base = ls.base(lc);
    const int ix = (int)(lc / kg.Mz), iz = (int)(lc - (long)ix * kg.Mz);
    const long st = ls.stride;
    // The stage twiddles tw[L, 2L) are staged in LDS behind the lines and
    // read from there: LDS reads are counted apart from the vector-memory
    // loads, which return in order, so a twiddle read never waits for the
    // source and h loads issued ahead of it (from global memory it would
    // wait for all of them).  The first stage, whose barrier makes them
    // visible, takes no twiddle.
    {
        C *const ltw = lds + 2 * B * PITCH;
        for (int i = tid; i < L; i += WG)
            ltw[i] = tw[L + i];
        tw = ltw - L; // indices L + [0, L) of the table
    }
    // The wavefront layout of the stages after the first: wavefront w owns
    // lines w LPW + [0, LPW) of the tile, thread jw of line bw.  (The
    // wavefront index is uniform: with one line per wavefront its
    // coordinates and k_x, k_z live in scalar registers.)
    constexpr int LPW = 64 / T;
    const int wv = __builtin_amdgcn_readfirstlane(tid / 64);
    const int bw = wv * LPW + (tid % 64) / T, jw = tid % T;
    const long linew = (long)tile_x<true>(bk) * B + bw;
    const long lcw = linew < ls.nlines ? linew : 0;
    const int ixw = (int)(lcw / kg.Mz), izw = (int)(lcw - (long)ixw * kg.Mz);
    const R kxw = (R)kg.kxf(ixw), kzw = (R)kg.kzf(izw);
    const bool b1w = fabs(kg.kzf(izw)) > DBL_EPSILON; // branch on the FP64 k
    const bool z0w = (ixw == 0) && (izw == 0);
    R inv[E];
#pragma unroll
    for (int s = 0; s < E; ++s) {
        const int n = last_point<L, P>(jw, s);
        inv[s] = (z0w && n == 0) ? (R)0 : (R)(1.0 / kg.ksq(ixw, n, izw));
    }
    // the two LDS buffers, at this thread's line of each layout
    C *const lb0 = lds + b * PITCH, *const lb1 = lds + (B + b) * PITCH;
    C *const lw0 = lds + bw * PITCH, *const lw1 = lds + (B + bw) * PITCH;
    // first-stage points of component c, in bounds for every lane (an idle
    // lane loads line 0's points and its results are never stored); the
    // loads of component c + 1 are issued before the transform of c, so
    // their latency hides behind it.  The loaded values are used as they
    // are: a select on them right after the load would wait for it there.
    // (Loading two components ahead measured no faster.)
    auto load = [&](int c, C *buf) {
        const C *src = W + c * M + base;
#pragma unroll
        for (int s = 0; s < E; ++s)
            buf[s] = src[(long)stage1_point<L, P>(j, s) * st];
    };
    // update_h's inputs (h and hdot at the points this thread ends with;
    // line 0's points for an idle lane, in bounds): with few points per
    // thread they are loaded before the last transform, so their latency
    // hides behind it (with E = 8 the registers are not there)
    const long Nh1 = 4 * N, Nh2 = Nh1 + Next, Ndh1 = Nh2 + Next,
               Ndh2 = Ndh1 + Next;
    const double2 *f2 = reinterpret_cast<const double2 *>(f);
    constexpr bool EARLY = E <= 4;
    double2 h1v[E], h2v[E], d1v[E], d2v[E];
    auto load_h = [&]() {
#pragma unroll
        for (int s = 0; s < E; ++s) {
            const long i = base + last_point<L, P>(j, s) * st;
            h1v[s] = f2[Nh1 / 2 + i];
            h2v[s] = f2[Nh2 / 2 + i];
            d1v[s] = f2[Ndh1 / 2 + i];
            d2v[s] = f2[Ndh2 / 2 + i];
        }
    };
    C o0[E], o1[E], bufs[2][E];
    load(0, bufs[0]);
    load(1, bufs[1]);
    auto step = [&](auto kc) {
        constexpr int K = decltype(kc)::value;
        if constexpr (K == GW_NC - 1 && EARLY) load_h();
        tt_component<L, P, K>(K % 2 ? lb1 : lb0, K % 2 ? lw1 : lw0, j, jw, tw,
                              bufs[K % 2], kg, kxw, kzw, b1w, z0w, inv, ga.m,
                              o0, o1);
        if constexpr (K + 2 < GW_NC) load(K + 2, bufs[K % 2]);
    };
    step(std::integral_constant<int, 0>{});
    step(std::integral_constant<int, 1>{});
    step(std::integral_constant<int, 2>{});
    step(std::integral_constant<int, 3>{});
    step(std::integral_constant<int, 4>{});
    // the two sums back to the load layout through LDS: o1 to buffer 1 (no
    // wavefront reads it after the last component's barrier), o0 to this
    // wavefront's own line of buffer 0 once its last reads of it are done
    static_assert(GW_NC == 5, "the last component is in buffer 0");
#pragma unroll
    for (int s = 0; s < E; ++s)
        lw1[Lds<L>::idx(last_point<L, P>(jw, s))] = o1[s];
    line_sync<true>();
#pragma unroll
    for (int s = 0; s < E; ++s)
        lw0[Lds<L>::idx(last_point<L, P>(jw, s))] = o0[s];
    lds_barrier();
#pragma unroll
    for (int s = 0; s < E; ++s) {
        const int n = Lds<L>::idx(last_point<L, P>(j, s));
        o0[s] = lb0[n];
        o1[s] = lb1[n];
    }
    if constexpr (!EARLY) load_h();
    if (!act)
        return;
    const HUpdate hu(f, result, N, Next, Ntot, dscal);
    const Rk4Ep ep = EP ? ep0.shifted(bk.z * e.f) : ep0;
#pragma unroll
    for (int s = 0; s < E; ++s) {
        const int n = last_point<L, P>(j, s);
        hu.template point<EP, false>(base + n * st, kg.ksq(ix, n, iz), h1v[s], h2v[s],
                              d1v[s], d2v[s], make_double2(o0[s].x, o0[s].y),
                              make_double2(o1[s].x, o1[s].y), ep);
    }
}

template <int L, int WG, class P, class C>
__global__ __launch_bounds__(WG) void k_y_tt_update_h(
    const C *W, long M, const double *__restrict__ f,
    double *__restrict__ result, long N, long Next, long Ntot, KGeom kg,
    const double *__restrict__ dscal, LineSet ls, const C *__restrict__ tw,
    Ens e, long rw, GwAxis ga)
{
    __shared__ C lds[tt_lds<L, WG, P>()];
    y_tt_update_h_body<L, WG, P, C>(hw_blk(), lds, W, M, f, result, N, Next,
                                    Ntot, kg, dscal, ls, tw, e, rw, ga);
}


// ---------------------------------------------------------------------------
// The same pass for grids that leave the chip idle: latency bounds it (one 64^3
// grid is 528 wavefronts, each running five transforms in turn), so the five
// components of a tile are transformed at the same time by a fifth of the
// work-group each, in one layout with work-group barriers, and after the last
// stage every thread takes points of the tile: five spectra from LDS, the
// projection in the order of tt_component, and update_h, whose inputs were
// loaded before the transforms.  Line plans have the radices of TTPlan and the
// sums their order, so the values are the same bit for bit.  7 x 16^3 with the
// RK4 epilogue 13.3 -> 6.2 us, 3 x 32^3 16.3 -> 7.4, 64^3 13.1 -> 12.0; the
// rule of tt_wide has the sizes where it loses.
// ---------------------------------------------------------------------------
template <int L> struct TTWidePlan { using P = typename TTPlan<L>::P; static constexpr int B = 8; };
template <> struct TTWidePlan<4> { using P = PlanT<4, 2, 2>; static constexpr int B = 64; };
template <> struct TTWidePlan<8> { using P = PlanT<4, 4, 2>; static constexpr int B = 32; };
template <> struct TTWidePlan<16> { using P = PlanT<4, 4, 4>; static constexpr int B = 16; };
template <> struct TTWidePlan<128> { using P = PlanT<8, 4, 4, 4, 2>; static constexpr int B = 8; };

// lines up to 128 points: 256 would need 175 KB of LDS for 128-byte runs, and
// with shorter ones it loses (64 x 256 x 32: 32-byte runs 24.8 us, 64-byte
// runs 26.2, components in turn 21.9)
constexpr int TT_WIDE_MAX = 128;

template <int L>
struct TTWide {
    using P = typename TTWidePlan<L>::P;
    static constexpr int B = TTWidePlan<L>::B, T = L / P::E;
    static constexpr int WG = GW_NC * B * T, LDS = GW_NC * B * Lds<L>::PITCH;
    static_assert(WG % 64 == 0 && WG <= 1024, "whole wavefronts");
};

template <int L, class C, bool EP>
__device__ __forceinline__ void y_tt_wide_body(
    const Blk &bk, C *lds, const C *W, long M, const double *__restrict__ f,
    double *__restrict__ result, long N, long Next, long Ntot,
    const KGeom &kg, const double *__restrict__ dscal, const LineSet &ls,
    const C *__restrict__ tw, const Ens &e, long rw, GwAxis ga,
    const Rk4Ep &ep0)
{
    using TT = TTWide<L>;
    using P = typename TT::P;
    using R = typename CT<C>::R;
    constexpr int B = TT::B, T = TT::T, WG = TT::WG, PITCH = Lds<L>::PITCH;
    constexpr int NP = (B * L + WG - 1) / WG; // points per thread
    W += bk.z * rw;
    f += bk.z * e.f;
    result += bk.z * e.f;
    dscal += bk.z * e.s;
    const int tid = threadIdx.x;
    const long line0 = (long)tile_x<true>(bk) * B;
    const long st = ls.stride;
    // the transform of component c: thread j of line b; idle lines transform
    // line 0 (in bounds)
    const int c = tid / (B * T), t = tid % (B * T), b = t % B, j = t / B;
    const long line = line0 + b;
    const C *src = W + c * M + ls.base(line < ls.nlines ? line : 0);
    C buf[P::E];
#pragma unroll
    for (int s = 0; s < P::E; ++s)
        buf[s] = src[(long)stage1_point<L, P>(j, s) * st];
    // this thread's points: line pb, point pn; h and hdot ahead
    const HUpdate hu(f, result, N, Next, Ntot, dscal);
    const double2 *f2 = reinterpret_cast<const double2 *>(f);
    double2 h1[NP], h2[NP], d1[NP], d2[NP];
#pragma unroll
    for (int p = 0; p < NP; ++p) {
        const int q = tid + p * WG, pb = q % B, pn = q / B;
        const long pl = line0 + pb;
        const long i = pn < L && pl < ls.nlines ? ls.base(pl) + pn * st : 0;
        h1[p] = f2[hu.Nh1 + i];
        h2[p] = f2[hu.Nh2 + i];
        d1[p] = f2[hu.Ndh1 + i];
        d2[p] = f2[hu.Ndh2 + i];
    }
    fft_line<L, -1, true, false, P>(lds + (c * B + b) * PITCH, j, tw,
                                    [&](int s, int) { return buf[s]; });
    const Rk4Ep ep = EP ? ep0.shifted(bk.z * e.f) : ep0;
#pragma unroll
    for (int p = 0; p < NP; ++p) {
        const int q = tid + p * WG, pb = q % B, pn = q / B;
        const long pl = line0 + pb;
        if (pn >= L || pl >= ls.nlines) continue;
        const int ix = (int)(pl / kg.Mz), iz = (int)(pl - (long)ix * kg.Mz);
        const bool zero = ix == 0 && iz == 0 && pn == 0;
        const bool b1 = fabs(kg.kzf(iz)) > DBL_EPSILON;
        const double ksq = kg.ksq(ix, pn, iz);
        const R inv = zero ? (R)0 : (R)(1.0 / ksq);
        const R kx = (R)kg.kxf(ix), ky = (R)kg.kyf(pn), kz = (R)kg.kzf(iz);
        const C *v = lds + pb * PITCH + Lds<L>::idx(pn);
        C o0, o1;
        auto add = [&](auto kc) {
            constexpr int K = decltype(kc)::value;
            R al, be;
            tt_source_coef<K>(kx, ky, kz, inv, b1, zero, ga.m, al, be);
            const C u = v[K * B * PITCH];
            if constexpr (K == 0) {
                o0 = CT<C>::make(al * u.x, al * u.y);
                o1 = CT<C>::make(be * u.x, be * u.y);
            } else {
                o0 = CT<C>::make(o0.x + al * u.x, o0.y + al * u.y);
                o1 = CT<C>::make(o1.x + be * u.x, o1.y + be * u.y);
            }
        };
        add(std::integral_constant<int, 0>{});
        add(std::integral_constant<int, 1>{});
        add(std::integral_constant<int, 2>{});
        add(std::integral_constant<int, 3>{});
        add(std::integral_constant<int, 4>{});
        hu.template point<EP, true>(ls.base(pl) + pn * st, ksq, h1[p], h2[p], d1[p],
                              d2[p], make_double2(o0.x, o0.y),
                              make_double2(o1.x, o1.y), ep);
    }
}

template <int L, class C, bool EP>
__global__ __launch_bounds__(TTWide<L>::WG) void k_y_tt_wide(
    const C *W, long M, const double *__restrict__ f,
    double *__restrict__ result, long N, long Next, long Ntot, KGeom kg,
    const double *__restrict__ dscal, LineSet ls, const C *__restrict__ tw,
    Ens e, long rw, GwAxis ga, Rk4Ep ep)
{
    __shared__ C lds[TTWide<L>::LDS];
    y_tt_wide_body<L, C, EP>(hw_blk(), lds, W, M, f, result, N, Next, Ntot, kg,
                             dscal, ls, tw, e, rw, ga, ep);
}

} // namespace ihg
