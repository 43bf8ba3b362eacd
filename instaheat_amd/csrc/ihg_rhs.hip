// ihg_rhs.hip -- the right-hand side mk_rhs (src/toolbox.c:75-626) as fused
// HIP kernels.
//
// Data flow of one call (no filter, no output):
//   derivatives     phi -> d_x phi, d_xx phi and d_y phi, d_yy phi, each from
//                   transforms along its own axis       (toolbox.c:132-139)
//   z pass          phi, its x and y derivatives, dphi, psi -> p, the part of
//                   the slope of dphi without means, block sums of rho and p;
//                   with GW the z r2c of five source products (pairs of rows
//                   in one complex row)                 (toolbox.c:140-243)
//   means           block sums -> rho_mean, pressure_mean, da   (:87, :241)
//   update          result[0..4N)                       (toolbox.c:282-299)
// GW on adds an x pass of the source components and one y pass that also does
// the TT projection and the h update (toolbox.c:311-424).
#include <algorithm>
#include <cfloat>
#include <cmath>
#include <type_traits>

#include "dispatch.h"
#include "fft_kernels.h"
#include "ihg_internal.h"
#include "mem.h"
#include "reduce.h"
#include "rhs_kernels.h"

namespace ihg {

static inline unsigned nblocks(long n, int per_block, unsigned cap)
{
    long b = (n + per_block - 1) / per_block;
    if (b < 1) b = 1;
    return (unsigned)(b > (long)cap ? cap : b);
}

// rho_mean, pressure_mean and da of every realization (one work-group each)
__global__ __launch_bounds__(MEANS_WG) void k_means(
    const double *__restrict__ partials, int nparts, long N,
    const double *__restrict__ f, double *__restrict__ result, long Ntot,
    double *__restrict__ dscal, Ens e)
{
    __shared__ double sh[MEANS_WG / 64];
    means_body(blockIdx.x, sh, partials, nparts, N, f, result, Ntot, dscal, e);
}

// (with the RK4 epilogue of the scale factor's slope)
__global__ __launch_bounds__(MEANS_WG) void k_means_rk4(
    const double *__restrict__ partials, int nparts, long N,
    const double *__restrict__ f, double *__restrict__ result, long Ntot,
    double *__restrict__ dscal, Ens e, Rk4Ep ep)
{
    __shared__ double sh[MEANS_WG / 64];
    means_body<true>(blockIdx.x, sh, partials, nparts, N, f, result, Ntot,
                     dscal, e, ep);
}

template <bool NT>
__global__ __launch_bounds__(RED_WG) void k_update_phi_psi(
    const double *__restrict__ f, double *__restrict__ result, long N,
    const double *__restrict__ dscal, Ens e)
{
    update_after_means_body<NT>(blockIdx.x, gridDim.x, blockIdx.z, f, result, N,
                                dscal, e);
}

template <bool NT>
__global__ __launch_bounds__(RED_WG) void k_update_phi_psi_rk4(
    const double *__restrict__ f, double *__restrict__ result, long N,
    const double *__restrict__ dscal, Ens e, Rk4Ep ep)
{
    update_after_means_body<NT, true>(blockIdx.x, gridDim.x, blockIdx.z, f,
                                      result, N, dscal, e, ep);
}

// k_means and the update in one launch for few partial sums: every
// work-group adds them up itself (the same sums bit for bit), the first of a
// realization also stores the means and does the scale factor.
template <bool EP, bool AHEAD>
__global__ __launch_bounds__(RED_WG) void k_means_update(
    const double *__restrict__ partials, int nparts, long N,
    const double *__restrict__ f, double *__restrict__ result, long Ntot,
    double *__restrict__ dscal, Ens e, Rk4Ep ep)
{
    __shared__ double sh[2 * MEANS_WG / 64];
    const unsigned z = blockIdx.z;
    double s0, s1;
    means_sums(partials + z * e.p, nparts, sh, s0, s1);
    const double rm = s0 / N, pm = s1 / N;
    if (blockIdx.x == 0 && threadIdx.x == 0)
        means_store<EP>(z, rm, pm, f, result, Ntot, dscal, e, ep);
    update_phi_psi_body<false, EP, AHEAD>(blockIdx.x, gridDim.x, z, f, result, N,
                                          rm, pm, e, ep);
}

template <int L, int WG, class P>
__global__ __launch_bounds__(WG) void k_y_tt_update_h_rk4(
    const double2 *W, long M, const double *__restrict__ f,
    double *__restrict__ result, long N, long Next, long Ntot, KGeom kg,
    const double *__restrict__ dscal, LineSet ls,
    const double2 *__restrict__ tw, Ens e, long rw, GwAxis ga, Rk4Ep ep)
{
    __shared__ double2 lds[tt_lds<L, WG, P>()];
    y_tt_update_h_body<L, WG, P, double2, true>(hw_blk(), lds, W, M, f, result,
                                                N, Next, Ntot, kg, dscal, ls,
                                                tw, e, rw, ga, ep);
}

// the y line lengths whose TT pass has the RK4 epilogue compiled in
template <class F>
static int dispatch_rk4_len(int L, F &&f)
{
    switch (L) {
    case 16: return f(std::integral_constant<int, 16>{});
    case 32: return f(std::integral_constant<int, 32>{});
    case 64: return f(std::integral_constant<int, 64>{});
    case 128: return f(std::integral_constant<int, 128>{});
    default: return set_error("no RK4 epilogue for %d-point lines", L);
    }
}

bool rk4_fusable(const ihg_ctx *c)
{
    if (!c->p.enable_gw) return true;
    const int L = c->Ny;
    return !c->p.gw_fp32 && (L == 16 || L == 32 || L == 64 || L == 128);
}

// ---------------------------------------------------------------------------
// launchers
// ---------------------------------------------------------------------------

static LineSet x_lineset(const ihg_ctx *c)
{
    const long plane = (long)c->Ny * c->Mz;
    return LineSet{plane, plane, 0, plane};
}

// The x and y gradients go to grad3 where the FP64 GW source keeps them; else
// to W + 3M and W + 4M, which nothing else uses during the z pass (the FP32
// source components fill less than the first half of W).  The filtered
// fluctuations of phi are in W + 5M, past the filter's four spectra and the
// five FP64 source components.
DerivIO deriv_io(const ihg_ctx *c, const double *f, int filtered, int nr)
{
    auto at = [&](int k) { return reinterpret_cast<double *>(c->W + k * c->M); };
    const bool many = nr > 1;
    const long rw = many ? 2 * c->ens.w : 0;
    DerivIO io{f, nullptr, nullptr, nullptr, many ? c->ens.f : 0, 0, rw};
    if (filtered) {
        io.phi = at(5);
        io.rphi = rw;
        io.dc = c->dscal + S_FILTER_DC;
        io.rdc = many ? c->ens.s : 0;
    }
    if (c->p.enable_gw && !c->p.gw_fp32) {
        io.gx = c->grad3;
        io.gy = c->grad3 + c->N;
        io.rxy = many ? c->ens.g : 0;
    } else {
        io.gx = at(3);
        io.gy = at(4);
    }
    return io;
}

// x and y derivative passes (pairs of z neighbours as complex values); the
// second derivatives go to result[N..2N) (x) and result[2N..3N) (y)
DerivXY deriv_axes(const ihg_ctx *c, const DerivIO &io, double *result, int nr)
{
    const long nzp = c->Nz / 2, plane = (long)c->Ny * nzp;
    const long rl = nr > 1 ? c->ens.f / 2 : 0;
    auto d2 = [](double *p) { return reinterpret_cast<double2 *>(p); };
    const double2 *phi = reinterpret_cast<const double2 *>(io.phi);
    DerivXY d;
    d.a[0] = DerivAxis{LineSet{plane, plane, 0, plane}, phi, d2(io.gx),
                       d2(result + c->N), c->kg.kx1 / c->Nx, c->kg.kx2 / c->Nx,
                       io.rphi / 2, rl, io.rxy / 2};
    d.a[1] = DerivAxis{LineSet{c->Nx * nzp, nzp, plane, nzp}, phi, d2(io.gy),
                       d2(result + 2 * c->N), c->kg.ky1 / c->Ny,
                       c->kg.ky2 / c->Ny, io.rphi / 2, rl, io.rxy / 2};
    return d;
}

FilterFac filter_fac(const ihg_ctx *c, int output, int nr)
{
    return FilterFac{c->filter, (long)c->Ny * c->Mz, c->Nx, c->Ny, c->Mz,
                     (double)c->N, output ? c->Wc : nullptr,
                     output ? c->Wc + c->M : nullptr, c->dscal + S_FILTER_DC,
                     nr > 1 ? c->ens.s : 0};
}

ZShift filter_shift(const ihg_ctx *c, int nr)
{
    ZShift z;
    z.dc = c->dscal + S_FILTER_DC;
    z.fl = reinterpret_cast<double *>(c->W + 5 * c->M);
    z.rdc = nr > 1 ? c->ens.s : 0;
    z.rfl = nr > 1 ? 2 * c->ens.w : 0;
    return z;
}

// Work-group size of the derivative and z passes: single wavefronts while
// 256 lanes a work-group would leave CUs idle.  Whole right-hand sides, 64 and
// 256 lanes in one of the passes (in brackets its work-groups of 256 lanes):
// derivatives 8 x 32^3 (256) 18.7 and 20.7 us, 64^3 (128) 19.5 and 20.8, 3 x
// 64^3 (384) 33.4 and 33.3, 4 x 64^3 (512) 42.5 and 41.3, 128^3 (1024) 74.2 and
// 70.7; z pass with GW 64^3 (128) 42.1 and 46.6, 128 x 64 x 128 (512) 104.6 and
// 104.5, without GW 128^3 (1024) 73.0 and 70.2.  (In the z pass lines of 16 and
// 32 points are faster with 64 lanes beyond the limit too: 48 x 32^3 (768) 139
// and 153 us, 256 x 256 x 16 (512) 109 and 132; the rule makes no difference
// between lengths.)
static int small_wg(long blocks256) { return blocks256 < 512 ? 64 : 256; }

template <int L, int WG>
static int launch_deriv(ihg_ctx *c, const DerivXY &d, int naxes, int nr)
{
    using P = typename DerivPlan<L>::P;
    constexpr int B = WG / (L / P::E);
    const long nl = naxes == 2 ? std::max(d.a[0].ls.nlines, d.a[1].ls.nlines)
                               : d.a[0].ls.nlines;
    const dim3 grid((unsigned)((nl + B - 1) / B), naxes, nr);
    hipLaunchKernelGGL((k_deriv<L, P, WG>), grid, dim3(WG), 0, c->stream, d,
                       c->tw);
    return hip_check(hipGetLastError(), "k_deriv");
}

static int deriv_pass(ihg_ctx *c, int len, const DerivXY &d, int naxes, int nr)
{
    return dispatch_len(len, [&](auto Lc) {
        constexpr int L = decltype(Lc)::value;
        using P = typename DerivPlan<L>::P;
        constexpr int WG = DerivPlan<L>::WG, B = WG / (L / P::E);
        return timed(c, F_DERIV, 24.0 * c->N * naxes * nr, [&]() {
            if constexpr (L / P::E <= 64)
                if (small_wg((d.a[0].ls.nlines + B - 1) / B * naxes * nr) == 64)
                    return launch_deriv<L, 64>(c, d, naxes, nr);
            return launch_deriv<L, WG>(c, d, naxes, nr);
        });
    });
}

// CUs of the chip: a work-group of the z pass with helper wavefronts fills one
constexpr unsigned NUM_CU = 256;

template <class C>
static int z_pass(ihg_ctx *c, const double *f, double *result, int output,
                  const DerivIO &io, int nr, int &nparts)
{
    const bool gw = c->p.enable_gw != 0;
    ZRhsArgs<C> a = z_rhs_args<C>(c, f, result, io, nr);
    if (output) {
        a.rho = c->rho;
        a.pressure = c->pressure;
    }
    return dispatch_len(c->Nz, [&](auto Lc) {
        constexpr int L = decltype(Lc)::value;
        const unsigned nb = z_rhs_blocks<L>(a.nrows, 256);
        const int wg = small_wg((long)nb * nr);
        const dim3 grid(wg == 64 ? z_rhs_blocks<L>(a.nrows, 64) : nb, 1, nr);
        nparts = (int)grid.x * (wg / 64);
        if (2L * nparts > c->npartials)
            return set_error("partials buffer too small");
        // phi, dphi, psi, two gradients, two second derivatives in; A, p
        // (rho and p on output calls, gradients and sources with GW) out
        const double rs = sizeof(typename CT<C>::R);
        const double bytes =
            (8.0 * c->N * (9 + (output ? 2 : 0)) +
             (gw ? (rs == 4 ? 3.0 : 1.0) * rs * c->N + GW_NC * sizeof(C) * c->M : 0.0)) * nr;
        return timed(c, F_Z_RHS, bytes, [&]() {
            auto go = [&](auto gwc) {
                constexpr bool G = decltype(gwc)::value;
                auto small = [&](auto wgc) {
                    constexpr int WG = decltype(wgc)::value;
                    hipLaunchKernelGGL((k_z_rhs<L, G, C, WG, (WG > 64)>), grid,
                                       dim3(WG), 0, c->stream, a);
                };
                // Helper wavefronts while the work-groups, two wavefronts a
                // SIMD at their registers, run all at once: five up to a
                // work-group a CU (7 x 16^3 11.0 -> 7.7 us, 3 x 32^3 13.5 ->
                // 9.8), three up to two (64^3, 512 work-groups: 15.4 -> 12.6;
                // with five 15.7), none beyond (64 x 256 x 32, 1024: 18 us,
                // with five 28).
                if (wg == 64 && G && grid.x * nr <= NUM_CU)
                    small(std::integral_constant<int, G ? 64 * GW_NC : 64>{});
                else if (wg == 64 && G && grid.x * nr <= 2 * NUM_CU)
                    small(std::integral_constant<int, G ? 192 : 64>{});
                else if (wg == 64)
                    small(std::integral_constant<int, 64>{});
                else
                    hipLaunchKernelGGL((k_z_rhs<L, G, C, 256>), grid, dim3(256), 0, c->stream, a);
            };
            if (gw)
                go(std::true_type{});
            else if constexpr (sizeof(typename CT<C>::R) == 8)
                go(std::false_type{});
            return hip_check(hipGetLastError(), "k_z_rhs");
        });
    });
}

int rhs_core(ihg_ctx *c, double *f, double *result, int output, int filtered,
             int nr, const Rk4Ep *ep)
{
    const long N = c->N;
    const Ens e = nr > 1 ? c->ens : Ens{};
    const DerivIO io = deriv_io(c, f, filtered, nr);
    const DerivXY d = deriv_axes(c, io, result, nr);
    if (c->Nx == c->Ny) {
        IHG_TRY(deriv_pass(c, c->Nx, d, 2, nr));
    } else {
        IHG_TRY(deriv_pass(c, c->Nx, d, 1, nr));
        IHG_TRY(deriv_pass(c, c->Ny, DerivXY{{d.a[1], d.a[0]}}, 1, nr));
    }
    int nparts = 0;
    if (c->p.enable_gw && c->p.gw_fp32)
        IHG_TRY(z_pass<float2>(c, f, result, output, io, nr, nparts));
    else
        IHG_TRY(z_pass<double2>(c, f, result, output, io, nr, nparts));
    // the epilogue reads y (and k1..k3) and writes the stage output beside
    // the slope: 2 (stage) or 4 (final, no slope written) more blocks
    const double ep_blocks = !ep ? 0.0 : (ep->mode == RK4_FINAL ? 4.0 : 8.0);
    // one pair of points a thread on small grids (32^3 with the epilogue 5.1
    // against 5.9 us, 7 x 16^3 + 3 x 32^3 5.9 and 6.8), two on larger ones
    // (64^3 6.2 against 7.0 us: the work-groups' sums count).  Near the limit
    // either choice is within 3 % of a right-hand side (131 to 197 k points:
    // without the epilogue two pairs gain up to 0.4 us from 164 k on and lose
    // up to 1 us at 131 k; with it one pair gains 0.2 to 1.7 us).
    const bool small = N * nr < 200000;
    const dim3 ugrid(nblocks(N, small ? RED_WG * 2 : RED_WG * 4, 65536), 1, nr);
    // One launch where the partial sums are few (64^3 has 512): 4.6 us against
    // 3.6 + 3.0 at 16^3, 6.3 against 4.4 + 5.2 at 64^3; every work-group then
    // reads all of them (at most 16 KB, from L2).
    if (nparts <= MEANS_WG && 4.0 * 8.0 * (double)N * nr < NT_BYTES)
        return timed(c, F_UPDATE, (9.0 + ep_blocks) * 8.0 * N * nr, [&]() {
            if (ep)
                hipLaunchKernelGGL((small ? k_means_update<true, true>
                                          : k_means_update<true, false>),
                                   ugrid, dim3(RED_WG), 0,
                                   c->stream, c->partials, nparts, N, f, result,
                                   c->Ntot, c->dscal, e, *ep);
            else
                hipLaunchKernelGGL((k_means_update<false, false>), ugrid, dim3(RED_WG), 0,
                                   c->stream, c->partials, nparts, N, f, result,
                                   c->Ntot, c->dscal, e, Rk4Ep{});
            return hip_check(hipGetLastError(), "k_means_update");
        });
    IHG_TRY(timed(c, F_MEANS, 16.0 * nparts * nr, [&]() {
        if (ep)
            hipLaunchKernelGGL(k_means_rk4, dim3(nr), dim3(MEANS_WG), 0,
                               c->stream, c->partials, nparts, N, f, result,
                               c->Ntot, c->dscal, e, *ep);
        else
            hipLaunchKernelGGL(k_means, dim3(nr), dim3(MEANS_WG), 0, c->stream,
                               c->partials, nparts, N, f, result, c->Ntot,
                               c->dscal, e);
        return hip_check(hipGetLastError(), "k_means");
    }));
    return timed(c, F_UPDATE, (9.0 + ep_blocks) * 8.0 * N * nr, [&]() {
        // the streaming hint when the four blocks of all realizations
        // outgrow the caches
        const bool nt = 4.0 * 8.0 * (double)N * nr >= NT_BYTES;
        if (ep)
            hipLaunchKernelGGL((nt ? k_update_phi_psi_rk4<true>
                                   : k_update_phi_psi_rk4<false>),
                               ugrid, dim3(RED_WG), 0, c->stream, f, result, N,
                               c->dscal, e, *ep);
        else
            hipLaunchKernelGGL((nt ? k_update_phi_psi<true>
                                   : k_update_phi_psi<false>),
                               ugrid, dim3(RED_WG), 0, c->stream, f, result, N,
                               c->dscal, e);
        return hip_check(hipGetLastError(), "k_update_phi_psi");
    });
}

// Whether the TT pass transforms the components side by side: up to about two
// 64^3 grids.  Measured side by side and in turn: 7 x 16^3 6.2 and 13.3 us, 3
// x 32^3 7.4 and 16.3, 64^3 (135 k modes) 12.0 and 13.1, 48 x 32^3 (836 k) 181
// and 157, 128^3 (1.06 M) 71.8 and 68.9, 4 x 128^3 467 and 432 us.  Near the
// limit, whole right-hand sides: 17 x 32^3 (296 k) 61.0 and 64.4, 130 x 16^3
// (300 k) 59.0 and 59.4, 512 x 64 x 16 (295 k) 78.1 and 81.3, 128 x 64 x 64 (270
// k) 65.8 and 66.7, 3 x 64^3 (406 k) 75.6 and 72.5.
// Lines of 128 points: a work-group takes 87 KB of LDS, one a CU, so the pass
// must fit in one round: 32 x 128 x 32 (68 work-groups) 42.1 and 45.7, 3 x 64 x
// 128 x 16 (216) 57.3 and 61.8, 32 x 128 x 128 (260) 75.0 and 69.3, 128 x 128 x
// 32 (272) 70.4 and 65.4.
static bool tt_wide(const ihg_ctx *c, int nr)
{
    if (c->Ny > TT_WIDE_MAX || c->M * nr >= 300000) return false;
    constexpr int B = TTWide<128>::B;
    const long lines = (long)c->Nx * c->Mz;
    return c->Ny < 128 || (lines + B - 1) / B * nr <= NUM_CU;
}

// GW source pipeline on complex type C after the z pass: x pass, fused y
// pass + TT + update_h.  Wk holds 6 M values of C; realization r of an
// ensemble finds them r * rw further on.
template <class C>
static int rhs_gw_t(ihg_ctx *c, C *Wk, const C *tw, const double *f,
                    double *result, int nr, long rw, const Rk4Ep *ep)
{
    const long N = c->N, M = c->M;
    const double cs = sizeof(C);
    const Ens e = nr > 1 ? c->ens : Ens{};
    if constexpr (std::is_same<C, float2>::value)
        IHG_TRY(x_pass_f32(c, Wk, -1, GW_NC, M, nr, rw));
    else
        IHG_TRY(x_pass(c, Wk, -1, GW_NC, M, nr, rw));
    // y pass of the sources, TT projection and update_h: the sources
    // and h1, h2, dh1, dh2 in; the four h blocks of result out
    const LineSet ls{(long)c->Nx * c->Mz, c->Mz, (long)c->Ny * c->Mz, c->Mz};
    const double epb = !ep ? 0.0 : (ep->mode == RK4_FINAL ? 8.0 : 16.0);
    const double bytes = (GW_NC * cs + (8.0 + epb) * 16.0) * M * nr;
    if (tt_wide(c, nr))
        return dispatch_len(c->Ny, [&](auto Lc) {
            constexpr int L = decltype(Lc)::value;
            if constexpr (L <= TT_WIDE_MAX) {
                using TT = TTWide<L>;
                const dim3 grid((unsigned)((ls.nlines + TT::B - 1) / TT::B), 1, nr);
                // the RK4 epilogue where rk4_fusable has it
                constexpr bool EP = std::is_same<C, double2>::value && L >= 16;
                if (ep && !EP)
                    return set_error("no RK4 epilogue for this TT pass");
                return timed(c, F_TT_UPDATE_H, bytes, [&]() {
                    if (ep)
                        hipLaunchKernelGGL((k_y_tt_wide<L, C, EP>), grid,
                                           dim3(TT::WG), 0, c->stream, Wk, M, f,
                                           result, N, c->Next, c->Ntot, c->kg,
                                           c->dscal, ls, tw, e, rw,
                                           gw_axis(c->kg), *ep);
                    else
                        hipLaunchKernelGGL((k_y_tt_wide<L, C, false>), grid,
                                           dim3(TT::WG), 0, c->stream, Wk, M, f,
                                           result, N, c->Next, c->Ntot, c->kg,
                                           c->dscal, ls, tw, e, rw,
                                           gw_axis(c->kg), Rk4Ep{});
                    return hip_check(hipGetLastError(), "k_y_tt_wide");
                });
            } else {
                return set_error("no wide TT pass for %d points", L);
            }
        });
    if constexpr (std::is_same<C, double2>::value) {
        if (ep)
            return dispatch_rk4_len(c->Ny, [&](auto Lc) {
                constexpr int L = decltype(Lc)::value;
                using TP = TTPlan<L>;
                constexpr int B = TP::WG / (L / TP::P::E);
                const unsigned nb = (unsigned)((ls.nlines + B - 1) / B);
                return timed(c, F_TT_UPDATE_H, bytes, [&]() {
                    hipLaunchKernelGGL((k_y_tt_update_h_rk4<L, TP::WG, typename TP::P>),
                                       dim3(nb, 1, nr), dim3(TP::WG), 0, c->stream, Wk,
                                       M, f, result, N, c->Next, c->Ntot, c->kg,
                                       c->dscal, ls, tw, e, rw, gw_axis(c->kg), *ep);
                    return hip_check(hipGetLastError(), "k_y_tt_update_h_rk4");
                });
            });
    } else if (ep) {
        return set_error("no RK4 epilogue for the FP32 GW source");
    }
    return dispatch_len(c->Ny, [&](auto Lc) {
        constexpr int L = decltype(Lc)::value;
        using TP = TTPlan<L>;
        constexpr int B = TP::WG / (L / TP::P::E);
        const unsigned nb = (unsigned)((ls.nlines + B - 1) / B);
        return timed(c, F_TT_UPDATE_H, bytes, [&]() {
            hipLaunchKernelGGL((k_y_tt_update_h<L, TP::WG, typename TP::P, C>),
                               dim3(nb, 1, nr), dim3(TP::WG), 0, c->stream, Wk,
                               M, f, result, N, c->Next, c->Ntot, c->kg,
                               c->dscal, ls, tw, e, rw, gw_axis(c->kg));
            return hip_check(hipGetLastError(), "k_y_tt_update_h");
        });
    });
}

int rhs_gw(ihg_ctx *c, const double *f, double *result, int nr,
           const Rk4Ep *ep)
{
    const long rw = nr > 1 ? c->ens.w : 0;
    if (c->p.gw_fp32)
        // FP32 values in the FP64 buffer, realizations at the same addresses
        return rhs_gw_t<float2>(c, reinterpret_cast<float2 *>(c->W), c->twf, f,
                                result, nr, 2 * rw, ep);
    return rhs_gw_t<double2>(c, c->W, c->tw, f, result, nr, rw, ep);
}

// mk_ffts_and_filter's filter branch (src/toolbox.c:164-171): phi, dphi,
// psi, dpsi (contiguous in f) filtered in place, all four in one batch.  An
// output call keeps the filtered spectra of phi (Wc) and psi (Wc + M); the
// fluctuations of the filtered phi stay in W + 5M for rhs_core.
int rhs_filter(ihg_ctx *c, double *f, int output, int nr)
{
    const long N = c->N, M = c->M;
    double2 *W = c->W;
    const Ens e = nr > 1 ? c->ens : Ens{};
    IHG_TRY(z_r2c_pass(c, f, W, 4, N, M, nr, e.f, e.w));
    IHG_TRY(y_pass(c, W, -1, 4, M, nr, e.w));
    IHG_TRY(dispatch_len(c->Nx, [&](auto Lc) {
        constexpr int L = decltype(Lc)::value;
        constexpr int WG = RoundtripWG<L>::WG;
        using SS = StridedShape<L, Plan<L>, WG>;
        const LineSet ls = x_lineset(c);
        const FilterFac fac = filter_fac(c, output, nr);
        return timed(c, F_X_ROUNDTRIP, (output ? 10.0 : 8.0) * 16.0 * M * nr, [&]() {
            hipLaunchKernelGGL((k_x_roundtrip<L, FilterFac, Plan<L>, WG>),
                               dim3((unsigned)((ls.nlines + SS::B - 1) / SS::B), 4, nr),
                               dim3(WG), 0, c->stream, W, ls, M, c->tw, fac, e.w);
            return hip_check(hipGetLastError(), "k_x_roundtrip");
        });
    }));
    IHG_TRY(y_pass(c, W, +1, 4, M, nr, e.w));
    const ZShift sh = filter_shift(c, nr);
    return z_c2r_pass(c, W, f, 4, M, N, nr, e.w, e.f, &sh);
}

} // namespace ihg
