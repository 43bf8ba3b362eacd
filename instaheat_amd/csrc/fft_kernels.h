// fft_kernels.h -- FFT pass kernels for the 3D r2c / c2r transforms.
//
// Layout (FFTW r2c_3d, the state layout of the reference): a real field is
// double[Nx][Ny][Nz] with z fastest; its half spectrum is
// complex[Nx][Ny][Nz/2+1].  A 3D r2c is a z pass (real rows -> half rows),
// then a y pass and an x pass on the half spectrum; c2r is the mirror.
//
// z passes transform two real rows at once as one complex row (real part one
// row, imaginary part the other) and split / merge the two Hermitian halves
// in LDS.  y and x passes are strided: a work-group owns B neighbouring lines,
// so every global access is a run of B consecutive complex values.
#pragma once

#include "fft_core.h"
#include "mem.h"

namespace ihg {

constexpr int FFT_WG = 256;

// Line plans of the z passes.  Their transposes are wavefront-local, so an
// extra stage costs LDS traffic but no work-group barrier, and fewer values
// per thread buy occupancy: at most 8 values per thread.  The short lines
// take 2 or 4, so that a small grid spreads over more lanes.
template <int L> struct ZPlanOf { using P = Plan<L>; };
template <> struct ZPlanOf<4> { using P = PlanT<2, 2, 2>; };
template <> struct ZPlanOf<8> { using P = PlanT<4, 4, 2>; };
template <> struct ZPlanOf<16> { using P = PlanT<4, 4, 4>; };
template <> struct ZPlanOf<256> { using P = PlanT<8, 8, 8, 4>; };
template <> struct ZPlanOf<512> { using P = PlanT<8, 8, 8, 8>; };

// Tile of a z pass: B lines of L points per work-group, T threads per line
template <int L>
struct Tile {
    using P = typename ZPlanOf<L>::P;
    static constexpr int E = P::E;
    static constexpr int T = L / E;
    static constexpr int B = FFT_WG / T;
    static constexpr int PITCH = Lds<L>::PITCH;
    // lines per wavefront (a line's T threads are consecutive lanes), so
    // each wavefront owns LPW lines and finishes them alone
    static constexpr int LPW = 64 / T;
};

// Geometry of a set of strided lines: line l starts at
// (l / inner) * outer_stride + (l % inner) and its points are `stride` apart.
struct LineSet {
    long nlines, inner, outer_stride, stride;
    __device__ __forceinline__ long base(long l) const
    {
        return (l / inner) * outer_stride + (l % inner);
    }
};

// Work-group coordinates of one pass: a standalone launch takes them from
// the hardware (hw_blk), a grouped launch -- passes of several grid sizes in
// one launch -- from its segment table.  gx is the number of tiles along x.
struct Blk {
    unsigned x, y, z, gx;
};

__device__ __forceinline__ Blk hw_blk()
{
    return Blk{blockIdx.x, blockIdx.y, blockIdx.z, gridDim.x};
}

// Tile index of a work-group along x.  The dispatcher hands work-groups to
// the eight XCDs in turn (work-group w to XCD w mod 8, w the linear
// work-group id; w and w + 8 land on one XCD whatever the other grid
// dimensions are), and every XCD has its own L2.  Strided tiles that are
// neighbours share a 128-byte line at their edges (the half-spectrum rows of
// Nz/2 + 1 complex values start off line boundaries), so with SWZ each XCD
// gets one contiguous run of tiles: XCD x takes tiles
// x*q + min(x, r) + [0, q + (x < r)), q = gx / 8, r = gx mod 8, in order.
// The map is a bijection of [0, gx).
template <bool SWZ>
__device__ __forceinline__ unsigned tile_x(const Blk &bk)
{
    if constexpr (!SWZ) {
        return bk.x;
    } else {
        const unsigned gx = bk.gx, bx = bk.x;
        const unsigned q = gx / 8, r = gx % 8, x = bx % 8;
        return x * q + (x < r ? x : r) + bx / 8;
    }
}

// ---------------------------------------------------------------------------
// strided complex-to-complex pass (y or x), in place or out of place,
// batched over blockIdx.y (arrays `batch` complex values apart).
// Lanes run fastest over the B lines of the tile, so for a fixed point n a
// wavefront touches B consecutive complex values.  The first Stockham stage
// loads straight from HBM into registers and the last stage stores straight
// from registers; only the transposes between stages go through LDS.
// ---------------------------------------------------------------------------
// The line plan P and the work-group size WG are template parameters so
// that an autotuner can pick them per line length (B = WG / (L / P::E)
// lines per work-group).
template <int L, class P = Plan<L>, int WG = FFT_WG>
struct StridedShape {
    static constexpr int B = WG / (L / P::E), PITCH = Lds<L>::PITCH;
    static constexpr int LDS = B * PITCH; // complex values of LDS
};

template <int L, int DIR, class C = double2, class P = Plan<L>,
          int WG = FFT_WG, bool SWZ = true>
__device__ __forceinline__ void c2c_strided_body(
    const Blk &bk, C *lds, const C *in, C *out, LineSet ls, long batch,
    const C *__restrict__ tw, long rr)
{
    constexpr int B = StridedShape<L, P, WG>::B, PITCH = Lds<L>::PITCH;
    const int tid = threadIdx.x;
    in += bk.y * batch + bk.z * rr;
    out += bk.y * batch + bk.z * rr;
    const int b = tid % B, j = tid / B;
    const long line = (long)tile_x<SWZ>(bk) * B + b;
    const bool act = line < ls.nlines;
    const long base = ls.base(act ? line : 0);
    const C *src = in + base;
    C *dst = out + base;
    const long st = ls.stride;
    auto rd = [&](int, int n) {
        const C v = ldn(src + n * st); // in bounds for every lane
        return act ? v : CT<C>::make(0, 0);
    };
    auto wr = [&](int, int n, C v) {
        if (act) stn(dst + n * st, v);
    };
    fft_line<L, DIR, true, true, P>(lds + b * PITCH, j, tw, rd, wr);
}

template <int L, int DIR, class C = double2, class P = Plan<L>,
          int WG = FFT_WG, bool SWZ = true>
__global__ __launch_bounds__(WG) void k_c2c_strided(
    const C *in, C *out, LineSet ls, long batch, const C *__restrict__ tw,
    long rr)
{
    __shared__ C lds[StridedShape<L, P, WG>::LDS];
    c2c_strided_body<L, DIR, C, P, WG, SWZ>(hw_blk(), lds, in, out, ls, batch,
                                            tw, rr);
}

// Candidate (plan, work-group size) pairs of the strided pass per line
// length; entry 0 is the default.  The autotuner times them on the
// context's own arrays and keeps the fastest.
template <class P_, int WG_, bool SWZ_ = true> struct StridedCand {
    using P = P_;
    static constexpr int WG = WG_;
    static constexpr bool SWZ = SWZ_;
};
template <class... Cs> struct CandList {
    static constexpr int n = sizeof...(Cs);
};
template <int L> struct StridedCands {
    using type = CandList<StridedCand<Plan<L>, 256>, StridedCand<Plan<L>, 256, false>>;
    static constexpr int x_default = 0;
};
template <> struct StridedCands<16> {
    using type = CandList<StridedCand<Plan<16>, 256>, StridedCand<Plan<16>, 256, false>,
                          StridedCand<PlanT<4, 4, 4>, 256>, StridedCand<Plan<16>, 128>>;
    static constexpr int x_default = 0;
};
template <> struct StridedCands<32> {
    using type = CandList<StridedCand<Plan<32>, 256>, StridedCand<Plan<32>, 256, false>,
                          StridedCand<PlanT<16, 16, 2>, 256>,
                          StridedCand<PlanT<4, 4, 4, 2>, 256>, StridedCand<Plan<32>, 128>>;
    static constexpr int x_default = 0;
};
template <> struct StridedCands<64> {
    using type = CandList<StridedCand<Plan<64>, 256>, StridedCand<Plan<64>, 256, false>,
                          StridedCand<PlanT<16, 16, 4>, 256>,
                          StridedCand<PlanT<4, 4, 4, 4>, 256>, StridedCand<Plan<64>, 128>>;
    static constexpr int x_default = 0;
};
template <> struct StridedCands<128> {
    using type = CandList<StridedCand<Plan<128>, 256>, StridedCand<Plan<128>, 256, false>,
                          StridedCand<PlanT<16, 16, 8>, 256>,
                          StridedCand<PlanT<4, 4, 4, 4, 2>, 256>, StridedCand<Plan<128>, 128>>;
    static constexpr int x_default = 0;
};
// 256-point x lines (points a whole y-z plane apart) run fastest with 32
// lines per work-group (512 B contiguous per point); y lines with 16.
template <> struct StridedCands<256> {
    using type = CandList<StridedCand<Plan<256>, 256>, StridedCand<Plan<256>, 256, false>,
                          StridedCand<Plan<256>, 512>, StridedCand<PlanT<8, 8, 8, 4>, 512>,
                          StridedCand<PlanT<4, 4, 4, 4, 4>, 512, false>>;
    static constexpr int x_default = 2;
};

// f(StridedCand<...>{}) for candidate `id` of a list (the default for an id
// out of range)
template <class F, class C0, class... Cs>
auto with_cand(int id, CandList<C0, Cs...>, F &&f)
{
    if constexpr (sizeof...(Cs) == 0) {
        return f(C0{});
    } else {
        if (id <= 0) return f(C0{});
        return with_cand(id - 1, CandList<Cs...>{}, f);
    }
}

// ---------------------------------------------------------------------------
// x-axis forward transform, a factor fac(bk, line, kx_index, value) and the
// backward transform, in place: the filter round trip, batched over
// blockIdx.y with arrays `batch` apart, realizations of an ensemble over
// blockIdx.z, `rr` apart.  The spectrum never leaves registers: the forward
// transform's last stage keeps its outputs, and the backward transform's
// first stage takes them through chain_slot; HBM is read and written once.
// ---------------------------------------------------------------------------
template <int L, class Fac, class P = Plan<L>, int WG = FFT_WG>
__device__ __forceinline__ void x_roundtrip_body(
    const Blk &bk, double2 *lds, double2 *data, LineSet ls, long batch,
    const double2 *__restrict__ tw, Fac fac, long rr)
{
    constexpr int E = P::E, B = StridedShape<L, P, WG>::B, PITCH = Lds<L>::PITCH;
    const int tid = threadIdx.x;
    data += bk.y * batch + bk.z * rr;
    const int b = tid % B, j = tid / B;
    const long line = (long)tile_x<true>(bk) * B + b;
    const bool act = line < ls.nlines;
    double2 *dst = data + ls.base(act ? line : 0);
    const long st = ls.stride;
    double2 *my = lds + b * PITCH;
    double2 spec[E];
    auto rd = [&](int, int n) {
        const double2 v = ldn(dst + n * st); // in bounds for every lane
        return act ? v : make_double2(0.0, 0.0);
    };
    auto keep = [&](int slot, int, double2 v) { spec[slot] = v; };
    fft_line<L, -1, true, true, P>(my, j, tw, rd, keep);
    lds_barrier(); // LDS reads of the forward transform are done
    auto rq = [&](int slot, int n) {
        return fac(bk, line, n, spec[chain_slot<L, P>(slot)]);
    };
    auto wq = [&](int, int n, double2 v) {
        if (act) stn(dst + n * st, v);
    };
    fft_line<L, +1, true, true, P>(my, j, tw, rq, wq);
}

// Work-group size of the round trip per line length.  Measured with 128, 256
// and 512 lanes: one 32^3 grid 5.1, 5.6, 7.3 us (9 work-groups at 256 leave
// the chip idle), 64^3 11.3, 11.5, 12.2, 128^3 38.8, 39.3, 55.5, 256^3 423,
// 343, 348 (128-byte runs at 128 lanes).
template <int L> struct RoundtripWG { static constexpr int WG = L <= 64 ? 128 : 256; };

template <int L, class Fac, class P = Plan<L>, int WG = FFT_WG>
__global__ __launch_bounds__(WG) void k_x_roundtrip(
    double2 *data, LineSet ls, long batch, const double2 *__restrict__ tw,
    Fac fac, long rr)
{
    __shared__ double2 lds[StridedShape<L, P, WG>::LDS];
    x_roundtrip_body<L, Fac, P, WG>(hw_blk(), lds, data, ls, batch, tw, fac, rr);
}

// ---------------------------------------------------------------------------
// Spectral derivatives along x or y: of every line of the real field phi the
// forward transform, times i k / L and -k^2 / L, and two backward transforms
// (the gradient component g, its Nyquist mode dropped, and the axis' part
// lap of the Laplacian).  A derivative along one axis needs no transform
// along the others: its multiplier depends on that axis' wave number alone,
// and |k|^2 is the sum of the three squares (src/toolbox.c:132-139).  The
// operators are real, so a line of neighbouring pairs (z, z + 1) is
// transformed as one complex line u + i v and gives (Du, Dv) with no
// Hermitian split: phi is read and g and lap are written in whole 16-byte
// pairs, aligned rows.  Geometry: `ls` in units of pairs.  The value phi[0]
// of the grid's first point is subtracted before the transform (its
// derivatives vanish): phi is a mean of order 1 with fluctuations of 1e-6 to
// 1e-2, and every line's transform would round at the size of the mean.  The
// difference of nearby numbers is exact.  (After the filter the derivatives
// are those of the filtered field before the mean is added and rounded in,
// FilterFac.)
// The bound is HBM traffic, 3 fields of 8 N bytes an axis: both axes at 256^3
// take 171 us (4.7 TB/s).  The z r2c, y and x fan-out passes of the derivatives
// through the 3D spectrum, which this replaces, took 307 us.  256-point lines:
// 16 values a thread in two stages with 296 registers (one wave a SIMD) 171
// us, 8 values in three stages 183, 16 values held to 256 registers 204, 512
// lanes a work-group 215.
// ---------------------------------------------------------------------------
struct DerivAxis {
    LineSet ls;
    const double2 *phi;
    double2 *g, *lap;
    double k1, k2;    // 2 pi / (L length), (2 pi / length)^2 / L
    long rp, rl, rg;  // realization strides of phi, lap, g (pairs)
};

template <int L, class P, int WG>
__device__ __forceinline__ void deriv_body(const Blk &bk, double2 *lds,
                                           const DerivAxis &a,
                                           const double2 *__restrict__ tw)
{
    constexpr int E = P::E, B = StridedShape<L, P, WG>::B, PITCH = Lds<L>::PITCH;
    const int tid = threadIdx.x;
    const int b = tid % B, j = tid / B;
    const long line = (long)bk.x * B + b;
    const bool act = line < a.ls.nlines;
    const long base = a.ls.base(act ? line : 0);
    const double2 *src = a.phi + bk.z * a.rp + base;
    double2 *gd = a.g + bk.z * a.rg + base, *ld = a.lap + bk.z * a.rl + base;
    const long st = a.ls.stride;
    double2 *my = lds + b * PITCH;
    double2 spec[E];
    const double phi0 = a.phi[bk.z * a.rp].x;
    // idle lanes transform line 0 (in bounds) and store nothing
    auto rd = [&](int, int n) {
        const double2 v = src[n * st];
        return make_double2(v.x - phi0, v.y - phi0);
    };
    auto keep = [&](int slot, int, double2 v) { spec[slot] = v; };
    fft_line<L, -1, true, true, P>(my, j, tw, rd, keep);
    lds_barrier(); // LDS reads of the forward transform are done
    auto rl = [&](int slot, int n) {
        const double2 v = spec[chain_slot<L, P>(slot)];
        const double m = n > L / 2 ? L - n : n, k = -(a.k2 * m * m);
        return make_double2(v.x * k, v.y * k);
    };
    auto wl = [&](int, int n, double2 v) {
        if (act) ld[n * st] = v;
    };
    fft_line<L, +1, true, true, P>(my, j, tw, rl, wl);
    lds_barrier();
    auto rg = [&](int slot, int n) {
        const double2 v = spec[chain_slot<L, P>(slot)];
        const double k = n > L / 2 ? a.k1 * (n - L) : (2 * n == L ? 0.0 : a.k1 * n);
        return make_double2(-v.y * k, v.x * k);
    };
    auto wg = [&](int, int n, double2 v) {
        if (act) gd[n * st] = v;
    };
    fft_line<L, +1, true, true, P>(my, j, tw, rg, wg);
}

// Line plans and work-group sizes of the derivative passes.  (One 16^3 grid:
// 16 values a thread 4.6 us, 4 values 3.4; 32^3 8 values 4.4, 4 values 4.1; at
// 64 and 128 points the longer plans are the faster ones, 45 against 47 us for
// 16 x 64^3.)
template <int L> struct DerivPlan { using P = Plan<L>; static constexpr int WG = FFT_WG; };
template <> struct DerivPlan<16> { using P = PlanT<4, 4, 4>; static constexpr int WG = FFT_WG; };
template <> struct DerivPlan<32> { using P = PlanT<4, 4, 4, 2>; static constexpr int WG = FFT_WG; };

// both axes (of one length) in one launch: blockIdx.y picks the axis
struct DerivXY {
    DerivAxis a[2];
};

template <int L, class P, int WG>
__global__ __launch_bounds__(WG) void k_deriv(DerivXY d,
                                              const double2 *__restrict__ tw)
{
    __shared__ double2 lds[StridedShape<L, P, WG>::LDS];
    deriv_body<L, P, WG>(hw_blk(), lds, d.a[blockIdx.y], tw);
}

// ---------------------------------------------------------------------------
// z passes
// ---------------------------------------------------------------------------

// Hermitian split after a forward transform of Z = A + iB (A, B real rows):
// A[k] = (Z[k] + conj Z[L-k]) / 2, B[k] = -i (Z[k] - conj Z[L-k]) / 2.
template <int L, class C>
__device__ __forceinline__ C herm_split(const C *line, int k, int s)
{
    using R = typename CT<C>::R;
    const C z1 = line[Lds<L>::idx(k)];
    const C z2 = cconj(line[Lds<L>::idx((L - k) & (L - 1))]);
    const R h = (R)0.5;
    if (s == 0)
        return CT<C>::make(h * (z1.x + z2.x), h * (z1.y + z2.y));
    return CT<C>::make(h * (z1.y - z2.y), -h * (z1.x - z2.x));
}

// Merge of two half rows A, B (Hermitian extension, imaginary parts of the
// k = 0 and k = L/2 bins dropped) into Z[n] = A_ext[n] + i B_ext[n].
// Written without branches: the mirrored index and the sign / zeroing of the
// imaginary parts are selects, so no value the caller computes is left to
// divergent control flow.
template <int L>
__device__ __forceinline__ double2 herm_merge(const double2 *__restrict__ A,
                                              const double2 *__restrict__ Bv,
                                              int n)
{
    const bool upper = n > L / 2;
    const int m = upper ? L - n : n;
    const double2 a = A[m], bb = Bv[m];
    // imaginary parts of the k = 0 and k = L/2 bins are dropped; the upper
    // half uses the conjugates
    const double edge = (m == 0 || m == L / 2) ? 0.0 : 1.0;
    const double sg = upper ? -1.0 : 1.0;
    const double ai = sg * edge * a.y, bi = sg * edge * bb.y;
    return make_double2(a.x - bi, ai + bb.x);
}

// Real rows -> half rows.  Line l = rows (2l, 2l+1) of `in` (nrows rows of
// L reals, batched over y with `rbatch` / `cbatch` strides, realizations
// over z `rin` / `rout` apart).
template <int L>
__device__ __forceinline__ void z_r2c_body(
    const Blk &bk, double2 *lds, const double *in, double2 *out, long nrows,
    long rbatch, long cbatch, const double2 *__restrict__ tw, long rin,
    long rout)
{
    using TL = Tile<L>;
    constexpr int MZ = L / 2 + 1;
    const int tid = threadIdx.x;
    in += bk.y * rbatch + bk.z * rin;
    out += bk.y * cbatch + bk.z * rout;
    const long nlines = nrows / 2;
    const int bc = tid / TL::T;
    const long line = (long)bk.x * TL::B + bc;
    const bool act = line < nlines;
    const double *ra = in + (act ? 2 * line : 0) * L;
    auto rd = [&](int, int n) {
        const double u = ldn(ra + n), v = ldn(ra + L + n); // in bounds
        return act ? make_double2(u, v) : make_double2(0.0, 0.0);
    };
    fft_line_wave<L, -1, typename TL::P>(lds + bc * TL::PITCH, tid % TL::T, tw, rd);
    // each wavefront splits and stores the 2 LPW rows of its own lines
    const int w = tid / 64, lane = tid % 64;
    const long row0 = 2 * ((long)bk.x * TL::B + w * TL::LPW);
    const double2 *wl = lds + w * TL::LPW * TL::PITCH;
    for (int idx = lane; idx < 2 * TL::LPW * MZ; idx += 64) {
        const int r = idx / MZ, k = idx - r * MZ;
        if (row0 + r < nrows)
            stn(out + row0 * MZ + idx,
                herm_split<L>(wl + (r >> 1) * TL::PITCH, k, r & 1));
    }
}

template <int L>
__global__ __launch_bounds__(FFT_WG) void k_z_r2c(
    const double *in, double2 *out, long nrows, long rbatch, long cbatch,
    const double2 *__restrict__ tw, long rin, long rout)
{
    __shared__ double2 lds[Tile<L>::B * Tile<L>::PITCH];
    z_r2c_body<L>(hw_blk(), lds, in, out, nrows, rbatch, cbatch, tw, rin, rout);
}

// A constant kept out of the transform of array 0 of a batch: the c2r pass
// writes u + *dc to the output and u itself to fl (strides per realization).
struct ZShift {
    const double *dc = nullptr;
    double *fl = nullptr;
    long rdc = 0, rfl = 0;
};

// Half rows -> real rows (the c2r z pass).
template <int L>
__device__ __forceinline__ void z_c2r_body(
    const Blk &bk, double2 *lds, const double2 *in, double *out, long nrows,
    long cbatch, long rbatch, const double2 *__restrict__ tw, long rin,
    long rout, const ZShift &sh)
{
    using TL = Tile<L>;
    constexpr int MZ = L / 2 + 1;
    const int tid = threadIdx.x;
    in += bk.y * cbatch + bk.z * rin;
    out += bk.y * rbatch + bk.z * rout;
    const long nlines = nrows / 2;
    const int bc = tid / TL::T;
    const long line = (long)bk.x * TL::B + bc;
    const bool act = line < nlines;
    const double2 *A = in + (act ? 2 * line : 0) * MZ;
    auto rd = [&](int, int n) {
        const double2 z = herm_merge<L>(A, A + MZ, n); // in bounds for every lane
        return act ? z : make_double2(0.0, 0.0);
    };
    fft_line_wave<L, +1, typename TL::P>(lds + bc * TL::PITCH, tid % TL::T, tw, rd);
    // each wavefront stores the 2 LPW rows of its own lines
    const int w = tid / 64, lane = tid % 64;
    const long row0 = 2 * ((long)bk.x * TL::B + w * TL::LPW);
    const double2 *wl = lds + w * TL::LPW * TL::PITCH;
    double c = 0.0, *fl = nullptr;
    if (sh.dc && bk.y == 0) {
        c = sh.dc[bk.z * sh.rdc];
        fl = sh.fl + bk.z * sh.rfl;
    }
    for (int idx = lane; idx < 2 * TL::LPW * L; idx += 64) {
        const int r = idx / L, n = idx - r * L;
        if (row0 + r < nrows) {
            const double2 z = wl[(r >> 1) * TL::PITCH + Lds<L>::idx(n)];
            const double v = (r & 1) ? z.y : z.x;
            if (fl) fl[row0 * L + idx] = v;
            stn(out + row0 * L + idx, v + c);
        }
    }
}

template <int L>
__global__ __launch_bounds__(FFT_WG) void k_z_c2r(
    const double2 *in, double *out, long nrows, long cbatch, long rbatch,
    const double2 *__restrict__ tw, long rin, long rout, ZShift sh)
{
    __shared__ double2 lds[Tile<L>::B * Tile<L>::PITCH];
    z_c2r_body<L>(hw_blk(), lds, in, out, nrows, cbatch, rbatch, tw, rin, rout,
                  sh);
}

} // namespace ihg
