// demag.hip -- zero-padded Newell-tensor demag convolution on gfx950.
//
// Replaces the cuFFT pipeline of native/backends/fdm/src/demag_fp64.cu:264-381
// (pack, 3 forward Z2Z transforms over the fully padded grid, 6-component
// complex tensor multiply, 3 inverse transforms, unpack).  The mathematics is
// that of crates/fullmag-engine/src/lib.rs:2306-2400,
//     H = IFFT( -K . FFT(Ms m) ) / Npad   on a (2nx, 2ny, 2nz) grid,
// organised around what is non-zero and around coalesced HBM access:
//
//   x fwd  R2C of 16 real rows per workgroup (two rows per complex transform,
//          only nx of 2nx inputs loaded); the nx+1 outputs of each row are
//          written transposed, so ky runs are contiguous in the spectrum.
//   y fwd  contiguous lines, ny of 2ny inputs loaded (3-D only).
//   z conv per (kx, ky): 3 components x (nz inputs -> 2nz), 3x3 tensor,
//          inverse, nz outputs; in registers for 2nz <= 16 (3-D only).
//   y inv  contiguous lines, 2ny inputs, ny outputs written (3-D only).
//   x inv  C2R of 16 rows, reading transposed runs, nx outputs per row,
//          scaled by 1/Npad and masked.
// Thin films (nz = 1, 2-D spectra): x fwd, y conv (forward y, tensor at
// kz = 0, inverse y in one kernel), x inv.
//
// Spectrum layout: spec[c][z][kx][ky] with z < nz (3-D) or a single plane
// (2-D), kx <= nx, ky < pitch (2ny in 3-D, ny in 2-D).  Slabs split into ky
// classes have a second one of pitch ny for the x passes.
// The Newell spectra are real (the padded kernel is even or odd along every
// axis); the tensor is stored on the non-negative octant as
// blocks per (kx, ky) column (kz <= nz, ky <= ny, kern_at) and mirrored with
// parity signs.
#include "demag.hpp"

#include <atomic>

#include <algorithm>
#include <cmath>
#include <cstdlib>
#include <type_traits>
namespace fm {
namespace {

// Octant extraction after the setup transform of layout spec[c][z][kx][ky]
// (z < pz, ky < py): entry (c, oz, kx, oy) of the tensor = Re spec[c][oz][kx][oy],
// stored at kern_at.  `total` counts kcomp * kz_n * hx * (ny + 1) entries.
template <typename Real>
__global__ void extract_octant_kernel(const cplx<double> *spec, Real *kern, int kz_n, int hx, int ny, int pz,
                                      int py, int64_t total, KernLayout kl) {
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= total) return;
    const int64_t ly = ny + 1;
    const int64_t per_comp = (int64_t)kz_n * hx * ly;
    const int c = (int)(i / per_comp);
    int64_t r = i - (int64_t)c * per_comp;
    const int oz = (int)(r / ((int64_t)hx * ly));
    r -= (int64_t)oz * hx * ly;
    const int kx = (int)(r / ly), oy = (int)(r - (int64_t)kx * ly);
    kern[kern_at(kl, c, oz, kx, oy)] = Real(spec[(((int64_t)c * pz + oz) * hx + kx) * py + oy].x);
}

// ---------------------------------------------------------------------------
// Launch geometry
// ---------------------------------------------------------------------------
size_t lds_budget() { return 65536; }

// Rows per x workgroup: the largest power of two <= 16 whose packed lines fit
// in 64 KB of LDS (padded stride when that still fits) and 512 lanes; a line
// longer than 64 KB takes one packed line (two rows) per workgroup when it
// fits in `limit`, the device's LDS per workgroup (160 KB on gfx950).  The
// kernels take pairs of rows, a power of two of them: `max_rows` is rounded
// down to one, and at least 2.
bool pick_x(const LinePlan &lp, size_t ce, int &xr, int &ls, int max_rows = 16, size_t limit = 65536) {
    while (max_rows & (max_rows - 1)) max_rows &= max_rows - 1;
    max_rows = std::max(2, max_rows);
    if (lp.fixed) {
        // two workgroups of a CU's 160 KB; a line distance of 4 mod 32 slots
        // puts eight lines read at one element index on different banks
        ls = fx_size(lp.n);
        ls += (36 - ls % 32) % 32;
        for (xr = max_rows; xr > 2; xr >>= 1)
            if (xr / 2 * lp.threads <= kMaxBlock && (size_t)(xr / 2) * ls * ce <= limit / 2) return true;
        return lp.threads <= kMaxBlock && (size_t)ls * ce <= limit;
    }
    for (xr = max_rows; xr >= 2; xr >>= 1) {
        const int lines = xr / 2;
        if (lines * lp.threads > kMaxBlock) continue;
        for (int pad = kPad; pad >= 0; --pad)
            if ((size_t)lines * (lp.n + pad) * ce <= 65536) {
                ls = lp.n + pad;
                return true;
            }
    }
    xr = 2;
    if (lp.threads > kMaxBlock) return false;
    for (int pad = kPad; pad >= 0; --pad)
        if ((size_t)(lp.n + pad) * ce <= limit) {
            ls = lp.n + pad;
            return true;
        }
    return false;
}

int ilog2(int v) {
    int r = 0;
    while ((1 << r) < v) ++r;
    return r;
}

int pick_lpw(const LinePlan &lp, size_t ce, int nlines_per_unit = 1) {
    int lpw = std::max(1, 256 / std::max(1, lp.threads * nlines_per_unit));
    while (lpw > 1 && ((size_t)lpw * nlines_per_unit * (lp.n + kPad) * ce > lds_budget() ||
                       lpw * nlines_per_unit * lp.threads > kMaxBlock))
        --lpw;
    return lpw;
}

// Columns per long-z workgroup: the largest power of two whose lines fit in
// `budget` bytes of LDS and kMaxBlock lanes.
int pick_ztile(const LinePlan &lp, int ncomp, size_t ce, size_t budget = 65536) {
    int tile = 64;
    while (tile > 1 && ((size_t)ncomp * tile * (lp.n + kPad) * ce > budget || ncomp * tile * lp.threads > kMaxBlock))
        tile >>= 1;
    return tile;
}

// LDS bytes one workgroup may allocate on `device`: lines longer than 64 KB
// use the device's per-workgroup limit (160 KB on gfx950).
size_t device_lds_limit(int device) {
    int lds = 0;
    if (hipDeviceGetAttribute(&lds, hipDeviceAttributeMaxSharedMemoryPerBlock, device) == hipSuccess &&
        (size_t)lds > 65536)
        return (size_t)lds;
    return 65536;
}

template <typename Real>
KernelView<Real> kview(const Context &c) {
    const DemagPlan &dp = c.dp;
    KernelView<Real> K;
    K.k = dp.projection ? nullptr : static_cast<const Real *>(dp.kern);
    K.kcomp = dp.kcomp;
    K.l = dp.kl;
    K.kz_n = dp.kz_n;
    K.ny = dp.py / 2;
    K.nz = dp.pz / 2;
    K.py = dp.py;
    K.pz = dp.pz;
    K.hx = dp.hx;
    K.kxs = 2.0 * kPi / (dp.px * c.dx);
    K.kys = 2.0 * kPi / (dp.py * c.dy);
    K.kzs = 2.0 * kPi / (dp.pz * c.dz);
    return K;
}

// The volume fraction of a tier backend in the field's precision (FP32
// under mixed precision).
template <typename Real>
const Real *phi_array(const Context &c) {
    if constexpr (sizeof(Real) == 4) return c.d_phi32;
    else return c.d_phi;
}

template <typename Real, typename S>
struct BoundaryCorrArgs {
    Real *out;
    const S *m;
    const Real *phi;  // volume fraction in the field's precision
    const double *ms_cell;
    double ms;
    int64_t n;
    const int32_t *cell;
    const uint32_t *off, *row;
    const int32_t *src;
    const Real *tensor;  // the field's precision (FP32 rows under mixed precision)
    uint32_t groups, stencil;
};

// Sparse near-field demag correction of the boundary tiers
// (native/backends/fdm/src/demag_boundary_fp64.cu:23-76): the field at a
// target cell gains -sum_s dN(t, s) . (phi_s Ms_s m_s) per row, dN symmetric
// with the components Nxx, Nxy, Nxz, Nyy, Nyz, Nzz; sources < 0 are skipped.
// One wavefront per target cell: its lanes share each row's stencil entries
// (entry lane + 64 u, u < 4, per pass), a butterfly reduction gives the row's
// sum in FP64, and the cell's rows are added in plan order, so a cell named
// by several rows gets all of them without atomics.  A pass issues all of a
// lane's loads together: its source indices, then the gathered sources and
// the tensors, with every address clamped to a valid entry; a skipped entry
// subtracts exactly zero.
template <typename Real, typename S>
__global__ void __launch_bounds__(256) boundary_corr_kernel(BoundaryCorrArgs<Real, S> a) {
    constexpr int U = 4;
    const uint32_t g = blockIdx.x * 4u + (threadIdx.x >> 6);
    const uint32_t lane = threadIdx.x & 63u;
    if (g >= a.groups) return;  // a whole wavefront
    const int64_t ti = a.cell[g], n = a.n;
    double h[3] = {double(a.out[ti]), double(a.out[n + ti]), double(a.out[2 * n + ti])};
    const double *msp = a.ms_cell;
    for (uint32_t e = a.off[g]; e < a.off[g + 1]; ++e) {
        const uint64_t r0 = (uint64_t)a.row[e] * a.stencil;
        double cx = 0.0, cy = 0.0, cz = 0.0;
        for (uint32_t s0 = 0; s0 < a.stencil; s0 += U * 64u) {
            int32_t si[U];
            bool ok[U];
#pragma unroll
            for (int u = 0; u < U; ++u) {
                const uint32_t s = s0 + lane + 64u * u;
                ok[u] = s < a.stencil;
                si[u] = a.src[r0 + (ok[u] ? s : 0u)];
            }
            double w[U], mv[U][3];
            Real nn[U][6];
#pragma unroll
            for (int u = 0; u < U; ++u) {
                ok[u] = ok[u] && si[u] >= 0;
                const int64_t j = ok[u] ? si[u] : 0;
                const double pv = double(a.phi[j]);
                const double cv = *(msp ? msp + j : &kNoArrayF64);
                w[u] = pv * (msp ? cv : a.ms);
#pragma unroll
                for (int q = 0; q < 3; ++q) mv[u][q] = double(a.m[q * n + j]);
                const Real *t = a.tensor + (r0 + (ok[u] ? s0 + lane + 64u * u : 0u)) * 6;
#pragma unroll
                for (int q = 0; q < 6; ++q) nn[u][q] = t[q];
            }
#pragma unroll
            for (int u = 0; u < U; ++u) {
                const double mx = w[u] * mv[u][0], my = w[u] * mv[u][1], mz = w[u] * mv[u][2];
                const double n0 = nn[u][0], n1 = nn[u][1], n2 = nn[u][2];
                const double n3 = nn[u][3], n4 = nn[u][4], n5 = nn[u][5];
                cx -= ok[u] ? n0 * mx + n1 * my + n2 * mz : 0.0;
                cy -= ok[u] ? n1 * mx + n3 * my + n4 * mz : 0.0;
                cz -= ok[u] ? n2 * mx + n4 * my + n5 * mz : 0.0;
            }
        }
#pragma unroll
        for (int off = 32; off > 0; off >>= 1) {
            cx += __shfl_xor(cx, off);
            cy += __shfl_xor(cy, off);
            cz += __shfl_xor(cz, off);
        }
        h[0] += cx;
        h[1] += cy;
        h[2] += cz;
    }
    if (lane == 0) {
        a.out[ti] = Real(h[0]);
        a.out[n + ti] = Real(h[1]);
        a.out[2 * n + ti] = Real(h[2]);
    }
}

// Whether the y and z passes run as one slab kernel: a short-z tensor, a
// scheduled y length of at most 512 and a slab that fits the LDS (and the
// `slab` knob's KB).  us per mixed Heun step, separate passes and slab:
// 64x64x4 43.7 and 37.8, 128x128x4 51.8 and 41.7, 256x256x4 83.8 and 65.3,
// 500x250x8 189 and 167, 256x256x8 116 and 108; FP64 128x128x4 67.8 and 49.5,
// 128x128x8 90.3 and 67.2, 500x250x4 177 and 146.  With 5 to 8 layers and
// lines of 32 lanes a workgroup has up to 12 wavefronts of at most 85 FP64
// values: FP64 spills (250x150x6 108 and 151).  FP32 there takes one round of
// one workgroup per CU for up to 256 slabs, which the skewed x frequencies give
// (classes and slab: 250x150x6 93.5 and 79.4, 256x256x6 102.2 and 86.8,
// 500x250x6 153.5 and 140.6, 100x150x7 71.3 and 66.5); a caller's spectra keep
// px / 2 + 1 slabs, and there it gains only where the columns divide into full
// rounds of nz T lanes per component (256x256x6, 2.7 rounds, 99 separate and
// 102; 256x192x6, 2 rounds, 94 and 90).
template <typename Real>
bool use_slab(const DemagPlan &dp) {
    if (dp.tune.slab <= 0 || dp.projection || dp.nz < 2 || dp.pz > z_reg_max<Real>() || !dp.ly.fixed ||
        !slab_length(dp.py))
        return false;
    const size_t bytes = (size_t)3 * dp.nz * fx_size(dp.py) * sizeof(cplx<Real>);
    if (bytes > (size_t)dp.tune.slab * 1024 || bytes > dp.lds_limit) return false;
    if (dp.nz <= 4 || fx_lanes(dp.py) < 32) return true;
    const int cols = dp.nz * fx_lanes(dp.py), rounds = (int)cdiv(dp.py, cols);
    return sizeof(Real) == 4 && (dp.own || 10 * dp.py >= 9 * rounds * cols);
}

template <typename Real>
bool class_rule(const DemagPlan &dp);
// Whether workgroups of `lds` bytes, `per_column` for each column or one for
// `per_group` of them, take fewer rounds over the chip for px / 2 columns than
// for px / 2 + 1, as many to a CU as its LDS holds.  A kernel's registers can
// hold it to fewer (class_kernel: three wavefronts per SIMD, 512 workgroups of
// 8 layers where the LDS counts 768 or 1024), so for ky classes this is where
// the columns divide into whole rounds by the LDS, not the rounds that run.
bool saves_round(const DemagPlan &dp, size_t lds, int per_group = 1, int per_column = 1) {
    int dev = 0, cus = 0;
    if (hipGetDevice(&dev) != hipSuccess ||
        hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || cus <= 0)
        return false;
    const int64_t slots = cus * std::max<int64_t>(1, (int64_t)(dp.lds_limit / lds)), h = dp.px / 2;
    return cdiv(per_column * cdiv(h + 1, per_group), slots) > cdiv(per_column * cdiv(h, per_group), slots);
}

// Whether the x transforms run at the frequencies k + 1/2 (plans with the
// library's own tensor): the padded rows leave room for a skew-cyclic
// convolution, whose spectrum has px / 2 columns and no Nyquist one, so the
// slab kernel's workgroups, one to three per CU, come to whole rounds where
// px does.  us per mixed Heun step without and with: 256x256x8 117.6 and 94.2
// (257 slabs of 104 KB are two rounds), 500x250x8 175.3 and 152.5, 256x256x4
// 73.4 and 71.1, 128x128x8 55.1 and 53.6; ky classes where saves_round
// counts one less, 256x300x8 138.9 and 132.2, 384x500x7 217.6 and 210.5.  It does
// not for others that gain (256x512x8 176.1 and 170.7, 64x400x8 90.0 and 80.6) and
// does for one that does not (384x512x8 238 and 238).  Elsewhere the factors in
// the x passes cost more than a column: 512x512x8 342 and 346, 512x512x1 73.8 and
// 75.5, 256x256x64 756 and 768.  In FP64 they cost 2 to 3 us per pass
// (128x128x4 52 and 57), which only a round saved gives back.
template <typename Real>
bool skew_rule(const DemagPlan &dp) {
    if (dp.tune.skew == 0 || !dp.three_d) return false;
    if (!use_slab<Real>(dp))
        return sizeof(Real) == 4 && class_rule<Real>(dp) &&
               saves_round(dp, (size_t)3 * dp.nz * fx_size(dp.py / kClasses) * sizeof(cplx<Real>), 1, kClasses);
    return sizeof(Real) == 4 || saves_round(dp, (size_t)3 * dp.nz * fx_size(dp.py) * sizeof(cplx<Real>));
}

// Whether a slab's ky classes go through the y transform and the z
// convolution in one kernel each: the plan's choice (class_rule, fixed at set-up
// with the tensor's layout), its second spectrum, and the knobs.
template <typename Real>
bool use_class(const DemagPlan &dp) {
    return dp.cls > 1 && dp.xspec && dp.ly.fixed && dp.tune.slab > 0;
}

// The x passes' spectrum.
template <typename Real>
SpecGeom x_geom(const DemagPlan &dp) {
    return SpecGeom{dp.hx, dp.three_d ? dp.nz : 1, use_class<Real>(dp) ? dp.xrows : dp.rows};
}
template <typename Real>
cplx<Real> *x_spec(const DemagPlan &dp) {
    return static_cast<cplx<Real> *>(use_class<Real>(dp) ? dp.xspec : dp.spec);
}

// x R2C of Ms src, the y and z transforms with the tensor product and the
// inverse y and z transforms: everything up to the x C2R, in the spectrum.
template <typename Real, typename S>
void demag_transform_t(Context &c, const S *src, const XArgs<Real> &xa, unsigned xgroups, size_t xlds,
                       bool weight_ms) {
    DemagPlan &dp = c.dp;
    cplx<Real> *spec = static_cast<cplx<Real> *>(dp.spec);
    const SpecGeom g{dp.hx, dp.three_d ? dp.nz : 1, dp.rows};
    {
        const MagSource<Real, S> ms{src,    c.d_mask, weight_ms ? c.d_ms_cell : nullptr, weight_ms ? c.ms : 1.0,
                                    dp.nx,  dp.ny,    dp.nz,
                                    (int64_t)c.n, weight_ms ? phi_array<Real>(c) : nullptr};
        Timed t(c, "demag_x_r2c");
        auto launch = [&](const auto &src_v) {
            launch_xfwd<Real>(c, xa, src_v, x_spec<Real>(dp), xgroups, (unsigned)dp.nz, 3, xlds);
        };
        if (ms.mask || ms.ms_cell || ms.phi)
            launch(MagSource<Real, S, true>{ms.m, ms.mask, ms.ms_cell, ms.ms, ms.nx, ms.ny, ms.nz, ms.n, ms.phi});
        else
            launch(ms);
    }
    const KernelView<Real> K = kview<Real>(c);
    if (use_class<Real>(dp)) {
        SlabArgs<Real> sa{};
        sa.data = spec;
        sa.tw = static_cast<const cplx<Real> *>(dp.tw_y);
        sa.twz = static_cast<const cplx<Real> *>(dp.tw_z);
        sa.twp = static_cast<const cplx<Real> *>(dp.tw_c);
        sa.nz = dp.nz;
        sa.ny = dp.ny;
        sa.hx = dp.hx;
        sa.pitch = dp.rows;
        sa.plane_stride = (int64_t)dp.hx * dp.rows;
        sa.in = static_cast<const cplx<Real> *>(dp.xspec);
        sa.in_pitch = dp.xrows;
        sa.in_plane = (int64_t)dp.hx * dp.xrows;
        sa.K = K;
        {
            Timed t(c, "demag_yz_class");
            launch_class<Real>(c, dp.ly, sa);
        }
        LineArgs<Real> la{};
        la.in = spec;
        la.in_pitch = dp.rows;
        la.data = static_cast<cplx<Real> *>(dp.xspec);
        la.line_pitch = dp.xrows;
        la.tw = sa.tw;
        la.lp = dp.ly;
        la.lines = 3ll * dp.nz * dp.hx;
        la.n_in = dp.py;
        la.n_out = dp.ny;
        la.inverse = 1;
        Timed t(c, "demag_y_inv");
        launch_class_inverse<Real>(c, dp.ly, la);
    } else if (dp.three_d && use_slab<Real>(dp)) {
        SlabArgs<Real> sa{};
        sa.data = spec;
        sa.tw = static_cast<const cplx<Real> *>(dp.tw_y);
        sa.twz = static_cast<const cplx<Real> *>(dp.tw_z);
        sa.nz = dp.nz;
        sa.ny = dp.ny;
        sa.hx = dp.hx;
        sa.pitch = dp.rows;
        sa.plane_stride = (int64_t)dp.hx * dp.rows;
        sa.K = K;
        Timed t(c, "demag_yz_slab");
        launch_slab<Real>(c, dp.ly, sa);
    } else if (dp.three_d) {
        LineArgs<Real> la{};
        la.data = spec;
        la.tw = static_cast<const cplx<Real> *>(dp.tw_y);
        la.lp = dp.ly;
        la.lines = 3ll * dp.nz * dp.hx;
        la.line_pitch = dp.rows;
        la.lpw = dp.y_lines_per_wg;
        {
            la.n_in = dp.ny;
            la.n_out = dp.py;
            la.inverse = 0;
            Timed t(c, "demag_y_fwd");
            launch_lines<Real>(c, dp.ly, la);
        }
        {
            Timed t(c, "demag_z_conv");
            if (dp.pz <= z_reg_max<Real>()) {
                ZArgs<Real> za{};
                za.data = spec;
                za.tw = static_cast<const cplx<Real> *>(dp.tw_z);
                za.nz = dp.nz;
                za.hx = dp.hx;
                za.py = dp.py;
                za.pitch = dp.rows;
                za.columns = (int64_t)dp.hx * dp.rows;
                za.zstride = (int64_t)dp.hx * dp.rows;
                za.comp_stride = (int64_t)dp.nz * dp.hx * dp.rows;
                za.K = K;
                za.xcd = dp.tune.xcd;
                launch_zreg<Real>(c, za);
            } else {
                ZLdsArgs<Real> za{};
                za.data = spec;
                za.tw = static_cast<const cplx<Real> *>(dp.tw_z);
                za.lp = dp.lz;
                za.n_in = dp.nz;
                za.n_out = dp.nz;
                za.tile = dp.z_tile;
                za.conv = 1;
                za.columns = (int64_t)dp.hx * dp.rows;
                za.zstride = (int64_t)dp.hx * dp.rows;
                za.comp_stride = (int64_t)dp.nz * dp.hx * dp.rows;
                za.py = dp.py;
                za.pitch = dp.rows;
                za.K = K;
                za.xcd = dp.tune.xcd;
                launch_zlds<Real>(c, za, 1);
            }
        }
        {
            la.n_in = dp.py;
            la.n_out = dp.ny;
            la.inverse = 1;
            Timed t(c, "demag_y_inv");
            launch_lines<Real>(c, dp.ly, la);
        }
    } else if (dp.y_split) {
        LineArgs<Real> la{};
        la.data = spec;
        la.tw = static_cast<const cplx<Real> *>(dp.tw_y);
        la.lp = dp.ly;
        la.lines = 3ll * dp.hx;
        la.line_pitch = dp.rows;
        la.lpw = dp.y_lines_per_wg;
        {
            la.n_in = dp.ny;
            la.n_out = dp.py;
            la.inverse = 0;
            Timed t(c, "demag_y_fwd");
            launch_lines<Real>(c, dp.ly, la);
        }
        {
            Timed t(c, "demag_y_conv");
            launch_film_tensor<Real>(c, spec, K, dp.hx, dp.py, (int64_t)dp.rows);
        }
        {
            la.n_in = dp.py;
            la.n_out = dp.ny;
            la.inverse = 1;
            Timed t(c, "demag_y_inv");
            launch_lines<Real>(c, dp.ly, la);
        }
    } else {
        YConvArgs<Real> ya{};
        ya.data = spec;
        ya.tw = static_cast<const cplx<Real> *>(dp.tw_y);
        ya.lp = dp.ly;
        ya.ny = dp.ny;
        ya.hx = dp.hx;
        ya.kpw = dp.yconv_kpw;
        ya.g = g;
        ya.K = K;
        Timed t(c, "demag_y_conv");
        launch_yconv<Real>(c, ya);
    }
}

template <typename Real, typename S>
void demag_eval_t(Context &c, const S *src, Real *out, bool weight_ms, int phase) {
    DemagPlan &dp = c.dp;
    cplx<Real> *spec = x_spec<Real>(dp);
    const SpecGeom g = x_geom<Real>(dp);
    const size_t ce = sizeof(cplx<Real>);
    XArgs<Real> xa{};
    xa.tw = static_cast<const cplx<Real> *>(dp.tw_x);
    xa.sw = static_cast<const cplx<Real> *>(dp.sw);
    xa.sw64 = static_cast<const cplx<double> *>(dp.sw64);
    xa.lp = dp.lx;
    xa.rows = dp.ny;
    xa.n_in = dp.nx;
    xa.n_out = dp.nx;
    xa.scale = Real(dp.inv_npad);
    xa.g = g;
    xa.xr = dp.xr;
    xa.xr_log2 = ilog2(dp.xr);
    xa.ls = dp.x_ls;
    const unsigned xgroups = (unsigned)cdiv(dp.ny, dp.xr);
    const size_t xlds = (size_t)(dp.xr / 2) * dp.x_ls * ce;
    if (phase != kDemagFinish) {
        c.spec_pre = false;  // the spectrum is overwritten
        demag_transform_t<Real, S>(c, src, xa, xgroups, xlds, weight_ms);
    }
    if (phase == kDemagSpectrum) return;
    {
        FieldSink<Real> sink{out, c.d_mask, dp.nx, dp.ny, (int64_t)c.n};
        Timed t(c, "demag_x_c2r");
        launch_xinv<Real>(c, xa, spec, sink, xgroups, (unsigned)dp.nz, xlds);
    }
    if (weight_ms && c.corr_groups > 0) {
        BoundaryCorrArgs<Real, S> ba{};
        ba.out = out;
        ba.m = src;
        ba.phi = phi_array<Real>(c);
        ba.ms_cell = c.d_ms_cell;
        ba.ms = c.ms;
        ba.n = (int64_t)c.n;
        ba.cell = c.d_corr_cell;
        ba.off = c.d_corr_off;
        ba.row = c.d_corr_row;
        ba.src = c.d_corr_src;
        ba.tensor = static_cast<const Real *>(c.d_corr_n);
        ba.groups = c.corr_groups;
        ba.stencil = c.corr_stencil;
        Timed t(c, "demag_boundary");
        const dim3 g1((unsigned)cdiv((int64_t)c.corr_groups, 4));  // one wavefront per target cell
        launch_rec(c, nullptr, g1, dim3(256), 0, 1, ba, [&] {
            hipLaunchKernelGGL((boundary_corr_kernel<Real, S>), g1, dim3(256), 0, c.stream, ba);
        });
    }
}

// exp(-i pi d / px) at x, d = x up to px / 2 and x - px beyond: the factors
// that shift a row's x frequencies by 1/2.
std::vector<cplx<double>> skew_table(int px) {
    std::vector<cplx<double>> w = twiddle_table(2 * px);
    w.resize(px);
    for (int x = px / 2 + 1; x < px; ++x) w[x] = {-w[x].x, -w[x].y};
    return w;
}

// Twiddle tables of the plan's lengths, in one allocation.
template <typename Real>
bool upload_twiddles(Context &c) {
    DemagPlan &dp = c.dp;
    std::vector<cplx<Real>> all;
    for (int n : {dp.px, dp.py, dp.three_d ? dp.pz : 1, dp.cls > 1 ? dp.py / dp.cls : 1})
        for (const cplx<double> &w : twiddle_table(n)) all.push_back({(Real)w.x, (Real)w.y});
    const size_t roots = all.size();
    // FP32: the inputs' factors in FP64 after the tables, on a 16-byte boundary
    size_t at64 = 0;
    if (dp.skew) {
        const std::vector<cplx<double>> w = skew_table(dp.px);
        for (const cplx<double> &v : w) all.push_back({(Real)v.x, (Real)v.y});
        if (sizeof(Real) == 4) {
            at64 = (all.size() + 1) / 2 * 2;
            all.resize(at64 + 2 * w.size());
            std::memcpy(&all[at64], w.data(), w.size() * sizeof(w[0]));
        } else {
            at64 = roots;
        }
    }
    const size_t bytes = all.size() * sizeof(cplx<Real>);
    if (!ctx_alloc(c, &dp.tw_x, bytes, "twiddle tables")) return false;
    dp.tw_y = static_cast<cplx<Real> *>(dp.tw_x) + dp.px;
    dp.sw = dp.skew ? static_cast<cplx<Real> *>(dp.tw_x) + roots : nullptr;
    dp.sw64 = dp.skew ? static_cast<cplx<Real> *>(dp.tw_x) + at64 : nullptr;
    dp.tw_z = static_cast<cplx<Real> *>(dp.tw_y) + dp.py;
    dp.tw_c = static_cast<cplx<Real> *>(dp.tw_z) + (dp.three_d ? dp.pz : 1);
    return ctx_upload(c, dp.tw_x, all.data(), bytes, "hipMemcpy(twiddles)", c.last_error);
}

// Transform lengths: 2n per axis where the tensor comes as spectra of that
// grid (or from the k-space projection); with the library's own Newell build
// the padded lengths of pick_padded, except for the z lengths up to `z_keep`,
// whose register kernels take 2nz as it is.
void pad_lengths(DemagPlan &dp, bool free, int z_keep) {
    dp.px = free ? pick_padded(dp.nx) : 2 * dp.nx;
    dp.py = free ? pick_padded(dp.ny) : 2 * dp.ny;
    dp.pz = !dp.three_d ? 1 : free && 2 * dp.nz > z_keep ? pick_padded(dp.nz) : 2 * dp.nz;
    dp.hx = dp.px / 2 + (dp.skew ? 0 : 1);
}

// Device bytes that the Newell set-up holds at once: the FP64 spectrum of the
// padded tensor and its octant, and `kept` complex and `tensor` real values of
// `real` bytes per component, plane and column that stay.
size_t setup_bytes(const DemagPlan &dp, size_t kept, size_t tensor, size_t real) {
    const size_t hx = dp.px / 2 + 1, cells = (size_t)dp.nx * dp.ny * dp.nz;
    return 6 * (size_t)dp.pz * hx * dp.py * sizeof(cplx<double>) + 6 * cells * sizeof(double) +
           (2 * kept + tensor) * hx * real;
}

// Whether `bytes` and a margin for the small tables are free on the device.
// Lines longer than 2n take up to 4/3 of the memory per axis (800 cells along
// each of three axes: 413 GB for the set-up's spectrum at 2048 points, 197 GB at
// 1600), so a grid whose padded set-up does not fit keeps 2n.
bool fits_device(size_t bytes) {
    size_t free = 0, total = 0;
    return hipMemGetInfo(&free, &total) != hipSuccess || bytes + (size_t(64) << 20) <= free;
}

bool plan_lines(DemagPlan &dp, std::string &err) {
    const DemagTuning &t = dp.tune;
    const bool fx = t.fixed != 0;
    if (!plan_line(dp.px, dp.lx, err, std::max(1, t.x_lanes), t.x_radix, fx)) return false;
    if (!plan_line(dp.py, dp.ly, err, std::max(1, t.y_lanes), t.y_radix, fx)) return false;
    // the scheduled z lines read the tensor entries directly (no projection
    // fallback) and keep a line in one wavefront
    const bool fz = fx && !dp.projection && fx_has(dp.pz) && fx_lanes(dp.pz) <= 64 && dp.pz > 16;
    if (dp.three_d && !plan_line(dp.pz, dp.lz, err, 1, 16, fz)) return false;
    return true;
}

}  // namespace

void parse_tuning_string(DemagTuning &t, const char *text) {
    if (!text) return;
    std::string s(text);
    size_t pos = 0;
    while (pos < s.size()) {
        size_t end = s.find(',', pos);
        if (end == std::string::npos) end = s.size();
        const std::string kv = s.substr(pos, end - pos);
        const size_t eq = kv.find('=');
        if (eq != std::string::npos) {
            const std::string k = kv.substr(0, eq);
            const int v = std::atoi(kv.c_str() + eq + 1);
            if (k == "x_radix") t.x_radix = v;
            else if (k == "x_lanes") t.x_lanes = v;
            else if (k == "x_rows") t.x_rows = v;
            else if (k == "y_radix") t.y_radix = v;
            else if (k == "y_lanes") t.y_lanes = v;
            else if (k == "y_lpw") t.y_lpw = v;
            else if (k == "fixed") t.fixed = v;
            else if (k == "xcd") t.xcd = v;
            else if (k == "y_pipe") t.y_pipe = v;
            else if (k == "y_pipe_f") t.y_pipe_f = v;
            else if (k == "z_tile") t.z_tile = v;
            else if (k == "zc") t.zc = v;
            else if (k == "y_split") t.y_split = v;
            else if (k == "pad") t.pad = v;
            else if (k == "slab") t.slab = v;
            else if (k == "skew") t.skew = v;
        }
        pos = end + 1;
    }
}

namespace {

void parse_tuning(DemagTuning &t) { parse_tuning_string(t, std::getenv("FULLMAG_FDM_TUNE")); }

// Padded forward transform of the Newell kernel, FP64, into a temporary
// spectrum spec[6][pz][hx][py].
bool newell_forward(Context &c, const DemagPlan &dp, double z_offset, cplx<double> **spec_out, std::string &err,
                    bool z_even = false) {
    const int pz = dp.three_d ? dp.pz : 1, nzo = dp.three_d ? dp.nz : 1;
    const SpecGeom g{dp.hx, pz, dp.py};
    const size_t ce = sizeof(cplx<double>);
    // one allocation: the spectrum (before it, the octant's tables), the
    // octant and the twiddle tables
    const size_t spec_bytes = std::max(6 * (size_t)pz * dp.hx * dp.py * ce,
                                       (newell_scratch(dp.nx, dp.ny, nzo) * sizeof(double) + ce - 1) / ce * ce);
    const size_t oct_bytes = 6 * (size_t)dp.nx * dp.ny * nzo * sizeof(double);
    std::vector<cplx<double>> tw = twiddle_table(dp.px);
    for (int n : {dp.py, pz}) {
        const std::vector<cplx<double>> w = twiddle_table(n);
        tw.insert(tw.end(), w.begin(), w.end());
    }
    const size_t roots = tw.size();
    if (dp.skew) {
        const std::vector<cplx<double>> w = skew_table(dp.px);
        tw.insert(tw.end(), w.begin(), w.end());
    }
    void *d_spec = nullptr;
    bool ok = hip_ok(hipMalloc(&d_spec, spec_bytes + oct_bytes + tw.size() * ce), "hipMalloc(newell)", err);
    double *d_oct = reinterpret_cast<double *>(static_cast<char *>(d_spec) + spec_bytes);
    cplx<double> *twx = reinterpret_cast<cplx<double> *>(static_cast<char *>(d_spec) + spec_bytes + oct_bytes);
    cplx<double> *twy = twx + dp.px, *twz = twy + dp.py;
    ok = ok && ctx_upload(c, twx, tw.data(), tw.size() * ce, "hipMemcpy(twiddles)", err);
    ok = ok && newell_octant(c, dp.nx, dp.ny, nzo, c.dx, c.dy, c.dz, z_offset, static_cast<double *>(d_spec), d_oct, err);
    int xr = 2, xls = dp.px;
    LinePlan lx, ly, lz;
    ok = ok && plan_line(dp.px, lx, err) && plan_line(dp.py, ly, err) && (!dp.three_d || plan_line(dp.pz, lz, err));
    if (ok && !pick_x(lx, ce, xr, xls, 16, dp.lds_limit)) {
        err = "Newell setup: x line does not fit in LDS";
        ok = false;
    }
    if (ok) {
        cplx<double> *spec = static_cast<cplx<double> *>(d_spec);
        NewellSource src{d_oct, dp.nx, dp.ny, nzo, dp.px, dp.py, pz, z_even ? 1 : 0};
        XArgs<double> xa{};
        xa.tw = twx;
        xa.sw = xa.sw64 = dp.skew ? twx + roots : nullptr;
        xa.lp = lx;
        xa.rows = dp.py;
        xa.n_in = dp.px;
        xa.n_out = 0;
        xa.scale = 1.0;
        xa.g = g;
        xa.xr = xr;
        xa.xr_log2 = ilog2(xr);
        xa.ls = xls;
        launch_xfwd<double>(c, xa, src, spec, (unsigned)cdiv(dp.py, xr), (unsigned)pz, 6, (size_t)(xr / 2) * xls * ce);
        LineArgs<double> la{};
        la.data = spec;
        la.tw = twy;
        la.lp = ly;
        la.lines = 6ll * pz * dp.hx;
        la.line_pitch = dp.py;
        la.lpw = pick_lpw(ly, ce);
        la.n_in = dp.py;
        la.n_out = dp.py;
        la.inverse = 0;
        if ((size_t)la.lpw * (ly.n + kPad) * ce > dp.lds_limit || la.lpw * ly.threads > kMaxBlock) {
            err = "Newell setup: y line does not fit in LDS";
            ok = false;
        }
        if (ok) launch_lines<double>(c, ly, la);
        if (ok && dp.three_d) {
            ZLdsArgs<double> za{};
            za.data = spec;
            za.tw = twz;
            za.lp = lz;
            za.n_in = dp.pz;
            za.n_out = dp.pz;
            za.tile = pick_ztile(lz, 1, ce);
            za.conv = 0;
            za.columns = (int64_t)dp.hx * dp.py;
            za.zstride = (int64_t)dp.hx * dp.py;
            za.comp_stride = (int64_t)dp.pz * dp.hx * dp.py;
            za.py = dp.py;
            za.pitch = dp.py;
            if ((size_t)za.tile * (lz.n + kPad) * ce > dp.lds_limit || za.tile * lz.threads > kMaxBlock) {
                err = "Newell setup: z line does not fit in LDS";
                ok = false;
            } else {
                launch_zlds<double>(c, za, 6);
            }
        }
        ok = ok && hip_ok(hipStreamSynchronize(c.stream), "Newell setup transform", err);
        ok = ok && hip_ok(hipGetLastError(), "Newell setup launch", err);
    }
    if (!ok) {
        if (d_spec) (void)hipFree(d_spec);
        return false;
    }
    *spec_out = static_cast<cplx<double> *>(d_spec);
    return true;
}

bool host_octant_from_spectra(const DemagPlan &dp, const fullmag_fdm_plan_desc &plan, std::vector<double> &kern,
                              std::string &err) {
    // Full spectra are [pz][py][px] interleaved complex; keep Re on the octant.
    const double *src[6] = {plan.demag_kernel_xx_spectrum, plan.demag_kernel_yy_spectrum,
                            plan.demag_kernel_zz_spectrum, plan.demag_kernel_xy_spectrum,
                            plan.demag_kernel_xz_spectrum, plan.demag_kernel_yz_spectrum};
    const int pz = dp.three_d ? dp.pz : 1;
    kern.assign((size_t)(dp.hx * dp.kl.skx), 0.0);
    // parity of the six components along (x, y, z)
    const int odd[6][3] = {{0, 0, 0}, {0, 0, 0}, {0, 0, 0}, {1, 1, 0}, {1, 0, 1}, {0, 1, 1}};
    double kmax = 0.0, bad = 0.0;
    for (int c = 0; c < 6; ++c) {
        const double *s = src[c];
        for (int z = 0; z < pz; ++z)
            for (int y = 0; y < dp.py; ++y)
                for (int x = 0; x < dp.px; ++x) {
                    const int64_t i = ((int64_t)z * dp.py + y) * dp.px + x;
                    const double re = s[2 * i], im = s[2 * i + 1];
                    kmax = std::max(kmax, std::fabs(re));
                    bad = std::max(bad, std::fabs(im));
                    const int ox = x <= dp.nx ? x : dp.px - x;
                    const int oy = y <= dp.ny ? y : dp.py - y;
                    const int oz = (pz == 1 || z <= dp.nz) ? z : pz - z;
                    double sg = 1.0;
                    if (odd[c][0] && x > dp.nx) sg = -sg;
                    if (odd[c][1] && y > dp.ny) sg = -sg;
                    if (odd[c][2] && pz > 1 && z > dp.nz) sg = -sg;
                    const int64_t j = ((int64_t)oz * dp.py + oy) * dp.px + ox;
                    bad = std::max(bad, std::fabs(re - sg * s[2 * j]));
                    if (x <= dp.nx && y <= dp.ny && (pz == 1 || z <= dp.nz) && c < dp.kcomp)
                        kern[kern_at(dp.kl, c, z, x, y)] = re;
                }
    }
    if (bad > 1e-8 * std::max(kmax, 1e-300)) {
        err = "demag kernel spectra are not real with Newell parity symmetry (deviation " + std::to_string(bad) +
              " vs max " + std::to_string(kmax) + ")";
        return false;
    }
    if (dp.kcomp == 4) {
        // thin film: xz and yz vanish on the film plane; check they are noise
        double m2 = 0.0;
        for (int c = 4; c < 6; ++c)
            for (int64_t i = 0; i < (int64_t)dp.px * dp.py; ++i) m2 = std::max(m2, std::fabs(src[c][2 * i]));
        if (m2 > 1e-8 * std::max(kmax, 1e-300)) {
            err = "thin-film demag spectra carry non-zero xz/yz components";
            return false;
        }
    }
    return true;
}

template <typename Real>
bool upload_kern(Context &c, const std::vector<double> &kern) {
    DemagPlan &dp = c.dp;
    dp.kern_elems = kern.size();
    const size_t bytes = kern.size() * sizeof(Real);
    if (!ctx_alloc(c, &dp.kern, bytes, "demag tensor")) return false;
    if (sizeof(Real) == sizeof(double))
        return ctx_upload(c, dp.kern, kern.data(), bytes, "hipMemcpy(tensor)", c.last_error);
    std::vector<float> f(kern.size());
    for (size_t i = 0; i < kern.size(); ++i) f[i] = (float)kern[i];
    return ctx_upload(c, dp.kern, f.data(), bytes, "hipMemcpy(tensor)", c.last_error);
}

// Whether the plan splits its slabs into ky classes: short z lines and a
// scheduled y length of 320 to 1024 whose slab does not fit the slab kernel.
// us per Heun step, separate passes and classes: mixed 512x512x4 187.1 and
// 167.9, 400x400x2 115.8 and 105.0, 300x384x5 145.2 and 133.0, 100x300x8 104.3
// and 96.6, 512x512x8 348.7 and 344.5; FP64
// 512x512x4 330.9 and 300.3, 200x400x3 126.5 and 118.0.  FP64 with more than
// four layers needs a component per lane: 512x512x8 651 and 670.  Where both
// fit, the slab kernel mostly wins (mixed 128x200x7 76.9 against 80.6,
// 500x250x8 175.7 against 186.5).
template <typename Real>
bool class_rule(const DemagPlan &dp) {
    return dp.three_d && !dp.projection && dp.nz >= 2 && dp.nz <= (sizeof(Real) == 4 ? 8 : 4) && dp.ly.fixed &&
           class_length(dp.py) && dp.tune.slab > 0 && !use_slab<Real>(dp);
}

// Rows per x workgroup where full workgroups are few: with fewer than 64 of more
// than one wavefront each, halving the rows (down to 4) spreads the same lanes
// over twice the CUs, for shorter runs per column.  us per step: 500x125x1
// mixed 53.6 with 16 rows (24 workgroups of 512 lanes), 51.3 with 8, 50.5 with
// 4; 200x30x2 mixed 48.1, 46.1, 44.6.  Not beyond: 256x256x1 mixed (48
// workgroups of 256) 49.8 with 16 and with 8, 512x512x1 mixed (96) 75.4 and
// 76.6, 64x64x1 FP64 (12 of one wavefront) 42.5 and 43.5.
int spread_rows(int xr, int threads, int rows, int planes) {
    while (xr > 4 && xr / 2 * threads > 64 && cdiv(rows, xr) * planes < 64)
        xr >>= 1;
    return xr;
}

// Launch geometry of the planned lines (no allocation): x rows per
// workgroup, y lines per workgroup, long-z tile, thin-film y convolution
// form.  `keep_split` >= 0 requires the thin-film form to stay as it is (a
// re-plan may not change the spectrum's row count).
template <typename Real>
bool plan_geometry(DemagPlan &dp, std::string &err, int keep_split = -1) {
    const size_t ce = sizeof(cplx<Real>);
    {
        const int64_t ly = dp.py / 2 + 1, nzo = dp.kz_n;
        KernLayout &l = dp.kl;
        const bool planes = dp.three_d && dp.pz <= z_reg_max<Real>();
        l.cls = dp.cls;
        l.yw = (int)cdiv(ly, (int64_t)dp.cls);
        const int64_t w = (int64_t)dp.cls * l.yw;
        l.sc = planes ? w : 1;
        l.soy = planes ? 1 : dp.kcomp;
        l.odd = w * dp.kcomp;
        l.soz = 2 * l.odd;
        l.skx = nzo * l.odd;
    }
    if (!pick_x(dp.lx, ce, dp.xr, dp.x_ls, dp.tune.x_rows > 0 ? dp.tune.x_rows : 16, dp.lds_limit)) {
        err = "x line FFT does not fit in one workgroup";
        return false;
    }
    if (dp.lx.fixed && dp.tune.x_rows <= 0) dp.xr = spread_rows(dp.xr, dp.lx.threads, dp.ny, 3 * dp.nz);
    if (dp.three_d) {
        dp.y_lines_per_wg = pick_lpw(dp.ly, ce);
        if (dp.tune.y_lpw > 0) dp.y_lines_per_wg = std::min(dp.y_lines_per_wg, dp.tune.y_lpw);
        if ((size_t)dp.y_lines_per_wg * (dp.ly.n + kPad) * ce > dp.lds_limit ||
            dp.y_lines_per_wg * dp.ly.threads > kMaxBlock) {
            err = "y line FFT does not fit in LDS or 512 lanes";
            return false;
        }
        if (dp.pz > z_reg_max<Real>()) {
            // at most 32 KB per workgroup: five or more workgroups share a CU
            // (measured at pz = 128: 209 us with 8 columns against 265 us
            // with 16 at 48 KB)
            dp.z_tile = pick_ztile(dp.lz, 3, ce, 32768);
            if (dp.tune.z_tile > 0) dp.z_tile = std::min(dp.z_tile, dp.tune.z_tile);
            if ((size_t)3 * dp.z_tile * (dp.lz.n + kPad) * ce > dp.lds_limit ||
                3 * dp.z_tile * dp.lz.threads > kMaxBlock) {
                err = "z line FFT does not fit in LDS or 512 lanes";
                return false;
            }
        }
    } else {
        // a scheduled column is three lines of whole wavefront shares: about
        // one wavefront per workgroup keeps the most workgroups in flight
        dp.yconv_kpw = dp.ly.fixed ? std::max(1, 64 / (3 * dp.ly.threads)) : pick_lpw(dp.ly, ce, 3);
        const bool split = dp.tune.y_split != 0 || (size_t)3 * dp.yconv_kpw * line_slots(dp.ly) * ce > dp.lds_limit ||
                           3 * dp.yconv_kpw * dp.ly.threads > 1024;
        if (keep_split >= 0 && split != (keep_split != 0)) {
            err = "schedule changes the thin-film y convolution form";
            return false;
        }
        dp.y_split = split;
        if (dp.y_split) {
            // the spectrum keeps all py ky entries of every kx row
            dp.rows = dp.py;
            dp.y_lines_per_wg = pick_lpw(dp.ly, ce);
            if ((size_t)dp.y_lines_per_wg * (dp.ly.n + kPad) * ce > dp.lds_limit ||
                dp.y_lines_per_wg * dp.ly.threads > kMaxBlock) {
                err = "thin-film y line FFT does not fit in LDS or 512 lanes";
                return false;
            }
        }
    }
    return true;
}

template <typename Real>
bool setup_tensor_t(Context &c, const fullmag_fdm_plan_desc &plan) {
    DemagPlan &dp = c.dp;
    const size_t ce = sizeof(cplx<Real>);
    dp.cls = class_rule<Real>(dp) ? kClasses : 1;
    if (!plan_geometry<Real>(dp, c.last_error)) return false;
    if (!upload_twiddles<Real>(c)) return false;
    dp.spec_elems = 3ull * (dp.three_d ? dp.nz : 1) * dp.hx * dp.rows;
    if (!ctx_alloc(c, &dp.spec, dp.spec_elems * ce, "demag spectrum")) return false;
    if (dp.projection) return true;
    if (plan.demag_kernel_spectrum_len != 0) {
        std::vector<double> kern;
        if (!host_octant_from_spectra(dp, plan, kern, c.last_error)) return false;
        return upload_kern<Real>(c, kern);
    }
    // In-library Newell build: octant, padded transform.
    cplx<double> *spec = nullptr;
    if (!newell_forward(c, dp, 0.0, &spec, c.last_error)) return false;
    dp.kern_elems = (uint64_t)(dp.hx * dp.kl.skx);
    const int64_t entries = (int64_t)dp.kcomp * dp.kz_n * dp.hx * (dp.py / 2 + 1);
    bool ok = ctx_alloc(c, &dp.kern, dp.kern_elems * sizeof(Real), "demag tensor") &&
              hip_ok(hipMemsetAsync(dp.kern, 0, dp.kern_elems * sizeof(Real), c.stream), "hipMemsetAsync(tensor)",
                     c.last_error);
    if (ok) {
        const int pz = dp.three_d ? dp.pz : 1;
        hipLaunchKernelGGL((extract_octant_kernel<Real>), dim3((unsigned)cdiv(entries, 256)), dim3(256), 0,
                           c.stream, spec, static_cast<Real *>(dp.kern), dp.kz_n, dp.hx, dp.py / 2, pz, dp.py, entries,
                           dp.kl);
        ok = hip_ok(hipStreamSynchronize(c.stream), "extract octant", c.last_error);
    }
    (void)hipFree(spec);
    return ok;
}

// The tensor first, then the classes' second spectrum: without memory for it
// the separate passes run.
template <typename Real>
bool setup_t(Context &c, const fullmag_fdm_plan_desc &plan) {
    DemagPlan &dp = c.dp;
    if (!setup_tensor_t<Real>(c, plan)) return false;
    if (dp.cls > 1) {
        dp.xrows = dp.ny + (dp.ny & 1);
        const std::string err = c.last_error;
        if (!ctx_alloc(c, &dp.xspec, 3ull * dp.nz * dp.hx * dp.xrows * sizeof(cplx<Real>), "demag spectrum")) {
            dp.xspec = nullptr;
            c.last_error = err;
        }
    }
    return true;
}

}  // namespace

bool demag_setup(Context &c, const fullmag_fdm_plan_desc &plan, bool newell_on_device) {
    DemagPlan &dp = c.dp;
    dp = DemagPlan{};
    if (!c.demag) return true;
    dp.enabled = true;
    dp.nx = c.nx;
    dp.ny = c.ny;
    dp.nz = c.nz;
    const uint64_t len2d = 2ull * (2ull * c.nx) * (2ull * c.ny);
    const bool have_spectra = plan.demag_kernel_spectrum_len != 0;
    dp.projection = !have_spectra && !newell_on_device;
    dp.three_d = !(c.nz == 1 && ((have_spectra && plan.demag_kernel_spectrum_len == len2d) ||
                                 (!have_spectra && newell_on_device)));
    dp.own = !have_spectra && newell_on_device;
    parse_tuning(dp.tune);
    pad_lengths(dp, dp.own && dp.tune.pad != 0, z_reg_max<double>());
    if (dp.own && (dp.px > 2 * dp.nx || dp.py > 2 * dp.ny || (dp.three_d && dp.pz > 2 * dp.nz))) {
        const size_t planes = dp.three_d ? 3 * (size_t)dp.nz : 3, oy = dp.py / 2 + 1, oz = dp.three_d ? dp.pz / 2 + 1 : 1;
        const size_t need = setup_bytes(dp, planes * dp.py, (dp.three_d ? 6 : 4) * oz * oy, c.real_bytes());
        if (!fits_device(need)) pad_lengths(dp, false, 0);
    }
    // an even row count keeps two rows of a spectrum column in one 16-byte access
    dp.rows = dp.three_d ? dp.py : dp.ny + (dp.ny & 1);
    dp.kcomp = dp.three_d ? 6 : 4;
    dp.kz_n = dp.three_d ? dp.pz / 2 + 1 : 1;
    dp.inv_npad = 1.0 / ((double)dp.px * dp.py * dp.pz);
    dp.lds_limit = device_lds_limit(c.device);
    if (!plan_lines(dp, c.last_error)) return false;
    dp.skew = !have_spectra && newell_on_device &&
              (c.mode == MODE_DOUBLE ? skew_rule<double>(dp) : skew_rule<float>(dp));
    dp.hx = dp.px / 2 + (dp.skew ? 0 : 1);
    if (c.mode == MODE_DOUBLE) return setup_t<double>(c, plan);
    return setup_t<float>(c, plan);
}

bool demag_replan(Context &c, const DemagTuning &t, std::string &err) {
    if (!c.demag) {
        c.dp.tune = t;
        return true;
    }
    DemagPlan dp = c.dp;
    dp.tune = t;
    if (!plan_lines(dp, err)) return false;
    const bool ok = c.mode == MODE_DOUBLE ? plan_geometry<double>(dp, err, c.dp.y_split ? 1 : 0)
                                          : plan_geometry<float>(dp, err, c.dp.y_split ? 1 : 0);
    if (!ok) return false;
    c.dp = dp;  // same buffers: their sizes do not depend on the schedule
    return true;
}

void demag_eval(Context &c, const void *src, bool src_f64, void *out, bool weight_ms, int phase) {
    if (c.mode == MODE_DOUBLE) {
        demag_eval_t<double, double>(c, static_cast<const double *>(src), static_cast<double *>(out), weight_ms, phase);
    } else if (src_f64) {
        demag_eval_t<float, double>(c, static_cast<const double *>(src), static_cast<float *>(out), weight_ms, phase);
    } else {
        demag_eval_t<float, float>(c, static_cast<const float *>(src), static_cast<float *>(out), weight_ms, phase);
    }
}

// ---------------------------------------------------------------------------
// Multilayer stack demag (crates/fullmag-engine/src/multilayer.rs:159-262):
// every layer's Ms m on the common convolution grid is transformed (x R2C,
// y lines, z lines for a 3-D grid; a thin common grid uses the 2-D
// transform, whose padded z plane would only repeat the first), the pair
// kernels are applied point by point in k-space,
//   H_d(k) = -sum_s K(d, s)(k) . M_s(k),
// and every layer's field is transformed back.  Layers on another grid than
// the common one go through the push/pull transfers of
// crates/fullmag-fdm-demag/src/transfer.rs.
// ---------------------------------------------------------------------------
namespace {

template <typename Real>
struct StackTensorArgs {
    const cplx<Real> *m;
    cplx<Real> *h;
    const Real *kern;       // per kernel 6 components of `points` reals
    const int *pair;        // kernel of (dst, src)
    const uint32_t *kimag;  // per kernel: bit c set when component c is imaginary
    int layers;
    int64_t points;        // planes * hx * py, the same linear index in spectra and kernels
    int64_t layer_stride;  // complex elements per layer spectrum
    int64_t comp_stride;   // complex elements per component of a spectrum (= points)
    int64_t kern_stride;   // reals per pair kernel (6 * points)
};

// acc += k m for a purely real (im = false) or purely imaginary (k i) kernel
// entry.
template <typename T>
__device__ __forceinline__ void kmad(cplx<T> &acc, T k, bool im, const cplx<T> &m) {
    if (im) {
        acc.x -= k * m.y;
        acc.y += k * m.x;
    } else {
        acc.x += k * m.x;
        acc.y += k * m.y;
    }
}

// One lane per k-point; for every destination layer the sources are summed
// in layer order (the order of the reference's kernel pairs for that
// destination).  Kernel components: xx, yy, zz, xy, xz, yz.  Every padded
// Newell component has a definite parity along each axis, so its transform
// is purely real (an even number of odd axes) or purely imaginary (odd): one
// real per component is stored.  LT > 0: that many layers, their sources held
// in registers; 0: any count, sources reloaded per destination.
template <typename Real, int LT>
__global__ void __launch_bounds__(256) stack_tensor_kernel(StackTensorArgs<Real> a) {
    const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (i >= a.points) return;
    const int64_t cs = a.comp_stride;
    const int L = LT > 0 ? LT : a.layers;
    constexpr int NR = LT > 0 ? LT : 1;
    cplx<Real> mr[NR][3];
    if (LT > 0) {
#pragma unroll
        for (int s = 0; s < NR; ++s) {
            const cplx<Real> *M = a.m + (int64_t)s * a.layer_stride + i;
            mr[s][0] = M[0];
            mr[s][1] = M[cs];
            mr[s][2] = M[2 * cs];
        }
    }
    for (int d = 0; d < L; ++d) {
        cplx<Real> hx{Real(0), Real(0)}, hy{Real(0), Real(0)}, hz{Real(0), Real(0)};
#pragma unroll
        for (int s = 0; s < (LT > 0 ? LT : 1); ++s) {
            for (int s2 = s; s2 < (LT > 0 ? s + 1 : L); ++s2) {
                const int u = a.pair[d * L + s2];
                const uint32_t im = a.kimag[u];
                const Real *K = a.kern + (int64_t)u * a.kern_stride + i;
                cplx<Real> mx, my, mz;
                if (LT > 0) {
                    mx = mr[s][0];
                    my = mr[s][1];
                    mz = mr[s][2];
                } else {
                    const cplx<Real> *M = a.m + (int64_t)s2 * a.layer_stride + i;
                    mx = M[0];
                    my = M[cs];
                    mz = M[2 * cs];
                }
                const Real kxx = K[0], kyy = K[cs], kzz = K[2 * cs], kxy = K[3 * cs], kxz = K[4 * cs], kyz = K[5 * cs];
                const bool ixx = im & 1u, iyy = im & 2u, izz = im & 4u, ixy = im & 8u, ixz = im & 16u, iyz = im & 32u;
                kmad(hx, kxx, ixx, mx); kmad(hx, kxy, ixy, my); kmad(hx, kxz, ixz, mz);
                kmad(hy, kxy, ixy, mx); kmad(hy, kyy, iyy, my); kmad(hy, kyz, iyz, mz);
                kmad(hz, kxz, ixz, mx); kmad(hz, kyz, iyz, my); kmad(hz, kzz, izz, mz);
            }
        }
        cplx<Real> *H = a.h + (int64_t)d * a.layer_stride + i;
        H[0] = {-hx.x, -hx.y};
        H[cs] = {-hy.x, -hy.y};
        H[2 * cs] = {-hz.x, -hz.y};
    }
}

struct GridXfer {
    int nx, ny, nz;     // native grid
    double ndx, ndy, ndz;
    int cx, cy, cz;     // common grid
    double cdx, cdy, cdz;
};

// push_m (transfer.rs:18-121): every common-grid cell is the overlap-volume
// weighted mean of the native cells it overlaps (FP64); SoA in, SoA out.
template <typename S>
__global__ void __launch_bounds__(256) stack_push_kernel(GridXfer g, const S *m, double *out) {
    const int64_t nc = (int64_t)g.cx * g.cy * g.cz, nn = (int64_t)g.nx * g.ny * g.nz;
    const int64_t p = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (p >= nc) return;
    const int x = (int)(p % g.cx), y = (int)((p / g.cx) % g.cy), z = (int)(p / ((int64_t)g.cx * g.cy));
    const double lo[3] = {x * g.cdx, y * g.cdy, z * g.cdz};
    const double hi[3] = {lo[0] + g.cdx, lo[1] + g.cdy, lo[2] + g.cdz};
    const double nd[3] = {g.ndx, g.ndy, g.ndz};
    const int nmax[3] = {g.nx, g.ny, g.nz};
    int a0[3], a1[3];
    for (int d = 0; d < 3; ++d) {
        a0[d] = max((int)floor(lo[d] / nd[d]), 0);
        a1[d] = min((int)ceil(hi[d] / nd[d]), nmax[d]);
    }
    double tot = 0.0, acc[3] = {0.0, 0.0, 0.0};
    for (int k = a0[2]; k < a1[2]; ++k)
        for (int j = a0[1]; j < a1[1]; ++j)
            for (int i = a0[0]; i < a1[0]; ++i) {
                const double o[3] = {i * g.ndx, j * g.ndy, k * g.ndz};
                double ov = 1.0;
                for (int d = 0; d < 3; ++d) ov *= fmax(fmin(hi[d], o[d] + nd[d]) - fmax(lo[d], o[d]), 0.0);
                if (ov > 0.0) {
                    const int64_t q = ((int64_t)k * g.ny + j) * g.nx + i;
                    for (int c = 0; c < 3; ++c) acc[c] += double(m[c * nn + q]) * ov;
                    tot += ov;
                }
            }
    for (int c = 0; c < 3; ++c) out[c * nc + p] = tot > 0.0 ? acc[c] / tot : 0.0;
}

// pull_h (transfer.rs:124-198): trilinear interpolation of the common grid at
// every native cell centre, neighbour indices clamped; inactive cells zero.
template <typename Real>
__global__ void __launch_bounds__(256) stack_pull_kernel(GridXfer g, const Real *h, const uint8_t *mask, Real *out) {
    const int64_t nc = (int64_t)g.cx * g.cy * g.cz, nn = (int64_t)g.nx * g.ny * g.nz;
    const int64_t p = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (p >= nn) return;
    const int x = (int)(p % g.nx), y = (int)((p / g.nx) % g.ny), z = (int)(p / ((int64_t)g.nx * g.ny));
    const double f[3] = {(x + 0.5) * g.ndx / g.cdx - 0.5, (y + 0.5) * g.ndy / g.cdy - 0.5,
                         (z + 0.5) * g.ndz / g.cdz - 0.5};
    const int cmax[3] = {g.cx, g.cy, g.cz};
    int b[3];
    double w[3];
    for (int d = 0; d < 3; ++d) {
        b[d] = (int)floor(f[d]);
        w[d] = f[d] - floor(f[d]);
    }
    double r[3] = {0.0, 0.0, 0.0};
    for (int dz = 0; dz < 2; ++dz)
        for (int dy = 0; dy < 2; ++dy)
            for (int dx = 0; dx < 2; ++dx) {
                const int ix = min(max(b[0] + dx, 0), cmax[0] - 1);
                const int iy = min(max(b[1] + dy, 0), cmax[1] - 1);
                const int iz = min(max(b[2] + dz, 0), cmax[2] - 1);
                const double ww = (dx == 0 ? 1.0 - w[0] : w[0]) * (dy == 0 ? 1.0 - w[1] : w[1]) *
                                  (dz == 0 ? 1.0 - w[2] : w[2]);
                const int64_t q = ((int64_t)iz * g.cy + iy) * g.cx + ix;
                for (int c = 0; c < 3; ++c) r[c] += double(h[c * nc + q]) * ww;
            }
    const bool act = !mask || mask[p];
    for (int c = 0; c < 3; ++c) out[c * nn + p] = act ? Real(r[c]) : Real(0);
}

// One real per kernel component: the imaginary part where bit c of `imag`
// is set, else the real part (the other part is zero up to rounding).
template <typename Real>
__global__ void __launch_bounds__(256) spec_part_kernel(const cplx<double> *in, Real *out, int64_t points,
                                                        uint32_t imag) {
    const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (i >= 6 * points) return;
    const int c = (int)(i / points);
    out[i] = Real(((imag >> c) & 1u) ? in[i].y : in[i].x);
}

// The ky octant of one kernel: out[kx][c][ky], ky <= py / 2.
template <typename Real>
__global__ void __launch_bounds__(256) stack_octant_kernel(const cplx<double> *in, Real *out, int hx, int py,
                                                           uint32_t imag) {
    const int hp = py / 2 + 1;
    const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (i >= (int64_t)hx * 6 * hp) return;
    const int ky = (int)(i % hp), c = (int)(i / hp % 6), kx = (int)(i / ((int64_t)hp * 6));
    const cplx<double> v = in[((int64_t)c * hx + kx) * py + ky];
    out[i] = Real(((imag >> c) & 1u) ? v.y : v.x);
}

GridXfer xfer_of(const Stack &s, const Context &l) {
    const Context &c = s.conv;
    return GridXfer{(int)l.nx, (int)l.ny, (int)l.nz, l.dx, l.dy, l.dz,
                    (int)c.nx, (int)c.ny, (int)c.nz, c.dx, c.dy, c.dz};
}

template <typename Real>
bool stack_setup_t(Stack &s, std::string &err) {
    Context &c = s.conv;
    DemagPlan &dp = c.dp;
    const size_t ce = sizeof(cplx<Real>);
    const int L = (int)s.layers.size();
    dp = DemagPlan{};
    dp.enabled = true;
    dp.nx = c.nx;
    dp.ny = c.ny;
    dp.nz = c.nz;
    dp.three_d = c.nz > 1;
    DemagTuning tune;
    parse_tuning(tune);
    dp.tune.y_split = tune.y_split;
    // pair kernels: the self kernel once, one shifted kernel per distinct
    // z distance dst - src (compared exactly)
    std::vector<double> shifts;
    s.pair.assign((size_t)L * L, 0);
    for (int d = 0; d < L; ++d)
        for (int q = 0; q < L; ++q) {
            if (d == q) continue;
            const double sh = s.oz[d] - s.oz[q];
            auto it = std::find(shifts.begin(), shifts.end(), sh);
            if (it == shifts.end()) {
                shifts.push_back(sh);
                it = shifts.end() - 1;
            }
            s.pair[(size_t)d * L + q] = 1 + (int)(it - shifts.begin());
        }
    s.nkern = 1 + (int)shifts.size();
    pad_lengths(dp, true, 0);
    if (dp.px > 2 * dp.nx || dp.py > 2 * dp.ny || (dp.three_d && dp.pz > 2 * dp.nz)) {
        const size_t points = (size_t)dp.pz * dp.py;
        if (!fits_device(setup_bytes(dp, 6 * points * L, 6 * points * s.nkern, c.real_bytes()))) pad_lengths(dp, false, 0);
    }
    dp.rows = dp.py;
    dp.inv_npad = 1.0 / ((double)dp.px * dp.py * dp.pz);
    dp.lds_limit = device_lds_limit(c.device);
    if (!plan_lines(dp, err)) return false;
    // The coupled y pass takes a thin stack whose column of 3 L lines fits one
    // workgroup; several columns where they are short.  Against the separate
    // passes, Heun steps of 2 to 5 layers of 64 x 64 to 512 x 512: 1.03 to
    // 1.6 times as fast wherever it fits, FP32 and FP64.
    s.kpw = std::max(1, 256 / (3 * L * dp.ly.threads));
    s.fused = !dp.three_d && dp.ly.fixed && !dp.tune.y_split &&
              ystack_fits<Real>(dp.py, L, s.kpw, std::min(dp.lds_limit, kLdsMax));
    // Frequencies k + 1/2 along x (skew_rule) where that saves a round: 3 films
    // of 512x512, 513 workgroups, mixed 138.3 and 125.4 us per step, FP64 214.8
    // and 203.1; without one saved, 100x300 four films FP64 79.5 and 83.0.
    dp.skew = tune.skew != 0 && s.fused &&
              saves_round(dp, (size_t)3 * L * s.kpw * line_slots(dp.ly) * ce, s.kpw);
    dp.hx = dp.px / 2 + (dp.skew ? 0 : 1);
    if (!pick_x(dp.lx, ce, dp.xr, dp.x_ls, 16, dp.lds_limit)) {
        err = "stack: x line FFT does not fit in one workgroup";
        return false;
    }
    dp.y_lines_per_wg = pick_lpw(dp.ly, ce);
    if ((size_t)dp.y_lines_per_wg * (dp.ly.n + kPad) * ce > dp.lds_limit ||
        dp.y_lines_per_wg * dp.ly.threads > kMaxBlock) {
        err = "stack: y line FFT does not fit in LDS or 512 lanes";
        return false;
    }
    if (dp.three_d) {
        dp.z_tile = pick_ztile(dp.lz, 1, ce);
        if ((size_t)dp.z_tile * (dp.lz.n + kPad) * ce > dp.lds_limit || dp.z_tile * dp.lz.threads > kMaxBlock) {
            err = "stack: z line FFT does not fit in LDS or 512 lanes";
            return false;
        }
    }
    if (!upload_twiddles<Real>(c)) {
        err = c.last_error;
        return false;
    }
    s.planes = dp.pz;
    const int64_t points = (int64_t)s.planes * dp.hx * dp.py;
    s.layer_spec = 3 * (uint64_t)points;
    if (!ctx_alloc(c, &s.spec_m, (size_t)L * s.layer_spec * ce, "stack spectra") ||
        (!s.fused && !ctx_alloc(c, &s.spec_h, (size_t)L * s.layer_spec * ce, "stack field spectra"))) {
        err = c.last_error;
        return false;
    }
    s.kern_stride = s.fused ? 6 * (uint64_t)dp.hx * (dp.py / 2 + 1) : 6 * (uint64_t)points;
    // components with an odd number of odd axes transform to imaginary
    // values: xz (odd in x) and yz (odd in y) of the shifted kernels, whose
    // z mirror keeps the sign, and of the thin self kernel (zero there); in
    // the 3-D self kernel they are also odd in z, so every component is real
    std::vector<uint32_t> kimag(s.nkern, (1u << 4) | (1u << 5));
    if (dp.three_d) kimag[0] = 0;
    if (!ctx_alloc(c, &s.kern, (size_t)s.nkern * s.kern_stride * sizeof(Real), "stack pair kernels") ||
        !ctx_alloc(c, (void **)&s.d_pair, s.pair.size() * sizeof(int), "stack pair table") ||
        !ctx_alloc(c, (void **)&s.d_kimag, kimag.size() * sizeof(uint32_t), "stack kernel parities") ||
        !ctx_upload(c, s.d_pair, s.pair.data(), s.pair.size() * sizeof(int), "hipMemcpy(pair table)", err) ||
        !ctx_upload(c, s.d_kimag, kimag.data(), kimag.size() * sizeof(uint32_t), "hipMemcpy(parities)", err))
        return false;
    for (int u = 0; u < s.nkern; ++u) {
        cplx<double> *spec = nullptr;
        if (!newell_forward(c, dp, u == 0 ? 0.0 : shifts[u - 1], &spec, err, u > 0)) return false;
        Real *dst = static_cast<Real *>(s.kern) + (uint64_t)u * s.kern_stride;
        const dim3 grid((unsigned)cdiv(s.kern_stride, 256));
        if (s.fused)
            hipLaunchKernelGGL((stack_octant_kernel<Real>), grid, dim3(256), 0, c.stream, spec, dst, dp.hx, dp.py,
                               kimag[u]);
        else
            hipLaunchKernelGGL((spec_part_kernel<Real>), grid, dim3(256), 0, c.stream, spec, dst, (int64_t)points,
                               kimag[u]);
        const bool ok = hip_ok(hipStreamSynchronize(c.stream), "stack kernel", err);
        (void)hipFree(spec);
        if (!ok) return false;
    }
    s.conv_m.assign(L, nullptr);
    s.conv_h.assign(L, nullptr);
    const uint64_t ncv = (uint64_t)c.nx * c.ny * c.nz;
    for (int l = 0; l < L; ++l) {
        const Context &lc = *s.layers[l];
        if (lc.nx == c.nx && lc.ny == c.ny && lc.nz == c.nz) continue;  // transfer.rs identity fast path
        if (!ctx_alloc(c, &s.conv_m[l], 3 * ncv * sizeof(double), "stack transfer m") ||
            !ctx_alloc(c, &s.conv_h[l], 3 * ncv * sizeof(Real), "stack transfer H")) {
            err = c.last_error;
            return false;
        }
    }
    return hip_ok(hipGetLastError(), "stack setup", err);
}

// y lines (3-D: per component, over the nz stored planes) and z lines of
// `layers` spectra, forward or inverse.
template <typename Real>
void stack_yz(Stack &s, cplx<Real> *spec, int layers, bool inverse) {
    Context &c = s.conv;
    const DemagPlan &dp = c.dp;
    const int64_t comp = (int64_t)s.planes * dp.hx * dp.py;
    auto zpass = [&](int l) {
        ZLdsArgs<Real> za{};
        za.data = spec + l * 3 * comp;
        za.tw = static_cast<const cplx<Real> *>(dp.tw_z);
        za.lp = dp.lz;
        za.n_in = inverse ? dp.pz : dp.nz;
        za.n_out = inverse ? dp.nz : dp.pz;
        za.tile = dp.z_tile;
        za.conv = 0;
        za.inverse = inverse ? 1 : 0;
        za.columns = (int64_t)dp.hx * dp.py;
        za.zstride = (int64_t)dp.hx * dp.py;
        za.comp_stride = comp;
        za.py = dp.py;
        za.pitch = dp.py;
        launch_zlds<Real>(c, za, 3);
    };
    for (int l = 0; dp.three_d && inverse && l < layers; ++l) zpass(l);
    LineArgs<Real> la{};
    la.tw = static_cast<const cplx<Real> *>(dp.tw_y);
    la.lp = dp.ly;
    la.line_pitch = dp.py;
    la.lpw = dp.y_lines_per_wg;
    la.n_in = inverse ? dp.py : dp.ny;
    la.n_out = inverse ? dp.ny : dp.py;
    la.inverse = inverse ? 1 : 0;
    if (dp.three_d) {
        la.lines = (int64_t)dp.nz * dp.hx;
        for (int k = 0; k < 3 * layers; ++k) {
            la.data = spec + k * comp;
            launch_lines<Real>(c, dp.ly, la);
        }
    } else {
        la.data = spec;
        la.lines = 3ll * layers * dp.hx;
        launch_lines<Real>(c, dp.ly, la);
    }
    for (int l = 0; dp.three_d && !inverse && l < layers; ++l) zpass(l);
}

template <typename Real, typename S>
void stack_eval_t(Stack &s, const S *const *src) {
    Context &c = s.conv;
    DemagPlan &dp = c.dp;
    const int L = (int)s.layers.size();
    XArgs<Real> xa{};
    xa.tw = static_cast<const cplx<Real> *>(dp.tw_x);
    xa.sw = static_cast<const cplx<Real> *>(dp.sw);
    xa.sw64 = static_cast<const cplx<double> *>(dp.sw64);
    xa.lp = dp.lx;
    xa.rows = dp.ny;
    xa.n_in = dp.nx;
    xa.n_out = dp.nx;
    xa.scale = Real(dp.inv_npad);
    xa.g = SpecGeom{dp.hx, s.planes, dp.py};
    xa.xr = dp.xr;
    xa.xr_log2 = ilog2(dp.xr);
    xa.ls = dp.x_ls;
    const unsigned xgroups = (unsigned)cdiv(dp.ny, dp.xr);
    const size_t xlds = (size_t)(dp.xr / 2) * dp.x_ls * sizeof(cplx<Real>);
    const int64_t ncv = (int64_t)c.nx * c.ny * c.nz;
    cplx<Real> *sm = static_cast<cplx<Real> *>(s.spec_m);
    cplx<Real> *sh = s.fused ? sm : static_cast<cplx<Real> *>(s.spec_h);
    // layers on the common grid go through the x passes together
    bool together = true, masked = false;
    for (int l = 0; l < L; ++l) {
        together = together && !s.conv_m[l];
        masked = masked || s.layers[l]->d_mask;
    }
    {
        Timed t(c, "stack_forward");
        for (int l0 = 0; together && l0 < L; l0 += kStackPack) {
            StackMag<Real, S> ms{};
            const int nl = std::min(kStackPack, L - l0);
            for (int l = 0; l < nl; ++l) {
                ms.m[l] = src[l0 + l];
                ms.mask[l] = s.layers[l0 + l]->d_mask;
                ms.ms[l] = s.layers[l0 + l]->ms;
            }
            ms.nx = dp.nx;
            ms.ny = dp.ny;
            ms.nz = dp.nz;
            ms.n = ncv;
            ms.layer_stride = (int64_t)s.layer_spec;
            launch_xfwd_stack<Real, S>(c, xa, ms, masked, sm + (uint64_t)l0 * s.layer_spec, xgroups, (unsigned)dp.nz,
                                       (unsigned)nl, xlds);
        }
        for (int l = 0; !together && l < L; ++l) {
            Context &lc = *s.layers[l];
            cplx<Real> *spec = sm + (uint64_t)l * s.layer_spec;
            if (s.conv_m[l]) {
                double *cm = static_cast<double *>(s.conv_m[l]);
                hipLaunchKernelGGL((stack_push_kernel<S>), dim3((unsigned)cdiv(ncv, 256)), dim3(256), 0, c.stream,
                                   xfer_of(s, lc), src[l], cm);
                MagSource<Real, double> ms{cm, nullptr, nullptr, lc.ms, dp.nx, dp.ny, dp.nz, ncv, nullptr};
                launch_xfwd<Real>(c, xa, ms, spec, xgroups, (unsigned)dp.nz, 3, xlds);
            } else {
                if (lc.d_mask) {
                    MagSource<Real, S, true> ms{src[l], lc.d_mask, nullptr, lc.ms, dp.nx, dp.ny, dp.nz, ncv, nullptr};
                    launch_xfwd<Real>(c, xa, ms, spec, xgroups, (unsigned)dp.nz, 3, xlds);
                } else {
                    MagSource<Real, S> ms{src[l], nullptr, nullptr, lc.ms, dp.nx, dp.ny, dp.nz, ncv, nullptr};
                    launch_xfwd<Real>(c, xa, ms, spec, xgroups, (unsigned)dp.nz, 3, xlds);
                }
            }
        }
        if (!s.fused) stack_yz<Real>(s, sm, L, false);
    }
    if (s.fused) {
        Timed t(c, "stack_tensor");
        YStackArgs<Real> ya{};
        ya.data = sm;
        ya.tw = static_cast<const cplx<Real> *>(dp.tw_y);
        ya.kern = static_cast<const Real *>(s.kern);
        ya.ny = dp.ny;
        ya.hx = dp.hx;
        ya.kpw = s.kpw;
        for (int d = 0; d < L; ++d)
            for (int q = 0; q < L; ++q) ya.kernel[d][q] = s.pair[(size_t)d * L + q];
        launch_ystack<Real>(c, dp.ly, L, ya);
    } else {
        Timed t(c, "stack_tensor");
        StackTensorArgs<Real> ta{};
        ta.m = sm;
        ta.h = sh;
        ta.kern = static_cast<const Real *>(s.kern);
        ta.pair = s.d_pair;
        ta.kimag = s.d_kimag;
        ta.layers = L;
        ta.points = (int64_t)s.planes * dp.hx * dp.py;
        ta.layer_stride = (int64_t)s.layer_spec;
        ta.comp_stride = ta.points;
        ta.kern_stride = (int64_t)s.kern_stride;
        const dim3 tg((unsigned)cdiv(ta.points, 256)), tb(256);
        switch (L) {
            case 1: hipLaunchKernelGGL((stack_tensor_kernel<Real, 1>), tg, tb, 0, c.stream, ta); break;
            case 2: hipLaunchKernelGGL((stack_tensor_kernel<Real, 2>), tg, tb, 0, c.stream, ta); break;
            case 3: hipLaunchKernelGGL((stack_tensor_kernel<Real, 3>), tg, tb, 0, c.stream, ta); break;
            case 4: hipLaunchKernelGGL((stack_tensor_kernel<Real, 4>), tg, tb, 0, c.stream, ta); break;
            default: hipLaunchKernelGGL((stack_tensor_kernel<Real, 0>), tg, tb, 0, c.stream, ta); break;
        }
    }
    {
        Timed t(c, "stack_inverse");
        if (!s.fused) stack_yz<Real>(s, sh, L, true);
        for (int l0 = 0; together && l0 < L; l0 += kStackPack) {
            StackField<Real> sf{};
            const int nl = std::min(kStackPack, L - l0);
            for (int l = 0; l < nl; ++l) {
                sf.out[l] = static_cast<Real *>(s.layers[l0 + l]->hd);
                sf.mask[l] = s.layers[l0 + l]->d_mask;
            }
            sf.nx = dp.nx;
            sf.ny = dp.ny;
            sf.n = ncv;
            sf.layer_stride = (int64_t)s.layer_spec;
            launch_xinv_stack<Real>(c, xa, sh + (uint64_t)l0 * s.layer_spec, sf, xgroups, (unsigned)dp.nz,
                                    (unsigned)nl, xlds);
        }
        for (int l = 0; !together && l < L; ++l) {
            Context &lc = *s.layers[l];
            const cplx<Real> *spec = sh + (uint64_t)l * s.layer_spec;
            const bool xfer = s.conv_h[l] != nullptr;
            Real *out = xfer ? static_cast<Real *>(s.conv_h[l]) : static_cast<Real *>(lc.hd);
            FieldSink<Real> sink{out, xfer ? nullptr : lc.d_mask, dp.nx, dp.ny, ncv};
            launch_xinv<Real>(c, xa, spec, sink, xgroups, (unsigned)dp.nz, xlds);
            if (xfer)
                hipLaunchKernelGGL((stack_pull_kernel<Real>), dim3((unsigned)cdiv(lc.n, 256)), dim3(256), 0,
                                   c.stream, xfer_of(s, lc), static_cast<const Real *>(s.conv_h[l]), lc.d_mask,
                                   static_cast<Real *>(lc.hd));
        }
    }
}

}  // namespace

bool stack_demag_setup(Stack &s, std::string &err) {
    if (!s.demag) return true;
    if (s.conv.mode == MODE_DOUBLE) return stack_setup_t<double>(s, err);
    return stack_setup_t<float>(s, err);
}

void stack_demag_eval(Stack &s, const void *const *src, bool src_state) {
    if (!s.demag) return;
    const int mode = s.conv.mode;
    const size_t L = s.layers.size();
    if (mode == MODE_DOUBLE) {
        std::vector<const double *> v(L);
        for (size_t l = 0; l < L; ++l) v[l] = static_cast<const double *>(src[l]);
        stack_eval_t<double, double>(s, v.data());
    } else if (mode == MODE_MIXED && src_state) {
        std::vector<const double *> v(L);
        for (size_t l = 0; l < L; ++l) v[l] = static_cast<const double *>(src[l]);
        stack_eval_t<float, double>(s, v.data());
    } else {
        std::vector<const float *> v(L);
        for (size_t l = 0; l < L; ++l) v[l] = static_cast<const float *>(src[l]);
        stack_eval_t<float, float>(s, v.data());
    }
}

bool newell_spectra_full(uint32_t nx, uint32_t ny, uint32_t nz, double dx, double dy, double dz, bool thin_film_2d,
                         double *out, std::string &err) {
    Context c;
    c.nx = nx; c.ny = ny; c.nz = nz; c.dx = dx; c.dy = dy; c.dz = dz;
    c.mode = MODE_DOUBLE;
    if (!hip_ok(hipGetDevice(&c.device), "hipGetDevice", err)) return false;
    if (!hip_ok(hipStreamCreateWithFlags(&c.stream, hipStreamNonBlocking), "hipStreamCreate", err)) return false;
    DemagPlan dp;
    dp.lds_limit = device_lds_limit(c.device);
    dp.nx = nx; dp.ny = ny; dp.nz = nz;
    dp.three_d = !thin_film_2d;
    pad_lengths(dp, false, 0);
    bool ok = true;
    cplx<double> *spec = nullptr;
    if (ok) ok = newell_forward(c, dp, 0.0, &spec, err);
    if (ok) {
        const int pz = dp.pz;
        const SpecGeom g{dp.hx, pz, dp.py};
        std::vector<cplx<double>> h((size_t)6 * pz * dp.hx * dp.py);
        ok = hip_ok(hipMemcpy(h.data(), spec, h.size() * sizeof(cplx<double>), hipMemcpyDeviceToHost),
                    "hipMemcpy(newell spectrum)", err);
        (void)hipFree(spec);
        if (ok) {
            const int64_t npad = (int64_t)dp.px * dp.py * pz;
            for (int comp = 0; comp < 6; ++comp)
                for (int z = 0; z < pz; ++z)
                    for (int y = 0; y < dp.py; ++y)
                        for (int x = 0; x < dp.px; ++x) {
                            cplx<double> v;
                            if (x < dp.hx) {
                                v = h[g.at(comp, z, x, y)];
                            } else {
                                // Hermitian continuation of a real kernel
                                v = h[g.at(comp, (pz - z) % pz, dp.px - x, (dp.py - y) % dp.py)];
                                v.y = -v.y;
                            }
                            const int64_t i = ((int64_t)z * dp.py + y) * dp.px + x;
                            out[comp * 2 * npad + 2 * i] = v.x;
                            out[comp * 2 * npad + 2 * i + 1] = v.y;
                        }
        }
    }
    (void)hipStreamDestroy(c.stream);
    return ok;
}

}  // namespace fm

