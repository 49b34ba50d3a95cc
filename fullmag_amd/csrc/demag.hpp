// demag.hpp -- types shared by the demag transform kernels (demag_x.hip,
// demag_y.hip, demag_z.hip) and their driver (demag.hip): tensor access,
// spectrum addressing, argument packs, and the launch functions each kernel
// file provides.  The kernel files are compiled once per field precision.
#pragma once

#include "context.hpp"

#include <type_traits>

namespace fm {

constexpr int kPad = 1;         // LDS line padding (complex slots) of runtime-planned lines
// LDS slots of one line.
inline int line_slots(const LinePlan &lp) { return lp.fixed ? fx_size(lp.n) : lp.n + kPad; }

// Stand-ins read in place of an absent optional per-cell array, so that the
// read itself needs no branch: an active-mask byte of 1 and a value of 1.
static __device__ const uint8_t kNoMask = 1;
static __device__ const double kNoArrayF64 = 1.0;
static __device__ const float kNoArrayF32 = 1.0f;
template <typename T>
__device__ __forceinline__ const T *no_array() {
    if constexpr (sizeof(T) == 4) return &kNoArrayF32;
    else return &kNoArrayF64;
}
constexpr int kMaxBlock = 512;  // lanes per workgroup for FFT kernels
// largest padded z length done in registers (a lane holds a column's 3 pz / 2
// inputs and one half of its padded spectrum; FP64 spreads the components over
// three wavefronts)
template <typename Real>
constexpr int z_reg_max() {
    return 16;
}

// Workgroup b runs on XCD b mod 8 (round-robin dispatch over the 8 XCDs of
// an MI355X).  Renumbered so that each XCD receives one contiguous range of
// logical workgroups.
__device__ __forceinline__ uint32_t xcd_block(uint32_t b, uint32_t g) {
    const uint32_t x = b & 7u, q = g >> 3, r = g & 7u;
    return x * q + (x < r ? x : r) + (b >> 3);
}

// ---------------------------------------------------------------------------
// Tensor access
// ---------------------------------------------------------------------------
template <typename Real>
struct KernelView {
    const Real *k = nullptr;  // octant tensor, nullptr for the projection fallback
    int kcomp = 6, kz_n = 1;
    KernLayout l;
    int ny = 0, nz = 0, py = 0, pz = 1, hx = 0;
    double kxs = 0, kys = 0, kzs = 0;  // 2 pi / (p d) per axis (projection)
};

// Position of oy within a row of the octant tensor (KernLayout): residue
// classes mod cls (a power of two) one after the other.
__host__ __device__ __forceinline__ int kern_y(const KernLayout &l, int oy) {
    return (oy & (l.cls - 1)) * l.yw + oy / l.cls;
}

// Entry (kx, oy, oz), component c of the octant tensor (KernLayout).
__host__ __device__ __forceinline__ int64_t kern_at(const KernLayout &l, int c, int oz, int kx, int oy) {
    return kx * l.skx + kern_y(l, oy) * l.soy + ((oz & 1) ? l.odd : 0) + (oz >> 1) * l.soz + c * l.sc;
}

// t = (xx, yy, zz, xy, xz, yz) at frequency (kx, ky, kz); kx <= nx.
template <typename Real>
__device__ __forceinline__ void tensor_at(const KernelView<Real> &K, int kx, int ky, int kz, Real t[6]) {
    if (K.k) {
        const bool ylo = ky <= K.ny;
        const int oy = ylo ? ky : K.py - ky;
        const Real sy = ylo ? Real(1) : Real(-1);
        int oz = 0;
        Real sz = Real(1);
        if (K.kz_n > 1) {
            const bool zlo = kz <= K.nz;
            oz = zlo ? kz : K.pz - kz;
            sz = zlo ? Real(1) : Real(-1);
        }
        const Real *e = K.k + kern_at(K.l, 0, oz, kx, oy);
        const int64_t sc = K.l.sc;
        t[0] = e[0];
        t[1] = e[sc];
        t[2] = e[2 * sc];
        t[3] = sy * e[3 * sc];
        if (K.kcomp == 6) {
            t[4] = sz * e[4 * sc];
            t[5] = sy * sz * e[5 * sc];
        } else {
            t[4] = Real(0);
            t[5] = Real(0);
        }
    } else {
        // native/backends/fdm/src/demag_fp64.cu:102-148: H(k) = -k (k.M) / k^2
        const int fy = ky <= K.py / 2 ? ky : ky - K.py;
        const int fz = kz <= K.pz / 2 ? kz : kz - K.pz;
        const double qx = kx * K.kxs, qy = fy * K.kys, qz = fz * K.kzs;
        const double q2 = qx * qx + qy * qy + qz * qz;
        if (q2 == 0.0) {
            for (int i = 0; i < 6; ++i) t[i] = Real(0);
            return;
        }
        const double r = 1.0 / q2;
        t[0] = Real(qx * qx * r); t[1] = Real(qy * qy * r); t[2] = Real(qz * qz * r);
        t[3] = Real(qx * qy * r); t[4] = Real(qx * qz * r); t[5] = Real(qy * qz * r);
    }
}

template <typename Real>
__device__ __forceinline__ void apply_tensor(const Real t[6], cplx<Real> &mx, cplx<Real> &my, cplx<Real> &mz) {
    const cplx<Real> X = mx, Y = my, Z = mz;
    mx = {-(t[0] * X.x + t[3] * Y.x + t[4] * Z.x), -(t[0] * X.y + t[3] * Y.y + t[4] * Z.y)};
    my = {-(t[3] * X.x + t[1] * Y.x + t[5] * Z.x), -(t[3] * X.y + t[1] * Y.y + t[5] * Z.y)};
    mz = {-(t[4] * X.x + t[5] * Y.x + t[2] * Z.x), -(t[4] * X.y + t[5] * Y.y + t[2] * Z.y)};
}

// ---------------------------------------------------------------------------
// Spectrum addressing: spec[c][z][kx][ky], `planes` z-planes, ky pitch.
// ---------------------------------------------------------------------------
struct SpecGeom {
    int hx;       // half-spectrum width px / 2 + 1, or px / 2 at the frequencies k + 1/2
    int planes;   // z planes stored
    int pitch;    // ky line length stored
    __device__ __host__ int64_t at(int c, int z, int kx, int ky) const {
        return (((int64_t)c * planes + z) * hx + kx) * pitch + ky;
    }
};

// ---------------------------------------------------------------------------
// x passes
// ---------------------------------------------------------------------------
template <typename Real>
struct XArgs {
    const cplx<Real> *tw;
    LinePlan lp;      // length px
    int xr, xr_log2;  // real rows per workgroup (power of two) and its log2
    int ls;           // LDS line stride (complex slots)
    int rows;         // valid real rows per (c, z) plane
    int n_in;         // forward: inputs loaded per row
    int n_out;        // inverse: outputs stored per row
    Real scale;       // inverse: 1/Npad
    // frequencies k + 1/2: exp(-i pi d / px) of the displacement d(x) (null: k),
    // and the same in FP64 for the inputs
    const cplx<Real> *sw;
    const cplx<double> *sw64;
    SpecGeom g;
};

// Ms m at (c, z, y, x) of the state; zero on inactive cells.  GATHER: the
// x pass reads the mask, volume fraction and per-cell Ms beside m with
// unconditional loads (a separate instantiation, so that the kernel for
// uniform material keeps its register budget).
template <typename Real, typename S, bool GATHER = false>
struct MagSource {
    const S *m;
    const uint8_t *mask;
    const double *ms_cell;
    double ms;
    int nx, ny, nz;
    int64_t n;
    // boundary tiers: every cell packs phi Ms m, mask or not (the volume
    // fraction in the field's precision)
    const Real *phi;
    __device__ double at(int c, int z, int y, int x) const {
        const int64_t i = ((int64_t)z * ny + y) * nx + x;
        if (phi) return double(m[(int64_t)c * n + i]) * (double(phi[i]) * (ms_cell ? ms_cell[i] : ms));
        if (mask && !mask[i]) return 0.0;
        const double w = ms_cell ? ms_cell[i] : ms;
        return double(m[(int64_t)c * n + i]) * w;
    }
    // The value with every load unconditional, so that a lane's loads all issue
    // before the first is used.  Without GATHER (no mask, no per-cell Ms) that is
    // one load; with it an absent array is read from a stand-in and its value
    // replaced after the load.
    __device__ double load(int c, int z, int y, int x) const {
        const int64_t i = ((int64_t)z * ny + y) * nx + x;
        const double mv = double(m[(int64_t)c * n + i]);
        if constexpr (!GATHER) return mv * ms;
        const double pv = double(*(phi ? phi + i : no_array<Real>()));
        const double cv = *(ms_cell ? ms_cell + i : &kNoArrayF64);
        const uint8_t kv = *(mask ? mask + i : &kNoMask);
        const double w = ms_cell ? cv : ms;
        const bool live = phi || kv != 0;
        return live ? mv * (phi ? pv * w : w) : 0.0;
    }
};

// Padded real-space Newell kernel at (c, z, y, x) of the (px, py, pz) grid,
// mirrored from the octant with the placement signs of
// crates/fullmag-fdm-demag/src/newell.rs:397-426 (the indices between the
// octant and its mirror image are never written there and stay zero).
struct NewellSource {
    const double *oct;  // [6][nz][ny][nx]
    int nx, ny, nz, px, py, pz;
    int z_even;  // the cross-layer kernel: mirrored z slots keep every sign (newell.rs:630-647)
    __device__ double at(int c, int zz, int yy, int x) const {
        if ((x >= nx && x <= px - nx) || (yy >= ny && yy <= py - ny) || (pz > 1 && zz >= nz && zz <= pz - nz))
            return 0.0;
        const int xi = x < nx ? x : px - x;
        const int yi = yy < ny ? yy : py - yy;
        const int zi = (pz == 1 || zz < nz) ? zz : pz - zz;
        const double sx = x < nx ? 1.0 : -1.0, sy = yy < ny ? 1.0 : -1.0;
        const double sz = (pz == 1 || zz < nz || z_even) ? 1.0 : -1.0;
        double s = 1.0;
        if (c == 3) s = sx * sy;
        else if (c == 4) s = sx * sz;
        else if (c == 5) s = sy * sz;
        return s * oct[(((int64_t)c * nz + zi) * ny + yi) * nx + xi];
    }
};

template <typename Real>
struct FieldSink {
    Real *out;
    const uint8_t *mask;
    int nx, ny;
    int64_t n;
    __device__ void operator()(int c, int z, int y, int x, Real v) const {
        const int64_t i = ((int64_t)z * ny + y) * nx + x;
        out[(int64_t)c * n + i] = (mask && !mask[i]) ? Real(0) : v;
    }
    // With a mask, operator() in two halves, so that a lane reads all its
    // mask bytes before its first store (a byte read may alias the stores,
    // so the compiler keeps each one behind the store before it).
    __device__ bool masked() const { return mask != nullptr; }
    __device__ uint8_t keep(int z, int y, int x) const { return mask[((int64_t)z * ny + y) * nx + x]; }
    __device__ void put(int c, int z, int y, int x, Real v, uint8_t keep) const {
        out[(int64_t)c * n + ((int64_t)z * ny + y) * nx + x] = keep ? v : Real(0);
    }
};

// ---------------------------------------------------------------------------
// Line passes and the thin-film y convolution
// ---------------------------------------------------------------------------
template <typename Real>
struct LineArgs {
    cplx<Real> *data;
    const cplx<Real> *tw;
    LinePlan lp;
    int64_t lines;      // number of lines
    int64_t line_pitch; // distance between consecutive lines
    int lpw;            // lines per workgroup
    int n_in, n_out;
    int inverse;
    int iters;          // line_pipe_kernel: line groups per workgroup
    const cplx<Real> *in;  // inverse from ky classes: rows of a class's entries after another's, in_pitch apart
    int64_t in_pitch;
};

// Thin film: per kx, the three components' ky lines (ny of 2ny inputs) are
// transformed, multiplied by the tensor at kz = 0, transformed back and the
// first ny outputs stored.
template <typename Real>
struct YConvArgs {
    cplx<Real> *data;
    const cplx<Real> *tw;
    LinePlan lp;  // length py
    int ny, hx, kpw;  // kx columns per workgroup
    SpecGeom g;
    KernelView<Real> K;
};

// Layers of a stack handed to one launch.
constexpr int kStackPack = 8;

// Ms m of up to kStackPack layers on the common grid (a mask where there is
// one), and where their fields go.
template <typename Real, typename S>
struct StackMag {
    const S *m[kStackPack];
    const uint8_t *mask[kStackPack];
    double ms[kStackPack];
    int nx, ny, nz;
    int64_t n;
    int64_t layer_stride;  // complex elements per layer spectrum
};
template <typename Real>
struct StackField {
    Real *out[kStackPack];
    const uint8_t *mask[kStackPack];
    int nx, ny;
    int64_t n;
    int64_t layer_stride;
};

// Thin stack of L <= kStackFused layers: per kx, the layers' 3 L ky lines are
// transformed, coupled by the pair kernels and transformed back in place.
constexpr int kStackFused = 5;
constexpr size_t kLdsMax = 163840;  // LDS of a CU, the most that a workgroup may take
// Whether `kpw` columns of L layers' scheduled lines fit a workgroup of `lds` bytes.
template <typename Real>
constexpr bool ystack_fits(int n, int L, int kpw = 1, size_t lds = kLdsMax) {
    return fx_has(n) && L <= kStackFused && 3 * L * fx_lanes(n) <= 1024 && lds <= kLdsMax &&
           (size_t)3 * L * kpw * fx_size(n) * sizeof(cplx<Real>) <= lds;
}
template <typename Real>
struct YStackArgs {
    cplx<Real> *data;       // [layer][c][kx][ky]
    const cplx<Real> *tw;
    const Real *kern;       // [kernel][kx][6][py / 2 + 1], the ky octant
    int ny, hx, kpw;        // kx columns per workgroup
    int kernel[kStackFused][kStackFused];  // of (dst, src)
};

// ---------------------------------------------------------------------------
// kx slabs: y transforms and z convolution together
// ---------------------------------------------------------------------------
template <typename Real>
struct SlabArgs {
    cplx<Real> *data;
    const cplx<Real> *tw, *twz;  // roots of lengths py and 2 nz
    int nz, ny, hx, pitch;
    int64_t plane_stride;        // between the (component, z) planes of the spectrum
    KernelView<Real> K;
    // ky classes (class_kernel): the x passes' spectrum, read, and the roots of
    // length py / kClasses
    const cplx<Real> *in, *twp;
    int in_pitch;
    int64_t in_plane;
};
// Residue classes of ky that class_kernel splits a slab into, and the padded y
// lengths it takes.
constexpr int kClasses = 4;
constexpr bool class_length(int n) {
    return n % kClasses == 0 && fx_has(n) && fx_lanes(n) >= 32 && fx_has(n / kClasses) && fx_lanes(n / kClasses) <= 16;
}
// Padded y lengths with a slab kernel: 24 lines of 32 lanes are 768.
constexpr bool slab_length(int n) { return fx_has(n) && fx_lanes(n) <= 32; }

// ---------------------------------------------------------------------------
// z passes
// ---------------------------------------------------------------------------
template <typename Real>
struct ZArgs {
    cplx<Real> *data;
    const cplx<Real> *tw;  // roots of length pz
    int nz, hx, py;
    int64_t columns;       // hx * pitch (pad columns ky >= py are skipped)
    int64_t zstride;       // hx * pitch (3-D demag layout)
    int64_t comp_stride;   // nz * hx * pitch
    int pitch;             // distance between kx rows of the spectrum (>= py)
    int xcd;               // renumber workgroups per XCD
    KernelView<Real> K;
};


// Long z lines: a workgroup holds `tile` consecutive columns (contiguous in
// ky) of all three components in LDS.  conv = 0: plain forward (or, with
// `inverse`, inverse) transform of one component (blockIdx.y = component),
// used by the Newell setup and the multilayer stack.
template <typename Real>
struct ZLdsArgs {
    cplx<Real> *data;
    const cplx<Real> *tw;
    LinePlan lp;      // length pz
    int n_in, n_out;
    int tile, conv;
    int inverse;  // conv = 0: the inverse transform (n_in = pz, n_out <= pz)
    int64_t columns, zstride, comp_stride;
    int py, pitch;
    int xcd;  // renumber workgroups per XCD
    KernelView<Real> K;
};

struct Timed {
    Context &c;
    int entry = -1;
    hipEvent_t ev{};
    Timed(Context &cc, const char *name) : c(cc) {
        if (c.timing) {
            entry = timing_entry(c, name);
            timing_begin(c, entry, &ev);
        }
    }
    ~Timed() {
        if (entry >= 0) timing_end(c, entry, ev);
    }
};

constexpr int scheduled_lengths() {
    int k = 0;
    for (int n = 1; n <= 4096; ++n) k += fx_has(n) ? 1 : 0;
    return k;
}

// Calls f(std::integral_constant<int, N>) with N the line length when `lp`
// has a compile-time schedule, else with N = 0 (runtime plan).
template <class F>
void with_line(const LinePlan &lp, F &&f) {
    static_assert(scheduled_lengths() == 26, "every length of fx_has is listed here");
    if (lp.fixed) {
        switch (lp.n) {
#define FM_LINE(N)                             \
    case N:                                    \
        static_assert(fx_has(N), "scheduled"); \
        f(std::integral_constant<int, N>{});   \
        return;
            FM_LINE(20) FM_LINE(24) FM_LINE(28) FM_LINE(32) FM_LINE(40) FM_LINE(48) FM_LINE(56) FM_LINE(64)
            FM_LINE(80) FM_LINE(96) FM_LINE(112) FM_LINE(128) FM_LINE(160) FM_LINE(192) FM_LINE(224) FM_LINE(256)
            FM_LINE(320) FM_LINE(384) FM_LINE(448) FM_LINE(512) FM_LINE(640) FM_LINE(768) FM_LINE(896)
            FM_LINE(1024) FM_LINE(2048) FM_LINE(4096)
#undef FM_LINE
            default: break;
        }
    }
    f(std::integral_constant<int, 0>{});
}

// ---------------------------------------------------------------------------
// Launches (recorded instead of issued while a batch records)
// ---------------------------------------------------------------------------
// demag_x.hip: x R2C of `src` into spec over `comps` components, and x C2R of
// spec into `sink`; grid (row groups, planes), dp supplies the geometry.
template <typename Real, class Src>
void launch_xfwd(Context &c, const XArgs<Real> &xa, const Src &src, cplx<Real> *spec, unsigned row_groups,
                 unsigned planes, unsigned comps, size_t lds);
template <typename Real>
void launch_xinv(Context &c, const XArgs<Real> &xa, const cplx<Real> *spec, const FieldSink<Real> &sink,
                 unsigned row_groups, unsigned planes, size_t lds);
// demag_y.hip: contiguous line passes, the thin-film y convolution and its
// split form's tensor pass.
template <typename Real>
void launch_lines(Context &c, const LinePlan &lp, LineArgs<Real> la);
template <typename Real>
void launch_yconv(Context &c, const YConvArgs<Real> &ya);
template <typename Real>
void launch_film_tensor(Context &c, cplx<Real> *spec, const KernelView<Real> &K, int hx, int py, int64_t rows);
// The stack's: x passes of `layers` <= kStackPack layers (spectra layer_stride
// apart), and the coupled y pass.
template <typename Real, typename S>
void launch_xfwd_stack(Context &c, const XArgs<Real> &xa, const StackMag<Real, S> &sm, bool masked, cplx<Real> *spec,
                       unsigned row_groups, unsigned planes, unsigned layers, size_t lds);
template <typename Real>
void launch_xinv_stack(Context &c, const XArgs<Real> &xa, const cplx<Real> *spec, const StackField<Real> &sf,
                       unsigned row_groups, unsigned planes, unsigned layers, size_t lds);
template <typename Real>
void launch_ystack(Context &c, const LinePlan &lp, int layers, const YStackArgs<Real> &ya);
// demag_s.hip: the slab kernel (slab_length(lp.n), 2 <= nz <= 8, a tensor).
template <typename Real>
void launch_slab(Context &c, const LinePlan &lp, const SlabArgs<Real> &sa);
template <typename Real>
void launch_class(Context &c, const LinePlan &lp, const SlabArgs<Real> &sa);
template <typename Real>
void launch_class_inverse(Context &c, const LinePlan &lp, const LineArgs<Real> &la);
// demag_z.hip: the register z convolution (pz <= 16) and the longer z lines
// (convolution, or plain transforms of `comps` components).
template <typename Real>
void launch_zreg(Context &c, const ZArgs<Real> &za);
template <typename Real>
void launch_zlds(Context &c, const ZLdsArgs<Real> &za, unsigned comps);

}  // namespace fm
