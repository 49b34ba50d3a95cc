// demag_z.hip -- z passes of the demag convolution: in registers for short
// lines, through LDS for long ones (see demag.hip for the pipeline).  Compiled
// once per field precision (FM_REAL).
#include "demag.hpp"

namespace fm {
namespace {

// Element `i` of an array whose base is uniform over the wavefront: the lane
// carries a 32-bit byte offset and the base stays in scalar registers.
template <typename T>
__device__ __forceinline__ T *lane_at(T *base, uint32_t i) {
    using B = typename std::conditional<std::is_const<T>::value, const char, char>::type;
    return reinterpret_cast<T *>(reinterpret_cast<B *>(base) + (uint32_t)(i * (uint32_t)sizeof(T)));
}

// V neighbouring columns, one 16-byte access.
template <typename Real, int V>
struct alignas(sizeof(cplx<Real>) * V) cvec {
    cplx<Real> c[V];
};

// Short z lines (pz = 2 NZ <= 16): one lane per (kx, ky) column, all three
// components in registers, no LDS and no barrier.  The NZ non-zero inputs of
// the padded line give the even kz = 2k as DFT_NZ(x)[k] and the odd
// kz = 2k + 1 as DFT_NZ(x_z w_pz^z)[k]; each half gets its tensor entries and
// is transformed back (the odd half times w_pz^-z), so only one half of the
// padded spectrum exists at a time and the input registers carry the odd
// half.  Consecutive lanes take consecutive columns, so every load and store
// is one contiguous run per wavefront, the tensor entries (oy fastest)
// included.  kz and pz - kz share an entry and, for kz > NZ, xz and yz change
// sign.  PROJ: the tensor is the k-space projection's, computed per kz.
// FP32 512x512x8: 52 us for 259 MB (5.0 TB/s), as much as the LDS-staged tile
// with two lanes per column took, a copy of the inputs straight to LDS (54 us)
// and one wavefront per component (57 us); 256x256x4 9.5 -> 7.9 us and
// 250x150x6 14.9 -> 10.9 us against that tile.
template <typename Real, int NZ, bool PROJ>
__device__ __forceinline__ void zreg_body(const ZArgs<Real> &a) {
    using C = cplx<Real>;
    constexpr int NE = NZ / 2 + 1, NO = (NZ + 1) / 2;  // octant entries of even and odd kz
    const uint32_t blk = a.xcd ? xcd_block(blockIdx.x, gridDim.x) : blockIdx.x;
    const uint32_t cl = blk * 256u + threadIdx.x;
    // a lane past the end repeats the last column: the kx of a wavefront's
    // lanes never falls below its first lane's (see kx0)
    const bool live = cl < a.columns;
    const uint32_t col = live ? cl : (uint32_t)a.columns - 1u;
    const int kx = (int)(col / (uint32_t)a.pitch), ky = (int)(col - (uint32_t)kx * (uint32_t)a.pitch);
    C x[3][NZ];
#pragma unroll
    for (int c = 0; c < 3; ++c)
#pragma unroll
        for (int z = 0; z < NZ; ++z) x[c][z] = *lane_at(a.data + c * a.comp_stride + z * a.zstride, col);
    const bool ylo = ky <= a.K.ny;
    const Real sy = ylo ? Real(1) : Real(-1);
    const int kx0 = __builtin_amdgcn_readfirstlane(kx);
    const Real *kb = a.K.k + kx0 * a.K.l.skx;
    const uint32_t ko = (uint32_t)((kx - kx0) * (int)a.K.l.skx + kern_y(a.K.l, ylo ? ky : a.py - ky));
    auto load = [&](Real (*t)[6], int n, int64_t off) {
#pragma unroll
        for (int i = 0; i < n; ++i)
#pragma unroll
            for (int q = 0; q < 6; ++q) t[i][q] = *lane_at(kb + off + i * a.K.l.soz + q * a.K.l.sc, ko);
    };
    // v = the kz = 2k + odd half; tensor, back to z
    auto half = [&](C (*v)[NZ], const Real (*t)[6], int odd) {
#pragma unroll
        for (int c = 0; c < 3; ++c) dft_any<Real, NZ>(v[c], a.tw, NZ, false);
#pragma unroll
        for (int k = 0; k < NZ; ++k) {
            const int kz = 2 * k + odd, i = (kz <= NZ ? kz : 2 * NZ - kz) >> 1;
            const Real sz = kz <= NZ ? Real(1) : Real(-1);
            Real tt[6];
            if constexpr (PROJ) {
                tensor_at(a.K, kx, ky, kz, tt);
            } else {
                tt[0] = t[i][0];
                tt[1] = t[i][1];
                tt[2] = t[i][2];
                tt[3] = sy * t[i][3];
                tt[4] = sz * t[i][4];
                tt[5] = sz * (sy * t[i][5]);
            }
            apply_tensor(tt, v[0][k], v[1][k], v[2][k]);
        }
#pragma unroll
        for (int c = 0; c < 3; ++c) dft_any<Real, NZ>(v[c], a.tw, NZ, true);
    };
    C y[3][NZ];
    {
        Real t[NE][6];
        if constexpr (!PROJ) load(t, NE, 0);
#pragma unroll
        for (int c = 0; c < 3; ++c)
#pragma unroll
            for (int z = 0; z < NZ; ++z) y[c][z] = x[c][z];
        half(y, t, 0);
    }
    {
        Real t[NO][6];
        if constexpr (!PROJ) load(t, NO, a.K.l.odd);
#pragma unroll
        for (int z = 1; z < NZ; ++z) {
            const C w = a.tw[z];
#pragma unroll
            for (int c = 0; c < 3; ++c) x[c][z] = cmul(x[c][z], w);
        }
        half(x, t, 1);
    }
#pragma unroll
    for (int z = 0; z < NZ; ++z) {
        const C w = cconj(a.tw[z]);
#pragma unroll
        for (int c = 0; c < 3; ++c) {
            const C o = cadd(y[c][z], z > 0 ? cmul(x[c][z], w) : x[c][z]);
            if (live) *lane_at(a.data + c * a.comp_stride + z * a.zstride, col) = o;
        }
    }
}

// The same in FP64 for NZ >= 3, where one column's three components take more
// registers than a lane has: one wavefront per component, so that two to four
// wavefronts share a SIMD.  The spectra of a half meet in LDS
// ([component][k][lane]): a wavefront reads the other two components and forms
// its own row of the tensor product.  The mirrored entries' signs go on the y
// and z vectors: xy and yz change with ky's mirror, xz and yz with kz's, which
// is the same as flipping y (z) before and after the product.
// 512x512x8: 157 us with four lanes per column and two shuffles per output,
// 177 us as zreg_body (one wavefront per SIMD), 109 us here (4.7 TB/s).
template <typename Real, int NZ>
__device__ __forceinline__ void zreg3_body(const ZArgs<Real> &a) {
    using C = cplx<Real>;
    constexpr int NE = NZ / 2 + 1;
    __shared__ C ex[3][NZ][64];
    const uint32_t blk = a.xcd ? xcd_block(blockIdx.x, gridDim.x) : blockIdx.x;
    const int lane = threadIdx.x & 63;
    const int c = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
    const uint32_t cl = blk * 64u + (uint32_t)lane;
    // a lane past the end repeats the last column: the kx of a wavefront's
    // lanes never falls below its first lane's (see kx0)
    const bool live = cl < a.columns;
    const uint32_t col = live ? cl : (uint32_t)a.columns - 1u;
    const int kx = (int)(col / (uint32_t)a.pitch), ky = (int)(col - (uint32_t)kx * (uint32_t)a.pitch);
    C *data = a.data + c * a.comp_stride;
    C x[NZ];
#pragma unroll
    for (int z = 0; z < NZ; ++z) x[z] = *lane_at(data + z * a.zstride, col);
    // this component's row of the tensor: its own entry, the next one's and
    // the one after
    const int e0 = c, e1 = c == 0 ? 3 : c == 1 ? 5 : 4, e2 = c == 0 ? 4 : c == 1 ? 3 : 5;
    const int c1 = c == 2 ? 0 : c + 1, c2 = c == 0 ? 2 : c - 1;
    const bool ylo = ky <= a.K.ny;
    const int kx0 = __builtin_amdgcn_readfirstlane(kx);
    const Real *kb = a.K.k + kx0 * a.K.l.skx;
    const uint32_t ko = (uint32_t)((kx - kx0) * (int)a.K.l.skx + kern_y(a.K.l, ylo ? ky : a.py - ky));
    const Real sy = ylo || c != 1 ? Real(1) : Real(-1), sz = c == 2 ? Real(-1) : Real(1);
    auto half = [&](C *v, int odd, int n, int64_t off) {
        Real t[NE][3];
#pragma unroll
        for (int i = 0; i < n; ++i) {
            const Real *p = kb + off + i * a.K.l.soz;
            t[i][0] = *lane_at(p + e0 * a.K.l.sc, ko);
            t[i][1] = *lane_at(p + e1 * a.K.l.sc, ko);
            t[i][2] = *lane_at(p + e2 * a.K.l.sc, ko);
        }
        dft_any<Real, NZ>(v, a.tw, NZ, false);
#pragma unroll
        for (int k = 0; k < NZ; ++k) {
            const Real g = 2 * k + odd <= NZ ? Real(1) : sz;
            ex[c][k][lane] = v[k] = {g * v[k].x, g * v[k].y};
        }
        __syncthreads();
#pragma unroll
        for (int k = 0; k < NZ; ++k) {
            const int kz = 2 * k + odd, i = (kz <= NZ ? kz : 2 * NZ - kz) >> 1;
            const Real g = kz <= NZ ? Real(-1) : -sz;
            const C p = ex[c1][k][lane], q = ex[c2][k][lane];
            v[k] = {g * (t[i][0] * v[k].x + t[i][1] * p.x + t[i][2] * q.x),
                    g * (t[i][0] * v[k].y + t[i][1] * p.y + t[i][2] * q.y)};
        }
        dft_any<Real, NZ>(v, a.tw, NZ, true);
    };
    C y[NZ];
#pragma unroll
    for (int z = 0; z < NZ; ++z) y[z] = x[z] = {sy * x[z].x, sy * x[z].y};
    half(y, 0, NE, 0);
#pragma unroll
    for (int z = 1; z < NZ; ++z) x[z] = cmul(x[z], a.tw[z]);
    __syncthreads();  // the even half's spectra have been read
    half(x, 1, (NZ + 1) / 2, a.K.l.odd);
#pragma unroll
    for (int z = 0; z < NZ; ++z) {
        const C o = cadd(y[z], z > 0 ? cmul(x[z], cconj(a.tw[z])) : x[z]);
        if (live) *lane_at(data + z * a.zstride, col) = {sy * o.x, sy * o.y};
    }
}
template <typename Real, int NZ>
__global__ void __launch_bounds__(192) zreg3_kernel(ZArgs<Real> a) {
    zreg3_body<Real, NZ>(a);
}
template <typename Real, int NZ>
__global__ void __launch_bounds__(192) zreg3_multi(const ZArgs<Real> *tab, int zdiv) {
    const ZArgs<Real> a = tab[blockIdx.z / zdiv];
    zreg3_body<Real, NZ>(a);
}

template <typename Real, int NZ, bool PROJ>
__global__ void __launch_bounds__(256) zreg_kernel(ZArgs<Real> a) {
    zreg_body<Real, NZ, PROJ>(a);
}
template <typename Real, int NZ>
__global__ void __launch_bounds__(256) zreg_multi(const ZArgs<Real> *tab, int zdiv) {
    const ZArgs<Real> a = tab[blockIdx.z / zdiv];
    zreg_body<Real, NZ, false>(a);
}

template <typename Real>
__global__ void __launch_bounds__(kMaxBlock) zlds_kernel(ZLdsArgs<Real> a) {
    extern __shared__ unsigned char smem_raw[];
    cplx<Real> *lds = reinterpret_cast<cplx<Real> *>(smem_raw);
    const int n = a.lp.n, ls = n + kPad, T = a.lp.threads;
    const int tid = threadIdx.x, nthr = blockDim.x;
    const int ncomp = a.conv ? 3 : 1;
    const int cbase = a.conv ? 0 : blockIdx.y;
    const int nslots = ncomp * a.tile;
    const int64_t col0 = (int64_t)blockIdx.x * a.tile;
    // batches of U loads per lane in flight before their LDS writes
    constexpr int U = 8;
    for (int base = tid; base < nslots * n; base += U * nthr) {
        cplx<Real> v[U];
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int idx = base + u * nthr;
            const int s = idx % nslots, e = idx / nslots;
            const int c = s / a.tile;
            const int64_t col = col0 + (s - c * a.tile);
            v[u] = {Real(0), Real(0)};
            if (idx < nslots * n && e < a.n_in && col < a.columns)
                v[u] = a.data[(cbase + c) * a.comp_stride + e * a.zstride + col];
        }
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int idx = base + u * nthr;
            if (idx < nslots * n) {
                const int s = idx % nslots, e = idx / nslots;
                lds[s * ls + lslot(a.lp, e)] = v[u];
            }
        }
    }
    __syncthreads();
    line_fft(lds + (tid / T) * ls, a.lp, tid % T, a.tw, !a.conv && a.inverse);
    __syncthreads();  // the tensor product and the stores cross lines
    if (a.conv) {
        // one pass per octant entry oz <= nz, applied at kz = oz and at its
        // mirror kz = pz - oz (xz and yz change sign): each tensor entry is
        // read once, as three 2-vector loads
        using V2 = typename std::conditional<sizeof(Real) == 4, float2, double2>::type;
        const int nzo = a.K.nz + 1;
        if (!a.K.k) {
            // k-space projection fallback: the tensor is computed per kz
            for (int idx = tid; idx < a.tile * n; idx += nthr) {
                const int j = idx % a.tile, e = idx / a.tile;
                const int64_t col = col0 + j;
                if (col >= a.columns) continue;
                const int kx = (int)(col / a.pitch), ky = (int)(col - (int64_t)kx * a.pitch);
                if (ky >= a.py) continue;
                Real t[6];
                tensor_at(a.K, kx, ky, e, t);
                const int se = lslot(a.lp, e);
                apply_tensor(t, lds[j * ls + se], lds[(a.tile + j) * ls + se], lds[(2 * a.tile + j) * ls + se]);
            }
        }
        for (int idx = tid; a.K.k && idx < a.tile * nzo; idx += nthr) {
            const int j = idx % a.tile, oz = idx / a.tile;
            const int64_t col = col0 + j;
            if (col >= a.columns) continue;
            const int kx = (int)(col / a.pitch), ky = (int)(col - (int64_t)kx * a.pitch);
            if (ky >= a.py) continue;
            const bool ylo = ky <= a.K.ny;
            const int oy = ylo ? ky : a.py - ky;
            const Real sy = ylo ? Real(1) : Real(-1);
            const V2 *e = reinterpret_cast<const V2 *>(a.K.k + kern_at(a.K.l, 0, oz, kx, oy));
            const V2 t01 = e[0], t23 = e[1], t45 = e[2];
            Real t[6] = {t01.x, t01.y, t23.x, sy * t23.y, t45.x, sy * t45.y};
            int se = lslot(a.lp, oz);
            apply_tensor(t, lds[j * ls + se], lds[(a.tile + j) * ls + se], lds[(2 * a.tile + j) * ls + se]);
            if (oz > 0 && oz < a.K.pz - oz) {
                t[4] = -t[4];
                t[5] = -t[5];
                se = lslot(a.lp, a.K.pz - oz);
                apply_tensor(t, lds[j * ls + se], lds[(a.tile + j) * ls + se], lds[(2 * a.tile + j) * ls + se]);
            }
        }
        __syncthreads();
        line_fft(lds + (tid / T) * ls, a.lp, tid % T, a.tw, true);
        __syncthreads();
    }
    for (int idx = tid; idx < nslots * a.n_out; idx += nthr) {
        const int s = idx % nslots, e = idx / nslots;
        const int c = s / a.tile;
        const int64_t col = col0 + (s - c * a.tile);
        if (col < a.columns) a.data[(cbase + c) * a.comp_stride + e * a.zstride + col] = lds[s * ls + lslot(a.lp, e)];
    }
}

// Long z lines of a scheduled length N with at most 64 lanes, C = 64 / T
// groups of V columns per wavefront.  Lane (t, g) = (lane / C, lane % C) holds
// elements t + e T of the V columns of group g, so a load instruction covers
// runs of C V consecutive columns (128 bytes for up to 128 z planes), and
// what it loads are the first pass's inputs: no index is divided and nothing
// is staged before the transform.  One wavefront per component, lines
// interleaved in LDS as [slot][group] with the V columns in one 16-byte
// access, so a pass needs no workgroup barrier and the twiddles serve V
// columns.  CONV: each tensor entry oz is loaded (beside the columns, before
// the transform) once per column and applied at kz = oz and pz - oz between
// two barriers; the inverse transform's last pass stores straight to memory.
// Bound by VALU work (about half of it butterflies; issued in 62 % of the SIMDs'
// cycles of the launch below) and by memory latency at nine wavefronts per CU
// (1.9 per SIMD on average).  256x256x64 mixed (257x512 columns of 128, 507 MB):
// 213 us with the staged lines of zlds_kernel, 131 us here, 147 us with one
// column per lane (twice the wavefronts, but each pays its own twiddles and
// 64-byte runs).  100^3 FP64: 214 -> 109 us.

// v[s][r] *= w^(r st) for the V columns s (see twiddle()).
template <typename T, int R, int V>
__device__ __forceinline__ void twiddle_cols(cplx<T> v[V][R], const cplx<T> *tw, int st, bool inv) {
    constexpr int LB = R == 2 ? 1 : R == 4 ? 2 : R == 8 ? 3 : 4;
    static_assert((1 << LB) == R, "power-of-two radix");
    const T sg = inv ? T(-1) : T(1);
    cplx<T> pw[LB], w[R];
#pragma unroll
    for (int b = 0; b < LB; ++b) {
        pw[b] = tw[st << b];
        pw[b].y *= sg;
    }
#pragma unroll
    for (int r = 1; r < R; ++r) {
        const int low = r & -r;
        const int lb = low == 1 ? 0 : low == 2 ? 1 : low == 4 ? 2 : 3;
        w[r] = r == low ? pw[lb] : cmul(w[r - low], pw[lb]);
#pragma unroll
        for (int s = 0; s < V; ++s) v[s][r] = cmul(v[s][r], w[r]);
    }
}

// One pass (see fx_pass) over the lane's V columns; `put(i, q)` takes output
// element i instead of LDS when LAST.
template <typename T, int N, int R, int NS, int V, int C, bool LAST, class Put>
__device__ __forceinline__ void col_pass(cvec<T, V> *l, int t, const cplx<T> *tw, bool inv, Put &&put) {
    constexpr int G = fx_pad(N), NT = fx_lanes(N), NR = N / R, ST = N / (NS * R);
    constexpr int MB = (NR + NT - 1) / NT;
    constexpr bool FULL = MB * NT == NR;
    cplx<T> v[MB][V][R];
    int base[MB];
#pragma unroll
    for (int b = 0; b < MB; ++b) {
        const int j0 = t + b * NT, j = FULL || j0 < NR ? j0 : 0, k = j % NS;
        const cvec<T, V> *p = l + fxslot<N>(j) * C;
#pragma unroll
        for (int r = 0; r < R; ++r) {
            const cvec<T, V> q = p[r * (NR + NR / G) * C];
#pragma unroll
            for (int s = 0; s < V; ++s) v[b][s][r] = q.c[s];
        }
        twiddle_cols<T, R, V>(v[b], tw, k * ST, inv);
#pragma unroll
        for (int s = 0; s < V; ++s) dft_any<T, R>(v[b][s], tw, N, inv);
        base[b] = (j / NS) * NS * R + k;
    }
    if constexpr (!LAST) pass_sync<N>();
#pragma unroll
    for (int b = 0; b < MB; ++b)
        if (FULL || t + b * NT < NR)
#pragma unroll
            for (int r = 0; r < R; ++r) {
                cvec<T, V> q;
#pragma unroll
                for (int s = 0; s < V; ++s) q.c[s] = v[b][s][r];
                if constexpr (LAST) put(base[b] + r * NS, q);
                else l[(fxslot<N>(base[b]) + r * (NS + NS / G)) * C] = q;
            }
    if constexpr (!LAST) pass_sync<N>();
}

// The first pass, from registers (see fx_first_pass).
template <typename T, int N, int V, int C>
__device__ __forceinline__ void col_first(cvec<T, V> *l, int t, const cplx<T> (*v)[fx_elems(N)], const cplx<T> *tw,
                                          bool inv) {
    constexpr int R = fx_radix(N, 0), B = fx_elems(N) / R, NT = fx_lanes(N);
#pragma unroll
    for (int b = 0; b < B; ++b) {
        cplx<T> u[V][R];
#pragma unroll
        for (int s = 0; s < V; ++s) {
#pragma unroll
            for (int r = 0; r < R; ++r) u[s][r] = v[s][b + r * B];
            dft_any<T, R>(u[s], tw, N, inv);
        }
#pragma unroll
        for (int r = 0; r < R; ++r) {
            cvec<T, V> q;
#pragma unroll
            for (int s = 0; s < V; ++s) q.c[s] = u[s][r];
            l[((t + b * NT) * (R + 1) + r) * C] = q;
        }
    }
    pass_sync<N>();
}

// Passes P.. of the schedule, the last through `put` when STORE.
template <typename T, int N, int P, int NS, int V, int C, bool STORE, class Put>
__device__ __forceinline__ void col_passes(cvec<T, V> *l, int t, const cplx<T> *tw, bool inv, Put &&put) {
    if constexpr (P < fx_npass(N)) {
        constexpr int R = fx_radix(N, P);
        col_pass<T, N, R, NS, V, C, STORE && P + 1 == fx_npass(N)>(l, t, tw, inv, put);
        col_passes<T, N, P + 1, NS * R, V, C, STORE>(l, t, tw, inv, put);
    }
}

template <int N>
constexpr bool zcol_has() {
    return N > 16 && fx_lanes(N) <= 64 && fx_npass(N) > 1;
}
// columns per lane: as many as fill a 16-byte access
template <typename Real>
constexpr int zcol_v() {
    return sizeof(Real) == 4 ? 2 : 1;
}

template <typename Real, int N, int V, bool CONV>
__global__ void __launch_bounds__(CONV ? 192 : 64) zcol_kernel(ZLdsArgs<Real> a) {
    using Cx = cplx<Real>;
    using Cv = cvec<Real, V>;
    constexpr int T = fx_lanes(N), E = fx_elems(N), C = 64 / T, NZO = N / 2 + 1;
    __shared__ Cv lds[CONV ? 3 : 1][fx_size(N) * C];
    const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
    const int g = lane % C, t = lane / C;
    const int comp = CONV ? w : (int)blockIdx.y;
    const uint32_t blk = a.xcd ? xcd_block(blockIdx.x, gridDim.x) : blockIdx.x;
    const int64_t col = ((int64_t)blk * C + g) * V;  // columns is even: a group is all in or all out
    const bool live = col < a.columns;
    Cx *data = a.data + comp * a.comp_stride + (live ? col : 0);
    Cv *l = lds[CONV ? w : 0] + g;
    const auto none = [](int, const Cv &) {};
    const auto store = [&](int i, const Cv &q) {
        if (live && i < a.n_out) *reinterpret_cast<Cv *>(data + i * a.zstride) = q;
    };
    {
        Cx v[V][E];
        const bool half = 2 * a.n_in <= N;
#pragma unroll
        for (int e = 0; e < E; ++e) {
            const int i = t + e * T;
            Cv q{};
            if (e < E / 2 || !half) {
                q = *reinterpret_cast<const Cv *>(data + (i < a.n_in ? i : 0) * a.zstride);
                if (i >= a.n_in) q = Cv{};
            }
#pragma unroll
            for (int s = 0; s < V; ++s) v[s][e] = q.c[s];
        }
        col_first<Real, N, V, C>(l, t, v, a.tw, !CONV && a.inverse);
    }
    if constexpr (!CONV) {
        col_passes<Real, N, 1, fx_radix(N, 0), V, C, true>(l, t, a.tw, a.inverse != 0, store);
    } else {
        // item tid + 192 u: entry oz = item / C of column group item % C
        constexpr int NU = (C * NZO + 191) / 192;
        constexpr int H = 3;  // 2-vectors per entry
        using V2 = typename std::conditional<sizeof(Real) == 4, float2, double2>::type;
        V2 k[NU][V][H];
#pragma unroll
        for (int u = 0; u < NU; ++u) {
            const int item = tid + 192 * u, oz = item < C * NZO ? item / C : 0;
            const int64_t cc = ((int64_t)blk * C + item % C) * V;
            const int64_t c0 = cc < a.columns ? cc : 0;
            const int kx = (int)((uint32_t)c0 / (uint32_t)a.pitch), ky = (int)((uint32_t)c0 % (uint32_t)a.pitch);
#pragma unroll
            for (int s = 0; s < V; ++s) {
                const int oy = ky + s <= a.K.ny ? ky + s : a.py - ky - s;
                const V2 *p = reinterpret_cast<const V2 *>(a.K.k + kern_at(a.K.l, 0, oz, kx, oy));
#pragma unroll
                for (int q = 0; q < H; ++q) k[u][s][q] = p[q];
            }
        }
        col_passes<Real, N, 1, fx_radix(N, 0), V, C, false>(l, t, a.tw, false, none);
        __syncthreads();
#pragma unroll
        for (int u = 0; u < NU; ++u) {
            const int item = tid + 192 * u;
            if (item < C * NZO) {
                const int oz = item / C, gi = item % C;
                const int64_t cc = ((int64_t)blk * C + gi) * V;
                const int ky = (int)((uint32_t)cc % (uint32_t)a.pitch);
                auto apply = [&](int kz, Real sz) {
                    const int at = fxslot<N>(kz) * C + gi;
                    Cv x = lds[0][at], y = lds[1][at], z = lds[2][at];
#pragma unroll
                    for (int s = 0; s < V; ++s) {
                        const Real sy = ky + s <= a.K.ny ? Real(1) : Real(-1);
                        const Real tt[6] = {k[u][s][0].x,      k[u][s][0].y,      k[u][s][1].x,
                                            sy * k[u][s][1].y, sz * k[u][s][2].x, sy * sz * k[u][s][2].y};
                        apply_tensor(tt, x.c[s], y.c[s], z.c[s]);
                    }
                    lds[0][at] = x;
                    lds[1][at] = y;
                    lds[2][at] = z;
                };
                apply(oz, Real(1));
                if (oz > 0 && oz < N - oz) apply(N - oz, Real(-1));
            }
        }
        __syncthreads();
        Cx v[V][E];
#pragma unroll
        for (int e = 0; e < E; ++e) {
            const Cv q = l[fxslot<N>(t + e * T) * C];
#pragma unroll
            for (int s = 0; s < V; ++s) v[s][e] = q.c[s];
        }
        pass_sync<N>();
        col_first<Real, N, V, C>(l, t, v, a.tw, true);
        col_passes<Real, N, 1, fx_radix(N, 0), V, C, true>(l, t, a.tw, true, store);
    }
}

}  // namespace

template <typename Real>
void launch_zreg(Context &c, const ZArgs<Real> &za) {
    const dim3 grid((unsigned)cdiv(za.columns, 256)), block(256);
    auto launch = [&](auto NZC) {
        constexpr int NZ = decltype(NZC)::value;
        const bool proj = !za.K.k;
        if constexpr (sizeof(Real) == 8 && NZ >= 3) {
            if (!proj) {
                const dim3 g3((unsigned)cdiv(za.columns, 64));
                launch_rec(c, reinterpret_cast<const void *>(&zreg3_multi<Real, NZ>), g3, dim3(192), 0, 1, za, [&] {
                    hipLaunchKernelGGL((zreg3_kernel<Real, NZ>), g3, dim3(192), 0, c.stream, za);
                });
                return;
            }
        }
        launch_rec(c, proj ? nullptr : reinterpret_cast<const void *>(&zreg_multi<Real, NZ>), grid, block, 0, 1, za, [&] {
            if (proj) hipLaunchKernelGGL((zreg_kernel<Real, NZ, true>), grid, block, 0, c.stream, za);
            else hipLaunchKernelGGL((zreg_kernel<Real, NZ, false>), grid, block, 0, c.stream, za);
        });
    };
    switch (za.nz) {
        case 1: launch(std::integral_constant<int, 1>{}); break;
        case 2: launch(std::integral_constant<int, 2>{}); break;
        case 3: launch(std::integral_constant<int, 3>{}); break;
        case 4: launch(std::integral_constant<int, 4>{}); break;
        case 5: launch(std::integral_constant<int, 5>{}); break;
        case 6: launch(std::integral_constant<int, 6>{}); break;
        case 7: launch(std::integral_constant<int, 7>{}); break;
        default: launch(std::integral_constant<int, 8>{}); break;
    }
}

template <typename Real>
void launch_zlds(Context &c, const ZLdsArgs<Real> &za, unsigned comps) {
    with_line(za.lp, [&](auto NC) {
        constexpr int N = decltype(NC)::value;
        if constexpr (zcol_has<N>()) {
            constexpr int V = zcol_v<Real>(), C = 64 / fx_lanes(N);
            const dim3 g((unsigned)cdiv(za.columns, C * V), comps);
            launch_rec(c, nullptr, g, dim3(za.conv ? 192 : 64), 0, 1, za, [&] {
                if (za.conv) hipLaunchKernelGGL((zcol_kernel<Real, N, V, true>), g, dim3(192), 0, c.stream, za);
                else hipLaunchKernelGGL((zcol_kernel<Real, N, V, false>), g, dim3(64), 0, c.stream, za);
            });
        } else {
            const int slots = (za.conv ? 3 : 1) * za.tile;
            const dim3 grid((unsigned)cdiv(za.columns, za.tile), comps), block((unsigned)(slots * za.lp.threads));
            const size_t lds = (size_t)slots * (za.lp.n + kPad) * sizeof(cplx<Real>);
            launch_rec(c, nullptr, grid, block, lds, 1, za, [&] {
                hipLaunchKernelGGL((zlds_kernel<Real>), grid, block, lds, c.stream, za);
            });
        }
    });
}

using R = FM_REAL;
template void launch_zreg<R>(Context &, const ZArgs<R> &);
template void launch_zlds<R>(Context &, const ZLdsArgs<R> &, unsigned);

}  // namespace fm
