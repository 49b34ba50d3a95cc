// demag_z.hip -- z passes of the demag convolution: in registers for short
// lines, through LDS for long ones (see demag.hip for the pipeline).  Compiled
// once per field precision (FM_REAL).
#include "demag.hpp"

namespace fm {
namespace {

// DFT of length N on registers with roots w_N^t = w_P^(S t) taken from the
// length-P = S N table (power-of-two N uses exact constants).
template <typename Real, int N, int S>
__device__ __forceinline__ void strided_dft(cplx<Real> *v, const cplx<Real> *tw_p, bool inv) {
    if constexpr (N == 1) {
        (void)v; (void)tw_p; (void)inv;
    } else if constexpr (N == 2 || N == 4 || N == 8 || N == 16) {
        dft_any<Real, N>(v, tw_p, N, inv);
    } else {
        cplx<Real> out[N];
#pragma unroll
        for (int q = 0; q < N; ++q) {
            cplx<Real> acc = v[0];
#pragma unroll
            for (int r = 1; r < N; ++r) {
                cplx<Real> w = tw_p[S * ((r * q) % N)];
                if (inv) w.y = -w.y;
                acc = cadd(acc, cmul(v[r], w));
            }
            out[q] = acc;
        }
#pragma unroll
        for (int q = 0; q < N; ++q) v[q] = out[q];
    }
}

template <typename Real, int N>
__device__ __forceinline__ void half_dft(cplx<Real> *v, const cplx<Real> *tw_p, bool inv) {
    if constexpr (N == 1) {
        (void)v; (void)tw_p; (void)inv;
    } else if constexpr (N == 2 || N == 4 || N == 8 || N == 16) {
        dft_any<Real, N>(v, tw_p, N, inv);
    } else {
        cplx<Real> out[N];
#pragma unroll
        for (int q = 0; q < N; ++q) {
            cplx<Real> acc = v[0];
#pragma unroll
            for (int r = 1; r < N; ++r) {
                cplx<Real> w = tw_p[2 * ((r * q) % N)];
                if (inv) w.y = -w.y;
                acc = cadd(acc, cmul(v[r], w));
            }
            out[q] = acc;
        }
#pragma unroll
        for (int q = 0; q < N; ++q) v[q] = out[q];
    }
}

// z convolution with two lanes per (kx, ky) column (pz = 2 NZ): lane parity p
// owns kz = 2k + p.  Forward: X[2k+p] = DFT_NZ(x_z w_pz^(p z))[k] (only the
// NZ non-zero inputs exist); tensor at its own kz; inverse:
// y_z = IDFT_NZ(Y_even)[z] + w_pz^(-z) IDFT_NZ(Y_odd)[z], z < NZ, summed
// across the lane pair with a shuffle.  All three components in registers.
// Consecutive lane pairs take consecutive columns.  Used where the staged
// tile does not apply (the k-space projection fallback).
template <typename Real, int NZ>
__global__ void __launch_bounds__(256) zconv_pair_kernel(ZArgs<Real> a) {
    const int64_t gid = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    const int p = (int)(gid & 1);
    // both lanes of a pair stay for the shuffle
    const int64_t col = gid >> 1;
    bool valid = col < a.columns;
    const int kx = valid ? (int)(col / a.pitch) : 0;
    const int ky = valid ? (int)(col - (int64_t)kx * a.pitch) : 0;
    valid = valid && ky < a.py;
    cplx<Real> v[3][NZ];
#pragma unroll
    for (int c = 0; c < 3; ++c) {
#pragma unroll
        for (int z = 0; z < NZ; ++z) {
            cplx<Real> x = {Real(0), Real(0)};
            if (valid) x = a.data[c * a.comp_stride + z * a.zstride + col];
            if (p && z) x = cmul(x, a.tw[z]);
            v[c][z] = x;
        }
        half_dft<Real, NZ>(v[c], a.tw, false);
    }
#pragma unroll
    for (int k = 0; k < NZ; ++k) {
        Real t[6];
        tensor_at(a.K, kx, ky, 2 * k + p, t);
        apply_tensor(t, v[0][k], v[1][k], v[2][k]);
    }
#pragma unroll
    for (int c = 0; c < 3; ++c) {
        half_dft<Real, NZ>(v[c], a.tw, true);
#pragma unroll
        for (int z = 0; z < NZ; ++z) {
            cplx<Real> y = v[c][z];
            if (p && z) y = cmul(y, cconj(a.tw[z]));
            const cplx<Real> o = {__shfl_xor(y.x, 1), __shfl_xor(y.y, 1)};
            v[c][z] = cadd(y, o);
        }
    }
    if (!valid) return;
#pragma unroll
    for (int c = 0; c < 3; ++c)
#pragma unroll
        for (int z = 0; z < NZ; ++z)
            if ((z & 1) == p) a.data[c * a.comp_stride + z * a.zstride + col] = v[c][z];
}

// The two-lane z convolution staged through LDS: a workgroup of 256 lanes
// owns 128 consecutive columns.  It loads the tile's 3 NZ rows of 128
// complex values (one row = one (component, z) plane segment) with 16-byte
// loads, all issued before any arithmetic; lane pair j computes column j
// from LDS exactly as zconv_pair_kernel does; the results go back through
// LDS and out with 16-byte stores.  The tile's whole input is in flight at
// once and no lane keeps loaded data in registers across the transform.
constexpr int kZTile = 128;

// Tile of kZTile consecutive columns starting at col0: 3 NZ rows, each row
// one contiguous run of the spectrum.  Lane t moves 16-byte units t + 256 i.
template <typename Real, int NZ, int TW = kZTile>
struct ZTile {
    using C = cplx<Real>;
    static constexpr int ROWS = 3 * NZ;
    static constexpr int V = sizeof(Real) == 4 ? 2 : 1;  // complex values per 16-byte access
    static constexpr int UNITS = TW / V;                 // accesses per row
    static constexpr int PER = (ROWS * UNITS + 255) / 256;
    C v[PER][V];

    __device__ __forceinline__ void fetch(const ZArgs<Real> &a, int64_t col0, int t) {
        if (col0 + TW <= a.columns) {
            // the whole tile lies inside the spectrum (every tile but possibly
            // the last): unconditional 16-byte loads, all issued before any
            // wait; a lane's unit past the tile re-reads the tile's last unit
            // and put() drops it
#pragma unroll
            for (int i = 0; i < PER; ++i) {
                const int idx = min(t + 256 * i, ROWS * UNITS - 1);
                const int r = idx / UNITS, u = idx - r * UNITS;
                const int c = r / NZ, z = r - c * NZ;
                const C *src = a.data + c * a.comp_stride + z * a.zstride + col0 + (int64_t)u * V;
                if constexpr (V == 2) {
                    const float4 q = *reinterpret_cast<const float4 *>(src);
                    v[i][0] = C{Real(q.x), Real(q.y)};
                    v[i][1] = C{Real(q.z), Real(q.w)};
                } else {
                    v[i][0] = *src;
                }
            }
            return;
        }
#pragma unroll
        for (int i = 0; i < PER; ++i) {
            const int idx = t + 256 * i;
#pragma unroll
            for (int e = 0; e < V; ++e) v[i][e] = C{Real(0), Real(0)};
            if (idx < ROWS * UNITS) {
                const int r = idx / UNITS, u = idx - r * UNITS;
                const int c = r / NZ, z = r - c * NZ;
                const int64_t col = col0 + (int64_t)u * V;
                const C *src = a.data + c * a.comp_stride + z * a.zstride + col;
                if (col + V <= a.columns) {
                    if constexpr (V == 2) {
                        const float4 q = *reinterpret_cast<const float4 *>(src);
                        v[i][0] = C{Real(q.x), Real(q.y)};
                        v[i][1] = C{Real(q.z), Real(q.w)};
                    } else {
                        v[i][0] = *src;
                    }
                } else {
                    for (int e = 0; e < V; ++e)
                        if (col + e < a.columns) v[i][e] = src[e];
                }
            }
        }
    }
    __device__ __forceinline__ void put(C (*tile)[TW + V], int t) const {
#pragma unroll
        for (int i = 0; i < PER; ++i) {
            const int idx = t + 256 * i;
            if (idx < ROWS * UNITS) {
                const int r = idx / UNITS, u = idx - r * UNITS;
#pragma unroll
                for (int e = 0; e < V; ++e) tile[r][u * V + e] = v[i][e];
            }
        }
    }
};

template <typename Real, int NZ, int TW = kZTile>
__device__ __forceinline__ void ztile_store(const ZArgs<Real> &a, cplx<Real> (*tile)[TW + ZTile<Real, NZ, TW>::V],
                                            int64_t col0, int t) {
    using C = cplx<Real>;
    using TL = ZTile<Real, NZ, TW>;
    constexpr int V = TL::V, UNITS = TL::UNITS;
#pragma unroll
    for (int i = 0; i < TL::PER; ++i) {
        const int idx = t + 256 * i;
        if (idx < TL::ROWS * UNITS) {
            const int r = idx / UNITS, u = idx - r * UNITS;
            const int c = r / NZ, z = r - c * NZ;
            const int64_t cl = col0 + (int64_t)u * V;
            C *dst = a.data + c * a.comp_stride + z * a.zstride + cl;
            if (cl + V <= a.columns) {
                if constexpr (V == 2) {
                    const C e0 = tile[r][u * 2], e1 = tile[r][u * 2 + 1];
                    *reinterpret_cast<float4 *>(dst) = float4{float(e0.x), float(e0.y), float(e1.x), float(e1.y)};
                } else {
                    *dst = tile[r][u];
                }
            } else {
                for (int e = 0; e < V; ++e)
                    if (cl + e < a.columns) dst[e] = tile[r][u * V + e];
            }
        }
    }
}

// The lane's half of its column's octant tensor block (the entries of its
// kz parity, six components each), in registers.  Issued at the start of the
// tile kernel together with the tile's loads, so one memory wait covers both.
// Pad columns and the projection fallback keep zeros.
// FP64 keeps only the block's address (30 doubles would double the
// registers) and reads each entry where it is applied.
template <typename Real, int NZ>
struct ZTensorRegs {
    static constexpr int NE = NZ / 2 + 1, NO = (NZ + 1) / 2;
    static constexpr bool REGS = sizeof(Real) == 4;
    static constexpr int NV = (6 * NE + 3) / 4;  // 16-byte loads of the longer (even) half
    Real k[REGS ? NV * 4 : 1];
    const Real *blk = nullptr;
    bool valid = false;
    __device__ __forceinline__ void load(const ZArgs<Real> &a, bool col_valid, int kx, int ky, int p) {
        valid = col_valid && a.K.k;
        const int oy = ky <= a.K.ny ? ky : a.py - ky;
        blk = valid ? a.K.k + kern_at(a.K.l, 0, p, kx, oy) : a.K.k;
        if constexpr (REGS) {
#pragma unroll
            for (int e = 0; e < NV * 4; ++e) k[e] = Real(0);
            if (!valid) return;
            const float4 *src = reinterpret_cast<const float4 *>(blk);
            const int nv = p ? (6 * NO + 3) / 4 : NV;
#pragma unroll
            for (int e = 0; e < NV; ++e) {
                if (e < nv) {
                    const float4 q = src[e];
                    k[4 * e] = q.x;
                    k[4 * e + 1] = q.y;
                    k[4 * e + 2] = q.z;
                    k[4 * e + 3] = q.w;
                }
            }
        }
    }
};

// The register convolution of one column of the tile (two lanes per column,
// as zconv_pair_kernel), in place in LDS: lane pair t/2 takes column t/2.  A
// column is read and written only by its own lane pair, which sits in one
// wave, so no barrier separates the reads from the writes.
template <typename Real, int NZ, int TW = kZTile>
__device__ __forceinline__ void ztile_convolve(const ZArgs<Real> &a, cplx<Real> (*tile)[TW + ZTile<Real, NZ, TW>::V],
                                               int j, int p, int ky, const ZTensorRegs<Real, NZ> &kr) {
    using C = cplx<Real>;
    C v[3][NZ];
#pragma unroll
    for (int c = 0; c < 3; ++c) {
#pragma unroll
        for (int z = 0; z < NZ; ++z) {
            C x = tile[c * NZ + z][j];
            if (p && z) x = cmul(x, a.tw[z]);
            v[c][z] = x;
        }
        half_dft<Real, NZ>(v[c], a.tw, false);
    }
    const Real sy = ky <= a.K.ny ? Real(1) : Real(-1);
#pragma unroll
    for (int k = 0; k < NZ; ++k) {
        // lane parity p owns kz = 2k + p; its octant entry is (kz or pz - kz) / 2
        const int kz0 = 2 * k, kz1 = 2 * k + 1;
        const int i0 = (kz0 <= NZ ? kz0 : 2 * NZ - kz0) >> 1, i1 = (kz1 <= NZ ? kz1 : 2 * NZ - kz1) >> 1;
        const Real s0 = kz0 <= NZ ? Real(1) : Real(-1), s1 = kz1 <= NZ ? Real(1) : Real(-1);
        const Real sz = p ? s1 : s0;
        Real tt[6];
        if constexpr (sizeof(Real) == 4) {
            // select between two fixed registers with a bit mask (an index
            // chosen at run time would move the array to scratch)
            const uint32_t msk = 0u - (uint32_t)p;
#pragma unroll
            for (int q = 0; q < 6; ++q) {
                const uint32_t b0 = __float_as_uint(kr.k[6 * i0 + q]), b1 = __float_as_uint(kr.k[6 * i1 + q]);
                tt[q] = __uint_as_float((b0 & ~msk) | (b1 & msk));
            }
        } else {
            const Real *e = kr.blk + 6 * (p ? i1 : i0);
#pragma unroll
            for (int q = 0; q < 6; ++q) tt[q] = kr.valid ? e[q] : Real(0);
        }
        tt[3] = sy * tt[3];
        tt[4] = sz * tt[4];
        tt[5] = sy * sz * tt[5];
        apply_tensor(tt, v[0][k], v[1][k], v[2][k]);
    }
#pragma unroll
    for (int c = 0; c < 3; ++c) {
        half_dft<Real, NZ>(v[c], a.tw, true);
#pragma unroll
        for (int z = 0; z < NZ; ++z) {
            C y = v[c][z];
            if (p && z) y = cmul(y, cconj(a.tw[z]));
            const C o = {__shfl_xor(y.x, 1), __shfl_xor(y.y, 1)};
            if ((z & 1) == p) tile[c * NZ + z][j] = cadd(y, o);
        }
    }
}

template <typename Real, int NZ, int TW>
__device__ __forceinline__ void zconv_tile_body(const ZArgs<Real> &a) {
    static_assert(TW == 128, "one column per lane pair of a 256-lane workgroup");
    using TL = ZTile<Real, NZ, TW>;
    __shared__ cplx<Real> tile[TL::ROWS][TW + TL::V];
    const uint32_t blk = a.xcd ? xcd_block(blockIdx.x, gridDim.x) : blockIdx.x;
    const int64_t col0 = (int64_t)blk * TW;
    const int t = (int)threadIdx.x;
    const int j = t >> 1, p = t & 1;
    const int64_t col = col0 + j;
    bool valid = col < a.columns;
    const int kx = valid ? (int)(col / a.pitch) : 0;
    const int ky = valid ? (int)(col - (int64_t)kx * a.pitch) : 0;
    valid = valid && ky < a.py;  // pad columns: transformed with a zero tensor, never read
    ZTensorRegs<Real, NZ> kr;
    kr.load(a, valid, kx, ky, p);
    {
        TL in;
        in.fetch(a, col0, t);
        in.put(tile, t);
    }
    __syncthreads();
    ztile_convolve<Real, NZ, TW>(a, tile, j, p, ky, kr);
    __syncthreads();
    ztile_store<Real, NZ, TW>(a, tile, col0, t);
}

template <typename Real, int NZ, int TW = kZTile>
__global__ void __launch_bounds__(256) zconv_tile_kernel(ZArgs<Real> a) {
    zconv_tile_body<Real, NZ, TW>(a);
}
template <typename Real, int NZ, int TW = kZTile>
__global__ void __launch_bounds__(256) zconv_tile_multi(const ZArgs<Real> *tab, int zdiv) {
    const ZArgs<Real> a = tab[blockIdx.z / zdiv];
    zconv_tile_body<Real, NZ, TW>(a);
}

// z convolution with four lanes per (kx, ky) column (pz = 2 NZ = 4 M, NZ
// even): lane q owns kz = 4k + q.  Forward: X[4k+q] = DFT_M(u)[k] with the
// folded input u_z = x_z w^(q z) + x_(z+M) w^(q (z+M)), z < M; tensor at its
// own kz; inverse: y_z = sum_q w^(-q z) IDFT_M(Y_q)[z mod M], summed over the
// quad with two shuffles; lane q stores the z = q (mod 4).  Workgroups are
// renumbered per XCD so the columns ky and py - ky of one kx row, which read
// the same tensor octant entries, share an L2.
template <typename Real, int NZ>
__device__ __forceinline__ void zconv_quad_body(const ZArgs<Real> &a) {
    static_assert(NZ % 2 == 0, "four lanes per column need an even nz");
    constexpr int M = NZ / 2, PZ = 2 * NZ;
    const uint32_t blk = a.xcd ? xcd_block(blockIdx.x, gridDim.x) : blockIdx.x;
    const int64_t gid = (int64_t)blk * blockDim.x + threadIdx.x;
    const int64_t col = gid >> 2;
    const int q = (int)(gid & 3);
    bool valid = col < a.columns;  // all four lanes of a quad stay for the shuffles
    const int kx = valid ? (int)(col / a.pitch) : 0;
    const int ky = valid ? (int)(col - (int64_t)kx * a.pitch) : 0;
    valid = valid && ky < a.py;
    // w^(q z), z < NZ: one gather per z, reused by all components and the inverse
    cplx<Real> wq[NZ];
#pragma unroll
    for (int z = 0; z < NZ; ++z) wq[z] = a.tw[(q * z) % PZ];
    cplx<Real> v[3][M];
#pragma unroll
    for (int c = 0; c < 3; ++c) {
#pragma unroll
        for (int z = 0; z < M; ++z) {
            cplx<Real> lo = {Real(0), Real(0)}, hi = {Real(0), Real(0)};
            if (valid) {
                lo = a.data[c * a.comp_stride + z * a.zstride + col];
                hi = a.data[c * a.comp_stride + (z + M) * a.zstride + col];
            }
            v[c][z] = cadd(cmul(lo, wq[z]), cmul(hi, wq[z + M]));
        }
        strided_dft<Real, M, 4>(v[c], a.tw, false);
    }
#pragma unroll
    for (int k = 0; k < M; ++k) {
        Real t[6];
        tensor_at(a.K, kx, ky, 4 * k + q, t);
        apply_tensor(t, v[0][k], v[1][k], v[2][k]);
    }
#pragma unroll
    for (int c = 0; c < 3; ++c) {
        strided_dft<Real, M, 4>(v[c], a.tw, true);
        cplx<Real> y[NZ];
#pragma unroll
        for (int z = 0; z < NZ; ++z) {
            cplx<Real> s = cmul(v[c][z % M], cconj(wq[z]));
            s.x += __shfl_xor(s.x, 1);
            s.y += __shfl_xor(s.y, 1);
            s.x += __shfl_xor(s.x, 2);
            s.y += __shfl_xor(s.y, 2);
            y[z] = s;
        }
        if (valid)
#pragma unroll
            for (int z = 0; z < NZ; ++z)
                if ((z & 3) == q) a.data[c * a.comp_stride + z * a.zstride + col] = y[z];
    }
}

template <typename Real, int NZ>
__global__ void __launch_bounds__(256) zconv_quad_kernel(ZArgs<Real> a) {
    zconv_quad_body<Real, NZ>(a);
}
template <typename Real, int NZ>
__global__ void __launch_bounds__(256) zconv_quad_multi(const ZArgs<Real> *tab, int zdiv) {
    const ZArgs<Real> a = tab[blockIdx.z / zdiv];
    zconv_quad_body<Real, NZ>(a);
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
// Bound by VALU work (about half of it butterflies) and by memory latency at
// nine wavefronts per CU.  256x256x64 mixed (257x512 columns of 128, 507 MB):
// 213 us with the staged lines of zlds_kernel, 131 us here, 147 us with one
// column per lane (twice the wavefronts, but each pays its own twiddles and
// 64-byte runs).  100^3 FP64: 214 -> 109 us.
template <typename Real, int V>
struct alignas(sizeof(cplx<Real>) * V) cvec {
    cplx<Real> c[V];
};

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
    const DemagPlan &dp = c.dp;
    const dim3 zb(256);
    const bool quad = dp.tune.z_quad && (dp.nz == 4 || dp.nz == 6 || dp.nz == 8);
    // the staged tiles read the tensor blocks directly (no projection fallback)
    const bool staged = !quad && !dp.projection;
    auto by_nz = [&](auto launch) {
        switch (dp.nz) {
            case 1: launch(std::integral_constant<int, 1>{}); break;
            case 2: launch(std::integral_constant<int, 2>{}); break;
            case 3: launch(std::integral_constant<int, 3>{}); break;
            case 4: launch(std::integral_constant<int, 4>{}); break;
            case 5: launch(std::integral_constant<int, 5>{}); break;
            case 6: launch(std::integral_constant<int, 6>{}); break;
            case 7: launch(std::integral_constant<int, 7>{}); break;
            default: launch(std::integral_constant<int, 8>{}); break;
        }
    };
    if (staged) {
        const dim3 zt((unsigned)cdiv(za.columns, kZTile));
        by_nz([&](auto NZC) {
            constexpr int NZ = decltype(NZC)::value;
            launch_rec(c, reinterpret_cast<const void *>(&zconv_tile_multi<Real, NZ>), zt, zb, 0, 1, za,
                       [&] { hipLaunchKernelGGL((zconv_tile_kernel<Real, NZ>), zt, zb, 0, c.stream, za); });
        });
    } else if (quad) {
        const dim3 zq((unsigned)cdiv(4 * za.columns, 256));
        auto quad_launch = [&](auto NZC) {
            constexpr int NZ = decltype(NZC)::value;
            launch_rec(c, reinterpret_cast<const void *>(&zconv_quad_multi<Real, NZ>), zq, zb, 0, 1, za,
                       [&] { hipLaunchKernelGGL((zconv_quad_kernel<Real, NZ>), zq, zb, 0, c.stream, za); });
        };
        switch (dp.nz) {
            case 4: quad_launch(std::integral_constant<int, 4>{}); break;
            case 6: quad_launch(std::integral_constant<int, 6>{}); break;
            default: quad_launch(std::integral_constant<int, 8>{}); break;
        }
    } else {
        const dim3 zg((unsigned)cdiv(2 * za.columns, 256));
        by_nz([&](auto NZC) {
            launch_rec(c, nullptr, zg, zb, 0, 1, za, [&] {
                hipLaunchKernelGGL((zconv_pair_kernel<Real, decltype(NZC)::value>), zg, zb, 0, c.stream, za);
            });
        });
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
