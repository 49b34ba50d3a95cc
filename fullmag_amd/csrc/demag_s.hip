// demag_s.hip -- y transforms and z convolution of one kx slab in one kernel
// (see demag.hip for the pipeline).  Compiled once per field precision
// (FM_REAL).
#include "demag.hpp"

namespace fm {
namespace {

// A workgroup holds the 3 nz ky lines of one kx in LDS: forward y transforms
// (ny inputs, T lanes per line), the z convolution of every (kx, ky) column on
// the LDS lines, inverse y transforms, ny outputs.  The padded ky spectrum
// never reaches memory and two launches go (the rule and both sides' times:
// use_slab).  Bound by latency: load, FFT, columns, FFT, store in turn, with
// one to three workgroups per CU to overlap them.
template <typename Real, int NZ>
struct SlabTensor {
    static constexpr int NE = NZ / 2 + 1, NO = (NZ + 1) / 2;
};

// Columns ky = CL k + q, k < N, with all three components in one lane (see
// zreg_body); their spectra back to put(line, k, value).
template <typename Real, int N, int NZ, int CL, class Put>
__device__ __forceinline__ void slab_columns(const SlabArgs<Real> &a, cplx<Real> *lds, int kx, int q, Put &&put) {
    using C = cplx<Real>;
    constexpr int NE = SlabTensor<Real, NZ>::NE, NO = SlabTensor<Real, NZ>::NO, S = fx_size(N);
    constexpr int LANES = 3 * NZ * fx_lanes(N), ROUNDS = (N + LANES - 1) / LANES;
#pragma unroll
    for (int r = 0; r < ROUNDS; ++r) {
        const int k0 = (int)threadIdx.x + r * LANES;
        if (k0 >= N) break;
        const int ky = CL * k0 + q;
        const bool ylo = ky <= CL * N / 2;
        const Real sy = ylo ? Real(1) : Real(-1);
        const Real *kp = a.K.k + kx * a.K.l.skx + kern_y(a.K.l, ylo ? ky : CL * N - ky);
        const C *col = lds + fxslot<N>(k0);
        auto half = [&](C (*v)[NZ], int n, int64_t off, int odd) {
            Real t[NE][6];
#pragma unroll
            for (int i = 0; i < n; ++i)
#pragma unroll
                for (int q = 0; q < 6; ++q) t[i][q] = kp[off + i * a.K.l.soz + q * a.K.l.sc];
#pragma unroll
            for (int c = 0; c < 3; ++c) dft_any<Real, NZ>(v[c], a.twz, NZ, false);
#pragma unroll
            for (int k = 0; k < NZ; ++k) {
                const int kz = 2 * k + odd, i = (kz <= NZ ? kz : 2 * NZ - kz) >> 1;
                const Real sz = kz <= NZ ? Real(1) : Real(-1);
                const Real tt[6] = {t[i][0], t[i][1], t[i][2], sy * t[i][3], sz * t[i][4], sz * (sy * t[i][5])};
                apply_tensor(tt, v[0][k], v[1][k], v[2][k]);
            }
#pragma unroll
            for (int c = 0; c < 3; ++c) dft_any<Real, NZ>(v[c], a.twz, NZ, true);
        };
        C x[3][NZ], y[3][NZ];
#pragma unroll
        for (int c = 0; c < 3; ++c)
#pragma unroll
            for (int z = 0; z < NZ; ++z) y[c][z] = x[c][z] = col[(c * NZ + z) * S];
        half(y, NE, 0, 0);
#pragma unroll
        for (int z = 1; z < NZ; ++z) {
            const C w = a.twz[z];
#pragma unroll
            for (int c = 0; c < 3; ++c) x[c][z] = cmul(x[c][z], w);
        }
        half(x, NO, a.K.l.odd, 1);
#pragma unroll
        for (int z = 0; z < NZ; ++z) {
            const C w = cconj(a.twz[z]);
#pragma unroll
            for (int c = 0; c < 3; ++c)
                put(c * NZ + z, k0, cadd(y[c][z], z > 0 ? cmul(x[c][z], w) : x[c][z]));
        }
    }
}

// Columns (CL = 1) with one component per lane (NZ >= 5; see zreg3_body): a half's
// spectra replace the column's inputs in LDS while they meet.
template <typename Real, int N, int NZ, class Put>
__device__ __forceinline__ void slab_rows(const SlabArgs<Real> &a, cplx<Real> *lds, int kx, Put &&put) {
    using C = cplx<Real>;
    constexpr int NE = SlabTensor<Real, NZ>::NE, NO = SlabTensor<Real, NZ>::NO, S = fx_size(N);
    constexpr int COLS = NZ * fx_lanes(N), ROUNDS = (N + COLS - 1) / COLS;
    const int c = (int)threadIdx.x / COLS, k0 = (int)threadIdx.x % COLS;
    const int e0 = c, e1 = c == 0 ? 3 : c == 1 ? 5 : 4, e2 = c == 0 ? 4 : c == 1 ? 3 : 5;
    const int c1 = c == 2 ? 0 : c + 1, c2 = c == 0 ? 2 : c - 1;
    const Real sz = c == 2 ? Real(-1) : Real(1);
    for (int r = 0; r < ROUNDS; ++r) {
        const bool live = k0 + r * COLS < N;  // every lane stays for the barriers
        const int ky = live ? k0 + r * COLS : 0;
        const bool ylo = ky <= N / 2;
        const Real sy = ylo || c != 1 ? Real(1) : Real(-1);
        const Real *kp = a.K.k + kx * a.K.l.skx + kern_y(a.K.l, ylo ? ky : N - ky);
        C *own = lds + c * NZ * S + fxslot<N>(ky);
        const C *p1 = lds + c1 * NZ * S + fxslot<N>(ky), *p2 = lds + c2 * NZ * S + fxslot<N>(ky);
        auto half = [&](C *v, int n, int64_t off, int odd) {
            Real t[NE][3];
#pragma unroll
            for (int i = 0; i < n; ++i) {
                const Real *p = kp + off + i * a.K.l.soz;
                t[i][0] = p[e0 * a.K.l.sc];
                t[i][1] = p[e1 * a.K.l.sc];
                t[i][2] = p[e2 * a.K.l.sc];
            }
            dft_any<Real, NZ>(v, a.twz, NZ, false);
#pragma unroll
            for (int k = 0; k < NZ; ++k) {
                const Real g = 2 * k + odd <= NZ ? Real(1) : sz;
                v[k] = {g * v[k].x, g * v[k].y};
                if (live) own[k * S] = v[k];
            }
            __syncthreads();
#pragma unroll
            for (int k = 0; k < NZ; ++k) {
                const int kz = 2 * k + odd, i = (kz <= NZ ? kz : 2 * NZ - kz) >> 1;
                const Real g = kz <= NZ ? Real(-1) : -sz;
                const C p = p1[k * S], q = p2[k * S];
                v[k] = {g * (t[i][0] * v[k].x + t[i][1] * p.x + t[i][2] * q.x),
                        g * (t[i][0] * v[k].y + t[i][1] * p.y + t[i][2] * q.y)};
            }
            dft_any<Real, NZ>(v, a.twz, NZ, true);
            __syncthreads();  // the half's spectra have been read
        };
        C x[NZ], y[NZ];
#pragma unroll
        for (int z = 0; z < NZ; ++z) {
            const C q = own[z * S];
            y[z] = x[z] = {sy * q.x, sy * q.y};
        }
        half(y, NE, 0, 0);
#pragma unroll
        for (int z = 1; z < NZ; ++z) x[z] = cmul(x[z], a.twz[z]);
        half(x, NO, a.K.l.odd, 1);
        if (live)
#pragma unroll
            for (int z = 0; z < NZ; ++z) {
                const C o = cadd(y[z], z > 0 ? cmul(x[z], cconj(a.twz[z])) : x[z]);
                put(c * NZ + z, ky, C{sy * o.x, sy * o.y});
            }
    }
}

// The z convolution of every column of the lines in LDS, ky = CL k + q: entry
// k of line c nz + z to put(line, k, value).  HIGH: nz 5 .. 8, else 2 .. 4.
template <typename Real, int N, bool HIGH, int CL, class Put>
__device__ __forceinline__ void slab_z(const SlabArgs<Real> &a, cplx<Real> *lds, int kx, int q, Put &&put) {
    if constexpr (HIGH && CL > 1) {
        switch (a.nz) {
            case 5: slab_columns<Real, N, 5, CL>(a, lds, kx, q, put); break;
            case 6: slab_columns<Real, N, 6, CL>(a, lds, kx, q, put); break;
            case 7: slab_columns<Real, N, 7, CL>(a, lds, kx, q, put); break;
            default: slab_columns<Real, N, 8, CL>(a, lds, kx, q, put); break;
        }
    } else if constexpr (HIGH) {
        switch (a.nz) {
            case 5: slab_rows<Real, N, 5>(a, lds, kx, put); break;
            case 6: slab_rows<Real, N, 6>(a, lds, kx, put); break;
            case 7: slab_rows<Real, N, 7>(a, lds, kx, put); break;
            default: slab_rows<Real, N, 8>(a, lds, kx, put); break;
        }
    } else {
        switch (a.nz) {
            case 2: slab_columns<Real, N, 2, CL>(a, lds, kx, q, put); break;
            case 3: slab_columns<Real, N, 3, CL>(a, lds, kx, q, put); break;
            default: slab_columns<Real, N, 4, CL>(a, lds, kx, q, put); break;
        }
    }
}

template <typename Real, int N, bool HIGH>
__device__ __forceinline__ void slab_body(const SlabArgs<Real> &a) {
    using C = cplx<Real>;
    constexpr int T = fx_lanes(N), E = fx_elems(N), S = fx_size(N);
    extern __shared__ unsigned char smem_raw[];
    C *lds = reinterpret_cast<C *>(smem_raw);
    const int kx = (int)blockIdx.x;
    const int l = (int)threadIdx.x / T, t = (int)threadIdx.x % T;  // line l = c nz + z
    C *line = lds + l * S;
    C *g = a.data + l * a.plane_stride + (int64_t)kx * a.pitch;
    {
        C v[E];
#pragma unroll
        for (int e = 0; e < E / 2; ++e) {
            const int i = t + e * T;
            const C q = g[i < a.ny ? i : 0];
            v[e] = i < a.ny ? q : C{Real(0), Real(0)};
        }
#pragma unroll
        for (int e = E / 2; e < E; ++e) v[e] = C{Real(0), Real(0)};
        fx_first_pass<Real, N>(line, t, v, a.tw, false);
        fx_rest<Real, N>(line, t, a.tw, false);
    }
    __syncthreads();
    slab_z<Real, N, HIGH, 1>(a, lds, kx, 0, [&](int ln, int k, const C &o) { lds[ln * S + fxslot<N>(k)] = o; });
    __syncthreads();
    C v[E];
    fx_load<Real, N>(line, t, v);
    fx_first_pass<Real, N>(line, t, v, a.tw, true);
    fx_rest_put<Real, N, 2>(line, t, a.tw, true, [&](int i, const C &q) {
        if (i < a.ny) g[i] = q;
    });
}

template <typename Real, int N, bool HIGH>
__global__ void __launch_bounds__((HIGH ? 24 : 12) * fx_lanes(N)) slab_kernel(SlabArgs<Real> a) {
    slab_body<Real, N, HIGH>(a);
}
template <typename Real, int N, bool HIGH>
__global__ void __launch_bounds__((HIGH ? 24 : 12) * fx_lanes(N)) slab_multi(const SlabArgs<Real> *tab, int zdiv) {
    const SlabArgs<Real> a = tab[blockIdx.z / zdiv];
    slab_body<Real, N, HIGH>(a);
}

// Class q of a slab too long for the LDS: ky = CL k + q, k < P = py / CL.  Its
// spectrum is the P-point transform of w^(q j) sum_f w^(q f P) x[j + f P],
// w = exp(-2 pi i / py), so a workgroup holds 3 nz lines of a quarter of the
// padded length; its z convolution goes straight to memory, a class's entries
// together, and the inverse y lines read it from there.  Against the y lines
// and zreg_kernel the padded spectrum is written once less and read once less
// (512x512x8 FP32: 207 MB read and written instead of 409), while the x
// spectrum is read by four workgroups, next to each other on one XCD.  Bound by
// latency at two workgroups per CU: 74 us there with VALU instructions issued
// in 46 % of the SIMDs' cycles, 1.7 wavefronts on a SIMD on average and 221 MB
// at 3.0 TB/s.  Three wavefronts per SIMD (168
// registers) take 76 us there, two 93 us, a component per lane (slab_rows)
// 106 us, a workgroup of one wavefront per 64 columns that walks over its
// lines 111 us; the two kernels it replaces 80 us.  Per step and the rule:
// class_rule.
template <typename Real, int P, int CL, bool HIGH>
__device__ __forceinline__ void class_body(const SlabArgs<Real> &a) {
    using C = cplx<Real>;
    constexpr int T = fx_lanes(P), E = fx_elems(P), S = fx_size(P);
    static_assert(CL == 4, "two inputs per element of a class's lines");
    extern __shared__ unsigned char smem_raw[];
    C *lds = reinterpret_cast<C *>(smem_raw);
    const int b = (int)xcd_block(blockIdx.x, gridDim.x), kx = b / CL, q = b % CL;
    const int l = (int)threadIdx.x / T, t = (int)threadIdx.x % T;  // line l = c nz + z
    C *line = lds + l * S;
    {
        const C *g = a.in + l * a.in_plane + (int64_t)kx * a.in_pitch;
        C x[2][E], w[E];
#pragma unroll
        for (int f = 0; f < 2; ++f)
#pragma unroll
            for (int e = 0; e < E; ++e) {
                const int i = t + e * T + f * P;
                x[f][e] = g[i < a.ny ? i : 0];
            }
#pragma unroll
        for (int e = 0; e < E; ++e) w[e] = a.tw[q * (t + e * T)];
        // w^(q P) = (-i)^q
        const Real cr = q == 0 ? Real(1) : q == 2 ? Real(-1) : Real(0);
        const Real ci = q == 1 ? Real(1) : q == 3 ? Real(-1) : Real(0);
        C v[E];
#pragma unroll
        for (int e = 0; e < E; ++e) {
            const int i = t + e * T;
            const C z{Real(0), Real(0)}, u0 = i < a.ny ? x[0][e] : z, u1 = i + P < a.ny ? x[1][e] : z;
            const C u{u0.x + (cr * u1.x + ci * u1.y), u0.y + (cr * u1.y - ci * u1.x)};
            v[e] = cmul(u, w[e]);
        }
        fx_first_pass<Real, P>(line, t, v, a.twp, false);
        fx_rest<Real, P>(line, t, a.twp, false);
    }
    __syncthreads();
    C *out = a.data + (int64_t)kx * a.pitch + q * P;
    slab_z<Real, P, HIGH, CL>(a, lds, kx, q, [&](int ln, int k, const C &o) { out[ln * a.plane_stride + k] = o; });
}
template <typename Real, int P, int CL, bool HIGH>
__global__ void __launch_bounds__((HIGH ? 24 : 12) * fx_lanes(P), sizeof(Real) == 4 ? 3 : 1) class_kernel(SlabArgs<Real> a) {
    class_body<Real, P, CL, HIGH>(a);
}
template <typename Real, int P, int CL, bool HIGH>
__global__ void __launch_bounds__((HIGH ? 24 : 12) * fx_lanes(P), sizeof(Real) == 4 ? 3 : 1) class_multi(const SlabArgs<Real> *tab, int zdiv) {
    const SlabArgs<Real> a = tab[blockIdx.z / zdiv];
    class_body<Real, P, CL, HIGH>(a);
}

}  // namespace

template <typename Real>
void launch_class(Context &c, const LinePlan &lp, const SlabArgs<Real> &sa) {
    with_line(lp, [&](auto NC) {
        constexpr int N = decltype(NC)::value;
        if constexpr (class_length(N)) {
            constexpr int P = N / kClasses;
            const dim3 grid((unsigned)(sa.hx * kClasses)), block((unsigned)(3 * sa.nz * fx_lanes(P)));
            const size_t lds = (size_t)3 * sa.nz * fx_size(P) * sizeof(cplx<Real>);
            auto launch = [&](auto high) {
                constexpr bool H = decltype(high)::value;
                launch_rec(c, reinterpret_cast<const void *>(&class_multi<Real, P, kClasses, H>), grid, block, lds, 1,
                           sa, [&] {
                               hipLaunchKernelGGL((class_kernel<Real, P, kClasses, H>), grid, block, lds, c.stream, sa);
                           });
            };
            if constexpr (sizeof(Real) == 4) {
                if (sa.nz > 4) {
                    launch(std::true_type{});
                    return;
                }
            }
            launch(std::false_type{});
        }
    });
}

template <typename Real>
void launch_slab(Context &c, const LinePlan &lp, const SlabArgs<Real> &sa) {
    with_line(lp, [&](auto NC) {
        constexpr int N = decltype(NC)::value;
        if constexpr (slab_length(N)) {
            const dim3 grid((unsigned)sa.hx), block((unsigned)(3 * sa.nz * lp.threads));
            const size_t lds = (size_t)3 * sa.nz * fx_size(N) * sizeof(cplx<Real>);
            auto launch = [&](auto high) {
                constexpr bool H = decltype(high)::value;
                launch_rec(c, reinterpret_cast<const void *>(&slab_multi<Real, N, H>), grid, block, lds, 1, sa, [&] {
                    hipLaunchKernelGGL((slab_kernel<Real, N, H>), grid, block, lds, c.stream, sa);
                });
            };
            if (sa.nz > 4) launch(std::true_type{});
            else launch(std::false_type{});
        }
    });
}

using R = FM_REAL;
template void launch_slab<R>(Context &, const LinePlan &, const SlabArgs<R> &);
template void launch_class<R>(Context &, const LinePlan &, const SlabArgs<R> &);

}  // namespace fm
