// demag_y.hip -- contiguous line passes of the demag convolution (the 3-D and
// split-film y transforms) and the thin-film y convolution (see demag.hip for
// the pipeline).  Compiled once per field precision (FM_REAL).
#include "demag.hpp"

namespace fm {
namespace {

// Lines without a compile-time schedule (and the Newell setup).
template <typename Real>
__global__ void __launch_bounds__(kMaxBlock) line_kernel(LineArgs<Real> a) {
    extern __shared__ unsigned char smem_raw[];
    cplx<Real> *lds = reinterpret_cast<cplx<Real> *>(smem_raw);
    const int n = a.lp.n, ls = n + kPad, T = a.lp.threads;
    // line j = tid / T of the workgroup belongs to its T lanes (blockDim.x = lpw T)
    const int j = threadIdx.x / T, t = threadIdx.x - j * T;
    const int64_t l = (int64_t)blockIdx.x * a.lpw + j;
    cplx<Real> *line = lds + j * ls;
    cplx<Real> *g = a.data + l * a.line_pitch;
    const bool live = l < a.lines;
    for (int e = t; e < n; e += T) {
        cplx<Real> v = {Real(0), Real(0)};
        if (e < a.n_in && live) v = g[e];
        line[lslot(a.lp, e)] = v;
    }
    __syncthreads();
    line_fft(line, a.lp, t, a.tw, a.inverse != 0);
    if (live)
        for (int e = t; e < a.n_out; e += T) g[e] = line[lslot(a.lp, e)];
}

// Contiguous line pass of a scheduled length N: a workgroup holds
// G = max(1, 64 / T) lines at a time (T lanes per line) and walks
// `iters` groups of lines.  With PIPE the global loads of the next group are
// issued into registers before the current group's LDS transform, so memory
// traffic overlaps the FFT; without it (one group per workgroup) the kernel
// holds no prefetch registers and more waves share each SIMD instead.
// Forward: N / 2 inputs per line (RAGGED: a.n_in, fewer), the rest zero, and N
// outputs; inverse: N inputs, a.n_out <= N / 2 outputs.
template <typename Real, int N, bool INV, bool PIPE, bool RAGGED, bool CLS = false>
__device__ __forceinline__ void line_pipe_body(const LineArgs<Real> &a) {
    constexpr int T = fx_lanes(N), E = fx_elems(N);
    constexpr int G = T >= 64 ? 1 : 64 / T;
    constexpr int NI = INV ? E : E / 2;
    static_assert(E % 2 == 0, "whole loads per lane");
    extern __shared__ unsigned char smem_raw[];
    cplx<Real> *lds = reinterpret_cast<cplx<Real> *>(smem_raw);
    const int j = (int)threadIdx.x / T, t = (int)threadIdx.x - j * T;
    cplx<Real> *line = lds + j * fx_size(N);
    // CLS: lane t takes the first pass of lane t1, so that neighbouring lanes
    // read neighbouring entries of one class
    constexpr int TC = T / kClasses;
    const int t1 = CLS ? (t % TC) * kClasses + t / TC : t;
    const int64_t first = (int64_t)blockIdx.x * (PIPE ? a.iters : 1) * G + j;
    cplx<Real> buf[NI];
    auto fetch = [&](int64_t l) {
        // a line past the end loads line 0 instead: its transform is never
        // stored, and unconditional loads issue together (a load guarded by
        // a select becomes a branch, and the join waits for the loads
        // issued before it)
        const cplx<Real> *g = a.data + (l < a.lines ? l : 0) * a.line_pitch;
        if constexpr (CLS) {
            // element i is entry i / kClasses of class i mod kClasses
            static_assert(T % kClasses == 0, "a lane stays in its class");
            g = a.in + (l < a.lines ? l : 0) * a.in_pitch + (t / TC) * (N / kClasses) + t % TC;
#pragma unroll
            for (int e = 0; e < NI; ++e) buf[e] = g[e * TC];
        } else if constexpr (!RAGGED) {
#pragma unroll
            for (int e = 0; e < NI; ++e) buf[e] = g[t + e * T];
        } else {
            // a line padded beyond 2 n_in: clamped addresses, zeros selected
            // after the loads
#pragma unroll
            for (int e = 0; e < NI; ++e) {
                const int i = t + e * T;
                const cplx<Real> q = g[i < a.n_in ? i : 0];
                buf[e] = i < a.n_in ? q : cplx<Real>{Real(0), Real(0)};
            }
        }
    };
    fetch(first);
    const int iters = PIPE ? a.iters : 1;
    for (int it = 0; it < iters; ++it) {
        const int64_t l = first + (int64_t)it * G;
        // the loaded elements are the first pass's inputs
        cplx<Real> v[E];
#pragma unroll
        for (int e = 0; e < E; ++e) v[e] = e < NI ? buf[e] : cplx<Real>{Real(0), Real(0)};
        if (PIPE && it + 1 < iters) fetch(l + G);
        fx_first_pass<Real, N>(line, t1, v, a.tw, INV);
        // the last pass stores from registers: consecutive lanes hold
        // consecutive elements, and the inverse produces only the half of
        // them that is kept
        const bool live = l < a.lines;
        cplx<Real> *g = a.data + (live ? l : 0) * a.line_pitch;
        fx_rest_put<Real, N, INV ? 2 : 1>(line, t, a.tw, INV, [&](int i, const cplx<Real> &q) {
            if (live && (!INV || i < a.n_out)) g[i] = q;
        });
        if (PIPE) __syncthreads();
    }
}

template <typename Real, int N, bool INV, bool PIPE, bool RAGGED>
__global__ void __launch_bounds__(256) line_pipe_kernel(LineArgs<Real> a) {
    line_pipe_body<Real, N, INV, PIPE, RAGGED>(a);
}
template <typename Real, int N, bool INV, bool PIPE, bool RAGGED>
__global__ void __launch_bounds__(256) line_pipe_multi(const LineArgs<Real> *tab, int zdiv) {
    const LineArgs<Real> a = tab[blockIdx.z / zdiv];
    line_pipe_body<Real, N, INV, PIPE, RAGGED>(a);
}

template <typename Real, int N>
__global__ void __launch_bounds__(256) line_class_kernel(LineArgs<Real> a) {
    line_pipe_body<Real, N, true, false, false, true>(a);
}
template <typename Real, int N>
__global__ void __launch_bounds__(256) line_class_multi(const LineArgs<Real> *tab, int zdiv) {
    const LineArgs<Real> a = tab[blockIdx.z / zdiv];
    line_pipe_body<Real, N, true, false, false, true>(a);
}

// MAXB: kMaxBlock, or 1024 for lines too long for three of them in
// kMaxBlock lanes.  Lines without a compile-time schedule.
template <typename Real>
__device__ __forceinline__ void yconv_body(const YConvArgs<Real> &a) {
    extern __shared__ unsigned char smem_raw[];
    cplx<Real> *lds = reinterpret_cast<cplx<Real> *>(smem_raw);
    const int n = a.lp.n, ls = n + kPad, T = a.lp.threads;
    const int tid = threadIdx.x, nthr = blockDim.x;
    const int kx0 = blockIdx.x * a.kpw;
    const int nl = 3 * a.kpw;  // slot s = c * kpw + j
    for (int idx = tid; idx < nl * n; idx += nthr) {
        const int s = idx / n, e = idx - s * n;
        const int c = s / a.kpw, kx = kx0 + (s - c * a.kpw);
        cplx<Real> v = {Real(0), Real(0)};
        if (e < a.ny && kx < a.hx) v = a.data[a.g.at(c, 0, kx, e)];
        lds[s * ls + lslot(a.lp, e)] = v;
    }
    __syncthreads();
    line_fft(lds + (tid / T) * ls, a.lp, tid % T, a.tw, false);
    for (int idx = tid; idx < a.kpw * n; idx += nthr) {
        const int j = idx / n, e = idx - j * n;
        const int kx = kx0 + j;
        if (kx >= a.hx) continue;
        Real t[6];
        tensor_at(a.K, kx, e, 0, t);
        const int se = lslot(a.lp, e);
        apply_tensor(t, lds[j * ls + se], lds[(a.kpw + j) * ls + se], lds[(2 * a.kpw + j) * ls + se]);
    }
    __syncthreads();
    line_fft(lds + (tid / T) * ls, a.lp, tid % T, a.tw, true);
    for (int idx = tid; idx < nl * a.ny; idx += nthr) {
        const int s = idx / a.ny, e = idx - s * a.ny;
        const int c = s / a.kpw, kx = kx0 + (s - c * a.kpw);
        if (kx < a.hx) a.data[a.g.at(c, 0, kx, e)] = lds[s * ls + lslot(a.lp, e)];
    }
}

template <typename Real, int MAXB>
__global__ void __launch_bounds__(MAXB) yconv_kernel(YConvArgs<Real> a) {
    yconv_body<Real>(a);
}
template <typename Real, int MAXB>
__global__ void __launch_bounds__(MAXB) yconv_multi(const YConvArgs<Real> *tab, int zdiv) {
    const YConvArgs<Real> a = tab[blockIdx.z / zdiv];
    yconv_body<Real>(a);
}

// The y convolution of a scheduled length N.  Same mapping (line s = c kpw + j
// of a workgroup holds component c of column j), but a lane's inputs go from
// memory straight into the first pass, and the tensor entries it will need
// are loaded beside them, so one memory wait covers both; every index is a
// compile-time shift or mask.  Bound by latency: a column is three short
// lines.  At 64x64 FP64 the runtime-plan form spilled to scratch at its
// 128-register budget.
template <typename Real, int N>
__device__ __forceinline__ void yconv_fx_body(const YConvArgs<Real> &a) {
    using C = cplx<Real>;
    constexpr int T = fx_lanes(N), E = fx_elems(N), NT = (E + 2) / 3, ls = fx_size(N);
    extern __shared__ unsigned char smem_raw[];
    C *lds = reinterpret_cast<C *>(smem_raw);
    const int tid = threadIdx.x, nthr = blockDim.x;
    const int kx0 = blockIdx.x * a.kpw;
    const int s = tid / T, t = tid % T, c = s / a.kpw, kxl = kx0 + (s - c * a.kpw);
    const bool live = kxl < a.hx;
    C *line = lds + s * ls;
    C *g = a.data + a.g.at(c, 0, live ? kxl : 0, 0);
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
    }
    // entry u: column j, ky = e of the workgroup's kpw N (kpw N / nthr = E / 3)
    Real k4[NT][4];
#pragma unroll
    for (int u = 0; u < NT; ++u) {
        const int idx = tid + u * nthr, j = idx / N, e = idx % N, kx = kx0 + j;
        const bool ok = j < a.kpw && kx < a.hx;
        const Real *K = a.K.k + kern_at(a.K.l, 0, 0, ok ? kx : 0, e <= N / 2 ? e : N - e);
#pragma unroll
        for (int q = 0; q < 4; ++q) k4[u][q] = K[q];
    }
    fx_rest<Real, N>(line, t, a.tw, false);
    __syncthreads();
#pragma unroll
    for (int u = 0; u < NT; ++u) {
        const int idx = tid + u * nthr, j = idx / N, e = idx % N;
        if (j < a.kpw) {
            const Real sy = e <= N / 2 ? Real(1) : Real(-1);
            const Real tt[6] = {k4[u][0], k4[u][1], k4[u][2], sy * k4[u][3], Real(0), Real(0)};
            const int se = fxslot<N>(e);
            apply_tensor(tt, lds[j * ls + se], lds[(a.kpw + j) * ls + se], lds[(2 * a.kpw + j) * ls + se]);
        }
    }
    __syncthreads();
    C v[E];
    fx_load<Real, N>(line, t, v);
    fx_first_pass<Real, N>(line, t, v, a.tw, true);
    fx_rest_put<Real, N, 2>(line, t, a.tw, true, [&](int i, const C &q) {
        if (live && i < a.ny) g[i] = q;
    });
}

template <typename Real, int N>
__global__ void __launch_bounds__(fx_lanes(N) > 64 ? 3 * fx_lanes(N) : 256) yconv_fx_kernel(YConvArgs<Real> a) {
    yconv_fx_body<Real, N>(a);
}
template <typename Real, int N>
__global__ void __launch_bounds__(fx_lanes(N) > 64 ? 3 * fx_lanes(N) : 256)
    yconv_fx_multi(const YConvArgs<Real> *tab, int zdiv) {
    const YConvArgs<Real> a = tab[blockIdx.z / zdiv];
    yconv_fx_body<Real, N>(a);
}

// acc += k m and acc += i k m for real k.
template <typename T>
__device__ __forceinline__ void mad_re(cplx<T> &acc, T k, const cplx<T> &m) {
    acc.x += k * m.x;
    acc.y += k * m.y;
}
template <typename T>
__device__ __forceinline__ void mad_im(cplx<T> &acc, T k, const cplx<T> &m) {
    acc.x -= k * m.y;
    acc.y += k * m.x;
}

// Thin stack: the 3 L ky lines of a kx column in one workgroup, transformed,
// coupled and transformed back without leaving LDS.  As line passes and a
// tensor pass the layers' spectra cross memory six times and the pair kernels
// are read at every ky; here twice, and the kernels on the ky octant.  Three
// 512 x 512 films, FP32: 3 x (6.6 + 6.1) + 25.9 us as three passes, 33.6 us
// here; bound by each workgroup's chain of load, transforms, coupling and
// store with two of them on a CU (the 513th column alone costs 6 us).
template <typename Real, int N, int L>
__global__ void __launch_bounds__(3 * L * fx_lanes(N) > 256 ? 3 * L * fx_lanes(N) : 256)
    ystack_kernel(YStackArgs<Real> a) {
    using C = cplx<Real>;
    constexpr int T = fx_lanes(N), E = fx_elems(N), ls = fx_size(N), NL = 3 * L, HP = N / 2 + 1;
    extern __shared__ unsigned char smem_raw[];
    C *lds = reinterpret_cast<C *>(smem_raw);
    const int tid = threadIdx.x, nthr = blockDim.x;
    const int kx0 = blockIdx.x * a.kpw;
    const int s = tid / T, t = tid % T, j = s / NL, kxl = kx0 + j;
    const bool live = kxl < a.hx;
    C *line = lds + s * ls;
    C *g = a.data + ((int64_t)(s - j * NL) * a.hx + (live ? kxl : kx0)) * N;
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
    }
    fx_rest<Real, N>(line, t, a.tw, false);
    __syncthreads();
    for (int idx = tid; idx < a.kpw * N; idx += nthr) {
        const int jc = idx / N, ky = idx % N, kx = kx0 + jc < a.hx ? kx0 + jc : kx0;
        const bool lo = ky <= N / 2;
        const Real sy = lo ? Real(1) : Real(-1);
        const int64_t o = (int64_t)kx * 6 * HP + (lo ? ky : N - ky), ks = (int64_t)a.hx * 6 * HP;
        C *col = lds + jc * NL * ls + fxslot<N>(ky);
        C m[L][3], h[L][3];
#pragma unroll
        for (int l = 0; l < L; ++l)
#pragma unroll
            for (int c = 0; c < 3; ++c) {
                m[l][c] = col[(3 * l + c) * ls];
                h[l][c] = {Real(0), Real(0)};
            }
#pragma unroll
        for (int d = 0; d < L; ++d)
#pragma unroll
            for (int q = 0; q < L; ++q) {
                C *hh = h[d];
                const C *mm = m[q];
                const Real *K = a.kern + (q == d ? 0 : a.kernel[d][q]) * ks + o;  // 0: self
                const Real kxx = K[0], kyy = K[HP], kzz = K[2 * HP], kxy = sy * K[3 * HP];
                const Real kxz = K[4 * HP], kyz = sy * K[5 * HP];
                mad_re(hh[0], kxx, mm[0]);
                mad_re(hh[0], kxy, mm[1]);
                mad_im(hh[0], kxz, mm[2]);
                mad_re(hh[1], kxy, mm[0]);
                mad_re(hh[1], kyy, mm[1]);
                mad_im(hh[1], kyz, mm[2]);
                mad_im(hh[2], kxz, mm[0]);
                mad_im(hh[2], kyz, mm[1]);
                mad_re(hh[2], kzz, mm[2]);
            }
#pragma unroll
        for (int l = 0; l < L; ++l)
#pragma unroll
            for (int c = 0; c < 3; ++c) col[(3 * l + c) * ls] = {-h[l][c].x, -h[l][c].y};
    }
    __syncthreads();
    C v[E];
    fx_load<Real, N>(line, t, v);
    fx_first_pass<Real, N>(line, t, v, a.tw, true);
    fx_rest_put<Real, N, 2>(line, t, a.tw, true, [&](int i, const C &q) {
        if (live && i < a.ny) g[i] = q;
    });
}

// Thin film, split form: the three components' ky spectra (all py entries,
// rows `rows` apart) are multiplied by the tensor at kz = 0 in place; the y
// transforms run before and after as line passes.  For films whose three
// lines do not fit one workgroup.
template <typename Real>
__global__ void __launch_bounds__(256) film_tensor_kernel(cplx<Real> *data, KernelView<Real> K, int hx, int py,
                                                          int64_t rows) {
    const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (i >= (int64_t)hx * py) return;
    const int kx = (int)(i / py), ky = (int)(i - (int64_t)kx * py);
    Real t[6];
    tensor_at(K, kx, ky, 0, t);
    const int64_t cs = (int64_t)hx * rows, o = (int64_t)kx * rows + ky;
    apply_tensor(t, data[o], data[cs + o], data[2 * cs + o]);
}

}  // namespace

template <typename Real>
void launch_lines(Context &c, const LinePlan &lp, LineArgs<Real> la) {
    const DemagPlan &dp = c.dp;
    const size_t ce = sizeof(cplx<Real>);
    with_line(lp, [&](auto NC) {
        constexpr int N = decltype(NC)::value;
        if constexpr (N > 0) {
            // the prefetching form (y_pipe > 1) and its absence (0) are knobs
            // of the power-of-two lengths
            constexpr bool P2 = fx_odd(N) == 1;
            if (!P2 || dp.tune.y_pipe > 0) {
                const bool inv = la.inverse != 0;
                constexpr int T = fx_lanes(N), G = T >= 64 ? 1 : 64 / T;
                la.iters = !P2 ? 1 : !inv && dp.tune.y_pipe_f > 0 ? dp.tune.y_pipe_f : dp.tune.y_pipe;
                const dim3 grid((unsigned)cdiv(la.lines, (int64_t)G * la.iters)), block((unsigned)(G * T));
                const size_t lds = (size_t)G * fx_size(N) * ce;
                auto launch = [&](auto invc, auto pipe, auto ragged) {
                    constexpr bool I = decltype(invc)::value, P = decltype(pipe)::value, G1 = decltype(ragged)::value;
                    launch_rec(c, P ? nullptr : reinterpret_cast<const void *>(&line_pipe_multi<Real, N, I, false, G1>),
                               grid, block, lds, 1, la, [&] {
                                   hipLaunchKernelGGL((line_pipe_kernel<Real, N, I, P, G1>), grid, block, lds,
                                                      c.stream, la);
                               });
                };
                const std::true_type yes;
                const std::false_type no;
                if constexpr (P2) {
                    if (la.iters > 1) {
                        if (inv) launch(yes, yes, no);
                        else if (2 * la.n_in == N) launch(no, yes, no);
                        else launch(no, yes, yes);
                        return;
                    }
                }
                if (inv) launch(yes, no, no);
                else if (2 * la.n_in == N) launch(no, no, no);
                else launch(no, no, yes);
                return;
            }
        }
        const dim3 grid((unsigned)cdiv(la.lines, la.lpw)), block((unsigned)(la.lpw * lp.threads));
        const size_t lds = (size_t)la.lpw * (lp.n + kPad) * ce;
        launch_rec(c, nullptr, grid, block, lds, 1, la,
                   [&] { hipLaunchKernelGGL((line_kernel<Real>), grid, block, lds, c.stream, la); });
    });
}

template <typename Real>
void launch_class_inverse(Context &c, const LinePlan &lp, const LineArgs<Real> &la) {
    with_line(lp, [&](auto NC) {
        constexpr int N = decltype(NC)::value;
        if constexpr (class_length(N)) {
            constexpr int T = fx_lanes(N), G = T >= 64 ? 1 : 64 / T;
            const dim3 grid((unsigned)cdiv(la.lines, (int64_t)G)), block((unsigned)(G * T));
            const size_t lds = (size_t)G * fx_size(N) * sizeof(cplx<Real>);
            launch_rec(c, reinterpret_cast<const void *>(&line_class_multi<Real, N>), grid, block, lds, 1, la, [&] {
                hipLaunchKernelGGL((line_class_kernel<Real, N>), grid, block, lds, c.stream, la);
            });
        }
    });
}

template <typename Real>
void launch_yconv(Context &c, const YConvArgs<Real> &ya) {
    const dim3 grid((unsigned)cdiv(ya.hx, ya.kpw)), block((unsigned)(3 * ya.kpw * ya.lp.threads));
    const size_t lds = (size_t)3 * ya.kpw * line_slots(ya.lp) * sizeof(cplx<Real>);
    with_line(ya.lp, [&](auto NC) {
        constexpr int N = decltype(NC)::value;
        if constexpr (N > 0) {
            launch_rec(c, reinterpret_cast<const void *>(&yconv_fx_multi<Real, N>), grid, block, lds, 1, ya,
                       [&] { hipLaunchKernelGGL((yconv_fx_kernel<Real, N>), grid, block, lds, c.stream, ya); });
        } else if (block.x > (unsigned)kMaxBlock) {
            launch_rec(c, reinterpret_cast<const void *>(&yconv_multi<Real, 1024>), grid, block, lds, 1, ya,
                       [&] { hipLaunchKernelGGL((yconv_kernel<Real, 1024>), grid, block, lds, c.stream, ya); });
        } else {
            launch_rec(c, reinterpret_cast<const void *>(&yconv_multi<Real, kMaxBlock>), grid, block, lds, 1, ya,
                       [&] { hipLaunchKernelGGL((yconv_kernel<Real, kMaxBlock>), grid, block, lds, c.stream, ya); });
        }
    });
}

template <typename Real>
void launch_ystack(Context &c, const LinePlan &lp, int layers, const YStackArgs<Real> &ya) {
    const dim3 grid((unsigned)cdiv(ya.hx, ya.kpw)), block((unsigned)(3 * layers * ya.kpw * lp.threads));
    const size_t lds = (size_t)3 * layers * ya.kpw * line_slots(lp) * sizeof(cplx<Real>);
    with_line(lp, [&](auto NC) {
        constexpr int N = decltype(NC)::value;
        auto launch = [&](auto lc) {
            constexpr int L = decltype(lc)::value;
            if constexpr (ystack_fits<Real>(N, L))  // the plan's rule
                hipLaunchKernelGGL((ystack_kernel<Real, N, L>), grid, block, lds, c.stream, ya);
        };
        switch (layers) {
            case 1: launch(std::integral_constant<int, 1>{}); break;
            case 2: launch(std::integral_constant<int, 2>{}); break;
            case 3: launch(std::integral_constant<int, 3>{}); break;
            case 4: launch(std::integral_constant<int, 4>{}); break;
            default: launch(std::integral_constant<int, 5>{}); break;
        }
    });
}

template <typename Real>
void launch_film_tensor(Context &c, cplx<Real> *spec, const KernelView<Real> &K, int hx, int py, int64_t rows) {
    const dim3 g1((unsigned)cdiv((int64_t)hx * py, 256));
    launch_rec(c, nullptr, g1, dim3(256), 0, 1, K, [&] {
        hipLaunchKernelGGL((film_tensor_kernel<Real>), g1, dim3(256), 0, c.stream, spec, K, hx, py, rows);
    });
}

using R = FM_REAL;
template void launch_lines<R>(Context &, const LinePlan &, LineArgs<R>);
template void launch_class_inverse<R>(Context &, const LinePlan &, const LineArgs<R> &);
template void launch_yconv<R>(Context &, const YConvArgs<R> &);
template void launch_ystack<R>(Context &, const LinePlan &, int, const YStackArgs<R> &);
template void launch_film_tensor<R>(Context &, cplx<R> *, const KernelView<R> &, int, int, int64_t);

}  // namespace fm
