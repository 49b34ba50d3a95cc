// demag_x.hip -- x passes of the demag convolution: real-to-complex of two
// packed rows per line and back (see demag.hip for the pipeline).  Compiled
// once per field precision (FM_REAL).
#include "demag.hpp"

namespace fm {
namespace {

// Forward real-to-complex along x for xr rows (y0 .. y0+xr-1) of plane
// (c = blockIdx.z, z = blockIdx.y).  Rows 2j, 2j+1 are packed as a + i b;
// with Z = FFT(a + i b):  A_k = (Z_k + conj Z_{N-k}) / 2,
// B_k = (Z_k - conj Z_{N-k}) / (2i), k = 0..N/2, stored at spec[c][z][k][y].
template <typename Real>
__device__ __forceinline__ void xfwd_split(cplx<Real> zk, cplx<Real> zn, cplx<Real> &A, cplx<Real> &B) {
    const Real h = Real(0.5);
    A = {h * (zk.x + zn.x), h * (zk.y - zn.y)};
    B = {h * (zk.y + zn.y), h * (zn.x - zk.x)};
}

// (a + i b) w, rounded once, as the inputs of a plan at integer frequencies
// are: Ms m rounded to FP32 and multiplied by an FP32 factor gave smooth states
// up to a fifth more error (rms of H_demag against FP64, 128x128x4 mixed: 3.0e-7
// at integer frequencies, 3.6e-7 so, 3.4e-7 with this product and 3.2e-7 with the
// exact powers of x_roots as well; 44.3, 44.3, 45.0 and 44.9 us per step).
template <typename Real>
__device__ __forceinline__ cplx<Real> skewed(double a, double b, const cplx<double> &w) {
    return {Real(a * w.x - b * w.y), Real(a * w.y + b * w.x)};
}

// Runtime-planned lines.
template <typename Real, class Src>
__device__ __forceinline__ void xfwd_body_rt(const XArgs<Real> &a, const Src &src, cplx<Real> *spec, int c) {
    extern __shared__ unsigned char smem_raw[];
    cplx<Real> *lds = reinterpret_cast<cplx<Real> *>(smem_raw);
    const int LINES = a.xr >> 1;
    const int n = a.lp.n, ls = a.ls, T = a.lp.threads;
    const int tid = threadIdx.x, nthr = blockDim.x;
    const int y0 = blockIdx.x * a.xr, z = blockIdx.y;
    // the T lanes of packed line j (= tid / T, blockDim.x = LINES * T) load it
    const int jl = tid / T, t = tid - jl * T, ya = y0 + 2 * jl;
    cplx<Real> *line = lds + jl * ls;
    for (int x = t; x < n; x += T) {
        cplx<Real> v = {Real(0), Real(0)};
        if (x < a.n_in) {
            const double va = ya < a.rows ? src.at(c, z, ya, x) : 0.0;
            const double vb = ya + 1 < a.rows ? src.at(c, z, ya + 1, x) : 0.0;
            if (a.sw64) v = skewed<Real>(va, vb, a.sw64[x]);
            else v = {Real(va), Real(vb)};
        }
        line[lslot(a.lp, x)] = v;
    }
    __syncthreads();
    line_fft(line, a.lp, t, a.tw, false);
    __syncthreads();  // the unpack reads every line
    // lane (j, k) splits line j into rows 2j (A) and 2j + 1 (B) at kx = k
    for (int idx = tid; idx < a.g.hx * LINES; idx += nthr) {
        const int j = idx & (LINES - 1), k = idx >> (a.xr_log2 - 1), y = y0 + 2 * j;
        if (y >= a.rows) continue;
        cplx<Real> A, B;
        xfwd_split(lds[j * ls + lslot(a.lp, k)], lds[j * ls + lslot(a.lp, a.sw ? n - 1 - k : k == 0 ? 0 : n - k)], A, B);
        cplx<Real> *dst = spec + a.g.at(c, z, k, y);
        dst[0] = A;
        if (y + 1 < a.rows) dst[1] = B;
    }
}

// Roots ahead of the passes (FxRoots) for powers of two; the other lengths'
// last pass has up to seven butterflies per lane (400x100x2 FP64, 896 points:
// 66.2 us per step with the table, 67.7 with the roots ahead).  FP32 at the
// frequencies k + 1/2 forms EXACT powers: a state's mean, which integer
// frequencies keep at k = 0 away from every twiddle, spreads over all of them
// there (rms of H_demag, smooth state, 128x128x4: 3.4 and 3.2e-7; 500x250x8
// random 2.4 and 2.2e-7 at 152.5 and 155.7 us per step, three 512x512 films 156.3
// and 157.9).  At integer frequencies they would cost more than they give (all lines
// so: 512x512x1 mixed 74.3 -> 76.2 us per step, 512x512x8 341 -> 349).
template <typename Real, int N, bool SKEW>
__device__ __forceinline__ auto x_roots(int t, const cplx<Real> *tw) {
    constexpr bool EXACT = SKEW && sizeof(Real) == 4;
    if constexpr (fx_odd(N) == 1) return FxRoots<Real, N, EXACT>(t, tw);
    else if constexpr (EXACT) return FxTable<Real>{tw};
    else return tw;
}

// Scheduled lines.  A lane's loads are all in flight before the first pass,
// which takes them from registers.  In the unpack a lane keeps its line (FP32:
// pair of rows) and walks kx = k0 + u T, so each step is one pointer
// increment and one LDS read per side at a fixed distance.
template <typename Real, class Src, int N, bool SKEW>
__device__ __forceinline__ void xfwd_body(const XArgs<Real> &a, const Src &src, cplx<Real> *spec, int c) {
    constexpr int E = fx_elems(N), T = fx_lanes(N);
    extern __shared__ unsigned char smem_raw[];
    cplx<Real> *lds = reinterpret_cast<cplx<Real> *>(smem_raw);
    const int LINES = a.xr >> 1, ls = a.ls;
    const int tid = threadIdx.x;
    const int y0 = blockIdx.x * a.xr, z = blockIdx.y;
    {
        const int jl = tid / T, t = tid % T, ya = y0 + 2 * jl;
        cplx<Real> *line = lds + jl * ls;
        cplx<Real> v[E];
        // branch-free: clamped addresses, every load issued before any is
        // used; elements t + e T with e >= E / 2 lie in the zero padding
        // (n_in <= N / 2) and are not loaded
        const bool oka = ya < a.rows, okb = ya + 1 < a.rows;
        const int yA = oka ? ya : 0, yB = okb ? ya + 1 : 0;
        constexpr int H = SKEW ? E / 2 : 1;
        double va[H], vb[H];
#pragma unroll
        for (int e = 0; e < E / 2; ++e) {
            const int x = t + e * T;
            const bool okx = x < a.n_in;
            const int xs = okx ? x : 0;
            const double qa = src.load(c, z, yA, xs), qb = src.load(c, z, yB, xs);
            if constexpr (SKEW) {
                va[e] = (okx && oka) ? qa : 0.0;
                vb[e] = (okx && okb) ? qb : 0.0;
            } else {
                v[e] = {(okx && oka) ? Real(qa) : Real(0), (okx && okb) ? Real(qb) : Real(0)};
            }
        }
        if constexpr (SKEW) {
            cplx<double> w[H];
#pragma unroll
            for (int e = 0; e < H; ++e) w[e] = a.sw64[t + e * T];
#pragma unroll
            for (int e = 0; e < H; ++e) v[e] = skewed<Real>(va[e], vb[e], w[e]);
        }
#pragma unroll
        for (int e = E / 2; e < E; ++e) v[e] = {Real(0), Real(0)};
        const auto roots = x_roots<Real, N, SKEW>(t, a.tw);
        fx_first_pass<Real, N>(line, t, v, a.tw, false);
        fx_rest<Real, N>(line, t, roots, false);
    }
    __syncthreads();  // the unpack reads every line
    if constexpr (sizeof(Real) == 8) {
        // FP64: one 16-byte complex per lane, consecutive lanes on consecutive rows
        constexpr int KS = T / 2;  // LINES T lanes over 2 LINES rows
        const int yl = tid & (a.xr - 1), k0 = tid >> a.xr_log2, y = y0 + yl;
        if (y >= a.rows) return;
        const cplx<Real> *ln = lds + (yl >> 1) * ls;
        cplx<Real> *dst = spec + a.g.at(c, z, k0, y);
        const bool odd = (yl & 1) != 0;
        auto one = [&](int k, int kn, cplx<Real> *d) {
            // A or B of xfwd_split, selected by value (a select of the two
            // structs goes through scratch)
            const cplx<Real> zk = ln[fxslot<N>(k)], zn = ln[fxslot<N>(kn)];
            const Real p = odd ? zk.y : zk.x, q = odd ? zn.y : zn.x;
            const Real r = odd ? zn.x : zk.y, s = odd ? zk.x : zn.y;
            *d = {Real(0.5) * (p + q), Real(0.5) * (r - s)};
        };
#pragma unroll
        for (int u = 0; u < E; ++u) {
            const int k = k0 + u * KS;
            one(k, SKEW ? N - 1 - k : u == 0 && k0 == 0 ? 0 : N - k, dst + (int64_t)(u * KS) * a.g.pitch);
        }
        if (!SKEW && k0 == 0) one(N / 2, N / 2, dst + (int64_t)(N / 2) * a.g.pitch);
    } else {
        // lane (j, k) splits line j into rows 2j (A) and 2j + 1 (B); the two
        // are adjacent in memory (one 16-byte store when the row pitch is even)
        const int j = tid & (LINES - 1), k0 = tid >> (a.xr_log2 - 1), y = y0 + 2 * j;
        if (y >= a.rows) return;
        const bool pair16 = (a.g.pitch & 1) == 0, two = y + 1 < a.rows;
        const cplx<Real> *ln = lds + j * ls;
        cplx<Real> *dst = spec + a.g.at(c, z, k0, y);
        auto one = [&](int k, int kn, cplx<Real> *d) {
            cplx<Real> A, B;
            xfwd_split(ln[fxslot<N>(k)], ln[fxslot<N>(kn)], A, B);
            if (two && pair16) {
                *reinterpret_cast<float4 *>(d) = float4{float(A.x), float(A.y), float(B.x), float(B.y)};
            } else {
                d[0] = A;
                if (two) d[1] = B;
            }
        };
#pragma unroll
        for (int u = 0; u < E / 2; ++u) {
            const int k = k0 + u * T;
            one(k, SKEW ? N - 1 - k : u == 0 && k0 == 0 ? 0 : N - k, dst + (int64_t)(u * T) * a.g.pitch);
        }
        if (!SKEW && k0 == 0) one(N / 2, N / 2, dst + (int64_t)(N / 2) * a.g.pitch);
    }
}

// Component c = blockIdx.z.
template <typename Real, class Src, int N = 0, bool SKEW = false>
__global__ void __launch_bounds__(kMaxBlock) xfwd_kernel(XArgs<Real> a, Src src, cplx<Real> *spec) {
    if constexpr (N > 0) xfwd_body<Real, Src, N, SKEW>(a, src, spec, (int)blockIdx.z);
    else xfwd_body_rt<Real, Src>(a, src, spec, (int)blockIdx.z);
}

// Multi-instance form: instance blockIdx.z / zdiv of the table, component
// blockIdx.z % zdiv.  Each multi-instance kernel copies its instance's
// arguments into a local before the body runs, so the body sees invariant
// values exactly as the plain kernel does (a reference into the table would be
// re-read after the body's stores, which changes how the compiler contracts
// the arithmetic, and with it the last bit of FP32 results).
template <typename Real, class Src>
struct XFwdPack {
    XArgs<Real> a;
    Src src;
    cplx<Real> *spec;
};
template <typename Real, class Src, int N, bool SKEW>
__global__ void __launch_bounds__(kMaxBlock) xfwd_multi(const XFwdPack<Real, Src> *tab, int zdiv) {
    const XFwdPack<Real, Src> p = tab[blockIdx.z / zdiv];
    xfwd_body<Real, Src, N, SKEW>(p.a, p.src, p.spec, (int)(blockIdx.z % zdiv));
}

// Entry l of an argument array, l uniform in the workgroup (selects of
// scalars: an index that is not a constant would put the array in scratch).
template <typename T>
__device__ __forceinline__ T entry_of(const T (&v)[kStackPack], int l) {
    T r = v[0];
#pragma unroll
    for (int q = 1; q < kStackPack; ++q) r = q == l ? v[q] : r;
    return r;
}

// Layer blockIdx.z / 3 of a stack, component blockIdx.z % 3: one launch for
// all layers, whose single passes of a few microseconds leave the chip partly
// idle (three 512 x 512 films, FP32: 3 x 6.7 us one by one).
template <typename Real, typename S, bool GATHER, int N, bool SKEW>
__global__ void __launch_bounds__(kMaxBlock) xfwd_stack_kernel(XArgs<Real> a, StackMag<Real, S> p, cplx<Real> *spec) {
    using Src = MagSource<Real, S, GATHER>;
    const int l = (int)blockIdx.z / 3, c = (int)blockIdx.z - 3 * l;
    const Src src{entry_of(p.m, l), GATHER ? entry_of(p.mask, l) : nullptr, nullptr, entry_of(p.ms, l),
                  p.nx, p.ny, p.nz, p.n, nullptr};
    cplx<Real> *sp = spec + l * p.layer_stride;
    if constexpr (N > 0) xfwd_body<Real, Src, N, SKEW>(a, src, sp, c);
    else xfwd_body_rt<Real, Src>(a, src, sp, c);
}

// Inverse complex-to-real along x: Z_k = A_k + i B_k for k <= N/2 and the
// Hermitian continuation A_{N-k} = conj A_k; z = IFFT(Z); rows a = Re z,
// b = Im z.  Reads spec[c][z][k][y0..y0+xr-1].
// Runtime-planned lines.
template <typename Real, class Sink>
__device__ __forceinline__ void xinv_body_rt(const XArgs<Real> &a, const cplx<Real> *spec, const Sink &sink, int c) {
    extern __shared__ unsigned char smem_raw[];
    cplx<Real> *lds = reinterpret_cast<cplx<Real> *>(smem_raw);
    const int LINES = a.xr >> 1;
    const int n = a.lp.n, ls = a.ls, T = a.lp.threads;
    const int tid = threadIdx.x, nthr = blockDim.x;
    const int y0 = blockIdx.x * a.xr, z = blockIdx.y;
    const int hx = a.g.hx;
    // consecutive lanes read consecutive rows of one kx column, in batches of
    // four loads per lane in flight before their LDS writes
    constexpr int U = 4;
    for (int base = tid; base < hx * LINES; base += U * nthr) {
        cplx<Real> A[U], B[U];
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int idx = base + u * nthr;
            const int j = idx & (LINES - 1), k = idx >> (a.xr_log2 - 1);
            const int ya = y0 + 2 * j;
            A[u] = B[u] = {Real(0), Real(0)};
            if (idx < hx * LINES) {
                if (ya < a.rows) A[u] = spec[a.g.at(c, z, k, ya)];
                if (ya + 1 < a.rows) B[u] = spec[a.g.at(c, z, k, ya + 1)];
            }
        }
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int idx = base + u * nthr;
            if (idx >= hx * LINES) break;
            const int j = idx & (LINES - 1), k = idx >> (a.xr_log2 - 1);
            lds[j * ls + lslot(a.lp, k)] = {A[u].x - B[u].y, A[u].y + B[u].x};
            if (a.sw || (k > 0 && k < n - k)) lds[j * ls + lslot(a.lp, a.sw ? n - 1 - k : n - k)] = {A[u].x + B[u].y, B[u].x - A[u].y};
        }
    }
    __syncthreads();
    const int jl = tid / T, t = tid - jl * T;
    const cplx<Real> *line = lds + jl * ls;
    line_fft(lds + jl * ls, a.lp, t, a.tw, true);
    // the lanes of line jl store its rows 2 jl (real part) and 2 jl + 1
    const int ya = y0 + 2 * jl;
    for (int x = t; x < a.n_out; x += T) {
        cplx<Real> v = line[lslot(a.lp, x)];
        if (a.sw) v = cmul(v, cconj(a.sw[x]));
        if (ya < a.rows) sink(c, z, ya, x, v.x * a.scale);
        if (ya + 1 < a.rows) sink(c, z, ya + 1, x, v.y * a.scale);
    }
}

// Scheduled lines.  Every load of a lane (kx = k0 + u T of one row pair) is in
// flight before the first LDS write; the addresses and LDS slots advance by
// fixed steps.
template <typename Real, class Sink, int N, bool SKEW>
__device__ __forceinline__ void xinv_body(const XArgs<Real> &a, const cplx<Real> *spec, const Sink &sink, int c) {
    constexpr int E = fx_elems(N), T = fx_lanes(N), H = E / 2, U = SKEW ? H : H + 1;
    extern __shared__ unsigned char smem_raw[];
    cplx<Real> *lds = reinterpret_cast<cplx<Real> *>(smem_raw);
    const int LINES = a.xr >> 1, ls = a.ls;
    const int tid = threadIdx.x;
    const int y0 = blockIdx.x * a.xr, z = blockIdx.y;
    const auto roots = x_roots<Real, N, SKEW>(tid % T, a.tw);
    // SKEW, FP32: the factors of the outputs a lane stores, ahead of the passes
    // (128x128x8 mixed 53.4 and 52.4 us per step, 256x256x4 71.1 and 70.5)
    constexpr int Q4 = SKEW && sizeof(Real) == 4 ? (N / 2 + 4 * T - 1) / (4 * T) : 1;
    cplx<Real> wq[Q4][4];
    if constexpr (SKEW && sizeof(Real) == 4) {
#pragma unroll
        for (int q = 0; q < Q4; ++q)
#pragma unroll
            for (int e = 0; e < 4; ++e) wq[q][e] = a.sw[4 * (tid % T + q * T) + e];
    }
    {
        // lane (j, k0): rows 2j and 2j + 1; consecutive lanes read
        // consecutive rows of one kx column (a row pair is one 16-byte load
        // in FP32 when the row pitch is even); u = H is kx = N / 2
        const int j = tid & (LINES - 1), k0 = tid >> (a.xr_log2 - 1), ya = y0 + 2 * j;
        const bool oka = ya < a.rows, okb = ya + 1 < a.rows;
        const cplx<Real> *s = spec + a.g.at(c, z, k0, oka ? ya : 0);
        cplx<Real> A[U], B[U];
        auto off = [&](int u) { return (int64_t)(u < H ? u * T : k0 == 0 ? N / 2 : 0) * a.g.pitch; };
        if (sizeof(Real) == 4 && (a.g.pitch & 1) == 0) {
#pragma unroll
            for (int u = 0; u < U; ++u) {
                // an even row pitch and an even ya keep the pair 16-byte aligned
                const float4 q = *reinterpret_cast<const float4 *>(s + off(u));
                A[u] = {Real(q.x), Real(q.y)};
                B[u] = {Real(q.z), Real(q.w)};
            }
        } else {
            const int nb = okb ? 1 : 0;
#pragma unroll
            for (int u = 0; u < U; ++u) {
                A[u] = s[off(u)];
                B[u] = s[off(u) + nb];
            }
        }
        cplx<Real> *ln = lds + j * ls;
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int k = u < H ? k0 + u * T : N / 2;
            if (!oka) A[u] = {Real(0), Real(0)};
            if (!okb) B[u] = {Real(0), Real(0)};
            if (u < H || k0 == 0) ln[fxslot<N>(k)] = {A[u].x - B[u].y, A[u].y + B[u].x};
            if (SKEW || (u < H && (u > 0 || k0 > 0)))
                ln[fxslot<N>(SKEW ? N - 1 - k : N - k)] = {A[u].x + B[u].y, B[u].x - A[u].y};
        }
    }
    __syncthreads();
    const int jl = tid / T, t = tid % T;
    cplx<Real> *line = lds + jl * ls;
    {
        cplx<Real> v[E];
        fx_load<Real, N>(line, t, v);
        fx_first_pass<Real, N>(line, t, v, a.tw, true);
        fx_rest<Real, N>(line, t, roots, true);
    }
    auto out = [&](int x) -> cplx<Real> {
        if constexpr (SKEW) return cmul(line[fxslot<N>(x)], cconj(a.sw[x]));
        else return line[fxslot<N>(x)];
    };
    // the lanes of line jl store its rows 2 jl (real part) and 2 jl + 1
    const int ya = y0 + 2 * jl;
    if constexpr (std::is_same<Sink, FieldSink<float>>::value) {
        if (2 * a.n_out <= N && sink.masked() && (a.n_out & 3) == 0 && (sink.n & 3) == 0) {
            // four consecutive outputs of a row per lane: their mask bytes in
            // one 4-byte load, every mask word read before the first store,
            // and the values in one 16-byte store (rows start on 16-byte
            // boundaries: nx = n_out and n are multiples of four)
            constexpr int TT = T, Q = (N / 2 + 4 * TT - 1) / (4 * TT);
            const bool oka = ya < a.rows, okb = ya + 1 < a.rows;
            const int yA = oka ? ya : 0, yB = okb ? ya + 1 : 0;
            uint32_t ka[Q], kb[Q];
#pragma unroll
            for (int q = 0; q < Q; ++q) {
                const int x = 4 * (t + q * TT);
                const int xs = x < a.n_out ? x : 0;
                ka[q] = *reinterpret_cast<const uint32_t *>(sink.mask + ((int64_t)z * sink.ny + yA) * sink.nx + xs);
                kb[q] = *reinterpret_cast<const uint32_t *>(sink.mask + ((int64_t)z * sink.ny + yB) * sink.nx + xs);
            }
#pragma unroll
            for (int q = 0; q < Q; ++q) {
                const int x = 4 * (t + q * TT);
                if (x < a.n_out) {
                    cplx<Real> v[4];
#pragma unroll
                    for (int e = 0; e < 4; ++e) {
                        v[e] = line[fxslot<N>(x + e)];
                        if constexpr (SKEW) v[e] = cmul(v[e], cconj(wq[q][e]));
                    }
                    auto row = [&](uint32_t k, int part) {
                        float o[4];
#pragma unroll
                        for (int e = 0; e < 4; ++e)
                            o[e] = ((k >> (8 * e)) & 0xffu) ? (part ? v[e].y : v[e].x) * a.scale : 0.0f;
                        return float4{o[0], o[1], o[2], o[3]};
                    };
                    const int64_t i = ((int64_t)z * sink.ny + ya) * sink.nx + x;
                    if (oka) *reinterpret_cast<float4 *>(sink.out + (int64_t)c * sink.n + i) = row(ka[q], 0);
                    if (okb)
                        *reinterpret_cast<float4 *>(sink.out + (int64_t)c * sink.n + i + sink.nx) = row(kb[q], 1);
                }
            }
            return;
        }
    }
    {
        if (2 * a.n_out <= N && sink.masked()) {
            // at most E / 2 outputs per row and lane: every mask byte read
            // (clamped addresses) before the first store
            const bool oka = ya < a.rows, okb = ya + 1 < a.rows;
            const int yA = oka ? ya : 0, yB = okb ? ya + 1 : 0;
            uint8_t ka[H], kb[H];
#pragma unroll
            for (int e = 0; e < H; ++e) {
                const int x = t + e * T;
                const int xs = x < a.n_out ? x : 0;
                ka[e] = sink.keep(z, yA, xs);
                kb[e] = sink.keep(z, yB, xs);
            }
#pragma unroll
            for (int e = 0; e < H; ++e) {
                const int x = t + e * T;
                if (x < a.n_out) {
                    const cplx<Real> v = out(x);
                    if (oka) sink.put(c, z, ya, x, v.x * a.scale, ka[e]);
                    if (okb) sink.put(c, z, ya + 1, x, v.y * a.scale, kb[e]);
                }
            }
            return;
        }
    }
    if constexpr (std::is_same<Sink, FieldSink<float>>::value) {
        if (2 * a.n_out <= N && !sink.masked() && (a.n_out & 3) == 0 && (sink.n & 3) == 0) {
            // four consecutive outputs of a row per lane and one 16-byte
            // store (rows start on 16-byte boundaries: nx = n_out and n are
            // multiples of four)
            constexpr int TT = T, Q = (N / 2 + 4 * TT - 1) / (4 * TT);
#pragma unroll
            for (int q = 0; q < Q; ++q) {
                const int x = 4 * (t + q * TT);
                if (x >= a.n_out) break;
                cplx<Real> v[4];
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    v[e] = line[fxslot<N>(x + e)];
                    if constexpr (SKEW) v[e] = cmul(v[e], cconj(wq[q][e]));
                }
                const int64_t i = ((int64_t)z * sink.ny + ya) * sink.nx + x;
                if (ya < a.rows)
                    *reinterpret_cast<float4 *>(sink.out + (int64_t)c * sink.n + i) =
                        float4{v[0].x * a.scale, v[1].x * a.scale, v[2].x * a.scale, v[3].x * a.scale};
                if (ya + 1 < a.rows)
                    *reinterpret_cast<float4 *>(sink.out + (int64_t)c * sink.n + i + sink.nx) =
                        float4{v[0].y * a.scale, v[1].y * a.scale, v[2].y * a.scale, v[3].y * a.scale};
            }
            return;
        }
    }
    for (int x = t; x < a.n_out; x += T) {
        const cplx<Real> v = out(x);
        if (ya < a.rows) sink(c, z, ya, x, v.x * a.scale);
        if (ya + 1 < a.rows) sink(c, z, ya + 1, x, v.y * a.scale);
    }
}

template <typename Real, class Sink, int N = 0, bool SKEW = false>
__global__ void __launch_bounds__(kMaxBlock) xinv_kernel(XArgs<Real> a, const cplx<Real> *spec, Sink sink) {
    if constexpr (N > 0) xinv_body<Real, Sink, N, SKEW>(a, spec, sink, (int)blockIdx.z);
    else xinv_body_rt<Real, Sink>(a, spec, sink, (int)blockIdx.z);
}

template <typename Real, int N, bool SKEW>
__global__ void __launch_bounds__(kMaxBlock)
    xinv_stack_kernel(XArgs<Real> a, const cplx<Real> *spec, StackField<Real> p) {
    using Sink = FieldSink<Real>;
    const int l = (int)blockIdx.z / 3, c = (int)blockIdx.z - 3 * l;
    const Sink sink{entry_of(p.out, l), entry_of(p.mask, l), p.nx, p.ny, p.n};
    const cplx<Real> *sp = spec + l * p.layer_stride;
    if constexpr (N > 0) xinv_body<Real, Sink, N, SKEW>(a, sp, sink, c);
    else xinv_body_rt<Real, Sink>(a, sp, sink, c);
}

template <typename Real, class Sink>
struct XInvPack {
    XArgs<Real> a;
    const cplx<Real> *spec;
    Sink sink;
};
template <typename Real, class Sink, int N, bool SKEW>
__global__ void __launch_bounds__(kMaxBlock) xinv_multi(const XInvPack<Real, Sink> *tab, int zdiv) {
    const XInvPack<Real, Sink> p = tab[blockIdx.z / zdiv];
    xinv_body<Real, Sink, N, SKEW>(p.a, p.spec, p.sink, (int)(blockIdx.z % zdiv));
}

}  // namespace

template <typename Real, class Src>
void launch_xfwd(Context &c, const XArgs<Real> &xa, const Src &src, cplx<Real> *spec, unsigned row_groups,
                 unsigned planes, unsigned comps, size_t lds) {
    const dim3 grid(row_groups, planes, comps), block((unsigned)((xa.xr / 2) * xa.lp.threads));
    if constexpr (std::is_same<Src, NewellSource>::value) {
        hipLaunchKernelGGL((xfwd_kernel<Real, Src, 0>), grid, block, lds, c.stream, xa, src, spec);
    } else {
        with_line(xa.lp, [&](auto NC) {
            constexpr int N = decltype(NC)::value;
            const XFwdPack<Real, Src> pk{xa, src, spec};
            auto launch = [&](auto skew) {
                constexpr bool SK = decltype(skew)::value;
                const void *multi = nullptr;
                if constexpr (N > 0) multi = reinterpret_cast<const void *>(&xfwd_multi<Real, Src, N, SK>);
                launch_rec(c, multi, grid, block, lds, (int)comps, pk, [&] {
                    hipLaunchKernelGGL((xfwd_kernel<Real, Src, N, SK>), grid, block, lds, c.stream, xa, src, spec);
                });
            };
            if (xa.sw) launch(std::true_type{});
            else launch(std::false_type{});
        });
    }
}

template <typename Real>
void launch_xinv(Context &c, const XArgs<Real> &xa, const cplx<Real> *spec, const FieldSink<Real> &sink,
                 unsigned row_groups, unsigned planes, size_t lds) {
    const dim3 grid(row_groups, planes, 3), block((unsigned)((xa.xr / 2) * xa.lp.threads));
    with_line(xa.lp, [&](auto NC) {
        constexpr int N = decltype(NC)::value;
        const XInvPack<Real, FieldSink<Real>> pk{xa, spec, sink};
        auto launch = [&](auto skew) {
            constexpr bool SK = decltype(skew)::value;
            const void *multi = nullptr;
            if constexpr (N > 0) multi = reinterpret_cast<const void *>(&xinv_multi<Real, FieldSink<Real>, N, SK>);
            launch_rec(c, multi, grid, block, lds, 3, pk, [&] {
                hipLaunchKernelGGL((xinv_kernel<Real, FieldSink<Real>, N, SK>), grid, block, lds, c.stream, xa, spec,
                                   sink);
            });
        };
        if (xa.sw) launch(std::true_type{});
        else launch(std::false_type{});
    });
}

template <typename Real, typename S>
void launch_xfwd_stack(Context &c, const XArgs<Real> &xa, const StackMag<Real, S> &sm, bool masked, cplx<Real> *spec,
                       unsigned row_groups, unsigned planes, unsigned layers, size_t lds) {
    const dim3 grid(row_groups, planes, 3 * layers), block((unsigned)((xa.xr / 2) * xa.lp.threads));
    with_line(xa.lp, [&](auto NC) {
        constexpr int N = decltype(NC)::value;
        auto launch = [&](auto skew) {
            constexpr bool SK = decltype(skew)::value;
            if (masked)
                hipLaunchKernelGGL((xfwd_stack_kernel<Real, S, true, N, SK>), grid, block, lds, c.stream, xa, sm, spec);
            else
                hipLaunchKernelGGL((xfwd_stack_kernel<Real, S, false, N, SK>), grid, block, lds, c.stream, xa, sm, spec);
        };
        if (xa.sw) launch(std::true_type{});
        else launch(std::false_type{});
    });
}

template <typename Real>
void launch_xinv_stack(Context &c, const XArgs<Real> &xa, const cplx<Real> *spec, const StackField<Real> &sf,
                       unsigned row_groups, unsigned planes, unsigned layers, size_t lds) {
    const dim3 grid(row_groups, planes, 3 * layers), block((unsigned)((xa.xr / 2) * xa.lp.threads));
    with_line(xa.lp, [&](auto NC) {
        constexpr int N = decltype(NC)::value;
        if (xa.sw)
            hipLaunchKernelGGL((xinv_stack_kernel<Real, N, true>), grid, block, lds, c.stream, xa, spec, sf);
        else
            hipLaunchKernelGGL((xinv_stack_kernel<Real, N, false>), grid, block, lds, c.stream, xa, spec, sf);
    });
}

using R = FM_REAL;
#define FM_XFWD(SRC) \
    template void launch_xfwd<R, SRC>(Context &, const XArgs<R> &, const SRC &, cplx<R> *, unsigned, unsigned, \
                                      unsigned, size_t);
using SrcState = MagSource<R, double>;
using SrcStateG = MagSource<R, double, true>;
FM_XFWD(SrcState)
FM_XFWD(SrcStateG)
#ifdef FM_REAL_IS_FLOAT
using SrcStage = MagSource<R, float>;
using SrcStageG = MagSource<R, float, true>;
FM_XFWD(SrcStage)
FM_XFWD(SrcStageG)
#else
FM_XFWD(NewellSource)
#endif
template void launch_xfwd_stack<R, double>(Context &, const XArgs<R> &, const StackMag<R, double> &, bool, cplx<R> *,
                                           unsigned, unsigned, unsigned, size_t);
#ifdef FM_REAL_IS_FLOAT
template void launch_xfwd_stack<R, float>(Context &, const XArgs<R> &, const StackMag<R, float> &, bool, cplx<R> *,
                                          unsigned, unsigned, unsigned, size_t);
#endif
template void launch_xinv_stack<R>(Context &, const XArgs<R> &, const cplx<R> *, const StackField<R> &, unsigned,
                                   unsigned, unsigned, size_t);
template void launch_xinv<R>(Context &, const XArgs<R> &, const cplx<R> *, const FieldSink<R> &, unsigned, unsigned,
                             size_t);

}  // namespace fm
