// fft.hpp -- line FFTs staged in LDS for the demag convolution.
//
// A "line" is one 1-D transform of length n held in LDS.  A workgroup holds
// several lines; each line is worked on by `threads` = n / (smallest radix)
// lanes, one butterfly per lane per pass, so every pass is read-all /
// barrier / write-all in place and a line needs only n complex slots of LDS.
//
// The passes are Stockham autosort DIT (natural-order output, no bit
// reversal): for radix R and span ns (product of the radices already
// applied) butterfly j reads x[j + r n/R], multiplies by w^(r k n/(ns R))
// with k = j mod ns, applies the R-point DFT and writes x[(j/ns) ns R + k + r ns].
// Twiddles come from a per-length table w[t] = exp(-2 pi i t / n) rounded
// from long double on the host, so FP64 transforms carry only butterfly
// rounding.  Forward is unnormalised exp(-i...), inverse unnormalised
// exp(+i...), the convention of crates/fullmag-engine/src/lib.rs:343-386.
#pragma once

#include "common.hpp"

#include <type_traits>
#include <vector>

namespace fm {

constexpr int kMaxPass = 16;

struct LinePlan {
    int n = 0;        // line length
    int npass = 0;    // number of Stockham passes
    int threads = 0;  // lanes per line (each holds up to 16 complex values)
    int swz = 0;      // 1: LDS slots XOR-swizzled within 16-element blocks
    int fixed = 0;    // 1: the compile-time schedule of length n (fx_has) runs this line
    int radix[kMaxPass] = {};
};

// LDS slot of line element i.  With swz set (n a multiple of 16) element
// 16b + c lives at 16b + (c ^ (b & 15)): the stride-16 writes of the first
// Stockham pass then spread over 32 banks instead of 2.  Bijective within
// each 16-element block.
__host__ __device__ __forceinline__ int lslot(const LinePlan &lp, int i) { return lp.swz ? (i ^ ((i >> 4) & 15)) : i; }

// Chooses radices from {16, 8, 4, 2, 3, 5, 7, 11, 13}, plus any larger prime
// factor of n as a direct-sum pass, and the lanes per line: the fewest lanes
// such that no lane holds more than 16 complex values in any pass, or
// `min_lanes` if larger (capped at the largest pass's butterfly count);
// power-of-two radices are capped at max_radix (16, 8 or 4).  With `fixed`, a
// length that has a compile-time schedule gets that schedule's lanes and
// radices (default knobs only).  Returns false (with `err`) for lengths
// needing more than kMaxPass passes or 1024 lanes.
bool plan_line(int n, LinePlan &lp, std::string &err, int min_lanes = 1, int max_radix = 16, bool fixed = false);

// Padded length of a linear convolution of n cells: any length >= 2n - 1
// gives the same field, so 2n where that has a compile-time schedule, else
// the next length that has one if it is at most 4/3 of 2n, else 2n.  us per step
// at 2n with a runtime plan and padded: 768x768x1 mixed 432 and 161 (1536 and
// 2048 points), 65x65x65 FP64 537 and 189 (130 and 160), 129x129x4 mixed 671 and
// 54 (258 has the factor 43), 1536x300x1 mixed 253 and 123; along z, where
// lengths above 1024 have runtime plans either way, 32x32x800 mixed 795 and 666.
int pick_padded(int n);

// w[t] = exp(-2 pi i t / n), t in [0, n), correctly rounded from long double.
std::vector<cplx<double>> twiddle_table(int n);

// ---------------------------------------------------------------------------
// Device butterflies
// ---------------------------------------------------------------------------

// cos/sin of 2 pi m / 16, m = 0..15 (exact decimal expansions).
#define FM_C1 0.92387953251128675613
#define FM_S1 0.38268343236508977173
#define FM_H 0.70710678118654752440

template <typename T>
__device__ __forceinline__ cplx<T> w16(int m, bool inv) {
    // returns exp(-+ 2 pi i m / 16) (forward: minus sign)
    const T c[16] = {T(1), T(FM_C1), T(FM_H), T(FM_S1), T(0), T(-FM_S1), T(-FM_H), T(-FM_C1),
                     T(-1), T(-FM_C1), T(-FM_H), T(-FM_S1), T(0), T(FM_S1), T(FM_H), T(FM_C1)};
    const T s[16] = {T(0), T(FM_S1), T(FM_H), T(FM_C1), T(1), T(FM_C1), T(FM_H), T(FM_S1),
                     T(0), T(-FM_S1), T(-FM_H), T(-FM_C1), T(-1), T(-FM_C1), T(-FM_H), T(-FM_S1)};
    m &= 15;
    return {c[m], inv ? s[m] : -s[m]};
}

template <typename T>
__device__ __forceinline__ void dft2(cplx<T> &a, cplx<T> &b) {
    cplx<T> t = a;
    a = cadd(t, b);
    b = csub(t, b);
}

// In-place 4-point DFT of (v[0], v[s], v[2s], v[3s]).
template <typename T>
__device__ __forceinline__ void dft4(cplx<T> &a0, cplx<T> &a1, cplx<T> &a2, cplx<T> &a3, bool inv) {
    cplx<T> s0 = cadd(a0, a2), d0 = csub(a0, a2);
    cplx<T> s1 = cadd(a1, a3), d1 = csub(a1, a3);
    // forward: -i * d1 ; inverse: +i * d1
    cplx<T> jd1 = inv ? cplx<T>{-d1.y, d1.x} : cplx<T>{d1.y, -d1.x};
    a0 = cadd(s0, s1);
    a2 = csub(s0, s1);
    a1 = cadd(d0, jd1);
    a3 = csub(d0, jd1);
}

// 8-point DFT: inner 4-point DFTs over even/odd samples, twiddle w8^(r2 q1),
// outer 2-point DFTs: X[q1 + 4 q2].
template <typename T>
__device__ __forceinline__ void dft8(cplx<T> *v, bool inv) {
    cplx<T> u0[4] = {v[0], v[2], v[4], v[6]};
    cplx<T> u1[4] = {v[1], v[3], v[5], v[7]};
    dft4(u0[0], u0[1], u0[2], u0[3], inv);
    dft4(u1[0], u1[1], u1[2], u1[3], inv);
#pragma unroll
    for (int q1 = 1; q1 < 4; ++q1) u1[q1] = cmul(u1[q1], w16<T>(2 * q1, inv));
#pragma unroll
    for (int q1 = 0; q1 < 4; ++q1) {
        cplx<T> a = u0[q1], b = u1[q1];
        dft2(a, b);
        v[q1] = a;
        v[q1 + 4] = b;
    }
}

// 16-point DFT as 4 x 4: inner DFTs over r1 (stride 4), twiddle w16^(r2 q1),
// outer DFTs over r2: X[q1 + 4 q2].
template <typename T>
__device__ __forceinline__ void dft16(cplx<T> *v, bool inv) {
    cplx<T> u[4][4];
#pragma unroll
    for (int r2 = 0; r2 < 4; ++r2) {
        cplx<T> a0 = v[r2], a1 = v[r2 + 4], a2 = v[r2 + 8], a3 = v[r2 + 12];
        dft4(a0, a1, a2, a3, inv);
        u[r2][0] = a0; u[r2][1] = a1; u[r2][2] = a2; u[r2][3] = a3;
    }
#pragma unroll
    for (int r2 = 1; r2 < 4; ++r2)
#pragma unroll
        for (int q1 = 1; q1 < 4; ++q1) u[r2][q1] = cmul(u[r2][q1], w16<T>(r2 * q1, inv));
#pragma unroll
    for (int q1 = 0; q1 < 4; ++q1) {
        cplx<T> a0 = u[0][q1], a1 = u[1][q1], a2 = u[2][q1], a3 = u[3][q1];
        dft4(a0, a1, a2, a3, inv);
        v[q1] = a0; v[q1 + 4] = a1; v[q1 + 8] = a2; v[q1 + 12] = a3;
    }
}

// Odd prime R: direct DFT with roots from the line's twiddle table.
template <typename T, int R>
__device__ __forceinline__ void dft_prime(cplx<T> *v, const cplx<T> *tw, int n, bool inv) {
    cplx<T> out[R];
    const int step = n / R;
#pragma unroll
    for (int q = 0; q < R; ++q) {
        cplx<T> acc = v[0];
#pragma unroll
        for (int r = 1; r < R; ++r) {
            cplx<T> w = tw[((r * q) % R) * step];
            if (inv) w.y = -w.y;
            acc = cadd(acc, cmul(v[r], w));
        }
        out[q] = acc;
    }
#pragma unroll
    for (int q = 0; q < R; ++q) v[q] = out[q];
}

// Odd prime R = 3, 5, 7 with literal roots: the pair sums s_r = v_r + v_(R-r)
// carry the cosines and the differences d_r the sines.
template <typename T, int R>
__device__ __forceinline__ void dft_odd(cplx<T> *v, bool inv) {
    static_assert(R == 3 || R == 5 || R == 7, "literal roots");
    constexpr int H = (R - 1) / 2;
    constexpr double C3[1] = {-0.5}, S3[1] = {0.86602540378443864676};
    constexpr double C5[2] = {0.30901699437494742410, -0.80901699437494742410},
                     S5[2] = {0.95105651629515357212, 0.58778525229247312917};
    constexpr double C7[3] = {0.62348980185873353053, -0.22252093395631440429, -0.90096886790241912624},
                     S7[3] = {0.78183148246802980871, 0.97492791218182360702, 0.43388373911755812048};
    cplx<T> s[H], d[H];
#pragma unroll
    for (int r = 1; r <= H; ++r) {
        s[r - 1] = cadd(v[r], v[R - r]);
        d[r - 1] = csub(v[r], v[R - r]);
    }
    cplx<T> o0 = v[0], out[R];
#pragma unroll
    for (int r = 0; r < H; ++r) o0 = cadd(o0, s[r]);
#pragma unroll
    for (int q = 1; q <= H; ++q) {
        cplx<T> a = v[0], b{T(0), T(0)};
#pragma unroll
        for (int r = 1; r <= H; ++r) {
            const int m = (q * r) % R, i = (m <= H ? m : R - m) - 1;
            const T c = T(R == 3 ? C3[i % 1] : R == 5 ? C5[i % 2] : C7[i]);
            const T w0 = T(R == 3 ? S3[i % 1] : R == 5 ? S5[i % 2] : S7[i]);
            const T w = m <= H ? w0 : -w0;
            a.x += c * s[r - 1].x;
            a.y += c * s[r - 1].y;
            b.x += w * d[r - 1].x;
            b.y += w * d[r - 1].y;
        }
        // forward: a - i b at q, a + i b at R - q; the inverse swaps them
        const cplx<T> lo{a.x + b.y, a.y - b.x}, hi{a.x - b.y, a.y + b.x};
        out[q] = inv ? hi : lo;
        out[R - q] = inv ? lo : hi;
    }
    v[0] = o0;
#pragma unroll
    for (int q = 1; q < R; ++q) v[q] = out[q];
}

template <typename T, int R>
__device__ __forceinline__ void dft_any(cplx<T> *v, const cplx<T> *tw, int n, bool inv);

constexpr int inv_mod(int a, int m, int x = 1) { return (a * x) % m == 1 % m ? x : inv_mod(a, m, x + 1); }

// R = A B with coprime A and B (Good and Thomas): inputs (B i + A j) mod R,
// A-point DFTs over i, B-point DFTs over j, no twiddles; outputs at the index
// that is p mod A and q mod B.
template <typename T, int A, int B>
__device__ __forceinline__ void dft_coprime(cplx<T> *v, const cplx<T> *tw, int n, bool inv) {
    constexpr int R = A * B;
    // 1 mod A and 0 mod B; 0 mod A and 1 mod B
    constexpr int EA = B * inv_mod(B, A), EB = A * inv_mod(A, B);
    cplx<T> u[B][A];
#pragma unroll
    for (int j = 0; j < B; ++j) {
#pragma unroll
        for (int i = 0; i < A; ++i) u[j][i] = v[(B * i + A * j) % R];
        dft_any<T, A>(u[j], tw, n, inv);
    }
#pragma unroll
    for (int p = 0; p < A; ++p) {
        cplx<T> w[B];
#pragma unroll
        for (int j = 0; j < B; ++j) w[j] = u[j][p];
        dft_any<T, B>(w, tw, n, inv);
#pragma unroll
        for (int q = 0; q < B; ++q) v[(p * EA + q * EB) % R] = w[q];
    }
}

template <typename T, int R>
__device__ __forceinline__ void dft_any(cplx<T> *v, const cplx<T> *tw, int n, bool inv) {
    if constexpr (R == 1) {
        (void)v;
    } else if constexpr (R == 2) {
        dft2(v[0], v[1]);
    } else if constexpr (R == 4) {
        dft4(v[0], v[1], v[2], v[3], inv);
    } else if constexpr (R == 8) {
        dft8(v, inv);
    } else if constexpr (R == 16) {
        dft16(v, inv);
    } else if constexpr (R == 12) {
        dft_coprime<T, 4, 3>(v, tw, n, inv);
    } else if constexpr (R == 6) {
        dft_coprime<T, 2, 3>(v, tw, n, inv);
    } else if constexpr (R == 10) {
        dft_coprime<T, 2, 5>(v, tw, n, inv);
    } else if constexpr (R == 14) {
        dft_coprime<T, 2, 7>(v, tw, n, inv);
    } else if constexpr (R == 3 || R == 5 || R == 7) {
        dft_odd<T, R>(v, inv);
    } else {
        dft_prime<T, R>(v, tw, n, inv);
    }
}

// v[r] *= w^(r st), r = 1..R-1, where w^t = tw[t] (r st < n).  For
// power-of-two R the roots w^(2^b st) are read from the table; each other power
// is one product of an earlier power and a table root, so no twiddle carries
// more than three extra roundings.  EXACT reads w^3 and w^12 too and forms the
// others as one product of w^1, w^2 or w^3 and w^4, w^8 or w^12.
template <int R, bool EXACT>
constexpr int root_count() {
    return R == 2 ? 1 : R == 4 ? 2 : R == 8 ? (EXACT ? 4 : 3) : EXACT ? 6 : 4;
}
template <bool EXACT>
constexpr int root_power(int i) {
    return !EXACT ? 1 << i : i < 3 ? i + 1 : 4 * (i - 2);
}
// The same for power-of-two R with the roots in hand.
template <typename T, int R, bool EXACT = false>
__device__ __forceinline__ void twiddle_by(cplx<T> *v, const cplx<T> *roots, bool inv) {
    // conjugation for the inverse as a product with -1 (exact), so the
    // table loads stay out of any branch
    const T sg = inv ? T(-1) : T(1);
    cplx<T> w[R];
#pragma unroll
    for (int i = 0; i < root_count<R, EXACT>(); ++i) w[root_power<EXACT>(i)] = {roots[i].x, sg * roots[i].y};
#pragma unroll
    for (int r = 1; r < R; ++r) {
        const int low = r & -r;
        if (!EXACT || R == 4) {
            if (r != low) w[r] = cmul(w[r - low], w[low]);
        } else if (r > 4 && r % 4 != 0) {
            w[r] = cmul(w[r & ~3], w[r & 3]);
        }
        v[r] = cmul(v[r], w[r]);
    }
}
template <typename T, int R, bool EXACT = false>
__device__ __forceinline__ void twiddle(cplx<T> *v, const cplx<T> *tw, int st, bool inv) {
    if constexpr (R == 2 || R == 4 || R == 8 || R == 16) {
        constexpr int LB = root_count<R, EXACT>();
        cplx<T> pw[LB];
#pragma unroll
        for (int b = 0; b < LB; ++b) pw[b] = tw[root_power<EXACT>(b) * st];
        twiddle_by<T, R, EXACT>(v, pw, inv);
    } else {
        const T sg = inv ? T(-1) : T(1);
#pragma unroll
        for (int r = 1; r < R; ++r) {
            cplx<T> w = tw[r * st];
            w.y *= sg;
            v[r] = cmul(v[r], w);
        }
    }
}

// Butterflies one lane may hold in a radix-R pass (16 complex values).
template <int R>
constexpr int lane_butterflies() {
    return R >= 16 ? 1 : 16 / R;
}

// One Stockham pass over a line in LDS.  Every lane of the workgroup must
// call it (it contains barriers); `t` is the lane's index within its line
// and `nt` the number of lanes per line.  Lane t handles butterflies t,
// t + nt, ... (at most lane_butterflies<R>()); the planner guarantees that
// covers all n/R of them.
template <typename T, int R>
__device__ __forceinline__ void stockham_pass(cplx<T> *line, const LinePlan &lp, int ns, int t, const cplx<T> *tw, bool inv) {
    constexpr int MB = lane_butterflies<R>();
    const int n = lp.n, nt = lp.threads;
    const int nr = n / R;
    cplx<T> v[MB][R];
    int base[MB];
#pragma unroll
    for (int b = 0; b < MB; ++b) {
        const int j = t + b * nt;
        base[b] = -1;
        if (j < nr) {
            const int k = j % ns;
#pragma unroll
            for (int r = 0; r < R; ++r) v[b][r] = line[lslot(lp, j + r * nr)];
            if (k != 0) twiddle<T, R>(v[b], tw, k * (n / (ns * R)), inv);
            dft_any<T, R>(v[b], tw, n, inv);
            base[b] = (j / ns) * ns * R + k;
        }
    }
    __syncthreads();
#pragma unroll
    for (int b = 0; b < MB; ++b) {
        if (base[b] >= 0) {
#pragma unroll
            for (int r = 0; r < R; ++r) line[lslot(lp, base[b] + r * ns)] = v[b][r];
        }
    }
    __syncthreads();
}

// One Stockham pass of a prime radix R above 13, known only at run time.
// Lane t owns the output slots o = t + m nt (m < 16; the planner gives such
// a line at least n / 16 lanes).  Slot o = (j / ns) ns R + q ns + k of
// butterfly j (k = j mod ns) is sum_r x[j + r n/R] w^(r e) with
// e = k n/(ns R) + q n/R, the twiddle and the R-point DFT in one direct sum
// over table roots (O(n R) work per pass).
template <typename T>
__device__ __forceinline__ void stockham_pass_prime(cplx<T> *line, const LinePlan &lp, int ns, int t, const cplx<T> *tw,
                                                 bool inv, int R) {
    const int n = lp.n, nt = lp.threads, nr = n / R, st = n / (ns * R);
    cplx<T> out[16];
#pragma unroll
    for (int m = 0; m < 16; ++m) {
        const int o = t + m * nt;
        if (o < n) {
            const int k = o % ns, q = (o / ns) % R, jb = o / (ns * R);
            const int j = jb * ns + k, e = k * st + q * nr;
            cplx<T> acc = line[lslot(lp, j)];
            int idx = e;
            for (int r = 1; r < R; ++r) {
                cplx<T> w = tw[idx];
                if (inv) w.y = -w.y;
                acc = cadd(acc, cmul(line[lslot(lp, j + r * nr)], w));
                idx += e;
                if (idx >= n) idx -= n;
            }
            out[m] = acc;
        }
    }
    __syncthreads();
#pragma unroll
    for (int m = 0; m < 16; ++m) {
        const int o = t + m * nt;
        if (o < n) line[lslot(lp, o)] = out[m];
    }
    __syncthreads();
}

// Full transform of one line.  Uniform across the workgroup.
template <typename T>
__device__ __forceinline__ void line_fft(cplx<T> *line, const LinePlan &lp, int t, const cplx<T> *tw, bool inv) {
    int ns = 1;
    for (int p = 0; p < lp.npass; ++p) {
        const int R = lp.radix[p];
        switch (R) {
            case 2: stockham_pass<T, 2>(line, lp, ns, t, tw, inv); break;
            case 3: stockham_pass<T, 3>(line, lp, ns, t, tw, inv); break;
            case 4: stockham_pass<T, 4>(line, lp, ns, t, tw, inv); break;
            case 5: stockham_pass<T, 5>(line, lp, ns, t, tw, inv); break;
            case 7: stockham_pass<T, 7>(line, lp, ns, t, tw, inv); break;
            case 8: stockham_pass<T, 8>(line, lp, ns, t, tw, inv); break;
            case 11: stockham_pass<T, 11>(line, lp, ns, t, tw, inv); break;
            case 13: stockham_pass<T, 13>(line, lp, ns, t, tw, inv); break;
            case 16: stockham_pass<T, 16>(line, lp, ns, t, tw, inv); break;
            default: stockham_pass_prime<T>(line, lp, ns, t, tw, inv, R); break;
        }
        ns *= R;
    }
}

// ---------------------------------------------------------------------------
// Compile-time schedules: 2^a (32..4096) and 5, 3 and 7 times a power of two
// (10, 12 or 14 times 2 .. 64)
// ---------------------------------------------------------------------------
// With n, the radices and the spans known at compile time every index is a
// shift, mask or constant product, the swizzle is fixed and each kernel holds
// one pass's registers.  Powers of two use 16 elements per lane and the
// radices plan_line() picks with default knobs (radix-16 passes, then an 8/4
// tail; 2^(4a+1) uses 16^(a-1) 8 4), so a line transformed by either path
// carries the same roundings.  The other lengths give a lane E = 12, 10 or 14
// elements, the inputs of one first-pass butterfly of that radix, and keep a
// power-of-two number of lanes per line, so that lines never straddle a
// wavefront; the remaining power of two is one or two passes of radix 16, 8,
// 4 or 2 in which some lanes may have no butterfly.
constexpr int clog2(int n) { return n <= 1 ? 0 : 1 + clog2(n / 2); }
constexpr int fx_odd(int n) { return n % 2 == 0 ? fx_odd(n / 2) : n; }

// Elements per lane.
constexpr int fx_elems(int n) {
    const int o = fx_odd(n);
    return o == 1 ? 16 : o == 3 ? 12 : o == 5 ? 10 : 14;
}
constexpr int fx_lanes(int n) { return n / fx_elems(n); }

constexpr bool fx_has(int n) {
    if (n < 20 || n % 2 != 0) return false;
    const int o = fx_odd(n);
    if (o == 1) return n >= 32 && n <= 4096;
    if (o != 3 && o != 5 && o != 7) return false;
    const int e = fx_elems(n), t = n / e;
    return t * e == n && t >= 2 && t <= 64;
}

constexpr int p2_npass(int n) {
    return (clog2(n) % 4 == 0) ? clog2(n) / 4 : (clog2(n) % 4 == 1 && clog2(n) < 4) ? 1 : clog2(n) / 4 + 1;
}

constexpr int p2_radix(int n, int p) {
    const int a = clog2(n) / 4, r = clog2(n) % 4;
    if (r == 0) return 16;
    if (r == 1) return a == 0 ? 2 : p < a - 1 ? 16 : p == a - 1 ? 8 : 4;
    if (r == 2) return p < a ? 16 : 4;
    return p < a ? 16 : 8;
}

// Passes and radices of a scheduled length: for the lengths with an odd
// factor, fx_elems() and then 2, 4, 8, 16, 8 4 or 16 4.
constexpr int fx_npass(int n) {
    if (fx_odd(n) == 1) return p2_npass(n);
    return fx_lanes(n) <= 16 ? 2 : 3;
}
constexpr int fx_radix(int n, int p) {
    if (fx_odd(n) == 1) return p2_radix(n, p);
    if (p == 0) return fx_elems(n);
    const int t = fx_lanes(n);
    if (t <= 16) return t;
    return p == 1 ? t / 4 : 4;
}

// LDS slot of element i of a scheduled line: one slot of padding after every
// G = fx_radix(n, 0) elements.  Every later pass reads with stride n / R and
// writes with span NS, both multiples of G, so all the slots of a butterfly
// are its first one plus compile-time offsets (an XOR swizzle costs two VALU
// operations per access instead: a fifth of all VALU work of a 1024-point
// line), and the first pass's stride-G writes spread over the banks.
// 512x512x8: FP64 y lines 54 -> 49 us, FP32 x R2C 20.8 -> 18.9 us; the FP32 y
// lines stay at 28 us (151 MB, bound by memory).
constexpr int fx_pad(int n) { return fx_radix(n, 0); }
template <int N>
__host__ __device__ constexpr int fxslot(int i) {
    return i + i / fx_pad(N);
}
// LDS slots of one line.
constexpr int fx_size(int n) { return n + n / fx_pad(n); }

// Ordering point between the reads and the writes of a pass.  With at most
// 64 lanes per line (a power of two), every line lies inside one wavefront,
// whose LDS operations execute in program order, so a wavefront-scope fence
// (which also keeps the compiler from moving LDS accesses across it) replaces
// the workgroup barrier and the other lines' waves run on independently.
// Callers that read other lines after the transform add their own barrier.
template <int N>
__device__ __forceinline__ void pass_sync() {
    if constexpr (fx_lanes(N) <= 64) {
        __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
        __builtin_amdgcn_wave_barrier();
    } else {
        __syncthreads();
    }
}

// The roots of a lane's butterflies in the passes after the first, loaded
// beside the line's inputs; a pass takes the table or this.  A pass that reads
// the table when it needs the roots waits for the L2 once more.  The x passes
// carry them (their workgroups of up to 512 lanes leave few others to cover
// the wait): per step 512x512x8 FP64 646.7 -> 637.7 us, mixed 345.9 -> 343.9,
// 250x150x6 single 94.8 -> 93.5.  In the film's y convolution they cost
// registers (512x512x1 FP64 90.1 -> 91.9 us) and in the slab kernel they gave
// nothing.
template <typename T, int N, bool EXACT = false>
struct FxRoots {
    static_assert(fx_npass(N) <= 3, "two passes of roots");
    cplx<T> w[2][8];
    __device__ __forceinline__ FxRoots(int t, const cplx<T> *tw) {
        if constexpr (fx_npass(N) > 1) fetch<1, fx_radix(N, 0)>(t, tw);
        if constexpr (fx_npass(N) > 2) fetch<2, fx_radix(N, 0) * fx_radix(N, 1)>(t, tw);
    }
    template <int P, int NS>
    __device__ __forceinline__ void fetch(int t, const cplx<T> *tw) {
        constexpr int R = fx_radix(N, P), NT = fx_lanes(N), NR = N / R, MB = (NR + NT - 1) / NT;
        constexpr int LB = root_count<R, EXACT>();
        static_assert(MB * LB <= 8, "roots of one pass");
#pragma unroll
        for (int b = 0; b < MB; ++b) {
            const int j0 = t + b * NT, j = MB * NT == NR || j0 < NR ? j0 : 0;
#pragma unroll
            for (int i = 0; i < LB; ++i) w[P - 1][b * LB + i] = tw[root_power<EXACT>(i) * ((j % NS) * (N / (NS * R)))];
        }
    }
};

// The table, its powers EXACT.
template <typename T>
struct FxTable {
    const cplx<T> *tw;
};

// One pass.  LAST: output element i goes to put(i, value) instead of LDS, and
// only the elements i < N / OUT_DIV are produced.
template <typename T, int N, int P, int R, int NS, bool LAST, int OUT_DIV, class Tw, class Put>
__device__ __forceinline__ void fx_pass(cplx<T> *line, int t, const Tw &tw, bool inv, Put &&put) {
    constexpr int G = fx_pad(N), NT = fx_lanes(N), NR = N / R, ST = N / (NS * R);
    constexpr int MB = (NR + NT - 1) / NT;  // butterflies per lane; the last may be beyond NR
    constexpr bool FULL = MB * NT == NR;
    static_assert(NR % G == 0 && NS % G == 0, "slots of a butterfly are equally spaced");
    cplx<T> v[MB][R];
    int base[MB];
#pragma unroll
    for (int b = 0; b < MB; ++b) {
        const int j0 = t + b * NT;
        const int j = FULL || j0 < NR ? j0 : 0;  // an idle lane repeats butterfly 0 and drops it
        const int k = j % NS;
        const cplx<T> *p = line + fxslot<N>(j);
#pragma unroll
        for (int r = 0; r < R; ++r) v[b][r] = p[r * (NR + NR / G)];
        // k = 0 multiplies by the table's exact w^0 = 1 (no branch: lanes of
        // one wave differ in k, and a branch would split the table loads)
        if constexpr (std::is_same<Tw, FxRoots<T, N, true>>::value)
            twiddle_by<T, R, true>(v[b], tw.w[P - 1] + b * root_count<R, true>(), inv);
        else if constexpr (std::is_same<Tw, FxRoots<T, N>>::value)
            twiddle_by<T, R>(v[b], tw.w[P - 1] + b * root_count<R, false>(), inv);
        else if constexpr (std::is_same<Tw, FxTable<T>>::value)
            twiddle<T, R, true>(v[b], tw.tw, k * ST, inv);
        else
            twiddle<T, R>(v[b], tw, k * ST, inv);
        dft_any<T, R>(v[b], nullptr, N, inv);
        base[b] = (j / NS) * NS * R + k;
    }
    if constexpr (!LAST) pass_sync<N>();
#pragma unroll
    for (int b = 0; b < MB; ++b)
        if (FULL || t + b * NT < NR) {
            if constexpr (LAST) {
#pragma unroll
                for (int r = 0; r < R / OUT_DIV; ++r) put(base[b] + r * NS, v[b][r]);
            } else {
                cplx<T> *p = line + fxslot<N>(base[b]);
#pragma unroll
                for (int r = 0; r < R; ++r) p[r * (NS + NS / G)] = v[b][r];
            }
        }
    if constexpr (!LAST) pass_sync<N>();
}

struct FxNoPut {
    template <typename T>
    __device__ __forceinline__ void operator()(int, const cplx<T> &) const {}
};

// Passes P.. of the schedule; the last through `put` when STORE.
template <typename T, int N, int P, int NS, bool STORE, int OUT_DIV, class Tw, class Put>
__device__ __forceinline__ void fx_passes(cplx<T> *line, int t, const Tw &tw, bool inv, Put &&put) {
    if constexpr (P < fx_npass(N)) {
        constexpr int R = fx_radix(N, P);
        fx_pass<T, N, P, R, NS, STORE && P + 1 == fx_npass(N), OUT_DIV>(line, t, tw, inv, put);
        fx_passes<T, N, P + 1, NS * R, STORE, OUT_DIV>(line, t, tw, inv, put);
    }
}

// The first pass, fed from registers: lane t holds elements t + e T (e < E),
// which are exactly the inputs of its E / R butterflies.  fx_rest runs the
// other passes, leaving the transform in the line; fx_rest_put hands its
// elements i < N / OUT_DIV to put(i, value) from registers.
template <typename T, int N>
__device__ __forceinline__ void fx_first_pass(cplx<T> *line, int t, const cplx<T> v[], const cplx<T> *tw, bool inv) {
    constexpr int R = fx_radix(N, 0), E = fx_elems(N), B = E / R, NT = fx_lanes(N);
    static_assert(B * R == E, "whole butterflies per lane");
#pragma unroll
    for (int b = 0; b < B; ++b) {
        cplx<T> u[R];
#pragma unroll
        for (int r = 0; r < R; ++r) u[r] = v[b + r * B];
        dft_any<T, R>(u, tw, N, inv);
        cplx<T> *p = line + (t + b * NT) * (R + 1);
#pragma unroll
        for (int r = 0; r < R; ++r) p[r] = u[r];
    }
    pass_sync<N>();
}
template <typename T, int N, class Tw>
__device__ __forceinline__ void fx_rest(cplx<T> *line, int t, const Tw &tw, bool inv) {
    fx_passes<T, N, 1, fx_radix(N, 0), false, 1>(line, t, tw, inv, FxNoPut{});
}
template <typename T, int N, int OUT_DIV, class Tw, class Put>
__device__ __forceinline__ void fx_rest_put(cplx<T> *line, int t, const Tw &tw, bool inv, Put &&put) {
    fx_passes<T, N, 1, fx_radix(N, 0), true, OUT_DIV>(line, t, tw, inv, put);
}

// Transform of a line in LDS, through the first pass's registers (its slots
// are this lane's own until pass_sync).
template <typename T, int N>
__device__ __forceinline__ void fx_load(const cplx<T> *line, int t, cplx<T> v[]) {
#pragma unroll
    for (int e = 0; e < fx_elems(N); ++e) v[e] = line[fxslot<N>(t + e * fx_lanes(N))];
    pass_sync<N>();
}

}  // namespace fm
