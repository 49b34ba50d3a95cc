// newell.hip -- Newell-Williams-Dunlop demag tensor on the displacement
// octant (FP64), for the in-library kernel build.
//
// Same tensor as crates/fullmag-fdm-demag/src/newell.rs:254-519 (Boris-style
// f/g tables, 27-point second-difference stencil with Kahan-Neumaier
// summation, point-dipole far field beyond 40 cells).  The reference places
// the octant into all eight sign octants of the padded grid on the host; here
// only the octant is produced and the device mirrors it with the parity signs
// while it transforms (demag.hip, NewellSource), so the host never holds the
// padded arrays.  A nonzero z_offset gives the cross-layer kernel of layers
// that far apart in z (newell.rs:528-651: every z coordinate, of the f/g
// tables and of the far field, is offset).
//
// The host's threads evaluate the tables (at most 42^3 entries of six
// functions with three logarithms and arc tangents each), the device takes
// the second differences and the far field, one lane per value.  The
// differences cancel to about 1e-4 of the table values, so another
// logarithm's last bit shows in the field at 1e-12: the device evaluating the
// tables with its own functions moved fields by up to 8e-12 and is not used.
// Sums, divisions and square roots round alike on both (this file is compiled
// without contraction), so the octant is the one a host loop over all cells
// gives, bit for bit.  Set-up of a 128x128x4 FP64 backend among other work:
// 8.0 ms with the whole octant on the host, 2.5 ms so.
#include "context.hpp"

#include <algorithm>
#include <cmath>
#include <thread>

namespace fm {
namespace {

// f(x, y, z): newell.rs:21-61 (log1p form, valid for signed arguments).
double nw_f(double x, double y, double z) {
    const double x2 = x * x, y2 = y * y, z2 = z * z;
    const double r2 = x2 + y2 + z2;
    if (r2 < 1e-300) return 0.0;
    const double r = std::sqrt(r2);
    double v = (2.0 * x2 - y2 - z2) * r / 6.0;
    const double sxz = x2 + z2, sxy = x2 + y2;
    if (sxz > 1e-300) {
        const double t = 2.0 * y * (y + r) / sxz;
        if (t > -1.0) v += y * (z2 - x2) / 4.0 * std::log1p(t);
    }
    if (sxy > 1e-300) {
        const double t = 2.0 * z * (z + r) / sxy;
        if (t > -1.0) v += z * (y2 - x2) / 4.0 * std::log1p(t);
    }
    if (std::fabs(x) > 1e-300) v -= x * y * z * std::atan(y * z / (x * r));
    return v;
}

// g(x, y, z): newell.rs:63-123.
double nw_g(double x, double y, double z) {
    const double x2 = x * x, y2 = y * y, z2 = z * z;
    const double r2 = x2 + y2 + z2;
    if (r2 < 1e-300) return 0.0;
    const double r = std::sqrt(r2);
    double v = -x * y * r / 3.0;
    const double sxy = x2 + y2, syz = y2 + z2, sxz = x2 + z2;
    if (sxy > 1e-300) {
        const double t = 2.0 * z * (z + r) / sxy;
        if (t > -1.0) v += x * y * z * std::log1p(t) / 2.0;
    }
    if (syz > 1e-300) {
        const double t = 2.0 * x * (x + r) / syz;
        if (t > -1.0) v += y * (3.0 * z2 - y2) * std::log1p(t) / 12.0;
    }
    if (sxz > 1e-300) {
        const double t = 2.0 * y * (y + r) / sxz;
        if (t > -1.0) v += x * (3.0 * z2 - x2) * std::log1p(t) / 12.0;
    }
    if (std::fabs(z) > 1e-300) v -= z2 * z / 6.0 * std::atan(x * y / (z * r));
    if (std::fabs(y) > 1e-300) v -= y2 * z / 2.0 * std::atan(x * z / (y * r));
    if (std::fabs(x) > 1e-300) v -= x2 * z / 2.0 * std::atan(y * z / (x * r));
    return v;
}

constexpr int kFar = 40;  // newell.rs:229

// One base function's values at grid offsets -1 .. min(n, 40) along each axis.
struct Table {
    int sx, sy;
    const double *v;  // value at grid offset (i-1, j-1, k-1)
    __device__ double at(int i, int j, int k) const { return v[((int64_t)k * sy + j) * sx + i]; }
};

// Second difference over the 27 neighbours of (i, j, k) with weights
// 8 / -4 / 2 / -1 (centre / faces / edges / corners), summed with
// Kahan-Neumaier compensation: newell.rs:150-203.  Table offsets are +1.
__device__ double stencil(const Table &t, int i, int j, int k, double hx, double hy, double hz) {
    double sum = 0.0, comp = 0.0;
    auto add = [&](double val) {
        const double s = sum + val;
        if (fabs(sum) >= fabs(val)) comp += (sum - s) + val;
        else comp += (val - s) + sum;
        sum = s;
    };
    const int a = i + 1, b = j + 1, c = k + 1;
    add(8.0 * t.at(a, b, c));
    add(-4.0 * t.at(a + 1, b, c)); add(-4.0 * t.at(a - 1, b, c));
    add(-4.0 * t.at(a, b + 1, c)); add(-4.0 * t.at(a, b - 1, c));
    add(-4.0 * t.at(a, b, c + 1)); add(-4.0 * t.at(a, b, c - 1));
    add(2.0 * t.at(a - 1, b - 1, c)); add(2.0 * t.at(a - 1, b + 1, c));
    add(2.0 * t.at(a + 1, b - 1, c)); add(2.0 * t.at(a + 1, b + 1, c));
    add(2.0 * t.at(a - 1, b, c - 1)); add(2.0 * t.at(a - 1, b, c + 1));
    add(2.0 * t.at(a + 1, b, c - 1)); add(2.0 * t.at(a + 1, b, c + 1));
    add(2.0 * t.at(a, b - 1, c - 1)); add(2.0 * t.at(a, b - 1, c + 1));
    add(2.0 * t.at(a, b + 1, c - 1)); add(2.0 * t.at(a, b + 1, c + 1));
    add(-t.at(a - 1, b - 1, c - 1)); add(-t.at(a - 1, b - 1, c + 1));
    add(-t.at(a - 1, b + 1, c - 1)); add(-t.at(a + 1, b - 1, c - 1));
    add(-t.at(a - 1, b + 1, c + 1)); add(-t.at(a + 1, b - 1, c + 1));
    add(-t.at(a + 1, b + 1, c - 1)); add(-t.at(a + 1, b + 1, c + 1));
    return (sum + comp) / (4.0 * kPi * hx * hy * hz);
}

// Point-dipole limit: newell.rs:212-226.
__device__ double dip_diag(double x, double y, double z, double vol) {
    const double r2 = x * x + y * y + z * z, r = sqrt(r2), r3 = r2 * r;
    return (1.0 / r3 - 3.0 * x * x / (r3 * r2)) / (4.0 * kPi) * vol;
}
__device__ double dip_off(double x, double y, double z, double vol) {
    const double r2 = x * x + y * y + z * z, r = sqrt(r2), r5 = r2 * r2 * r;
    return -3.0 * x * y / (4.0 * kPi * r5) * vol;
}

struct OctantArgs {
    int nx, ny, nz, sx, sy, sz;
    double dx, dy, dz, z0;
};

// Component blockIdx.y at one displacement per lane; 27 cached table reads or
// one square root and two divisions per 8 bytes written.
__global__ void __launch_bounds__(256) newell_octant_kernel(OctantArgs a, const double *tables, double *out) {
    const int64_t per = (int64_t)a.nx * a.ny * a.nz, o = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (o >= per) return;
    const int i = (int)(o % a.nx), j = (int)(o / a.nx % a.ny), k = (int)(o / ((int64_t)a.nx * a.ny));
    const int c = (int)blockIdx.y;
    const bool far = i >= kFar || j >= kFar || k >= kFar || i * i + j * j + k * k >= kFar * kFar;
    double v;
    if (far) {
        const double x = i * a.dx, y = j * a.dy, z = k * a.dz + a.z0, vol = a.dx * a.dy * a.dz;
        switch (c) {
            case 0: v = dip_diag(x, y, z, vol); break;
            case 1: v = dip_diag(y, x, z, vol); break;
            case 2: v = dip_diag(z, y, x, vol); break;
            case 3: v = dip_off(x, y, z, vol); break;
            case 4: v = dip_off(x, z, y, vol); break;
            default: v = dip_off(y, z, x, vol); break;
        }
    } else {
        const Table t{a.sx, a.sy, tables + (int64_t)c * a.sx * a.sy * a.sz};
        // argument order of the cell sizes follows newell.rs:386-392
        switch (c) {
            case 1: v = stencil(t, i, j, k, a.dy, a.dx, a.dz); break;
            case 2: v = stencil(t, i, j, k, a.dz, a.dy, a.dx); break;
            case 4: v = stencil(t, i, j, k, a.dx, a.dz, a.dy); break;
            case 5: v = stencil(t, i, j, k, a.dy, a.dz, a.dx); break;
            default: v = stencil(t, i, j, k, a.dx, a.dy, a.dz); break;
        }
    }
    out[(int64_t)c * per + o] = v;
}

OctantArgs octant_args(int nx, int ny, int nz, double dx, double dy, double dz, double z0) {
    return OctantArgs{nx, ny, nz, std::min(nx, kFar) + 2, std::min(ny, kFar) + 2, std::min(nz, kFar) + 2, dx, dy, dz, z0};
}

}  // namespace

size_t newell_scratch(int nx, int ny, int nz) {
    const OctantArgs a = octant_args(nx, ny, nz, 0, 0, 0, 0);
    return 6 * (size_t)a.sx * a.sy * a.sz;
}

bool newell_octant(Context &c, int nx, int ny, int nz, double dx, double dy, double dz, double z_offset,
                   double *scratch, double *out, std::string &err) {
    const OctantArgs a = octant_args(nx, ny, nz, dx, dy, dz, z_offset);
    const size_t per = (size_t)a.sx * a.sy * a.sz;
    std::vector<double> t(6 * per);
    const int rows = a.sy * a.sz;
    auto fill = [&](int first, int step) {
        for (int row = first; row < rows; row += step) {
            const double y = (row % a.sy - 1.0) * dy, z = (row / a.sy - 1.0) * dz + z_offset;
            double *v = t.data() + (size_t)row * a.sx;
            for (int i = 0; i < a.sx; ++i, ++v) {
                const double x = (i - 1.0) * dx;
                v[0] = nw_f(x, y, z);
                v[per] = nw_f(y, x, z);
                v[2 * per] = nw_f(z, y, x);
                v[3 * per] = nw_g(x, y, z);
                v[4 * per] = nw_g(x, z, y);
                v[5 * per] = nw_g(y, z, x);
            }
        }
    };
    // 0.2 us per point, and up to a millisecond until a thread runs on an idle
    // core: at 10,584 points (128x128x4) a set-up among other work takes 2.8 ms
    // with one thread, 2.5 ms with two or three, 2.6 to 6.5 with four, 5.1 to
    // 6.8 with eight or sixteen
    const int nt = (int)std::min<size_t>({std::max(1u, std::thread::hardware_concurrency()), 8, 1 + per / 4096});
    std::vector<std::thread> th;
    for (int i = 1; i < nt; ++i) th.emplace_back(fill, i, nt);
    fill(0, nt);
    for (auto &x : th) x.join();
    if (!ctx_upload(c, scratch, t.data(), t.size() * sizeof(double), "hipMemcpy(newell tables)", err)) return false;
    const int64_t cells = (int64_t)nx * ny * nz;
    hipLaunchKernelGGL(newell_octant_kernel, dim3((unsigned)cdiv(cells, 256), 6), dim3(256), 0, c.stream, a, scratch,
                       out);
    return hip_ok(hipGetLastError(), "newell octant launch", err);
}

}  // namespace fm
