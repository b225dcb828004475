// sx_multipole_cylinder.hip -- the cylinder average as sums per Bessel order.
//
//   A_lm(t) = sqrt(2 pi) sum_j b_j e^{i |z_j q_z|} F_lm(r_j q_r, phi_j - phi_q)
//
// (MPCylinderScatterDevice::scatter, multipole_scatter_device.cpp:900-987), F_lm
// being J_n cos or sin of n (phi - phi_q) times a constant, n = 2l or 2l - 1.
// All moments of a shell follow from, per order n,
//   G_n = sum_j b_j e^{i |z_j q_z|} J_n(r_j q_r) (cos n phi_j, sin n phi_j),
// four FP64 sums.  One wavefront takes a shell, 64 frames (lane = frame) and
// part of an atom range: the recurrences in n yield J_n and cos, sin of n phi one
// after the other, and each is used at once, so that nothing of the factors
// is stored (Miller's values wait in LDS for their norm).  Nothing is shared between
// shells except the atoms' coordinates, so there are no barriers.
//
// Bound by FP64 issue and the latency of its chains: per (atom, frame, shell)
// about 10 operations an order and 130 to 180 for the first two functions or
// Miller's recurrence; the sums of 21 orders leave two wavefronts a SIMD.
// 10,000 atoms x 2,000 frames, 41 moments, 10 shells: 6.8 ms, 7.2 ms a call (45 ms a
// call when a pre-pass stored J_n of every (shell, order, atom, frame), 34 GB here, and each
// wavefront of 8 moments formed its own phases).
#include <algorithm>
#include <cmath>

#include "sx_special_device.h"

namespace sx {

namespace {

constexpr int kBlockWaves = 4;
constexpr double kPi = 3.14159265358979323846;
// Upward recurrence from the asymptotic J_0, J_1 above this argument (and
// above the largest order), Miller's downward one up to it.
constexpr int kAsymptotic = 25;
// Terms of the asymptotic series in 1 / x, P and Q together: at x = 25 the
// first one left out is below 2e-17.
constexpr int kHankel = 20;

// c_k(nu) = prod_{i <= k} (4 nu^2 - (2i - 1)^2) / (k! 8^k), the coefficients of
// Hankel's expansion, with the signs of P = c_0 - c_2 / x^2 + .. and
// Q = (c_1 - c_3 / x^2 + ..) / x; first nu = 0, then nu = 1.
struct HankelTable {
    double p[2][kHankel / 2], q[2][kHankel / 2];
};
constexpr HankelTable make_hankel() {
    HankelTable h{};
    for (int nu = 0; nu < 2; ++nu) {
        double c = 1.0;
        for (int k = 0; k < kHankel; ++k) {
            const double v = (k / 2) & 1 ? -c : c;
            if (k & 1) h.q[nu][k / 2] = v;
            else h.p[nu][k / 2] = v;
            c *= (4.0 * nu * nu - (2.0 * k + 1.0) * (2.0 * k + 1.0)) / (8.0 * (k + 1.0));
        }
    }
    return h;
}
__constant__ const HankelTable kHankelTable = make_hankel();

// P and Q of order nu at 1 / x = ix, y = ix^2; the coefficients by scalar loads.
__device__ __forceinline__ void hankel_pq(int nu, double ix, double y, double &p, double &q) {
    int zo = nu;
    asm volatile("" : "+s"(zo));
    const auto P = uniform(&kHankelTable.p[0][0]) + zo * (kHankel / 2), C = uniform(&kHankelTable.q[0][0]) + zo * (kHankel / 2);
    p = P[kHankel / 2 - 1];
    q = C[kHankel / 2 - 1];
#pragma unroll
    for (int k = kHankel / 2 - 2; k >= 0; --k) {
        p = fma(p, y, P[k]);
        q = fma(q, y, C[k]);
    }
    q *= ix;
}

// J_0(x), J_1(x), x > kAsymptotic: sqrt(2 / (pi x)) (P cos chi - Q sin chi),
// chi = x - pi/4 - nu pi/2, from sin and cos of x.
__device__ __forceinline__ void bessel01_large(double x, double ix, double &j0, double &j1) {
    double s, c, p, q;
    sincos_reduced(x, s, c);
    // sqrt(1 / (pi x)): cos, sin(x - pi/4) = (c +- s) / sqrt(2) take the 2
    const double a = sqrt(ix * 0.31830988618379067154), y = ix * ix, u = a * (c + s), v = a * (s - c);
    hankel_pq(0, ix, y, p, q);
    j0 = fma(p, u, -q * v);
    hankel_pq(1, ix, y, p, q);
    j1 = fma(p, v, q * u);
}

struct CylinderSumArgs {
    const float *rr, *zz;       // r, z of every (atom, frame) in the axis frame
    const double2 *angle;       // cos phi, sin phi
    size_t NFp, NAp, range;
    const float *b;
    int per_shell_b;
    const double *q;            // q_r, phi_q, q_z per shell
    int ns, N1, groups;         // orders, groups of orders
    int sub, items, start;      // parts per range; wavefronts; start of Miller's recurrence (even)
    double large;               // arguments above take the upward recurrence
    double2 *parts;             // [split * sub][ns][N1][2][NFp]
};

// Orders [g NG, g NG + NG) of a shell.
template <int NG>
__global__ __launch_bounds__(kBlockWaves *kWave, 2) void cylinder_sums_kernel(CylinderSumArgs a) {
    __shared__ double mil[kBlockWaves][NG][kWave];
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
    // shells fastest: the wavefronts of a workgroup read the same atoms
    int i = blockIdx.x * kBlockWaves + wave;
    if (i >= a.items) return;  // no barriers
    const int s = i % a.ns;
    i /= a.ns;
    const int g = i % a.groups;
    i /= a.groups;
    const int tiles = (int)(a.NFp / kWave), z = i / tiles;
    const size_t t = (size_t)(i % tiles) * kWave + lane;
    const size_t r0 = (size_t)(z / a.sub) * a.range, r1 = min(a.NAp, r0 + a.range);
    const size_t len = r1 > r0 ? r1 - r0 : 0;
    const size_t j0 = r0 + len * (z % a.sub) / a.sub, j1 = r0 + len * (z % a.sub + 1) / a.sub;
    const int n0 = g * NG, nk = min(NG, a.N1 - n0);
    const auto Q = uniform(a.q) + 3 * s;
    const auto B = uniform(a.b) + (a.per_shell_b ? (size_t)s * a.NAp : 0);
    const double qr = Q[0], qz = Q[2];
    double *M = &mil[wave][0][lane];

    double acc[NG][4];
#pragma unroll
    for (int k = 0; k < NG; ++k)
#pragma unroll
        for (int v = 0; v < 4; ++v) acc[k][v] = 0.0;

#pragma unroll 1
    for (size_t j = j0; j < j1; ++j) {
        const float bj = B[j];
        if (bj == 0.f) continue;  // padding atoms and zero lengths add nothing
        const size_t e = j * a.NFp + t;
        const double x = (double)a.rr[e] * qr, zq = fabs((double)a.zz[e] * qz);
        const double2 an = a.angle[e];
        double ws, wc;
        sincos_reduced(zq, ws, wc);
        double wr = (double)bj * wc, wi = (double)bj * ws;
        // J_n of this group's orders into LDS, the lane's own column
        if (x > a.large) {
            const double ix = reciprocal(x), dx = ix + ix;
            double ja, jb, tn = 0.0;  // J_{n-1}, J_n, n
            bessel01_large(x, ix, jb, ja);
            ja = -ja;  // J_{-1} = -J_1
            auto step = [&]() {
                const double nx = fma(tn * dx, jb, -ja);
                ja = jb;
                jb = nx;
                tn += 1.0;
            };
#pragma unroll 1
            for (int n = 0; n < n0; ++n) step();
#pragma unroll 2
            for (int k = 0; k < nk; ++k) {
                M[k * kWave] = jb;
                step();
            }
        } else if (x < 1e-5) {
            // (x/2)^n / n! (1 - (x/2)^2 / (n + 1)), to (x/2)^4
            const double h = 0.5 * x;
            double p = 1.0;
#pragma unroll 1
            for (int n = 1; n <= n0; ++n) p *= h / (double)n;
#pragma unroll 1
            for (int k = 0; k < nk; ++k) {
                M[k * kWave] = p * (1.0 - h * h / (double)(n0 + k + 1));
                p *= h / (double)(n0 + k + 1);
            }
        } else {
            // from 1e-5 on the values stay in range from the start at 1e-280
            const double dx = 2.0 * reciprocal(x);
            double fp1 = 0.0, f = 1e-280, norm = 0.0;  // f_{n+1}, f_n
            int n = a.start;
            double tn = (double)n;
            // two steps, to the even order below; its value into the norm
            auto two = [&]() {
                const double f1 = fma(tn * dx, f, -fp1);
                const double f2 = fma((tn - 1.0) * dx, f1, -f);
                fp1 = f1;
                f = f2;
                tn -= 2.0;
                n -= 2;
                norm += f;
            };
#pragma unroll 1
            while (n > n0 + NG) two();
            // n even, at most n0 + NG; f_n and f_{n+1} of each step where they are in the group
#pragma unroll 1
            for (;;) {
                const int k = n - n0;
                if (k >= 0 && k < NG) M[k * kWave] = f;
                if (k >= -1 && k + 1 < NG) M[(k + 1) * kWave] = fp1;
                if (k <= 0 || n == 0) break;
                two();
            }
#pragma unroll 1
            while (n > 0) two();
            // J_0 + 2 sum J_2k = 1; f = f_0 is in the sum once
            const double inorm = reciprocal(fma(2.0, norm, -f));
            wr *= inorm;
            wi *= inorm;
        }
        // cos, sin of n phi by c_{n+1} = 2 cos(phi) c_n - c_{n-1}
        const double c2 = an.x + an.x;
        double cn = 1.0, sn = 0.0, cp = an.x, sp = -an.y;  // of n = 0 and -1
        auto turn = [&]() {
            const double cx = fma(c2, cn, -cp), sx = fma(c2, sn, -sp);
            cp = cn;
            sp = sn;
            cn = cx;
            sn = sx;
        };
#pragma unroll 1
        for (int n = 0; n < n0; ++n) turn();
#pragma unroll
        for (int k = 0; k < NG; ++k)
            if (k < nk) {
                const double jn = M[k * kWave];
                const double u = jn * wr, v = jn * wi;
                acc[k][0] = fma(u, cn, acc[k][0]);
                acc[k][1] = fma(v, cn, acc[k][1]);
                acc[k][2] = fma(u, sn, acc[k][2]);
                acc[k][3] = fma(v, sn, acc[k][3]);
                // formed here: moved behind the other orders, as the compiler
                // would, they keep every order's factors in registers
#pragma unroll
                for (int w = 0; w < 4; ++w) asm volatile("" : "+v"(acc[k][w]));
                turn();
            }
    }
#pragma unroll
    for (int k = 0; k < NG; ++k)
        if (k < nk) {
            double2 *p = a.parts + (((size_t)z * a.ns + s) * a.N1 + n0 + k) * 2 * a.NFp + t;
            p[0] = make_double2(acc[k][0], acc[k][1]);
            p[a.NFp] = make_double2(acc[k][2], acc[k][3]);
        }
}

__global__ __launch_bounds__(256) void cylinder_angles_kernel(const float *__restrict__ phi, size_t n,
                                                              double2 *__restrict__ angle) {
    const size_t e = (size_t)blockIdx.x * 256 + threadIdx.x;
    if (e >= n) return;
    double s, c;
    sincos((double)phi[e], &s, &c);
    angle[e] = make_double2(c, s);
}

// amp[(range, shell, moment)][t] from the sums of the moment's order.
__global__ __launch_bounds__(kWave) void cylinder_amplitudes_kernel(const double2 *__restrict__ parts, int sub, int ns,
                                                                    int N1, size_t NFp, int nmo,
                                                                    const int *__restrict__ moments,
                                                                    const double *__restrict__ q,
                                                                    float2 *__restrict__ amp) {
    const size_t t = (size_t)blockIdx.x * kWave + threadIdx.x;
    const int k = blockIdx.y, s = blockIdx.z % ns, sp = blockIdx.z / ns;
    const int l = moments[2 * k], m = moments[2 * k + 1];
    const int n = l == 0 ? 0 : (m <= 1 ? 2 * l : 2 * l - 1);
    double2 gc = make_double2(0.0, 0.0), gs = gc;
    for (int u = 0; u < sub; ++u) {
        const double2 *p = parts + (((size_t)(sp * sub + u) * ns + s) * N1 + n) * 2 * NFp + t;
        gc.x += p[0].x;
        gc.y += p[0].y;
        gs.x += p[NFp].x;
        gs.y += p[NFp].y;
    }
    double cq, sq;
    sincos((double)n * q[3 * s + 1], &sq, &cq);
    double f = sqrt(2.0 * kPi);
    double re = gc.x, im = gc.y;
    if (l > 0) {
        // cos or sin of n (phi - phi_q)
        if (m & 1) {
            re = gs.x * cq - gc.x * sq;
            im = gs.y * cq - gc.y * sq;
        } else {
            re = gc.x * cq + gs.x * sq;
            im = gc.y * cq + gs.y * sq;
        }
        f *= sqrt(2.0) * ((l & 1) ? -1.0 : 1.0);
        if (m >= 2) {  // times -i
            const double r = re;
            re = im;
            im = -r;
        }
    }
    amp[(((size_t)sp * ns + s) * nmo + k) * NFp + t] = make_float2((float)(f * re), (float)(f * im));
}

using CylinderFn = void (*)(CylinderSumArgs);
struct CylinderKernel {
    int ng;
    CylinderFn fn;
};
const CylinderKernel kKernels[] = {{5, cylinder_sums_kernel<5>},
                                   {9, cylinder_sums_kernel<9>},
                                   {13, cylinder_sums_kernel<13>},
                                   {17, cylinder_sums_kernel<17>},
                                   {21, cylinder_sums_kernel<21>}};

// Orders in as few equal groups as the largest kernel allows, in the
// smallest kernel that holds a group.
const CylinderKernel &cylinder_kernel(int N1, int *groups) {
    *groups = (N1 + 20) / 21;
    const int per = (N1 + *groups - 1) / *groups;
    for (const CylinderKernel &k : kKernels)
        if (k.ng >= per) return k;
    return kKernels[4];
}

}  // namespace

size_t cylinder_parts_bytes(int N1, size_t NFp, int ns, int split, int sub) {
    return sizeof(double2) * 2 * N1 * NFp * (size_t)ns * split * sub;
}

// Ranges are cut into parts, of at least 8 atoms, until the wavefronts fill
// whole rounds of the two a SIMD that fit.  (An atom's chain of recurrences takes
// 2 to 6 us and calls of few atoms leave SIMDs idle: 1,000 atoms x 100 frames x 1
// shell, whole calls with parts of 32 and of 8 atoms: (16, 0) alone 319 and 179 us,
// l <= 10 250 and 170 us.)
int cylinder_parts_per_range(int N1, size_t NFp, size_t NAp, int ns, int split, int cus) {
    int groups = 1;
    (void)cylinder_kernel(N1, &groups);
    const long base = (long)(NFp / kWave) * ns * groups * split, resident = 8L * cus;
    const long most = std::max<long>(1, std::min<long>(32, (long)(NAp / split / 8)));
    int sub = 1;
    double best = 0.0;
    for (long s = 1; s <= most; ++s) {
        const double rounds = (double)((base * s + resident - 1) / resident) / (double)s;
        if (s == 1 || rounds < best * 0.97) {
            best = rounds;
            sub = (int)s;
        }
    }
    return sub;
}

hipError_t launch_cylinder_sums(const MultipoleArgs &m, int N1, int sub, void *angles, void *parts,
                                hipStream_t stream) {
    const size_t n = m.NAp * m.NFp;
    if (N1 < 1 || N1 > kCylinderSumN1 || !cylinder_sums_grid_fits(m.nmo, m.ns, m.split)) return hipErrorInvalidValue;
    CylinderSumArgs a;
    a.rr = static_cast<const float *>(m.sph);
    const float *phi = a.rr + n;
    a.zz = a.rr + 2 * n;
    a.angle = static_cast<const double2 *>(angles);
    a.NFp = m.NFp;
    a.NAp = m.NAp;
    a.range = (m.NAp + m.split - 1) / m.split;
    a.b = m.b;
    a.per_shell_b = m.per_shell_b;
    a.q = m.qinfo;
    a.ns = m.ns;
    a.N1 = N1;
    const CylinderKernel &k = cylinder_kernel(N1, &a.groups);
    a.sub = sub;
    const int large = std::max(kAsymptotic, N1 - 1);
    a.large = (double)large;
    a.start = (large + 32 + (int)(2.0 * std::sqrt(2.0 * large)) + 1) & ~1;
    a.parts = static_cast<double2 *>(parts);
    const unsigned tiles = (unsigned)(m.NFp / kWave);
    const size_t items = (size_t)tiles * m.ns * a.groups * m.split * sub;
    if (items > (size_t)1 << 30) return hipErrorInvalidValue;
    a.items = (int)items;
    hipLaunchKernelGGL(cylinder_angles_kernel, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, stream, phi, n,
                       static_cast<double2 *>(angles));
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
    hipLaunchKernelGGL(k.fn, dim3((unsigned)((items + kBlockWaves - 1) / kBlockWaves)), dim3(kBlockWaves * kWave), 0,
                       stream, a);
    e = hipGetLastError();
    if (e != hipSuccess) return e;
    hipLaunchKernelGGL(cylinder_amplitudes_kernel, dim3(tiles, (unsigned)m.nmo, (unsigned)(m.split * m.ns)),
                       dim3(kWave), 0, stream, a.parts, sub, m.ns, N1, m.NFp, m.nmo, m.moments, m.qinfo, m.amp);
    return hipGetLastError();
}

}  // namespace sx
