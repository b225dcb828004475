// sx_multipole_sphere.hip -- the sphere average as sums over products of a
// radial and an angular factor.
//
//   A_lm(t) = 4 pi i^l sum_j [b_j j_l(|q| r_j)] conj(Y_lm(theta_j, phi_j))
//
// (MPSphereScatterDevice::scatter, multipole_scatter_device.cpp:428-498).
// Every term is the product of a factor of (shell, degree) and one of
// (degree, order), so a workgroup forms each factor once per (atom, frame):
// its wavefronts first put the Bessel functions of a few shells, the powers
// u^m, u = -sin(theta) e^{i phi}, and cos(theta) of a few atoms x 64 frames into LDS, then
// each sums the products of its own (degree, order) pairs in registers,
// lane = frame.  Both signs of an order come from the same sums.
//
// Legendre functions by the recurrence in the degree, scaled such that one of
// its coefficients is 1: P_lm ~ s_lm u^m T_lm with
//   T_l = alpha_lm cos(theta) T_{l-1} - T_{l-2},  T_m = 1,
// two FP64 operations a degree; s_lm and the normalisation multiply the
// finished sums.  Two orders m, m + 1 (m even) run side by side and share the
// Bessel functions that they read.
//
// Per (atom, frame): 4 FMAs a shell and entry (pair of orders at a degree)
// plus 8 operations shared by the shells, about 80 operations for the Bessel
// functions of a shell; at most 100 sums a lane, so that two wavefronts a SIMD
// fit without scratch.  Bound by the latency of those two (scalar and LDS loads
// per entry, the recurrences of the factors).  20,000 atoms x 2,000 frames,
// 121 moments, 10 shells: 15.8 ms, 16.5 ms a call (128 ms a call when each wavefront
// of 8 moments ran their Legendre recurrences itself and read Bessel functions
// from a table of 36 GB).
#include <algorithm>
#include <cmath>

#include "sx_special_device.h"

namespace sx {

namespace {

constexpr int kWaves = 8;
constexpr int kThreads = kWaves * kWave;
constexpr int kFewEntries = 2;  // entries a wavefront of the kernels that take lists of few pairs
constexpr double kPi = 3.14159265358979323846;

// w j_l(x), l0 <= l < L1, to J[l * stride]: upward where x exceeds the largest
// degree, else by Miller's downward recurrence, normalised to j_0 or j_1; below 1e-8
// by the leading term, x^l / (2l + 1)!!, whose relative error is x^2.
// From 1e-8 the recurrence stays in range from its start at 1e-280.
// Miller's recurrence starts at degree `start`.
// (LOW: l0 may be above 0; without it the loops stay those of all degrees.)
template <bool LOW>
__device__ __forceinline__ void bessel_to_lds(double w, double x, int l0, int L1, int start, double *J, int stride) {
    if (x < 1e-8) {
        double j = w;
#pragma unroll 1
        for (int l = 0; l < L1; ++l) {
            if (!LOW || l >= l0) J[l * stride] = j;
            j *= x / (2.0 * l + 3.0);
        }
        return;
    }
    double s, c;
    sincos_reduced(x, s, c);
    const double ix = reciprocal(x);
    const double j0 = w * s * ix, j1 = fma(-w, c, j0) * ix;
    const int L = L1 - 1;
    if (x > (double)L) {
        if (!LOW || l0 == 0) J[0] = j0;
        if (L1 > 1 && (!LOW || l0 <= 1)) J[stride] = j1;
        double a = j0, b = j1;
        int l = 2;
#pragma unroll 1
        for (; LOW && l < l0; ++l) {
            const double n = fma((2.0 * l - 1.0) * ix, b, -a);
            a = b;
            b = n;
        }
#pragma unroll 2
        for (; l < L1; ++l) {
            const double n = fma((2.0 * l - 1.0) * ix, b, -a);
            a = b;
            b = n;
            J[l * stride] = n;
        }
        return;
    }
    int n = start;
    double fp1 = 0.0, f = 1e-280;  // f_{n+1}, f_n
#pragma unroll 2
    for (; n > L; --n) {
        const double fm1 = fma((2.0 * n + 1.0) * ix, f, -fp1);
        fp1 = f;
        f = fm1;
    }
    const int low = LOW ? max(l0, 2) : 1;
#pragma unroll 2
    for (; n >= low; --n) {
        J[n * stride] = f;
        const double fm1 = fma((2.0 * n + 1.0) * ix, f, -fp1);
        fp1 = f;
        f = fm1;
    }
#pragma unroll 1
    for (; LOW && n > 0; --n) {
        const double fm1 = fma((2.0 * n + 1.0) * ix, f, -fp1);
        fp1 = f;
        f = fm1;
    }
    // f = f_0, fp1 = f_1
    const double sc = fabs(j0) >= fabs(j1) || L == 0 ? j0 / f : j1 / fp1;
    if (!LOW || l0 == 0) J[0] = j0;
    if (L >= 1 && (!LOW || l0 <= 1)) J[stride] = j1;
#pragma unroll 1
    for (int l = LOW ? low : 2; l < L1; ++l) J[l * stride] *= sc;
}

struct SphereSumArgs {
    const float *srf;                       // r of every (atom, frame)
    const double *sct, *sst, *ssp, *scp;    // cos theta, sin theta, sin phi, cos phi
    size_t NFp, NAp, range;                 // atoms per range (the last may be shorter)
    const float *b;
    int per_shell_b;
    const double *q;                        // |q| per shell
    int ns, L1, M1, CA, sub;                // degrees, orders, atoms per step, parts per range
    int l0, m0;                             // lists of few pairs: the lowest degree and order that have entries
    int start;                              // of Miller's recurrence, L + 32 + 2 sqrt(2 L) for x <= L
    int nd;                                 // pairs of orders x degree in all
    const SphereEntry *sched;               // [kWaves][ND]
    const double *alpha;                    // [M1 + 1][L1]
    double2 *parts;                         // [split * sub][ns][2 nd][NFp]
};

// Block (frame tile, MS shells, part of an atom range).
template <int MS, int ND>
__global__ __launch_bounds__(kThreads) void sphere_sums_kernel(SphereSumArgs a) {
    extern __shared__ double lds[];
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
    const size_t t = (size_t)blockIdx.x * kWave + lane;
    const int s0 = blockIdx.y * MS, z = blockIdx.z;
    const size_t r0 = (size_t)(z / a.sub) * a.range, r1 = min(a.NAp, r0 + a.range);
    const size_t len = r1 > r0 ? r1 - r0 : 0;
    const size_t j0 = r0 + len * (z % a.sub) / a.sub, j1 = r0 + len * (z % a.sub + 1) / a.sub;
    // LDS of one atom, from the lowest degree and order on: J [L1 - l0][MS][64],
    // F [M1 - m0] double2 [64], cos theta [64]
    constexpr bool LOW = ND == kFewEntries;
    const int l0 = LOW ? a.l0 : 0, m0 = LOW ? a.m0 : 0;
    const int jrows = (a.L1 - l0) * MS, frows = 2 * (a.M1 - m0);
    const int per_atom = (jrows + frows + 1) * kWave;

    const auto alpha = uniform(a.alpha), Q = uniform(a.q);
    const auto B = uniform(a.b);
    const auto sched = uniform(a.sched) + wave * ND;
    double acc[ND][MS][4];
#pragma unroll
    for (int k = 0; k < ND; ++k)
#pragma unroll
        for (int s = 0; s < MS; ++s)
#pragma unroll
            for (int i = 0; i < 4; ++i) acc[k][s][i] = 0.0;

    for (size_t jc = j0; jc < j1; jc += a.CA) {
        const int na = (int)min((size_t)a.CA, j1 - jc);
        // the factors of na atoms: one (atom, shell) or (atom, angles) a wavefront at a time
#pragma unroll 1
        for (int i = wave; i < na * (MS + 1); i += kWaves) {
            const int c = i / (MS + 1), s = i - c * (MS + 1);
            const size_t j = jc + c, e = j * a.NFp + t;
            double *A = lds + c * per_atom + lane;
            if (s < MS) {
                double *J = A + s * kWave;
                const int sh = min(s0 + s, a.ns - 1);
                const float w = B[(a.per_shell_b ? (size_t)sh * a.NAp : 0) + j];
                if (w == 0.f) {
                    for (int l = 0; l < a.L1 - l0; ++l) J[l * (MS * kWave)] = 0.0;
                } else {
                    bessel_to_lds<LOW>((double)w, Q[sh] * (double)a.srf[e], l0, a.L1, a.start, J - l0 * (MS * kWave),
                                       MS * kWave);
                }
            } else {
                const double st = a.sst[e], ur = -st * a.scp[e], ui = -st * a.ssp[e];
                double2 *F = reinterpret_cast<double2 *>(lds + c * per_atom + jrows * kWave) + lane;
                double fr = 1.0, fi = 0.0;
#pragma unroll 1
                for (int m = 0; m < a.M1; ++m) {
                    if (!LOW || m >= m0) F[(m - m0) * kWave] = make_double2(fr, fi);
                    const double nr = fma(fr, ur, -fi * ui);
                    fi = fma(fr, ui, fi * ur);
                    fr = nr;
                }
                A[(jrows + frows) * kWave] = a.sct[e];
            }
        }
        __syncthreads();
#pragma unroll 1
        for (int c = 0; c < na; ++c) {
            const double *A = lds + c * per_atom + lane;
            const double2 *F = reinterpret_cast<const double2 *>(lds + c * per_atom + jrows * kWave) + lane;
            const double ct = A[(jrows + frows) * kWave];
            double ta1 = 0.0, tb1 = 0.0, ta2 = 0.0, tb2 = 0.0;
            double2 f1 = make_double2(0.0, 0.0), f2 = f1;
            // the wavefront's entries, read again for every atom through an index
            // that the compiler cannot hoist: held across the loop they would take
            // the registers of the sums
            int zo = 0;
            asm volatile("" : "+s"(zo));
#pragma unroll
            for (int k = 0; k < ND; ++k) {
                const auto E = sched + (k + zo);
                const int skip = E->skip;
                if (skip >= 0) {
                    // a run of degrees starts: T_{m-1} = 0, T_{m-2} = -1 give T_m = 1
                    f1 = F[E->f1 * kWave];
                    f2 = F[E->f2 * kWave];
                    ta1 = 0.0;
                    tb1 = -1.0;
                    ta2 = -1.0;
                    tb2 = 0.0;
                    const auto al = alpha + E->first;
#pragma unroll 1
                    for (int i = 0; i < skip; ++i) {
                        const double n1 = fma(al[i] * ct, ta1, -tb1);
                        const double n2 = fma(al[a.L1 + i] * ct, ta2, -tb2);
                        tb1 = ta1;
                        ta1 = n1;
                        tb2 = ta2;
                        ta2 = n2;
                    }
                }
                const double n1 = fma(E->alpha1 * ct, ta1, -tb1), n2 = fma(E->alpha2 * ct, ta2, -tb2);
                tb1 = ta1;
                ta1 = n1;
                tb2 = ta2;
                ta2 = n2;
                const double x1 = n1 * f1.x, y1 = n1 * f1.y, x2 = n2 * f2.x, y2 = n2 * f2.y;
                const double *J = A + E->l * (MS * kWave);
#pragma unroll
                for (int s = 0; s < MS; ++s) {
                    const double jv = J[s * kWave];
                    acc[k][s][0] = fma(jv, x1, acc[k][s][0]);
                    acc[k][s][1] = fma(jv, y1, acc[k][s][1]);
                    acc[k][s][2] = fma(jv, x2, acc[k][s][2]);
                    acc[k][s][3] = fma(jv, y2, acc[k][s][3]);
                    // the sums are formed here: moved behind the other entries, as the
                    // compiler would, they keep every entry's factors in registers
#pragma unroll
                    for (int i = 0; i < 4; ++i) asm volatile("" : "+v"(acc[k][s][i]));
                }
            }
        }
        __syncthreads();
    }
#pragma unroll
    for (int k = 0; k < ND; ++k) {
        const int d = sched[k].pair;
        if (d < 0) break;
#pragma unroll
        for (int s = 0; s < MS; ++s) {
            if (s0 + s >= a.ns) break;
            double2 *p = a.parts + (((size_t)z * a.ns + s0 + s) * 2 * a.nd + 2 * d) * a.NFp + t;
            p[0] = make_double2(acc[k][s][0], acc[k][s][1]);
            p[a.NFp] = make_double2(acc[k][s][2], acc[k][s][3]);
        }
    }
}

// amp[(range, shell, moment)][t] from the sums of the moment's (degree,
// |order|): K i^l (C - i S) for m >= 0, K (-1)^m i^l (C + i S) for m < 0.
__global__ __launch_bounds__(kWave) void sphere_amplitudes_kernel(const double2 *__restrict__ parts, int sub, int ns,
                                                                  int nd, size_t NFp, int nmo,
                                                                  const int2 *__restrict__ entry,
                                                                  const double *__restrict__ scale,
                                                                  float2 *__restrict__ amp) {
    const size_t t = (size_t)blockIdx.x * kWave + threadIdx.x;
    const int k = blockIdx.y, s = blockIdx.z % ns, sp = blockIdx.z / ns;
    const int2 en = entry[k];  // entry of parts; l & 3, + 4 for m < 0, + 8 for odd m < 0
    double2 v = make_double2(0.0, 0.0);
    for (int u = 0; u < sub; ++u) {
        const double2 p = parts[(((size_t)(sp * sub + u) * ns + s) * 2 * nd + en.x) * NFp + t];
        v.x += p.x;
        v.y += p.y;
    }
    const double K = (en.y & 8) ? -scale[k] : scale[k];
    double re = K * v.x, im = (en.y & 4) ? K * v.y : -K * v.y;
    if (en.y & 1) {
        const double r = re;
        re = -im;
        im = r;
    }
    if (en.y & 2) {
        re = -re;
        im = -im;
    }
    amp[(((size_t)sp * ns + s) * nmo + k) * NFp + t] = make_float2((float)re, (float)im);
}

using SumsFn = void (*)(SphereSumArgs);
struct SumsKernel {
    int nd, ms;
    SumsFn fn;
};
// pairs a wavefront x shells a workgroup: 4 nd ms <= 100 sums a lane
const SumsKernel kKernels[] = {
    {2, 1, sphere_sums_kernel<1, 2>},  {2, 3, sphere_sums_kernel<3, 2>},  {2, 6, sphere_sums_kernel<6, 2>},
    {2, 8, sphere_sums_kernel<8, 2>},  {4, 1, sphere_sums_kernel<1, 4>},  {4, 2, sphere_sums_kernel<2, 4>},
    {4, 4, sphere_sums_kernel<4, 4>},  {4, 6, sphere_sums_kernel<6, 4>},  {5, 1, sphere_sums_kernel<1, 5>},
    {5, 2, sphere_sums_kernel<2, 5>},  {5, 3, sphere_sums_kernel<3, 5>},  {5, 5, sphere_sums_kernel<5, 5>},
    {8, 1, sphere_sums_kernel<1, 8>},  {8, 2, sphere_sums_kernel<2, 8>},  {8, 3, sphere_sums_kernel<3, 8>},
    {11, 1, sphere_sums_kernel<1, 11>}, {11, 2, sphere_sums_kernel<2, 11>},
};
constexpr size_t kLdsBytes = 160 << 10;
// Lists of at most one pair a wavefront: the sums no longer cover the latency of
// the factors' loads and chains, so that workgroups take at most 3 shells and half
// of the LDS, which then starts at their lowest degree and order, so that two and
// more share a CU, and ranges are cut for four.  5,000 atoms x 2,000 frames x 5 shells,
// whole calls: (0, 0) 1.72 -> 1.17 ms, l <= 3 1.98 -> 1.43 ms, (16, 0) 3.43 -> 2.86 ms,
// (16, 16) 3.20 -> 2.46 ms (2.76 ms by the moment's own recurrence from a table of
// Bessel functions; the other single moments were no faster that way either).
constexpr int kFewShells = 3, kFewPerCu = 4;

size_t lds_per_atom(int degrees, int ms, int orders) {
    return sizeof(double) * kWave * ((size_t)degrees * ms + 2 * orders + 1);
}

}  // namespace

bool make_sphere_plan(const int *moments, int nmo, int ns, SpherePlan *plan) {
    int lmax = 0, mmax = 0;
    for (int k = 0; k < nmo; ++k) {
        lmax = std::max(lmax, moments[2 * k]);
        mmax = std::max(mmax, std::abs(moments[2 * k + 1]));
    }
    if (lmax >= kSphereSumL1 || nmo > 65535) return false;
    SpherePlan p;
    p.L1 = lmax + 1;
    p.M1 = mmax + 1;
    // the (even order, degree) pairs that occur, runs of degrees per order
    std::vector<int> pair_of((size_t)(mmax / 2 + 1) * p.L1, -1);
    for (int k = 0; k < nmo; ++k) pair_of[(size_t)(std::abs(moments[2 * k + 1]) / 2) * p.L1 + moments[2 * k]] = 0;
    std::vector<int2> pairs;
    for (int h = 0; h <= mmax / 2; ++h)
        for (int l = 2 * h; l < p.L1; ++l)
            if (pair_of[(size_t)h * p.L1 + l] == 0) {
                pair_of[(size_t)h * p.L1 + l] = (int)pairs.size();
                pairs.push_back(make_int2(l, 2 * h));
            }
    p.nd = (int)pairs.size();
    const int per_wave = (p.nd + kWaves - 1) / kWaves;
    const bool few = per_wave == 1;
    if (few) {
        p.l0 = pairs[0].x;
        for (const int2 &q : pairs) p.l0 = std::min(p.l0, q.x);
        p.m0 = pairs[0].y;
    }
    const int degrees = p.L1 - p.l0, orders = p.M1 - p.m0;
    p.per_cu = few ? kFewPerCu : 1;
    // the kernel of the fewest operations: 8 a pair and 4 a pair and shell,
    // about 80 a shell for its Bessel functions, 60 for the angles, per group of shells
    double best = 0.0;
    p.kernel = -1;
    for (int i = 0; i < (int)(sizeof(kKernels) / sizeof(kKernels[0])); ++i) {
        const SumsKernel &k = kKernels[i];
        if (few && (k.nd != kFewEntries || k.ms > kFewShells)) continue;
        if (k.nd < per_wave || lds_per_atom(degrees, k.ms, orders) > kLdsBytes) continue;
        const int groups = (ns + k.ms - 1) / k.ms;
        const double cost = groups * (p.nd * (8.0 + 4.0 * k.ms) + 80.0 * k.ms + 60.0) + 0.01 * k.nd;
        if (p.kernel < 0 || cost < best) {
            best = cost;
            p.kernel = i;
        }
    }
    if (p.kernel < 0) return false;
    const SumsKernel &kk = kKernels[p.kernel];
    p.groups = (ns + kk.ms - 1) / kk.ms;
    p.CA = (int)std::max<size_t>(1, std::min<size_t>(8, kLdsBytes / (few ? 2 : 1) / lds_per_atom(degrees, kk.ms, orders)));
    // P_lm normalised as Y_lm: P_l = a_l (x P_{l-1} - e_l P_{l-2}), a_l =
    // sqrt((4 l^2 - 1) / (l^2 - m^2)), e_l = sqrt(((l-1)^2 - m^2) / (4 (l-1)^2 - 1));
    // P_l = s_l T_l with s_l = a_l e_l s_{l-2}
    p.alpha.assign((size_t)(p.M1 + 1) * p.L1, 0.0);
    std::vector<double> s((size_t)(p.M1 + 1) * p.L1, 0.0);
    for (int m = 0; m <= mmax + 1 && m < p.L1; ++m) {
        double *al = p.alpha.data() + (size_t)m * p.L1, *sm = s.data() + (size_t)m * p.L1;
        double c = (2.0 * m + 1.0) / (4.0 * kPi);
        for (int i = 1; i <= m; ++i) c *= (2.0 * i - 1.0) / (2.0 * i);
        sm[m] = std::sqrt(c);
        for (int l = m + 1; l < p.L1; ++l) {
            const double al2 = std::sqrt((4.0 * l * l - 1.0) / ((double)l * l - (double)m * m));
            const double e =
                l > m + 1 ? std::sqrt(((l - 1.0) * (l - 1.0) - (double)m * m) / (4.0 * (l - 1.0) * (l - 1.0) - 1.0)) : 0.0;
            sm[l] = l > m + 1 ? al2 * e * sm[l - 2] : sm[m];
            al[l] = al2 * sm[l - 1] / sm[l];
        }
    }
    // every wavefront's entries; the unused last ones of some repeat degree 0 without a place for the sums
    p.sched.assign((size_t)kWaves * kk.nd, SphereEntry{0.0, 0.0, 0, 0, 0, 0, 0, -1});
    for (int w = 0; w < kWaves; ++w) {
        const int d0 = p.nd * w / kWaves, d1 = p.nd * (w + 1) / kWaves;
        for (int d = d0; d < d1; ++d) {
            const int l = pairs[d].x, m = pairs[d].y;
            const bool next = d > d0 && pairs[d - 1].y == m && pairs[d - 1].x == l - 1;
            SphereEntry &e = p.sched[(size_t)w * kk.nd + d - d0];
            e.alpha1 = p.alpha[(size_t)m * p.L1 + l];
            e.alpha2 = p.alpha[(size_t)(m + 1) * p.L1 + l];
            e.l = l - p.l0;
            e.skip = next ? -1 : l - m;
            e.first = m * p.L1 + m;
            e.f1 = m - p.m0;
            e.f2 = std::min(m + 1, mmax) - p.m0;
            e.pair = d;
        }
    }
    p.entry.resize(nmo);
    p.scale.resize(nmo);
    for (int k = 0; k < nmo; ++k) {
        const int l = moments[2 * k], m = moments[2 * k + 1], am = std::abs(m);
        p.entry[k] = make_int2(2 * pair_of[(size_t)(am / 2) * p.L1 + l] + (am & 1),
                               (l & 3) + (m < 0 ? 4 : 0) + (m < 0 && (am & 1) ? 8 : 0));
        p.scale[k] = 4.0 * kPi * s[(size_t)am * p.L1 + l];
    }
    *plan = std::move(p);
    return true;
}

size_t sphere_parts_bytes(const SpherePlan &p, size_t NFp, int ns, int split, int sub) {
    return sizeof(double2) * 2 * p.nd * NFp * (size_t)ns * split * sub;
}

// One workgroup a CU (LDS and registers; per_cu for lists of few pairs): ranges
// are cut into parts, of at least 32 atoms, until the workgroups fill whole
// rounds of the CUs.
int sphere_parts_per_range(const SpherePlan &p, size_t NFp, size_t NAp, int split, int cus) {
    const long base = (long)(NFp / kWave) * p.groups * split, resident = (long)cus * p.per_cu;
    const long most = std::max<long>(1, std::min<long>(32, (long)(NAp / split / 32)));
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

size_t sphere_table_bytes(const SpherePlan &p) {
    return sizeof(SphereEntry) * p.sched.size() + sizeof(double) * (p.alpha.size() + p.scale.size()) +
           sizeof(int2) * p.entry.size();
}

void sphere_tables(const SpherePlan &p, void *out) {
    char *o = static_cast<char *>(out);
    auto put = [&](const auto &v) {
        const size_t n = sizeof(v[0]) * v.size();
        std::copy_n(reinterpret_cast<const char *>(v.data()), n, o);
        o += n;
    };
    put(p.sched);
    put(p.alpha);
    put(p.scale);
    put(p.entry);
}

hipError_t launch_sphere_sums(const MultipoleArgs &m, const SpherePlan &p, const void *tables, int sub, void *parts,
                              hipStream_t stream) {
    const size_t n = m.NAp * m.NFp;
    SphereSumArgs a;
    a.srf = static_cast<const float *>(m.sph);
    const double *d = reinterpret_cast<const double *>(static_cast<const char *>(m.sph) + sizeof(float) * n);
    a.sct = d;
    a.sst = d + n;
    a.ssp = d + 2 * n;
    a.scp = d + 3 * n;
    a.NFp = m.NFp;
    a.NAp = m.NAp;
    a.range = (m.NAp + m.split - 1) / m.split;
    a.b = m.b;
    a.per_shell_b = m.per_shell_b;
    a.q = m.qinfo;
    a.ns = m.ns;
    a.L1 = p.L1;
    a.M1 = p.M1;
    a.CA = p.CA;
    a.sub = sub;
    a.l0 = p.l0;
    a.m0 = p.m0;
    a.start = p.L1 - 1 + 32 + (int)(2.0 * std::sqrt(2.0 * (p.L1 - 1)));
    a.nd = p.nd;
    const char *tb = static_cast<const char *>(tables);
    a.sched = reinterpret_cast<const SphereEntry *>(tb);
    a.alpha = reinterpret_cast<const double *>(tb + sizeof(SphereEntry) * p.sched.size());
    const double *scale = a.alpha + p.alpha.size();
    const int2 *entry = reinterpret_cast<const int2 *>(scale + p.scale.size());
    a.parts = static_cast<double2 *>(parts);
    const SumsKernel &k = kKernels[p.kernel];
    const size_t lds = lds_per_atom(p.L1 - p.l0, k.ms, p.M1 - p.m0) * p.CA;
    hipError_t e =
        hipFuncSetAttribute((const void *)k.fn, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
    if (e != hipSuccess) return e;
    const unsigned tiles = (unsigned)(m.NFp / kWave);
    if (!sphere_sums_grid_fits(m.ns, m.split)) return hipErrorInvalidValue;
    hipLaunchKernelGGL(k.fn, dim3(tiles, (unsigned)p.groups, (unsigned)(m.split * sub)), dim3(kThreads), lds, stream, a);
    e = hipGetLastError();
    if (e != hipSuccess) return e;
    hipLaunchKernelGGL(sphere_amplitudes_kernel, dim3(tiles, (unsigned)m.nmo, (unsigned)(m.split * m.ns)), dim3(kWave),
                       0, stream, a.parts, sub, m.ns, p.nd, m.NFp, m.nmo, entry, scale, m.amp);
    return hipGetLastError();
}

}  // namespace sx
