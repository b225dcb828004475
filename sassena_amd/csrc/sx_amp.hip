// sx_amp.hip -- staging transposes and the coherent amplitude kernel.
//
// Amplitude ("all" scattering, reference loop all_vectors_scatter_device.cpp:418-438):
//   A_v(t) = sum_j b_j exp(i q_v . r_j(t))
// Each lane of a wavefront owns one frame t and each wavefront a block of VB
// q vectors (wave-uniform, held in SGPRs), so the atom sum needs no cross-lane
// reduction and every coordinate load is a coalesced 256-byte row of the
// atom-major SoA block.  The phase is formed in FP64 in turns (q pre-divided
// by 2 pi), reduced to [0, 1) turns in FP64 (v_fract_f64), and evaluated with
// the hardware v_sin_f32 / v_cos_f32, which take turns (max abs error 1.3e-7
// over the reduced range, measured against FP64 on gfx950).  Sums run in FP32
// over 64 atoms and are folded into FP64 totals.
//
// When the vectors of all shells are one orientation set scaled by |q_s|
// (orientation types file and sphere, abstract_vectors_scatter_device.cpp:115-129),
// amp_oriented_kernel forms d = u_m . r once per atom and orientation and the
// phase of each shell as the single FP64 product (|q_s| / 2 pi) d, or, with
// linearly spaced shells, steps the phasor from shell to shell (sx_amp_device.h).
#include <algorithm>
#include <cmath>

#include "sx_amp_device.h"

namespace sx {

// ---------------------------------------------------------------- staging --

// src: frames [nf][NA][3] (frames F0.. of the host block); tile 64 atoms x TF
// frames, its loads (192 floats a frame) in flight together.  Bound by latency
// for small blocks: 1,000 atoms x 200 frames took 32 us with one frame's loads
// after the other and 64 workgroups, and takes 9 us so.
template <int TF>
__global__ __launch_bounds__(256) void stage_frames_kernel(const float *__restrict__ src, int NA,
                                                           int F0, int nf, float *__restrict__ coords,
                                                           size_t NAp, size_t NFp) {
    __shared__ float tile[3][64][TF + 1];
    const int a0 = blockIdx.x * 64, f0 = blockIdx.y * TF;
    const int tid = threadIdx.x;
    const int cols = min(192, 3 * (NA - a0));
#pragma unroll 12
    for (int i = 0; i < TF * 192 / 256; ++i) {
        const int e = i * 256 + tid, tf = e / 192, col = e - tf * 192;
        const int f = f0 + tf;
        if (col < cols && f < nf) tile[col % 3][col / 3][tf] = src[((size_t)f * NA + a0) * 3 + col];
    }
    __syncthreads();
    const int tf = tid % TF;
    for (int row = tid / TF; row < 192; row += 256 / TF) {
        const int c = row / 64, ja = row % 64;
        const int a = a0 + ja, f = f0 + tf;
        if (a < NA && f < nf) coords[(size_t)c * NAp * NFp + (size_t)a * NFp + F0 + f] = tile[c][ja][tf];
    }
}

// src: atoms [na][NF][3] (atoms A0.. of the host block).
__global__ __launch_bounds__(256) void stage_atoms_kernel(const float *__restrict__ src, int A0, int na,
                                                          int NF, float *__restrict__ coords, size_t NAp,
                                                          size_t NFp) {
    const int t = blockIdx.x * 256 + threadIdx.x;
    const int ja = blockIdx.y;
    if (t >= NF || ja >= na) return;
    const float *p = src + ((size_t)ja * NF + t) * 3;
    const size_t row = (size_t)(A0 + ja) * NFp + t;
    coords[row] = p[0];
    coords[NAp * NFp + row] = p[1];
    coords[2 * NAp * NFp + row] = p[2];
}

hipError_t launch_stage_frames(const float *src, size_t NA, size_t F0, size_t nf, float *coords, size_t NAp,
                               size_t NFp, hipStream_t stream) {
    // tiles of 16 frames (64-byte row segments) while those of 64 are fewer than
    // two a CU
    const size_t ta = (NA + 63) / 64;
    if (ta * ((nf + 63) / 64) < 512)
        hipLaunchKernelGGL(stage_frames_kernel<16>, dim3((unsigned)ta, (unsigned)((nf + 15) / 16)), dim3(256), 0, stream,
                           src, (int)NA, (int)F0, (int)nf, coords, NAp, NFp);
    else
        hipLaunchKernelGGL(stage_frames_kernel<64>, dim3((unsigned)ta, (unsigned)((nf + 63) / 64)), dim3(256), 0, stream,
                           src, (int)NA, (int)F0, (int)nf, coords, NAp, NFp);
    return hipGetLastError();
}

hipError_t launch_stage_atoms(const float *src, size_t a0, size_t na, size_t NF, float *coords, size_t NAp,
                              size_t NFp, hipStream_t stream) {
    dim3 grid((unsigned)((NF + 255) / 256), (unsigned)na);
    hipLaunchKernelGGL(stage_atoms_kernel, grid, dim3(256), 0, stream, src, (int)a0, (int)na, (int)NF, coords,
                       NAp, NFp);
    return hipGetLastError();
}

// Largest |x| over n floats, as the bit pattern of a non-negative float
// (ordered like unsigned integers) in *out, which the caller zeroes first.
// One atomic a workgroup: one a wavefront of 4,096 workgroups, all on one word,
// took 142 us for 1,000 atoms x 200 frames, which takes 3.6 us so.
__global__ __launch_bounds__(256) void absmax_kernel(const float *__restrict__ x, size_t n,
                                                     unsigned *__restrict__ out) {
    __shared__ float part[4];
    float m = 0.f;
    const size_t i0 = (size_t)blockIdx.x * 256 + threadIdx.x, step = (size_t)gridDim.x * 256;
    const float4 *x4 = reinterpret_cast<const float4 *>(x);  // (device allocations are aligned)
#pragma unroll 4
    for (size_t i = i0; i < n / 4; i += step) {
        const float4 v = x4[i];
        m = fmaxf(fmaxf(m, fmaxf(fabsf(v.x), fabsf(v.y))), fmaxf(fabsf(v.z), fabsf(v.w)));
    }
    for (size_t i = n / 4 * 4 + i0; i < n; i += step) m = fmaxf(m, fabsf(x[i]));
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) m = fmaxf(m, __shfl_xor(m, off, 64));
    if ((threadIdx.x & 63) == 0) part[threadIdx.x >> 6] = m;
    __syncthreads();
    if (threadIdx.x == 0)
        atomicMax(out, __float_as_uint(fmaxf(fmaxf(part[0], part[1]), fmaxf(part[2], part[3]))));
}

__global__ void zero_u32_kernel(unsigned *p) { *p = 0u; }

hipError_t launch_absmax(const float *x, size_t n, unsigned *out, hipStream_t stream) {
    hipLaunchKernelGGL(zero_u32_kernel, dim3(1), dim3(1), 0, stream, out);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
    if (reinterpret_cast<size_t>(x) % sizeof(float4)) return hipErrorInvalidValue;
    // 32 floats a thread, up to eight workgroups a CU
    const size_t blocks = std::min<size_t>(2048, std::max<size_t>(1, (n + 8191) / 8192));
    hipLaunchKernelGGL(absmax_kernel, dim3((unsigned)blocks), dim3(256), 0, stream, x, n, out);
    return hipGetLastError();
}

// -------------------------------------------------------------- amplitude --

struct AmpKernelArgs {
    const float *X, *Y, *Z;
    size_t NFp;
    const double *qrev;
    const float *b;
    const int *brow;
    size_t NAp;
    int V, ftiles, vgroups, split, atoms_per_split;
    float2 *amp;
};

template <int VB, bool PER_ROW_B>
__global__ __launch_bounds__(256) void amp_all_kernel(AmpKernelArgs a) {
    // XCD-aware work order: hardware hands consecutive workgroups to the 8
    // XCDs round-robin; give each XCD a contiguous run of items so that the
    // wavefronts sharing one frame tile and atom range share that XCD's L2.
    // A wavefront an item: four to a workgroup in this order, also across the ends
    // of a frame tile's vectors, so that no wavefront runs on vectors that are
    // not there (200 vectors: 25 wavefronts a tile and range, not 7 workgroups of 4;
    // 20,000 atoms x 2,000 frames: 3.20 -> 2.90 ms a call).
    const int nitems = a.ftiles * a.split * a.vgroups;
    const int per = ((nitems + 3) / 4 + 7) >> 3;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int item = ((int)(blockIdx.x & 7) * per + (int)(blockIdx.x >> 3)) * 4 + wave;
    if (item >= nitems) return;
    const int vg = item % a.vgroups;
    const int rest = item / a.vgroups;
    const int sp = rest % a.split;
    const int ft = rest / a.split;

    const int lane = threadIdx.x & 63;
    const int vbase = vg * VB;
    const size_t t = (size_t)ft * kWave + lane;

    double qx[VB], qy[VB], qz[VB];
    int brow[VB];
#pragma unroll
    for (int i = 0; i < VB; ++i) {
        const int v = min(vbase + i, a.V - 1);
        qx[i] = a.qrev[3 * v];
        qy[i] = a.qrev[3 * v + 1];
        qz[i] = a.qrev[3 * v + 2];
        brow[i] = PER_ROW_B ? a.brow[v] : 0;
    }

    // FP32 sums over kFold atoms, folded into FP64 totals
    constexpr int kFold = 64;
    double tr[VB], ti[VB];
#pragma unroll
    for (int i = 0; i < VB; ++i) tr[i] = ti[i] = 0.0;

    const size_t j0 = (size_t)sp * a.atoms_per_split;
    const size_t j1 = min(a.NAp, j0 + (size_t)a.atoms_per_split);
    // buffer loads: the batch's first row as the base, the atom's row as the scalar and
    // the lane's frame as the vector offset, so that no VALU instruction goes on addresses
    // (601 for 8 atoms x 8 vectors, 626 with plain loads: 2.90 -> 2.78 ms a call of 20,000
    // atoms x 2,000 frames x 200 vectors)
    const unsigned voff = (unsigned)(t * sizeof(float));
    const int rows = (int)(kAtomChunk * a.NFp * sizeof(float));

    for (size_t jf = j0; jf < j1; jf += kFold) {
        const size_t jend = min(j1, jf + (size_t)kFold);
        float cr[VB], ci[VB];
#pragma unroll
        for (int i = 0; i < VB; ++i) cr[i] = ci[i] = 0.f;
#pragma unroll 1
        for (size_t j = jf; j < jend; j += kAtomChunk) {
            float xs[kAtomChunk], ys[kAtomChunk], zs[kAtomChunk];
            const __amdgpu_buffer_rsrc_t rx =
                __builtin_amdgcn_make_buffer_rsrc((void *)(a.X + j * a.NFp), (short)0, rows, kBufferDword3);
            const __amdgpu_buffer_rsrc_t ry =
                __builtin_amdgcn_make_buffer_rsrc((void *)(a.Y + j * a.NFp), (short)0, rows, kBufferDword3);
            const __amdgpu_buffer_rsrc_t rz =
                __builtin_amdgcn_make_buffer_rsrc((void *)(a.Z + j * a.NFp), (short)0, rows, kBufferDword3);
#pragma unroll
            for (int c = 0; c < kAtomChunk; ++c) {
                const int so = (int)(c * a.NFp * sizeof(float));
                xs[c] = __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(rx, voff, so, 0));
                ys[c] = __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(ry, voff, so, 0));
                zs[c] = __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(rz, voff, so, 0));
            }
#pragma unroll
            for (int c = 0; c < kAtomChunk; ++c) {
                const double xd = xs[c], yd = ys[c], zd = zs[c];
                const float b0 = a.b[j + c];
#pragma unroll
                for (int i = 0; i < VB; ++i) {
                    const float bj = PER_ROW_B ? a.b[(size_t)brow[i] * a.NAp + j + c] : b0;
                    double p = qx[i] * xd;
                    p = fma(qy[i], yd, p);
                    p = fma(qz[i], zd, p);
                    const float f = (float)__builtin_amdgcn_fract(p);
                    cr[i] = fmaf(bj, __builtin_amdgcn_cosf(f), cr[i]);
                    ci[i] = fmaf(bj, __builtin_amdgcn_sinf(f), ci[i]);
                }
            }
        }
#pragma unroll
        for (int i = 0; i < VB; ++i) {
            tr[i] += (double)cr[i];
            ti[i] += (double)ci[i];
        }
    }

#pragma unroll
    for (int i = 0; i < VB; ++i) {
        const int v = vbase + i;
        if (v < a.V) a.amp[((size_t)sp * a.V + v) * a.NFp + t] = make_float2((float)tr[i], (float)ti[i]);
    }
}


// Work item of an oriented launch: XCD x = blockIdx & 7 takes an equal
// share of the (frame tile, atom range, orientation group) items of every
// shell tile, the shell tiles one after another.  At any time the CUs then
// run tiles of one shell group: with the shell tile varying fastest, the
// dispatch order tied each CU to the items of one shell tile, so tiles of
// unequal cost (exactly stepped and corrected ones, a partial last tile) left
// some CUs idle while others finished theirs.
//
// A wavefront an item (og: its group of VM orientations), four to a workgroup in
// this order, also across the ends of a frame tile's orientations.
struct OrientItem {
    int ft, sp, og, sg;
};

__device__ __forceinline__ bool orient_item(const OrientKernelArgs &a, OrientItem &w) {
    const int nsub = a.ftiles * a.split * a.ogroups;
    const int per = ((nsub + 3) / 4 + 7) >> 3;
    const int local = (int)(blockIdx.x >> 3);
    w.sg = local / per;
    const int r = ((int)(blockIdx.x & 7) * per + (local - w.sg * per)) * 4 +
                  __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    if (w.sg >= a.sgroups || r >= nsub) return false;
    w.og = r % a.ogroups;
    const int rest = r / a.ogroups;
    w.sp = rest % a.split;
    w.ft = rest / a.split;
    return true;
}

static int oriented_grid(int ftiles, int split, int ogroups, int sgroups) {
    return (((ftiles * split * ogroups + 3) / 4 + 7) / 8) * 8 * sgroups;
}

template <int VM, int VS, bool PER_ROW_B>
__global__ __launch_bounds__(256, 2) void amp_oriented_kernel(OrientKernelArgs a) {
    OrientItem w;
    if (!orient_item(a, w)) return;
    oriented_tile<VM, VS, PER_ROW_B>(a, w.ft, w.sp, w.og, w.sg * VS);
}

// Shells each on their own phase (mode 0) in tiles of 2 orientations x VS <= 8
// shells, VS such that the last tile is as full as the others (21 shells: three
// tiles of 7, not 8 + 8 + 5 padded to 8).  The sums of a term do not depend on the
// tile.  7,001 atoms x 1,501 frames x 21 shells x 67 orientations, a factor per
// atom and shell: 5.35 -> 4.66 ms with this and the wavefront items.
template <int VS, bool PER_ROW_B>
__global__ __launch_bounds__(256, 2) void amp_direct_kernel(OrientKernelArgs a) {
    OrientItem w;
    if (!orient_item(a, w)) return;
    oriented_tile_body<2, VS, PER_ROW_B, 0, true>(a, w.ft, w.sp, w.og, w.sg * VS, nullptr);
}

// Shells that are an arithmetic progression up to small residuals (modes 2-5
// of oriented_tile_body, by the tile line's flags); one factor per atom.
// The FP64 totals take the dynamic LDS (kResidualLds<VM, VS> bytes).
template <int VM, int VS>
__global__ __launch_bounds__(256, 2) void amp_oriented_res_kernel(OrientKernelArgs a) {
    extern __shared__ double tot_lds[];
    OrientItem w;
    if (!orient_item(a, w)) return;
    residual_tile<VM, VS>(a, w.ft, w.sp, w.og, w.sg * VS, tot_lds);
}

// Oriented tile shapes (orientations x shells per wavefront), picked by the
// host autotuner: 0: 2x8, 1: 4x4, 2: 1x8, 3: 1x16, 4: 1x20.
static const int kShapeVM[kOrientShapes] = {2, 4, 1, 1, 1};
static const int kShapeVS[kOrientShapes] = {8, 4, 8, 16, 20};

int orient_shape_vm(int shape) { return kShapeVM[shape]; }
int orient_shape_vs(int shape) { return kShapeVS[shape]; }

template <int VM, int VS>
static hipError_t launch_oriented_shape(const OrientKernelArgs &k, bool per_row, int blocks, hipStream_t stream) {
    if (k.ap == 2) {
        if (per_row) return hipErrorInvalidValue;
        const void *fn = (const void *)amp_oriented_res_kernel<VM, VS>;
        const size_t lds = kResidualLds<VM, VS>;
        hipError_t e = hipFuncSetAttribute(fn, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
        if (e != hipSuccess) return e;
        hipLaunchKernelGGL((amp_oriented_res_kernel<VM, VS>), dim3(blocks), dim3(256), lds, stream, k);
    } else if (per_row)
        hipLaunchKernelGGL((amp_oriented_kernel<VM, VS, true>), dim3(blocks), dim3(256), 0, stream, k);
    else
        hipLaunchKernelGGL((amp_oriented_kernel<VM, VS, false>), dim3(blocks), dim3(256), 0, stream, k);
    return hipGetLastError();
}

OrientKernelArgs make_orient_args(const OrientArgs &a) {
    constexpr int CH = 16;
    const int VM = kShapeVM[a.shape], VS = kShapeVS[a.shape];
    OrientKernelArgs k;
    k.X = a.coords;
    k.Y = a.coords + a.NAp * a.NFp;
    k.Z = a.coords + 2 * a.NAp * a.NFp;
    k.NFp = a.NFp;
    k.qlen = a.qlen;
    k.u = a.u;
    k.b = a.b;
    k.NAp = a.NAp;
    k.natoms = a.natoms ? std::min(a.natoms, a.NAp) : a.NAp;
    k.NM = a.NM;
    k.ns = a.ns;
    k.V = a.NM * a.ns;
    k.ftiles = (int)(a.NFp / kWave);
    k.ogroups = (a.NM + VM - 1) / VM;
    k.sgroups = (a.ns + VS - 1) / VS;
    k.split = a.split;
    size_t aps = (k.natoms + a.split - 1) / a.split;
    aps = (aps + CH - 1) / CH * CH;
    k.atoms_per_split = (int)aps;
    k.per_shell_b = a.per_shell_b;
    k.amp = a.amp;
    k.ap = a.ap;
    k.qstep = a.qstep;
    k.q0 = a.q0;
    k.qres = a.qres;
    k.lines = a.ap == 2 ? a.lines : nullptr;
    k.pack = nullptr;
    k.parts = nullptr;
    k.sub = 1;
    k.NF = 0;
    return k;
}

int tile_lines(const double *ql, int ns, double rmax, const ShellGrid &g, const int *firsts, const int *vs,
               int ntiles, TileLine *lines, float *res) {
    double qmax = 0.0;
    for (int s = 0; s < ns; ++s) qmax = std::max(qmax, std::fabs(ql[s]));
    const double tol = 1e-12 * qmax;
    double bound = kMaxShellResidual * qmax;
    if (rmax > 0.0) bound = std::min(bound, kMaxResidualPhase / kTwoPiTurns / rmax);
    int plain = 0;
    for (int t = 0; t < ntiles; ++t) {
        const int first = firsts[t], VS = vs[t], C = VS / 2, n = std::min(VS, ns - first);
        const int mid = first + C;
        // candidate steps: the call's, and that of the exact run through the middle
        double steps[2] = {g.step, 0.0};
        int nsteps = 1;
        if (mid < ns && g.runs[mid].last > mid) steps[nsteps++] = g.runs[mid].step;
        else if (mid - 1 >= first && mid - 1 < ns && g.runs[mid - 1].last >= mid) steps[nsteps++] = g.runs[mid - 1].step;
        else if (mid >= ns && g.runs[first].last > first) steps[nsteps++] = g.runs[first].step;
        int best_flags = 4;
        double best_max = 0.0;
        TileLine best{};
        for (int c = 0; c < nsteps; ++c) {
            const double st = steps[c];
            const double qm = mid < ns ? ql[mid] : ql[first] + (double)C * st;
            int flags = 0;
            double mx = 0.0;
            for (int k = 0; k < n; ++k) {
                const double r = std::fabs(ql[first + k] - (qm + (double)(k - C) * st));
                mx = std::max(mx, r);
                if (r > tol) flags |= k > C ? kTileCorrectUp : k < C ? kTileCorrectDown : 0;
            }
            if (mx > bound) continue;
            const int pop = (flags & 1) + (flags >> 1);
            const int bpop = best_flags > 3 ? 3 : (best_flags & 1) + (best_flags >> 1);
            if (best_flags > 3 || pop < bpop || (pop == bpop && mx < best_max)) {
                best_flags = flags;
                best_max = mx;
                best = TileLine{qm, st, flags, 0};
            }
        }
        if (best_flags > 3) {
            // the call's ideal grid and its residuals (within the bounds)
            best = TileLine{g.q0 + (double)mid * g.step, g.step, kTileCorrectUp | kTileCorrectDown, 0};
        }
        lines[first] = best;
        for (int k = 0; k < n; ++k) {
            const double r = ql[first + k] - (best.qmid + (double)(k - C) * best.step);
            res[first + k] = std::fabs(r) <= tol ? 0.f : (float)(kTwoPiTurns * r);
        }
        if (!(best.flags & kTileCorrectUp)) plain += std::max(0, n - C - 1);
        if (!(best.flags & kTileCorrectDown)) plain += std::min(n, C);
        if (n > C) plain += 1;  // the middle shell lies on the line
    }
    return plain;
}

int shell_progression(const double *qlen, int ns, double rmax, ShellGrid *g) {
    *g = ShellGrid{};
    if (ns < 2) return 0;
    const double d = (qlen[ns - 1] - qlen[0]) / (double)(ns - 1);
    double qmax = 0.0, emax = 0.0;
    for (int s = 0; s < ns; ++s) qmax = std::max(qmax, std::fabs(qlen[s]));
    g->res.resize(ns);
    for (int s = 0; s < ns; ++s) {
        const double e = qlen[s] - (qlen[0] + (double)s * d);
        g->res[s] = e;
        emax = std::max(emax, std::fabs(e));
    }
    g->q0 = qlen[0];
    g->step = d;
    const double tol = 1e-12 * qmax;
    if (emax <= tol) {
        g->mode = 1;
    } else if (emax <= kMaxShellResidual * qmax && emax * rmax <= kMaxResidualPhase / kTwoPiTurns) {
        g->mode = 2;
        g->runs.resize(ns);
        for (int s = 0; s < ns; ++s) {
            // extend the run from s while every shell inside stays on the line
            // through its end points
            int last = s;
            double step = 0.0;
            for (int e = s + 1; e < std::min(ns, s + kMaxRunShells); ++e) {
                const double st = (qlen[e] - qlen[s]) / (double)(e - s);
                bool on = true;
                for (int k = s + 1; k < e && on; ++k)
                    on = std::fabs(qlen[k] - (qlen[s] + (double)(k - s) * st)) <= tol;
                if (!on) break;
                last = e;
                step = st;
            }
            g->runs[s] = ShellRun{step, last, 0};
        }
    } else {
        g->res.clear();
        g->step = 0.0;
    }
    return g->mode;
}

template <int VS>
static void launch_direct(const OrientKernelArgs &k, bool per_row, int blocks, hipStream_t stream) {
    if (per_row)
        hipLaunchKernelGGL((amp_direct_kernel<VS, true>), dim3(blocks), dim3(256), 0, stream, k);
    else
        hipLaunchKernelGGL((amp_direct_kernel<VS, false>), dim3(blocks), dim3(256), 0, stream, k);
}

hipError_t launch_amp_oriented(const OrientArgs &a, hipStream_t stream) {
    if (a.shape < 0 || a.shape >= kOrientShapes) return hipErrorInvalidValue;
    const OrientKernelArgs k = make_orient_args(a);
    const int blocks = oriented_grid(k.ftiles, k.split, k.ogroups, k.sgroups);
    const bool per_row = a.per_shell_b != 0;
    if (a.shape == 0 && a.ap == 0) {
        switch ((a.ns + k.sgroups - 1) / k.sgroups) {
            case 1: launch_direct<1>(k, per_row, blocks, stream); break;
            case 2: launch_direct<2>(k, per_row, blocks, stream); break;
            case 3: launch_direct<3>(k, per_row, blocks, stream); break;
            case 4: launch_direct<4>(k, per_row, blocks, stream); break;
            case 5: launch_direct<5>(k, per_row, blocks, stream); break;
            case 6: launch_direct<6>(k, per_row, blocks, stream); break;
            case 7: launch_direct<7>(k, per_row, blocks, stream); break;
            default: launch_direct<8>(k, per_row, blocks, stream); break;
        }
        return hipGetLastError();
    }
    switch (a.shape) {
        case 0: return launch_oriented_shape<2, 8>(k, per_row, blocks, stream);
        case 1: return launch_oriented_shape<4, 4>(k, per_row, blocks, stream);
        case 2: return launch_oriented_shape<1, 8>(k, per_row, blocks, stream);
        case 3: return launch_oriented_shape<1, 16>(k, per_row, blocks, stream);
        default: return launch_oriented_shape<1, 20>(k, per_row, blocks, stream);
    }
}

// ------------------------------------------------------- few frames ------

// pack[t][j] = (x, y, z, b) of atom j at frame t < NF (b: one factor per atom,
// or nullptr); padding atoms as staged.
__global__ __launch_bounds__(256) void pack_frames_kernel(const float *__restrict__ X, const float *__restrict__ Y,
                                                          const float *__restrict__ Z, const float *__restrict__ b,
                                                          size_t NAp, size_t NFp, float4 *__restrict__ pack) {
    const size_t j = (size_t)blockIdx.x * 256 + threadIdx.x, t = blockIdx.y;
    if (j >= NAp) return;
    const size_t e = j * NFp + t;
    pack[t * NAp + j] = make_float4(X[e], Y[e], Z[e], b ? b[j] : 0.f);
}

// Work of a wavefront of the few-frames launch, items in the order
// (frame, range, part, shell tile, orientation group), the last fastest, so that the
// wavefronts of a CU read the same atoms.
struct FewItem {
    int t, sp, part, sg, og;
};

__device__ __forceinline__ bool few_item(const OrientKernelArgs &a, FewItem &w) {
    int i = __builtin_amdgcn_readfirstlane((int)blockIdx.x * 4 + (int)(threadIdx.x >> 6));
    w.og = i % a.ogroups;
    i /= a.ogroups;
    w.sg = i % a.sgroups;
    i /= a.sgroups;
    w.part = i % a.sub;
    i /= a.sub;
    w.sp = i % a.split;
    w.t = i / a.split;
    return w.t < a.NF;
}

template <int VS, bool PER_ROW_B>
__global__ __launch_bounds__(256, 2) void amp_few_kernel(OrientKernelArgs a) {
    FewItem w;
    if (!few_item(a, w)) return;
    oriented_tile<1, VS, PER_ROW_B, true, true>(a, w.t, w.sp, w.og, w.sg * VS, w.part);
}

template <int VS>
__global__ __launch_bounds__(256, 2) void amp_few_res_kernel(OrientKernelArgs a) {
    extern __shared__ double tot_lds[];
    FewItem w;
    if (!few_item(a, w)) return;
    residual_tile<1, VS, true>(a, w.t, w.sp, w.og, w.sg * VS, tot_lds, w.part);
}

// amp[v][t] = the ranges' amplitudes, each rounded to FP32 from the FP64 sum
// of its parts, added in FP32 in the ranges' order.
__global__ __launch_bounds__(kWave) void few_amplitudes_kernel(const double2 *__restrict__ parts, int split, int sub,
                                                             int V, int NF, size_t NFp, float2 *__restrict__ amp) {
    const size_t i = (size_t)blockIdx.x * kWave + threadIdx.x, n = (size_t)V * NF;
    if (i >= n) return;
    float2 s = make_float2(0.f, 0.f);
    for (int k = 0; k < split; ++k) {
        double2 v = make_double2(0.0, 0.0);
#pragma unroll 8
        for (int p = 0; p < sub; ++p) {
            const double2 x = parts[((size_t)k * sub + p) * n + i];
            v.x += x.x;
            v.y += x.y;
        }
        const float re = (float)v.x, im = (float)v.y;
        s.x = k ? s.x + re : re;
        s.y = k ? s.y + im : im;
    }
    amp[(i / NF) * NFp + i % NF] = s;
}

// Lane = orientation pays where the frames' padding (NFp lanes for NF frames)
// exceeds that of the orientations by a third: one frame of 100,000 atoms, 40
// shells x 500 orientations: 18.4 ms with lane = frame, 0.47 ms so (packing and
// adding the parts 0.03 ms more), bound by instruction issue as the other form
// is.  Up to that third the other form's coalesced coordinates need no packing.
bool few_frames(size_t NF, size_t NFp, int NM) {
    const double lanes = (double)NF * ((NM + kWave - 1) / kWave * kWave);
    return NFp == (size_t)kWave && lanes * 4.0 / 3.0 <= (double)NFp * NM;
}

// Parts of an atom range, of at least 4 folds: about 4096 wavefronts in all.
int few_parts(size_t NF, size_t NAp, int NM, int ns, int split, int shape) {
    const long items = (long)NF * split * ((NM + kWave - 1) / kWave) * ((ns + kShapeVS[shape] - 1) / kShapeVS[shape]);
    const long most = std::max<long>(1, (long)(NAp / split / 256));
    return (int)std::max<long>(1, std::min(most, 4096 / std::max<long>(items, 1)));
}

template <int VS>
static hipError_t launch_few_shape(const OrientKernelArgs &k, bool per_row, unsigned blocks, hipStream_t stream) {
    if (k.ap == 2) {
        if (per_row) return hipErrorInvalidValue;
        const void *fn = (const void *)amp_few_res_kernel<VS>;
        const size_t lds = kResidualLds<1, VS>;
        hipError_t e = hipFuncSetAttribute(fn, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
        if (e != hipSuccess) return e;
        hipLaunchKernelGGL((amp_few_res_kernel<VS>), dim3(blocks), dim3(256), lds, stream, k);
    } else if (per_row)
        hipLaunchKernelGGL((amp_few_kernel<VS, true>), dim3(blocks), dim3(256), 0, stream, k);
    else
        hipLaunchKernelGGL((amp_few_kernel<VS, false>), dim3(blocks), dim3(256), 0, stream, k);
    return hipGetLastError();
}

hipError_t launch_amp_few(const OrientArgs &a, int NF, int sub, float4 *pack, double2 *parts, hipStream_t stream) {
    if (a.shape < 0 || a.shape >= kOrientShapes || sub < 1 || NF < 1 || (size_t)NF > a.NFp) return hipErrorInvalidValue;
    OrientKernelArgs k = make_orient_args(a);
    k.ogroups = (a.NM + kWave - 1) / kWave;
    k.pack = pack;
    k.parts = parts;
    k.sub = sub;
    k.NF = NF;
    hipLaunchKernelGGL(pack_frames_kernel, dim3((unsigned)((a.NAp + 255) / 256), (unsigned)NF), dim3(256), 0, stream,
                       k.X, k.Y, k.Z, a.per_shell_b ? nullptr : a.b, a.NAp, a.NFp, pack);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
    const size_t items = (size_t)NF * a.split * sub * k.sgroups * k.ogroups;
    if (items > (size_t)1 << 30) return hipErrorInvalidValue;
    const unsigned blocks = (unsigned)((items + 3) / 4);
    const bool per_row = a.per_shell_b != 0;
    switch (kShapeVS[a.shape]) {
        case 4: e = launch_few_shape<4>(k, per_row, blocks, stream); break;
        case 8: e = launch_few_shape<8>(k, per_row, blocks, stream); break;
        case 16: e = launch_few_shape<16>(k, per_row, blocks, stream); break;
        default: e = launch_few_shape<20>(k, per_row, blocks, stream); break;
    }
    if (e != hipSuccess) return e;
    hipLaunchKernelGGL(few_amplitudes_kernel, dim3((unsigned)(((size_t)k.V * NF + kWave - 1) / kWave)), dim3(kWave), 0,
                       stream, parts, a.split, sub, k.V, NF, a.NFp, a.amp);
    return hipGetLastError();
}

template <int VM, int VS>
static hipError_t oriented_occupancy(bool per_row, int mode, int *blocks) {
    if (mode == 2) {
        const void *k = (const void *)amp_oriented_res_kernel<VM, VS>;
        const size_t lds = kResidualLds<VM, VS>;
        hipError_t e = hipFuncSetAttribute(k, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
        if (e != hipSuccess) return e;
        return hipOccupancyMaxActiveBlocksPerMultiprocessor(blocks, k, 256, lds);
    }
    const void *k = per_row ? (const void *)amp_oriented_kernel<VM, VS, true>
                            : (const void *)amp_oriented_kernel<VM, VS, false>;
    return hipOccupancyMaxActiveBlocksPerMultiprocessor(blocks, k, 256, 0);
}

hipError_t oriented_blocks_per_cu(int shape, bool per_row, int mode, int *blocks) {
    *blocks = 0;
    switch (shape) {
        case 0: return oriented_occupancy<2, 8>(per_row, mode, blocks);
        case 1: return oriented_occupancy<4, 4>(per_row, mode, blocks);
        case 2: return oriented_occupancy<1, 8>(per_row, mode, blocks);
        case 3: return oriented_occupancy<1, 16>(per_row, mode, blocks);
        case 4: return oriented_occupancy<1, 20>(per_row, mode, blocks);
        default: return hipErrorInvalidValue;
    }
}

int oriented_base_blocks(size_t NFp, int NM, int ns, int shape) {
    const int VM = kShapeVM[shape], VS = kShapeVS[shape];
    return (int)(NFp / kWave) * ((NM + 4 * VM - 1) / (4 * VM)) * ((ns + VS - 1) / VS);
}

hipError_t launch_amp_all(const AmpArgs &a, hipStream_t stream) {
    AmpKernelArgs k;
    k.X = a.coords;
    k.Y = a.coords + a.NAp * a.NFp;
    k.Z = a.coords + 2 * a.NAp * a.NFp;
    k.NFp = a.NFp;
    k.qrev = a.qrev;
    k.b = a.b;
    k.brow = a.brow;
    k.NAp = a.NAp;
    k.V = a.V;
    k.ftiles = (int)(a.NFp / kWave);
    k.vgroups = (a.V + a.vb - 1) / a.vb;
    k.split = a.split;
    size_t aps = (a.NAp + a.split - 1) / a.split;
    aps = (aps + kAtomChunk - 1) / kAtomChunk * kAtomChunk;
    k.atoms_per_split = (int)aps;
    k.amp = a.amp;
    const int nitems = (k.ftiles * k.split * k.vgroups + 3) / 4;
    const int blocks = ((nitems + 7) / 8) * 8;
    const bool per_row = a.brow != nullptr;
#define SX_AMP_CASE(VBV)                                                                         \
    case VBV:                                                                                    \
        if (per_row)                                                                             \
            hipLaunchKernelGGL((amp_all_kernel<VBV, true>), dim3(blocks), dim3(256), 0, stream, k);  \
        else                                                                                     \
            hipLaunchKernelGGL((amp_all_kernel<VBV, false>), dim3(blocks), dim3(256), 0, stream, k); \
        break;
    switch (a.vb) {
        SX_AMP_CASE(4)
        SX_AMP_CASE(8)
        SX_AMP_CASE(16)
        default:
            return hipErrorInvalidValue;
    }
#undef SX_AMP_CASE
    return hipGetLastError();
}

hipError_t all_blocks_per_cu(int vb, bool per_row, int *blocks) {
    *blocks = 0;
    const void *k = nullptr;
    switch (vb) {
        case 4: k = per_row ? (const void *)amp_all_kernel<4, true> : (const void *)amp_all_kernel<4, false>; break;
        case 8: k = per_row ? (const void *)amp_all_kernel<8, true> : (const void *)amp_all_kernel<8, false>; break;
        case 16: k = per_row ? (const void *)amp_all_kernel<16, true> : (const void *)amp_all_kernel<16, false>; break;
        default: return hipErrorInvalidValue;
    }
    return hipOccupancyMaxActiveBlocksPerMultiprocessor(blocks, k, 256, 0);
}

}  // namespace sx
