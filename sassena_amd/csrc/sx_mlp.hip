// sx_mlp.hip -- the small network of the learned control variate, trained and
// evaluated by hand-written gfx950 kernels.
//
// y = W3 . tanh(W2 tanh(W1 x + b1) + b2) + b3 with 16 inputs (zero padded),
// two hidden layers of 128 and one output.  W1 and W2 are BF16 operands of
// v_mfma_f32_16x16x16_bf16 (FP32 accumulation); the output layer, biases,
// activations and optimizer state are FP32.
// Operand layouts of the 16x16x16 MFMA (lane l, register j < 4):
//   A[m][k]: m = l % 16, k = 4 (l / 16) + j;  B[k][n]: k = 4 (l / 16) + j,
//   n = l % 16;  D[m][n]: m = 4 (l / 16) + j, n = l % 16.
// A D tile of h1 is therefore the A operand of h1^T and a D tile of dz2 the B
// operand of dz2, so the weight gradients need no shuffles.
//
// A step is bound by latency, not by its 0.5 GFLOP: a workgroup takes 64 rows
// with 16 wavefronts, wavefront = (16 rows) x (2 of 8 column tiles), so that
// every stage is a few MFMAs deep; the weights are kept as ready operand
// fragments (8 B a lane, loaded at the start straight into registers);
// activations and their derivatives pass between wavefronts through LDS, as
// fragments for the weight gradients and as rows for the next layer.  A second
// launch sums the workgroups' partials and applies Adam.
//
// Every sum has one order, whichever wavefronts hold its terms, so that results
// neither vary from run to run nor follow the layout: an output adds its columns
// tile after tile, then over the 16 of a tile; a workgroup's weight gradients
// are those of its 16-row tiles added one after the other, as are db3 and the
// loss; the gradients of its columns are those of its 4-row groups; the
// workgroups follow in order.  Products that enter a sum do so by fmaf, which
// leaves the compiler no choice of which one to fuse.  (Adam carries a rounding
// of one sum into the fourth digit of the parameters within 500 steps.)
// 4,096 rows a step: 14 + 4 us (133 + 16 us when each of four wavefronts took 16
// rows through all columns, copied W2 into LDS and added its gradients there
// by LDS atomics).
#include <hip/hip_runtime.h>

#include <cmath>
#include <cstdarg>
#include <cstdint>
#include <cstdio>
#include <string>
#include <vector>

#include "../../include/sassena_amd.h"

namespace sxm {

constexpr int IN = 16, H = 128;
constexpr int OFF_W1 = 0, OFF_B1 = OFF_W1 + IN * H, OFF_W2 = OFF_B1 + H, OFF_B2 = OFF_W2 + H * H,
              OFF_W3 = OFF_B2 + H, OFF_B3 = OFF_W3 + H, NPARAM = OFF_B3 + 1;
constexpr int ROWS_PER_BLOCK = 64;
constexpr int kStepThreads = 1024;
// A workgroup's gradients and loss: the 64 tiles of W2 and the 8 of W1 as
// fragments [tile][lane][4], then b1, b2, W3, b3 and the loss, padded to 16 B.
constexpr int PK_W2 = 0, PK_W1 = PK_W2 + H * H, PK_B1 = PK_W1 + IN * H, PK_B3 = PK_B1 + 3 * H, PK_LOSS = PK_B3 + 1,
              PK = (PK_LOSS + 1 + 3) / 4 * 4;
// BF16 operand fragments: W1 [nt][lane][4], W2 [nt][kt][lane][4] (B operand of
// h1 W2), W2^T [nt][kt][lane][4] (B operand of dz2 W2^T).
constexpr int FR_W1 = 0, FR_W2 = FR_W1 + IN * H, FR_W2T = FR_W2 + H * H, FR = FR_W2T + H * H;

typedef short bf16x4 __attribute__((ext_vector_type(4)));
typedef float f32x4 __attribute__((ext_vector_type(4)));

__device__ __forceinline__ short to_bf16(float f) {
    // round to nearest even (finite inputs)
    unsigned u = __float_as_uint(f);
    u += 0x7fffu + ((u >> 16) & 1u);
    return (short)(u >> 16);
}
__device__ __forceinline__ float from_bf16(short s) { return __uint_as_float(((unsigned)(unsigned short)s) << 16); }

__device__ __forceinline__ f32x4 mfma(bf16x4 a, bf16x4 b, f32x4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(a, b, c, 0, 0, 0);
}

// Row index of batch row r of step `step`: a hashed draw from [0, n).
__device__ __forceinline__ unsigned pick_row(unsigned long long seed, unsigned step, unsigned r, unsigned n) {
    unsigned long long z = seed ^ ((unsigned long long)step << 32) ^ r;
    z += 0x9e3779b97f4a7c15ull;
    z = (z ^ (z >> 30)) * 0xbf58476d1ce4e5b9ull;
    z = (z ^ (z >> 27)) * 0x94d049bb133111ebull;
    z ^= z >> 31;
    return (unsigned)(z % n);
}

struct StepArgs {
    const float *x;        // [n][IN] inputs
    const float *t;        // [n] targets (nullptr: forward only)
    unsigned n;            // rows available
    unsigned rows;         // rows in this batch
    int sample;            // 1: draw rows with pick_row, 0: rows 0..rows-1
    unsigned long long seed;
    unsigned step;
    const short *frag;     // BF16 operand fragments of W1, W2, W2^T
    const float *p;        // FP32 parameters (b1, b2, W3, b3 used from here)
    float *y;              // [rows] outputs (optional)
    float *partial;        // [blocks][PK] gradients and loss of each workgroup (training)
};

// Row stride of the row-major LDS tiles: 132 shorts, so that the 16 rows of an
// A operand start in different banks.
constexpr int LD = H + 4;

// Forward (and backward when a.t != nullptr) of ROWS_PER_BLOCK rows.
__global__ __launch_bounds__(kStepThreads) void mlp_step_kernel(StepArgs a) {
    __shared__ short rows_lds[ROWS_PER_BLOCK * LD];  // h1, then dz2: A operands
    __shared__ bf16x4 h1f[4 * 8 * 64];               // D tiles [row tile][column tile][lane]
    __shared__ bf16x4 xf[4 * 64];                    // x^T: A operand of dW1
    __shared__ float yrow[ROWS_PER_BLOCK];
    __shared__ float sums[2][16];                    // db3 and loss per 4-row group
    __shared__ union {
        float h2[4][4][8][64];                       // [row tile][row mod 4][column tile][lane]
        struct {
            bf16x4 dzf[4 * 8 * 64];                  // dz2, then dz1: D tiles
            float cols[3][16][H];                    // db1, db2, dW3 per 4-row group
        };
    } u;
    bf16x4 *dzf = u.dzf;
    auto &cols = u.cols;
    const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
    const int rt = wave & 3, cq = wave >> 2;         // row tile, column quarter (tiles 2 cq, 2 cq + 1)
    const bool train = a.t != nullptr;
    const int lr = lane & 15, lg = lane >> 4;        // MFMA lane row/col and k group
    const bf16x4 *F = reinterpret_cast<const bf16x4 *>(a.frag);

    // operand fragments of this wavefront's columns
    bf16x4 w1f[2], w2f[2][8], w2t[2][8];
#pragma unroll
    for (int i = 0; i < 2; ++i) {
        const int nt = 2 * cq + i;
        w1f[i] = F[FR_W1 / 4 + nt * 64 + lane];
#pragma unroll
        for (int kt = 0; kt < 8; ++kt) {
            w2f[i][kt] = F[FR_W2 / 4 + (nt * 8 + kt) * 64 + lane];
            if (train) w2t[i][kt] = F[FR_W2T / 4 + (nt * 8 + kt) * 64 + lane];
        }
    }
    // the input row of lane row lr, and those of the D-layout rows 4 lg + j
    const unsigned row0 = blockIdx.x * ROWS_PER_BLOCK + rt * 16;
    int ra = -1;
    if (row0 + lr < a.rows) ra = (int)(a.sample ? pick_row(a.seed, a.step, row0 + lr, a.n) : row0 + lr);
    f32x4 xv = {0.f, 0.f, 0.f, 0.f};
    if (ra >= 0) xv = *reinterpret_cast<const f32x4 *>(a.x + (size_t)ra * IN + 4 * lg);
    int rd[4];
    float tv[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        rd[j] = __shfl(ra, 4 * lg + j, 64);
        tv[j] = train && rd[j] >= 0 ? a.t[rd[j]] : 0.f;
    }
    bf16x4 xa;
#pragma unroll
    for (int j = 0; j < 4; ++j) xa[j] = to_bf16(xv[j]);
    if (train && cq == 0) {
        // x[row lr][4 lg + j] is element (k = 4 lg + j, row lr) of x^T: lane
        // (lr / 4) * 16 + k, register lr % 4 of its A operand
        short *xs = reinterpret_cast<short *>(xf + rt * 64);
#pragma unroll
        for (int j = 0; j < 4; ++j) xs[((lr >> 2) * 16 + 4 * lg + j) * 4 + (lr & 3)] = xa[j];
    }

    // ---- layer 1: h1 = tanh(x W1 + b1)
    float h1[2][4];
#pragma unroll
    for (int i = 0; i < 2; ++i) {
        const int nt = 2 * cq + i;
        f32x4 acc = {0.f, 0.f, 0.f, 0.f};
        acc = mfma(xa, w1f[i], acc);
        const float bias = a.p[OFF_B1 + 16 * nt + lr];
        bf16x4 f;
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            h1[i][j] = tanhf(acc[j] + bias);
            f[j] = to_bf16(h1[i][j]);
            rows_lds[(rt * 16 + 4 * lg + j) * LD + 16 * nt + lr] = f[j];
        }
        h1f[(rt * 8 + nt) * 64 + lane] = f;
    }
    __syncthreads();
    // ---- layer 2: h2 = tanh(h1 W2 + b2)
    const short *arow = rows_lds + (rt * 16 + lr) * LD + 4 * lg;
    float h2[2][4], w3[2];
    {
        f32x4 acc[2] = {{0.f, 0.f, 0.f, 0.f}, {0.f, 0.f, 0.f, 0.f}};
#pragma unroll
        for (int kt = 0; kt < 8; ++kt) {
            const bf16x4 av = *reinterpret_cast<const bf16x4 *>(arow + 16 * kt);
#pragma unroll
            for (int i = 0; i < 2; ++i) acc[i] = mfma(av, w2f[i][kt], acc[i]);
        }
#pragma unroll
        for (int i = 0; i < 2; ++i) {
            const int c = 16 * (2 * cq + i) + lr;
            const float bias = a.p[OFF_B2 + c];
            w3[i] = a.p[OFF_W3 + c];
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                h2[i][j] = tanhf(acc[i][j] + bias);
                u.h2[rt][j][2 * cq + i][lane] = h2[i][j];
            }
        }
    }
    __syncthreads();
    // ---- layer 3: y[r] = h2[r] . W3 + b3, rows 4 lg + cq: tile after tile, then
    // over the 16 lanes of a k group
    {
        float s = 0.f;
#pragma unroll
        for (int nt = 0; nt < 8; ++nt) s = fmaf(u.h2[rt][cq][nt][lane], a.p[OFF_W3 + 16 * nt + lr], s);
#pragma unroll
        for (int off = 8; off > 0; off >>= 1) s += __shfl_xor(s, off, 64);
        s += a.p[OFF_B3];
        const unsigned r = 4 * lg + cq;
        if (lr == 0) {
            yrow[rt * 16 + r] = s;
            if (a.y && row0 + r < a.rows) a.y[row0 + r] = s;
        }
    }
    if (!train) return;
    __syncthreads();  // h2 is read: dz2 and the columns' sums take its place
    float yr[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) yr[j] = yrow[rt * 16 + 4 * lg + j];

    // ---- loss and dy = 2 (y - t) / rows (rows beyond the batch contribute 0)
    float dy[4], dsum = 0.f, lsum = 0.f;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        const float e = rd[j] >= 0 ? yr[j] - tv[j] : 0.f;
        dy[j] = 2.f * e / (float)a.rows;
        dsum += dy[j];
        lsum = fmaf(e, e, lsum);
    }
    if (cq == 0 && lr == 0) {
        sums[0][rt * 4 + lg] = dsum;
        sums[1][rt * 4 + lg] = lsum;
    }
    // ---- dz2 = dy W3 (1 - h2^2); dW3 = sum dy h2; db2 = sum dz2
#pragma unroll
    for (int i = 0; i < 2; ++i) {
        const int nt = 2 * cq + i, c = 16 * nt + lr;
        float gw3 = 0.f, gb2 = 0.f;
        bf16x4 f;
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const float dw = dy[j] * w3[i], d = fmaf(-h2[i][j], h2[i][j], 1.f);
            gw3 = fmaf(dy[j], h2[i][j], gw3);
            gb2 = fmaf(dw, d, gb2);
            f[j] = to_bf16(dw * d);
            rows_lds[(rt * 16 + 4 * lg + j) * LD + c] = f[j];  // h1's rows were read before the last barrier
        }
        dzf[(rt * 8 + nt) * 64 + lane] = f;
        cols[2][rt * 4 + lg][c] = gw3;
        cols[1][rt * 4 + lg][c] = gb2;
    }
    __syncthreads();
    float *dst = a.partial + (size_t)blockIdx.x * PK;
    const f32x4 zero = {0.f, 0.f, 0.f, 0.f};
    // ---- dW2[k][c] = sum_r h1[r][k] dz2[r][c]: A = h1^T (D tiles of h1), B = dz2 (D tiles);
    // row of tiles wave / 2, four of its tiles, each row tile's product added to the last
    {
        const int mt = wave >> 1, c0 = (wave & 1) * 4;
        f32x4 acc[4] = {zero, zero, zero, zero};
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const bf16x4 av = h1f[(r * 8 + mt) * 64 + lane];
#pragma unroll
            for (int i = 0; i < 4; ++i) acc[i] += mfma(av, dzf[(r * 8 + c0 + i) * 64 + lane], zero);
        }
#pragma unroll
        for (int i = 0; i < 4; ++i)
            *reinterpret_cast<f32x4 *>(dst + PK_W2 + ((mt * 8 + c0 + i) * 64 + lane) * 4) = acc[i];
    }
    // ---- dh1 = dz2 W2^T, dz1 = dh1 (1 - h1^2); db1 = sum dz1
    bf16x4 d1[2];
    {
        f32x4 acc[2] = {{0.f, 0.f, 0.f, 0.f}, {0.f, 0.f, 0.f, 0.f}};
#pragma unroll
        for (int kt = 0; kt < 8; ++kt) {
            const bf16x4 av = *reinterpret_cast<const bf16x4 *>(arow + 16 * kt);
#pragma unroll
            for (int i = 0; i < 2; ++i) acc[i] = mfma(av, w2t[i][kt], acc[i]);
        }
#pragma unroll
        for (int i = 0; i < 2; ++i) {
            float gb1 = 0.f;
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                const float d = fmaf(-h1[i][j], h1[i][j], 1.f);
                gb1 = fmaf(acc[i][j], d, gb1);
                d1[i][j] = to_bf16(acc[i][j] * d);
            }
            cols[0][rt * 4 + lg][16 * (2 * cq + i) + lr] = gb1;
        }
    }
    __syncthreads();  // dz2's fragments are read
#pragma unroll
    for (int i = 0; i < 2; ++i) dzf[(rt * 8 + 2 * cq + i) * 64 + lane] = d1[i];
    __syncthreads();
    // ---- dW1[k][c] = sum_r x[r][k] dz1[r][c]
    if (wave < 8) {
        f32x4 acc = zero;
#pragma unroll
        for (int r = 0; r < 4; ++r) acc += mfma(xf[r * 64 + lane], dzf[(r * 8 + wave) * 64 + lane], zero);
        *reinterpret_cast<f32x4 *>(dst + PK_W1 + (wave * 64 + lane) * 4) = acc;
    } else {
        const int i = tid - 512;
        if (i < 3 * H) {
            float s = 0.f;
#pragma unroll
            for (int k = 0; k < 16; ++k) s += cols[i / H][k][i % H];
            dst[PK_B1 + i] = s;
        } else if (i < 3 * H + 2) {
            float s = 0.f;
            for (int r = 0; r < 16; r += 4) {
                const float *g = sums[i - 3 * H] + r;
                s += ((g[0] + g[1]) + g[2]) + g[3];
            }
            dst[PK_B3 + i - 3 * H] = s;
        }
    }
}

// The parameter of entry e of a workgroup's gradients (e < PK_LOSS).
__device__ __forceinline__ int packed_param(int e) {
    if (e >= PK_B1) {
        const int q = e - PK_B1;
        return q < H ? OFF_B1 + q : q < 2 * H ? OFF_B2 + q - H : q < 3 * H ? OFF_W3 + q - 2 * H : OFF_B3;
    }
    const bool second = e < PK_W1;
    const int r = second ? e : e - PK_W1, tile = r >> 8, lane = (r >> 2) & 63, j = r & 3;
    const int row = (second ? 16 * (tile >> 3) : 0) + 4 * (lane >> 4) + j, col = 16 * (tile & 7) + (lane & 15);
    return (second ? OFF_W2 : OFF_W1) + row * H + col;
}

// The BF16 operand fragments of parameter i (of W1 or W2) with value v.
__device__ __forceinline__ void put_fragment(short *frag, int i, float v) {
    const short b = to_bf16(v);
    if (i >= OFF_W1 && i < OFF_B1) {
        const int k = (i - OFF_W1) / H, n = (i - OFF_W1) % H;
        frag[FR_W1 + (((n >> 4) * 64) + (k >> 2) * 16 + (n & 15)) * 4 + (k & 3)] = b;
    } else if (i >= OFF_W2 && i < OFF_B2) {
        const int k = (i - OFF_W2) / H, n = (i - OFF_W2) % H;
        frag[FR_W2 + (((n >> 4) * 8 + (k >> 4)) * 64 + ((k >> 2) & 3) * 16 + (n & 15)) * 4 + (k & 3)] = b;
        frag[FR_W2T + (((k >> 4) * 8 + (n >> 4)) * 64 + ((n >> 2) & 3) * 16 + (k & 15)) * 4 + (n & 3)] = b;
    }
}

// Sums the workgroups' gradients in their order into grad, and optionally
// applies one Adam step to the FP32 parameters and refreshes the BF16
// fragments.  A thread loads 4 entries of every kSlices-th workgroup into LDS,
// kStaged workgroups at a time; then each entry has a thread that adds them.
constexpr int kSlices = 16, kGroups = 16, kStaged = 64;
__global__ __launch_bounds__(kSlices *kGroups) void mlp_reduce_adam_kernel(
    const float *__restrict__ partial, int blocks, float *__restrict__ grad, float *__restrict__ loss,
    float *__restrict__ p, float *__restrict__ m, float *__restrict__ v, short *__restrict__ frag, int apply, float lr,
    float b1c, float b2c) {
    __shared__ f32x4 sh[kStaged][kGroups];
    const int g = threadIdx.x % kGroups, sl = threadIdx.x / kGroups;
    const int e0 = ((int)blockIdx.x * kGroups + g) * 4;
    const int gi = threadIdx.x >> 2, j = threadIdx.x & 3, e = ((int)blockIdx.x * kGroups + gi) * 4 + j;
    float gr = 0.f;
    for (int b0 = 0; b0 < blocks; b0 += kStaged) {
        const int nb = min(kStaged, blocks - b0);
        f32x4 x[kStaged / kSlices];
#pragma unroll
        for (int k = 0; k < kStaged / kSlices; ++k) {
            const int b = sl + k * kSlices;
            if (b < nb && e0 < PK) x[k] = *reinterpret_cast<const f32x4 *>(partial + (size_t)(b0 + b) * PK + e0);
        }
#pragma unroll
        for (int k = 0; k < kStaged / kSlices; ++k) {
            const int b = sl + k * kSlices;
            if (b < nb && e0 < PK) sh[b][g] = x[k];
        }
        __syncthreads();
        if (threadIdx.x < kGroups * 4) {
            // one entry a thread
#pragma unroll 16
            for (int b = 0; b < nb; ++b) gr += sh[b][gi][j];
        }
        __syncthreads();
    }
    if (threadIdx.x >= kGroups * 4 || e > PK_LOSS) return;
    if (e == PK_LOSS) {
        if (loss) *loss = gr;
        return;
    }
    const int i = packed_param(e);
    grad[i] = gr;
    if (!apply) return;
    const float beta1 = 0.9f, beta2 = 0.999f, eps = 1e-8f;
    const float mi = beta1 * m[i] + (1.f - beta1) * gr;
    const float vi = beta2 * v[i] + (1.f - beta2) * gr * gr;
    m[i] = mi;
    v[i] = vi;
    const float pi = p[i] - lr * (mi / b1c) / (sqrtf(vi / b2c) + eps);
    p[i] = pi;
    put_fragment(frag, i, pi);
}

__global__ void mlp_fragments_kernel(const float *__restrict__ p, short *__restrict__ frag) {
    const int i = blockIdx.x * 256 + threadIdx.x;
    if (i < NPARAM) put_fragment(frag, i, p[i]);
}

}  // namespace sxm

struct sx_mlp {
    int device = 0;
    std::string err;
    hipStream_t stream = nullptr;
    float *p = nullptr, *m = nullptr, *v = nullptr, *grad = nullptr, *partial = nullptr, *loss = nullptr;
    short *frag = nullptr;
    float *x = nullptr, *t = nullptr, *y = nullptr;
    size_t xcap = 0, pcap_blocks = 0;
    unsigned long long adam_t = 0;
};

namespace {

int mfail(sx_mlp *n, int code, const char *fmt, ...) {
    char buf[512];
    va_list ap;
    va_start(ap, fmt);
    vsnprintf(buf, sizeof buf, fmt, ap);
    va_end(ap);
    if (n) n->err = buf;
    return code;
}

#define SXM_HIP(n, expr)                                                                                    \
    do {                                                                                                    \
        hipError_t e_ = (expr);                                                                             \
        if (e_ != hipSuccess) {                                                                             \
            (void)hipGetLastError(); /* reported here, and not by the next call's launches too */           \
            return mfail((n), e_ == hipErrorOutOfMemory ? SX_ERR_NOMEM : SX_ERR_HIP, "%s failed: %s (%s:%d)", \
                         #expr, hipGetErrorString(e_), __FILE__, __LINE__);                                 \
        }                                                                                                   \
    } while (0)

// The capacities hold only for buffers that are there: 0 until every allocation succeeded.
int ensure_rows(sx_mlp *n, size_t rows) {
    if (rows <= n->xcap) return SX_OK;
    n->xcap = 0;
    for (float **q : {&n->x, &n->t, &n->y})
        if (*q) {
            (void)hipFree(*q);
            *q = nullptr;
        }
    SXM_HIP(n, hipMalloc(&n->x, sizeof(float) * sxm::IN * rows));
    SXM_HIP(n, hipMalloc(&n->t, sizeof(float) * rows));
    SXM_HIP(n, hipMalloc(&n->y, sizeof(float) * rows));
    n->xcap = rows;
    return SX_OK;
}

int ensure_partials(sx_mlp *n, size_t blocks) {
    if (blocks <= n->pcap_blocks) return SX_OK;
    n->pcap_blocks = 0;
    if (n->partial) (void)hipFree(n->partial);
    n->partial = nullptr;
    SXM_HIP(n, hipMalloc(&n->partial, sizeof(float) * sxm::PK * blocks));
    n->pcap_blocks = blocks;
    return SX_OK;
}

int check_rows(sx_mlp *n, const float *x, size_t rows) {
    if (!x || rows == 0 || rows > (size_t)1 << 28) return mfail(n, SX_ERR_ARG, "bad row count %zu", rows);
    for (size_t i = 0; i < rows * sxm::IN; ++i)
        if (!std::isfinite(x[i])) return mfail(n, SX_ERR_ARG, "non-finite input at %zu", i);
    return SX_OK;
}

// One pass over `rows` rows (sampled from n when sample != 0): forward,
// and backward + reduction (+ Adam when apply) when t is given.
int step(sx_mlp *n, unsigned nrows_avail, unsigned rows, int sample, unsigned long long seed, unsigned stepno,
         bool train, int apply, float lr) {
    const unsigned blocks = (rows + sxm::ROWS_PER_BLOCK - 1) / sxm::ROWS_PER_BLOCK;
    if (train) {
        int rc = ensure_partials(n, blocks);
        if (rc != SX_OK) return rc;
    }
    sxm::StepArgs a;
    a.x = n->x;
    a.t = train ? n->t : nullptr;
    a.n = nrows_avail;
    a.rows = rows;
    a.sample = sample;
    a.seed = seed;
    a.step = stepno;
    a.frag = n->frag;
    a.p = n->p;
    a.y = train ? nullptr : n->y;
    a.partial = n->partial;
    hipLaunchKernelGGL(sxm::mlp_step_kernel, dim3(blocks), dim3(sxm::kStepThreads), 0, n->stream, a);
    SXM_HIP(n, hipGetLastError());
    if (train) {
        float b1c = 1.f, b2c = 1.f;
        if (apply) {
            n->adam_t++;
            b1c = 1.f - powf(0.9f, (float)n->adam_t);
            b2c = 1.f - powf(0.999f, (float)n->adam_t);
        }
        constexpr int per = 4 * sxm::kGroups;
        hipLaunchKernelGGL(sxm::mlp_reduce_adam_kernel, dim3((sxm::PK + per - 1) / per),
                           dim3(sxm::kSlices * sxm::kGroups), 0, n->stream, n->partial, (int)blocks, n->grad, n->loss,
                           n->p, n->m, n->v, n->frag, apply, lr, b1c, b2c);
        SXM_HIP(n, hipGetLastError());
    }
    return SX_OK;
}

}  // namespace

extern "C" {

size_t sx_mlp_param_count(void) { return (size_t)sxm::NPARAM; }

const char *sx_mlp_last_error(const sx_mlp *n) { return n ? n->err.c_str() : "null network"; }

int sx_mlp_create(int device, unsigned long long seed, sx_mlp **out) {
    if (!out) return SX_ERR_ARG;
    *out = nullptr;
    int ndev = 0;
    if (hipGetDeviceCount(&ndev) != hipSuccess || device < 0 || device >= ndev) return SX_ERR_HIP;
    if (hipSetDevice(device) != hipSuccess) return SX_ERR_HIP;
    sx_mlp *n = new (std::nothrow) sx_mlp();
    if (!n) return SX_ERR_NOMEM;
    n->device = device;
    int rc = SX_OK;
    auto fail = [&](hipError_t e) {
        if (e != hipSuccess && rc == SX_OK) rc = SX_ERR_HIP;
    };
    fail(hipStreamCreateWithFlags(&n->stream, hipStreamNonBlocking));
    fail(hipMalloc(&n->p, sizeof(float) * sxm::NPARAM));
    fail(hipMalloc(&n->m, sizeof(float) * sxm::NPARAM));
    fail(hipMalloc(&n->v, sizeof(float) * sxm::NPARAM));
    fail(hipMalloc(&n->grad, sizeof(float) * sxm::NPARAM));
    fail(hipMalloc(&n->loss, sizeof(float)));
    fail(hipMalloc(&n->frag, sizeof(short) * sxm::FR));
    if (rc != SX_OK) {
        sx_mlp_destroy(n);
        return rc;
    }
    // Glorot-uniform weights from a seeded generator, zero biases
    std::vector<float> p(sxm::NPARAM, 0.f);
    unsigned long long s = seed * 6364136223846793005ull + 1442695040888963407ull;
    auto uni = [&]() {
        s = s * 6364136223846793005ull + 1442695040888963407ull;
        return (double)(s >> 11) / 9007199254740992.0;
    };
    const double l1 = std::sqrt(6.0 / (sxm::IN + sxm::H)), l2 = std::sqrt(6.0 / (2 * sxm::H)),
                 l3 = std::sqrt(6.0 / (sxm::H + 1));
    for (int i = 0; i < sxm::IN * sxm::H; ++i) p[sxm::OFF_W1 + i] = (float)((2 * uni() - 1) * l1);
    for (int i = 0; i < sxm::H * sxm::H; ++i) p[sxm::OFF_W2 + i] = (float)((2 * uni() - 1) * l2);
    for (int i = 0; i < sxm::H; ++i) p[sxm::OFF_W3 + i] = (float)((2 * uni() - 1) * l3);
    rc = sx_mlp_set_params(n, p.data(), p.size());
    if (rc != SX_OK) {
        sx_mlp_destroy(n);
        return rc;
    }
    *out = n;
    return SX_OK;
}

void sx_mlp_destroy(sx_mlp *n) {
    if (!n) return;
    (void)hipSetDevice(n->device);
    if (n->stream) (void)hipStreamSynchronize(n->stream);
    for (float *q : {n->p, n->m, n->v, n->grad, n->partial, n->loss, n->x, n->t, n->y})
        if (q) (void)hipFree(q);
    if (n->frag) (void)hipFree(n->frag);
    if (n->stream) (void)hipStreamDestroy(n->stream);
    delete n;
}

int sx_mlp_set_params(sx_mlp *n, const float *params, size_t count) {
    if (!n) return SX_ERR_ARG;
    if (!params || count != (size_t)sxm::NPARAM) return mfail(n, SX_ERR_ARG, "expected %d parameters", sxm::NPARAM);
    SXM_HIP(n, hipSetDevice(n->device));
    SXM_HIP(n, hipMemcpyAsync(n->p, params, sizeof(float) * sxm::NPARAM, hipMemcpyHostToDevice, n->stream));
    SXM_HIP(n, hipMemsetAsync(n->m, 0, sizeof(float) * sxm::NPARAM, n->stream));
    SXM_HIP(n, hipMemsetAsync(n->v, 0, sizeof(float) * sxm::NPARAM, n->stream));
    hipLaunchKernelGGL(sxm::mlp_fragments_kernel, dim3((sxm::NPARAM + 255) / 256), dim3(256), 0, n->stream, n->p,
                       n->frag);
    SXM_HIP(n, hipGetLastError());
    SXM_HIP(n, hipStreamSynchronize(n->stream));
    n->adam_t = 0;
    return SX_OK;
}

int sx_mlp_get_params(sx_mlp *n, float *params, size_t count) {
    if (!n) return SX_ERR_ARG;
    if (!params || count != (size_t)sxm::NPARAM) return mfail(n, SX_ERR_ARG, "expected %d parameters", sxm::NPARAM);
    SXM_HIP(n, hipSetDevice(n->device));
    SXM_HIP(n, hipMemcpyAsync(params, n->p, sizeof(float) * sxm::NPARAM, hipMemcpyDeviceToHost, n->stream));
    SXM_HIP(n, hipStreamSynchronize(n->stream));
    return SX_OK;
}

int sx_mlp_gradients(sx_mlp *n, const float *x, const float *t, size_t rows, float *grads, float *loss) {
    if (!n) return SX_ERR_ARG;
    int rc = check_rows(n, x, rows);
    if (rc != SX_OK) return rc;
    if (!t || !grads) return mfail(n, SX_ERR_ARG, "null targets or gradient buffer");
    SXM_HIP(n, hipSetDevice(n->device));
    rc = ensure_rows(n, rows);
    if (rc != SX_OK) return rc;
    SXM_HIP(n, hipMemcpyAsync(n->x, x, sizeof(float) * sxm::IN * rows, hipMemcpyHostToDevice, n->stream));
    SXM_HIP(n, hipMemcpyAsync(n->t, t, sizeof(float) * rows, hipMemcpyHostToDevice, n->stream));
    rc = step(n, (unsigned)rows, (unsigned)rows, 0, 0, 0, true, 0, 0.f);
    if (rc != SX_OK) return rc;
    SXM_HIP(n, hipMemcpyAsync(grads, n->grad, sizeof(float) * sxm::NPARAM, hipMemcpyDeviceToHost, n->stream));
    float l = 0.f;
    SXM_HIP(n, hipMemcpyAsync(&l, n->loss, sizeof(float), hipMemcpyDeviceToHost, n->stream));
    SXM_HIP(n, hipStreamSynchronize(n->stream));
    if (loss) *loss = l / (float)rows;
    return SX_OK;
}

int sx_mlp_train(sx_mlp *n, const float *x, const float *t, size_t rows, int steps, int batch, float lr,
                 unsigned long long seed, float *final_loss) {
    if (!n) return SX_ERR_ARG;
    int rc = check_rows(n, x, rows);
    if (rc != SX_OK) return rc;
    if (!t || steps <= 0 || batch <= 0 || batch > (1 << 20) || !(lr > 0.f))
        return mfail(n, SX_ERR_ARG, "bad training arguments");
    SXM_HIP(n, hipSetDevice(n->device));
    rc = ensure_rows(n, rows);
    if (rc != SX_OK) return rc;
    SXM_HIP(n, hipMemcpyAsync(n->x, x, sizeof(float) * sxm::IN * rows, hipMemcpyHostToDevice, n->stream));
    SXM_HIP(n, hipMemcpyAsync(n->t, t, sizeof(float) * rows, hipMemcpyHostToDevice, n->stream));
    for (int s = 0; s < steps; ++s) {
        // cosine decay to 5 % of the initial rate
        const float lrs = lr * (0.05f + 0.95f * 0.5f * (1.f + cosf(3.14159265f * (float)s / (float)steps)));
        rc = step(n, (unsigned)rows, (unsigned)batch, 1, seed, (unsigned)s, true, 1, lrs);
        if (rc != SX_OK) return rc;
    }
    float l = 0.f;
    SXM_HIP(n, hipMemcpyAsync(&l, n->loss, sizeof(float), hipMemcpyDeviceToHost, n->stream));
    SXM_HIP(n, hipStreamSynchronize(n->stream));
    if (final_loss) *final_loss = l / (float)batch;
    return SX_OK;
}

int sx_mlp_predict(sx_mlp *n, const float *x, size_t rows, float *y) {
    if (!n) return SX_ERR_ARG;
    int rc = check_rows(n, x, rows);
    if (rc != SX_OK) return rc;
    if (!y) return mfail(n, SX_ERR_ARG, "null output");
    SXM_HIP(n, hipSetDevice(n->device));
    rc = ensure_rows(n, rows);
    if (rc != SX_OK) return rc;
    SXM_HIP(n, hipMemcpyAsync(n->x, x, sizeof(float) * sxm::IN * rows, hipMemcpyHostToDevice, n->stream));
    rc = step(n, (unsigned)rows, (unsigned)rows, 0, 0, 0, false, 0, 0.f);
    if (rc != SX_OK) return rc;
    SXM_HIP(n, hipMemcpyAsync(y, n->y, sizeof(float) * rows, hipMemcpyDeviceToHost, n->stream));
    SXM_HIP(n, hipStreamSynchronize(n->stream));
    return SX_OK;
}

}  // extern "C"
