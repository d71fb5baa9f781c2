// hfem_mlp: learned constitutive surrogate for MisesMat.
//
// Network: 13 inputs -> 3 x 128 hidden (SiLU) -> 27 outputs, FP32 master
// weights in one flat buffer (W1 128x13, b1, W2 128x128, b2, W3 128x128, b3,
// W4 27x128, b4; row = output unit).
//   inputs  (eps_{n+1} - epsp_n) (6), epsp_n (6), kappa_n (1); the return
//           map of misesmat.C:181-263 depends on the strain only through
//           eps_{n+1} - epsp_n, so this difference is the strain input;
//           all scaled by E / sig0 (the yield strain is 1)
//   outputs sigma_{n+1} (6) and the upper triangle of the consistent
//           tangent (21, row-major), each as its departure from the elastic
//           trial: o_sigma = (D_e (eps - epsp_n) - sigma) / sig0 and
//           o_D = (D_e - D) / E, so both vanish on the elastic branch and the
//           network learns only the plastic correction
// Training data: random strain paths driven through the plain return
// mapping (mises_return / mises_tangent, the device form of MisesMat):
// each path starts virgin and takes 1..maxsteps Gaussian increments of
// every Voigt strain component; every step is one sample.
// Training: mean-squared error over the 27 scaled outputs, Adam, batches
// drawn with replacement by a counter-based hash; three FP32 launches a step.
// Inference: BF16 operands on MFMA (v_mfma_f32_32x32x16_bf16) with FP32
// accumulation, weights staged in LDS in operand order.

#include <algorithm>
#include <cmath>
#include <cstring>
#include <vector>

#include "hipfem_internal.h"
#include "hipfem_material.h"

namespace hipfem {

constexpr int MLP_IN = 13, MLP_H = 128, MLP_OUT = 27;
constexpr int OFF_W1 = 0;
constexpr int OFF_B1 = OFF_W1 + MLP_H * MLP_IN;
constexpr int OFF_W2 = OFF_B1 + MLP_H;
constexpr int OFF_B2 = OFF_W2 + MLP_H * MLP_H;
constexpr int OFF_W3 = OFF_B2 + MLP_H;
constexpr int OFF_B3 = OFF_W3 + MLP_H * MLP_H;
constexpr int OFF_W4 = OFF_B3 + MLP_H;
constexpr int OFF_B4 = OFF_W4 + MLP_OUT * MLP_H;
constexpr int MLP_NPARAM = OFF_B4 + MLP_OUT;
constexpr int MLP_SLABS = 64;   // most weight-gradient slabs of a batch

// --------------------------------------------------------------- hashing RNG
__host__ __device__ inline uint64_t mix64(uint64_t x)
{
    x += 0x9E3779B97F4A7C15ull;
    x = (x ^ (x >> 30)) * 0xBF58476D1CE4E5B9ull;
    x = (x ^ (x >> 27)) * 0x94D049BB133111EBull;
    return x ^ (x >> 31);
}

__host__ __device__ inline double unit_open(uint64_t h) { return ((double)(h >> 11) + 0.5) * (1.0 / 9007199254740992.0); }

__host__ __device__ inline int path_length(uint64_t seed, int64_t p, int maxsteps)
{
    return 1 + (int)(mix64(seed ^ (0xD1B54A32D192ED03ull * (uint64_t)(p + 1))) % (uint64_t)maxsteps);
}

// --------------------------------------------------------- training samples
__global__ void k_mlp_paths(int64_t npaths, const int64_t *__restrict__ off, int64_t nsamples, uint64_t seed,
                            double E, double nu, double sig0, double H, double stdev, float in_scale,
                            float sig_scale, float tan_scale, float *__restrict__ X, float *__restrict__ Y)
{
    const int64_t p = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
    if (p >= npaths) return;
    const int64_t o = off[p], L = off[p + 1] - o;
    double eps[6] = {0, 0, 0, 0, 0, 0}, epsp[6] = {0, 0, 0, 0, 0, 0}, kappa = 0.0;
    uint64_t ctr = mix64(seed * 0x632BE59BD9B4E019ull + (uint64_t)p);
    for (int64_t s = 0; s < L && o + s < nsamples; s++) {
#pragma unroll
        for (int i = 0; i < 6; i += 2) {   // Box-Muller pairs
            const uint64_t h1 = mix64(ctr++), h2 = mix64(ctr++);
            const double r = sqrt(-2.0 * log(unit_open(h1))), t = 6.283185307179586 * unit_open(h2);
            eps[i] += stdev * r * cos(t);
            eps[i + 1] += stdev * r * sin(t);
        }
        MisesOut m;
        mises_return(E, nu, sig0, H, eps, epsp, kappa, m);
        double D[36];
        mises_tangent(E, nu, sig0, H, kappa, m.kappa, m.sdev, D);
        float *x = X + (o + s) * MLP_IN;
        float *y = Y + (o + s) * MLP_OUT;
        double el[6], st[6];
#pragma unroll
        for (int i = 0; i < 6; i++) el[i] = eps[i] - epsp[i];
        elastic_trial(E, nu, el, st);
#pragma unroll
        for (int i = 0; i < 6; i++) {
            x[i] = (float)(el[i] * in_scale);
            x[6 + i] = (float)(epsp[i] * in_scale);
            y[i] = (float)((st[i] - m.sig[i]) * sig_scale);
        }
        x[12] = (float)(kappa * in_scale);
        int k = 0;
        for (int r = 0; r < 6; r++)
            for (int c = r; c < 6; c++, k++) y[6 + k] = (float)((elastic_upper(E, nu, k) - D[6 * r + c]) * tan_scale);
#pragma unroll
        for (int i = 0; i < 6; i++) epsp[i] = m.epsp[i];
        kappa = m.kappa;
    }
}

// ------------------------------------------------------------- FP32 kernels
// A training step is three launches: k_mlp_step (forward and backward of the
// batch, 16 rows a workgroup), k_mlp_wgrad (weight-gradient slabs over the
// rows) and k_mlp_apply (slabs summed, Adam).  All products run on the FP32
// matrix instructions (FP32 operands and accumulation).
//
// Besides the parameters the device holds copies that the products can read
// along their contiguous dimension: W1 padded to 16 columns, and W2, W3, W4
// transposed (W4's rows padded to 32).
constexpr int AUX_W1 = 0;                        // 128 x 16
constexpr int AUX_T2 = AUX_W1 + MLP_H * 16;      // 128 x 128: [in][out]
constexpr int AUX_T3 = AUX_T2 + MLP_H * MLP_H;
constexpr int AUX_T4 = AUX_T3 + MLP_H * MLP_H;   // 128 x 32: [in][out]
constexpr int MLP_NAUX = AUX_T4 + MLP_H * 32;

// where parameter i has a copy (-1: a bias)
__device__ __forceinline__ int aux_of(int i)
{
    if (i < OFF_B1) return AUX_W1 + (i / MLP_IN) * 16 + i % MLP_IN;
    if (i >= OFF_W2 && i < OFF_B2) return AUX_T2 + (i - OFF_W2) % MLP_H * MLP_H + (i - OFF_W2) / MLP_H;
    if (i >= OFF_W3 && i < OFF_B3) return AUX_T3 + (i - OFF_W3) % MLP_H * MLP_H + (i - OFF_W3) / MLP_H;
    if (i >= OFF_W4 && i < OFF_B4) return AUX_T4 + (i - OFF_W4) % MLP_H * 32 + (i - OFF_W4) / MLP_H;
    return -1;
}

__global__ void k_mlp_aux(const float *__restrict__ p, float *__restrict__ aux)
{
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= MLP_NPARAM) return;
    const int j = aux_of(i);
    if (j >= 0) aux[j] = p[i];
}

typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef float f32x16 __attribute__((__vector_size__(16 * sizeof(float))));

__device__ __forceinline__ float sigmoidf_(float z) { return 1.f / (1.f + expf(-z)); }

constexpr int TR = 16;            // batch rows per workgroup of k_mlp_step
constexpr int TLD = MLP_H + 4;    // LDS row of an activation tile

// acc += A (16 rows in LDS, row stride TLD) times the 16 columns whose
// operand rows b holds: lane (c, q) of b is the row of column c, entries
// [4 NV q, 4 NV (q + 1)); the four lane groups take the four quarters of the
// inner dimension, so both operands are read 16 bytes at a time
template <int NV>
__device__ __forceinline__ f32x4 tile_product(const float *sA, const f32x4 b[NV], int c, int q, f32x4 acc)
{
#pragma unroll
    for (int v = 0; v < NV; v++) {
        const f32x4 a = *reinterpret_cast<const f32x4 *>(sA + c * TLD + 4 * NV * q + 4 * v);
#pragma unroll
        for (int i = 0; i < 4; i++) acc = __builtin_amdgcn_mfma_f32_16x16x4f32(a[i], b[v][i], acc, 0, 0, 0);
    }
    return acc;
}

template <int NV>
__device__ __forceinline__ void load_operand(const float *__restrict__ row, int q, f32x4 b[NV])
{
#pragma unroll
    for (int v = 0; v < NV; v++) b[v] = *reinterpret_cast<const f32x4 *>(row + 4 * NV * q + 4 * v);
}

// what a step reads and writes; row r of the batch is sample
// hash(seed, step, r) mod nsamples (drawn with replacement), or row r of X, Y
struct StepArgs {
    int B;
    const float *X, *Y;
    int64_t nsamples;      // 0: rows as they lie
    uint64_t seed;
    int64_t step;
    const float *p, *aux;
    float scale;           // 1 / (27 B)
    float *xb;             // B16 x 16 inputs
    float *h;              // 3 x B16 x 128 activations
    float *dz;             // 3 x B16 x 128 gradients before the activation
    float *dy;             // B16 x 32 output gradients
    float *yp;             // predictions (forward only), B x 27
    double *loss;          // per workgroup: sum of squared errors
};

// Forward (and, BWD, backward) of 16 rows: eight waves, wave w owns units
// 16 w .. 16 w + 15 of every hidden layer.  Activations pass through LDS; the
// derivative of SiLU stays in the registers of the lane that meets the same
// (row, unit) again on the way back.  Each layer's weights are loaded before
// the barrier that ends the layer before it.
//
// Bound: the chain of seven dependent products, each 32 matrix instructions
// a wave and its weights from L2: 21 us for 4,096 rows (256 workgroups).  With
// one launch a product (64 x 64 tiles on the vector units, 64 to 128 workgroups)
// and one for each elementwise pass a training step took 503 us; it takes 46.
template <bool BWD>
__global__ __launch_bounds__(512) void k_mlp_step(StepArgs A)
{
    __shared__ __align__(16) float sA[2][TR * TLD];
    __shared__ double sL[8];
    const int t = threadIdx.x, w = t >> 6, l = t & 63, c = l & 15, q = l >> 4;
    const int r0 = blockIdx.x * TR, B16 = gridDim.x * TR, u = 16 * w + c;
    const float *P = A.p;
    f32x4 b1[1], b[8];
    load_operand<1>(A.aux + AUX_W1 + u * 16, q, b1);
    load_operand<8>(P + OFF_W2 + u * MLP_H, q, b);
    auto sample = [&](int r) -> int64_t {
        r = min(r, A.B - 1);   // the rows past the batch repeat its last one, with no gradient
        if (!A.nsamples) return r;
        return (int64_t)(mix64(A.seed ^ mix64((uint64_t)A.step * 0x9E3779B97F4A7C15ull + (uint64_t)r)) %
                         (uint64_t)A.nsamples);
    };
    if (t < TR * 16) {
        const int r = t >> 4, k = t & 15;
        const float x = k < MLP_IN ? A.X[sample(r0 + r) * MLP_IN + k] : 0.f;
        sA[0][r * TLD + k] = x;
        if constexpr (BWD) A.xb[(size_t)(r0 + r) * 16 + k] = x;
    }
    __syncthreads();
    float dsilu[3][4];
    f32x4 acc;
#pragma unroll
    for (int L = 0; L < 3; L++) {
        const f32x4 zero = {0.f, 0.f, 0.f, 0.f};
        if (L == 0)
            acc = tile_product<1>(sA[0], b1, c, q, zero);
        else
            acc = tile_product<8>(sA[L & 1], b, c, q, zero);
        if (L == 1) load_operand<8>(P + OFF_W3 + u * MLP_H, q, b);
        if (L == 2) load_operand<8>(P + OFF_W4 + min(u, MLP_OUT - 1) * MLP_H, q, b);
        const float bias = P[(L == 0 ? OFF_B1 : L == 1 ? OFF_B2 : OFF_B3) + u];
#pragma unroll
        for (int i = 0; i < 4; i++) {
            const float z = acc[i] + bias, s = sigmoidf_(z), h = z * s;
            dsilu[L][i] = s * (1.f + z * (1.f - s));
            sA[(L + 1) & 1][(4 * q + i) * TLD + u] = h;
            if constexpr (BWD) A.h[((size_t)L * B16 + r0 + 4 * q + i) * MLP_H + u] = h;
        }
        __syncthreads();
    }
    // output layer on the first two waves: 27 of 32 columns
    double loss = 0.0;
    if (w < 2) {
        acc = tile_product<8>(sA[1], b, c, q, f32x4{0.f, 0.f, 0.f, 0.f});
        const float bias = u < MLP_OUT ? P[OFF_B4 + u] : 0.f;
#pragma unroll
        for (int i = 0; i < 4; i++) {
            const int r = r0 + 4 * q + i;
            const bool live = r < A.B && u < MLP_OUT;
            const float y = acc[i] + bias;
            if constexpr (BWD) {
                const float d = live ? y - A.Y[sample(r) * MLP_OUT + u] : 0.f;
                const float dy = 2.f * A.scale * d;
                loss += (double)d * (double)d;
                sA[0][(4 * q + i) * TLD + u] = dy;
                A.dy[(size_t)r * 32 + u] = dy;
            } else {
                if (live) A.yp[(size_t)r * MLP_OUT + u] = y;
            }
        }
    }
    if constexpr (!BWD) return;
    f32x4 b4[2];
    load_operand<2>(A.aux + AUX_T4 + u * 32, q, b4);
    load_operand<8>(A.aux + AUX_T3 + u * MLP_H, q, b);
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) loss += __shfl_xor(loss, off, 64);
    if (l == 0) sL[w] = loss;
    __syncthreads();
    if (t == 0) A.loss[blockIdx.x] = sL[0] + sL[1];
#pragma unroll
    for (int L = 2; L >= 0; L--) {
        const f32x4 zero = {0.f, 0.f, 0.f, 0.f};
        if (L == 2)
            acc = tile_product<2>(sA[0], b4, c, q, zero);
        else
            acc = tile_product<8>(sA[L & 1 ? 1 : 0], b, c, q, zero);
        if (L == 1) load_operand<8>(A.aux + AUX_T2 + u * MLP_H, q, b);
#pragma unroll
        for (int i = 0; i < 4; i++) {
            const float d = acc[i] * dsilu[L][i];
            if (L) sA[L & 1 ? 0 : 1][(4 * q + i) * TLD + u] = d;
            A.dz[((size_t)L * B16 + r0 + 4 * q + i) * MLP_H + u] = d;
        }
        if (L) __syncthreads();
    }
}

// acc (32 x 32 tiles NM x NN) += sum over rows [k0, k1) of a[k][m] b[k][n]
// (row strides lda, ldb; a multiple of 8 rows); lanes 32..63 take the odd rows.
// csum: the sums of a's columns (the bias gradient), in four running sums a
// lane against the rounding of one long one, and over the two lanes of a column.
template <int NM, int NN>
__device__ __forceinline__ void rank_update(const float *__restrict__ a, int lda, const float *__restrict__ b, int ldb,
                                            int k0, int k1, int l, f32x16 acc[NM][NN], float csum[NM])
{
    const int m = l & 31;
    float cs[NM][4] = {};
#pragma unroll 2
    for (int k = k0 + (l >> 5); k < k1; k += 8) {
#pragma unroll
        for (int u = 0; u < 4; u++) {
            const int r = k + 2 * u;
            float x[NM], y[NN];
#pragma unroll
            for (int i = 0; i < NM; i++) x[i] = a[(size_t)r * lda + 32 * i + m];
#pragma unroll
            for (int j = 0; j < NN; j++) y[j] = b[(size_t)r * ldb + 32 * j + (ldb < 32 ? m & (ldb - 1) : m)];
#pragma unroll
            for (int i = 0; i < NM; i++) {
                cs[i][u] += x[i];
#pragma unroll
                for (int j = 0; j < NN; j++)
                    acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x2f32(x[i], y[j], acc[i][j], 0, 0, 0);
            }
        }
    }
#pragma unroll
    for (int i = 0; i < NM; i++) {
        csum[i] = (cs[i][0] + cs[i][1]) + (cs[i][2] + cs[i][3]);
        csum[i] += __shfl_xor(csum[i], 32, 64);
    }
}

// row of value r of lane l in a 32 x 32 tile (column l % 32)
__device__ __forceinline__ int tile_row(int l, int r) { return 8 * (r >> 2) + 4 * (l >> 5) + (r & 3); }

template <int NM, int NN>
__device__ __forceinline__ void store_tiles(const f32x16 acc[NM][NN], int l, float *__restrict__ out, int m0, int mmax,
                                            int n0, int nmax)
{
#pragma unroll
    for (int i = 0; i < NM; i++)
#pragma unroll
        for (int j = 0; j < NN; j++)
#pragma unroll
            for (int r = 0; r < 16; r++) {
                const int m = m0 + 32 * i + tile_row(l, r), n = n0 + 32 * j + (l & 31);
                if (m < mmax && n < nmax) out[m * nmax + n] = acc[i][j][r];
            }
}

// Gradient slab z of the parameters: sums over rows [rows z, rows (z + 1)) of
// dZ_L^T H_{L-1} and of dZ_L.  Blocks (0, z) and (1, z): layers 2 and 3, a
// 64 x 64 quarter a wave; block (2, z): layer 1 (32 units a wave) and the
// output layer (32 inputs a wave).
//
// Bound: the latency of the row loads (70 % of the waves' time is waiting, the
// vector units issue in 7 % of the cycles), eight pairs of rows in flight: 19 us
// for 4,096 rows in 64 slabs.
__global__ __launch_bounds__(256) void k_mlp_wgrad(int B16, int rows, const float *__restrict__ xb,
                                                   const float *__restrict__ h, const float *__restrict__ dz,
                                                   const float *__restrict__ dy, float *__restrict__ slabs)
{
    const int w = threadIdx.x >> 6, l = threadIdx.x & 63, z = blockIdx.y;
    const int k0 = z * rows, k1 = min(B16, k0 + rows);
    float *out = slabs + (size_t)z * MLP_NPARAM;
    const size_t layer = (size_t)B16 * MLP_H;
    if (blockIdx.x < 2) {
        const int L = blockIdx.x + 1, m0 = 64 * (w >> 1), n0 = 64 * (w & 1);
        f32x16 acc[2][2] = {};
        float cs[2];
        rank_update<2, 2>(dz + L * layer + m0, MLP_H, h + (L - 1) * layer + n0, MLP_H, k0, k1, l, acc, cs);
        store_tiles<2, 2>(acc, l, out + (L == 1 ? OFF_W2 : OFF_W3), m0, MLP_H, n0, MLP_H);
#pragma unroll
        for (int i = 0; i < 2; i++) {
            if (n0 == 0 && l < 32) out[(L == 1 ? OFF_B2 : OFF_B3) + m0 + 32 * i + l] = cs[i];
        }
    } else {
        f32x16 acc[1][1] = {};
        float cs[1];
        // 16 input columns: the tile's upper half repeats them, and is not stored
        rank_update<1, 1>(dz + 32 * w, MLP_H, xb, 16, k0, k1, l, acc, cs);
        store_tiles<1, 1>(acc, l, out + OFF_W1, 32 * w, MLP_H, 0, MLP_IN);
        if (l < 32) out[OFF_B1 + 32 * w + l] = cs[0];
        f32x16 acc4[1][1] = {};
        rank_update<1, 1>(dy, 32, h + 2 * layer + 32 * w, MLP_H, k0, k1, l, acc4, cs);
        // the tile's columns are inputs 32 w ..: rows of W4 are 128 long
#pragma unroll
        for (int r = 0; r < 16; r++) {
            const int u = tile_row(l, r);
            if (u < MLP_OUT) out[OFF_W4 + u * MLP_H + 32 * w + (l & 31)] = acc4[0][0][r];
        }
        if (w == 0 && l < MLP_OUT) out[OFF_B4 + l] = cs[0];
    }
}

// g = sum of the S slabs (in order), and with adam the Adam update of the
// parameters and their copies; block 0 also sums the loss partials.  Sixteen
// slabs at a time are summed pairwise: with 64 of them added one after the
// other the sums round a bias gradient of 4,096 rows to 1.2e-7 of itself, so to
// 4.5e-8 (FP64 sums: 3e-8, but 20 % on the training step).
__global__ __launch_bounds__(256) void k_mlp_apply(int S, const float *__restrict__ slabs, int nloss,
                                                   const double *__restrict__ lossp, double lscale,
                                                   double *__restrict__ loss, float *__restrict__ g,
                                                   float *__restrict__ p, float *__restrict__ aux,
                                                   float *__restrict__ m, float *__restrict__ v, int adam, float lr, float b1,
                                                   float b2, float eps, float bc1, float bc2)
{
    const int i = blockIdx.x * 256 + threadIdx.x;
    if (i < MLP_NPARAM) {
        float s = 0.f;
        for (int z0 = 0; z0 < S; z0 += 16) {
            float x[16];
#pragma unroll
            for (int j = 0; j < 16; j++) x[j] = z0 + j < S ? slabs[(size_t)(z0 + j) * MLP_NPARAM + i] : 0.f;
#pragma unroll
            for (int w = 8; w > 0; w >>= 1)
#pragma unroll
                for (int j = 0; j < w; j++) x[j] += x[j + w];
            s += x[0];
        }
        g[i] = s;
        if (adam) {
            const float mi = b1 * m[i] + (1.f - b1) * s;
            const float vi = b2 * v[i] + (1.f - b2) * s * s;
            m[i] = mi;
            v[i] = vi;
            const float pi = p[i] - lr * (mi / bc1) / (sqrtf(vi / bc2) + eps);
            p[i] = pi;
            const int j = aux_of(i);
            if (j >= 0) aux[j] = pi;
        }
    }
    if (blockIdx.x != 0) return;
    __shared__ double sh[4];
    double s = 0.0;
    for (int k = threadIdx.x; k < nloss; k += 256) s += lossp[k];
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) s += __shfl_xor(s, off, 64);
    if (threadIdx.x % 64 == 0) sh[threadIdx.x / 64] = s;
    __syncthreads();
    if (threadIdx.x == 0) *loss = (sh[0] + sh[1] + sh[2] + sh[3]) * lscale;
}

// --------------------------------------------------------- BF16 inference
typedef __bf16 bf16x8 __attribute__((__vector_size__(8 * sizeof(__bf16))));

__host__ __device__ inline uint16_t f2bf(float f)
{
    uint32_t u;
    memcpy(&u, &f, 4);
    u += 0x7FFFu + ((u >> 16) & 1u);   // round to nearest even (finite inputs)
    return (uint16_t)(u >> 16);
}

// operand-order weight blocks: layer (KS k-steps of 16, NT n-tiles of 32);
// block (nt, ks) holds 64 lanes x 8 values: lane l -> output j = 32 nt + l%32,
// inputs k = 16 ks + 8 (l/32) + v
constexpr int BF_L1 = 4 * 1 * 512, BF_L2 = 4 * 8 * 512, BF_L3 = 4 * 8 * 512, BF_L4 = 1 * 8 * 512;
constexpr int BF_TOTAL = BF_L1 + BF_L2 + BF_L3 + BF_L4;   // bf16 values (76 KiB)
constexpr int ACT_LD = MLP_H + 8;                          // padded LDS row (bf16)

__device__ __forceinline__ float bf2f(uint16_t b)
{
    uint32_t u = (uint32_t)b << 16;
    float f;
    memcpy(&f, &u, 4);
    return f;
}

// z silu(z) = z / (1 + e^-z) with the hardware exp2 and reciprocal (the
// result is rounded to BF16, 8 bits, right after), then to BF16 by
// v_cvt_pk_bf16_f32 (round to nearest even, as f2bf)
__device__ __forceinline__ uint16_t silu_bf16(float z)
{
    const float h = z * __builtin_amdgcn_rcpf(1.f + __builtin_amdgcn_exp2f(-1.4426950408889634f * z));
    const __bf16 b = (__bf16)h;
    uint16_t u;
    memcpy(&u, &b, 2);
    return u;
}

constexpr int BF_WAVES = 8;   // waves per workgroup sharing the LDS weights

__global__ __launch_bounds__(64 * BF_WAVES) void k_mlp_bf16(int n, const float *__restrict__ X,
                                                             float *__restrict__ Y, const uint16_t *__restrict__ wpk,
                                                             const float *__restrict__ params)
{
    extern __shared__ uint16_t lds[];
    uint16_t *sW = lds;                                   // BF_TOTAL
    uint16_t *sA = lds + BF_TOTAL;                        // BF_WAVES waves x 32 x ACT_LD
    for (int i = threadIdx.x; i < BF_TOTAL / 8; i += 64 * BF_WAVES)
        reinterpret_cast<uint4 *>(sW)[i] = reinterpret_cast<const uint4 *>(wpk)[i];
    const int wv = threadIdx.x >> 6, l = threadIdx.x & 63;
    uint16_t *act = sA + wv * 32 * ACT_LD;
    const uint16_t *W1 = sW, *W2 = sW + BF_L1, *W3 = W2 + BF_L2, *W4 = W3 + BF_L3;
    const int ntile = (n + 31) / 32;
    __syncthreads();
    for (int base = blockIdx.x * BF_WAVES; base < ntile; base += gridDim.x * BF_WAVES) {
        const int tile = base + wv;
        const int row0 = tile * 32;
        // layer 1: A operand straight from X (13 inputs, zero padded to 16)
        bf16x8 a;
        {
            const int i = row0 + (l & 31);
            uint16_t v8[8];
#pragma unroll
            for (int v = 0; v < 8; v++) {
                const int k = 8 * (l >> 5) + v;
                v8[v] = (i < n && k < MLP_IN) ? f2bf(X[(int64_t)i * MLP_IN + k]) : (uint16_t)0;
            }
            memcpy(&a, v8, 16);
        }
        f32x16 acc[4];
#pragma unroll
        for (int nt = 0; nt < 4; nt++) {
            acc[nt] = (f32x16){0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0};
            const bf16x8 b = *reinterpret_cast<const bf16x8 *>(W1 + (nt * 64 + l) * 8);
            acc[nt] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b, acc[nt], 0, 0, 0);
        }
        // hidden layers: bias + SiLU into LDS, read back as the next A operand
        for (int layer = 0; layer < 3; layer++) {
            const float *bias = params + (layer == 0 ? OFF_B1 : layer == 1 ? OFF_B2 : OFF_B3);
#pragma unroll
            for (int nt = 0; nt < 4; nt++) {
                const int j = nt * 32 + (l & 31);
                const float bj = bias[j];
#pragma unroll
                for (int r = 0; r < 16; r++) act[tile_row(l, r) * ACT_LD + j] = silu_bf16(acc[nt][r] + bj);
            }
            wave_lds_fence();   // the activation tile is the wave's own
            const uint16_t *Wn = layer == 0 ? W2 : layer == 1 ? W3 : W4;
#pragma unroll
            for (int nt = 0; nt < 4; nt++) acc[nt] = (f32x16){0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0};
            if (layer < 2) {
#pragma unroll
                for (int ks = 0; ks < 8; ks++) {
                    const bf16x8 av =
                        *reinterpret_cast<const bf16x8 *>(act + (l & 31) * ACT_LD + ks * 16 + 8 * (l >> 5));
#pragma unroll
                    for (int nt = 0; nt < 4; nt++) {
                        const bf16x8 b = *reinterpret_cast<const bf16x8 *>(Wn + ((nt * 8 + ks) * 64 + l) * 8);
                        acc[nt] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(av, b, acc[nt], 0, 0, 0);
                    }
                }
            } else {
#pragma unroll
                for (int ks = 0; ks < 8; ks++) {
                    const bf16x8 av =
                        *reinterpret_cast<const bf16x8 *>(act + (l & 31) * ACT_LD + ks * 16 + 8 * (l >> 5));
                    const bf16x8 b = *reinterpret_cast<const bf16x8 *>(Wn + (ks * 64 + l) * 8);
                    acc[0] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(av, b, acc[0], 0, 0, 0);
                }
            }
            wave_lds_fence();   // the activation tile is the wave's own
        }
        // output layer: 27 of 32 columns
        const int j = l & 31;
        if (j < MLP_OUT) {
            const float bj = params[OFF_B4 + j];
#pragma unroll
            for (int r = 0; r < 16; r++) {
                const int i = row0 + tile_row(l, r);
                if (i < n) Y[(int64_t)i * MLP_OUT + j] = acc[0][r] + bj;
            }
        }
    }
}

// pack W (out x in, FP32) of one layer into operand-order BF16 blocks
__global__ void k_pack_bf16(const float *__restrict__ W, int nout, int nin, int NT, int KS, uint16_t *__restrict__ out)
{
    const int idx = blockIdx.x * blockDim.x + threadIdx.x;
    if (idx >= NT * KS * 512) return;
    const int v = idx & 7, l = (idx >> 3) & 63, blk = idx >> 9;
    const int nt = blk / KS, ks = blk % KS;
    const int j = nt * 32 + (l & 31), k = ks * 16 + 8 * (l >> 5) + v;
    out[idx] = (j < nout && k < nin) ? f2bf(W[j * nin + k]) : (uint16_t)0;
}

}  // namespace hipfem

using namespace hipfem;

struct hfem_mlp {
    hipfem_ctx *ctx = nullptr;
    double E = 0, nu = 0, sig0 = 0, H = 0;
    float in_scale = 1, sig_scale = 1, tan_scale = 1;
    float *d_p = nullptr, *d_g = nullptr, *d_m = nullptr, *d_v = nullptr;
    int64_t adam_t = 0;
    // training set
    int64_t nsamples = 0;
    float *d_X = nullptr, *d_Y = nullptr;
    // copies of the weights that the FP32 products read (valid when
    // aux_version == param_version)
    float *d_aux = nullptr;
    long aux_version = -1;
    // work buffers for batches of up to cap rows (a multiple of TR)
    int cap = 0;
    float *d_xb = nullptr, *d_h = nullptr, *d_dz = nullptr, *d_dy = nullptr;
    double *d_lossp = nullptr;   // per workgroup
    float *d_ws = nullptr;       // gradient slabs
    // host-array rows and predictions of hfem_mlp_forward / _gradients
    int io_cap = 0;
    float *d_ix = nullptr, *d_iy = nullptr;
    double *d_loss = nullptr;
    // BF16 operand-order weights (valid when packed_version == param_version)
    uint16_t *d_wpk = nullptr;
    long param_version = 0, packed_version = -1;
};

static int mlp_ensure_batch(hfem_mlp *m, int B)
{
    if (B <= m->cap) return 0;
    HIPFEM_CHECK(hipStreamSynchronize(m->ctx->stream));   // a step may still use the buffers
    void *ps[] = {m->d_xb, m->d_h, m->d_dz, m->d_dy, m->d_lossp};
    m->d_xb = m->d_h = m->d_dz = m->d_dy = nullptr;
    m->d_lossp = nullptr;
    m->cap = 0;
    for (void *p : ps)
        if (p) HIPFEM_CHECK(hipFree(p));
    const size_t b = ((size_t)B + TR - 1) / TR * TR;
    HIPFEM_REQUIRE(b <= INT32_MAX, HIPFEM_ETOOBIG, "batch of %d rows too large", B);
    HIPFEM_CHECK(hipMalloc(&m->d_xb, sizeof(float) * b * 16));
    HIPFEM_CHECK(hipMalloc(&m->d_h, sizeof(float) * b * 3 * MLP_H));
    HIPFEM_CHECK(hipMalloc(&m->d_dz, sizeof(float) * b * 3 * MLP_H));
    HIPFEM_CHECK(hipMalloc(&m->d_dy, sizeof(float) * b * 32));
    HIPFEM_CHECK(hipMalloc(&m->d_lossp, sizeof(double) * (b / TR)));
    if (!m->d_ws) HIPFEM_CHECK(hipMalloc(&m->d_ws, sizeof(float) * (size_t)MLP_SLABS * MLP_NPARAM));
    m->cap = (int)b;
    return 0;
}

// device buffers for n host rows (inputs, targets or predictions)
static int mlp_ensure_io(hfem_mlp *m, int n)
{
    if (n <= m->io_cap) return 0;
    void *ps[] = {m->d_ix, m->d_iy};
    m->d_ix = m->d_iy = nullptr;
    m->io_cap = 0;
    for (void *p : ps)
        if (p) HIPFEM_CHECK(hipFree(p));
    HIPFEM_CHECK(hipMalloc(&m->d_ix, sizeof(float) * (size_t)n * MLP_IN));
    HIPFEM_CHECK(hipMalloc(&m->d_iy, sizeof(float) * (size_t)n * MLP_OUT));
    m->io_cap = n;
    return 0;
}

// the weight copies of the current parameters
static int mlp_ensure_aux(hfem_mlp *m)
{
    if (m->d_aux && m->aux_version == m->param_version) return 0;
    hipStream_t s = m->ctx->stream;
    if (!m->d_aux) {
        HIPFEM_CHECK(hipMalloc(&m->d_aux, sizeof(float) * MLP_NAUX));
        k_zero_f32<<<(MLP_NAUX + 255) / 256, 256, 0, s>>>(MLP_NAUX, m->d_aux);
    }
    k_mlp_aux<<<(MLP_NPARAM + 255) / 256, 256, 0, s>>>(m->d_p, m->d_aux);
    HIPFEM_CHECK(hipGetLastError());
    m->aux_version = m->param_version;
    return 0;
}

// forward, backward and gradients of the B rows that a names into d_g, loss
// into d_loss; with adam the Adam update (bias corrections bc1, bc2)
static int mlp_step(hfem_mlp *m, StepArgs a, bool adam, float lr, float bc1, float bc2)
{
    hipStream_t s = m->ctx->stream;
    const int nwg = (a.B + TR - 1) / TR, B16 = nwg * TR;
    a.p = m->d_p;
    a.aux = m->d_aux;
    a.scale = 1.f / (float)((int64_t)a.B * MLP_OUT);
    a.xb = m->d_xb;
    a.h = m->d_h;
    a.dz = m->d_dz;
    a.dy = m->d_dy;
    a.yp = nullptr;
    a.loss = m->d_lossp;
    k_mlp_step<true><<<nwg, 512, 0, s>>>(a);
    // slabs of at least 64 rows, a multiple of 8 each (rank_update)
    const int rows = std::max(64, ((B16 + MLP_SLABS - 1) / MLP_SLABS + 7) / 8 * 8), S = (B16 + rows - 1) / rows;
    k_mlp_wgrad<<<dim3(3, S), 256, 0, s>>>(B16, rows, m->d_xb, m->d_h, m->d_dz, m->d_dy, m->d_ws);
    k_mlp_apply<<<(MLP_NPARAM + 255) / 256, 256, 0, s>>>(S, m->d_ws, nwg, m->d_lossp,
                                                         1.0 / (double)((int64_t)a.B * MLP_OUT), m->d_loss, m->d_g,
                                                         m->d_p, m->d_aux, m->d_m, m->d_v, adam, lr, 0.9f, 0.999f, 1e-8f,
                                                         bc1, bc2);
    HIPFEM_CHECK(hipGetLastError());
    return 0;
}

static int mlp_free(hfem_mlp *m)
{
    void *ps[] = {m->d_p, m->d_g, m->d_m, m->d_v, m->d_X, m->d_Y, m->d_xb, m->d_h, m->d_dz, m->d_dy, m->d_lossp,
                  m->d_ix, m->d_iy, m->d_aux, m->d_loss, m->d_wpk, m->d_ws};
    for (void *p : ps)
        if (p) HIPFEM_CHECK(hipFree(p));
    return 0;
}

extern "C" int hfem_mlp_nparams(void) { return MLP_NPARAM; }

extern "C" int hfem_mlp_create(hipfem_ctx *ctx, const double *mat4, uint64_t seed, hfem_mlp **out)
{
    HIPFEM_REQUIRE(ctx && mat4 && out, HIPFEM_EINVAL, "hfem_mlp_create: null argument");
    HIPFEM_REQUIRE(mat4[0] > 0 && mat4[2] > 0, HIPFEM_EINVAL, "hfem_mlp_create: E and sig0 must be positive");
    DeviceGuard g(ctx->device);
    hfem_mlp *m = new hfem_mlp();
    m->ctx = ctx;
    m->E = mat4[0];
    m->nu = mat4[1];
    m->sig0 = mat4[2];
    m->H = mat4[3];
    m->in_scale = (float)(m->E / m->sig0);
    m->sig_scale = (float)(1.0 / m->sig0);
    m->tan_scale = (float)(1.0 / m->E);
    auto fail = [&](int rc) { mlp_free(m); delete m; return rc; };
    // U(-1/sqrt(fan_in), 1/sqrt(fan_in)) for weights and biases
    std::vector<float> p(MLP_NPARAM);
    const int fan[4] = {MLP_IN, MLP_H, MLP_H, MLP_H};
    const int offs[5] = {OFF_W1, OFF_W2, OFF_W3, OFF_W4, MLP_NPARAM};
    for (int L = 0; L < 4; L++) {
        const double a = 1.0 / std::sqrt((double)fan[L]);
        for (int i = offs[L]; i < offs[L + 1]; i++)
            p[i] = (float)(a * (2.0 * unit_open(mix64(seed * 0x9E3779B97F4A7C15ull + (uint64_t)i)) - 1.0));
    }
    const size_t nb = sizeof(float) * MLP_NPARAM;
    if (hipMalloc(&m->d_p, nb) != hipSuccess || hipMalloc(&m->d_g, nb) != hipSuccess ||
        hipMalloc(&m->d_m, nb) != hipSuccess || hipMalloc(&m->d_v, nb) != hipSuccess ||
        hipMalloc(&m->d_loss, sizeof(double)) != hipSuccess) {
        set_error("hfem_mlp_create: out of device memory");
        return fail(HIPFEM_ENOMEM);
    }
    if (hipMemcpy(m->d_p, p.data(), nb, hipMemcpyHostToDevice) != hipSuccess ||
        hipMemset(m->d_m, 0, nb) != hipSuccess || hipMemset(m->d_v, 0, nb) != hipSuccess ||
        hipMemset(m->d_g, 0, nb) != hipSuccess) {
        set_error("hfem_mlp_create: upload failed");
        return fail(HIPFEM_EHIP);
    }
    ctx_retain(ctx);
    *out = m;
    return 0;
}

extern "C" void hfem_mlp_destroy(hfem_mlp *m)
{
    if (!m) return;
    hipfem_ctx *c = m->ctx;
    {
        DeviceGuard g(c->device);
        (void)hipStreamSynchronize(c->stream);
        mlp_free(m);
        delete m;
    }
    ctx_release(c);
}

extern "C" int hfem_mlp_scales(const hfem_mlp *m, double *scales3)
{
    HIPFEM_REQUIRE(m && scales3, HIPFEM_EINVAL, "null argument");
    scales3[0] = m->in_scale;
    scales3[1] = m->sig_scale;
    scales3[2] = m->tan_scale;
    return 0;
}

extern "C" int hfem_mlp_get_params(hfem_mlp *m, float *p)
{
    HIPFEM_REQUIRE(m && p, HIPFEM_EINVAL, "null argument");
    DeviceGuard g(m->ctx->device);
    HIPFEM_CHECK(hipStreamSynchronize(m->ctx->stream));
    HIPFEM_CHECK(hipMemcpy(p, m->d_p, sizeof(float) * MLP_NPARAM, hipMemcpyDeviceToHost));
    return 0;
}

extern "C" int hfem_mlp_set_params(hfem_mlp *m, const float *p)
{
    HIPFEM_REQUIRE(m && p, HIPFEM_EINVAL, "null argument");
    DeviceGuard g(m->ctx->device);
    HIPFEM_CHECK(hipStreamSynchronize(m->ctx->stream));
    HIPFEM_CHECK(hipMemcpy(m->d_p, p, sizeof(float) * MLP_NPARAM, hipMemcpyHostToDevice));
    m->param_version++;
    return 0;
}

extern "C" int hfem_mlp_generate(hfem_mlp *m, int64_t nsamples, uint64_t seed, double stdev, int maxsteps)
{
    HIPFEM_REQUIRE(m && nsamples > 0 && stdev > 0 && maxsteps > 0, HIPFEM_EINVAL, "generate: bad arguments");
    DeviceGuard g(m->ctx->device);
    hipStream_t s = m->ctx->stream;
    // path offsets: path p holds 1..maxsteps samples (same length rule on the device)
    std::vector<int64_t> off(1, 0);
    while (off.back() < nsamples) off.push_back(off.back() + path_length(seed, (int64_t)off.size() - 1, maxsteps));
    const int64_t npaths = (int64_t)off.size() - 1;
    int64_t *d_off = nullptr;
    HIPFEM_CHECK(hipStreamSynchronize(s));
    if (m->d_X) HIPFEM_CHECK(hipFree(m->d_X));
    if (m->d_Y) HIPFEM_CHECK(hipFree(m->d_Y));
    m->d_X = m->d_Y = nullptr;
    m->nsamples = 0;
    HIPFEM_CHECK(hipMalloc(&m->d_X, sizeof(float) * (size_t)nsamples * MLP_IN));
    HIPFEM_CHECK(hipMalloc(&m->d_Y, sizeof(float) * (size_t)nsamples * MLP_OUT));
    HIPFEM_CHECK(hipMalloc(&d_off, sizeof(int64_t) * off.size()));
    HIPFEM_CHECK(hipMemcpyAsync(d_off, off.data(), sizeof(int64_t) * off.size(), hipMemcpyHostToDevice, s));
    k_mlp_paths<<<(unsigned)((npaths + 127) / 128), 128, 0, s>>>(npaths, d_off, nsamples, seed, m->E, m->nu, m->sig0,
                                                                 m->H, stdev, m->in_scale, m->sig_scale,
                                                                 m->tan_scale, m->d_X, m->d_Y);
    HIPFEM_CHECK(hipGetLastError());
    HIPFEM_CHECK(hipStreamSynchronize(s));
    HIPFEM_CHECK(hipFree(d_off));
    m->nsamples = nsamples;
    return 0;
}

extern "C" int hfem_mlp_get_samples(hfem_mlp *m, int64_t first, int64_t count, float *X, float *Y)
{
    HIPFEM_REQUIRE(m && first >= 0 && count >= 0 && first + count <= m->nsamples, HIPFEM_ERANGE,
                   "get_samples: range outside the training set");
    DeviceGuard g(m->ctx->device);
    HIPFEM_CHECK(hipStreamSynchronize(m->ctx->stream));
    if (X) HIPFEM_CHECK(hipMemcpy(X, m->d_X + first * MLP_IN, sizeof(float) * count * MLP_IN, hipMemcpyDeviceToHost));
    if (Y) HIPFEM_CHECK(hipMemcpy(Y, m->d_Y + first * MLP_OUT, sizeof(float) * count * MLP_OUT, hipMemcpyDeviceToHost));
    return 0;
}

extern "C" int hfem_mlp_train(hfem_mlp *m, int steps, int batch, double lr, double lr_final, uint64_t seed,
                              double *final_loss)
{
    HIPFEM_REQUIRE(m && steps >= 0 && batch > 0 && lr > 0, HIPFEM_EINVAL, "train: bad arguments");
    HIPFEM_REQUIRE(m->nsamples > 0, HIPFEM_EINVAL, "train: no training set (call hfem_mlp_generate)");
    DeviceGuard g(m->ctx->device);
    hipStream_t s = m->ctx->stream;
    int rc = mlp_ensure_batch(m, batch);
    if (rc) return rc;
    rc = mlp_ensure_aux(m);
    if (rc) return rc;
    const float b1 = 0.9f, b2 = 0.999f;
    for (int it = 0; it < steps; it++) {
        m->adam_t++;
        // cosine decay from lr to lr_final
        const double c = 0.5 * (1.0 + std::cos(3.141592653589793 * (double)it / std::max(1, steps)));
        const float lrt = (float)(lr_final + (lr - lr_final) * c);
        const float bc1 = 1.f - std::pow(b1, (float)m->adam_t), bc2 = 1.f - std::pow(b2, (float)m->adam_t);
        StepArgs a = {};
        a.B = batch;
        a.X = m->d_X;
        a.Y = m->d_Y;
        a.nsamples = m->nsamples;
        a.seed = seed;
        a.step = it;
        rc = mlp_step(m, a, true, lrt, bc1, bc2);
        if (rc) return rc;
    }
    m->param_version++;
    m->aux_version = m->param_version;   // the update wrote the copies too
    if (final_loss) {
        HIPFEM_CHECK(hipMemcpyAsync(final_loss, m->d_loss, sizeof(double), hipMemcpyDeviceToHost, s));
    }
    HIPFEM_CHECK(hipStreamSynchronize(s));
    return 0;
}

// host-array helpers: run the FP32 forward (and backward) on n given rows
extern "C" int hfem_mlp_forward(hfem_mlp *m, int n, const float *X, float *Y)
{
    HIPFEM_REQUIRE(m && n >= 0 && X && Y, HIPFEM_EINVAL, "forward: bad arguments");
    DeviceGuard g(m->ctx->device);
    if (n == 0) return 0;
    int rc = mlp_ensure_io(m, n);
    if (rc) return rc;
    rc = mlp_ensure_aux(m);
    if (rc) return rc;
    hipStream_t s = m->ctx->stream;
    HIPFEM_CHECK(hipMemcpyAsync(m->d_ix, X, sizeof(float) * n * MLP_IN, hipMemcpyHostToDevice, s));
    StepArgs a = {};
    a.B = n;
    a.X = m->d_ix;
    a.p = m->d_p;
    a.aux = m->d_aux;
    a.yp = m->d_iy;
    k_mlp_step<false><<<(n + TR - 1) / TR, 512, 0, s>>>(a);
    HIPFEM_CHECK(hipGetLastError());
    HIPFEM_CHECK(hipMemcpyAsync(Y, m->d_iy, sizeof(float) * n * MLP_OUT, hipMemcpyDeviceToHost, s));
    HIPFEM_CHECK(hipStreamSynchronize(s));
    return 0;
}

extern "C" int hfem_mlp_gradients(hfem_mlp *m, int n, const float *X, const float *Y, float *grad, double *loss)
{
    HIPFEM_REQUIRE(m && n > 0 && X && Y && grad, HIPFEM_EINVAL, "gradients: bad arguments");
    DeviceGuard g(m->ctx->device);
    int rc = mlp_ensure_batch(m, n);
    if (rc) return rc;
    rc = mlp_ensure_io(m, n);
    if (rc) return rc;
    rc = mlp_ensure_aux(m);
    if (rc) return rc;
    hipStream_t s = m->ctx->stream;
    HIPFEM_CHECK(hipMemcpyAsync(m->d_ix, X, sizeof(float) * n * MLP_IN, hipMemcpyHostToDevice, s));
    HIPFEM_CHECK(hipMemcpyAsync(m->d_iy, Y, sizeof(float) * n * MLP_OUT, hipMemcpyHostToDevice, s));
    StepArgs a = {};
    a.B = n;
    a.X = m->d_ix;
    a.Y = m->d_iy;
    rc = mlp_step(m, a, false, 0.f, 1.f, 1.f);
    if (rc) return rc;
    HIPFEM_CHECK(hipMemcpyAsync(grad, m->d_g, sizeof(float) * MLP_NPARAM, hipMemcpyDeviceToHost, s));
    if (loss) HIPFEM_CHECK(hipMemcpyAsync(loss, m->d_loss, sizeof(double), hipMemcpyDeviceToHost, s));
    HIPFEM_CHECK(hipStreamSynchronize(s));
    return 0;
}

namespace hipfem {
void mlp_info(const hfem_mlp *m, hipfem_ctx **ctx, double mat4[4], float scales[3])
{
    *ctx = m->ctx;
    mat4[0] = m->E;
    mat4[1] = m->nu;
    mat4[2] = m->sig0;
    mat4[3] = m->H;
    scales[0] = m->in_scale;
    scales[1] = m->sig_scale;
    scales[2] = m->tan_scale;
}

// BF16 inference of n rows of device X into device Y on the context stream
int mlp_infer_bf16_dev(hfem_mlp *m, int n, const float *dX, float *dY)
{
    hipStream_t s = m->ctx->stream;
    if (m->packed_version != m->param_version || !m->d_wpk) {
        if (!m->d_wpk) HIPFEM_CHECK(hipMalloc(&m->d_wpk, sizeof(uint16_t) * BF_TOTAL));
        uint16_t *w = m->d_wpk;
        k_pack_bf16<<<(BF_L1 + 255) / 256, 256, 0, s>>>(m->d_p + OFF_W1, MLP_H, MLP_IN, 4, 1, w);
        k_pack_bf16<<<(BF_L2 + 255) / 256, 256, 0, s>>>(m->d_p + OFF_W2, MLP_H, MLP_H, 4, 8, w + BF_L1);
        k_pack_bf16<<<(BF_L3 + 255) / 256, 256, 0, s>>>(m->d_p + OFF_W3, MLP_H, MLP_H, 4, 8, w + BF_L1 + BF_L2);
        k_pack_bf16<<<(BF_L4 + 255) / 256, 256, 0, s>>>(m->d_p + OFF_W4, MLP_OUT, MLP_H, 1, 8,
                                                        w + BF_L1 + BF_L2 + BF_L3);
        HIPFEM_CHECK(hipGetLastError());
        m->packed_version = m->param_version;
    }
    if (n <= 0) return 0;
    const size_t lds = sizeof(uint16_t) * (BF_TOTAL + BF_WAVES * 32 * ACT_LD);
    int dev = 0, maxlds = 0;
    HIPFEM_CHECK(hipGetDevice(&dev));
    HIPFEM_CHECK(hipDeviceGetAttribute(&maxlds, hipDeviceAttributeMaxSharedMemoryPerBlock, dev));
    HIPFEM_REQUIRE((size_t)maxlds >= lds, HIPFEM_EINVAL,
                   "surrogate inference needs %zu bytes of LDS per workgroup, the device offers %d", lds, maxlds);
    const int ntile = (n + 31) / 32;
    // one workgroup per CU (the LDS holds one), each looping over its tiles
    const int grid = std::max(1, std::min((ntile + BF_WAVES - 1) / BF_WAVES, 256));
    k_mlp_bf16<<<grid, 64 * BF_WAVES, lds, s>>>(n, dX, dY, m->d_wpk, m->d_p);
    HIPFEM_CHECK(hipGetLastError());
    return 0;
}
}  // namespace hipfem

extern "C" int hfem_mlp_infer_bf16(hfem_mlp *m, int n, const float *X, float *Y)
{
    HIPFEM_REQUIRE(m && n >= 0 && X && Y, HIPFEM_EINVAL, "infer: bad arguments");
    DeviceGuard g(m->ctx->device);
    hipStream_t s = m->ctx->stream;
    float *dX = nullptr, *dY = nullptr;
    HIPFEM_CHECK(hipMalloc(&dX, sizeof(float) * std::max(1, n) * MLP_IN));
    HIPFEM_CHECK(hipMalloc(&dY, sizeof(float) * std::max(1, n) * MLP_OUT));
    int rc = 0;
    if (n) HIPFEM_CHECK(hipMemcpyAsync(dX, X, sizeof(float) * n * MLP_IN, hipMemcpyHostToDevice, s));
    rc = mlp_infer_bf16_dev(m, n, dX, dY);
    if (!rc && n) {
        HIPFEM_CHECK(hipMemcpyAsync(Y, dY, sizeof(float) * n * MLP_OUT, hipMemcpyDeviceToHost, s));
    }
    HIPFEM_CHECK(hipStreamSynchronize(s));
    HIPFEM_CHECK(hipFree(dX));
    HIPFEM_CHECK(hipFree(dY));
    return rc;
}
