// mlp.hip -- neighbour-count forecaster: a 4-64-64-1 MLP (tanh, softplus Poisson rate)
// trained online with hand-written forward / backward / reduction / Adam kernels.
//
// Parameter layout (float32, 4545 values): W1[64][4], b1[64], W2[64][64], b2[64],
// w3[64], b3.  Loss: mean Poisson NLL  lambda - y log(lambda + 1e-6).
// Forward (k_mlp_forward): one thread per sample, parameters read with wave-uniform addresses
// (scalar loads, no per-lane traffic).  Training: k_mlp_backward and k_mlp_update below.
#include <vector>

#include "mlp.hpp"

namespace gplum {

constexpr int OFF_W1 = 0, OFF_B1 = 256, OFF_W2 = 320, OFF_B2 = 4416, OFF_W3 = 4480, OFF_B3 = 4544;
static_assert(OFF_B3 + 1 == MLP_NPARAM, "parameter layout");
constexpr float MLP_EPS = 1e-6f;

__device__ inline float softplus_f(float z) { return z > 20.f ? z : log1pf(expf(z)); }
__device__ inline float sigmoid_f(float z) { return 1.f / (1.f + expf(-z)); }

// per-sample forward pass; h1, h2 in registers.  The weights are read with
// wave-uniform addresses straight from global memory, which the compiler turns into
// scalar loads: every lane uses the same weight, so no LDS traffic per FMA.
__device__ inline float mlp_eval(const float *__restrict__ s, const float x[MLP_NIN], float h1[MLP_NH],
                                 float h2[MLP_NH], float *zout) {
    // every loop fully unrolled: h1/h2 are indexed by compile-time constants and stay
    // in registers (a runtime index would put them in scratch memory)
#pragma unroll
    for (int p = 0; p < MLP_NH; p++) {
        float a = s[OFF_B1 + p];
#pragma unroll
        for (int q = 0; q < MLP_NIN; q++) a = __builtin_fmaf(s[OFF_W1 + p * MLP_NIN + q], x[q], a);
        h1[p] = tanhf(a);
    }
#pragma unroll
    for (int p = 0; p < MLP_NH; p++) {
        float a = s[OFF_B2 + p];
#pragma unroll
        for (int q = 0; q < MLP_NH; q++) a = __builtin_fmaf(s[OFF_W2 + p * MLP_NH + q], h1[q], a);
        h2[p] = tanhf(a);
    }
    float z = s[OFF_B3];
#pragma unroll
    for (int p = 0; p < MLP_NH; p++) z = __builtin_fmaf(s[OFF_W3 + p], h2[p], z);
    *zout = z;
    return softplus_f(z);
}

__global__ __launch_bounds__(256) void k_mlp_forward(const float *__restrict__ theta, const float *__restrict__ x,
                                                     int n, float *__restrict__ lam) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    float xi[MLP_NIN], h1[MLP_NH], h2[MLP_NH], z;
#pragma unroll
    for (int q = 0; q < MLP_NIN; q++) xi[q] = x[(size_t)q * n + i];
    lam[i] = mlp_eval(theta, xi, h1, h2, &z);
}

// --------------------------------------------------------------- training
//
// A training step is 0.1 GFLOP and 0.2 MB: bound by how many CUs take part and by the latency of
// its few dependent stages.  A workgroup of 4 waves takes tiles of 32 samples (8192 samples: one
// tile on every CU); the 64 x 64 layer runs forward and backward on the FP32 matrix
// instruction (16 x 16 x 4: FP32 operands and sums), wave w owning hidden units 16 w ... 16 w + 15, with W2
// as operands in registers.  The gradient is summed in FP64 (products of two FP32 values are
// exact there): W2's on the FP64 matrix instruction, the others per lane, over the tiles of a
// workgroup in registers; the workgroups' sums are added in a fixed order by k_mlp_update, which
// also takes the Adam step.  One thread per sample (32 workgroups, weights by scalar loads, the
// activations through memory to a second and third pass): 94 + 18 + 17 + 5 us per step of
// 8192 samples.
typedef float mlp_v4f __attribute__((ext_vector_type(4)));
typedef double mlp_v4d __attribute__((ext_vector_type(4)));

constexpr int MLP_TILE = 32;         // samples per tile
constexpr int MLP_LD = 68;           // row stride of a tile in LDS: 16 rows x 4 columns hit 64 banks
constexpr int MLP_MAX_WG = 256;

static int mlp_grid(int n) { return std::min(ceil_div(n, MLP_TILE), MLP_MAX_WG); }

__global__ __launch_bounds__(256) void k_mlp_backward(const float *__restrict__ s, const float *__restrict__ x,
                                                      const float *__restrict__ y, int n, double *__restrict__ part,
                                                      double *__restrict__ loss_part) {
    __shared__ float s_h[MLP_TILE][MLP_LD], s_d[MLP_TILE][MLP_LD], s_x[MLP_TILE][MLP_NIN];
    __shared__ float s_z[4][MLP_TILE], s_dz[MLP_TILE];
    const int t = (int)threadIdx.x, w = t >> 6, l = t & 63, r = l >> 4, c = l & 15;
    // layer 1: lane t evaluates units u0 .. u0 + 7 of sample t % 32
    const int si = t & 31, u0 = (t >> 5) * 8;
    float w1[8][MLP_NIN], b1[8];
#pragma unroll
    for (int u = 0; u < 8; u++) {
        b1[u] = s[OFF_B1 + u0 + u];
#pragma unroll
        for (int q = 0; q < MLP_NIN; q++) w1[u][q] = s[OFF_W1 + (u0 + u) * MLP_NIN + q];
    }
    // W2 as right operand B[k][n] (lane: k = 4 ks + r, n = unit): forward W2[n][k], backward W2[k][n]
    const int unit = 16 * w + c;
    float wf[16], wb[16];
#pragma unroll
    for (int ks = 0; ks < 16; ks++) {
        wf[ks] = s[OFF_W2 + unit * MLP_NH + 4 * ks + r];
        wb[ks] = s[OFF_W2 + (4 * ks + r) * MLP_NH + unit];
    }
    const float b2 = s[OFF_B2 + unit], w3 = s[OFF_W3 + unit], b3 = s[OFF_B3];
    mlp_v4d g2[4] = {};
    double gb1 = 0., gb2 = 0., gw3 = 0., gb3 = 0., loss = 0., gw1[MLP_NIN] = {};
    const int tiles = (n + MLP_TILE - 1) / MLP_TILE;
    for (int tile = (int)blockIdx.x; tile < tiles; tile += (int)gridDim.x) {
        const int i0 = MLP_TILE * tile;
        {
            float xi[MLP_NIN];
#pragma unroll
            for (int q = 0; q < MLP_NIN; q++) xi[q] = (i0 + si < n) ? x[(size_t)q * n + i0 + si] : 0.f;
            if (t < MLP_TILE)
#pragma unroll
                for (int q = 0; q < MLP_NIN; q++) s_x[t][q] = xi[q];
#pragma unroll
            for (int u = 0; u < 8; u++) {
                float a = b1[u];
#pragma unroll
                for (int q = 0; q < MLP_NIN; q++) a = __builtin_fmaf(w1[u][q], xi[q], a);
                s_h[si][u0 + u] = tanhf(a);
            }
        }
        __syncthreads();
        // h2 of samples 16 h + 4 r + j, unit `unit`; the output layer's sum over the units
        float h2[2][4];
#pragma unroll
        for (int h = 0; h < 2; h++) {
            mlp_v4f acc = {b2, b2, b2, b2};
#pragma unroll
            for (int ks = 0; ks < 16; ks++)
                acc = __builtin_amdgcn_mfma_f32_16x16x4f32(s_h[16 * h + c][4 * ks + r], wf[ks], acc, 0, 0, 0);
#pragma unroll
            for (int j = 0; j < 4; j++) {
                h2[h][j] = tanhf(acc[j]);
                float z = w3 * h2[h][j];
#pragma unroll
                for (int d = 1; d < 16; d <<= 1) z += __shfl_xor(z, d);
                if (c == 0) s_z[w][16 * h + 4 * r + j] = z;
            }
        }
        __syncthreads();
        if (t < MLP_TILE) {
            float dz = 0.f;
            if (i0 + t < n) {
                const float z = b3 + ((s_z[0][t] + s_z[1][t]) + (s_z[2][t] + s_z[3][t]));
                const float lam = softplus_f(z), yi = y[i0 + t];
                loss += (double)lam - (double)yi * log((double)lam + (double)MLP_EPS);
                dz = (1.f - yi / (lam + MLP_EPS)) * sigmoid_f(z) / (float)n;
            }
            s_dz[t] = dz;
            gb3 += (double)dz;
        }
        __syncthreads();
#pragma unroll
        for (int h = 0; h < 2; h++)
#pragma unroll
            for (int j = 0; j < 4; j++) {
                const int row = 16 * h + 4 * r + j;
                const float dz = s_dz[row], d2 = dz * w3 * (1.f - h2[h][j] * h2[h][j]);
                s_d[row][unit] = d2;
                gb2 += (double)d2;
                gw3 += (double)dz * (double)h2[h][j];
            }
        __syncthreads();
#pragma unroll
        for (int h = 0; h < 2; h++) {
            mlp_v4f acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int ks = 0; ks < 16; ks++)
                acc = __builtin_amdgcn_mfma_f32_16x16x4f32(s_d[16 * h + c][4 * ks + r], wb[ks], acc, 0, 0, 0);
#pragma unroll
            for (int j = 0; j < 4; j++) {
                const int row = 16 * h + 4 * r + j;
                const float h1 = s_h[row][unit], d1 = acc[j] * (1.f - h1 * h1);
                gb1 += (double)d1;
#pragma unroll
                for (int q = 0; q < MLP_NIN; q++) gw1[q] += (double)d1 * (double)s_x[row][q];
            }
        }
        // dW2[p][q] += d2[sample][p] h1[sample][q]: rows p = 16 w + ..., columns 16 u + c
#pragma unroll
        for (int ks = 0; ks < MLP_TILE / 4; ks++) {
            const double a = (double)s_d[4 * ks + r][unit];
#pragma unroll
            for (int u = 0; u < 4; u++)
                g2[u] = __builtin_amdgcn_mfma_f64_16x16x4f64(a, (double)s_h[4 * ks + r][16 * u + c], g2[u], 0, 0, 0);
        }
        __syncthreads();
    }
    double *o = part + (size_t)blockIdx.x * MLP_NPARAM;
    auto rows_sum = [](double v) {                        // over the four lanes of a unit
        v += __shfl_xor(v, 16);
        return v + __shfl_xor(v, 32);
    };
    gb1 = rows_sum(gb1);
    gb2 = rows_sum(gb2);
    gw3 = rows_sum(gw3);
#pragma unroll
    for (int q = 0; q < MLP_NIN; q++) gw1[q] = rows_sum(gw1[q]);
    if (r == 0) {
        o[OFF_B1 + unit] = gb1;
        o[OFF_B2 + unit] = gb2;
        o[OFF_W3 + unit] = gw3;
#pragma unroll
        for (int q = 0; q < MLP_NIN; q++) o[OFF_W1 + unit * MLP_NIN + q] = gw1[q];
    }
    // the FP64 instruction's result: row 4 j + r, column c
#pragma unroll
    for (int u = 0; u < 4; u++)
#pragma unroll
        for (int j = 0; j < 4; j++) o[OFF_W2 + (16 * w + 4 * j + r) * MLP_NH + 16 * u + c] = g2[u][j];
    if (t < MLP_TILE) {
#pragma unroll
        for (int d = 1; d < MLP_TILE; d <<= 1) {
            gb3 += __shfl_xor(gb3, d);
            loss += __shfl_xor(loss, d);
        }
        if (t == 0) {
            o[OFF_B3] = gb3;
            loss_part[blockIdx.x] = loss;
        }
    }
}

// grad = the workgroups' sums added in order (8 runs of workgroups, then the runs); adam: theta's
// step too.  32 parameters per workgroup.
struct AdamStep {
    int on;
    float lr, b1, b2, c1, c2;
};
__global__ __launch_bounds__(256) void k_mlp_update(int nparts, const double *__restrict__ part, float *__restrict__ grad,
                                                    float *__restrict__ theta, float *__restrict__ m, float *__restrict__ v,
                                                    AdamStep a) {
    __shared__ double s_sum[8][32];
    const int kk = (int)threadIdx.x & 31, run = (int)threadIdx.x >> 5, k = (int)blockIdx.x * 32 + kk;
    const int per = (nparts + 7) / 8, c1 = min(nparts, (run + 1) * per);
    double acc = 0.;
    if (k < MLP_NPARAM)
#pragma unroll 8
        for (int c = run * per; c < c1; c++) acc += part[(size_t)c * MLP_NPARAM + k];
    s_sum[run][kk] = acc;
    __syncthreads();
    if (threadIdx.x >= 32 || k >= MLP_NPARAM) return;
    for (int q = 1; q < 8; q++) acc += s_sum[q][kk];
    const float g = (float)acc;
    grad[k] = g;
    if (!a.on) return;
    const float mk = a.b1 * m[k] + (1.f - a.b1) * g;
    const float vk = a.b2 * v[k] + (1.f - a.b2) * g * g;
    m[k] = mk;
    v[k] = vk;
    theta[k] -= a.lr * (mk / a.c1) / (sqrtf(vk / a.c2) + 1e-8f);
}

// ---------------------------------------------- prediction on the matrix cores
//
// The rates that size the candidate buffers (fc_plan) need no more than a few digits:
// the 64x64 hidden layer runs on MFMA (v_mfma_f32_16x16x16bf16_1k: bf16 operands,
// FP32 accumulation) and tanh comes from the hardware exp and reciprocal.  A wave
// takes 16 samples per tile: lane l evaluates layer 1 for sample l % 16 and the
// sixteen hidden units 16 s + 4 (l / 16) + j (s, j = 0..3), which are exactly its A
// operands (A[i][k] = h1 of sample i, unit k) of the four K-steps; W2 is held as the B
// operands (B[k][n] = W2[n][k]) for the four 16-column output tiles; the accumulators
// (D[i][n], i = 4 (l / 16) + j, n = 16 t + l % 16) start at b2, and the output layer
// sums w3 h2 over the 16 lanes of a row.  Agrees with k_mlp_forward to bf16 precision.
typedef short mlp_v4s __attribute__((ext_vector_type(4)));

__device__ inline short bf16_rn(float x) {                // round to nearest even
    const unsigned u = __float_as_uint(x);
    return (short)((u + 0x7FFFu + ((u >> 16) & 1u)) >> 16);
}
__device__ inline float tanh_fast(float a) {               // 1 - 2 / (1 + e^(2a))
    return 1.f - 2.f * __builtin_amdgcn_rcpf(1.f + __expf(2.f * a));
}

constexpr int MLP_PRED_BLOCK = 256;

__global__ __launch_bounds__(MLP_PRED_BLOCK) void k_mlp_predict(const float *__restrict__ s,
                                                                const float *__restrict__ x, int n,
                                                                float *__restrict__ lam) {
    const int l = (int)threadIdx.x & 63;
    const int r = l >> 4, c = l & 15;
    // this lane's layer-1 units, W2 as B operands, b2 / w3 of its output columns
    float w1[16][MLP_NIN], b1[16];
#pragma unroll
    for (int u = 0; u < 16; u++) {
        const int k = 16 * (u >> 2) + 4 * r + (u & 3);
        b1[u] = s[OFF_B1 + k];
#pragma unroll
        for (int q = 0; q < MLP_NIN; q++) w1[u][q] = s[OFF_W1 + k * MLP_NIN + q];
    }
    mlp_v4s bw[4][4];
    float b2[4], w3[4];
#pragma unroll
    for (int t = 0; t < 4; t++) {
        const int nn = 16 * t + c;
        b2[t] = s[OFF_B2 + nn];
        w3[t] = s[OFF_W3 + nn];
#pragma unroll
        for (int ks = 0; ks < 4; ks++)
#pragma unroll
            for (int j = 0; j < 4; j++) bw[t][ks][j] = bf16_rn(s[OFF_W2 + nn * MLP_NH + 16 * ks + 4 * r + j]);
    }
    const float b3 = s[OFF_B3];
    const int waves = (int)(gridDim.x * (MLP_PRED_BLOCK / 64));
    const int tiles = (n + 15) / 16;
    for (int tile = (int)blockIdx.x * (MLP_PRED_BLOCK / 64) + ((int)threadIdx.x >> 6); tile < tiles;
         tile += waves) {
        const int i = 16 * tile + c;
        float xi[MLP_NIN];
#pragma unroll
        for (int q = 0; q < MLP_NIN; q++) xi[q] = (i < n) ? x[(size_t)q * n + i] : 0.f;
        mlp_v4s a[4];
#pragma unroll
        for (int u = 0; u < 16; u++) {
            float z = b1[u];
#pragma unroll
            for (int q = 0; q < MLP_NIN; q++) z = __builtin_fmaf(w1[u][q], xi[q], z);
            a[u >> 2][u & 3] = bf16_rn(tanh_fast(z));
        }
        float zp[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int t = 0; t < 4; t++) {
            mlp_v4f acc = {b2[t], b2[t], b2[t], b2[t]};
#pragma unroll
            for (int ks = 0; ks < 4; ks++) acc = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(a[ks], bw[t][ks], acc, 0, 0, 0);
#pragma unroll
            for (int j = 0; j < 4; j++) zp[j] = __builtin_fmaf(w3[t], tanh_fast(acc[j]), zp[j]);
        }
        // sum over the 16 output columns of the row (lanes 16 r .. 16 r + 15)
#pragma unroll
        for (int d = 8; d > 0; d >>= 1)
#pragma unroll
            for (int j = 0; j < 4; j++) zp[j] += __shfl_xor(zp[j], d);
        // lane c < 4 of row r writes sample 4 r + c of the tile
        const int o = 16 * tile + 4 * r + c;
        float zo = zp[0];
#pragma unroll
        for (int j = 1; j < 4; j++) zo = (c == j) ? zp[j] : zo;
        if (c < 4 && o < n) lam[o] = softplus_f(zo + b3);
    }
}

// ------------------------------------------------------------------ host

int Forecaster::ensure(int nsamp) {
    GPLUM_ENSURE(theta, MLP_NPARAM);
    GPLUM_ENSURE(grad, MLP_NPARAM);
    GPLUM_ENSURE(m, MLP_NPARAM);
    GPLUM_ENSURE(v, MLP_NPARAM);
    GPLUM_ENSURE(part, (size_t)MLP_NPARAM * mlp_grid(nsamp));
    GPLUM_ENSURE(loss_part, mlp_grid(nsamp));
    return GPLUM_OK;
}

int Forecaster::init_params(hipStream_t st, unsigned seed) {
    if (initialized) return GPLUM_OK;
    int rc = ensure(1);
    if (rc) return rc;
    std::vector<float> h(MLP_NPARAM, 0.f);
    // deterministic LCG + Box-Muller: W ~ N(0, 1/fan_in), biases 0, b3 = -2
    unsigned long long s = 0x9E3779B97F4A7C15ull ^ seed;
    auto uni = [&]() {
        s = s * 6364136223846793005ull + 1442695040888963407ull;
        return ((s >> 11) + 0.5) * (1.0 / 9007199254740992.0);
    };
    auto gauss = [&]() { return std::sqrt(-2.0 * std::log(uni())) * std::cos(6.283185307179586 * uni()); };
    for (int k = OFF_W1; k < OFF_B1; k++) h[k] = (float)(gauss() / 2.0);
    for (int k = OFF_W2; k < OFF_B2; k++) h[k] = (float)(gauss() / 8.0);
    for (int k = OFF_W3; k < OFF_B3; k++) h[k] = (float)(gauss() / 8.0);
    h[OFF_B3] = -2.f;
    GPLUM_HIP(hipMemcpyAsync(theta.p, h.data(), sizeof(float) * MLP_NPARAM, hipMemcpyHostToDevice, st));
    GPLUM_HIP(hipMemsetAsync(m.p, 0, sizeof(float) * MLP_NPARAM, st));
    GPLUM_HIP(hipMemsetAsync(v.p, 0, sizeof(float) * MLP_NPARAM, st));
    adam_t = 0;
    initialized = true;
    return GPLUM_OK;
}

int Forecaster::forward(const float *d_x, int n, float *d_lam, hipStream_t st) {
    if (n <= 0) return GPLUM_OK;
    hipLaunchKernelGGL(k_mlp_forward, dim3(ceil_div(n, 256)), dim3(256), 0, st, theta.p, d_x, n, d_lam);
    GPLUM_HIP(hipGetLastError());
    return GPLUM_OK;
}

int Forecaster::predict(const float *d_x, int n, float *d_lam, hipStream_t st) {
    if (n <= 0) return GPLUM_OK;
    const int tiles = ceil_div(n, 16);
    const int blocks = std::min(ceil_div(tiles, MLP_PRED_BLOCK / 64), 2048);
    hipLaunchKernelGGL(k_mlp_predict, dim3(blocks), dim3(MLP_PRED_BLOCK), 0, st, theta.p, d_x, n, d_lam);
    GPLUM_HIP(hipGetLastError());
    return GPLUM_OK;
}

int Forecaster::gradient(const float *d_x, const float *d_y, int n, double *loss, bool step, hipStream_t st) {
    int rc = ensure(n);
    if (rc) return rc;
    AdamStep a{0, lr, 0.9f, 0.999f, 1.f, 1.f};
    if (step) {
        adam_t++;
        a.on = 1;
        a.c1 = 1.f - std::pow(a.b1, (float)adam_t);
        a.c2 = 1.f - std::pow(a.b2, (float)adam_t);
    }
    const int grid = mlp_grid(n);
    hipLaunchKernelGGL(k_mlp_backward, dim3(grid), dim3(256), 0, st, theta.p, d_x, d_y, n, part.p, loss_part.p);
    hipLaunchKernelGGL(k_mlp_update, dim3(ceil_div(MLP_NPARAM, 32)), dim3(256), 0, st, grid, part.p, grad.p, theta.p, m.p, v.p,
                       a);
    GPLUM_HIP(hipGetLastError());
    if (loss) return read_loss(n, loss, st);
    return GPLUM_OK;
}

int Forecaster::read_loss(int n, double *loss, hipStream_t st) {
    std::vector<double> h(mlp_grid(n));
    GPLUM_HIP(hipMemcpyAsync(h.data(), loss_part.p, sizeof(double) * h.size(), hipMemcpyDeviceToHost, st));
    GPLUM_HIP(hipStreamSynchronize(st));
    double s = 0.;
    for (double x : h) s += x;
    *loss = s / n;
    return GPLUM_OK;
}

}  // namespace gplum

// ------------------------------------------------------------------ C ABI (tests)

namespace {
struct MlpCtx {
    hipStream_t st = nullptr;
    gplum::Forecaster f;
    gplum::DArray<float> x, y, lam;
};
thread_local MlpCtx t_mlp;

int mlp_ctx_init(MlpCtx &c) {
    if (!c.st) GPLUM_HIP(hipStreamCreateWithFlags(&c.st, hipStreamNonBlocking));
    return GPLUM_OK;
}
}  // namespace

extern "C" int gplum_mlp_forward(const float *theta, const float *x, int n, float *lam) {
    if (!theta || (n > 0 && (!x || !lam)) || n < 0) return gplum::fail(GPLUM_E_ARG, "bad arguments");
    MlpCtx &c = t_mlp;
    int rc = mlp_ctx_init(c);
    if (rc) return rc;
    if ((rc = c.f.ensure(1))) return rc;
    GPLUM_ENSURE(c.x, 4 * (size_t)n + 4);
    GPLUM_ENSURE(c.lam, (size_t)n + 1);
    GPLUM_HIP(hipMemcpyAsync(c.f.theta.p, theta, sizeof(float) * gplum::MLP_NPARAM, hipMemcpyHostToDevice, c.st));
    GPLUM_HIP(hipMemcpyAsync(c.x.p, x, sizeof(float) * 4 * n, hipMemcpyHostToDevice, c.st));
    if ((rc = c.f.forward(c.x.p, n, c.lam.p, c.st))) return rc;
    GPLUM_HIP(hipMemcpyAsync(lam, c.lam.p, sizeof(float) * n, hipMemcpyDeviceToHost, c.st));
    GPLUM_HIP(hipStreamSynchronize(c.st));
    return GPLUM_OK;
}

extern "C" int gplum_mlp_predict(const float *theta, const float *x, int n, float *lam) {
    if (!theta || (n > 0 && (!x || !lam)) || n < 0) return gplum::fail(GPLUM_E_ARG, "bad arguments");
    MlpCtx &c = t_mlp;
    int rc = mlp_ctx_init(c);
    if (rc) return rc;
    if ((rc = c.f.ensure(1))) return rc;
    GPLUM_ENSURE(c.x, 4 * (size_t)n + 4);
    GPLUM_ENSURE(c.lam, (size_t)n + 1);
    GPLUM_HIP(hipMemcpyAsync(c.f.theta.p, theta, sizeof(float) * gplum::MLP_NPARAM, hipMemcpyHostToDevice, c.st));
    GPLUM_HIP(hipMemcpyAsync(c.x.p, x, sizeof(float) * 4 * n, hipMemcpyHostToDevice, c.st));
    if ((rc = c.f.predict(c.x.p, n, c.lam.p, c.st))) return rc;
    GPLUM_HIP(hipMemcpyAsync(lam, c.lam.p, sizeof(float) * n, hipMemcpyDeviceToHost, c.st));
    GPLUM_HIP(hipStreamSynchronize(c.st));
    return GPLUM_OK;
}

extern "C" int gplum_mlp_loss_grad(const float *theta, const float *x, const float *y, int n, double *loss,
                                   float *grad) {
    if (!theta || !x || !y || !grad || n <= 0) return gplum::fail(GPLUM_E_ARG, "bad arguments");
    MlpCtx &c = t_mlp;
    int rc = mlp_ctx_init(c);
    if (rc) return rc;
    if ((rc = c.f.ensure(n))) return rc;
    GPLUM_ENSURE(c.x, 4 * (size_t)n);
    GPLUM_ENSURE(c.y, (size_t)n);
    GPLUM_HIP(hipMemcpyAsync(c.f.theta.p, theta, sizeof(float) * gplum::MLP_NPARAM, hipMemcpyHostToDevice, c.st));
    GPLUM_HIP(hipMemcpyAsync(c.x.p, x, sizeof(float) * 4 * n, hipMemcpyHostToDevice, c.st));
    GPLUM_HIP(hipMemcpyAsync(c.y.p, y, sizeof(float) * n, hipMemcpyHostToDevice, c.st));
    if ((rc = c.f.gradient(c.x.p, c.y.p, n, loss, false, c.st))) return rc;
    GPLUM_HIP(hipMemcpyAsync(grad, c.f.grad.p, sizeof(float) * gplum::MLP_NPARAM, hipMemcpyDeviceToHost, c.st));
    GPLUM_HIP(hipStreamSynchronize(c.st));
    return GPLUM_OK;
}

extern "C" int gplum_mlp_train(float *theta, const float *x, const float *y, int n, int n_steps, float lr,
                               double *loss_first, double *loss_last) {
    if (!theta || !x || !y || n <= 0 || n_steps < 0 || !(lr > 0.f))
        return gplum::fail(GPLUM_E_ARG, "bad arguments");
    MlpCtx &c = t_mlp;
    int rc = mlp_ctx_init(c);
    if (rc) return rc;
    gplum::Forecaster &f = c.f;   // the thread's buffers, with a fresh Adam state for this call
    if ((rc = f.ensure(n))) return rc;
    f.adam_t = 0;
    f.lr = lr;
    GPLUM_ENSURE(c.x, 4 * (size_t)n);
    GPLUM_ENSURE(c.y, (size_t)n);
    GPLUM_HIP(hipMemcpyAsync(f.theta.p, theta, sizeof(float) * gplum::MLP_NPARAM, hipMemcpyHostToDevice, c.st));
    GPLUM_HIP(hipMemsetAsync(f.m.p, 0, sizeof(float) * gplum::MLP_NPARAM, c.st));
    GPLUM_HIP(hipMemsetAsync(f.v.p, 0, sizeof(float) * gplum::MLP_NPARAM, c.st));
    GPLUM_HIP(hipMemcpyAsync(c.x.p, x, sizeof(float) * 4 * n, hipMemcpyHostToDevice, c.st));
    GPLUM_HIP(hipMemcpyAsync(c.y.p, y, sizeof(float) * n, hipMemcpyHostToDevice, c.st));
    for (int s = 0; s < n_steps; s++) {
        double *lp = (s == 0) ? loss_first : nullptr;
        if ((rc = f.gradient(c.x.p, c.y.p, n, lp, true, c.st))) return rc;
    }
    if (loss_last) {
        if ((rc = f.gradient(c.x.p, c.y.p, n, loss_last, false, c.st))) return rc;
    }
    GPLUM_HIP(hipMemcpyAsync(theta, f.theta.p, sizeof(float) * gplum::MLP_NPARAM, hipMemcpyDeviceToHost, c.st));
    GPLUM_HIP(hipStreamSynchronize(c.st));
    return GPLUM_OK;
}
