// closure.hip -- learned subgrid closure: features, network inference and
// training, and its right-hand side.
//
// No counterpart in the reference (its fluxes are the resolved ones only,
// mhdrhs.f90:60-119). On a coarse grid the filtered equations carry
// unresolved flux terms: the subgrid Reynolds stress R_ij, Maxwell stress
// M_ij, electromotive force and energy flux. A small network maps the resolved
// state at a point and its 3^3-stencil gradients to those 18 terms; the step
// adds the divergence of the momentum-flux and energy-flux corrections and the
// curl of the EMF correction to the right-hand side.
//
//   features (28): rho, u (3), B (3), then d/dx, d/dy, d/dz of rho, ux, uy,
//                  uz, Bx, By, Bz (central differences, periodic), each
//                  normalised as (f - mean) / std
//   network:       28 -> 64 (tanh) -> 64 (tanh) -> 18, FP32
//   outputs (18):  R xx, xy, xz, yy, yz, zz; M xx, xy, xz, yy, yz, zz;
//                  EMF x, y, z; energy flux x, y, z;
//                  physical value = output * ystd
//
// Parameter vector (FP32): W1[28][64], b1[64], W2[64][64], b2[64],
// W3[64][18], b3[18], then xmean[28], xstd[28], ystd[18].
#include "internal.hpp"

namespace laps {

namespace {

constexpr int kThreadsCl = 256;

}  // namespace

// ---------------------------------------------------------------- features

__global__ void k_cl_features(const double* __restrict__ S, int nx, int ny, int nz, double dx, double dy, double dz,
                              const float* __restrict__ norm, float* __restrict__ X) {
    const long long N = (long long)nx * ny * nz;
    const long long i = blockIdx.x * (long long)blockDim.x + threadIdx.x;
    if (i >= N) return;
    const int ix = (int)(i % nx);
    const int iy = (int)((i / nx) % ny);
    const int iz = (int)(i / ((long long)nx * ny));
    const long long xp = i - ix + (ix + 1 == nx ? 0 : ix + 1), xm = i - ix + (ix == 0 ? nx - 1 : ix - 1);
    const long long sy = nx, sz = (long long)nx * ny;
    const long long yp = i + (iy + 1 == ny ? -(long long)(ny - 1) * sy : sy);
    const long long ym = i + (iy == 0 ? (long long)(ny - 1) * sy : -sy);
    const long long zp = i + (iz + 1 == nz ? -(long long)(nz - 1) * sz : sz);
    const long long zm = i + (iz == 0 ? (long long)(nz - 1) * sz : -sz);
    // fields: rho = S[0], u = S[8..10] (primitives), B = S[4..6]
    const int fld[7] = {0, 8, 9, 10, 4, 5, 6};
    float f[28];
#pragma unroll
    for (int q = 0; q < 7; ++q) {
        const double* g = S + fld[q] * N;
        f[q] = (float)g[i];
        f[7 + 3 * q] = (float)((g[xp] - g[xm]) / (2.0 * dx));
        f[8 + 3 * q] = (float)((g[yp] - g[ym]) / (2.0 * dy));
        f[9 + 3 * q] = (float)((g[zp] - g[zm]) / (2.0 * dz));
    }
    const float* mean = norm;
    const float* sd = norm + kClIn;
#pragma unroll
    for (int q = 0; q < kClIn; ++q) X[i * kClIn + q] = (f[q] - mean[q]) / sd[q];
}

// ---------------------------------------------------------------- network
//
// The three layers are small dense products over the samples, run on the FP32 matrix units
// (v_mfma_f32_16x16x4_f32, twice the FP32 vector rate). A work-group of four waves takes tiles
// of 16*MT samples; wave w owns the columns 16w..16w+15 of a hidden layer and keeps its weight
// operands in registers over all tiles, so the weights are read once per work-group and only
// the activations go through LDS. Operand layout of the instruction, for lane (g = lane / 16,
// c = lane % 16): A holds row c at k-slot g, B holds column c at k-slot g, and register i of
// the result is row 4g + i, column c. Which k a slot stands for is free as long as A and B
// agree, and is chosen so that a lane's operands are neighbours in memory. tanhf is the library's: 1.41
// units in the last place at most over all floats. A polynomial below 0.55 and the hardware exponential and
// reciprocal above reach 1.96; they are ahead in large batches (262144 samples forward 68 us with tanhf, 59
// with them, the gradient 177 and 154), level at 4096 samples and behind in k_cl_net (68 and 71).

typedef float f32x4 __attribute__((ext_vector_type(4)));

__device__ __forceinline__ f32x4 mfma16(float a, float b, f32x4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
}

// LDS row strides: 68 floats put the 16-float operand reads of 16 rows, and the column writes of
// the results, on distinct banks, and keep the reads 16-byte aligned
constexpr int kHS = 68;   // hidden activations (64 used)
constexpr int kYS = 36;   // outputs (18 used, columns 18-31 zero)
constexpr int kXS = 36;   // features (28 used)

// weight operands of wave w for the forward layers: k-slot (g, s) is k = 7g + s of the inputs and
// k = 16g + s of the hidden layers
struct FwdWeights {
    float w1[7], w2[16], w3[16], b1, b2, b3;
    __device__ __forceinline__ void load(const float* __restrict__ P, int w, int g, int c) {
        const float* B1 = P + kClIn * kClH;
        const float* W2 = B1 + kClH;
        const float* B2 = W2 + kClH * kClH;
        const float* W3 = B2 + kClH;
        const float* B3 = W3 + kClH * kClOut;
        const int o = 16 * w + c, n = 16 * (w & 1) + c;
        const int nc = n < kClOut ? n : 0;
#pragma unroll
        for (int s = 0; s < 7; ++s) w1[s] = P[(7 * g + s) * kClH + o];
#pragma unroll
        for (int s = 0; s < 16; ++s) {
            w2[s] = W2[(16 * g + s) * kClH + o];
            const float t = W3[(16 * g + s) * kClOut + nc];
            w3[s] = n < kClOut ? t : 0.f;
        }
        b1 = B1[o];
        b2 = B2[o];
        b3 = n < kClOut ? B3[nc] : 0.f;
    }
};

// one row of a hidden tile times 16 k-slots of the wave's weights
__device__ __forceinline__ f32x4 hidden_product(const float* __restrict__ row, const float (&wt)[16], f32x4 acc) {
    const f32x4* r4 = reinterpret_cast<const f32x4*>(row);
#pragma unroll
    for (int q = 0; q < 4; ++q) {
        const f32x4 a = r4[q];
#pragma unroll
        for (int s = 0; s < 4; ++s) acc = mfma16(a[s], wt[4 * q + s], acc);
    }
    return acc;
}

// Forward pass of a tile whose input operands x[mt][s] (row 16 mt + c, input 7g + s) are in
// registers. h1, h2: this lane's activations (row 16 mt + 4g + i, column 16w + c), also in the LDS
// tiles sH1, sH2. Returns the outputs of m-tile w / 2, columns 16 (w % 2) + c (waves with w / 2 <
// MT). Ends without a barrier after the last read of sH2.
template <int MT>
__device__ __forceinline__ f32x4 net_forward(const float (&x)[MT][7], const FwdWeights& wt, float* sH1, float* sH2,
                                             int w, int g, int c, f32x4 (&h1)[MT], f32x4 (&h2)[MT]) {
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) {
        f32x4 acc = {wt.b1, wt.b1, wt.b1, wt.b1};
#pragma unroll
        for (int s = 0; s < 7; ++s) acc = mfma16(x[mt][s], wt.w1[s], acc);
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            h1[mt][i] = tanhf(acc[i]);
            sH1[(16 * mt + 4 * g + i) * kHS + 16 * w + c] = h1[mt][i];
        }
    }
    __syncthreads();
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) {
        f32x4 acc = {wt.b2, wt.b2, wt.b2, wt.b2};
        acc = hidden_product(sH1 + (16 * mt + c) * kHS + 16 * g, wt.w2, acc);
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            h2[mt][i] = tanhf(acc[i]);
            sH2[(16 * mt + 4 * g + i) * kHS + 16 * w + c] = h2[mt][i];
        }
    }
    __syncthreads();
    f32x4 y = {wt.b3, wt.b3, wt.b3, wt.b3};
    if (w / 2 < MT) y = hidden_product(sH2 + (16 * (w / 2) + c) * kHS + 16 * g, wt.w3, y);
    return y;
}

// Network on caller samples: X (n, 28) -> Y (n, 18). Bound by the matrix units (24 us at their
// peak), tanh and the barriers between the layers: 262144 samples in 68 us, against 282 us with
// one work-item per sample, FP32 vector products and the weights in LDS.
__global__ __launch_bounds__(kThreadsCl) void k_mlp_fwd(const float* __restrict__ X, long long n,
                                                        const float* __restrict__ P, float* __restrict__ Y) {
    constexpr int MT = 2;
    __shared__ __align__(16) float sH1[16 * MT * kHS], sH2[16 * MT * kHS];
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6, g = lane >> 4, c = lane & 15;
    FwdWeights wt;
    wt.load(P, w, g, c);
    const int col = 16 * (w & 1) + c;
    for (long long s0 = blockIdx.x * (16LL * MT); s0 < n; s0 += (long long)gridDim.x * (16 * MT)) {
        float x[MT][7];
#pragma unroll
        for (int mt = 0; mt < MT; ++mt) {
            const long long r = s0 + 16 * mt + c;
            const float* xr = X + (r < n ? r : n - 1) * kClIn + 7 * g;
#pragma unroll
            for (int s = 0; s < 7; ++s) x[mt][s] = xr[s];
        }
        f32x4 h1[MT], h2[MT];
        const f32x4 y = net_forward<MT>(x, wt, sH1, sH2, w, g, c, h1, h2);
        if (col < kClOut) {
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const long long r = s0 + 16 * (w / 2) + 4 * g + i;
                if (r < n) Y[r * kClOut + col] = y[i];
            }
        }
    }
}

// Gradient of the mean-squared-error loss L = sum (Y - T)^2 / (n 18) over the samples: forward,
// backward and the weight gradients of a tile in one work-group, the weight gradients kept as
// matrix accumulators over the work-group's tiles (no activation or delta reaches memory) and
// written once as its row of `part` (the gradient, then the squared error in FP64).
// A lane's own deltas are the B operand of the weight gradients (k-slot (g, (mt, i)) is row
// 16 mt + 4g + i), so only the A operands, the activations by column, are read from LDS. The sum
// over samples is fixed by n alone (tiles dealt to work-groups in turn, mlp_part_rows). Bound by
// the latency of the six products of a tile when a work-group has one tile: 4096 samples in 12.8
// us and the reduction in 4.2, against 3.1 ms for the separate forward, delta and weight-gradient
// kernels, whose weight gradients ran one work-item per weight over all samples; 262144 samples
// in 177 us against 128 ms.
template <int MT>
__global__ __launch_bounds__(kThreadsCl) void k_mlp_grad(const float* __restrict__ X, const float* __restrict__ T,
                                                         long long n, const float* __restrict__ P,
                                                         float* __restrict__ part) {
    __shared__ __align__(16) float sH1[16 * MT * kHS], sH2[16 * MT * kHS], sD2[16 * MT * kHS], sY[16 * MT * kYS];
    __shared__ float sB3[4][16];
    __shared__ double sE[4];
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6, g = lane >> 4, c = lane & 15;
    FwdWeights wt;
    wt.load(P, w, g, c);
    // the transposed layers: dH2 = dY W3^T (k = 5g + s of the outputs, 18 padded to 20),
    // dH1 = dZ2 W2^T (k = 16g + s)
    const float* W2 = P + kClIn * kClH + kClH;
    const float* W3 = W2 + kClH * kClH + kClH;
    float w3t[5], w2t[16];
#pragma unroll
    for (int s = 0; s < 5; ++s) {
        const int o = 5 * g + s;
        const float t = W3[(16 * w + c) * kClOut + (o < kClOut ? o : 0)];
        w3t[s] = o < kClOut ? t : 0.f;
    }
#pragma unroll
    for (int s = 0; s < 16; ++s) w2t[s] = W2[(16 * w + c) * kClH + 16 * g + s];
    const int col = 16 * (w & 1) + c, mq0 = 2 * (w >> 1);
    const float sc = 2.0f / (float)((double)n * kClOut);
    const f32x4 zero = {0.f, 0.f, 0.f, 0.f};
    f32x4 a1[2] = {zero, zero}, a2[4] = {zero, zero, zero, zero}, a3[2] = {zero, zero};
    float gb1 = 0.f, gb2 = 0.f, gb3 = 0.f;
    double err = 0.0;
    for (long long s0 = blockIdx.x * (16LL * MT); s0 < n; s0 += (long long)gridDim.x * (16 * MT)) {
        float x[MT][7];
#pragma unroll
        for (int mt = 0; mt < MT; ++mt) {
            const long long r = s0 + 16 * mt + c;
            const float* xr = X + (r < n ? r : n - 1) * kClIn + 7 * g;
#pragma unroll
            for (int s = 0; s < 7; ++s) x[mt][s] = xr[s];
        }
        f32x4 h1[MT], h2[MT];
        const f32x4 y = net_forward<MT>(x, wt, sH1, sH2, w, g, c, h1, h2);
        if (w / 2 < MT) {
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const int row = 16 * (w / 2) + 4 * g + i;
                const long long r = s0 + row;
                float dy = 0.f;
                if (r < n && col < kClOut) {
                    const float d = y[i] - T[r * kClOut + col];
                    err += (double)(d * d);
                    dy = sc * d;
                }
                gb3 += dy;
                sY[row * kYS + col] = dy;
            }
        }
        __syncthreads();
        f32x4 d2[MT], d1[MT];
#pragma unroll
        for (int mt = 0; mt < MT; ++mt) {
            f32x4 acc = zero;
            const float* yr = sY + (16 * mt + c) * kYS + 5 * g;
#pragma unroll
            for (int s = 0; s < 5; ++s) acc = mfma16(yr[s], w3t[s], acc);
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const int row = 16 * mt + 4 * g + i;
                d2[mt][i] = s0 + row < n ? acc[i] * (1.f - h2[mt][i] * h2[mt][i]) : 0.f;
                gb2 += d2[mt][i];
                sD2[row * kHS + 16 * w + c] = d2[mt][i];
            }
        }
        __syncthreads();
#pragma unroll
        for (int mt = 0; mt < MT; ++mt) {
            const f32x4 acc = hidden_product(sD2 + (16 * mt + c) * kHS + 16 * g, w2t, zero);
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                d1[mt][i] = s0 + 16 * mt + 4 * g + i < n ? acc[i] * (1.f - h1[mt][i] * h1[mt][i]) : 0.f;
                gb1 += d1[mt][i];
            }
        }
#pragma unroll
        for (int mt = 0; mt < MT; ++mt)
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const int row = 16 * mt + 4 * g + i;
                const long long r = s0 + row;
#pragma unroll
                for (int q = 0; q < 2; ++q) {
                    const int a = 16 * q + c;
                    const float xa = X[(r < n ? r : n - 1) * kClIn + (a < kClIn ? a : 0)];
                    a1[q] = mfma16(a < kClIn ? xa : 0.f, d1[mt][i], a1[q]);
                }
#pragma unroll
                for (int q = 0; q < 4; ++q) a2[q] = mfma16(sH1[row * kHS + 16 * q + c], d2[mt][i], a2[q]);
                const float dy = sY[row * kYS + col];
#pragma unroll
                for (int q = 0; q < 2; ++q) a3[q] = mfma16(sH2[row * kHS + 16 * (mq0 + q) + c], dy, a3[q]);
            }
        __syncthreads();  // the tile's activations are read before the next tile's are written
    }
    // the work-group's row: weights from the accumulators (row 4g + i, column c of a tile), biases
    // and the squared error summed over the lanes that share a column
    float* G = part + blockIdx.x * (long long)kClPart;
    float* gW2 = G + kClIn * kClH + kClH;
    float* gW3 = gW2 + kClH * kClH + kClH;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
#pragma unroll
        for (int q = 0; q < 2; ++q) {
            const int a = 16 * q + 4 * g + i;
            if (a < kClIn) G[a * kClH + 16 * w + c] = a1[q][i];
            if (col < kClOut) gW3[(16 * (mq0 + q) + 4 * g + i) * kClOut + col] = a3[q][i];
        }
#pragma unroll
        for (int q = 0; q < 4; ++q) gW2[(16 * q + 4 * g + i) * kClH + 16 * w + c] = a2[q][i];
    }
#pragma unroll
    for (int o = 16; o < 64; o <<= 1) {
        gb1 += __shfl_xor(gb1, o);
        gb2 += __shfl_xor(gb2, o);
        gb3 += __shfl_xor(gb3, o);
    }
    for (int o = 1; o < 64; o <<= 1) err += __shfl_xor(err, o);
    if (g == 0) {
        G[kClIn * kClH + 16 * w + c] = gb1;
        gW2[kClH * kClH + 16 * w + c] = gb2;
        sB3[w][c] = gb3;
    }
    if (lane == 0) sE[w] = err;
    __syncthreads();
    if (threadIdx.x < kClOut) {
        const int t = threadIdx.x;
        gW3[kClH * kClOut + t] = sB3[t >> 4][t & 15] + sB3[2 + (t >> 4)][t & 15];
    }
    if (threadIdx.x == 0) *(double*)(G + kClNParam) = (sE[0] + sE[1]) + (sE[2] + sE[3]);
}

// Sum of the `rows` rows of `part` in a fixed order (8 interleaved sums of a column, then their
// sum), 32 columns per block: the gradient into G (if set); with m and v, the Adam update of P from
// the same sums, so a training step is two launches and the gradient need not reach memory. The last
// block adds the squared error, in FP64 as the rows hold it, and rounds it once, times loss_scale,
// into loss.
__global__ __launch_bounds__(kThreadsCl) void k_mlp_reduce(const float* __restrict__ part, int rows,
                                                           float* __restrict__ G, float* __restrict__ loss,
                                                           double loss_scale, float* __restrict__ P,
                                                           float* __restrict__ m, float* __restrict__ v, float lr,
                                                           float b1t, float b2t) {
    if (blockIdx.x == gridDim.x - 1) {
        __shared__ double se[kThreadsCl / 64];
        double e = 0.0;
        for (int r = threadIdx.x; r < rows; r += kThreadsCl) e += *(const double*)(part + r * (long long)kClPart + kClNParam);
        for (int o = 1; o < 64; o <<= 1) e += __shfl_xor(e, o);
        if ((threadIdx.x & 63) == 0) se[threadIdx.x >> 6] = e;
        __syncthreads();
        if (loss && threadIdx.x == 0) loss[0] = (float)(((se[0] + se[1]) + (se[2] + se[3])) * loss_scale);
        return;
    }
    __shared__ float s[8][32];
    const int cx = threadIdx.x & 31, ry = threadIdx.x >> 5;
    const int i = blockIdx.x * 32 + cx;
    float a = 0.f;
    if (i < kClNParam) {
#pragma unroll 8
        for (int r = ry; r < rows; r += 8) a += part[r * (long long)kClPart + i];
    }
    s[ry][cx] = a;
    __syncthreads();
    if (ry != 0 || i >= kClNParam) return;
    const float g = ((s[0][cx] + s[1][cx]) + (s[2][cx] + s[3][cx])) + ((s[4][cx] + s[5][cx]) + (s[6][cx] + s[7][cx]));
    if (G) G[i] = g;
    if (m) {
        const float b1 = 0.9f, b2 = 0.999f, eps = 1e-8f;
        const float mi = b1 * m[i] + (1.f - b1) * g;
        const float vi = b2 * v[i] + (1.f - b2) * g * g;
        m[i] = mi;
        v[i] = vi;
        const float mh = mi / (1.f - b1t), vh = vi / (1.f - b2t);
        P[i] -= lr * mh / (sqrtf(vh) + eps);
    }
}

// ---------------------------------------------------------------- closure terms

// Features, network and correction fields of a step in one kernel: the 28 features are formed from
// the real state S in LDS, and of the outputs only the 12 real fields the step transforms reach
// memory (and the 18 outputs Y where the caller asks for them). Correction fields:
// C[0..5] = momentum flux tau_ij = R_ij - M_ij + delta_ij q (xx, xy, xz, yy,
// yz, zz), C[6..8] = EMF correction, C[9..11] = energy-flux correction. q is
// the subgrid part of the total pressure p + B^2/2 with
// p = (gamma-1)(e - rho u.u/2 - B^2/2): q = -(gamma-1)/2 (tr R + tr M) + tr M / 2.
// At 64^3: 68 us, against 21 + 229 + 9 us for the feature, network and term kernels. Held to 128
// registers (40 bytes spilled) for four work-groups per CU; uncapped it holds 144, three, and the
// last quarter of the 1024 work-groups waits.
__global__ __launch_bounds__(kThreadsCl, 4) void k_cl_net(const double* __restrict__ S, int nx, int ny, int nz,
                                                       double dx, double dy, double dz,
                                                       const float* __restrict__ P, double gamma,
                                                       float* __restrict__ Y, double* __restrict__ C) {
    constexpr int MT = 2, TS = 16 * MT;
    constexpr int YD = 19;  // row stride of the outputs in LDS (FP64, physical units)
    __shared__ __align__(16) float sH1[TS * kHS], sH2[TS * kHS], sX[TS * kXS];
    __shared__ double sY[TS * YD];
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6, g = lane >> 4, c = lane & 15;
    FwdWeights wt;
    wt.load(P, w, g, c);
    const float* norm = P + kClNParam;
    const float* ystd = norm + 2 * kClIn;
    const long long N = (long long)nx * ny * nz;
    // features: a work-item takes point m of the tile and one kind (the value or the derivative
    // along one axis) of fields 0-3 or 4-6 of rho, u, B (S[0], S[8..10], S[4..6]); a tile's loads
    // are issued while the network of the tile before it runs
    const int m = threadIdx.x & 31, kind = (threadIdx.x >> 5) & 3, half = threadIdx.x >> 7;
    const double d2 = 2.0 * (kind == 1 ? dx : (kind == 2 ? dy : dz));
    const int col = 16 * (w & 1) + c;
    const double ys = col < kClOut ? (double)ystd[col] : 0.0;
    const double* f0[4];
    float mean[4], sd[4];
    int xk[4];
#pragma unroll
    for (int t = 0; t < 4; ++t) {
        const int q = half ? (t < 3 ? 4 + t : 6) : t;  // the last slot of the upper half repeats field 6
        const int fld = half ? (t < 3 ? 4 + t : 6) : (t == 0 ? 0 : 7 + t);
        f0[t] = S + fld * N;
        xk[t] = kind == 0 ? q : 6 + 3 * q + kind;
        mean[t] = norm[xk[t]];
        sd[t] = norm[kClIn + xk[t]];
    }
    double fp[4], fm[4];
    auto fetch = [&](long long s0) {
        const long long i = s0 + m < N ? s0 + m : N - 1;
        const long long sy = nx, sz = (long long)nx * ny;
        long long ip = i, im = i;
        if (kind == 1) {
            const int ix = (int)((unsigned)i % (unsigned)nx);  // N < 2^31 on the supported grids
            ip = ix + 1 == nx ? i - (nx - 1) : i + 1;
            im = ix == 0 ? i + (nx - 1) : i - 1;
        } else if (kind == 2) {
            const int iy = (int)((unsigned)i / (unsigned)nx % (unsigned)ny);
            ip = iy + 1 == ny ? i - (ny - 1) * sy : i + sy;
            im = iy == 0 ? i + (ny - 1) * sy : i - sy;
        } else if (kind == 3) {
            const int iz = (int)((unsigned)i / (unsigned)sz);
            ip = iz + 1 == nz ? i - (nz - 1) * sz : i + sz;
            im = iz == 0 ? i + (nz - 1) * sz : i - sz;
        }
#pragma unroll
        for (int t = 0; t < 4; ++t) {
            fp[t] = f0[t][ip];
            fm[t] = f0[t][im];
        }
    };
    const long long step = (long long)gridDim.x * TS;
    long long s0 = blockIdx.x * (long long)TS;
    if (s0 < N) fetch(s0);
    for (; s0 < N; s0 += step) {
#pragma unroll
        for (int t = 0; t < 4; ++t) {
            const float v = kind == 0 ? (float)fp[t] : (float)((fp[t] - fm[t]) / d2);  // as k_cl_features has it
            sX[m * kXS + xk[t]] = (v - mean[t]) / sd[t];
        }
        if (s0 + step < N) fetch(s0 + step);
        __syncthreads();
        float x[MT][7];
#pragma unroll
        for (int mt = 0; mt < MT; ++mt)
#pragma unroll
            for (int s = 0; s < 7; ++s) x[mt][s] = sX[(16 * mt + c) * kXS + 7 * g + s];
        f32x4 h1[MT], h2[MT];
        const f32x4 y = net_forward<MT>(x, wt, sH1, sH2, w, g, c, h1, h2);
        if (col < kClOut) {
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const int r = 16 * (w / 2) + 4 * g + i;
                sY[r * YD + col] = (double)y[i] * ys;
                if (Y && s0 + r < N) Y[(s0 + r) * kClOut + col] = y[i];
            }
        }
        __syncthreads();
        if (C && s0 + m < N) {
            // a work-item forms field f of its point, and field f + 8 of those that have one
            const double* o = sY + m * YD;
            const int f = threadIdx.x >> 5;
            double v;
            if (f < 6) {
                v = o[f] - o[6 + f];
                if (f == 0 || f == 3 || f == 5) {
                    const double trR = o[0] + o[3] + o[5], trM = o[6] + o[9] + o[11];
                    v += -0.5 * (gamma - 1.0) * (trR + trM) + 0.5 * trM;
                }
            } else {
                v = o[6 + f];
            }
            C[f * N + s0 + m] = v;
            if (f < 4) C[(f + 8) * N + s0 + m] = o[f + 14];
        }
    }
}

// Spectral right-hand side of the correction fields (spectra Ch on a box of nky x nkz rows of
// stride rs, the full spectrum or the kept box, FP64, 12 fields): momentum_i -= i k'_j tau_ij (as calc_rhs does for
// the resolved momentum flux, mhdrhs.f90:206-222), B -= i k' x E (the
// induction term of the electric field E, mhdrhs.f90:224-233) and e -= i k'.F
// (the energy flux, mhdrhs.f90:234-236). Out: 7 fields, momentum x, y, z, B x,
// y, z, energy.
__global__ void k_cl_rhs(const cpx<double>* __restrict__ Ch, long long M, int rs, int nkx, int nky,
                         const double* __restrict__ wx, const double* __restrict__ wy, const double* __restrict__ wz,
                         cpx<double>* __restrict__ R) {
    const long long i = blockIdx.x * (long long)blockDim.x + threadIdx.x;
    if (i >= M) return;
    const int kx = (int)(i % rs);
    if (kx >= nkx) return;  // row padding
    const int iy = (int)((i / rs) % nky);
    const int iz = (int)(i / ((long long)rs * nky));
    const double k[3] = {wx[kx], wy[iy], wz[iz]};
    auto t = [&](int a, int b) {
        const int idx[3][3] = {{0, 1, 2}, {1, 3, 4}, {2, 4, 5}};
        return Ch[idx[a][b] * M + i];
    };
    // -i * (k . v) for complex v: -i (x + iy) = y - ix
#pragma unroll
    for (int a = 0; a < 3; ++a) {
        double sx = 0.0, sy = 0.0;
#pragma unroll
        for (int b = 0; b < 3; ++b) {
            const cpx<double> v = t(a, b);
            sx += k[b] * v.x;
            sy += k[b] * v.y;
        }
        R[a * M + i] = cpx<double>{sy, -sx};
    }
    const cpx<double> E[3] = {Ch[6 * M + i], Ch[7 * M + i], Ch[8 * M + i]};
#pragma unroll
    for (int a = 0; a < 3; ++a) {
        const int b = (a + 1) % 3, c = (a + 2) % 3;
        const double sx = k[b] * E[c].x - k[c] * E[b].x, sy = k[b] * E[c].y - k[c] * E[b].y;
        R[(3 + a) * M + i] = cpx<double>{sy, -sx};
    }
    double sx = 0.0, sy = 0.0;
#pragma unroll
    for (int b = 0; b < 3; ++b) {
        const cpx<double> v = Ch[(9 + b) * M + i];
        sx += k[b] * v.x;
        sy += k[b] * v.y;
    }
    R[6 * M + i] = cpx<double>{sy, -sx};
}

// ---------------------------------------------------------------- training data

// Box filter of a fine state and of its flux products, one work-item per coarse cell (mean over
// r^3 fine cells): out[q][coarse cell], q = 0..7 rho, m x y z, B x y z, e; 8..13 m_i u_j and
// 14..19 B_i B_j (xx, xy, xz, yy, yz, zz); 20..22 E = -u x B + (d_i/rho) J x B; 23..25 the
// energy flux (e + p + B^2/2) u - (u.B) B (mhdrhs.f90:60-119). S = [uu(8), uu_prim(4)] and J
// (3 fields) are the fine real fields, FP64.
__global__ void k_cl_filter(const double* __restrict__ S, const double* __restrict__ J, int nx, int ny, int nz, int r,
                            double di, double* __restrict__ out) {
    const int cx = nx / r, cy = ny / r, cz = nz / r;
    const long long Nc = (long long)cx * cy * cz;
    const long long ic = blockIdx.x * (long long)blockDim.x + threadIdx.x;
    if (ic >= Nc) return;
    const int x0 = (int)(ic % cx) * r, y0 = (int)((ic / cx) % cy) * r, z0 = (int)(ic / ((long long)cx * cy)) * r;
    const long long N = (long long)nx * ny * nz;
    double acc[kClFilt];
#pragma unroll
    for (int q = 0; q < kClFilt; ++q) acc[q] = 0.0;
    const int pr[6][2] = {{0, 0}, {0, 1}, {0, 2}, {1, 1}, {1, 2}, {2, 2}};
    for (int dz = 0; dz < r; ++dz)
        for (int dy = 0; dy < r; ++dy)
            for (int dx = 0; dx < r; ++dx) {
                const long long i = ((long long)(z0 + dz) * ny + (y0 + dy)) * nx + (x0 + dx);
                double w[8], u[3], b[3], j[3];
#pragma unroll
                for (int q = 0; q < 8; ++q) w[q] = S[q * N + i];
#pragma unroll
                for (int a = 0; a < 3; ++a) {
                    u[a] = S[(8 + a) * N + i];
                    b[a] = w[4 + a];
                    j[a] = J[a * N + i];
                }
                const double p = S[11 * N + i], rho = w[0];
#pragma unroll
                for (int q = 0; q < 8; ++q) acc[q] += w[q];
#pragma unroll
                for (int c = 0; c < 6; ++c) {
                    acc[8 + c] += w[1 + pr[c][0]] * u[pr[c][1]];
                    acc[14 + c] += b[pr[c][0]] * b[pr[c][1]];
                }
                const double h = di / rho;
                const double ub = u[0] * b[0] + u[1] * b[1] + u[2] * b[2];
                const double et = w[7] + p + 0.5 * (b[0] * b[0] + b[1] * b[1] + b[2] * b[2]);
#pragma unroll
                for (int a = 0; a < 3; ++a) {
                    const int s = (a + 1) % 3, t = (a + 2) % 3;
                    acc[20 + a] += -(u[s] * b[t] - u[t] * b[s]) + h * (j[s] * b[t] - j[t] * b[s]);
                    acc[23 + a] += et * u[a] - ub * b[a];
                }
            }
    const double inv = 1.0 / ((double)r * r * r);
#pragma unroll
    for (int q = 0; q < kClFilt; ++q) out[q * Nc + ic] = acc[q] * inv;
}

// One field q of the 26 of k_cl_filter (same numbering and formulas) at every fine point, not
// averaged: the input of the spectral (sharp cut-off) filter, one transform per field. Only the
// inputs field q needs are read.
__global__ void k_cl_point(const double* __restrict__ S, const double* __restrict__ J, long long N, int q, double di,
                           double* __restrict__ out) {
    const int pr[6][2] = {{0, 0}, {0, 1}, {0, 2}, {1, 1}, {1, 2}, {2, 2}};
    for (long long i = blockIdx.x * (long long)blockDim.x + threadIdx.x; i < N; i += (long long)gridDim.x * blockDim.x) {
        double v;
        if (q < 8) {
            v = S[q * N + i];
        } else if (q < 14) {
            v = S[(1 + pr[q - 8][0]) * N + i] * S[(8 + pr[q - 8][1]) * N + i];            // m_i u_j
        } else if (q < 20) {
            v = S[(4 + pr[q - 14][0]) * N + i] * S[(4 + pr[q - 14][1]) * N + i];          // B_i B_j
        } else if (q < 23) {
            const int a = q - 20, s1 = (a + 1) % 3, t1 = (a + 2) % 3;
            const double us = S[(8 + s1) * N + i], ut = S[(8 + t1) * N + i];
            const double bs = S[(4 + s1) * N + i], bt = S[(4 + t1) * N + i];
            const double h = di / S[i];
            v = -(us * bt - ut * bs) + h * (J[s1 * N + i] * bt - J[t1 * N + i] * bs);   // E = -u x B + (d_i/rho) J x B
        } else {
            const int a = q - 23;
            double u[3], b[3];
#pragma unroll
            for (int c = 0; c < 3; ++c) {
                u[c] = S[(8 + c) * N + i];
                b[c] = S[(4 + c) * N + i];
            }
            const double ub = u[0] * b[0] + u[1] * b[1] + u[2] * b[2];
            const double et = S[7 * N + i] + S[11 * N + i] + 0.5 * (b[0] * b[0] + b[1] * b[1] + b[2] * b[2]);
            v = et * u[a] - ub * b[a];                                                   // energy flux
        }
        out[i] = v;
    }
}

// Sharp spectral cut-off between a fine and a coarse full spectrum (layout [z][y][KXP] with kx
// fastest): the modes with kx < nxc/2, |my| < nyc/2 and |mz| < nzc/2 (signed; the coarse
// Nyquist rows are dropped, so the cut is the same for +k and -k). dir > 0: gather into the
// coarse spectrum C (zero outside the cut); dir < 0: scatter C into the fine spectrum F (the
// caller zeroes F first).
__global__ void k_spec_cut(cpx<double>* __restrict__ F, int nyf, int nzf, int kxpf, cpx<double>* __restrict__ C,
                           int nxc, int nyc, int nzc, int kxpc, int dir) {
    const long long Mc = (long long)kxpc * nyc * nzc;
    for (long long i = blockIdx.x * (long long)blockDim.x + threadIdx.x; i < Mc; i += (long long)gridDim.x * blockDim.x) {
        const int kx = (int)(i % kxpc);
        const int ky = (int)((i / kxpc) % nyc);
        const int kz = (int)(i / ((long long)kxpc * nyc));
        const int my = ky <= nyc / 2 ? ky : ky - nyc;
        const int mz = kz <= nzc / 2 ? kz : kz - nzc;
        const bool kept = kx < nxc / 2 && 2 * my < nyc && -2 * my < nyc && 2 * mz < nzc && -2 * mz < nzc;
        const long long f =
            kept ? ((long long)(mz >= 0 ? mz : nzf + mz) * nyf + (my >= 0 ? my : nyf + my)) * kxpf + kx : 0;
        if (dir > 0) C[i] = kept ? F[f] : cpx<double>{0.0, 0.0};
        else if (kept) F[f] = C[i];
    }
}

// ---------------------------------------------------------------- launchers

static unsigned blocks_for(long long n) { return (unsigned)((n + kThreadsCl - 1) / kThreadsCl); }

hipError_t launch_cl_features(const double* S, int nx, int ny, int nz, double dx, double dy, double dz,
                              const float* norm, float* X, hipStream_t s) {
    const long long N = (long long)nx * ny * nz;
    hipLaunchKernelGGL(k_cl_features, dim3(blocks_for(N)), dim3(kThreadsCl), 0, s, S, nx, ny, nz, dx, dy, dz, norm,
                       X);
    return hipGetLastError();
}

hipError_t launch_cl_point(const double* S, const double* J, long long N, int q, double di, double* out,
                           hipStream_t s) {
    const long long nb = blocks_for(N) < 65536 ? blocks_for(N) : 65536;
    hipLaunchKernelGGL(k_cl_point, dim3((unsigned)nb), dim3(kThreadsCl), 0, s, S, J, N, q, di, out);
    return hipGetLastError();
}

hipError_t launch_spec_cut(cpx<double>* F, int nyf, int nzf, int kxpf, cpx<double>* C, int nxc, int nyc, int nzc,
                           int kxpc, int dir, hipStream_t s) {
    const long long Mc = (long long)kxpc * nyc * nzc;
    const long long nb = blocks_for(Mc) < 65536 ? blocks_for(Mc) : 65536;
    hipLaunchKernelGGL(k_spec_cut, dim3((unsigned)nb), dim3(kThreadsCl), 0, s, F, nyf, nzf, kxpf, C, nxc, nyc, nzc,
                       kxpc, dir);
    return hipGetLastError();
}

hipError_t launch_cl_filter(const double* S, const double* J, int nx, int ny, int nz, int r, double di, double* out,
                            hipStream_t s) {
    const long long Nc = (long long)(nx / r) * (ny / r) * (nz / r);
    hipLaunchKernelGGL(k_cl_filter, dim3(blocks_for(Nc)), dim3(kThreadsCl), 0, s, S, J, nx, ny, nz, r, di, out);
    return hipGetLastError();
}

hipError_t launch_mlp_fwd(const float* X, long long n, const float* P, float* Y, hipStream_t s) {
    const long long nt = (n + 31) / 32;
    hipLaunchKernelGGL(k_mlp_fwd, dim3((unsigned)(nt < 1024 ? nt : 1024)), dim3(kThreadsCl), 0, s, X, n, P, Y);
    return hipGetLastError();
}

// Samples per tile: 16 while that gives each of the 256 CUs at most one tile (4096 samples: 12.8
// us, half of a 32-sample tile's chain of products), 32 above (half the partial rows and weight
// reads per sample: 8192 samples in 15.2 us).
static int mlp_tile(long long n) { return n <= 16LL * 256 ? 16 : 32; }

// Rows of partial sums k_mlp_grad writes for n samples: one per work-group, at most one
// work-group per CU up to LAPS_MLP_NOALLOC_MAX samples and two per CU beyond.
int mlp_part_rows(long long n) {
    const int t = mlp_tile(n);
    const long long tiles = (n + t - 1) / t;
    return (int)(tiles < 512 ? tiles : 512);
}

static hipError_t launch_partials(const float* X, const float* T, long long n, const float* P, float* part,
                                  hipStream_t s) {
    const dim3 grid((unsigned)mlp_part_rows(n));
    if (mlp_tile(n) == 16)
        hipLaunchKernelGGL((k_mlp_grad<1>), grid, dim3(kThreadsCl), 0, s, X, T, n, P, part);
    else
        hipLaunchKernelGGL((k_mlp_grad<2>), grid, dim3(kThreadsCl), 0, s, X, T, n, P, part);
    return hipGetLastError();
}

// Gradient of the loss over n samples into G (kClNParam) and the mean squared error into loss[0]
// (may be null); part holds mlp_part_rows(n) * kClPart floats, 8-byte aligned.
hipError_t launch_mlp_grad(const float* X, const float* T, long long n, const float* P, float* part, float* G,
                           float* loss, hipStream_t s) {
    hipError_t e = launch_partials(X, T, n, P, part, s);
    if (e != hipSuccess) return e;
    hipLaunchKernelGGL(k_mlp_reduce, dim3((kClNParam + 31) / 32 + 1), dim3(kThreadsCl), 0, s, part, mlp_part_rows(n), G,
                       loss, 1.0 / ((double)n * kClOut), nullptr, nullptr, nullptr, 0.f, 0.f, 0.f);
    return hipGetLastError();
}

// One Adam step of P on n samples (m, v: the moments; b1t, b2t: the powers of the betas); the mean
// squared error before the step into loss[0].
hipError_t launch_mlp_train_step(const float* X, const float* T, long long n, float* P, float* part, float* m,
                                 float* v, float* loss, float lr, float b1t, float b2t, hipStream_t s) {
    hipError_t e = launch_partials(X, T, n, P, part, s);
    if (e != hipSuccess) return e;
    hipLaunchKernelGGL(k_mlp_reduce, dim3((kClNParam + 31) / 32 + 1), dim3(kThreadsCl), 0, s, part, mlp_part_rows(n), nullptr,
                       loss, 1.0 / ((double)n * kClOut), P, m, v, lr, b1t, b2t);
    return hipGetLastError();
}

hipError_t launch_cl_net(const double* S, int nx, int ny, int nz, double dx, double dy, double dz, const float* P,
                         double gamma, float* Y, double* C, hipStream_t s) {
    const long long nt = ((long long)nx * ny * nz + 31) / 32;
    hipLaunchKernelGGL(k_cl_net, dim3((unsigned)(nt < 1024 ? nt : 1024)), dim3(kThreadsCl), 0, s, S, nx, ny, nz,
                       dx, dy, dz, P, gamma, Y, C);
    return hipGetLastError();
}

hipError_t launch_cl_rhs(const cpx<double>* Ch, const Box& b, BoxTables t, cpx<double>* R, hipStream_t s) {
    hipLaunchKernelGGL(k_cl_rhs, dim3(blocks_for(b.modes())), dim3(kThreadsCl), 0, s, Ch, b.modes(), b.KXP, b.KX, b.CY,
                       t.wx, t.wy, t.wz, R);
    return hipGetLastError();
}

}  // namespace laps
