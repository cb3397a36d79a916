// Learned closure for coarse (p = 1 Legendre) periodic-box runs: per-element
// features and training targets, a small MLP (70 -> 128 -> 128 -> 40, GELU,
// BF16 weights with FP32 accumulation) with its own forward, backward and
// Adam kernels, and RK4 stepping of the coarse solver with the corrected
// tendency dU/dt = M^-1 R(U) + C(U).  No reference counterpart.
#include "dg_amd.h"

#include <hip/hip_runtime.h>

#include <mutex>

#include <cmath>
#include <cstddef>
#include <cstdint>
#include <cstring>
#include <random>
#include <sstream>
#include <stdexcept>
#include <string>
#include <type_traits>
#include <vector>

#include "dg_solver_impl.hpp"

namespace {

constexpr int NF = 70, NH = 128, NO = 40;      // features, hidden width, outputs
constexpr int NP = NF * NH + NH + NH * NH + NH + NH * NO + NO;
constexpr int OFF_W1 = 0, OFF_B1 = NF * NH, OFF_W2 = OFF_B1 + NH, OFF_B2 = OFF_W2 + NH * NH;
constexpr int OFF_W3 = OFF_B2 + NH, OFF_B3 = OFF_W3 + NH * NO;
constexpr int TB = 256;

struct ClosureError : std::runtime_error {
    using std::runtime_error::runtime_error;
};

void hcheck(hipError_t e, const char* what) {
    if (e != hipSuccess) {
        std::ostringstream o;
        o << what << ": " << hipGetErrorString(e);
        throw ClosureError(o.str());
    }
}

unsigned nblk(long n) { return (unsigned)((n + TB - 1) / TB); }

// ---------------------------------------------------------------------------
// bf16 storage (round to nearest even), FP32 arithmetic
// ---------------------------------------------------------------------------
__host__ __device__ inline uint16_t to_bf16(float f) {
    uint32_t u;
    std::memcpy(&u, &f, 4);
    u += 0x7fffu + ((u >> 16) & 1u);
    return (uint16_t)(u >> 16);
}

__device__ inline float gelu(float z) { return 0.5f * z * (1.0f + erff(z * 0.70710678118654752f)); }
// gelu(z), and its derivative in d
__device__ inline float gelu_both(float z, float& d) {
    const float e = 1.0f + erff(z * 0.70710678118654752f);
    d = 0.5f * e + z * 0.39894228040143268f * expf(-0.5f * z * z);
    return 0.5f * z * e;
}

// Gaussian jitter of the mini-batch features, noise standard deviations in
// normalised units (raw units: noise / scale); counter-based hash RNG
// (splitmix64) and the Box-Muller transform
__device__ inline unsigned long long mix64(unsigned long long z) {
    z += 0x9e3779b97f4a7c15ull;
    z = (z ^ (z >> 30)) * 0xbf58476d1ce4e5b9ull;
    z = (z ^ (z >> 27)) * 0x94d049bb133111ebull;
    return z ^ (z >> 31);
}
__device__ inline float jitter(float noise, float scale, unsigned long long t, unsigned long long key) {
    const unsigned long long h = mix64(key ^ mix64(t));
    const float u1 = ((float)(h >> 40) + 0.5f) * (1.0f / 16777216.0f);
    const float u2 = ((float)((h >> 16) & 0xffffffu) + 0.5f) * (1.0f / 16777216.0f);
    const float g = sqrtf(-2.0f * logf(u1)) * cosf(6.283185307179586f * u2);
    return noise * g / scale;
}

__global__ void to_bf16_kernel(const float* __restrict__ p, uint16_t* __restrict__ pb, int n) {
    const int i = blockIdx.x * TB + threadIdx.x;
    if (i < n) pb[i] = to_bf16(p[i]);
}

// ---------------------------------------------------------------------------
// Coarse-state features and targets (p = 1 Legendre periodic box)
// ---------------------------------------------------------------------------

// face mean of element block u (8 x 5) on face (d, side), variable s:
// (1/4) sum_ab w_a w_b U(face point (a, b)) on the (p+2) = 3-point rule,
// factored as sum_b u_b phi_r(+-1) m_t1 m_t2 with the basis means
// m_j = (1/2) sum_a w_a phi_j(x_a)
__device__ double face_mean(const dg::KTables& T, const double* m, const double* u, int d, int side, int s) {
    const double* phi = side ? T.phip : T.phim;
    double acc = 0.;
    for (int k = 0; k < 2; ++k)
        for (int j = 0; j < 2; ++j)
            for (int i = 0; i < 2; ++i) {
                const int b = i + 2 * j + 4 * k;
                const int r = d == 0 ? i : (d == 1 ? j : k);
                const int t1 = d == 0 ? j : i, t2 = d == 2 ? j : k;
                acc = fma(u[b * 5 + s], phi[r] * m[t1] * m[t2], acc);
            }
    return acc;
}

// X[e] = own 40 coefficients, then for the faces x-, x+, y-, y+, z-, z+ the
// jump of the face-mean state (neighbour's matching face minus own), 5
// each.  32 threads per element (32-bit index arithmetic: E 32 < 2^32):
// all copy the 40 coefficients, threads 0..29 then take the 30 jumps
constexpr int FT = 32;
__global__ void features_kernel(const double* __restrict__ U, float* __restrict__ X,
                                const dg::KTables* __restrict__ Tp, dg::KGeom G) {
    const unsigned t = blockIdx.x * TB + threadIdx.x;
    const unsigned e = t / FT, q = t % FT;
    if (e >= G.E) return;
    const double* u = U + (size_t)e * 40;
    float* x = X + (size_t)e * NF;
    x[q] = (float)u[q];
    if (q < 40 - FT) x[FT + q] = (float)u[FT + q];
    if (q >= 30) return;
    const int c = 40 + (int)q;
    const dg::KTables& T = *Tp;
    double m[2];
    for (int jj = 0; jj < 2; ++jj) {
        double a = 0.;
        for (int g = 0; g < 3; ++g) a += T.w[g] * T.B[g][jj];
        m[jj] = 0.5 * a;
    }
    const int f = (c - 40) / 5, s = (c - 40) % 5, d = f >> 1, side = f & 1;
    const unsigned nx = G.ne[0], ny = G.ne[1], nz = G.ne[2];
    const unsigned eyz = e / nx;
    unsigned cc[3] = {e - eyz * nx, eyz % ny, eyz / ny};
    const unsigned nd = d == 0 ? nx : (d == 1 ? ny : nz);
    cc[d] = side ? (cc[d] + 1 == nd ? 0u : cc[d] + 1) : (cc[d] == 0 ? nd - 1 : cc[d] - 1);
    const unsigned en = cc[0] + nx * (cc[1] + ny * cc[2]);
    x[c] = (float)(face_mean(T, m, U + (size_t)en * 40, d, 1 - side, s) - face_mean(T, m, u, d, side, s));
}

// coarse state = Legendre modes (i, j, k) <= 1 of the fine state (the L2
// projection onto p = 1 for an orthogonal basis on affine elements)
__global__ void truncate_kernel(const double* __restrict__ Uf, double* __restrict__ Uc, int Pf, long E) {
    const long t = (long)blockIdx.x * TB + threadIdx.x;
    if (t >= E * 40) return;
    const long e = t / 40;
    const int r = (int)(t % 40), b = r / 5, s = r % 5;
    const int i = b & 1, j = (b >> 1) & 1, k = b >> 2, n = Pf + 1;
    Uc[t] = Uf[(e * n * n * n + i + n * j + n * n * k) * 5 + s];
}

// Y = trunc(Df) - Dc, in FP32
__global__ void target_kernel(const double* __restrict__ Df, const double* __restrict__ Dc, float* __restrict__ Y,
                              int Pf, long E) {
    const long t = (long)blockIdx.x * TB + threadIdx.x;
    if (t >= E * 40) return;
    const long e = t / 40;
    const int r = (int)(t % 40), b = r / 5, s = r % 5;
    const int i = b & 1, j = (b >> 1) & 1, k = b >> 2, n = Pf + 1;
    Y[t] = (float)(Df[(e * n * n * n + i + n * j + n * n * k) * 5 + s] - Dc[t]);
}

// Fused inference for the closure step and dg_mlp_forward, on the matrix
// cores: v_mfma_f32_16x16x16_bf16 tiles (bf16 operands, FP32 accumulation)
// for the three layers, with the normalisation, GELU, de-normalisation and
// the fallback bound around them.  The grid is persistent (at most one
// block per CU): a block stages the three weight matrices once, transposed
// to [output][input] in LDS, then walks tiles of 16 rows per wave; a wave
// takes its rows through all three layers by itself.  Activations enter each
// layer rounded to bf16.
//
// Operand layout of the 16x16x16 bf16 MFMA (lane l, element q = 0..3):
// A[l % 16][4 (l / 16) + q], B[4 (l / 16) + q][l % 16]; the result lane l
// holds D[4 (l / 16) + q][l % 16].
typedef short bf16x4 __attribute__((ext_vector_type(4)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
constexpr int K1 = 80;                         // layer-1 inputs padded to whole 16-wide k steps
constexpr int L1S = K1 + 4, L2S = NH + 4;      // LDS row strides (bf16), padded off the bank period
constexpr int N3 = 48;                         // layer-3 outputs padded to whole 16-column tiles
constexpr int WV = 64;                         // lanes per wave
constexpr int MAX_INFER_BLOCKS = 256;          // a block per CU
constexpr int GCHUNKS = 32;                   // most row chunks of one weight-gradient pass

// WN pairs of waves with 16 rows each; the rows hold the features, then each
// layer's activations and the de-normalised outputs in place
template <int WN>
struct InferLDS {
    uint16_t w1[NH][L1S];                      // W1^T; inputs k >= NF are zero
    uint16_t w2[NH][L2S];                      // W2^T
    uint16_t w3[N3][L2S];                      // W3^T; outputs n >= NO are zero
    uint16_t a[16 * WN][L2S];
};

__device__ inline bf16x4 ld_bf16x4(const uint16_t* q) { return *reinterpret_cast<const bf16x4*>(q); }

// The weights' LDS image (w1, w2, w3 of InferLDS, contiguous) in global
// memory, built once per change of the bf16 weights: element i of the image
// is W1^T / W2^T / W3^T at (row, column) with the padding zero
constexpr int IMG1 = NH * L1S, IMG2 = NH * L2S, IMG3 = N3 * L2S, IMG = IMG1 + IMG2 + IMG3;

__global__ void pack_infer_weights(const uint16_t* __restrict__ W, uint16_t* __restrict__ img) {
    const int i = blockIdx.x * TB + threadIdx.x;
    if (i >= IMG) return;
    uint16_t v = 0;
    if (i < IMG1) {
        const int n = i / L1S, k = i % L1S;
        if (k < NF) v = W[OFF_W1 + k * NH + n];
    } else if (i < IMG1 + IMG2) {
        const int n = (i - IMG1) / L2S, k = (i - IMG1) % L2S;
        if (k < NH) v = W[OFF_W2 + k * NH + n];
    } else {
        const int n = (i - IMG1 - IMG2) / L2S, k = (i - IMG1 - IMG2) % L2S;
        if (n < NO && k < NH) v = W[OFF_W3 + k * NO + n];
    }
    img[i] = v;
}

// acc[j] += A[16 rows][K] x W^T[16 j .. 16 j + 15][K] for j < NT
// W^T from the rows of the first tile on
template <int NT, int K, int LA, int LW>
__device__ __forceinline__ void mfma_layer(const uint16_t (*A)[LA], const uint16_t (*Wt)[LW], int lane, f32x4* acc) {
    const int c = lane & 15, kq = 4 * (lane >> 4);
#pragma unroll 2
    for (int kk = 0; kk < K; kk += 16) {
        const bf16x4 a = ld_bf16x4(&A[c][kk + kq]);
#pragma unroll
        for (int j = 0; j < NT; ++j)
            acc[j] = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(a, ld_bf16x4(&Wt[16 * j + c][kk + kq]), acc[j], 0, 0,
                                                              0);
    }
}

// Features of the elements r0 .. r0 + nr - 1 of a box, normalised and rounded,
// into the 16 rows of a pair of waves (lane 0 .. 127; features_kernel's values: the 40 coefficients,
// then per face the jump of the face mean).  A lane takes one variable and
// direction of an element, both faces.
__device__ __forceinline__ void pair_features(const double* __restrict__ U, const dg::KTables& T, const dg::KGeom& G,
                                              const float* __restrict__ xs, long r0, int nr, int lane,
                                              uint16_t (*a)[L2S]) {
    auto put = [&](int r, int k, float x) { a[r][k] = to_bf16((x - xs[k]) * xs[NF + k]); };
#pragma unroll
    for (int t0 = 0; t0 < 16 * 40; t0 += 2 * WV) {
        const int t = t0 + lane, r = t / 40;
        if (r < nr) put(r, t - 40 * r, (float)U[r0 * 40 + t]);
    }
    double m[2], P[2][8];                      // weights of the - and + face means, b = r + 2 t1 + 4 t2
    for (int jj = 0; jj < 2; ++jj) {
        double v = 0.;
        for (int g = 0; g < 3; ++g) v += T.w[g] * T.B[g][jj];
        m[jj] = 0.5 * v;
    }
#pragma unroll
    for (int b = 0; b < 8; ++b) {
        P[0][b] = T.phim[b & 1] * m[b >> 1 & 1] * m[b >> 2];
        P[1][b] = T.phip[b & 1] * m[b >> 1 & 1] * m[b >> 2];
    }
#pragma unroll 1
    for (int t = lane; t < 16 * 15; t += 2 * WV) {
        const int r = t / 15, ds = t - 15 * r, d = ds / 5, s = ds - 5 * d;
        if (r >= nr) continue;
        const unsigned e = (unsigned)(r0 + r), nx = G.ne[0], ny = G.ne[1], nz = G.ne[2];
        const unsigned yz = e / nx, z = yz / ny;
        const unsigned c = d == 0 ? e - yz * nx : (d == 1 ? yz - z * ny : z);
        const unsigned st = d == 0 ? 1u : (d == 1 ? nx : nx * ny), n = d == 0 ? nx : (d == 1 ? ny : nz);
        const unsigned em = e - st + (c == 0 ? st * n : 0u), ep = e + st - (c + 1 == n ? st * n : 0u);
        const double *u = U + (size_t)e * 40 + s, *um = U + (size_t)em * 40 + s, *up = U + (size_t)ep * 40 + s;
        double om = 0., op = 0., nm = 0., np = 0.;
#pragma unroll
        for (int b = 0; b < 8; ++b) {          // mode b = i + 2 j + 4 k; its (r, t1, t2) along d
            const int b1 = (b >> 1 & 1) | (b & 1) << 1 | (b & 4), b2 = (b >> 2) | (b & 1) << 1 | (b >> 1 & 1) << 2;
            const double wm = d == 0 ? P[0][b] : (d == 1 ? P[0][b1] : P[0][b2]);
            const double wp = d == 0 ? P[1][b] : (d == 1 ? P[1][b1] : P[1][b2]);
            om = fma(u[b * 5], wm, om);
            op = fma(u[b * 5], wp, op);
            nm = fma(um[b * 5], wp, nm);
            np = fma(up[b * 5], wm, np);
        }
        put(r, 40 + 10 * d + s, (float)(nm - om));
        put(r, 45 + 10 * d + s, (float)(np - op));
    }
    for (int t = lane; t < 16 * (K1 - NF); t += 2 * WV) a[t / (K1 - NF)][NF + t % (K1 - NF)] = 0;
}

// Rows X (STATE: the features of the box state U) through the network; the two
// waves of a pair take half of each layer's columns.  Bound: VALU issue, more
// than half of it in the error functions (256 per row; 32 of some 50
// instructions per lane).  32768 elements: 26.9 us with the features, against
// 19.4 for a features kernel and 30.2 for four waves a block that took two
// tiles one after the other.
template <int WN, bool STATE>
__global__ __launch_bounds__(2 * WN * WV) void mlp_infer_kernel(const float* __restrict__ X, const double* __restrict__ U,
                                                                const dg::KTables* __restrict__ Tp, dg::KGeom G,
                                                                const uint16_t* __restrict__ Wimg,
                                                                const float* __restrict__ P,
                                                                const float* __restrict__ xs, float* __restrict__ C,
                                                                double bound, long rows,
                                                                unsigned long long* __restrict__ count) {
    constexpr int MT = 2 * WN * WV, MR = WN * 16;
    __shared__ alignas(16) InferLDS<WN> L;
    int t = threadIdx.x;
    // the weights' LDS image, a straight 16-byte copy
    static_assert(offsetof(InferLDS<WN>, w2) == IMG1 * 2 && offsetof(InferLDS<WN>, w3) == (IMG1 + IMG2) * 2 &&
                      offsetof(InferLDS<WN>, a) == IMG * 2 && IMG * 2 % 16 == 0,
                  "contiguous weight image");
    static_assert((NO + 1) * 4 <= L2S * 2 && K1 <= L2S, "outputs and features fit a row");
    {
        constexpr int NV = IMG * 2 / 16;
        const uint4* src = reinterpret_cast<const uint4*>(Wimg);
        uint4* dst = reinterpret_cast<uint4*>(&L.w1[0][0]);
        for (int i = t; i < NV; i += 4 * MT) {
            // four loads in flight before the stores
            const int i1 = i + MT, i2 = i + 2 * MT, i3 = i + 3 * MT;
            const uint4 v0 = src[i];
            const uint4 v1 = i1 < NV ? src[i1] : v0, v2 = i2 < NV ? src[i2] : v0, v3 = i3 < NV ? src[i3] : v0;
            dst[i] = v0;
            if (i1 < NV) dst[i1] = v1;
            if (i2 < NV) dst[i2] = v2;
            if (i3 < NV) dst[i3] = v3;
        }
    }
    const long ntile = (rows + MR - 1) / MR;
    for (long tile = blockIdx.x; tile < ntile; tile += gridDim.x) {
        // nothing of a tile is kept over the loop (addresses and biases held
        // in registers for the next tile, which is rare, spill)
        asm volatile("" : "+v"(t));
        asm volatile("" : "+s"(P), "+s"(xs));
        const int lane = t & 63, pl = t & 127, half = t >> 6 & 1, pair = t >> 7;
        const int c = lane & 15, rq = 4 * (lane >> 4);
        uint16_t(*const a)[L2S] = L.a + 16 * pair;
        const long r0 = tile * MR + 16 * pair;
        const int nr = (int)(rows - r0 < 16 ? rows - r0 : 16);     // may be 0 or less in the last tile
        if constexpr (!STATE) {
            // the features: all global loads first, then the stores
            constexpr int PER = 16 * K1 / (2 * WV);
            float xv[PER];
#pragma unroll
            for (int u = 0; u < PER; ++u) {
                const int i = pl + u * 2 * WV, r = i / K1, k = i % K1;
                xv[u] = (r < nr && k < NF) ? X[(r0 + r) * NF + k] : 0.f;
            }
#pragma unroll
            for (int u = 0; u < PER; ++u) {
                const int i = pl + u * 2 * WV, r = i / K1, k = i % K1;
                a[r][k] = (r < nr && k < NF) ? to_bf16((xv[u] - xs[k]) * xs[NF + k]) : (uint16_t)0;
            }
        } else {
            pair_features(U, *Tp, G, xs, r0, nr, pl, a);
        }
        __syncthreads();                       // also the staged weights
        // two hidden layers, GELU
        f32x4 acc[4];
        auto hidden = [&](auto first) {
            constexpr bool one = decltype(first)::value;
            const float* b = P + (one ? OFF_B1 : OFF_B2) + 64 * half;
#pragma unroll
            for (int j = 0; j < 4; ++j) acc[j] = f32x4{b[16 * j + c], b[16 * j + c], b[16 * j + c], b[16 * j + c]};
            if constexpr (one) mfma_layer<4, K1, L2S, L1S>(a, L.w1 + 64 * half, lane, acc);
            else mfma_layer<4, NH, L2S, L2S>(a, L.w2 + 64 * half, lane, acc);
            __syncthreads();
#pragma unroll
            for (int j = 0; j < 4; ++j) {
#pragma unroll
                for (int q = 0; q < 4; ++q) a[rq + q][64 * half + 16 * j + c] = to_bf16(gelu(acc[j][q]));
                __builtin_amdgcn_sched_barrier(0);     // four error functions in flight, not sixteen
            }
            __syncthreads();
        };
        hidden(std::true_type());
        hidden(std::false_type());
        // layer 3: NH -> NO, de-normalised; tiles 0 and 1, and tile 2
#pragma unroll
        for (int j = 0; j < 2; ++j) {
            const int n = 32 * half + 16 * j + c;
            const float b = n < NO ? P[OFF_B3 + n] : 0.f;
            acc[j] = f32x4{b, b, b, b};
        }
        if (half) mfma_layer<1, NH, L2S, L2S>(a, L.w3 + 32, lane, acc);
        else mfma_layer<2, NH, L2S, L2S>(a, L.w3, lane, acc);
        __syncthreads();
        float* const o = reinterpret_cast<float*>(&a[0][0]);
        constexpr int OS = L2S / 2;            // a row in floats
#pragma unroll
        for (int j = 0; j < 2; ++j) {
            const int n = 32 * half + 16 * j + c;
            if (n < NO) {
                const float ys = xs[2 * NF + n];
#pragma unroll
                for (int q = 0; q < 4; ++q) o[(rq + q) * OS + n] = acc[j][q] * ys;
            }
        }
        __syncthreads();
        // fallback bound per row (count null: no bound), then the store
        if (count) {
            if (pl < nr) {
                double n2 = 0.;
                for (int i = 0; i < NO; ++i) n2 += (double)o[pl * OS + i] * o[pl * OS + i];
                if (!(sqrt(n2) <= bound)) {
                    for (int i = 0; i < NO; ++i) o[pl * OS + i] = 0.f;
                    atomicAdd(count, 1ull);
                }
            }
            __syncthreads();
        }
        for (int i = pl; i < nr * NO; i += 2 * WV) C[r0 * NO + i] = o[i / NO * OS + i % NO];
        __syncthreads();                       // the rows are free for the next tile
    }
}

// ---------------------------------------------------------------------------
// Training on the matrix cores: FP32 GEMM tiles (v_mfma_f32_16x16x4f32,
// FP32 operands and accumulation).  In one 16x16x4 step lane l supplies
// A[l % 16][l / 16] and B[l / 16][l % 16] and holds D[4 (l / 16) + r][l % 16],
// r = 0..3, of the 16x16 result.  The layer inputs and the gradients stay
// FP32 and the weights are the bf16 working copy widened exactly, so the
// arithmetic is that of a plain FP32 network with bf16 weights up to the
// order of the FP32 sums.
// ---------------------------------------------------------------------------
constexpr int RT = 16;                         // rows of a train_rows workgroup
constexpr int RW = NH / 16;                    // its waves: a 16-column tile of the hidden layers each
constexpr int RB = RW * WV;
constexpr int GW = 4;                          // waves of a weight-gradient workgroup

__device__ __forceinline__ f32x4 mfma4(float a, float b, f32x4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
}

// The bf16 weights in the order of train_rows' lanes: for each 16-column tile
// of a layer's outputs, 16 bytes per lane of the weights of eight MFMA steps;
// forward W1, W2, W3, then W3 and W2 for the backward steps (rows as
// columns).  17 16-byte loads per lane in place of 124 2-byte ones.
constexpr int ST1 = (NF + 3) / 4, ST2 = NH / 4, ST3 = NO / 4;      // MFMA steps over the layers' inputs
constexpr int S1 = (ST1 + 7) / 8, S2 = (ST2 + 7) / 8, S3 = (ST3 + 7) / 8;
constexpr int TG = WV * 8;                     // weights of one tile and eight steps
constexpr int LI1 = 0, LI2 = LI1 + RW * S1 * TG, LI3 = LI2 + RW * S2 * TG, LB3 = LI3 + (NO + 15) / 16 * S2 * TG,
              LB2 = LB3 + RW * S3 * TG, LANE_IMG = LB2 + RW * S2 * TG;
__device__ __forceinline__ int lane_slot(int img, int groups, int k, int n) {   // input k, output n
    return img + ((n / 16 * groups + k / 32) * WV + (k & 3) * 16 + (n & 15)) * 8 + (k / 4 & 7);
}
__device__ __forceinline__ void store_lane_weights(uint16_t* img, int i, uint16_t v) {
    if (i < OFF_B1) {
        img[lane_slot(LI1, S1, i / NH, i % NH)] = v;
    } else if (i >= OFF_W2 && i < OFF_B2) {
        const int k = (i - OFF_W2) / NH, n = (i - OFF_W2) % NH;
        img[lane_slot(LI2, S2, k, n)] = v;
        img[lane_slot(LB2, S2, n, k)] = v;
    } else if (i >= OFF_W3 && i < OFF_B3) {
        const int k = (i - OFF_W3) / NO, n = (i - OFF_W3) % NO;
        img[lane_slot(LI3, S2, k, n)] = v;
        img[lane_slot(LB3, S3, n, k)] = v;
    }
}
__global__ void pack_lane_weights(const uint16_t* __restrict__ pb, uint16_t* __restrict__ img) {
    const int i = blockIdx.x * TB + threadIdx.x;
    if (i < NP) store_lane_weights(img, i, pb[i]);
}
// x is in its register here: what follows does not wait for its load (nor,
// the counter of loads and stores being one, for stores issued in between)
template <class T>
__device__ __forceinline__ void arrived(T& x) {
    asm volatile("" : "+v"(x));
}
template <int S>
struct LaneWeights {
    uint4 v[S];
    __device__ __forceinline__ void arrive() {
#pragma unroll
        for (int g = 0; g < S; ++g) {
            arrived(v[g].x);
            arrived(v[g].y);
            arrived(v[g].z);
            arrived(v[g].w);
        }
    }
    __device__ __forceinline__ void load(const uint16_t* img, int tile, int lane) {
#pragma unroll
        for (int g = 0; g < S; ++g) v[g] = *reinterpret_cast<const uint4*>(img + ((tile * S + g) * WV + lane) * 8);
    }
    __device__ __forceinline__ float operator[](int i) const {
        const uint4& q = v[i / 8];
        const int h = i % 8 / 2;
        const uint32_t x = h == 0 ? q.x : (h == 1 ? q.y : (h == 2 ? q.z : q.w));
        const uint32_t u = i & 1 ? x & 0xffff0000u : x << 16;
        float f;
        std::memcpy(&f, &u, 4);
        return f;
    }
};

// Position of a workgroup in the launch's sequence: the grid is a multiple
// of 8, workgroups go round the 8 XCDs, and each XCD walks a contiguous
// eighth, so that train_wgrad finds the rows of its chunks in its own L2.
__device__ __forceinline__ unsigned xcd_walk() {
    return (blockIdx.x & 7u) * (gridDim.x >> 3) + (blockIdx.x >> 3);
}

// Forward pass, loss and the gradients of the layer outputs for 16 rows of a
// mini-batch: gathered (rows idx, or row m itself for null), jittered and
// normalised rows Xn, activations H1 and H2, gradients G3 (mean squared error
// in normalised target units, 2 (O - Y / yscale) / (M NO)), G2 and G1, and
// the rows' sum of squared errors in part.  A wave keeps the pre-activations
// of its column tile in registers from the forward to the backward pass, the
// layers meet in LDS (row strides 4 modulo 64 banks and 4 rows x 16 columns
// per access: no conflicts), and all weights are on their way to registers
// while the rows are gathered.
// Bound: latency and issue of the two waves per SIMD that 4096 rows are (256
// workgroups): some 2000 instructions a wave, many of them the error function,
// and 124 dependent MFMAs behind the gather.  4096 rows take 13.6 us (26 with
// 2-byte weight loads); one launch in place of the eight of gather, jitter,
// three forward layers, loss and two backward ones.  A mini-batch of 4096
// with its parameter update: 118 us in 13 launches before, 33 in 3.
struct TrainRows {
    const float *X, *Y, *xs, *p;
    const uint16_t* img;             // lane_slot's order
    const int* idx;
    long nrows, M;
    float noise;
    unsigned long long key;
    float *Xn, *H1, *H2, *G1, *G2, *G3;
    double* part;
};

__global__ __launch_bounds__(RB) void train_rows(TrainRows A) {
    constexpr int SX = 76, SH = NH + 4, SO = 44;
    static_assert(NO % 4 == 0 && 4 * ST1 <= SX && NO <= SO, "LDS rows");
    __shared__ float xn[RT * SX], h1[RT * SH], h2[RT * SH], g2[RT * SH], g3[RT * SO];
    __shared__ long row[RT];
    __shared__ double red[RW];
    const int tid = threadIdx.x, w = tid / WV, lane = tid & (WV - 1), c = lane & 15, kq = lane >> 4;
    const int n = 16 * w + c, no = n < NO ? n : 0;
    const long r0 = (long)xcd_walk() * RT;
    if (r0 >= A.M) return;
    LaneWeights<S1> w1;
    LaneWeights<S2> w2, w3, t2;
    LaneWeights<S3> t3;
    w1.load(A.img + LI1, w, lane);
    w2.load(A.img + LI2, w, lane);
    w3.load(A.img + LI3, 16 * w < NO ? w : 0, lane);
    t3.load(A.img + LB3, w, lane);
    t2.load(A.img + LB2, w, lane);
    float b1 = A.p[OFF_B1 + n], b2 = A.p[OFF_B2 + n], b3 = A.p[OFF_B3 + no], ys = A.xs[2 * NF + no];
    if (tid < RT) {
        const long m = r0 + tid < A.M ? r0 + tid : A.M - 1;
        long r = m;
        if (A.idx) {
            r = A.idx[m];
            r = r < 0 ? 0 : (r >= A.nrows ? A.nrows - 1 : r);
        }
        row[tid] = r;
    }
    __syncthreads();
    float y[4];                                // targets of the output tile, in flight over the layers
#pragma unroll
    for (int r = 0; r < 4; ++r) y[r] = A.Y[row[4 * kq + r] * NO + no];
    for (int t = tid; t < RT * SX; t += RB) {
        const int q = t / SX, k = t - q * SX;
        const long m = r0 + q;
        float a = 0.f;
        if (k < NF && m < A.M) {
            a = A.X[row[q] * NF + k];
            if (A.noise > 0.f) a += jitter(A.noise, A.xs[NF + k], (unsigned long long)(m * NF + k), A.key);
            a = (a - A.xs[k]) * A.xs[NF + k];
            A.Xn[m * NF + k] = a;
        }
        xn[t] = a;
    }
    w1.arrive();
    w2.arrive();
    w3.arrive();
    t3.arrive();
    t2.arrive();
    for (float& v : y) arrived(v);
    arrived(b1);
    arrived(b2);
    arrived(b3);
    arrived(ys);
    __syncthreads();
    auto layer = [&](const float* in, int stride, const auto& wt, auto steps, f32x4 acc) {
        constexpr int K = decltype(steps)::value;
#pragma unroll
        for (int i = 0; i < K; ++i) acc = mfma4(in[c * stride + 4 * i + kq], wt[i], acc);
        return acc;
    };
    auto bias = [](float b) { return f32x4{b, b, b, b}; };
    // the tile to LDS and to memory (whose arrays hold whole tiles of rows)
    auto put = [&](float* o, int stride, float* out, int width, int r, float v) {
        o[(4 * kq + r) * stride + n] = v;
        out[(r0 + 4 * kq) * width + n + r * width] = v;
    };
    float dz1[4], dz2[4];
    const f32x4 z1 = layer(xn, SX, w1, std::integral_constant<int, ST1>(), bias(b1));
#pragma unroll
    for (int r = 0; r < 4; ++r) put(h1, SH, A.H1, NH, r, gelu_both(z1[r], dz1[r]));
    __syncthreads();
    const f32x4 z2 = layer(h1, SH, w2, std::integral_constant<int, ST2>(), bias(b2));
#pragma unroll
    for (int r = 0; r < 4; ++r) put(h2, SH, A.H2, NH, r, gelu_both(z2[r], dz2[r]));
    __syncthreads();
    double e2 = 0.;
    if (16 * w < NO) {
        const f32x4 o = layer(h2, SH, w3, std::integral_constant<int, ST2>(), bias(b3));
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const int q = 4 * kq + r;
            const float d = r0 + q < A.M ? o[r] - y[r] / ys : 0.f;
            if (n < NO) {
                put(g3, SO, A.G3, NO, r, 2.0f * d / (float)(A.M * NO));
                e2 += (double)d * d;
            }
        }
    }
    for (int off = WV / 2; off > 0; off >>= 1) e2 += __shfl_down(e2, off, WV);
    if (lane == 0) red[w] = e2;
    __syncthreads();
    if (tid == 0) {
        double v = 0.;
        for (int i = 0; i < RW; ++i) v += red[i];
        A.part[r0 / RT] = v;
    }
    const f32x4 zero = {0.f, 0.f, 0.f, 0.f};
    const f32x4 d2 = layer(g3, SO, t3, std::integral_constant<int, ST3>(), zero);
#pragma unroll
    for (int r = 0; r < 4; ++r) put(g2, SH, A.G2, NH, r, d2[r] * dz2[r]);
    __syncthreads();
    const f32x4 d1 = layer(g2, SH, t2, std::integral_constant<int, ST2>(), zero);
#pragma unroll
    for (int r = 0; r < 4; ++r) A.G1[(r0 + 4 * kq) * NH + n + r * NH] = d1[r] * dz1[r];
}

// Weight and bias gradients of a layer with K inputs and N outputs, partial
// over one chunk of rows: part[k][n] = sum_{m in [mb, me)} A[m][k] G[m][n],
// with the row k = K the bias (A = 1), for the 16 rows k0 .. of the layer and
// all its columns.  The waves split the chunk's rows and add their tiles in
// LDS, in a fixed order.  A lane reads four neighbouring columns at once:
// tile j of a group of four holds the columns 4 c + j.  Bound: latency (4096
// rows: 64 MFMAs per wave, 8.8 us for the three layers).
template <int K, int N>
__device__ __forceinline__ void wgrad_tile(const float* __restrict__ A, const float* __restrict__ G,
                                           float* __restrict__ part, int k0, long mb, long me, f32x4* red) {
    constexpr int NG = (N + 63) / 64, NJ = 4 * NG;
    const int wv = threadIdx.x / WV, lane = threadIdx.x & (WV - 1), c = lane & 15, kq = lane >> 4;
    const int k = k0 + c;
    f32x4 acc[NJ];
#pragma unroll
    for (int j = 0; j < NJ; ++j) acc[j] = f32x4{0.f, 0.f, 0.f, 0.f};
    for (long m4 = mb + 4 * wv; m4 < me; m4 += 4 * GW) {
        const long m = m4 + kq;
        const bool ok = m < me;                // all rows but the last ones of the batch's last chunk
        const long mc = ok ? m : mb;
        float a = A[mc * K + (k < K ? k : 0)];
        a = ok ? (k < K ? a : (k == K ? 1.f : 0.f)) : 0.f;
#pragma unroll
        for (int q = 0; q < NG; ++q) {
            const int n = 64 * q + 4 * c;      // the columns past N are not stored
            f32x4 g = *reinterpret_cast<const f32x4*>(G + mc * N + (n < N ? n : 0));
            if (m4 + 4 > me && !ok) g = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int j = 0; j < 4; ++j) acc[4 * q + j] = mfma4(a, g[j], acc[4 * q + j]);
        }
    }
#pragma unroll
    for (int j = 0; j < NJ; ++j) red[(wv * NJ + j) * WV + lane] = acc[j];
    __syncthreads();
    for (int i = threadIdx.x; i < NG * WV; i += GW * WV) {
        const int q = i / WV, l = i % WV, n = 64 * q + 4 * (l & 15);
        if (n >= N) continue;
        f32x4 v[4];
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            v[j] = red[(4 * q + j) * WV + l];
#pragma unroll
            for (int w = 1; w < GW; ++w) v[j] += red[(w * NJ + 4 * q + j) * WV + l];
        }
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const int kk = k0 + 4 * (l >> 4) + r;
            if (kk <= K) *reinterpret_cast<f32x4*>(part + kk * N + n) = f32x4{v[0][r], v[1][r], v[2][r], v[3][r]};
        }
    }
}

// All three layers in one launch: workgroup (16-row k tile of a layer, chunk)
constexpr int KT1 = (NF + 16) / 16, KT2 = (NH + 16) / 16;      // k tiles with the bias row
static_assert(NH % 64 == 0 && NO % 4 == 0 && OFF_W2 % 4 == 0 && OFF_W3 % 4 == 0 && NP % 4 == 0,
              "16-byte groups of columns");
__global__ __launch_bounds__(GW * WV) void train_wgrad(TrainRows A, float* __restrict__ gpart, long chunk) {
    __shared__ f32x4 red[GW * (NH / 16) * WV];
    const unsigned u = xcd_walk(), s = u / (KT1 + 2 * KT2);
    const int t = (int)(u - s * (KT1 + 2 * KT2));
    const long mb = (long)s * chunk, me = mb + chunk < A.M ? mb + chunk : A.M;
    if (mb >= A.M) return;
    float* part = gpart + (size_t)s * NP;
    if (t < KT2) wgrad_tile<NH, NH>(A.H1, A.G2, part + OFF_W2, 16 * t, mb, me, red);
    else if (t < KT2 + KT1) wgrad_tile<NF, NH>(A.Xn, A.G1, part + OFF_W1, 16 * (t - KT2), mb, me, red);
    else wgrad_tile<NH, NO>(A.H2, A.G3, part + OFF_W3, 16 * (t - KT2 - KT1), mb, me, red);
}

// g[i] = sum_s part[s][i] over the row chunks (fixed order), with ADAM then
// the Adam update (Kingma & Ba 2015) of the FP32 master parameters and their
// BF16 working copy; the last workgroup adds the rows' squared errors
// (nb partial sums) times inv to the loss, in a fixed order.
struct AdamStep {
    float *p, *m1, *m2;
    uint16_t *pb, *img;
    float lr, b1, b2, eps, c1, c2;
};
template <bool ADAM>
__global__ __launch_bounds__(WV) void train_update(const float* __restrict__ part, float* __restrict__ g, int nchunk,
                                                   AdamStep S, const double* __restrict__ e2, long nb, double inv,
                                                   double* __restrict__ loss) {
    if (blockIdx.x == gridDim.x - 1) {
        double v = 0.;
        for (long i = threadIdx.x; i < nb; i += WV) v += e2[i];
        for (int off = WV / 2; off > 0; off >>= 1) v += __shfl_down(v, off, WV);
        if (threadIdx.x == 0) loss[0] += v * inv;
        return;
    }
    const int i = blockIdx.x * WV + threadIdx.x;
    if (i >= NP) return;
    float v = 0.f;
#pragma unroll 8
    for (int s = 0; s < nchunk; ++s) v += part[(size_t)s * NP + i];
    if constexpr (ADAM) {
        const float a = S.b1 * S.m1[i] + (1.f - S.b1) * v;
        const float q2 = S.b2 * S.m2[i] + (1.f - S.b2) * v * v;
        S.m1[i] = a;
        S.m2[i] = q2;
        const float q = S.p[i] - S.lr * (a / S.c1) / (sqrtf(q2 / S.c2) + S.eps);
        S.p[i] = q;
        const uint16_t h = to_bf16(q);
        S.pb[i] = h;
        store_lane_weights(S.img, i, h);
    } else {
        g[i] = v;
    }
}

__global__ void clear_f64_kernel(double* p) { p[threadIdx.x] = 0.; }

// Y = trunc(Df) - Dc + (trunc(Uf) - Uc) / tau, for a coarse state Uc of
// its own (a coarse run beside the fine one): the tendency mismatch at Uc
// plus a relaxation of Uc toward the fine state's projection
__global__ void target_at_kernel(const double* __restrict__ Df, const double* __restrict__ Dc,
                                 const double* __restrict__ Uf, const double* __restrict__ Uc, double rtau,
                                 float* __restrict__ Y, int Pf, long E) {
    const long t = (long)blockIdx.x * TB + threadIdx.x;
    if (t >= E * 40) return;
    const long e = t / 40;
    const int r = (int)(t % 40), b = r / 5, s = r % 5;
    const int i = b & 1, j = (b >> 1) & 1, k = b >> 2, n = Pf + 1;
    const long f = (e * n * n * n + i + n * j + n * n * k) * 5 + s;
    Y[t] = (float)(Df[f] - Dc[t] + (Uf[f] - Uc[t]) * rtau);
}

// Device scratch of dg_closure_step_noalloc: the corrections [E][NO] and the
// 64-bit fallback counter of up to NOALLOC_MAX_ELEMS elements (32^3, the
// closure's box), 5.2 MB, in a
// file-scope array that each GPU holds until the process ends.  Host code
// never passes the array's name to a kernel (on the host it is a stand-in,
// not a device address): it uses the address hipGetSymbolAddress returns
// for the current device (noalloc_scratch).
constexpr long NOALLOC_MAX_ELEMS = 32768;
constexpr size_t NOALLOC_C = (size_t)NOALLOC_MAX_ELEMS * NO;        // floats
constexpr size_t NOALLOC_FLOATS = NOALLOC_C + 2;        // + the counter (8 B, 8-aligned)
static_assert((NOALLOC_C * sizeof(float)) % 8 == 0, "counter alignment");
static __device__ __align__(256) float scratch[NOALLOC_FLOATS];

// one thread clears *p (a vector store: the address is lane-indexed)
__global__ void clear_u64_kernel(unsigned long long* p) { p[threadIdx.x] = 0ull; }

thread_local std::string g_mlp_error;

}  // namespace

// ---------------------------------------------------------------------------
// MLP object
// ---------------------------------------------------------------------------
struct dg_mlp {
    int device = 0;
    hipStream_t stream = nullptr;
    float* p = nullptr;          // master parameters [NP]
    uint16_t* pb = nullptr;      // BF16 working copy
    uint16_t* img = nullptr;     // the inference kernel's LDS image of the bf16 weights
    uint16_t* lane_img = nullptr;   // the training kernels' copy (lane_slot)
    bool img_stale = true;       // pb changed since img was built
    float* g = nullptr;          // gradient
    float* m1 = nullptr;         // Adam moments
    float* m2 = nullptr;
    float* xs = nullptr;         // feature mean [NF], scale [NF], target scale [NO]
    long cap = 0;                // rows the activation buffers hold
    float *Xn = nullptr, *H1 = nullptr, *H2 = nullptr, *G3 = nullptr, *G2 = nullptr, *G1 = nullptr;
    double* part = nullptr;
    float* gpart = nullptr;      // per-chunk weight-gradient partials [GCHUNKS][NP]
    double* lacc = nullptr;      // training loss accumulator (device)
    long step = 0;
    std::string err;
};

namespace {

void free_acts(dg_mlp* m) {
    for (float* q : {m->Xn, m->H1, m->H2, m->G3, m->G2, m->G1})
        if (q) (void)hipFree(q);
    if (m->part) (void)hipFree(m->part);
    if (m->gpart) (void)hipFree(m->gpart);
    if (m->lacc) (void)hipFree(m->lacc);
    m->Xn = m->H1 = m->H2 = m->G3 = m->G2 = m->G1 = nullptr;
    m->part = nullptr;
    m->gpart = nullptr;
    m->lacc = nullptr;
    m->cap = 0;
}

// The inference kernel on a persistent grid of at most one block per CU (the
// weight image is rebuilt first, on the same stream, when pb changed), on rows
// X, or for null X on the features of the state U of the box s.  Four pairs
// of waves a block while that is a tile per CU; above, eight share the staged
// weights (one tile per CU in place of two one after the other).
void launch_infer(dg_mlp* m, const float* X, const dg_solver* s, const double* U, float* C, double bound, long rows,
                  unsigned long long* count, hipStream_t st) {
    if (m->img_stale) {
        hipLaunchKernelGGL(pack_infer_weights, dim3(nblk(IMG)), dim3(TB), 0, st, m->pb, m->img);
        hcheck(hipGetLastError(), "weight image kernel");
        m->img_stale = false;
    }
    const dg::KTables* tab = s ? s->dtab : nullptr;
    const dg::KGeom g = s ? s->geo : dg::KGeom{};
    auto launch = [&](auto waves, auto state) {
        constexpr int WN = decltype(waves)::value;
        const long ntile = (rows + 16 * WN - 1) / (16 * WN);
        const unsigned grid = (unsigned)(ntile < MAX_INFER_BLOCKS ? ntile : MAX_INFER_BLOCKS);
        hipLaunchKernelGGL((mlp_infer_kernel<WN, decltype(state)::value>), dim3(grid), dim3(2 * WN * WV), 0, st, X, U, tab, g, m->img, m->p, m->xs, C,
                           bound, rows, count);
    };
    const bool few = rows <= 4 * 16 * MAX_INFER_BLOCKS;
    std::integral_constant<int, 4> w4;
    std::integral_constant<int, 8> w8;
    if (X) few ? launch(w4, std::false_type()) : launch(w8, std::false_type());
    else few ? launch(w4, std::true_type()) : launch(w8, std::true_type());
    hcheck(hipGetLastError(), "inference kernel");
}

void ensure_acts(dg_mlp* m, long rows) {
    rows = (rows + RT - 1) / RT * RT;          // train_rows writes whole tiles
    if (rows <= m->cap) return;
    free_acts(m);
    auto al = [&](float** q, long n) { hcheck(dg::device_malloc(q, (size_t)n * sizeof(float)), "hipMalloc(mlp)"); };
    al(&m->H1, rows * NH);
    al(&m->H2, rows * NH);
    al(&m->G3, rows * NO);
    al(&m->G2, rows * NH);
    al(&m->G1, rows * NH);
    al(&m->Xn, rows * NF);
    hcheck(dg::device_malloc(&m->part, (size_t)((rows + RT - 1) / RT) * sizeof(double)), "hipMalloc(mlp)");
    hcheck(dg::device_malloc(&m->gpart, (size_t)GCHUNKS * NP * sizeof(float)), "hipMalloc(mlp)");
    hcheck(dg::device_malloc(&m->lacc, sizeof(double)), "hipMalloc(mlp)");
    m->cap = rows;
}

// the weight-gradient row chunks of a batch of M rows: at most GCHUNKS
// chunks of at least 64 rows
long grad_chunk(long M) {
    const long c = (M + GCHUNKS - 1) / GCHUNKS;
    return c < 64 ? 64 : c;
}

// the training kernels' copy of the bf16 weights, before a run of mini-batches
// (train_update keeps it from one to the next)
void pack_lanes(dg_mlp* m) {
    hipLaunchKernelGGL(pack_lane_weights, dim3(nblk(NP)), dim3(TB), 0, m->stream, m->pb, m->lane_img);
    hcheck(hipGetLastError(), "weight copy kernel");
}

// Loss and gradient of a mini-batch of M rows: the batch's mean squared error
// is added to m->lacc on the device (no host synchronisation); the gradient
// goes into m->g, or with adam straight into the parameters.
void mini_batch(dg_mlp* m, const float* X, const float* Y, const int* idx, long nrows, long M, float noise,
                const AdamStep* adam) {
    hipStream_t st = m->stream;
    TrainRows A;
    A.X = X;
    A.Y = Y;
    A.xs = m->xs;
    A.p = m->p;
    A.img = m->lane_img;
    A.idx = idx;
    A.nrows = nrows;
    A.M = M;
    A.noise = noise;
    A.key = (unsigned long long)m->step * 0x100000001ull;
    A.Xn = m->Xn;
    A.H1 = m->H1;
    A.H2 = m->H2;
    A.G1 = m->G1;
    A.G2 = m->G2;
    A.G3 = m->G3;
    A.part = m->part;
    const unsigned nr = (unsigned)((M + RT - 1) / RT);
    hipLaunchKernelGGL(train_rows, dim3((nr + 7u) & ~7u), dim3(RB), 0, st, A);
    const long chunk = grad_chunk(M);
    const unsigned nch = (unsigned)((M + chunk - 1) / chunk);
    hipLaunchKernelGGL(train_wgrad, dim3((nch * (KT1 + 2 * KT2) + 7u) & ~7u), dim3(GW * WV), 0, st, A, m->gpart, chunk);
    const dim3 ug((NP + WV - 1) / WV + 1);
    const double inv = 1.0 / (double)(M * NO);
    if (adam)
        hipLaunchKernelGGL((train_update<true>), ug, dim3(WV), 0, st, m->gpart, m->g, (int)nch, *adam, m->part,
                           (long)nr, inv, m->lacc);
    else
        hipLaunchKernelGGL((train_update<false>), ug, dim3(WV), 0, st, m->gpart, m->g, (int)nch, AdamStep{}, m->part,
                           (long)nr, inv, m->lacc);
    hcheck(hipGetLastError(), "mlp training kernels");
}

// m->lacc = 0 (a kernel: no memset node on a captured stream)
void clear_loss(dg_mlp* m) {
    hipLaunchKernelGGL(clear_f64_kernel, dim3(1), dim3(1), 0, m->stream, m->lacc);
    hcheck(hipGetLastError(), "clear kernel");
}

double read_loss(dg_mlp* m) {
    double v = 0.;
    hcheck(hipMemcpyAsync(&v, m->lacc, sizeof(double), hipMemcpyDeviceToHost, m->stream), "hipMemcpy");
    hcheck(hipStreamSynchronize(m->stream), "hipStreamSynchronize");
    return v;
}

template <class F>
int mlp_guard(std::string& err, F&& f) {
    try {
        f();
        err.clear();
        return DG_OK;
    } catch (const std::invalid_argument& e) {
        err = e.what();
        return DG_ERR_ARGUMENT;
    } catch (const dg::UnsupportedError& e) {
        err = e.what();
        return DG_ERR_UNSUPPORTED;
    } catch (const std::domain_error& e) {
        err = e.what();
        return DG_ERR_NUMERICS;
    } catch (const std::exception& e) {
        err = e.what();
        return DG_ERR_DEVICE;
    }
}

void need_ptr(const void* p, const char* what) {
    if (!p) throw std::invalid_argument(std::string(what) + " is NULL");
}

// the coarse / fine solvers this module works with: 3D Legendre periodic boxes
void check_box(const dg_solver* s, const char* what, int order) {
    need_ptr(s, what);
    if ((unsigned long long)s->geo.E * NF >= (1ull << 32))
        throw std::invalid_argument(std::string(what) + ": too many elements for the closure features");
    if (s->cfg.dim != 3 || s->geo.mapped || s->cfg.basis != dg::Basis::LegendreHex || s->geo.fp32)
        throw dg::UnsupportedError(std::string(what) + ": a 3D affine FP64 LegendreHex periodic box is required");
    if (order > 0 && s->P != order)
        throw dg::UnsupportedError(std::string(what) + ": order " + std::to_string(order) + " is required");
}

// dD = M^-1 R(U) of solver s (dt = 1), with its own stage registers as scratch
void tendency(dg_solver* s, const double* U, double* D) {
    dg::StageArgs a{};
    a.Ust = U;
    a.R = s->Ua;
    a.mode = dg::MODE_RESIDUAL;
    hcheck(launch_solver_stage(s, a, nullptr, s->stream), "stage kernel");
    hcheck(dg::launch_inv_mass(s->P, 1.0, s->Ua, D, s->dtab, s->geo, s->stream), "inverse mass kernel");
}

// The device address of `scratch` on the current device, looked up once
// per device (under a lock) and kept; no heap memory is involved.
constexpr int NOALLOC_MAX_DEVICES = 64;
float* noalloc_scratch(int device) {
    static std::mutex mu;
    static float* addr[NOALLOC_MAX_DEVICES] = {};
    if (device < 0 || device >= NOALLOC_MAX_DEVICES) throw std::invalid_argument("device index out of range");
    std::lock_guard<std::mutex> lk(mu);
    if (!addr[device]) {
        void* ptr = nullptr;
        hcheck(hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch)), "hipGetSymbolAddress(scratch)");
        if (!ptr) throw std::runtime_error("hipGetSymbolAddress(scratch) returned NULL");
        addr[device] = static_cast<float*>(ptr);
    }
    return addr[device];
}

// argument checks of the closure step; returns the time step
double closure_check(dg_solver* s, dg_mlp* m, double dt_step, int nsteps) {
    check_box(s, "solver", 1);
    need_ptr(m, "mlp");
    if (nsteps < 0) throw std::invalid_argument("nsteps < 0");
    const double dt = dt_step > 0.0 ? dt_step : s->dt;
    if (!(dt > 0.0)) throw std::invalid_argument("no time step");
    if (s->cfg.stepper != dg::Stepper::RK4) throw dg::UnsupportedError("the closure steps RK4 only");
    hcheck(hipSetDevice(s->device), "hipSetDevice");
    return dt;
}

// nsteps corrected RK4 steps with the given corrections C [E][NO] and fallback
// counter cnt (device memory)
void closure_steps(dg_solver* s, dg_mlp* m, double dt, double bound, int nsteps, float* C,
                   unsigned long long* cnt, long* n_fallback) {
    const long E = s->geo.E;
    // the counter is cleared by a kernel (no memset node if the caller
    // captures the solver's stream)
    hipLaunchKernelGGL(clear_u64_kernel, dim3(1), dim3(1), 0, s->stream, cnt);
    hcheck(hipGetLastError(), "clear kernel");
    // the network's parameters are written by its own stream (training)
    hcheck(hipStreamSynchronize(m->stream), "hipStreamSynchronize");
    auto stage = [&](const double* Ust, double* Uout, int mode, double alpha) {
        // everything on the solver's stream: the network on the state's
        // features with its fallback, and the stage kernel whose RK epilogue takes
        // dU = dt (M^-1 R + C)
        launch_infer(m, nullptr, s, Ust, C, bound, E, cnt, s->stream);
        dg::StageArgs a{};
        a.Ust = Ust;
        a.U0 = s->U0;
        a.Uout = Uout;
        a.acc = s->acc;
        a.cmp = s->cmp;
        a.dt = dt;
        a.alpha = alpha;
        a.mode = mode;
        hcheck(launch_solver_stage(s, a, C, s->stream), "corrected stage kernel");
    };
    for (int k = 0; k < nsteps; ++k) {
        // the stage kernel reads the neighbours of Ust: stages ping-pong
        // U0 -> Ua -> Ub -> Ua -> U0, as in dg_step
        stage(s->U0, s->Ua, dg::MODE_RK_FIRST, 0.5);
        s->time += dt / 2.0;
        stage(s->Ua, s->Ub, dg::MODE_RK_MID, 0.5);
        stage(s->Ub, s->Ua, dg::MODE_RK_MID, 1.0);
        s->time += dt / 2.0;
        stage(s->Ua, s->U0, dg::MODE_RK_LAST, 0.0);
    }
    unsigned long long c = 0;
    hcheck(hipMemcpyAsync(&c, cnt, sizeof(c), hipMemcpyDeviceToHost, s->stream), "hipMemcpyAsync");
    hcheck(hipStreamSynchronize(s->stream), "hipStreamSynchronize");
    if (n_fallback) *n_fallback = (long)c;
}

}  // namespace

extern "C" {

int dg_mlp_create(unsigned long long seed, dg_mlp** out) {
    if (out) *out = nullptr;
    dg_mlp* m = nullptr;
    const int rc = mlp_guard(g_mlp_error, [&] {
        need_ptr(out, "out");
        m = new dg_mlp();
        hcheck(hipGetDevice(&m->device), "hipGetDevice");
        hcheck(hipStreamCreateWithFlags(&m->stream, hipStreamNonBlocking), "hipStreamCreate");
        hcheck(dg::device_malloc(&m->p, NP * sizeof(float)), "hipMalloc(mlp)");
        hcheck(dg::device_malloc(&m->pb, NP * sizeof(uint16_t)), "hipMalloc(mlp)");
        hcheck(dg::device_malloc(&m->img, IMG * sizeof(uint16_t)), "hipMalloc(mlp)");
        hcheck(dg::device_malloc(&m->lane_img, LANE_IMG * sizeof(uint16_t)), "hipMalloc(mlp)");
        hcheck(dg::launch_zero(m->lane_img, LANE_IMG * sizeof(uint16_t), m->stream), "zero kernel");   // the padding
        hcheck(dg::device_malloc(&m->g, NP * sizeof(float)), "hipMalloc(mlp)");
        hcheck(dg::device_malloc(&m->m1, NP * sizeof(float)), "hipMalloc(mlp)");
        hcheck(dg::device_malloc(&m->m2, NP * sizeof(float)), "hipMalloc(mlp)");
        hcheck(dg::device_malloc(&m->xs, (2 * NF + NO) * sizeof(float)), "hipMalloc(mlp)");
        // He-normal hidden layers, a small output layer (the correction
        // starts near zero), zero biases; identity scaling
        std::mt19937_64 rng(seed);
        std::normal_distribution<float> nd(0.f, 1.f);
        std::vector<float> h(NP, 0.f);
        for (int i = 0; i < NF * NH; ++i) h[OFF_W1 + i] = nd(rng) * std::sqrt(2.f / NF);
        for (int i = 0; i < NH * NH; ++i) h[OFF_W2 + i] = nd(rng) * std::sqrt(2.f / NH);
        for (int i = 0; i < NH * NO; ++i) h[OFF_W3 + i] = nd(rng) * 0.1f * std::sqrt(1.f / NH);
        hcheck(hipMemcpy(m->p, h.data(), NP * sizeof(float), hipMemcpyHostToDevice), "hipMemcpy");
        std::vector<float> z(NP, 0.f);
        hcheck(hipMemcpy(m->m1, z.data(), NP * sizeof(float), hipMemcpyHostToDevice), "hipMemcpy");
        hcheck(hipMemcpy(m->m2, z.data(), NP * sizeof(float), hipMemcpyHostToDevice), "hipMemcpy");
        std::vector<float> xs(2 * NF + NO, 1.f);
        for (int i = 0; i < NF; ++i) xs[i] = 0.f;
        hcheck(hipStreamSynchronize(m->stream), "hipStreamSynchronize");
        hcheck(hipMemcpy(m->xs, xs.data(), xs.size() * sizeof(float), hipMemcpyHostToDevice), "hipMemcpy");
        hipLaunchKernelGGL(to_bf16_kernel, dim3(nblk(NP)), dim3(TB), 0, m->stream, m->p, m->pb, NP);
        m->img_stale = true;
        hcheck(hipGetLastError(), "to_bf16");
        hcheck(hipStreamSynchronize(m->stream), "hipStreamSynchronize");
    });
    if (rc != DG_OK) {
        if (m) dg_mlp_destroy(m);
        return rc;
    }
    *out = m;
    return DG_OK;
}

int dg_mlp_destroy(dg_mlp* m) {
    if (!m) return DG_OK;
    (void)hipSetDevice(m->device);
    free_acts(m);
    for (float* q : {m->p, m->g, m->m1, m->m2, m->xs})
        if (q) (void)hipFree(q);
    if (m->pb) (void)hipFree(m->pb);
    if (m->img) (void)hipFree(m->img);
    if (m->lane_img) (void)hipFree(m->lane_img);
    if (m->stream) (void)hipStreamDestroy(m->stream);
    delete m;
    return DG_OK;
}

const char* dg_mlp_last_error(const dg_mlp* m) { return m ? m->err.c_str() : g_mlp_error.c_str(); }

int dg_mlp_num_params(long* n) {
    if (!n) return DG_ERR_ARGUMENT;
    *n = NP;
    return DG_OK;
}

int dg_mlp_get_params(const dg_mlp* m, float* host) {
    return mlp_guard(m ? const_cast<dg_mlp*>(m)->err : g_mlp_error, [&] {
        need_ptr(m, "mlp");
        need_ptr(host, "host");
        hcheck(hipMemcpy(host, m->p, NP * sizeof(float), hipMemcpyDeviceToHost), "hipMemcpy");
    });
}

int dg_mlp_set_params(dg_mlp* m, const float* host) {
    return mlp_guard(m ? m->err : g_mlp_error, [&] {
        need_ptr(m, "mlp");
        need_ptr(host, "host");
        // work already queued on the network's stream may read the parameters
        hcheck(hipStreamSynchronize(m->stream), "hipStreamSynchronize");
        hcheck(hipMemcpy(m->p, host, NP * sizeof(float), hipMemcpyHostToDevice), "hipMemcpy");
        hipLaunchKernelGGL(to_bf16_kernel, dim3(nblk(NP)), dim3(TB), 0, m->stream, m->p, m->pb, NP);
        m->img_stale = true;
        hcheck(hipGetLastError(), "to_bf16");
        hcheck(hipStreamSynchronize(m->stream), "hipStreamSynchronize");
    });
}

int dg_mlp_set_scaling(dg_mlp* m, const float* x_mean, const float* x_scale, const float* y_scale) {
    return mlp_guard(m ? m->err : g_mlp_error, [&] {
        need_ptr(m, "mlp");
        need_ptr(x_mean, "x_mean");
        need_ptr(x_scale, "x_scale");
        need_ptr(y_scale, "y_scale");
        std::vector<float> xs(2 * NF + NO);
        for (int i = 0; i < NF; ++i) {
            xs[i] = x_mean[i];
            xs[NF + i] = x_scale[i];
        }
        for (int i = 0; i < NO; ++i) {
            if (!(y_scale[i] > 0.f)) throw std::invalid_argument("y_scale entries must be > 0");
            xs[2 * NF + i] = y_scale[i];
        }
        hcheck(hipStreamSynchronize(m->stream), "hipStreamSynchronize");
        hcheck(hipMemcpy(m->xs, xs.data(), xs.size() * sizeof(float), hipMemcpyHostToDevice), "hipMemcpy");
    });
}

int dg_mlp_forward(dg_mlp* m, const float* X_dev, float* Y_dev, long rows) {
    return mlp_guard(m ? m->err : g_mlp_error, [&] {
        need_ptr(m, "mlp");
        need_ptr(X_dev, "X");
        need_ptr(Y_dev, "Y");
        if (rows < 1) throw std::invalid_argument("rows < 1");
        hcheck(hipSetDevice(m->device), "hipSetDevice");
        // the closure step's inference kernel, without the fallback bound
        launch_infer(m, X_dev, nullptr, nullptr, Y_dev, 0.0, rows, nullptr, m->stream);
        hcheck(hipStreamSynchronize(m->stream), "hipStreamSynchronize");
    });
}

int dg_mlp_gradient(dg_mlp* m, const float* X_dev, const float* Y_dev, long rows, float* grad_host, double* loss) {
    return mlp_guard(m ? m->err : g_mlp_error, [&] {
        need_ptr(m, "mlp");
        need_ptr(X_dev, "X");
        need_ptr(Y_dev, "Y");
        if (rows < 1) throw std::invalid_argument("rows < 1");
        hcheck(hipSetDevice(m->device), "hipSetDevice");
        ensure_acts(m, rows);
        clear_loss(m);
        pack_lanes(m);
        mini_batch(m, X_dev, Y_dev, nullptr, rows, rows, 0.f, nullptr);
        const double l = read_loss(m);
        if (loss) *loss = l;
        if (grad_host) hcheck(hipMemcpy(grad_host, m->g, NP * sizeof(float), hipMemcpyDeviceToHost), "hipMemcpy");
    });
}

int dg_mlp_train(dg_mlp* m, const float* X_dev, const float* Y_dev, long nrows, const int* idx_dev, long nidx,
                 int batch, float lr, float noise, double* mean_loss) {
    return mlp_guard(m ? m->err : g_mlp_error, [&] {
        need_ptr(m, "mlp");
        need_ptr(X_dev, "X");
        need_ptr(Y_dev, "Y");
        need_ptr(idx_dev, "idx");
        if (nrows < 1 || nidx < 1 || batch < 1) throw std::invalid_argument("empty training set or batch");
        if (nidx < batch) throw std::invalid_argument("fewer row indices than one mini-batch (nidx < batch)");
        hcheck(hipSetDevice(m->device), "hipSetDevice");
        ensure_acts(m, batch);
        clear_loss(m);
        pack_lanes(m);
        long nb = 0;
        for (long i0 = 0; i0 + batch <= nidx; i0 += batch) {
            const float b1 = 0.9f, b2 = 0.999f, k = (float)(m->step + 1);
            const AdamStep adam{m->p, m->m1, m->m2, m->pb, m->lane_img, lr, b1, b2, 1e-8f, 1.f - std::pow(b1, k), 1.f - std::pow(b2, k)};
            m->img_stale = true;
            mini_batch(m, X_dev, Y_dev, idx_dev + i0, nrows, batch, noise, &adam);
            ++nb;
            ++m->step;
        }
        const double sum = read_loss(m);
        if (mean_loss) *mean_loss = nb ? sum / nb : 0.;
    });
}

int dg_closure_features(dg_solver* s, const double* U_dev, float* X_dev) {
    return mlp_guard(g_mlp_error, [&] {
        check_box(s, "solver", 1);
        need_ptr(U_dev, "U");
        need_ptr(X_dev, "X");
        hcheck(hipSetDevice(s->device), "hipSetDevice");
        hipLaunchKernelGGL(features_kernel, dim3(nblk((long)s->geo.E * FT)), dim3(TB), 0, s->stream, U_dev, X_dev,
                           s->dtab, s->geo);
        hcheck(hipGetLastError(), "features kernel");
        hcheck(hipStreamSynchronize(s->stream), "hipStreamSynchronize");
    });
}

int dg_closure_target(dg_solver* fine, const double* Uf_dev, dg_solver* coarse, double* Uc_dev, float* Y_dev) {
    return mlp_guard(g_mlp_error, [&] {
        check_box(fine, "fine solver", 0);
        check_box(coarse, "coarse solver", 1);
        need_ptr(Uf_dev, "Uf");
        need_ptr(Uc_dev, "Uc");
        need_ptr(Y_dev, "Y");
        if (fine->P < 2) throw std::invalid_argument("the fine solver's order must exceed 1");
        for (int d = 0; d < 3; ++d)
            if (fine->geo.ne[d] != coarse->geo.ne[d] || fine->geo.h[d] != coarse->geo.h[d] ||
                fine->geo.lo[d] != coarse->geo.lo[d])
                throw std::invalid_argument("fine and coarse solvers must share the mesh");
        if (fine->device != coarse->device) throw std::invalid_argument("the solvers live on different devices");
        hcheck(hipSetDevice(fine->device), "hipSetDevice");
        hcheck(hipStreamSynchronize(coarse->stream), "hipStreamSynchronize");
        const long E = fine->geo.E;
        // fine tendency into the fine handle's Ub, then the coarse state and its tendency
        tendency(fine, Uf_dev, fine->Ub);
        hipLaunchKernelGGL(truncate_kernel, dim3(nblk(E * 40)), dim3(TB), 0, fine->stream, Uf_dev, Uc_dev, fine->P, E);
        hcheck(hipGetLastError(), "truncate kernel");
        hcheck(hipStreamSynchronize(fine->stream), "hipStreamSynchronize");
        tendency(coarse, Uc_dev, coarse->Ub);
        hcheck(hipStreamSynchronize(coarse->stream), "hipStreamSynchronize");
        hipLaunchKernelGGL(target_kernel, dim3(nblk(E * 40)), dim3(TB), 0, fine->stream, fine->Ub, coarse->Ub, Y_dev,
                           fine->P, E);
        hcheck(hipGetLastError(), "target kernel");
        hcheck(hipStreamSynchronize(fine->stream), "hipStreamSynchronize");
    });
}

int dg_closure_target_at(dg_solver* fine, const double* Uf_dev, dg_solver* coarse, const double* Uc_dev, double tau,
                         float* Y_dev) {
    return mlp_guard(g_mlp_error, [&] {
        check_box(fine, "fine solver", 0);
        check_box(coarse, "coarse solver", 1);
        need_ptr(Uf_dev, "Uf");
        need_ptr(Uc_dev, "Uc");
        need_ptr(Y_dev, "Y");
        if (fine->P < 2) throw std::invalid_argument("the fine solver's order must exceed 1");
        if (!(tau > 0.0)) throw std::invalid_argument("tau must be > 0");
        for (int d = 0; d < 3; ++d)
            if (fine->geo.ne[d] != coarse->geo.ne[d] || fine->geo.h[d] != coarse->geo.h[d] ||
                fine->geo.lo[d] != coarse->geo.lo[d])
                throw std::invalid_argument("fine and coarse solvers must share the mesh");
        if (fine->device != coarse->device) throw std::invalid_argument("the solvers live on different devices");
        hcheck(hipSetDevice(fine->device), "hipSetDevice");
        const long E = fine->geo.E;
        tendency(fine, Uf_dev, fine->Ub);
        hcheck(hipStreamSynchronize(fine->stream), "hipStreamSynchronize");
        tendency(coarse, Uc_dev, coarse->Ub);
        hcheck(hipStreamSynchronize(coarse->stream), "hipStreamSynchronize");
        hipLaunchKernelGGL(target_at_kernel, dim3(nblk(E * 40)), dim3(TB), 0, fine->stream, fine->Ub, coarse->Ub,
                           Uf_dev, Uc_dev, 1.0 / tau, Y_dev, fine->P, E);
        hcheck(hipGetLastError(), "target kernel");
        hcheck(hipStreamSynchronize(fine->stream), "hipStreamSynchronize");
    });
}

int dg_closure_step(dg_solver* s, dg_mlp* m, double dt_step, double bound, int nsteps, long* n_fallback) {
    return mlp_guard(g_mlp_error, [&] {
        const double dt = closure_check(s, m, dt_step, nsteps);
        const long E = s->geo.E;
        // the corrections and the counter live on the solver handle from the
        // first call on (freed by dg_destroy)
        if (!s->cl_C) hcheck(dg::device_malloc(&s->cl_C, (size_t)E * NO * sizeof(float)), "hipMalloc");
        if (!s->cl_cnt) hcheck(dg::device_malloc(&s->cl_cnt, sizeof(unsigned long long)), "hipMalloc");
        closure_steps(s, m, dt, bound, nsteps, s->cl_C, s->cl_cnt, n_fallback);
    });
}

int dg_closure_step_noalloc(dg_solver* s, dg_mlp* m, double dt_step, double bound, int nsteps, long* n_fallback) {
    return mlp_guard(g_mlp_error, [&] {
        const double dt = closure_check(s, m, dt_step, nsteps);
        const long E = s->geo.E;
        if (E > NOALLOC_MAX_ELEMS)
            throw std::invalid_argument("dg_closure_step_noalloc: " + std::to_string(E) + " elements exceed the " +
                                        std::to_string(NOALLOC_MAX_ELEMS) + " of its static scratch (use dg_closure_step)");
        // the device is current (closure_check): its own copy of the array
        float* base = noalloc_scratch(s->device);
        float* C = base;
        auto* cnt = reinterpret_cast<unsigned long long*>(base + NOALLOC_C);
        closure_steps(s, m, dt, bound, nsteps, C, cnt, n_fallback);
    });
}

}  // extern "C"
