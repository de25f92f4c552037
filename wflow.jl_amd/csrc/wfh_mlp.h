// wfh_mlp.h - the learned Newton warm start: an 8-64-64-1 perceptron with BF16 weights and
// activations and FP32 accumulation, evaluated and trained with gfx950 matrix-core instructions
// (v_mfma_f32_32x32x16_bf16), one wave per 64 samples. Included by wflow_hip.hip.
//
// Network (unit indices 0..63 of both hidden layers are the matrix-core row indices below):
//   z1 = W1 x + b1,  h1 = bf16(relu(z1))          W1: [64][8]  (x: 8 normalised features, bf16)
//   z2 = W2 h1 + b2, h2 = relu(z2)                 W2: [64][64]
//   y  = w3 . h2 + b3                              w3: [64] (FP32)
// Training minimises the mean squared error with Adam on FP32 master weights; the BF16 operand
// copies are re-derived after every update. The backward pass rounds the output gradient of
// layer 2 and of layer 1 to BF16 where they enter a matrix-core product.
//
// Matrix-core lane layouts (checked on the device by tests/test_gpu_mlp.py):
//   A (32x16): lane l holds row l % 32, k = 8 (l / 32) + j, j = 0..7
//   B (16x32): lane l holds col l % 32, k = 8 (l / 32) + j
//   D (32x32): lane l, register r holds row 8 (r / 4) + 4 (l / 32) + r % 4, col l % 32
// Samples are columns: lane l owns sample l; a column block c holds samples 32 c .. 32 c + 31.
// A layer's D tile can be the next layer's B operand without moving data between lanes when the
// next layer's k positions are the D rows in register order: k position 16 kb + 8 h + j of
// in-block kb (0, 1) of a 32-unit block is unit 8 (2 kb + j / 4) + 4 h + j % 4 of that block.

namespace {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x16 __attribute__((ext_vector_type(16)));

constexpr int MLP_IN = 8, MLP_H = 64;
// flat parameter vector: W1 [64][8], b1 [64], W2 [64][64], b2 [64], w3 [64], b3
constexpr int MLP_OW1 = 0, MLP_OB1 = MLP_OW1 + MLP_H * MLP_IN, MLP_OW2 = MLP_OB1 + MLP_H,
              MLP_OB2 = MLP_OW2 + MLP_H * MLP_H, MLP_OW3 = MLP_OB2 + MLP_H, MLP_OB3 = MLP_OW3 + MLP_H,
              MLP_NPARAM = MLP_OB3 + 1;

// in-unit of k position (kb2 = 0..3 over 64 units, lane half h, j = 0..7)
__host__ __device__ inline int mlp_kunit(int kb2, int h, int j) {
    return 32 * (kb2 >> 1) + 8 * (2 * (kb2 & 1) + (j >> 2)) + 4 * h + (j & 3);
}
// unit held by lane half h, register r of a D tile of row block rb
__host__ __device__ inline int mlp_dunit(int rb, int h, int r) { return 32 * rb + 8 * (r >> 2) + 4 * h + (r & 3); }

// Operand copies of the weights (device), in the order one lane reads them.
struct MlpOps {
    bf16x8 a1[2][64];        // layer 1, row block hb: lane < 32 W1[32 hb + lane][0..7], lane >= 32 zero
    bf16x8 a2[2][4][64];     // layer 2, row block ob, k block kb2: W2[32 ob + l % 32][kunit(kb2, l / 32, j)]
    bf16x8 a2t[2][4][64];    // W2 transposed (backward): W2[kunit(kb2, l / 32, j)][32 ub + l % 32]
    float b1[2][2][16];      // [row block][lane half][register]: b1 of the unit in that D slot
    float b2[2][2][16];
    float w3[2][2][16];
    float b3;
    float x_mean[MLP_IN], x_inv_std[MLP_IN];  // feature normalisation
    float y_mean, y_std;                      // target scaling
};

__device__ __forceinline__ bf16x8 bf8_zero() {
    bf16x8 z;
#pragma unroll
    for (int j = 0; j < 8; ++j) z[j] = (__bf16)0.0f;
    return z;
}

__device__ __forceinline__ bf16x8 shfl_bf8(const bf16x8 v, const int src) {
    union {
        bf16x8 b;
        int w[4];
    } u;
    u.b = v;
#pragma unroll
    for (int k = 0; k < 4; ++k) u.w[k] = __shfl(u.w[k], src);
    return u.b;
}

// Forward pass of one wave: lane l's normalised features x (8 floats) -> network output
// (normalised target space). With T != nullptr the intermediate tiles are kept for the backward
// pass: z1/z2 pre-activations (with bias) per column block.
struct MlpTape {
    f32x16 z1[2][2];  // [column block][row block]
    f32x16 z2[2][2];
    bf16x8 xb;        // own features (bf16)
};

__device__ __forceinline__ float mlp_forward(const MlpOps& W, const float* x, MlpTape* T) {
    const int lane = threadIdx.x & 63, h = lane >> 5;
    bf16x8 xb;
#pragma unroll
    for (int j = 0; j < 8; ++j) xb[j] = (__bf16)((x[j] - W.x_mean[j]) * W.x_inv_std[j]);
    if (T) T->xb = xb;
    const bf16x8 xhi = shfl_bf8(xb, (lane & 31) + 32);
    float part[2];
#pragma unroll
    for (int c = 0; c < 2; ++c) {
        const bf16x8 b1op = h ? bf8_zero() : (c == 0 ? xb : xhi);
        bf16x8 b2op[4];
#pragma unroll
        for (int hb = 0; hb < 2; ++hb) {
            f32x16 z = {};
            z = __builtin_amdgcn_mfma_f32_32x32x16_bf16(W.a1[hb][lane], b1op, z, 0, 0, 0);
#pragma unroll
            for (int r = 0; r < 16; ++r) z[r] += W.b1[hb][h][r];
            if (T) T->z1[c][hb] = z;
#pragma unroll
            for (int kb = 0; kb < 2; ++kb)
#pragma unroll
                for (int j = 0; j < 8; ++j) b2op[2 * hb + kb][j] = (__bf16)fmaxf(z[8 * kb + j], 0.0f);
        }
        float acc = 0.0f;
#pragma unroll
        for (int ob = 0; ob < 2; ++ob) {
            f32x16 z = {};
#pragma unroll
            for (int kb2 = 0; kb2 < 4; ++kb2)
                z = __builtin_amdgcn_mfma_f32_32x32x16_bf16(W.a2[ob][kb2][lane], b2op[kb2], z, 0, 0, 0);
#pragma unroll
            for (int r = 0; r < 16; ++r) {
                z[r] += W.b2[ob][h][r];
                acc += fmaxf(z[r], 0.0f) * W.w3[ob][h][r];
            }
            if (T) T->z2[c][ob] = z;
        }
        part[c] = acc + __shfl_xor(acc, 32);
    }
    return (h ? part[1] : part[0]) + W.b3;
}

// The forward pass as a call of its own, with the weights read from global memory (L2): for
// callers that consult the network rarely, so that their own register allocation and LDS are
// not shaped by it.
__device__ __noinline__ float mlp_forward_call(const MlpOps* W, float x0, float x1, float x2, float x3, float x4,
                                               float x5, float x6, float x7) {
    const float x[8] = {x0, x1, x2, x3, x4, x5, x6, x7};
    return mlp_forward(*W, x, nullptr);
}

// ---- training ----------------------------------------------------------------------------
// One block of four waves takes 256 samples of x [n][8], t [n] (normalised targets), wave w the
// tile of samples 64 w .. 64 w + 63: partial gradients of the mean squared error over n samples
// into part[blockIdx.x][MLP_NPARAM], loss sum into loss[blockIdx.x].
// A minibatch has few blocks (32 for 8192 samples), so the time of one block is what counts: the
// four tiles run side by side, the products over the samples are split by quadrant of W2 (one per
// wave, samples in ascending order), and a unit's sum over the samples is a left fold by one lane
// over a row in LDS, the order in which LDS atomics of one wave would add.
// Measured: an epoch of 300,000 rows in minibatches of 8192 5.10 -> 0.81 ms (17 us for this kernel
// and 4.7 us for the Adam step a minibatch; one wave with four tiles in a row and LDS atomics per unit,
// an Adam step, a layout launch and a read-back of the loss took 138 us). Bound by latency: 32 of 256
// CUs have work.
constexpr int MLP_GS = 256;                // samples of a block
constexpr int MLP_FP = MLP_GS + 4;         // row pitch of the float tile: 16-byte rows, lanes on distinct banks
constexpr int MLP_BP = MLP_GS + 8;         // row pitch of the bf16 tiles
__global__ void __launch_bounds__(256) k_mlp_grad(const MlpOps* __restrict__ Wp, const float* __restrict__ x,
                                                  const float* __restrict__ t, long long n, float inv_n,
                                                  float* __restrict__ part, float* __restrict__ loss) {
    __shared__ __attribute__((aligned(16))) float F[MLP_H][MLP_FP];    // [unit][sample]: relu(z2), then dz1
    __shared__ __attribute__((aligned(16))) __bf16 G[MLP_H][MLP_BP];   // [unit][sample]: layer output gradients
    __shared__ __attribute__((aligned(16))) __bf16 H[MLP_H][MLP_BP];   // [unit][sample]: h1
    __shared__ __attribute__((aligned(16))) __bf16 XT[MLP_IN][MLP_BP]; // [feature][sample]
    __shared__ __attribute__((aligned(16))) float DY[MLP_GS];
    __shared__ float ERR[MLP_GS];
    const MlpOps& W = *Wp;
    const int lane = threadIdx.x & 63, h = lane >> 5, col = lane & 31;
    const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    const int s0 = 64 * wave;  // the wave's first sample in the block
    float* P = part + (size_t)blockIdx.x * MLP_NPARAM;
    f32x16 g1[2][2];  // dz1 of the wave's tile: [column block][row block]
    {
        const long long s = (long long)blockIdx.x * MLP_GS + s0 + lane;
        const bool valid = s < n;
        float xv[8];
#pragma unroll
        for (int j = 0; j < 8; ++j) xv[j] = valid ? x[s * 8 + j] : W.x_mean[j];
        const float tv = valid ? t[s] : 0.0f;
        MlpTape T;
        const float y = mlp_forward(W, xv, &T);
        const float err = valid ? y - tv : 0.0f;
        const float dy = 2.0f * err * inv_n;
        DY[s0 + lane] = dy;
        ERR[s0 + lane] = err;
#pragma unroll
        for (int j = 0; j < 8; ++j) XT[j][s0 + lane] = T.xb[j];
#pragma unroll
        for (int c = 0; c < 2; ++c) {
            const int sc = s0 + 32 * c + col;
#pragma unroll
            for (int hb = 0; hb < 2; ++hb)
#pragma unroll
                for (int r = 0; r < 16; ++r) H[mlp_dunit(hb, h, r)][sc] = (__bf16)fmaxf(T.z1[c][hb][r], 0.0f);
            // layer 2 output gradients
            const float dyc = __shfl(dy, 32 * c + col);
            bf16x8 bg[4];
#pragma unroll
            for (int ob = 0; ob < 2; ++ob)
#pragma unroll
                for (int r = 0; r < 16; ++r) {
                    const float z = T.z2[c][ob][r];
                    const int u = mlp_dunit(ob, h, r);
                    const __bf16 g = (__bf16)(z > 0.0f ? W.w3[ob][h][r] * dyc : 0.0f);
                    F[u][sc] = fmaxf(z, 0.0f);
                    G[u][sc] = g;
                    bg[2 * ob + (r >> 3)][r & 7] = g;
                }
            // dh1 = W2^T g2 (B from the g2 tiles in register order), dz1 = dh1 (z1 > 0)
#pragma unroll
            for (int ub = 0; ub < 2; ++ub) {
                f32x16 d = {};
#pragma unroll
                for (int kb2 = 0; kb2 < 4; ++kb2)
                    d = __builtin_amdgcn_mfma_f32_32x32x16_bf16(W.a2t[ub][kb2][lane], bg[kb2], d, 0, 0, 0);
#pragma unroll
                for (int r = 0; r < 16; ++r) g1[c][ub][r] = T.z1[c][ub][r] > 0.0f ? d[r] : 0.0f;
            }
        }
    }
    __syncthreads();
    // dW2 = G h1^T over the block's samples (k = samples), quadrant (vb, ub) by wave
    {
        const int vb = wave >> 1, ub = wave & 1;
        f32x16 g = {};
#pragma unroll
        for (int kb = 0; kb < MLP_GS / 16; ++kb) {
            const bf16x8 a = *reinterpret_cast<const bf16x8*>(&G[32 * vb + col][16 * kb + 8 * h]);
            const bf16x8 b = *reinterpret_cast<const bf16x8*>(&H[32 * ub + col][16 * kb + 8 * h]);
            g = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b, g, 0, 0, 0);
        }
#pragma unroll
        for (int r = 0; r < 16; ++r) P[MLP_OW2 + mlp_dunit(vb, h, r) * MLP_H + 32 * ub + col] = g[r];
    }
    // sums over the samples: dw3 (wave 0), db2 (wave 1), one unit per lane; db3 and the loss (wave 2)
    if (wave == 0) {
        float acc = 0.0f;
#pragma unroll 16
        for (int s = 0; s < MLP_GS; s += 4) {
            const float4 z = *reinterpret_cast<const float4*>(&F[lane][s]);
            const float4 d = *reinterpret_cast<const float4*>(&DY[s]);
            acc += z.x * d.x;
            acc += z.y * d.y;
            acc += z.z * d.z;
            acc += z.w * d.w;
        }
        P[MLP_OW3 + lane] = acc;
    } else if (wave == 1) {
        const float w3 = W.w3[h][(lane >> 2) & 1][4 * ((lane & 31) >> 3) + (lane & 3)];
        float acc = 0.0f;
#pragma unroll 16
        for (int s = 0; s < MLP_GS; s += 4) {
            const float4 z = *reinterpret_cast<const float4*>(&F[lane][s]);
            const float4 d = *reinterpret_cast<const float4*>(&DY[s]);
            acc += z.x > 0.0f ? w3 * d.x : 0.0f;
            acc += z.y > 0.0f ? w3 * d.y : 0.0f;
            acc += z.z > 0.0f ? w3 * d.z : 0.0f;
            acc += z.w > 0.0f ? w3 * d.w : 0.0f;
        }
        P[MLP_OB2 + lane] = acc;
    } else if (wave == 2) {
        float gb3 = 0.0f, lsum = 0.0f;
#pragma unroll
        for (int k = 0; k < MLP_GS; k += 64) {
            lsum += ERR[k + lane] * ERR[k + lane];
            gb3 += DY[k + lane];
        }
#pragma unroll
        for (int mask = 1; mask < 64; mask <<= 1) {
            gb3 += __shfl_xor(gb3, mask);
            lsum += __shfl_xor(lsum, mask);
        }
        if (lane == 0) {
            P[MLP_OB3] = gb3;
            loss[blockIdx.x] = lsum;
        }
    }
    __syncthreads();
#pragma unroll
    for (int c = 0; c < 2; ++c)
#pragma unroll
        for (int ub = 0; ub < 2; ++ub)
#pragma unroll
            for (int r = 0; r < 16; ++r) {
                const int u = mlp_dunit(ub, h, r), sc = s0 + 32 * c + col;
                F[u][sc] = g1[c][ub][r];
                G[u][sc] = (__bf16)g1[c][ub][r];
            }
    __syncthreads();
    if (wave < 2) {
        // dW1 = dz1 x^T, row block by wave (B columns beyond the 8 features are zero)
        f32x16 g = {};
#pragma unroll
        for (int kb = 0; kb < MLP_GS / 16; ++kb) {
            const bf16x8 a = *reinterpret_cast<const bf16x8*>(&G[32 * wave + col][16 * kb + 8 * h]);
            const bf16x8 b = col < 8 ? *reinterpret_cast<const bf16x8*>(&XT[col & 7][16 * kb + 8 * h]) : bf8_zero();
            g = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b, g, 0, 0, 0);
        }
#pragma unroll
        for (int r = 0; r < 16; ++r)
            if (col < 8) P[MLP_OW1 + mlp_dunit(wave, h, r) * MLP_IN + col] = g[r];
    } else if (wave == 2) {
        float acc = 0.0f;
#pragma unroll 16
        for (int s = 0; s < MLP_GS; s += 4) {
            const float4 g = *reinterpret_cast<const float4*>(&F[lane][s]);
            acc += g.x;
            acc += g.y;
            acc += g.z;
            acc += g.w;
        }
        P[MLP_OB1 + lane] = acc;
    }
}

// lane half and register of unit u in a D tile (inverse of mlp_dunit), and lane half and j of
// in-unit u in a k block (inverse of mlp_kunit; the k block is 2 (u / 32) + (u / 16) % 2)
__device__ inline int mlp_unit_half(int u) { return (u >> 2) & 1; }
__device__ inline int mlp_unit_reg(int u) { return 4 * ((u & 31) >> 3) + (u & 3); }
__device__ inline int mlp_unit_j(int u) { return 4 * ((u >> 3) & 1) + (u & 3); }

// The operand copies of one master parameter (flat index i).
__device__ __forceinline__ void mlp_put(MlpOps* __restrict__ W, const int i, const float v) {
    if (i < MLP_OB1) {
        const int u = i / MLP_IN;
        W->a1[u >> 5][u & 31][i % MLP_IN] = (__bf16)v;
    } else if (i >= MLP_OW2 && i < MLP_OB2) {
        const int o = (i - MLP_OW2) / MLP_H, u = (i - MLP_OW2) % MLP_H;  // W2[o][u]
        W->a2[o >> 5][u >> 4][32 * mlp_unit_half(u) + (o & 31)][mlp_unit_j(u)] = (__bf16)v;
        W->a2t[u >> 5][o >> 4][32 * mlp_unit_half(o) + (u & 31)][mlp_unit_j(o)] = (__bf16)v;
    } else if (i == MLP_OB3) {
        W->b3 = v;
    } else {
        const int u = i < MLP_OW2 ? i - MLP_OB1 : i < MLP_OW3 ? i - MLP_OB2 : i - MLP_OW3;
        float* q = i < MLP_OW2 ? &W->b1[0][0][0] : i < MLP_OW3 ? &W->b2[0][0][0] : &W->w3[0][0][0];
        q[32 * (u >> 5) + 16 * mlp_unit_half(u) + mlp_unit_reg(u)] = v;
    }
}

// Sum of the per-block partial gradients in block order, then one Adam step on the FP32 master
// parameters and their operand copies (adam_t = the step number, 1-based; lr = 0 leaves the
// parameters, moments and copies unchanged and only sums the gradient into grad). One wave per
// block: the loads of one parameter's column of partials are what takes the time, so they are
// spread over the CUs and kept 32 in flight.
__global__ void __launch_bounds__(64) k_mlp_adam(const float* __restrict__ part, int nblocks, float* __restrict__ p,
                                                 float* __restrict__ m1, float* __restrict__ m2,
                                                 float* __restrict__ grad, MlpOps* __restrict__ W, float lr,
                                                 int adam_t) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= MLP_NPARAM) return;
    float g = 0.0f;
    int b = 0;
    for (; b + 32 <= nblocks; b += 32) {
        float v[32];
#pragma unroll
        for (int k = 0; k < 32; ++k) v[k] = part[(size_t)(b + k) * MLP_NPARAM + i];
#pragma unroll
        for (int k = 0; k < 32; ++k) g += v[k];
    }
    for (; b < nblocks; ++b) g += part[(size_t)b * MLP_NPARAM + i];
    grad[i] = g;
    if (lr == 0.0f) return;
    const float be1 = 0.9f, be2 = 0.999f;
    m1[i] = be1 * m1[i] + (1.0f - be1) * g;
    m2[i] = be2 * m2[i] + (1.0f - be2) * g * g;
    const float mh = m1[i] / (1.0f - powf(be1, (float)adam_t));
    const float vh = m2[i] / (1.0f - powf(be2, (float)adam_t));
    const float v = p[i] - lr * mh / (sqrtf(vh) + 1e-8f);
    p[i] = v;
    mlp_put(W, i, v);
}

// Operand copies from the master parameters (one block of 256 threads).
__global__ void k_mlp_layout(const float* __restrict__ p, MlpOps* __restrict__ W) {
    for (int idx = threadIdx.x; idx < 2 * 64; idx += blockDim.x) {  // a1
        const int hb = idx / 64, l = idx % 64;
        bf16x8 v;
#pragma unroll
        for (int j = 0; j < 8; ++j)
            v[j] = (__bf16)(l < 32 ? p[MLP_OW1 + (32 * hb + l) * MLP_IN + j] : 0.0f);
        W->a1[hb][l] = v;
    }
    for (int idx = threadIdx.x; idx < 2 * 4 * 64; idx += blockDim.x) {  // a2, a2t
        const int ob = idx / 256, kb2 = (idx / 64) % 4, l = idx % 64;
        bf16x8 v, vt;
#pragma unroll
        for (int j = 0; j < 8; ++j) {
            const int u = mlp_kunit(kb2, l >> 5, j);
            v[j] = (__bf16)p[MLP_OW2 + (32 * ob + (l & 31)) * MLP_H + u];
            vt[j] = (__bf16)p[MLP_OW2 + u * MLP_H + 32 * ob + (l & 31)];
        }
        W->a2[ob][kb2][l] = v;
        W->a2t[ob][kb2][l] = vt;
    }
    for (int idx = threadIdx.x; idx < 2 * 2 * 16; idx += blockDim.x) {
        const int rb = idx / 32, hh = (idx / 16) % 2, r = idx % 16;
        const int u = mlp_dunit(rb, hh, r);
        W->b1[rb][hh][r] = p[MLP_OB1 + u];
        W->b2[rb][hh][r] = p[MLP_OB2 + u];
        W->w3[rb][hh][r] = p[MLP_OW3 + u];
    }
    if (threadIdx.x == 0) W->b3 = p[MLP_OB3];
}

// Network outputs (normalised target space) for n samples x [n][8], tiles of 64 samples dealt to
// the waves in turn. A wave holds all weights in registers (136 of the 256 that two waves per SIMD
// leave) and loads the next tile's rows while it computes one, so a tile moves its 36 B a sample
// and nothing else. One million rows: 48 -> 29 us for the call, 21 us of it this kernel (four-byte
// copies of the 20 KB of operands into LDS for every 256 samples took the time before); bound by the
// VALU work between the products. The operations are mlp_forward's, except that layer 2 starts its products from
// the bias and folds the output with fused multiply-adds (nothing is rounded to bf16 after them).
// VEC: x is 16-byte aligned, rows are read as two float4.
template <bool VEC>
__device__ __forceinline__ void mlp_row(const float* __restrict__ x, const long long s, float* v) {
    if (VEC) {
        const float4 a = reinterpret_cast<const float4*>(x)[2 * s], b = reinterpret_cast<const float4*>(x)[2 * s + 1];
        v[0] = a.x, v[1] = a.y, v[2] = a.z, v[3] = a.w, v[4] = b.x, v[5] = b.y, v[6] = b.z, v[7] = b.w;
    } else {
#pragma unroll
        for (int j = 0; j < 8; ++j) v[j] = x[s * 8 + j];
    }
}

template <bool VEC>
__global__ void __launch_bounds__(256, 2) k_mlp_predict(const MlpOps* __restrict__ Wp, const float* __restrict__ x,
                                                        long long n, float* __restrict__ y) {
    const MlpOps& W = *Wp;
    const int lane = threadIdx.x & 63, h = lane >> 5;
    const long long stride = (long long)gridDim.x * blockDim.x;
    long long s = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    const bool any = s - lane < n;  // the wave has a tile (uniform; a lane past n repeats the last row)
    if (!any) return;
    float xv[8];
    mlp_row<VEC>(x, s < n ? s : n - 1, xv);
    bf16x8 a1[2], a2[2][4];
    f32x16 b1[2], b2[2], w3[2];
#pragma unroll
    for (int rb = 0; rb < 2; ++rb) {
        a1[rb] = W.a1[rb][lane];
#pragma unroll
        for (int k = 0; k < 4; ++k) a2[rb][k] = W.a2[rb][k][lane];
#pragma unroll
        for (int r = 0; r < 16; ++r) b1[rb][r] = W.b1[rb][h][r], b2[rb][r] = W.b2[rb][h][r], w3[rb][r] = W.w3[rb][h][r];
    }
    const float b3 = W.b3;
    float mean[8], inv[8];
#pragma unroll
    for (int j = 0; j < 8; ++j) mean[j] = W.x_mean[j], inv[j] = W.x_inv_std[j];
    for (; s - lane < n; s += stride) {
        bf16x8 xb;
#pragma unroll
        for (int j = 0; j < 8; ++j) xb[j] = (__bf16)((xv[j] - mean[j]) * inv[j]);
        const long long sn = s + stride;
        if (sn - lane < n) mlp_row<VEC>(x, sn < n ? sn : n - 1, xv);
        const bf16x8 xhi = shfl_bf8(xb, (lane & 31) + 32);
        float part[2];
#pragma unroll
        for (int c = 0; c < 2; ++c) {
            const bf16x8 b1op = h ? bf8_zero() : (c == 0 ? xb : xhi);
            bf16x8 b2op[4];
#pragma unroll
            for (int hb = 0; hb < 2; ++hb) {
                f32x16 z = {};
                z = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a1[hb], b1op, z, 0, 0, 0);
#pragma unroll
                for (int r = 0; r < 16; ++r) b2op[2 * hb + (r >> 3)][r & 7] = (__bf16)fmaxf(z[r] + b1[hb][r], 0.0f);
            }
            float acc[2] = {0.0f, 0.0f};
#pragma unroll
            for (int ob = 0; ob < 2; ++ob) {
                f32x16 z = b2[ob];
#pragma unroll
                for (int k = 0; k < 4; ++k)
                    z = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a2[ob][k], b2op[k], z, 0, 0, 0);
#pragma unroll
                for (int r = 0; r < 16; ++r) acc[ob] = __builtin_fmaf(fmaxf(z[r], 0.0f), w3[ob][r], acc[ob]);
            }
            const float a = acc[0] + acc[1];
            part[c] = a + __shfl_xor(a, 32);
        }
        if (s < n) y[s] = (h ? part[1] : part[0]) + b3;
    }
}

}  // namespace

struct wfh_mlp {
    int device = 0;
    hipStream_t stream = nullptr;
    float *p = nullptr, *m1 = nullptr, *m2 = nullptr, *grad = nullptr;  // master parameters, Adam moments
    MlpOps* ops = nullptr;
    MlpOps host_ops{};
    float* part = nullptr;
    float* loss = nullptr;
    int64_t part_blocks = 0, loss_blocks = 0;
    int adam_t = 0;
    std::string err;
};

namespace {
int32_t mfail(wfh_mlp* x, int32_t code, const std::string& msg) {
    if (x) x->err = msg;
    return code;
}
#define MHIP(x, call)                                                                                          \
    do {                                                                                                       \
        hipError_t e_ = (call);                                                                                \
        if (e_ != hipSuccess) return mfail((x), WFH_ERR_HIP, std::string(#call ": ") + hipGetErrorString(e_)); \
    } while (0)

int32_t mlp_relayout(wfh_mlp* x) {
    // normalisation lives in the host copy; the kernel fills the operand part
    MHIP(x, hipMemcpyAsync(x->ops, &x->host_ops, sizeof(MlpOps), hipMemcpyHostToDevice, x->stream));
    hipLaunchKernelGGL(k_mlp_layout, dim3(1), dim3(256), 0, x->stream, x->p, x->ops);
    MHIP(x, hipGetLastError());
    return WFH_OK;
}

// room for the partial gradients of `blocks` blocks and the loss sums of `losses`
int32_t mlp_ensure_part(wfh_mlp* x, int64_t blocks, int64_t losses) {
    if (blocks > x->part_blocks) {
        if (x->part) hipFree(x->part);
        x->part = nullptr;
        x->part_blocks = 0;
        MHIP(x, hipMalloc(&x->part, (size_t)blocks * MLP_NPARAM * sizeof(float)));
        x->part_blocks = blocks;
    }
    if (losses > x->loss_blocks) {
        if (x->loss) hipFree(x->loss);
        x->loss = nullptr;
        x->loss_blocks = 0;
        MHIP(x, hipMalloc(&x->loss, (size_t)losses * sizeof(float)));
        x->loss_blocks = losses;
    }
    return WFH_OK;
}
}  // namespace

extern "C" int32_t wfh_mlp_create(int32_t device, uint64_t seed, wfh_mlp** out) {
    if (!out) return WFH_ERR_ARG;
    *out = nullptr;
    wfh_mlp* x = new wfh_mlp();
    x->device = device;
    auto bail = [&](int32_t code, const std::string& m) {
        g_create_error = m;
        wfh_mlp_destroy(x);
        return code;
    };
    if (hipSetDevice(device) != hipSuccess || hipStreamCreate(&x->stream) != hipSuccess)
        return bail(WFH_ERR_HIP, "mlp: device / stream");
    if (hipMalloc(&x->p, MLP_NPARAM * sizeof(float)) != hipSuccess ||
        hipMalloc(&x->m1, MLP_NPARAM * sizeof(float)) != hipSuccess ||
        hipMalloc(&x->m2, MLP_NPARAM * sizeof(float)) != hipSuccess ||
        hipMalloc(&x->grad, MLP_NPARAM * sizeof(float)) != hipSuccess ||
        hipMalloc(&x->ops, sizeof(MlpOps)) != hipSuccess)
        return bail(WFH_ERR_HIP, "mlp: hipMalloc");
    // He-uniform initialisation from a 64-bit LCG (reproducible for a seed)
    std::vector<float> p(MLP_NPARAM, 0.0f), z(MLP_NPARAM, 0.0f);
    uint64_t st = seed * 6364136223846793005ULL + 1442695040888963407ULL;
    auto uni = [&]() {
        st = st * 6364136223846793005ULL + 1442695040888963407ULL;
        return (double)(st >> 11) * (1.0 / 9007199254740992.0) * 2.0 - 1.0;
    };
    for (int i = 0; i < MLP_H * MLP_IN; ++i) p[MLP_OW1 + i] = (float)(uni() * std::sqrt(6.0 / MLP_IN));
    for (int i = 0; i < MLP_H * MLP_H; ++i) p[MLP_OW2 + i] = (float)(uni() * std::sqrt(6.0 / MLP_H));
    for (int i = 0; i < MLP_H; ++i) p[MLP_OW3 + i] = (float)(uni() * std::sqrt(3.0 / MLP_H));
    if (hipMemcpy(x->p, p.data(), MLP_NPARAM * sizeof(float), hipMemcpyHostToDevice) != hipSuccess ||
        hipMemcpy(x->m1, z.data(), MLP_NPARAM * sizeof(float), hipMemcpyHostToDevice) != hipSuccess ||
        hipMemcpy(x->m2, z.data(), MLP_NPARAM * sizeof(float), hipMemcpyHostToDevice) != hipSuccess)
        return bail(WFH_ERR_HIP, "mlp: upload");
    for (int j = 0; j < MLP_IN; ++j) {
        x->host_ops.x_mean[j] = 0.0f;
        x->host_ops.x_inv_std[j] = 1.0f;
    }
    x->host_ops.y_mean = 0.0f;
    x->host_ops.y_std = 1.0f;
    if (mlp_relayout(x) || hipStreamSynchronize(x->stream) != hipSuccess) return bail(WFH_ERR_HIP, "mlp: layout");
    *out = x;
    return WFH_OK;
}

extern "C" int32_t wfh_mlp_set_normalization(wfh_mlp* x, const float* x_mean, const float* x_std, float y_mean,
                                             float y_std) {
    if (!x || !x_mean || !x_std) return WFH_ERR_ARG;
    for (int j = 0; j < MLP_IN; ++j) {
        if (!(x_std[j] > 0.0f) || !std::isfinite(x_mean[j])) return mfail(x, WFH_ERR_ARG, "bad normalisation");
        x->host_ops.x_mean[j] = x_mean[j];
        x->host_ops.x_inv_std[j] = 1.0f / x_std[j];
    }
    if (!(y_std > 0.0f) || !std::isfinite(y_mean)) return mfail(x, WFH_ERR_ARG, "bad target scaling");
    x->host_ops.y_mean = y_mean;
    x->host_ops.y_std = y_std;
    MHIP(x, hipSetDevice(x->device));
    int32_t rc = mlp_relayout(x);
    if (rc) return rc;
    MHIP(x, hipStreamSynchronize(x->stream));
    return WFH_OK;
}

// params: [MLP_NPARAM] host floats in the flat order W1, b1, W2, b2, w3, b3
extern "C" int32_t wfh_mlp_set_params(wfh_mlp* x, const float* params) {
    if (!x || !params) return WFH_ERR_ARG;
    MHIP(x, hipSetDevice(x->device));
    MHIP(x, hipMemcpy(x->p, params, MLP_NPARAM * sizeof(float), hipMemcpyHostToDevice));
    int32_t rc = mlp_relayout(x);
    if (rc) return rc;
    MHIP(x, hipStreamSynchronize(x->stream));
    return WFH_OK;
}

extern "C" int32_t wfh_mlp_get_params(wfh_mlp* x, float* params) {
    if (!x || !params) return WFH_ERR_ARG;
    MHIP(x, hipSetDevice(x->device));
    MHIP(x, hipStreamSynchronize(x->stream));
    MHIP(x, hipMemcpy(params, x->p, MLP_NPARAM * sizeof(float), hipMemcpyDeviceToHost));
    return WFH_OK;
}

// One pass over n samples (device arrays x [n][8], t [n] normalised targets) in minibatches of
// `batch` samples (a multiple of 64), one Adam step each (lr > 0), or with lr = 0 one gradient
// of the whole set (no update). Returns the mean squared error of the pass in *loss and the
// last minibatch's gradient (the whole set's with lr = 0) in grad (host, [MLP_NPARAM]) if given.
extern "C" int32_t wfh_mlp_train(wfh_mlp* x, const float* xs, const float* ts, int64_t n, int64_t batch, float lr,
                                 double* loss, float* grad) {
    if (!x || !xs || !ts || n <= 0) return WFH_ERR_ARG;
    if (lr == 0.0f) batch = ((n + 63) / 64) * 64;
    if (batch < 64 || batch % 64) return mfail(x, WFH_ERR_ARG, "batch must be a positive multiple of 64");
    MHIP(x, hipSetDevice(x->device));
    // the loss sums of every minibatch's blocks are kept and read back once, at the end
    const auto nblocks = [](int64_t rows) { return (rows + MLP_GS - 1) / MLP_GS; };
    const int64_t full = n / batch, rest = n % batch;
    const int64_t total = full * nblocks(batch) + nblocks(rest);
    int32_t rc = mlp_ensure_part(x, nblocks(std::min<int64_t>(batch, n)), total);
    if (rc) return rc;
    float* lossp = x->loss;
    for (int64_t s0 = 0; s0 < n; s0 += batch) {
        const int64_t nb = std::min<int64_t>(batch, n - s0);
        const int blocks = (int)nblocks(nb);
        hipLaunchKernelGGL(k_mlp_grad, dim3(blocks), dim3(256), 0, x->stream, (const MlpOps*)x->ops, xs + s0 * 8,
                           ts + s0, (long long)nb, 1.0f / (float)nb, x->part, lossp);
        if (lr != 0.0f) ++x->adam_t;
        hipLaunchKernelGGL(k_mlp_adam, dim3((MLP_NPARAM + 63) / 64), dim3(64), 0, x->stream, (const float*)x->part,
                           blocks, x->p, x->m1, x->m2, x->grad, x->ops, lr, x->adam_t);
        MHIP(x, hipGetLastError());
        lossp += blocks;
    }
    std::vector<float> lbuf(total);
    MHIP(x, hipMemcpyAsync(lbuf.data(), x->loss, total * sizeof(float), hipMemcpyDeviceToHost, x->stream));
    MHIP(x, hipStreamSynchronize(x->stream));
    double lsum = 0.0;
    for (float v : lbuf) lsum += v;
    if (loss) *loss = lsum / (double)n;
    if (grad) MHIP(x, hipMemcpy(grad, x->grad, MLP_NPARAM * sizeof(float), hipMemcpyDeviceToHost));
    return WFH_OK;
}

// Network outputs (normalised target space) for device arrays x [n][8] -> y [n].
extern "C" int32_t wfh_mlp_predict(wfh_mlp* x, const float* xs, int64_t n, float* ys) {
    if (!x || !xs || !ys || n < 0) return WFH_ERR_ARG;
    MHIP(x, hipSetDevice(x->device));
    if (n > 0) {
        // a grid of two waves per SIMD (two blocks of four waves on each of 256 CUs) at most: the
        // weights are loaded once per wave. One million rows: 28.9 us, 32.4 with 256 blocks and 29.5 with
        // 1024.
        const unsigned blocks = (unsigned)std::min<int64_t>((n + 255) / 256, 512);
        auto k = reinterpret_cast<uintptr_t>(xs) % 16 == 0 ? k_mlp_predict<true> : k_mlp_predict<false>;
        hipLaunchKernelGGL(k, dim3(blocks), dim3(256), 0, x->stream, (const MlpOps*)x->ops, xs, (long long)n, ys);
    }
    MHIP(x, hipGetLastError());
    MHIP(x, hipStreamSynchronize(x->stream));
    return WFH_OK;
}

extern "C" const char* wfh_mlp_last_error(const wfh_mlp* x) { return x ? x->err.c_str() : g_create_error.c_str(); }

extern "C" void wfh_mlp_destroy(wfh_mlp* x) {
    if (!x) return;
    if (x->stream) hipStreamSynchronize(x->stream);
    for (void* q : {(void*)x->p, (void*)x->m1, (void*)x->m2, (void*)x->grad, (void*)x->ops, (void*)x->part,
                    (void*)x->loss})
        if (q) hipFree(q);
    if (x->stream) hipStreamDestroy(x->stream);
    delete x;
}
