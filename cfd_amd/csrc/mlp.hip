// A small MLP on the matrix cores (gfx950 MFMA, BF16 inputs, FP32
// accumulation): 16 -> 64 -> 64 -> 16 (tanh, tanh, linear), one row per mesh
// node.  It warm-starts the mesh-Laplace solves (see the session); this file
// holds the inference and training kernels.
//
// Layout on the matrix cores: nodes run along the N dimension, so a layer is
// Z(out x nodes) = W^T(out x in) . H(in x nodes) + b.  With
// v_mfma_f32_16x16x16bf16_1k (wave64) lane l holds
//   A[row = l%16][k = 4(l/16)+j],  B[k = 4(l/16)+j][col = l%16],
//   D[row = 4(l/16)+i][col = l%16]           (i, j = 0..3)
// so a layer's D tile (16 outputs x 16 nodes) is, element for element, the B
// operand of the next layer: activations never leave the registers.  Weight
// gradients need dZ and H with nodes along K; those tiles are transposed
// through LDS.
//
// Rounding: inputs, weights, activations fed to the next layer and the
// back-propagated dZ are rounded to BF16 (round to nearest even); accumulations, the output, tanh and bias gradients are FP32.
#include "cfd_internal.hpp"

namespace cfd {

namespace {

typedef short bf16x2 __attribute__((ext_vector_type(2)));
typedef short bf16x4 __attribute__((ext_vector_type(4)));
typedef float f32x4 __attribute__((ext_vector_type(4)));

// round to nearest even, infinities kept, NaN quiet (v_cvt_pk_bf16_f32; an
// integer rounding took five instructions a value)
__device__ __forceinline__ bf16x2 pack2(float a, float b) {
    typedef float f32x2 __attribute__((ext_vector_type(2)));
    typedef __bf16 bfx2 __attribute__((ext_vector_type(2)));
    return __builtin_bit_cast(bf16x2, __builtin_convertvector(f32x2{a, b}, bfx2));
}
__device__ __forceinline__ unsigned short f2bf(float f) { return (unsigned short)pack2(f, f)[0]; }

__device__ __forceinline__ bf16x4 pack4(const f32x4& v) {
    const bf16x2 lo = pack2(v[0], v[1]), hi = pack2(v[2], v[3]);
    return bf16x4{lo[0], lo[1], hi[0], hi[1]};
}

__device__ __forceinline__ f32x4 mfma(bf16x4 a, bf16x4 b, f32x4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(a, b, c, 0, 0, 0);
}

__device__ __forceinline__ bf16x4 load4(const unsigned short* p) {  // p: 8-byte aligned
    return *reinterpret_cast<const bf16x4*>(p);
}
// A operand of W^T (rows = outputs, cols = inputs), tile (mt, kb), from the
// BF16 copy stored row-major [out][in] with `in` columns
__device__ __forceinline__ bf16x4 load_wt(const unsigned short* __restrict__ w, int in, int mt,
                                          int kb, int lane) {
    return load4(w + (size_t)(mt * 16 + (lane & 15)) * in + kb * 16 + 4 * (lane >> 4));
}
// A operand of W (rows = inputs, cols = outputs) from the same [out][in] copy:
// tile (kt, mb) = W[kt*16 + l%16][mb*16 + 4(l/16)+j] = Wt[mb*16 + 4(l/16)+j][kt*16 + l%16]
__device__ __forceinline__ bf16x4 load_w(const unsigned short* __restrict__ w, int in, int kt,
                                         int mb, int lane) {
    const int c = kt * 16 + (lane & 15), r0 = mb * 16 + 4 * (lane >> 4);
    bf16x4 r;
    r[0] = (short)w[(size_t)(r0 + 0) * in + c];
    r[1] = (short)w[(size_t)(r0 + 1) * in + c];
    r[2] = (short)w[(size_t)(r0 + 2) * in + c];
    r[3] = (short)w[(size_t)(r0 + 3) * in + c];
    return r;
}
__device__ __forceinline__ f32x4 bias4(const float* __restrict__ b, int mt, int lane) {
    const float* p = b + mt * 16 + 4 * (lane >> 4);
    f32x4 r;
    r[0] = p[0];
    r[1] = p[1];
    r[2] = p[2];
    r[3] = p[3];
    return r;
}
__device__ __forceinline__ f32x4 tanh4(f32x4 z) {
    f32x4 h;
    for (int i = 0; i < 4; ++i) h[i] = tanhf(z[i]);
    return h;
}

struct MlpDev {
    const unsigned short *w1, *w2, *w3;  // BF16 [out][in]
    const float *b1, *b2, *b3;           // FP32
};

// forward of one tile of 16 nodes; x4 = this lane's B operand of the input
__device__ __forceinline__ void mlp_tile_forward(const MlpDev& m, bf16x4 x4, int lane, f32x4 (&z1)[4],
                                                 f32x4 (&h1)[4], f32x4 (&z2)[4], f32x4 (&h2)[4],
                                                 f32x4& z3) {
#pragma unroll
    for (int mt = 0; mt < 4; ++mt) {
        z1[mt] = mfma(load_wt(m.w1, kMlpIn, mt, 0, lane), x4, bias4(m.b1, mt, lane));
        h1[mt] = tanh4(z1[mt]);
    }
    bf16x4 hb[4];
#pragma unroll
    for (int kb = 0; kb < 4; ++kb) hb[kb] = pack4(h1[kb]);
#pragma unroll
    for (int mt = 0; mt < 4; ++mt) {
        f32x4 acc = bias4(m.b2, mt, lane);
#pragma unroll
        for (int kb = 0; kb < 4; ++kb) acc = mfma(load_wt(m.w2, kMlpHid, mt, kb, lane), hb[kb], acc);
        z2[mt] = acc;
        h2[mt] = tanh4(acc);
    }
#pragma unroll
    for (int kb = 0; kb < 4; ++kb) hb[kb] = pack4(h2[kb]);
    f32x4 acc = bias4(m.b3, 0, lane);
#pragma unroll
    for (int kb = 0; kb < 4; ++kb) acc = mfma(load_wt(m.w3, kMlpHid, 0, kb, lane), hb[kb], acc);
    z3 = acc;
}

// this lane's B operand of the input tile: features X[node][16] (BF16)
// (sample q = node0 + l%16 is node q * stride; samples q >= n are zero)
__device__ __forceinline__ bf16x4 load_x(const unsigned short* __restrict__ X, long long node0, int n,
                                         int lane, int stride = 1) {
    const long long node = node0 + (lane & 15);
    bf16x4 r = {0, 0, 0, 0};
    if (node < n) r = load4(X + node * stride * kMlpIn + 4 * (lane >> 4));
    return r;
}

// Inference: out[node][0..1] (FP32) for every node; one wave per 16 nodes
__global__ void __launch_bounds__(64) k_mlp_forward(MlpDev m, const unsigned short* __restrict__ X,
                                                     int n, float* __restrict__ out) {
    const int lane = threadIdx.x;
    const long long node0 = (long long)blockIdx.x * 16;
    f32x4 z1[4], h1[4], z2[4], h2[4], z3;
    mlp_tile_forward(m, load_x(X, node0, n, lane), lane, z1, h1, z2, h2, z3);
    const long long node = node0 + (lane & 15);
    if (lane < 16 && node < n) {  // rows 0 and 1 of the output tile
        out[2 * node] = z3[0];
        out[2 * node + 1] = z3[1];
    }
}

// A 16x16 tile in LDS, BF16, as its rows (features) by columns (nodes): written
// from D layout (lane l holds [4(l/16)+i][l%16]), read in A layout
// ([l%16][4(l/16)+j]).  Rows are 40 bytes apart: 8-byte reads, and the rows of
// the four reading quarters start in different banks.
constexpr int kTileRow = 20;
struct MlpTile {
    unsigned short m[16 * kTileRow];
    __device__ __forceinline__ void put(const bf16x4& d, int lane) {
#pragma unroll
        for (int i = 0; i < 4; ++i)
            m[(4 * (lane >> 4) + i) * kTileRow + (lane & 15)] = (unsigned short)d[i];
    }
    __device__ __forceinline__ bf16x4 get(int lane) const {
        return load4(m + (lane & 15) * kTileRow + 4 * (lane >> 4));
    }
};

// Training: loss sum((y - t)^2)/n over outputs 0..1 of the n sampled nodes
// q * stride (q < n); `tiles` tiles of 16 samples per block.  Writes this
// block's gradient partial (kMlpParams floats, parameter layout of the master
// copy) and its loss partial.
//
// Four waves a block: wave w forms rows 16 w .. of every hidden layer, of the
// errors behind it and of the weight gradients that belong to them.  The
// layers' outputs and the errors pass through LDS, once as the B operands of
// the next product (lane for lane as they were formed) and once as tiles read
// transposed; everything of a tile has two copies, so that a wave may begin
// the next tile while another one reads this one.  A wave's weights stay in
// registers for all tiles.
//
// Bound by the latency of one tile's chain (three layers, two errors, a barrier
// each) and, with the chip full, the tanh: 32,768 samples 61 us with one wave a
// block (the whole chain, 5,000 instructions a tile, on one SIMD), 20.3 us so.
// Three blocks a CU: the registers of a fourth would be spilled (25-29 us).
constexpr int kGradWaves = 4;
__global__ void __launch_bounds__(64 * kGradWaves, 3)
k_mlp_grad(MlpDev m, const unsigned short* __restrict__ X, const float* __restrict__ T, int n,
           int stride, int tiles, float inv_n, float* __restrict__ gpart,
           float* __restrict__ lpart) {
    __shared__ bf16x4 sh1[2][4][64], sh2[2][4][64], sd2[2][4][64];  // B operands
    __shared__ bf16x4 sw3[4][64];  // the output layer's A operands, alike for all waves
    __shared__ __align__(8) MlpTile th1[2][4], th2[4], td2[4], td1[4], td3[4];
    __shared__ float sm[kGradWaves][16 * 17];
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    const int r4 = 4 * (lane >> 4), c = lane & 15;
    const f32x4 zero = {0.f, 0.f, 0.f, 0.f};
    // weight-gradient accumulators, D layout: dW1t tile w (64x16), dW2t tiles
    // (w, kb) (64x64), dW3t tile w (16x64); bias sums per row
    f32x4 g1 = zero, g2[4] = {zero, zero, zero, zero}, g3 = zero, gb1 = zero, gb2 = zero, gb3 = zero;
    const bf16x4 w1 = load_wt(m.w1, kMlpIn, w, 0, lane), w3b = load_w(m.w3, kMlpHid, w, 0, lane);
    const f32x4 b1 = bias4(m.b1, w, lane), b2 = bias4(m.b2, w, lane), b3 = bias4(m.b3, 0, lane);
    bf16x4 w2[4], w2b[4];
    sw3[w][lane] = load_wt(m.w3, kMlpHid, 0, w, lane);
#pragma unroll
    for (int k = 0; k < 4; ++k) {
        w2[k] = load_wt(m.w2, kMlpHid, w, k, lane);
        w2b[k] = load_w(m.w2, kMlpHid, w, k, lane);
    }
    float loss = 0.f;
    for (int tt = 0; tt < tiles; ++tt) {
        const long long node0 = ((long long)blockIdx.x * tiles + tt) * 16;
        if (node0 >= n) break;  // uniform over the block
        const int u = tt & 1;
        const bf16x4 x4 = load_x(X, node0, n, lane, stride);
        // input tile with nodes along K: B[node = 4(l/16)+j][in = l%16]
        bf16x4 bx;
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const long long nd = node0 + r4 + j;
            bx[j] = nd < n ? (short)X[nd * stride * kMlpIn + c] : (short)0;
        }
        const long long q = node0 + c, node = q * stride;
        float t0 = 0.f, t1 = 0.f;
        if (q < n && r4 == 0) {
            t0 = T[2 * node];
            t1 = T[2 * node + 1];
        }
        const f32x4 h1 = tanh4(mfma(w1, x4, b1));
        const bf16x4 h1b = pack4(h1);
        sh1[u][w][lane] = h1b;
        th1[u][w].put(h1b, lane);
        __syncthreads();
        f32x4 acc = b2;
#pragma unroll
        for (int k = 0; k < 4; ++k) acc = mfma(w2[k], sh1[u][k][lane], acc);
        const f32x4 h2 = tanh4(acc);
        const bf16x4 h2b = pack4(h2);
        sh2[u][w][lane] = h2b;
        th2[w].put(h2b, lane);
        __syncthreads();
        f32x4 z3 = b3;  // alike in every wave
#pragma unroll
        for (int k = 0; k < 4; ++k) z3 = mfma(sw3[k][lane], sh2[u][k][lane], z3);
        // dZ3 (D layout): rows 0, 1 carry the loss; padded rows and samples 0
        f32x4 dz3 = zero;
        if (q < n && r4 == 0) {
            const float d0 = z3[0] - t0, d1 = z3[1] - t1;
            loss += d0 * d0 + d1 * d1;
            dz3[0] = 2.f * d0 * inv_n;
            dz3[1] = 2.f * d1 * inv_n;
        }
        // dH2 = W3 dZ3 (64 x 16 nodes), dZ2 = dH2 (1 - h2^2)
        const bf16x4 dz3b = pack4(dz3);
        td3[w].put(dz3b, lane);
        f32x4 dh = mfma(w3b, dz3b, zero), dz2, dz1;
#pragma unroll
        for (int i = 0; i < 4; ++i) dz2[i] = dh[i] * (1.f - h2[i] * h2[i]);
        const bf16x4 dz2b = pack4(dz2);
        sd2[u][w][lane] = dz2b;
        td2[w].put(dz2b, lane);
        __syncthreads();
        // dH1 = W2 dZ2, dZ1 = dH1 (1 - h1^2)
        dh = zero;
#pragma unroll
        for (int k = 0; k < 4; ++k) dh = mfma(w2b[k], sd2[u][k][lane], dh);
#pragma unroll
        for (int i = 0; i < 4; ++i) dz1[i] = dh[i] * (1.f - h1[i] * h1[i]);
        td1[w].put(pack4(dz1), lane);
        __builtin_amdgcn_wave_barrier();  // read below by the wave's other lanes
        // bias gradients: row sums over the 16 nodes (reduced at the end)
        gb1 += dz1;
        gb2 += dz2;
        gb3 += dz3;
        // weight gradients dWt(out x in) += dZ(out x nodes) H^T(nodes x in):
        // A = dZ with nodes along K, B = H^T, both read transposed (the wave's
        // own tiles but h1's)
        g3 = mfma(td3[w].get(lane), th2[w].get(lane), g3);
        const bf16x4 a2 = td2[w].get(lane);
#pragma unroll
        for (int k = 0; k < 4; ++k) g2[k] = mfma(a2, th1[u][k].get(lane), g2[k]);
        g1 = mfma(td1[w].get(lane), bx, g1);
    }
    // store this block's partial in the master layout
    float* gp = gpart + (size_t)blockIdx.x * kMlpParams;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        gp[kMlpW1 + (w * 16 + r4 + i) * kMlpIn + c] = g1[i];
#pragma unroll
        for (int k = 0; k < 4; ++k)
            gp[kMlpW2 + (w * 16 + r4 + i) * kMlpHid + k * 16 + c] = g2[k][i];
        gp[kMlpW3 + (r4 + i) * kMlpHid + w * 16 + c] = g3[i];
    }
    // bias: sum over the 16 node columns (lanes with the same l/16), fixed order
    auto rowsum = [&](const f32x4& v, float* dst) {
        float* sw = sm[w];
#pragma unroll
        for (int i = 0; i < 4; ++i) sw[(r4 + i) * 17 + c] = v[i];
        __syncthreads();
        if (lane < 16) {
            float s = 0.f;
            for (int q = 0; q < 16; ++q) s += sw[lane * 17 + q];
            if (dst) dst[lane] = s;
        }
        __syncthreads();
    };
    rowsum(gb1, gp + kMlpB1 + w * 16);
    rowsum(gb2, gp + kMlpB2 + w * 16);
    rowsum(gb3, w == 0 ? gp + kMlpB3 : nullptr);
    // loss partial
    for (int off = 32; off > 0; off >>= 1) loss += __shfl_down(loss, off, 64);
    if (threadIdx.x == 0) lpart[blockIdx.x] = loss;
}

// One Adam step of a parameter on the FP32 master copy (rows of W3 and b3
// beyond the used outputs stay zero), then the weight's BF16 copy
struct MlpAdam {
    float *w, *mom, *vel;
    unsigned short* wb;
    float lr, b1, b2, eps, c1, c2;
};
__device__ __forceinline__ void adam_step(const MlpAdam& a, int p, float g) {
    const bool used = !((p >= kMlpW3 && p < kMlpB3 && (p - kMlpW3) / kMlpHid >= kMlpOutUsed) ||
                        (p >= kMlpB3 && p - kMlpB3 >= kMlpOutUsed));
    if (used) {
        const float mm = a.b1 * a.mom[p] + (1.f - a.b1) * g;
        const float vv = a.b2 * a.vel[p] + (1.f - a.b2) * g * g;
        a.mom[p] = mm;
        a.vel[p] = vv;
        a.w[p] = a.w[p] - a.lr * (mm * a.c1) / (sqrtf(vv * a.c2) + a.eps);
    }
    if (p < kMlpB3 && !(p >= kMlpB1 && p < kMlpW2) && !(p >= kMlpB2 && p < kMlpW3))
        a.wb[p] = f2bf(a.w[p]);
}

// grad[p] = sum over blocks of gpart[b][p]; the loss likewise from lpart (as
// column kMlpParams).  A block sums 64 columns; each of its kRedWaves waves
// sums one contiguous range of the partial blocks, and the waves' sums are
// added in wave order: a fixed order for a given block count.  kAdam: the
// parameter's Adam step in the same launch.
constexpr int kRedWaves = 16;
template <bool kAdam>
__global__ void __launch_bounds__(64 * kRedWaves)
k_mlp_reduce(const float* __restrict__ gpart, const float* __restrict__ lpart, int nblocks,
             float* __restrict__ grad, float* __restrict__ loss, MlpAdam adam) {
    __shared__ float sm[kRedWaves][65];
    const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
    const int p = blockIdx.x * 64 + lane;
    const int b0 = (int)((long long)nblocks * wv / kRedWaves);
    const int b1 = (int)((long long)nblocks * (wv + 1) / kRedWaves);
    float s = 0.f;
    if (p < kMlpParams) {
#pragma unroll 8
        for (int b = b0; b < b1; ++b) s += gpart[(size_t)b * kMlpParams + p];
    } else if (p == kMlpParams) {
#pragma unroll 8
        for (int b = b0; b < b1; ++b) s += lpart[b];
    }
    sm[wv][lane] = s;
    __syncthreads();
    if (wv == 0) {
        float t = 0.f;
#pragma unroll
        for (int w = 0; w < kRedWaves; ++w) t += sm[w][lane];
        if (p < kMlpParams) {
            grad[p] = t;
            if (kAdam) adam_step(adam, p, t);
        } else if (p == kMlpParams) {
            *loss = t;
        }
    }
}

__global__ void k_mlp_to_bf16(const float* __restrict__ w, unsigned short* __restrict__ wb) {
    const int p = blockIdx.x * blockDim.x + threadIdx.x;
    if (p < kMlpParams) wb[p] = f2bf(w[p]);
}

MlpDev mlp_dev(const MlpWeights& w) {
    MlpDev m;
    m.w1 = w.wb.p + kMlpW1;
    m.w2 = w.wb.p + kMlpW2;
    m.w3 = w.wb.p + kMlpW3;
    m.b1 = w.w.p + kMlpB1;
    m.b2 = w.w.p + kMlpB2;
    m.b3 = w.w.p + kMlpB3;
    return m;
}

}  // namespace

void MlpWeights::init(const float* host_params, hipStream_t s) {
    w.alloc(kMlpParams);
    m.alloc(kMlpParams);
    v.alloc(kMlpParams);
    wb.alloc(kMlpParams);
    grad.alloc(kMlpParams);
    loss.alloc(1);
    w.upload(host_params, kMlpParams, s);
    m.zero(s);
    v.zero(s);
    step = 0;
    k_mlp_to_bf16<<<grid_for(kMlpParams), kBlock, 0, s>>>(w.p, wb.p);
    CFD_HIP(hipGetLastError());
}

void mlp_forward(const MlpWeights& w, const unsigned short* X, int n, float* out, hipStream_t s) {
    if (n <= 0) return;
    k_mlp_forward<<<(n + 15) / 16, 64, 0, s>>>(mlp_dev(w), X, n, out);
    CFD_HIP(hipGetLastError());
}

// gradient and loss over the samples; adam: with the Adam step
static int gradient(MlpWeights& w, const unsigned short* X, const float* T, int n,
                    int tiles_per_block, hipStream_t s, int stride, const MlpAdam* adam) {
    CFD_CHECK(n > 0 && tiles_per_block > 0 && stride > 0, "arg: MLP training needs nodes");
    const int ns = (n + stride - 1) / stride;  // samples 0, stride, 2 stride, ... < n
    const int nb = (ns + 16 * tiles_per_block - 1) / (16 * tiles_per_block);
    if ((size_t)nb * kMlpParams > w.gpart.n) w.gpart.alloc((size_t)nb * kMlpParams);
    if ((size_t)nb > w.lpart.n) w.lpart.alloc(nb);
    k_mlp_grad<<<nb, 64 * kGradWaves, 0, s>>>(mlp_dev(w), X, T, ns, stride, tiles_per_block, 1.0f / (float)ns,
                                 w.gpart.p, w.lpart.p);
    const auto reduce = adam ? k_mlp_reduce<true> : k_mlp_reduce<false>;
    reduce<<<kMlpParams / 64 + 1, 64 * kRedWaves, 0, s>>>(w.gpart.p, w.lpart.p, nb, w.grad.p,
                                                          w.loss.p, adam ? *adam : MlpAdam{});
    CFD_HIP(hipGetLastError());
    return ns;
}

int mlp_gradient(MlpWeights& w, const unsigned short* X, const float* T, int n, int tiles_per_block,
                 hipStream_t s, int stride) {
    return gradient(w, X, T, n, tiles_per_block, s, stride, nullptr);
}

int mlp_train(MlpWeights& w, const unsigned short* X, const float* T, int n, int tiles_per_block,
              float lr, hipStream_t s, int stride) {
    const float b1 = 0.9f, b2 = 0.999f, eps = 1e-8f;
    ++w.step;
    const float c1 = 1.0f / (1.0f - std::pow(b1, (float)w.step));
    const float c2 = 1.0f / (1.0f - std::pow(b2, (float)w.step));
    const MlpAdam adam{w.w.p, w.m.p, w.v.p, w.wb.p, lr, b1, b2, eps, c1, c2};
    return gradient(w, X, T, n, tiles_per_block, s, stride, &adam);
}

}  // namespace cfd
