// The network in two kernels, for nets whose activations fit the LDS of a
// CU (every width the surrogate uses).
//
//   mlp_rows_kernel   one workgroup takes 16 samples through the whole
//                     network: every layer's product (MFMA 16x16x32 BF16),
//                     bias, GELU, and, when training, the loss and the
//                     backward products.  Activations never leave the LDS.
//   mlp_grad_kernel   every layer's weight gradient (a wavefront per 16x16
//                     tile, the batch as the contraction), the bias
//                     gradients and, when training, Adam on the parameters
//                     the gradient belongs to, in the same pass.
//
// The layer-by-layer form they replace launched 15 kernels a training step
// (gathers, products, column sums, loss, Adam), most of them one to a few
// workgroups long: 422 us a step for 256 samples of 3-256-256-256-65, 47 us
// with the two (an epoch of 8192 samples, uploads included: 13.49 ms before,
// 1.51 ms).  A forward of 512 samples went from 89.0 to 34.6 us.
//
// Operand layout.  v_mfma_f32_16x16x32_bf16 wants 8 consecutive k per lane
// from both operands, so everything a product reads is kept with its
// contraction index contiguous and padded with zeros to a multiple of 32:
// the weights twice, [out][in] for the forward and [in][out] for the
// backward products; the layer inputs and the output gradients of a batch
// as [feature][sample] for the weight gradients.  Every operand load is then
// one aligned 16-byte load per lane without a bounds check.
#pragma once

#include "common.hpp"
#include "reduce.hpp"

namespace vfps_impl {

typedef unsigned short u16x8 __attribute__((ext_vector_type(8)));
typedef unsigned short u16x4 __attribute__((ext_vector_type(4)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x4 __attribute__((ext_vector_type(4)));

// float -> bfloat16, round to nearest even (NaN stays NaN)
__host__ __device__ inline uint16_t f2bf(float f)
{
    uint32_t u = __builtin_bit_cast(uint32_t, f);
    if ((u & 0x7F800000u) == 0x7F800000u && (u & 0x007FFFFFu)) {
        return (uint16_t)((u >> 16) | 0x0040u);
    }
    u += 0x7FFFu + ((u >> 16) & 1u);
    return (uint16_t)(u >> 16);
}

__host__ __device__ inline float bf2f(uint16_t h)
{
    return __builtin_bit_cast(float, (uint32_t)h << 16);
}

// GELU with the exact Gaussian CDF: x Phi(x), and its derivative
__device__ inline float gelu(float x)
{
    return 0.5f * x * (1.0f + erff(x * 0.70710678118654752f));
}
__device__ inline float gelu_grad(float x)
{
    const float cdf = 0.5f * (1.0f + erff(x * 0.70710678118654752f));
    const float pdf = 0.39894228040143268f * expf(-0.5f * x * x);
    return cdf + x * pdf;
}

__device__ __forceinline__ f32x4 mfma_bf16(u16x8 a, u16x8 b, f32x4 c)
{
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(
        __builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b), c, 0, 0,
        0);
}

// Adam (Kingma & Ba): m = b1 m + (1-b1) g; v = b2 v + (1-b2) g^2;
// p -= lr (m / (1 - b1^t)) / (sqrt(v / (1 - b2^t)) + eps)
struct AdamArgs {
    float lr, b1, b2, eps, c1, c2;  // c1 = 1 - b1^t, c2 = 1 - b2^t
};

__device__ __forceinline__ float adam_update(const AdamArgs& a, float g,
                                             float* p, float* m, float* v)
{
    const float mi = a.b1 * *m + (1.0f - a.b1) * g;
    const float vi = a.b2 * *v + (1.0f - a.b2) * g * g;
    *m = mi;
    *v = vi;
    const float mh = mi / a.c1;
    const float vh = vi / a.c2;
    const float pi = *p - a.lr * mh / (sqrtf(vh) + a.eps);
    *p = pi;
    return pi;
}

constexpr uint32_t MLP_MAX_LAYERS = 8;
constexpr uint32_t MLP_ROWS = 16;        // samples per workgroup
constexpr uint32_t MLP_THREADS = 1024;
constexpr uint32_t MLP_WAVES = MLP_THREADS / 64;
constexpr uint32_t MLP_FRAGS = 8;        // operand loads in flight per tile
// LDS a workgroup may use (the hardware has 160 KiB per CU)
constexpr size_t MLP_LDS_MAX = 150 * 1024;

// The network's shape and where everything lies.
struct MlpNet {
    uint32_t L = 0;                       // layers
    uint32_t w[MLP_MAX_LAYERS + 1] = {};  // widths
    uint32_t wp[MLP_MAX_LAYERS + 1] = {}; // widths, up to a multiple of 32
    uint32_t po[MLP_MAX_LAYERS] = {};     // weights in the parameter vector
    uint32_t bo[MLP_MAX_LAYERS] = {};     // biases in the parameter vector
    uint32_t wo[MLP_MAX_LAYERS] = {};     // padded BF16 weights
    uint32_t ao[MLP_MAX_LAYERS] = {};     // rows of a layer's input [feature]
    uint32_t go[MLP_MAX_LAYERS] = {};     // rows of a layer's dZ [feature]
    uint32_t nbias = 0;                   // bias partials per workgroup
    uint32_t to[MLP_MAX_LAYERS] = {};     // a layer's bias partials
    // LDS (4-byte words)
    uint32_t zo[MLP_MAX_LAYERS] = {};     // hidden pre-activations [16][wp+4]
    uint32_t yo = 0;                      // outputs [16][w + 1]
    uint32_t tgt = 0, lab = 0;            // targets [16][w - 1], labels [16]
    uint32_t act[2] = {};                 // BF16 activations [16][as]
    uint32_t as = 0;                      // their row stride (halves)
    uint32_t lds_words = 0;
    uint32_t wsize = 0, arows = 0, grows = 0;
    uint32_t bmax = 0;                    // samples, up to a multiple of 32
};

// The layout, or L = 0 if the network does not fit.
inline MlpNet mlp_net(const uint32_t* dims, uint32_t ndims, uint32_t max_batch)
{
    MlpNet n;
    if (ndims < 2 || ndims - 1 > MLP_MAX_LAYERS) return MlpNet{};
    n.L = ndims - 1;
    auto up32 = [](uint32_t v) { return (v + 31u) & ~31u; };
    uint32_t widest = 0, po = 0, z = 0;
    for (uint32_t l = 0; l <= n.L; l++) {
        n.w[l] = dims[l];
        n.wp[l] = up32(dims[l]);
        widest = std::max(widest, n.wp[l]);
    }
    for (uint32_t l = 0; l < n.L; l++) {
        n.po[l] = po;
        po += dims[l] * dims[l + 1];
        n.bo[l] = po;
        po += dims[l + 1];
        n.wo[l] = n.wsize;
        n.wsize += n.wp[l] * n.wp[l + 1];
        n.ao[l] = n.arows;
        n.arows += n.wp[l];
        n.go[l] = n.grows;
        n.grows += n.wp[l + 1];
        n.to[l] = n.nbias;
        n.nbias += n.wp[l + 1];
    }
    for (uint32_t l = 0; l + 1 < n.L; l++) {
        n.zo[l] = z;
        z += MLP_ROWS * (n.wp[l + 1] + 4);
    }
    const uint32_t out = n.w[n.L];
    n.yo = z;
    z += MLP_ROWS * (out + 1);
    n.tgt = z;
    z += MLP_ROWS * (out - 1);
    n.lab = z;
    z += MLP_ROWS;
    z = (z + 3u) & ~3u;
    n.as = widest + 8;  // rows 4 banks apart, 16-byte aligned
    for (uint32_t k = 0; k < 2; k++) {
        n.act[k] = z;
        z += MLP_ROWS * n.as / 2;
    }
    n.lds_words = z;
    n.bmax = up32(max_batch);
    if ((size_t)z * 4 > MLP_LDS_MAX) return MlpNet{};
    return n;
}

struct MlpRowsArgs {
    const uint16_t* W;       // padded BF16 weights [out][in] per layer
    const uint16_t* WT;      // the same, [in][out]
    const float* p;          // parameters (biases)
    const float* x;          // samples [.][w0]
    const uint32_t* idx;     // rows of the batch in x, T, lab (null: 0, 1, ..)
    uint32_t B;              // samples in the batch
    float* Y;                // forward only: outputs [B][out]
    // training
    const float* T;          // [.][out - 1]
    const float* labels;     // [.]
    float wl;                // weight of the label's loss
    uint16_t* AT;            // layer inputs [feature][bmax]
    uint16_t* GT;            // layer dZ [feature][bmax]
    float* dbp;              // bias partials [workgroup][nbias]
    double* lossp;           // loss partials [workgroup]
};

// up to MLP_FRAGS operand fragments of one 16-column tile, k from 0: 16
// bytes per lane each (a fragment past K rereads the last one, unused)
__device__ __forceinline__ void mlp_frags(u16x8 (&f)[MLP_FRAGS],
                                          const uint16_t* q, uint32_t K)
{
#pragma unroll
    for (uint32_t t = 0; t < MLP_FRAGS; t++) {
        const uint32_t k = t * 32u < K ? t * 32u : K - 32u;
        f[t] = *reinterpret_cast<const u16x8*>(q + k);
    }
}

// 16 rows through one product: act [16][as] (BF16, LDS) times the 16
// columns of the fragments f (the first MLP_FRAGS of the column block q)
__device__ __forceinline__ f32x4 mlp_tile(const uint16_t* act, uint32_t as,
                                          uint32_t r16, uint32_t kq,
                                          const u16x8 (&f)[MLP_FRAGS],
                                          const uint16_t* q, uint32_t K)
{
    f32x4 acc = {0.0f, 0.0f, 0.0f, 0.0f};
    const uint16_t* a = act + r16 * as + kq;
#pragma unroll
    for (uint32_t t = 0; t < MLP_FRAGS; t++) {
        if (t * 32u < K) {
            acc = mfma_bf16(*reinterpret_cast<const u16x8*>(a + t * 32u), f[t],
                            acc);
        }
    }
    for (uint32_t k = MLP_FRAGS * 32u; k < K; k += 32u) {
        acc = mfma_bf16(*reinterpret_cast<const u16x8*>(a + k),
                        *reinterpret_cast<const u16x8*>(q + k), acc);
    }
    return acc;
}

// Bound: the latency of one pass through the layers (16 workgroups for 256
// samples: the smallest MFMA tile is 16 rows, and 16 rows of the surrogate
// are 4.8 M products, 1 us of a CU's matrix cores).  Each wavefront owns
// 16-column tiles and loads the next layer's first operand fragments (8 KB)
// before the barrier that ends this one, so that the weights' trip from the
// other XCDs' writes overlaps the epilogue.  3-256-256-256-65: forward of
// 512 samples, all layers and the transfer, in one launch (was six).
template <bool TRAIN>
__global__ void __launch_bounds__(MLP_THREADS)
mlp_rows_kernel(MlpNet n, MlpRowsArgs a)
{
    extern __shared__ __align__(16) float lds[];
    __shared__ double red[16];
    const uint32_t tid = threadIdx.x, lane = tid & 63u, wave = tid >> 6;
    const uint32_t r16 = lane & 15u, q4 = lane >> 4, kq = q4 * 8u;
    const uint32_t r0 = blockIdx.x * MLP_ROWS;
    const uint32_t L = n.L, out = n.w[L];
    uint16_t* act = reinterpret_cast<uint16_t*>(lds + n.act[0]);
    uint16_t* nxt = reinterpret_cast<uint16_t*>(lds + n.act[1]);
    float* y = lds + n.yo;
    u16x8 f[MLP_FRAGS];

    // this wavefront's first tile of a product with weights q [N][K]
    auto fetch = [&](const uint16_t* q, uint32_t N, uint32_t K) {
        if (wave * 16u < N) {
            mlp_frags(f, q + (size_t)(wave * 16u + r16) * K + kq, K);
        }
    };
    // the product of the 16 rows in act with q [N][K]; then(acc, column)
    // per tile; the fragments of the first tile are in f
    auto product = [&](const uint16_t* q, uint32_t N, uint32_t K, auto&& then) {
        for (uint32_t tj = wave * 16u; tj < N; tj += MLP_WAVES * 16u) {
            const uint16_t* col = q + (size_t)(tj + r16) * K + kq;
            if (tj != wave * 16u) {
                mlp_frags(f, col, K);
            }
            then(mlp_tile(act, n.as, r16, kq, f, col, K), tj + r16);
        }
    };

    fetch(a.W + n.wo[0], n.wp[1], n.wp[0]);
    auto sample = [&](uint32_t r) -> size_t {
        return a.idx ? a.idx[r0 + r] : r0 + r;
    };
    // inputs (rows past the batch: zeros), targets and labels
    for (uint32_t t = tid; t < MLP_ROWS * n.wp[0]; t += MLP_THREADS) {
        const uint32_t r = t / n.wp[0], c = t % n.wp[0];
        act[r * n.as + c] = r0 + r < a.B && c < n.w[0]
                                ? f2bf(a.x[sample(r) * n.w[0] + c])
                                : (uint16_t)0;
    }
    if constexpr (TRAIN) {
        const uint32_t S = out - 1;
        for (uint32_t t = tid; t < MLP_ROWS * S; t += MLP_THREADS) {
            const uint32_t r = t / S, c = t % S;
            lds[n.tgt + t] = r0 + r < a.B ? a.T[sample(r) * S + c] : 0.0f;
        }
        if (tid < MLP_ROWS) {
            lds[n.lab + tid] = r0 + tid < a.B ? a.labels[sample(tid)] : 0.0f;
        }
    }
    __syncthreads();
    if constexpr (TRAIN) {
        for (uint32_t t = tid; t < MLP_ROWS * n.wp[0]; t += MLP_THREADS) {
            const uint32_t c = t / MLP_ROWS, r = t % MLP_ROWS;
            a.AT[(size_t)(n.ao[0] + c) * n.bmax + r0 + r] = act[r * n.as + c];
        }
    }

    // ---- forward -------------------------------------------------------------
    for (uint32_t l = 0; l < L; l++) {
        const uint32_t N = n.w[l + 1], NP = n.wp[l + 1];
        const float* bias = a.p + n.bo[l];
        const bool last = l + 1 == L;
        product(a.W + n.wo[l], NP, n.wp[l], [&](f32x4 acc, uint32_t j) {
            const float b = j < N ? bias[j] : 0.0f;
            u16x4 packed;
#pragma unroll
            for (uint32_t r = 0; r < 4; r++) {
                const uint32_t i = q4 * 4u + r;
                const float z = acc[r] + b;
                if (!last) {
                    const uint16_t h = f2bf(gelu(z));
                    nxt[i * n.as + j] = h;
                    // (rows past the batch add nothing to the gradients)
                    packed[r] = r0 + i < a.B ? h : (uint16_t)0;
                    if (TRAIN) lds[n.zo[l] + i * (NP + 4u) + j] = z;
                } else if (j < N) {
                    if (TRAIN) {
                        y[i * (N + 1u) + j] = z;
                    } else if (r0 + i < a.B) {
                        a.Y[(size_t)(r0 + i) * N + j] = z;
                    }
                }
            }
            if (TRAIN && !last) {
                *reinterpret_cast<u16x4*>(a.AT + (size_t)(n.ao[l + 1] + j) * n.bmax +
                                          r0 + q4 * 4u) = packed;
            }
        });
        if (!last) {
            fetch(a.W + n.wo[l + 1], n.wp[l + 2], NP);
        } else if (TRAIN && L > 1) {
            fetch(a.WT + n.wo[l], n.wp[l], NP);
        }
        __syncthreads();
        uint16_t* t = act;
        act = nxt;
        nxt = t;
    }
    if constexpr (!TRAIN) {
        return;
    }

    // ---- loss and its gradient with respect to the outputs ----------------------
    // The first S outputs are regressed onto the targets (mean squared
    // error), the last is the logit of the label (binary cross entropy,
    // weight wl); loss = (1/B) sum_b [ (1/S) sum_k (y-t)^2 + wl BCE ].
    {
        const uint32_t S = out - 1, NP = n.wp[L];
        double loss = 0.0;
        for (uint32_t t = tid; t < MLP_ROWS * NP; t += MLP_THREADS) {
            const uint32_t r = t / NP, k = t % NP;
            float g = 0.0f;
            if (k < out && r0 + r < a.B) {
                const float v = y[r * (out + 1u) + k];
                if (k < S) {
                    const float d = v - lds[n.tgt + r * S + k];
                    loss += (double)d * (double)d / (double)S;
                    g = 2.0f * d / (float)(S * a.B);
                } else {
                    const float lab = lds[n.lab + r];
                    // BCE with logits: max(y,0) - y*lab + log(1 + exp(-|y|))
                    loss += (double)a.wl *
                            ((double)fmaxf(v, 0.0f) - (double)v * lab +
                             log1p(exp(-fabs((double)v))));
                    const float sg = 1.0f / (1.0f + expf(-v));
                    g = a.wl * (sg - lab) / (float)a.B;
                }
            }
            if (k < out) y[r * (out + 1u) + k] = g;
            act[r * n.as + k] = f2bf(g);
        }
        loss = block_sum(loss, red);  // (its barriers order act and y too)
        if (tid == 0) {
            a.lossp[blockIdx.x] = loss;
        }
        float* db = a.dbp + (size_t)blockIdx.x * n.nbias + n.to[L - 1];
        for (uint32_t k = tid; k < NP; k += MLP_THREADS) {
            u16x8 h[2];
            float s = 0.0f;
#pragma unroll
            for (uint32_t r = 0; r < MLP_ROWS; r++) {
                h[r >> 3][r & 7u] = act[r * n.as + k];
                if (k < out) s += y[r * (out + 1u) + k];
            }
            db[k] = s;
            u16x8* dst = reinterpret_cast<u16x8*>(
                a.GT + (size_t)(n.go[L - 1] + k) * n.bmax + r0);
            dst[0] = h[0];
            dst[1] = h[1];
        }
    }

    // ---- backward: dZ of layer l - 1 from dZ of layer l ---------------------------
    for (uint32_t l = L - 1; l > 0; l--) {
        const uint32_t NP = n.wp[l];
        const float* z = lds + n.zo[l - 1];
        float* db = a.dbp + (size_t)blockIdx.x * n.nbias + n.to[l - 1];
        product(a.WT + n.wo[l], NP, n.wp[l + 1], [&](f32x4 acc, uint32_t j) {
            u16x4 packed;
            float s = 0.0f;
#pragma unroll
            for (uint32_t r = 0; r < 4; r++) {
                const uint32_t i = q4 * 4u + r;
                const float dz = r0 + i < a.B
                                     ? acc[r] * gelu_grad(z[i * (NP + 4u) + j])
                                     : 0.0f;
                s += dz;
                packed[r] = f2bf(dz);
                nxt[i * n.as + j] = packed[r];
            }
            *reinterpret_cast<u16x4*>(a.GT + (size_t)(n.go[l - 1] + j) * n.bmax +
                                      r0 + q4 * 4u) = packed;
            s += __shfl_xor(s, 16, 64);
            s += __shfl_xor(s, 32, 64);
            if (q4 == 0) db[j] = s;
        });
        if (l > 1) {
            fetch(a.WT + n.wo[l - 1], n.wp[l - 1], NP);
        }
        __syncthreads();
        uint16_t* t = act;
        act = nxt;
        nxt = t;
    }
}

struct MlpGradArgs {
    const uint16_t* AT;
    const uint16_t* GT;
    const float* dbp;
    const double* lossp;
    uint32_t B;
    float* g;                // gradients
    float* loss;             // [1] the batch's loss
    // Adam
    float* p;
    float* m;
    float* v;
    uint16_t* W;
    uint16_t* WT;
    AdamArgs adam;
};

// 16x16 weight-gradient tiles of the network
__host__ __device__ inline uint32_t mlp_grad_tiles(const MlpNet& n, uint32_t l)
{
    return ((n.w[l + 1] + 15u) / 16u) * ((n.w[l] + 15u) / 16u);
}

constexpr uint32_t MLP_GRAD_THREADS = 256;

// Workgroups [0, tiles/4): a tile of dW = dZ^T A per wavefront; then the
// biases, a thread each; the last workgroup's last thread adds the loss.
// Bound: the operands' trip from L2 (608 tiles of 16 KB for the surrogate
// at 256 samples).
template <bool ADAM>
__global__ void __launch_bounds__(MLP_GRAD_THREADS)
mlp_grad_kernel(MlpNet n, MlpGradArgs a, uint32_t tile_blocks)
{
    const uint32_t tid = threadIdx.x, lane = tid & 63u, wave = tid >> 6;
    const uint32_t K = (a.B + 31u) & ~31u;
    const uint32_t nwg = K / MLP_ROWS;  // workgroups of the rows kernel
    if (blockIdx.x < tile_blocks) {
        uint32_t tile = blockIdx.x * (MLP_GRAD_THREADS / 64u) + wave;
        uint32_t l = 0;
        while (l < n.L && tile >= mlp_grad_tiles(n, l)) {
            tile -= mlp_grad_tiles(n, l);
            l++;
        }
        if (l == n.L) return;
        const uint32_t ni = n.w[l], no = n.w[l + 1];
        const uint32_t tk = (ni + 15u) / 16u;
        const uint32_t j0 = (tile / tk) * 16u, k0 = (tile % tk) * 16u;
        const uint32_t r16 = lane & 15u, q4 = lane >> 4;
        const uint16_t* ga = a.GT + (size_t)(n.go[l] + j0 + r16) * n.bmax + q4 * 8u;
        const uint16_t* xa = a.AT + (size_t)(n.ao[l] + k0 + r16) * n.bmax + q4 * 8u;
        const uint32_t k = k0 + r16;
        // the parameters and moments of this lane's four entries, fetched
        // beside the operands
        float pv[4], mv[4], vv[4];
        if (ADAM) {
#pragma unroll
            for (uint32_t r = 0; r < 4; r++) {
                const uint32_t j = j0 + q4 * 4u + r;
                const size_t o = n.po[l] + (size_t)(j < no ? j : no - 1u) * ni +
                                 (k < ni ? k : ni - 1u);
                pv[r] = a.p[o];
                mv[r] = a.m[o];
                vv[r] = a.v[o];
            }
        }
        f32x4 acc = {0.0f, 0.0f, 0.0f, 0.0f};
        for (uint32_t b = 0; b < K; b += MLP_FRAGS * 32u) {
            u16x8 fg[MLP_FRAGS], fx[MLP_FRAGS];
            mlp_frags(fg, ga + b, K - b);
            mlp_frags(fx, xa + b, K - b);
#pragma unroll
            for (uint32_t t = 0; t < MLP_FRAGS; t++) {
                if (b + t * 32u < K) acc = mfma_bf16(fg[t], fx[t], acc);
            }
        }
        u16x4 packed = {0, 0, 0, 0};
#pragma unroll
        for (uint32_t r = 0; r < 4; r++) {
            const uint32_t j = j0 + q4 * 4u + r;
            if (j >= no || k >= ni) continue;
            const size_t o = n.po[l] + (size_t)j * ni + k;
            a.g[o] = acc[r];
            if (ADAM) {
                packed[r] = f2bf(adam_update(a.adam, acc[r], pv + r, mv + r, vv + r));
                a.p[o] = pv[r];
                a.m[o] = mv[r];
                a.v[o] = vv[r];
                a.W[n.wo[l] + (size_t)j * n.wp[l] + k] = packed[r];
            }
        }
        if (ADAM && k < ni) {
            // (rows past the layer's last keep their zeros)
            *reinterpret_cast<u16x4*>(a.WT + n.wo[l] + (size_t)k * n.wp[l + 1] +
                                      j0 + q4 * 4u) = packed;
        }
        return;
    }
    const uint32_t t = (blockIdx.x - tile_blocks) * MLP_GRAD_THREADS + tid;
    if (t < n.nbias) {
        uint32_t l = 0;
        while (l + 1 < n.L && t >= n.to[l + 1]) l++;
        const uint32_t j = t - n.to[l];
        if (j < n.w[l + 1]) {
            float s = 0.0f;
            for (uint32_t w = 0; w < nwg; w++) {
                s += a.dbp[(size_t)w * n.nbias + t];
            }
            const uint32_t o = n.bo[l] + j;
            a.g[o] = s;
            if (ADAM) {
                adam_update(a.adam, s, a.p + o, a.m + o, a.v + o);
            }
        }
    }
    if (blockIdx.x == gridDim.x - 1 && tid == MLP_GRAD_THREADS - 1) {
        double s = 0.0;
        for (uint32_t w = 0; w < nwg; w++) s += a.lossp[w];
        *a.loss = (float)(s / (double)a.B);
    }
}

// both padded BF16 copies of the weights from the FP32 parameters
__global__ void __launch_bounds__(256)
mlp_pack_kernel(MlpNet n, const float* __restrict__ p, uint16_t* __restrict__ W,
                uint16_t* __restrict__ WT)
{
    for (uint32_t t = blockIdx.x * 256u + threadIdx.x; t < n.wsize;
         t += gridDim.x * 256u) {
        uint32_t l = 0;
        while (l + 1 < n.L && t >= n.wo[l + 1]) l++;
        const uint32_t e = t - n.wo[l];
        const uint32_t j = e / n.wp[l], k = e % n.wp[l];
        const bool in = j < n.w[l + 1] && k < n.w[l];
        const uint16_t h = in ? f2bf(p[n.po[l] + (size_t)j * n.w[l] + k])
                              : (uint16_t)0;
        W[t] = h;
        WT[n.wo[l] + (size_t)k * n.wp[l + 1] + j] = h;
    }
}

}  // namespace vfps_impl
