// The network in two kernels, for nets whose activations fit the LDS of a
// CU (every width the surrogate uses).
//
//   mlp_rows_kernel   one workgroup takes 4, 8 or 16 samples through the whole
//                     network: every layer's product (MFMA 16x16x32 BF16),
//                     bias, GELU, and, when training, the loss and the
//                     backward products.  Activations never leave the LDS.
//   mlp_grad_kernel   every layer's weight gradient (a wavefront per 16x16
//                     tile, the batch as the contraction), the bias
//                     gradients, the loss and, when training, Adam on the
//                     parameters the gradient belongs to, in the same pass.
//
// The layer-by-layer form they replace launched 15 kernels a training step
// (gathers, products, column sums, loss, Adam), most of them one to a few
// workgroups long: 422 us a step for 256 samples of 3-256-256-256-65; the two
// take 21.2 and 6.4 us (an epoch of 8192 samples, uploads included: 13.5 ms
// before, 1.07 ms).  A forward of 512 samples went from 88.6 to 27.4 us.
//
// Operand layout.  v_mfma_f32_16x16x32_bf16 wants 8 consecutive k per lane
// from both operands: lane l holds column (or row) l % 16, k = 8 (l / 16) ...
// + 7 of a 16 x 32 fragment.  Everything a product reads from memory is kept
// in that order, a fragment after the other (mlp_frag), padded with zeros to
// whole fragments: the weights twice, once per direction, and the layer
// inputs and output gradients of a batch (samples as the contraction).  A
// fragment load is then 1 KB in a row and needs no bounds check.  With
// row-major matrices a load touched 16 rows, and the 128 KB of a layer took
// a workgroup 4 us (30 us a launch for the training kernel, 20.6 with
// fragments).
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
// both, from one error function
__device__ inline float gelu_both(float x, float* grad)
{
    const float e = 1.0f + erff(x * 0.70710678118654752f);
    const float pdf = 0.39894228040143268f * expf(-0.5f * x * x);
    *grad = 0.5f * e + x * pdf;
    return 0.5f * x * e;
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

// place of (column c, contraction index k) in a matrix of K contraction
// indexes (K % 32 == 0) held as fragments
__host__ __device__ __forceinline__ size_t mlp_frag(uint32_t c, uint32_t k,
                                                    uint32_t K)
{
    return ((size_t)(c >> 4) * (K >> 5) + (k >> 5)) * 512u +
           (((k & 31u) >> 3) * 16u + (c & 15u)) * 8u + (k & 7u);
}

constexpr uint32_t MLP_MAX_LAYERS = 8;
constexpr uint32_t MLP_ROWS = 16;        // most samples per workgroup
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
    uint32_t nbias = 0;                   // all layers' dZ columns
    uint32_t to[MLP_MAX_LAYERS] = {};     // a layer's first one
    // LDS (4-byte words)
    uint32_t zo[MLP_MAX_LAYERS] = {};     // hidden layers: gelu', then dZ
                                          // [16][wp + 4]
    uint32_t yo = 0;                      // outputs, then dZ [16][w + 1]
    uint32_t tgt = 0;                     // targets, then the outputs'
                                          // differences from them [16][w - 1]
    uint32_t lab = 0, logit = 0;          // labels, their outputs [16]
    uint32_t act[2] = {};                 // BF16 activations [16][as]
    uint32_t tr = 0;                      // layer inputs, then dZ [feature][.]
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
    n.logit = z;
    z += MLP_ROWS;
    z = (z + 3u) & ~3u;
    n.as = widest + 8;  // rows 4 banks apart, 16-byte aligned
    for (uint32_t k = 0; k < 2; k++) {
        n.act[k] = z;
        z += MLP_ROWS * n.as / 2;
    }
    n.tr = z;
    z += (n.arows + n.grows) * MLP_ROWS / 2;
    n.lds_words = z;
    n.bmax = up32(max_batch);
    if ((size_t)z * 4 > MLP_LDS_MAX) return MlpNet{};
    return n;
}

struct MlpRowsArgs {
    const uint16_t* W;       // BF16 weights per layer: columns out, k in
    const uint16_t* WT;      // the same, columns in, k out
    const float* p;          // parameters (biases)
    const float* x;          // samples [.][w0]
    const uint32_t* idx;     // rows of the batch in x, T, lab (null: 0, 1, ..)
    uint32_t B;              // samples in the batch
    float* Y;                // forward only: outputs [B][out]
    // training
    const float* T;          // [.][out - 1]
    const float* labels;     // [.]
    float wl;                // weight of the label's loss
    uint16_t* AT;            // layer inputs: columns features, k samples
    uint16_t* GT;            // layer dZ, the same way
    float* dz;               // FP32 dZ [sample][nbias]
    double* terms;           // loss terms [sample][out]
};

// up to MLP_FRAGS fragments from q on, of `count` (one past them rereads the
// last, unused)
__device__ __forceinline__ void mlp_frags(u16x8 (&f)[MLP_FRAGS],
                                          const uint16_t* q, uint32_t count,
                                          uint32_t lane)
{
#pragma unroll
    for (uint32_t t = 0; t < MLP_FRAGS; t++) {
        const uint32_t e = t < count ? t : count - 1u;
        f[t] = *reinterpret_cast<const u16x8*>(q + e * 512u + lane * 8u);
    }
}

// 16 rows through one product: act [16][as] (BF16, LDS) times the 16
// columns whose fragments are f (the first MLP_FRAGS of the K / 32 at q).
__device__ __forceinline__ f32x4 mlp_tile(const uint16_t* act, uint32_t as,
                                          uint32_t lane,
                                          const u16x8 (&f)[MLP_FRAGS],
                                          const uint16_t* q, uint32_t K)
{
    f32x4 acc = {0.0f, 0.0f, 0.0f, 0.0f};
    const uint16_t* a = act + (lane & 15u) * as + (lane >> 4) * 8u;
#pragma unroll
    for (uint32_t t = 0; t < MLP_FRAGS; t++) {
        if (t * 32u < K) {
            acc = mfma_bf16(*reinterpret_cast<const u16x8*>(a + t * 32u), f[t],
                            acc);
        }
    }
    for (uint32_t k = MLP_FRAGS * 32u; k < K; k += 32u) {
        acc = mfma_bf16(*reinterpret_cast<const u16x8*>(a + k),
                        *reinterpret_cast<const u16x8*>(q + k * 16u + lane * 8u),
                        acc);
    }
    return acc;
}

// Bound: the latency of one pass through the layers.  Samples per workgroup:
// 4 RR, the fewest that still need no more workgroups than the GPU has CUs
// (mlp_rows_per_lane).  The products cost a CU 1 us whatever of their 16 rows
// is in use, but a GELU with its derivative is about 130 instructions: with
// 16 samples a workgroup's four wavefronts per SIMD spend 3 us a layer on
// them, and a batch of 256 is 16 workgroups; with 4 samples it is 64 (a
// launch of 256 samples, operands still row by row: 34 us with 16, 30 with 4).
// A lane of a product's result holds rows 4 q .. 4 q + 3 of one column, so
// sample s = q RR + r is given MFMA row 4 q + r: every lane then has RR
// samples (the rows between hold stale values that no other row sees).
// Each wavefront owns 16-column tiles and loads the next layer's first
// operand fragments (8 KB) and bias before the epilogue of its last tile, so
// that their trip overlaps it.  What the gradient products read is kept in
// LDS and stored at the end: a store in between would be waited for by the
// next use of a load (the counter drains in order).
template <bool TRAIN, int RR>
__global__ void __launch_bounds__(MLP_THREADS)
mlp_rows_kernel(MlpNet n, MlpRowsArgs a)
{
    extern __shared__ __align__(16) float lds[];
    constexpr uint32_t R = 4u * RR;  // samples of this workgroup
    typedef uint16_t packed_t __attribute__((ext_vector_type(RR == 1 ? 2 : RR)));
    const uint32_t tid = threadIdx.x, lane = tid & 63u, wave = tid >> 6;
    const uint32_t r16 = lane & 15u, q4 = lane >> 4;
    const uint32_t r0 = blockIdx.x * R;
    const uint32_t s0 = q4 * RR;     // this lane's first sample
    const uint32_t L = n.L, out = n.w[L];
    uint16_t* act = reinterpret_cast<uint16_t*>(lds + n.act[0]);
    uint16_t* nxt = reinterpret_cast<uint16_t*>(lds + n.act[1]);
    float* y = lds + n.yo;
    u16x8 f[MLP_FRAGS];
    float bias0 = 0.0f;  // bias of this lane's column of the first tile

    // act row of sample s
    auto row = [](uint32_t s) { return s / RR * 4u + s % RR; };
    // layer inputs (arows features), then dZ (grows), R samples each
    uint16_t* tr = reinterpret_cast<uint16_t*>(lds + n.tr);
    // this lane's RR samples of one feature
    auto keep = [&](uint32_t feature, packed_t v) {
        if constexpr (RR == 1) {
            tr[feature * R + s0] = v[0];
        } else {
            *reinterpret_cast<packed_t*>(tr + feature * R + s0) = v;
        }
    };
    // this wavefront's tile tj of a product with the fragments q of N columns
    // and K contraction indexes (bias: of the columns, the first nb)
    auto fetch = [&](const uint16_t* q, uint32_t tj, uint32_t N, uint32_t K,
                     const float* bias, uint32_t nb) {
        if (tj < N) {
            mlp_frags(f, q + (size_t)tj * K, K / 32u, lane);
            bias0 = tj + r16 < nb ? bias[tj + r16] : 0.0f;
        }
    };
    auto fetch_forward = [&](uint32_t l, uint32_t tj) {
        fetch(a.W + n.wo[l], tj, n.wp[l + 1], n.wp[l], a.p + n.bo[l], n.w[l + 1]);
    };
    auto fetch_backward = [&](uint32_t l, uint32_t tj) {
        fetch(a.WT + n.wo[l], tj, n.wp[l], n.wp[l + 1], nullptr, 0);
    };
    // the product of the rows in act with q (N columns, K contraction
    // indexes); then(acc, column, bias) per tile.  The operands of the first
    // tile are in f and bias0; here(tj) fetches those of a later one, next()
    // those of the product that follows.
    auto product = [&](const uint16_t* q, uint32_t N, uint32_t K, auto&& here,
                       auto&& next, auto&& then) {
        constexpr uint32_t step = MLP_WAVES * 16u;
        if (wave * 16u >= N) next();
        for (uint32_t tj = wave * 16u; tj < N; tj += step) {
            if (tj != wave * 16u) here(tj);
            const f32x4 acc =
                mlp_tile(act, n.as, lane, f, q + (size_t)tj * K, K);
            const float b = bias0;
            if (tj + step >= N) next();
            then(acc, tj + r16, b);
        }
    };

    auto sample = [&](uint32_t s) -> size_t {
        return a.idx ? a.idx[r0 + s] : r0 + s;
    };
    // inputs (samples past the batch: zeros), targets and labels
    for (uint32_t t = tid; t < R * n.wp[0]; t += MLP_THREADS) {
        const uint32_t s = t / n.wp[0], c = t % n.wp[0];
        act[row(s) * n.as + c] = r0 + s < a.B && c < n.w[0]
                                     ? f2bf(a.x[sample(s) * n.w[0] + c])
                                     : (uint16_t)0;
    }
    fetch_forward(0, wave * 16u);
    if constexpr (TRAIN) {
        const uint32_t S = out - 1;
        for (uint32_t t = tid; t < R * S; t += MLP_THREADS) {
            const uint32_t s = t / S, c = t % S;
            lds[n.tgt + t] = r0 + s < a.B ? a.T[sample(s) * S + c] : 0.0f;
        }
        if (tid < R) {
            lds[n.lab + tid] = r0 + tid < a.B ? a.labels[sample(tid)] : 0.0f;
        }
    }
    __syncthreads();
    if constexpr (TRAIN) {
        for (uint32_t t = tid; t < R * n.wp[0]; t += MLP_THREADS) {
            const uint32_t c = t / R, s = t % R;
            tr[(n.ao[0] + c) * R + s] = act[row(s) * n.as + c];
        }
    }

    // ---- forward -------------------------------------------------------------
    for (uint32_t l = 0; l < L; l++) {
        const uint32_t N = n.w[l + 1], NP = n.wp[l + 1];
        const bool last = l + 1 == L;
        auto next = [&]() {
            if (!last) {
                fetch_forward(l + 1, wave * 16u);
            } else if (TRAIN && L > 1) {
                fetch_backward(l, wave * 16u);
            }
        };
        product(a.W + n.wo[l], NP, n.wp[l],
                [&](uint32_t tj) { fetch_forward(l, tj); }, next,
                [&](f32x4 acc, uint32_t j, float b) {
            packed_t packed;
#pragma unroll
            for (uint32_t r = 0; r < (uint32_t)RR; r++) {
                const uint32_t s = s0 + r;
                const float z = acc[r] + b;
                if (!last) {
                    float h, grad = 0.0f;
                    if (TRAIN) {
                        h = gelu_both(z, &grad);
                        lds[n.zo[l] + s * (NP + 4u) + j] = grad;
                    } else {
                        h = gelu(z);
                    }
                    // (columns up to whole fragments stay zero: 0 times an
                    // infinite activation is no number, and the next
                    // product's zero weights would carry it to every output)
                    const uint16_t hb = j < N ? f2bf(h) : (uint16_t)0;
                    nxt[row(s) * n.as + j] = hb;
                    // (samples past the batch add nothing to the gradients)
                    packed[r] = r0 + s < a.B ? hb : (uint16_t)0;
                } else if (j < N) {
                    if (TRAIN) {
                        y[s * (N + 1u) + j] = z;
                    } else if (r0 + s < a.B) {
                        a.Y[(size_t)(r0 + s) * N + j] = z;
                    }
                }
            }
            if (TRAIN && !last) {
                keep(n.ao[l + 1] + j, packed);
            }
        });
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
        for (uint32_t t = tid; t < R * NP; t += MLP_THREADS) {
            const uint32_t s = t / NP, k = t % NP;
            float g = 0.0f;
            if (k < out && r0 + s < a.B) {
                const float v = y[s * (out + 1u) + k];
                if (k < S) {
                    const float d = v - lds[n.tgt + s * S + k];
                    lds[n.tgt + s * S + k] = d;
                    g = 2.0f * d / (float)(S * a.B);
                } else {
                    const float sg = 1.0f / (1.0f + expf(-v));
                    lds[n.logit + s] = v;
                    g = a.wl * (sg - lds[n.lab + s]) / (float)a.B;
                }
            }
            if (k < out) y[s * (out + 1u) + k] = g;
            act[row(s) * n.as + k] = f2bf(g);
        }
        __syncthreads();
        for (uint32_t k = tid; k < NP; k += MLP_THREADS) {
#pragma unroll
            for (uint32_t s = 0; s < R; s++) {
                tr[(n.arows + n.go[L - 1] + k) * R + s] = act[row(s) * n.as + k];
            }
        }
    }

    // ---- backward: dZ of layer l - 1 from dZ of layer l ---------------------------
    for (uint32_t l = L - 1; l > 0; l--) {
        const uint32_t NP = n.wp[l];
        float* grad = lds + n.zo[l - 1];
        auto next = [&]() {
            if (l > 1) fetch_backward(l - 1, wave * 16u);
        };
        product(a.WT + n.wo[l], NP, n.wp[l + 1],
                [&](uint32_t tj) { fetch_backward(l, tj); }, next,
                [&](f32x4 acc, uint32_t j, float) {
            packed_t packed;
#pragma unroll
            for (uint32_t r = 0; r < (uint32_t)RR; r++) {
                const uint32_t s = s0 + r;
                float& g = grad[s * (NP + 4u) + j];
                // (columns up to whole fragments: zeros, as forward)
                const float dz = r0 + s < a.B && j < n.w[l] ? acc[r] * g : 0.0f;
                g = dz;
                packed[r] = f2bf(dz);
                nxt[row(s) * n.as + j] = packed[r];
            }
            keep(n.arows + n.go[l - 1] + j, packed);
        });
        __syncthreads();
        uint16_t* t = act;
        act = nxt;
        nxt = t;
    }
    if (L == 1) __syncthreads();
    // ---- what the gradient products and biases read -------------------------------
    for (uint32_t t = tid; t < (n.arows + n.grows) * RR; t += MLP_THREADS) {
        const uint32_t feature = t / RR, c = t % RR;
        const bool in = feature < n.arows;
        *reinterpret_cast<u16x4*>(
            (in ? a.AT : a.GT) +
            mlp_frag(in ? feature : feature - n.arows, r0 + 4u * c, n.bmax)) =
            *reinterpret_cast<const u16x4*>(tr + feature * R + 4u * c);
    }
    for (uint32_t l = 0; l < L; l++) {
        const uint32_t NP = n.wp[l + 1];
        for (uint32_t t = tid; t < R * NP; t += MLP_THREADS) {
            const uint32_t s = t / NP, j = t % NP;
            a.dz[(size_t)(r0 + s) * n.nbias + n.to[l] + j] =
                l + 1 < L  ? lds[n.zo[l] + s * (NP + 4u) + j]
                : j < out  ? y[s * (out + 1u) + j]
                           : 0.0f;
        }
    }
    for (uint32_t t = tid; t < R * out; t += MLP_THREADS) {
        const uint32_t s = t / out, k = t % out, S = out - 1;
        double e = 0.0;
        if (k < S) {
            const float d = lds[n.tgt + s * S + k];
            e = (double)d * (double)d / (double)S;
        } else {
            // BCE with logits: max(y,0) - y*lab + log(1 + exp(-|y|))
            const float v = lds[n.logit + s];
            e = (double)a.wl * ((double)fmaxf(v, 0.0f) -
                                (double)v * lds[n.lab + s] +
                                log1p(exp(-fabs((double)v))));
        }
        if (r0 + s < a.B) a.terms[(size_t)(r0 + s) * out + k] = e;
    }
}

// Samples per lane (RR) of a batch of B samples on a GPU of ncu CUs.
inline uint32_t mlp_rows_per_lane(uint32_t B, uint32_t ncu)
{
    const uint32_t rows = (B + 31u) & ~31u;
    return rows <= 4u * ncu ? 1u : rows <= 8u * ncu ? 2u : 4u;
}

struct MlpGradArgs {
    const uint16_t* AT;
    const uint16_t* GT;
    const float* dz;
    const double* terms;
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

constexpr uint32_t MLP_BIAS_COLS = 32;   // (a layer's columns are whole 32s)
constexpr uint32_t MLP_BIAS_ROWS = 256;  // samples staged at once
constexpr uint32_t MLP_BIAS_STRIDE = MLP_BIAS_ROWS + 4;

// workgroups beside the tiles': the biases' and one for the loss
__host__ __device__ inline uint32_t mlp_grad_sums(const MlpNet& n)
{
    return n.nbias / MLP_BIAS_COLS + 1u;
}

// Workgroups [0, tiles/4): a tile of dW = dZ^T A per wavefront; then the
// biases, 32 columns of dZ each; the last workgroup adds the loss.
// The sums that no matrix product fixes keep one order whatever the batch's
// split over workgroups: a bias gradient adds its samples one after another
// in FP32 (as colsum_kernel), the loss its terms as loss_kernel does.  So a
// training run gives the same bits as layer by layer.  (Partial sums of the
// rows kernel's workgroups took 1.3 us less a step of 256 samples, 27.6 in
// all, in other last bits.)
// Bound: the operands' trip from L2 (608 tiles of 16 KB for the surrogate
// at 256 samples).
template <bool ADAM>
__global__ void __launch_bounds__(MLP_GRAD_THREADS)
mlp_grad_kernel(MlpNet n, MlpGradArgs a, uint32_t tile_blocks)
{
    const uint32_t tid = threadIdx.x, lane = tid & 63u, wave = tid >> 6;
    const uint32_t K = (a.B + 31u) & ~31u;
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
        const uint16_t* ga = a.GT + (size_t)(n.go[l] + j0) * n.bmax;
        const uint16_t* xa = a.AT + (size_t)(n.ao[l] + k0) * n.bmax;
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
            mlp_frags(fg, ga + b * 16u, (K - b) / 32u, lane);
            mlp_frags(fx, xa + b * 16u, (K - b) / 32u, lane);
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
                a.W[n.wo[l] + mlp_frag(j, k, n.wp[l])] = packed[r];
            }
        }
        if (ADAM && k < ni) {
            // (rows past the layer's last keep their zeros)
            *reinterpret_cast<u16x4*>(
                a.WT + n.wo[l] + mlp_frag(k, j0 + q4 * 4u, n.wp[l + 1])) = packed;
        }
        return;
    }
    const uint32_t c0 = (blockIdx.x - tile_blocks) * MLP_BIAS_COLS;
    if (c0 < n.nbias) {
        __shared__ __align__(16) float cols[MLP_BIAS_COLS * MLP_BIAS_STRIDE];
        uint32_t l = 0;
        while (l + 1 < n.L && c0 >= n.to[l + 1]) l++;
        const uint32_t j = c0 - n.to[l] + tid;
        const bool mine = tid < MLP_BIAS_COLS && j < n.w[l + 1];
        const uint32_t o = n.bo[l] + (mine ? j : 0u);
        float pv = 0.0f, mv = 0.0f, vv = 0.0f;
        if (ADAM) {
            pv = a.p[o];
            mv = a.m[o];
            vv = a.v[o];
        }
        float s = 0.0f;
        for (uint32_t b0 = 0; b0 < K; b0 += MLP_BIAS_ROWS) {
            // (samples from the batch's end to K are zeros, which change no
            // sum that starts at +0)
            const uint32_t nr = min(MLP_BIAS_ROWS, K - b0);
            constexpr uint32_t QUADS = MLP_BIAS_COLS / 4;
            constexpr uint32_t STEP = MLP_GRAD_THREADS / QUADS;
            constexpr uint32_t LOADS = MLP_BIAS_ROWS / STEP;
            const uint32_t q = tid % QUADS, r = tid / QUADS;
            f32x4 v[LOADS];
#pragma unroll
            for (uint32_t i = 0; i < LOADS; i++) {
                const uint32_t b = b0 + min(r + i * STEP, nr - 1u);
                v[i] = *reinterpret_cast<const f32x4*>(
                    a.dz + (size_t)b * n.nbias + c0 + q * 4u);
            }
#pragma unroll
            for (uint32_t i = 0; i < LOADS; i++) {
#pragma unroll
                for (uint32_t e = 0; e < 4; e++) {
                    cols[(q * 4u + e) * MLP_BIAS_STRIDE + r + i * STEP] = v[i][e];
                }
            }
            __syncthreads();
            if (tid < MLP_BIAS_COLS) {
                const f32x4* p4 = reinterpret_cast<const f32x4*>(
                    cols + tid * MLP_BIAS_STRIDE);
                for (uint32_t b = 0; b < nr; b += 32u) {
                    f32x4 x[8];
#pragma unroll
                    for (uint32_t i = 0; i < 8; i++) x[i] = p4[b / 4u + i];
#pragma unroll
                    for (uint32_t i = 0; i < 8; i++) {
                        s = s + x[i].x;
                        s = s + x[i].y;
                        s = s + x[i].z;
                        s = s + x[i].w;
                    }
                }
            }
            __syncthreads();
        }
        if (mine) {
            a.g[o] = s;
            if (ADAM) {
                adam_update(a.adam, s, &pv, &mv, &vv);
                a.p[o] = pv;
                a.m[o] = mv;
                a.v[o] = vv;
            }
        }
        return;
    }
    __shared__ double red[16];
    const uint32_t total = a.B * n.w[n.L];
    double s = 0.0;
    constexpr uint32_t AHEAD = 16;
    for (uint32_t t = tid; t < total; t += AHEAD * MLP_GRAD_THREADS) {
        double e[AHEAD];
#pragma unroll
        for (uint32_t i = 0; i < AHEAD; i++) {
            e[i] = a.terms[min(t + i * MLP_GRAD_THREADS, total - 1u)];
        }
#pragma unroll
        for (uint32_t i = 0; i < AHEAD; i++) {
            if (t + i * MLP_GRAD_THREADS < total) s += e[i];
        }
    }
    s = block_sum(s, red);
    if (tid == 0) {
        *a.loss = (float)(s / (double)a.B);
    }
}

// The update of all parameters from gradients already there, and of both
// padded BF16 copies of the weights, whose zeros between stay.  (With the
// copies made by mlp_pack_kernel afterwards a step of 3-256-256-256-65 took
// 18.6 us in place of 13.)
__global__ void __launch_bounds__(256)
mlp_adam_kernel(MlpNet n, AdamArgs a, uint32_t count, float* __restrict__ p,
                const float* __restrict__ g, float* __restrict__ m,
                float* __restrict__ v, uint16_t* __restrict__ W,
                uint16_t* __restrict__ WT)
{
    for (uint32_t i = blockIdx.x * 256u + threadIdx.x; i < count;
         i += gridDim.x * 256u) {
        const uint16_t h = f2bf(adam_update(a, g[i], p + i, m + i, v + i));
        // the layer's places, picked with fixed indexes: all arguments then
        // come in one trip (they lie in host memory)
        uint32_t po = 0, bo = 0, w = 1, wo = 0, wpi = 0, wpo = 0;
#pragma unroll
        for (uint32_t l = 0; l < MLP_MAX_LAYERS; l++) {
            if (l < n.L && i >= n.po[l]) {
                po = n.po[l];
                bo = n.bo[l];
                w = n.w[l];
                wo = n.wo[l];
                wpi = n.wp[l];
                wpo = n.wp[l + 1];
            }
        }
        if (i >= bo) continue;
        const uint32_t j = (i - po) / w, k = (i - po) % w;
        W[wo + mlp_frag(j, k, wpi)] = h;
        WT[wo + mlp_frag(k, j, wpo)] = h;
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
        W[n.wo[l] + mlp_frag(j, k, n.wp[l])] = h;
        WT[n.wo[l] + mlp_frag(k, j, n.wp[l + 1])] = h;
    }
}

}  // namespace vfps_impl
