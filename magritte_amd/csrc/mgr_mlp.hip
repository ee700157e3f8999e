// mgr_mlp.hip -- the learned warm start: a multilayer perceptron
// 8 -> 128 -> 128 -> 7 (GELU) that predicts per-cell log10 level-population
// fractions from local density, temperature, velocity gradient and a
// first-pass J, trained on populations the plain method converged.  It has no
// counterpart in the reference, whose starting point is LTE
// (Simulation::compute_LTE_level_populations, sim_lines.tpp:10-16); the plain
// LTE-started iteration stays the fallback, and the ALI loop that follows the
// warm start is unchanged, so converged populations are those of the plain
// method.
//
// Arithmetic: every matrix product runs on the CDNA4 matrix cores with
// bfloat16 operands, round to nearest even, and FP32 accumulation:
// v_mfma_f32_16x16x32_bf16 wherever K is a multiple of 32 (the hidden layer,
// the output layer, the back-propagation through W2 and the weight gradients,
// whose K is the tile's 64 rows), v_mfma_f32_16x16x16_bf16 for the two
// products with K = 16 (the 8 inputs and the 7 outputs, padded); biases,
// GELU, the loss and Adam run in FP32 on the FP32 master weights.
//
// Training runs without host round trips: minibatches are consecutive slices
// of a pseudo-random permutation of the rows computed on the device (a
// four-round Feistel network over the next even power of two with cycle
// walking, keyed per epoch), Adam's step count and the epoch's loss live in
// device memory, and each epoch is one hipGraph replay.
//
// Work mapping: the products are formed transposed, neurons by rows
// (D = W^T H^T), 16 rows (cells) to a wavefront: a lane's results, four
// consecutive neurons of one row, are then K values of the next product's
// right operand as they stand.  The M rows of two tiles take the neurons of 32
// in alternate fours (neuron), which puts the operand's eight values in order.
// Prediction: a wave's rows stay in its registers from the inputs to the outputs.
// Training: a workgroup takes tiles of 64 rows with 8 waves, two for the same 16
// rows, which form one half of the neurons each and hand each other their
// operands through LDS.  The weight gradients reduce over rows: their operands
// are transposed on the matrix cores (a product with the unit matrix, exact)
// and pass through LDS too, and each wave forms an eighth of the gradients over
// the 64 rows, accumulating in registers over all the tiles a workgroup takes.
// Per-workgroup partial gradients are reduced in a fixed order by the Adam
// kernel, so training is deterministic.
//
// MFMA operand layouts (lane l, r = l % 16, g = l / 16):
//   16x16x16: A[m = r][k = 4g + j], B[k = 4g + j][n = r], j = 0..3;
//   16x16x32: A[m = r][k = 8g + j], B[k = 8g + j][n = r], j = 0..7;
//   both:     D[m = 4g + j][n = r], j = 0..3.
#include <algorithm>
#include <cmath>
#include <cstring>
#include <vector>

#include "mgr_common.hpp"

using namespace mgr;

namespace {

constexpr int IN = MGR_MLP_IN;        // 8 features
constexpr int HID = MGR_MLP_HIDDEN;   // 128
constexpr int OUT = MGR_MLP_OUT;      // 7 levels
constexpr int KIN = 16;               // IN padded to one MFMA K step
constexpr int NOUT = 16;              // OUT padded to one MFMA N tile
constexpr int ROWS = 64;              // rows per workgroup tile
constexpr int THREADS = 256;           // of the forward kernel
constexpr int GRAD_THREADS = 512;      // of the gradient kernel

// packed FP32 parameters: W1 [IN][HID], b1, W2 [HID][HID], b2, W3 [HID][OUT], b3
constexpr int OFF_W1 = 0;
constexpr int OFF_B1 = OFF_W1 + IN * HID;
constexpr int OFF_W2 = OFF_B1 + HID;
constexpr int OFF_B2 = OFF_W2 + HID * HID;
constexpr int OFF_W3 = OFF_B2 + HID;
constexpr int OFF_B3 = OFF_W3 + HID * OUT;
constexpr int NPAR = OFF_B3 + OUT;

// bf16 weights as left operands A[m][k], one word per lane and MFMA: frag16
// for K = 16 (8 bytes), frag32 for K = 32 (16 bytes)
//   W1F  m = neuron, k = input (padded)     forward, layer 1
//   W2F  m = neuron, k = neuron of layer 1  forward, layer 2
//   W2B  m = neuron of layer 1, k = neuron  backward, dH1 = dZ2 W2^T
//   W3F  m = output (padded), k = neuron    forward, layer 3
//   W3B  m = neuron, k = output (padded)    backward, dH2 = dY W3^T
// neurons in m in the order of neuron_row, in k as they are.
// The padding entries are zero from the network's creation on.
constexpr int BF_W1F = 0;
constexpr int BF_W2F = BF_W1F + HID * KIN;
constexpr int BF_W3F = BF_W2F + HID * HID;
constexpr int BF_FORWARD = BF_W3F + NOUT * HID;   // what the forward pass needs
constexpr int BF_W2B = BF_FORWARD;
constexpr int BF_W3B = BF_W2B + HID * HID;
constexpr int BF_TOTAL = BF_W3B + HID * NOUT;

__device__ __forceinline__ int frag16(int m, int k) { return m / 16 * 256 + (k / 4 * 16 + m % 16) * 4 + k % 4; }
__device__ __forceinline__ int frag32(int m, int k)
{
    return ((m / 16 * (HID / 32) + k / 32) * 64 + k % 32 / 8 * 16 + m % 16) * 8 + k % 8;
}
// The neuron in row m of tile t, and the row (16 t + m) of a neuron.
__device__ __forceinline__ int neuron(int t, int m) { return t / 2 * 32 + m / 4 * 8 + t % 2 * 4 + m % 4; }
__device__ __forceinline__ int neuron_row(int u) { return (u / 32 * 2 + u % 8 / 4) * 16 + u % 32 / 8 * 4 + u % 4; }

// Partial gradients of a workgroup: the words as the threads hold them, so that
// they are written whole, with the loss at NPAR
//   W2 [q][i][thread][4], W1 [wave][g < 2][r][4], W3 [wave][g][r < OUT][4], b1, b2, b3
constexpr int PG_W1 = HID * HID;
constexpr int PG_W3 = PG_W1 + IN * HID;
constexpr int PG_B = PG_W3 + HID * OUT;

// LDS of the training kernel, 160 KB: the weights; the transposed operands of the
// weight gradients, tile t of two waves' 32 rows at ((t 2 + rows / 32) 64 + lane) 8
// + (rows / 16 % 2) 4; and one layer's right operands of the next product, K step
// kt of rows / 16 at ((rows / 16 4 + kt) 64 + lane) 8 (layer 2's pass through
// the tiles T_DZ1, which are written last)
constexpr int T_H1 = 0, T_DZ2 = 8, T_H2 = 16, T_DZ1 = 24, T_X = 32, T_DY = 33, T_TILES = 34;
constexpr int L_TILES = BF_TOTAL;                       // bf16 elements before the tiles
constexpr int L_PASS = L_TILES + T_TILES * 2 * 64 * 8;
constexpr size_t LDS_TRAIN = (size_t)(L_PASS + ROWS * HID) * 2;
static_assert(LDS_TRAIN <= 160 * 1024, "a CU's LDS");
constexpr int NBIAS = HID + HID + NOUT;
constexpr size_t LDS_FORWARD = (size_t)BF_FORWARD * 2 + NBIAS * sizeof(float) + ROWS * NOUT * sizeof(float);

typedef short s4 __attribute__((ext_vector_type(4)));
typedef short s8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf4 __attribute__((ext_vector_type(4)));
typedef float f4 __attribute__((ext_vector_type(4)));

__device__ __forceinline__ uint16_t f2bf(float x)
{
    uint32_t u = __float_as_uint(x);
    u += 0x7FFFu + ((u >> 16) & 1u);
    return (uint16_t)(u >> 16);
}
__device__ __forceinline__ float bf2f(uint16_t h) { return __uint_as_float((uint32_t)h << 16); }
__device__ __forceinline__ s4 ld4(const uint16_t *p) { return *reinterpret_cast<const s4 *>(p); }
__device__ __forceinline__ s8 ld8(const uint16_t *p) { return *reinterpret_cast<const s8 *>(p); }
// the same rounding (to nearest even) of four values
__device__ __forceinline__ s4 to_bf(f4 x) { return __builtin_bit_cast(s4, __builtin_convertvector(x, bf4)); }
__device__ __forceinline__ s8 join(s4 a, s4 b) { return __builtin_shufflevector(a, b, 0, 1, 2, 3, 4, 5, 6, 7); }

__device__ __forceinline__ f4 mfma(s4 a, s4 b, f4 c)
{
    return __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(a, b, c, 0, 0, 0);
}
__device__ __forceinline__ f4 mfma32(s8 a, s8 b, f4 c)
{
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf8, a), __builtin_bit_cast(bf8, b), c, 0, 0, 0);
}

constexpr float SQRT_2_OVER_PI = 0.7978845608028654f;
constexpr float GELU_C = 0.044715f;

// GELU (tanh form) and its derivative.  With p = 1 / (exp(2u) + 1),
// u = sqrt(2/pi) (z + c z^3) held to +-15, t = tanh u = 1 - 2 p, gelu =
// z (1 + t) / 2 and gelu' = (1 + t) / 2 + z (1 - t^2) u' / 2.  The reciprocal
// is the correctly rounded one.
__device__ __forceinline__ void gelu(float z, float &h, float &grad)
{
#pragma clang fp contract(off)
    float u = SQRT_2_OVER_PI * fmaf(z, z * (GELU_C * z), z);
    u = __builtin_amdgcn_fmed3f(u, -15.0f, 15.0f);
    const float d = __builtin_amdgcn_exp2f(u * (2.0f * 1.44269504f)) + 1.0f;
    float p = __builtin_amdgcn_rcpf(d);
    p = fmaf(fmaf(-d, p, 1.0f), p, p);   // the quotient 1 / d for every d in [1, 2^48)
    const float t = fmaf(-2.0f, p, 1.0f);
    const float w = fmaf(0.5f, t, 0.5f);
    h = z * w;
    const float du = 0.5f * SQRT_2_OVER_PI * fmaf(z, 3.0f * GELU_C * z, 1.0f);
    grad = du * (z * fmaf(-t, t, 1.0f)) + w;
}

struct Norm {
    float xm[IN], xs[IN], ym[OUT], ys[OUT];
};

// Device state of a training run: the epoch (counted from -1, advanced by
// k_epoch_begin at the start of every epoch replay), its permutation key
// and the shape of the permutation domain.
struct TrainState {
    int64_t  epoch;
    uint64_t seed, key;
    uint32_t n;              // rows permuted
    int      half;           // bits of each Feistel half
    uint32_t mask;           // (1 << half) - 1
};

// A four-round Feistel network on [0, 2^(2 half)): a bijection for any key.
__device__ __forceinline__ uint32_t feistel(uint32_t x, int half, uint32_t mask, uint64_t key)
{
    uint32_t L = x >> half, R = x & mask;
    for (int i = 0; i < 4; i++) {
        uint32_t f = R * 0x85EBCA6Bu + ((uint32_t)(key >> (16 * i)) ^ (0x9E3779B9u * (uint32_t)(i + 1)));
        f ^= f >> 13;
        f *= 0xC2B2AE35u;
        f ^= f >> 16;
        const uint32_t nl = R;
        R = (L ^ f) & mask;
        L = nl;
    }
    return (L << half) | R;
}

// Row at position i of the epoch's permutation of [0, n): the Feistel
// bijection, walked along its cycle until it lands inside [0, n) (the
// restriction of a permutation to a subset by cycle walking is a
// permutation of the subset).
__device__ __forceinline__ int64_t permuted_row(const TrainState &st, int64_t i)
{
    uint32_t x = (uint32_t)i;
    do { x = feistel(x, st.half, st.mask, st.key); } while (x >= st.n);
    return (int64_t)x;
}

__device__ __forceinline__ uint64_t mix64(uint64_t z)
{
    z += 0x9E3779B97F4A7C15ull;
    z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ull;
    z = (z ^ (z >> 27)) * 0x94D049BB133111EBull;
    return z ^ (z >> 31);
}

__global__ void k_epoch_begin(TrainState *st)
{
    st->epoch++;
    st->key = mix64(st->seed ^ mix64((uint64_t)st->epoch));
}

// Source row of batch row `row` (b0 + row of the epoch order, or idx[row],
// or row itself).
__device__ __forceinline__ int64_t source_row(const TrainState *st, const int64_t *idx, int64_t b0, int64_t row)
{
    if (st) return permuted_row(*st, b0 + row);
    return idx ? idx[row] : row;
}

// The parameter of word e of the partial gradients.
__device__ __forceinline__ int param_of(int e)
{
    const int j = e % 4;
    if (e < PG_W1) {
        const int lane = e / 4 % 64, wave = e / 256 % 8, i = e / 2048 % 4, q = e / 8192;
        return OFF_W2 + neuron(wave % 4 * 2 + q, lane / 16 * 4 + j) * HID + neuron(wave / 4 * 4 + i, lane % 16);
    }
    if (e < PG_W3) {
        const int i = (e - PG_W1) / 4, lane = i % 32, wave = i / 32;
        return OFF_W1 + (lane / 16 * 4 + j) * HID + neuron(wave, lane % 16);
    }
    if (e < PG_B) {
        const int i = (e - PG_W3) / 4, r = i % OUT, g = i / OUT % 4, wave = i / (4 * OUT);
        return OFF_W3 + neuron(wave, 4 * g + j) * OUT + r;
    }
    const int b = e - PG_B;
    return b < HID ? OFF_B1 + b : b < 2 * HID ? OFF_B2 + b - HID : OFF_B3 + b - 2 * HID;
}

// Copy the first `total` bf16 weights into LDS.
__device__ __forceinline__ void load_weights(uint16_t *s, const uint16_t *__restrict__ wbf, int total)
{
    const uint4 *src = reinterpret_cast<const uint4 *>(wbf);
    uint4 *dst = reinterpret_cast<uint4 *>(s);
#pragma unroll 10
    for (int i = threadIdx.x; i < total / 8; i += blockDim.x) dst[i] = src[i];
}

// The lane's inputs 4g .. 4g+3 normalised, as right operand: zeros in the
// padding and for a row that is not in the batch.
__device__ __forceinline__ s4 input_operand(f4 x, bool valid, f4 xm, f4 xs)
{
    const f4 v = (x - xm) / xs;
    return to_bf(valid ? v : f4{0.f, 0.f, 0.f, 0.f});
}

// GELU of four pre-activations as an operand, and its derivatives.
__device__ __forceinline__ s4 activate(f4 z, f4 &grad)
{
    f4 h;
#pragma unroll
    for (int j = 0; j < 4; j++) {
        float hj, dj;
        gelu(z[j], hj, dj);
        h[j] = hj;
        grad[j] = dj;
    }
    return to_bf(h);
}

// A K = 128 product of one M tile: its four operands w ((kt 64 + lane) 8) by b.
__device__ __forceinline__ f4 product(const uint16_t *w, const s8 b[4])
{
    const int lane = threadIdx.x & 63;
    f4 z = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int kt = 0; kt < 4; kt++) z = mfma32(ld8(w + (kt * 64 + lane) * 8), b[kt], z);
    return z;
}

// Outputs 4g + j of the 16 rows of one wave, row r of lane (r, g), with biases sB.
__device__ __forceinline__ f4 forward_rows(const uint16_t *s, const float *sB, s4 x)
{
    const int lane = threadIdx.x & 63, g = lane >> 4;
    f4 none;
    s4 h[8];
    s8 b[4];
#pragma unroll
    for (int mt = 0; mt < 8; mt++)
        h[mt] = activate(mfma(ld4(s + BF_W1F + (mt * 64 + lane) * 4), x, f4{0.f, 0.f, 0.f, 0.f}) +
                             *reinterpret_cast<const f4 *>(sB + neuron(mt, 4 * g)),
                         none);
#pragma unroll
    for (int kt = 0; kt < 4; kt++) b[kt] = join(h[2 * kt], h[2 * kt + 1]);
#pragma unroll
    for (int mt = 0; mt < 8; mt++)
        h[mt] = activate(product(s + BF_W2F + mt * 4 * 64 * 8, b) +
                             *reinterpret_cast<const f4 *>(sB + HID + neuron(mt, 4 * g)),
                         none);
#pragma unroll
    for (int kt = 0; kt < 4; kt++) b[kt] = join(h[2 * kt], h[2 * kt + 1]);
    return product(s + BF_W3F, b) + *reinterpret_cast<const f4 *>(sB + 2 * HID + 4 * g);
}

// Loss and gradients over rows [0, n) of a batch of X/T (rows b0 .. b0+n-1 of
// the epoch's permutation with st, else through idx when given, else the
// rows themselves): grid-stride over 64-row tiles; per-workgroup partial
// gradients (PG_W1) and partial loss go to part[blockIdx.x * (NPAR + 1)].
//
// Bound by vector instructions, most of them the GELUs', and per launch by the
// weights' way into LDS and the 74 KB of partial gradients.  With activations in
// row-major LDS (16-way bank conflicts on every operand) and gradient operands
// gathered two bytes at a time a 16384-row batch took 40 us and 400000 rows 590
// us; with 4 waves that hold all 128 neurons of their rows (413 registers, of
// which the upper half is moved in and out) 24 and 251; here 22 and 215.
__global__ __launch_bounds__(GRAD_THREADS) void k_mlp_grad(const float *__restrict__ X, const float *__restrict__ T,
                                                           const TrainState *st, const int64_t *__restrict__ idx,
                                                           int64_t b0, int64_t n, int64_t n_total,
                                                           const uint16_t *__restrict__ wbf,
                                                           const float *__restrict__ P,
                                                           const Norm *__restrict__ norm, float *__restrict__ part)
{
    extern __shared__ __align__(16) uint16_t s[];
    uint16_t *sT = s + L_TILES, *pass = s + L_PASS, *pass2 = sT + T_DZ1 * 2 * 64 * 8;
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63, r = lane & 15, g = lane >> 4;
    const int rb = wave & 3, mt0 = wave / 4 * 4;   // the wave's 16 rows and its first tile of neurons
    const float inv = 2.0f / ((float)n_total * (float)OUT);
    s4 unit;   // the unit matrix as right operand
    for (int j = 0; j < 4; j++) unit[j] = 4 * g + j == r ? 0x3F80 : 0;
    const f4 zero = {0.f, 0.f, 0.f, 0.f};
    auto put = [&](int t, s4 operand) {
        // rows 4g + j of neuron r: exact, the values are bf16
        const s4 v = to_bf(mfma(operand, unit, zero));
        *reinterpret_cast<s4 *>(sT + ((t * 2 + (rb >> 1)) * 64 + lane) * 8 + (rb & 1) * 4) = v;
    };
    auto get = [&](int t, int p) { return ld8(sT + ((t * 2 + p) * 64 + lane) * 8); };
    // this wave's half of a layer to the rows' two waves, and the whole of it
    auto give = [&](uint16_t *to, const s4 h[4]) {
#pragma unroll
        for (int i = 0; i < 2; i++)
            *reinterpret_cast<s8 *>(to + ((rb * 4 + mt0 / 2 + i) * 64 + lane) * 8) = join(h[2 * i], h[2 * i + 1]);
    };
    auto take = [&](const uint16_t *from, s8 b[4]) {
#pragma unroll
        for (int kt = 0; kt < 4; kt++) b[kt] = ld8(from + ((rb * 4 + kt) * 64 + lane) * 8);
    };

    f4 gW2[2][4], gW1 = zero, gW3 = zero;
#pragma unroll
    for (int i = 0; i < 4; i++) gW2[0][i] = gW2[1][i] = zero;
    float gb = 0.0f, loss = 0.0f;
    // the sum of a transposed operand's column m over the tile's rows, in their order
    auto column = [&](int t, int m, float sum) {
#pragma unroll
        for (int i = 0; i < 8; i++) {
            const s8 v = ld8(sT + ((t * 2 + i / 4) * 64 + i % 4 * 16 + m) * 8);
            for (int j = 0; j < 8; j++) sum += bf2f((uint16_t)v[j]);
        }
        return sum;
    };
    // bias gradients: dZ1 of threads 0..127, dZ2 of 128..255, dY of wave 4
    const int column_row = neuron_row(threadIdx.x % HID);
    const int column_tile = wave == 4 ? T_DY : (threadIdx.x < HID ? T_DZ1 : T_DZ2) + column_row / 16;
    const int column_m = wave == 4 ? r : column_row % 16;

    // a tile's inputs and targets are read before the weights, or the tile before, are dealt with
    f4 next_x = zero, next_t = zero;
    bool next_valid = false;
    auto fetch = [&](int64_t tile) {
        // the rows of two waves alternate in fours, as the neurons of two tiles do
        const int64_t row = tile * ROWS + neuron(rb, r);
        next_valid = row < n;
        if (!next_valid || g > 1) return;
        const int64_t src = source_row(st, idx, b0, row);
        next_x = *reinterpret_cast<const f4 *>(X + src * IN + 4 * g);
        for (int j = 0; j < 4; j++)
            if (4 * g + j < OUT) next_t[j] = T[src * OUT + 4 * g + j];
    };
    fetch(blockIdx.x);
    load_weights(s, wbf, BF_TOTAL);

    const int64_t ntiles = (n + ROWS - 1) / ROWS;
    for (int64_t tile = blockIdx.x; tile < ntiles; tile += gridDim.x) {
        // the biases and the normalisation are read again for every tile (out of
        // the cache): kept in registers they would push others out to memory
        const float *Pt = P;
        const Norm *nt = norm;
        asm volatile("" : "+s"(Pt), "+s"(nt));
        auto bias = [&](int layer, int i) {
            return *reinterpret_cast<const f4 *>(Pt + layer + neuron(mt0 + i, 4 * g));
        };
        const bool valid = next_valid && g < 2;
        f4 xn = next_x, t = next_t;   // normalised
        for (int j = 0; j < 4; j++) {
            if (g < 2) xn[j] = (xn[j] - nt->xm[4 * g + j]) / nt->xs[4 * g + j];
            if (4 * g + j < OUT) t[j] = (t[j] - nt->ym[4 * g + j]) / nt->ys[4 * g + j];
        }
        const s4 x = to_bf(valid ? xn : zero);
        __syncthreads();   // the weights are in place, the previous tile's operands consumed
        fetch(tile + gridDim.x);
        s4 h[4];
        s8 b[4];
        f4 g1[4], g2[4];
#pragma unroll
        for (int i = 0; i < 4; i++) {
            h[i] = activate(mfma(ld4(s + BF_W1F + ((mt0 + i) * 64 + lane) * 4), x, zero) + bias(OFF_B1, i), g1[i]);
            put(T_H1 + mt0 + i, h[i]);
        }
        give(pass, h);
        __syncthreads();
        take(pass, b);
#pragma unroll
        for (int i = 0; i < 4; i++) {
            h[i] = activate(product(s + BF_W2F + (mt0 + i) * 4 * 64 * 8, b) + bias(OFF_B2, i), g2[i]);
            put(T_H2 + mt0 + i, h[i]);
        }
        give(pass2, h);
        __syncthreads();
        take(pass2, b);
        const f4 y = product(s + BF_W3F, b);
        // dY = 2 (y - t) / (n_total OUT) on valid rows and outputs
        f4 d = zero;
        for (int j = 0; j < 4; j++)
            if (valid && 4 * g + j < OUT) {
                const float e = y[j] + Pt[OFF_B3 + 4 * g + j] - t[j];
                if (wave < 4) loss += e * e;
                d[j] = e * inv;
            }
        const s4 dy = to_bf(d);
        if (wave < 4) put(T_X, x);
        else put(T_DY, dy);
        // dH2 = dY W3^T, dZ2 = dH2 * gelu'(Z2)
#pragma unroll
        for (int i = 0; i < 4; i++) {
            h[i] = to_bf(mfma(ld4(s + BF_W3B + ((mt0 + i) * 64 + lane) * 4), dy, zero) * g2[i]);
            put(T_DZ2 + mt0 + i, h[i]);
        }
        give(pass, h);
        __syncthreads();
        take(pass, b);
        // dH1 = dZ2 W2^T, dZ1 = dH1 * gelu'(Z1)
#pragma unroll
        for (int i = 0; i < 4; i++)
            put(T_DZ1 + mt0 + i, to_bf(product(s + BF_W2B + (mt0 + i) * 4 * 64 * 8, b) * g1[i]));
        __syncthreads();
        // an eighth of the gradients over the tile's rows: W2 of 32 neurons by 64, W1 and W3 of 16
#pragma unroll
        for (int p = 0; p < 2; p++) {
            const s8 ha = get(T_H1 + 2 * rb, p), hb = get(T_H1 + 2 * rb + 1, p);
#pragma unroll
            for (int i = 0; i < 4; i++) {
                const s8 dz = get(T_DZ2 + mt0 + i, p);
                gW2[0][i] = mfma32(ha, dz, gW2[0][i]);
                gW2[1][i] = mfma32(hb, dz, gW2[1][i]);
            }
            gW1 = mfma32(get(T_X, p), get(T_DZ1 + wave, p), gW1);
            gW3 = mfma32(get(T_H2 + wave, p), get(T_DY, p), gW3);
        }
        if (wave < 5) gb = column(column_tile, column_m, gb);
    }

    float *out = part + (int64_t)blockIdx.x * (NPAR + 1);
#pragma unroll
    for (int q = 0; q < 2; q++)
#pragma unroll
        for (int i = 0; i < 4; i++)
            *reinterpret_cast<f4 *>(out + ((q * 4 + i) * GRAD_THREADS + threadIdx.x) * 4) = gW2[q][i];
    if (g < 2) *reinterpret_cast<f4 *>(out + PG_W1 + (wave * 32 + lane) * 4) = gW1;
    if (r < OUT) *reinterpret_cast<f4 *>(out + PG_W3 + ((wave * 4 + g) * OUT + r) * 4) = gW3;
    if (wave < 4) out[PG_B + threadIdx.x] = gb;
    if (wave == 4 && g == 0 && r < OUT) out[PG_B + 2 * HID + r] = gb;
    // loss: wave sums, then one lane adds the waves' in order
    for (int off = 32; off > 0; off >>= 1) loss += __shfl_down(loss, off, 64);
    __syncthreads();   // the operands are consumed
    float *wl = reinterpret_cast<float *>(sT);
    if (lane == 0) wl[wave] = loss;
    __syncthreads();
    if (threadIdx.x == 0) out[NPAR] = (wl[0] + wl[1]) + (wl[2] + wl[3]);
}

// bf16 copies of master parameter p in the weight layouts.
__device__ __forceinline__ void repack_param(int p, float x, uint16_t *__restrict__ wbf)
{
    const uint16_t h = f2bf(x);
    if (p < OFF_B1) {                        // W1 [i][o]
        const int i = (p - OFF_W1) / HID, o = (p - OFF_W1) % HID;
        wbf[BF_W1F + frag16(neuron_row(o), i)] = h;
    } else if (p >= OFF_W2 && p < OFF_B2) {  // W2 [i][o]
        const int k = p - OFF_W2, i = k / HID, o = k % HID;
        wbf[BF_W2F + frag32(neuron_row(o), i)] = h;
        wbf[BF_W2B + frag32(neuron_row(i), o)] = h;
    } else if (p >= OFF_W3 && p < OFF_B3) {  // W3 [i][o]
        const int k = p - OFF_W3, i = k / OUT, o = k % OUT;
        wbf[BF_W3F + frag32(o, i)] = h;
        wbf[BF_W3B + frag16(neuron_row(i), o)] = h;
    }
}

// Sum the G partials of each parameter in a fixed order (8 interleaved
// sequential sums, then a fixed tree: deterministic), optionally apply one
// Adam step and refresh the parameter's bf16 copies.  Blocks of 256 threads
// cover 32 parameters (p = NPAR is the loss); with 16 loads of a thread in
// flight, 256 partials (19 MB) take 7.9 us, with the compiler's
// choice 13.  In a training run (st given)
// the step is step0 + epoch * nbatch + batch + 1 and the loss sum is added to
// loss_acc[epoch]; otherwise c1, c2 are given.
constexpr int RED_P = 32, RED_W = 8;
__global__ __launch_bounds__(RED_P * RED_W) void k_mlp_reduce_adam(
    const float *__restrict__ part, int G, float *__restrict__ grad_out, float *__restrict__ P,
    float *__restrict__ m, float *__restrict__ v, uint16_t *__restrict__ wbf, int do_adam, float lr, float c1,
    float c2, const TrainState *st, int64_t step0, int64_t nbatch, int64_t batch, float *__restrict__ loss_acc)
{
    __shared__ float sh[RED_W][RED_P];
    const int pi = threadIdx.x % RED_P, wi = threadIdx.x / RED_P;
    const int e = blockIdx.x * RED_P + pi;
    float s = 0.0f;
    if (e <= NPAR) {
#pragma unroll 16
        for (int w = wi; w < G; w += RED_W) s += part[(int64_t)w * (NPAR + 1) + e];
    }
    sh[wi][pi] = s;
    __syncthreads();
    if (wi != 0 || e > NPAR) return;
    const int p = e < NPAR ? param_of(e) : NPAR;
    const float gsum = ((sh[0][pi] + sh[1][pi]) + (sh[2][pi] + sh[3][pi])) +
                       ((sh[4][pi] + sh[5][pi]) + (sh[6][pi] + sh[7][pi]));
    if (grad_out) grad_out[p] = gsum;
    if (st && p == NPAR && loss_acc) loss_acc[st->epoch] += gsum;
    if (!do_adam || p == NPAR) return;
    if (st) {
        const float t = (float)(step0 + st->epoch * nbatch + batch + 1);
        c1 = 1.0f - powf(0.9f, t);
        c2 = 1.0f - powf(0.999f, t);
    }
    const float b1 = 0.9f, b2 = 0.999f, eps = 1e-8f;
    const float mm = b1 * m[p] + (1.0f - b1) * gsum;
    const float vv = b2 * v[p] + (1.0f - b2) * gsum * gsum;
    m[p] = mm;
    v[p] = vv;
    const float x = P[p] - lr * (mm / c1) / (sqrtf(vv / c2) + eps);
    P[p] = x;
    if (wbf) repack_param(p, x, wbf);
}

// FP32 master parameters -> the bf16 layouts.
__global__ void k_mlp_pack(const float *__restrict__ P, uint16_t *__restrict__ wbf)
{
    const int p = blockIdx.x * blockDim.x + threadIdx.x;
    if (p < NPAR) repack_param(p, P[p], wbf);
}

// Forward only: Y (de-normalised) for rows [0, n), or, with pop != null, the
// level populations pop[p V + i] = pop_tot[p] 10^y_i / sum_i 10^y_i.
__global__ __launch_bounds__(THREADS) void k_mlp_forward(const float *__restrict__ X, int64_t n,
                                                         const uint16_t *__restrict__ wbf,
                                                         const float *__restrict__ P,
                                                         const Norm *__restrict__ norm, float *__restrict__ Y,
                                                         const double *__restrict__ pop_tot,
                                                         double *__restrict__ pop)
{
    extern __shared__ __align__(16) uint16_t s[];
    float *sB = reinterpret_cast<float *>(s + BF_FORWARD);
    float(*sy)[NOUT] = reinterpret_cast<float(*)[NOUT]>(sB + NBIAS);
    load_weights(s, wbf, BF_FORWARD);
    for (int i = threadIdx.x; i < NBIAS; i += THREADS)
        sB[i] = i < HID           ? P[OFF_B1 + i]
                : i < 2 * HID     ? P[OFF_B2 + i - HID]
                : i < 2 * HID + OUT ? P[OFF_B3 + i - 2 * HID]
                                  : 0.0f;
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63, r = lane & 15, g = lane >> 4;
    f4 xm{}, xs{1.f, 1.f, 1.f, 1.f}, ym{}, ys{};
    for (int j = 0; j < 4; j++) {
        if (g < 2) {
            xm[j] = norm->xm[4 * g + j];
            xs[j] = norm->xs[4 * g + j];
        }
        if (4 * g + j < OUT) {
            ym[j] = norm->ym[4 * g + j];
            ys[j] = norm->ys[4 * g + j];
        }
    }
    const int64_t ntiles = (n + ROWS - 1) / ROWS;
    for (int64_t tile = blockIdx.x; tile < ntiles; tile += gridDim.x) {
        const int64_t row = tile * ROWS + wave * 16 + r;
        const bool valid = row < n && g < 2;
        const s4 x = input_operand(valid ? *reinterpret_cast<const f4 *>(X + row * IN + 4 * g) : xm, valid, xm, xs);
        __syncthreads();   // the weights are in place, the previous tile's outputs read
        const f4 y = forward_rows(s, sB, x);
        for (int j = 0; j < 4; j++) {
            const int i = 4 * g + j;
            const float v = y[j] * ys[j] + ym[j];
            sy[wave * 16 + r][i] = v;
            if (Y && row < n && i < OUT) Y[row * OUT + i] = v;
        }
        __syncthreads();
        if (pop && threadIdx.x < ROWS) {
            const int64_t row = tile * ROWS + threadIdx.x;
            if (row < n) {
                double f[OUT], sum = 0.0;
                double mx = -1e300;
                for (int i = 0; i < OUT; i++) mx = fmax(mx, (double)sy[threadIdx.x][i]);
                for (int i = 0; i < OUT; i++) {
                    f[i] = exp10((double)sy[threadIdx.x][i] - mx);
                    sum += f[i];
                }
                for (int i = 0; i < OUT; i++) pop[row * OUT + i] = pop_tot[row] * (f[i] / sum);
            }
        }
    }
}

// The warm start's guard: a cell whose predicted populations are not all
// finite and positive, or give one of its lines an opacity <= 0 (the sign of
// n_j B_a - n_i B_s, as the emissivity/opacity kernel forms it), takes back
// the populations it held before the prediction.  near_bad is cleared for that
// kernel, which sets it anew.
__global__ void k_warm_guard(int64_t N, int V, int L, const int32_t *__restrict__ irad,
                             const int32_t *__restrict__ jrad, const double *__restrict__ Ba,
                             const double *__restrict__ Bs, const double *__restrict__ prev,
                             double *__restrict__ pop, unsigned long long *__restrict__ count,
                             int32_t *__restrict__ near_bad)
{
    const int64_t p = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (p >= N) return;
    if (p == 0) *near_bad = 0;
    double *x = pop + p * V;
    bool ok = true;
    for (int i = 0; i < V; i++) ok = ok && x[i] > 0.0 && __builtin_isfinite(x[i]);
    for (int k = 0; k < L; k++) ok = ok && (x[jrad[k]] * Ba[k] - x[irad[k]] * Bs[k] > 0.0);
    if (!ok) {
        for (int i = 0; i < V; i++) x[i] = prev[p * V + i];
        atomicAdd(count, 1ull);
    }
}

// Per-cell features of the warm start (after a first radiation field and
// J_eff from the starting populations):
//   0 log10 n(collision partner 0)   1 log10 T   2 log10 n(species)
//   3 log10 max over neighbours |v_nb - v_p| / |x_nb - x_p|  (s^-1)
//   4..7 log10 (Jlin_k / B_nu_k(T)) for transitions k = 0..3 (0 if absent)
__global__ void k_features(int64_t N, int L, int nspecs, int num, int partner, const double *__restrict__ abundance,
                           const double *__restrict__ T, const double *__restrict__ pos,
                           const double *__restrict__ vel, const int64_t *__restrict__ nb_off,
                           const int32_t *__restrict__ nb, const double *__restrict__ frequency,
                           const double *__restrict__ Jlin, float *__restrict__ X)
{
    const int64_t p = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (p >= N) return;
    const double floor_ = 1e-30;
    const double npart = abundance[p * nspecs + (partner >= 0 ? partner : num)];
    float *x = X + p * IN;
    x[0] = (float)log10(fmax(npart, floor_));
    x[1] = (float)log10(fmax(T[p], floor_));
    x[2] = (float)log10(fmax(abundance[p * nspecs + num], floor_));
    double gmax = 0.0;
    for (int64_t e = nb_off[p]; e < nb_off[p + 1]; e++) {
        const int64_t q = nb[e];
        double dv2 = 0.0, dx2 = 0.0;
        for (int d = 0; d < 3; d++) {
            const double dv = vel[3 * q + d] - vel[3 * p + d];
            const double dx = pos[3 * q + d] - pos[3 * p + d];
            dv2 += dv * dv;
            dx2 += dx * dx;
        }
        if (dx2 > 0.0) gmax = fmax(gmax, sqrt(dv2 / dx2));
    }
    x[3] = (float)log10(fmax(gmax * CC, floor_));
    for (int k = 0; k < 4; k++) {
        float f = 0.0f;
        if (k < L && Jlin) {   // Jlin null: no first pass, the inputs are 0
            const double nu = frequency[k];
            const double B = TWO_HH_OVER_CC_SQUARED * nu * nu * nu / expm1(HH_OVER_KB * nu / T[p]);
            f = (float)log10(fmax(Jlin[p * L + k] / B, floor_));
        }
        x[4 + k] = f;
    }
}

}  // namespace

struct mgr_mlp {
    int device = 0;
    hipStream_t stream = nullptr;
    std::string err;
    float *P = nullptr, *m = nullptr, *v = nullptr;   // [NPAR] master and Adam moments
    uint16_t *wbf = nullptr;                          // [BF_TOTAL]
    Norm *norm = nullptr;
    Norm h_norm;
    int64_t step = 0;
    bool jlin_inputs = true;   // reads inputs 4..7 (Jlin / B_nu after a first pass)
    int fail(int code, const std::string &msg)
    {
        err = msg;
        return code;
    }
};

#define MLP_HIP(call)                                                                \
    do {                                                                             \
        hipError_t e_ = (call);                                                      \
        if (e_ != hipSuccess) {                                                      \
            mlp->fail(MGR_ERR_DEVICE, std::string(#call) + ": " + hipGetErrorString(e_)); \
            return MGR_ERR_DEVICE;                                                   \
        }                                                                            \
    } while (0)

static int mlp_pack(mgr_mlp *mlp)
{
    hipLaunchKernelGGL(k_mlp_pack, dim3((NPAR + 255) / 256), dim3(256), 0, mlp->stream, mlp->P, mlp->wbf);
    MLP_HIP(hipGetLastError());
    return MGR_OK;
}

static int mlp_lds_attr(mgr_mlp *mlp)
{
    MLP_HIP(hipFuncSetAttribute((const void *)k_mlp_grad, hipFuncAttributeMaxDynamicSharedMemorySize, (int)LDS_TRAIN));
    MLP_HIP(hipFuncSetAttribute((const void *)k_mlp_forward, hipFuncAttributeMaxDynamicSharedMemorySize, (int)LDS_FORWARD));
    return MGR_OK;
}

extern "C" int64_t mgr_mlp_num_params(void) { return NPAR; }

extern "C" const char *mgr_mlp_last_error(const mgr_mlp *mlp) { return mlp ? mlp->err.c_str() : "null mlp"; }

extern "C" int mgr_mlp_create(int device, uint64_t seed, mgr_mlp **out)
{
    if (!out) return MGR_ERR_ARGUMENT;
    *out = nullptr;
    mgr_mlp *mlp = new mgr_mlp();
    mlp->device = device;
    auto bail = [&](int rc) {
        mgr_mlp_destroy(mlp);
        return rc;
    };
    if (hipSetDevice(device) != hipSuccess) return bail(MGR_ERR_DEVICE);
    if (hipStreamCreate(&mlp->stream) != hipSuccess) return bail(MGR_ERR_DEVICE);
    if (mgr::device_malloc(&mlp->P, NPAR * sizeof(float)) != hipSuccess || mgr::device_malloc(&mlp->m, NPAR * sizeof(float)) != hipSuccess ||
        mgr::device_malloc(&mlp->v, NPAR * sizeof(float)) != hipSuccess ||
        mgr::device_malloc(&mlp->wbf, BF_TOTAL * sizeof(uint16_t)) != hipSuccess ||
        mgr::device_malloc(&mlp->norm, sizeof(Norm)) != hipSuccess)
        return bail(MGR_ERR_NOMEM);
    // He-style initialisation from a 64-bit LCG + Box-Muller, zero biases
    std::vector<float> P(NPAR, 0.0f);
    uint64_t st = seed * 6364136223846793005ULL + 1442695040888963407ULL;
    auto uni = [&]() {
        st = st * 6364136223846793005ULL + 1442695040888963407ULL;
        return ((st >> 11) + 0.5) * (1.0 / 9007199254740992.0);
    };
    auto gauss = [&]() { return std::sqrt(-2.0 * std::log(uni())) * std::cos(2.0 * PI * uni()); };
    for (int i = 0; i < IN * HID; i++) P[OFF_W1 + i] = (float)(gauss() * std::sqrt(2.0 / IN));
    for (int i = 0; i < HID * HID; i++) P[OFF_W2 + i] = (float)(gauss() * std::sqrt(2.0 / HID));
    for (int i = 0; i < HID * OUT; i++) P[OFF_W3 + i] = (float)(gauss() * std::sqrt(1.0 / HID));
    for (int i = 0; i < IN; i++) { mlp->h_norm.xm[i] = 0.0f; mlp->h_norm.xs[i] = 1.0f; }
    for (int i = 0; i < OUT; i++) { mlp->h_norm.ym[i] = 0.0f; mlp->h_norm.ys[i] = 1.0f; }
    if (hipMemcpy(mlp->P, P.data(), NPAR * sizeof(float), hipMemcpyHostToDevice) != hipSuccess ||
        hipMemset(mlp->m, 0, NPAR * sizeof(float)) != hipSuccess ||
        hipMemset(mlp->v, 0, NPAR * sizeof(float)) != hipSuccess ||
        hipMemset(mlp->wbf, 0, BF_TOTAL * sizeof(uint16_t)) != hipSuccess ||
        hipMemcpy(mlp->norm, &mlp->h_norm, sizeof(Norm), hipMemcpyHostToDevice) != hipSuccess)
        return bail(MGR_ERR_DEVICE);
    int rc = mlp_lds_attr(mlp);
    if (!rc) rc = mlp_pack(mlp);
    if (!rc && hipStreamSynchronize(mlp->stream) != hipSuccess) rc = MGR_ERR_DEVICE;
    if (rc) return bail(rc);
    *out = mlp;
    return MGR_OK;
}

extern "C" void mgr_mlp_destroy(mgr_mlp *mlp)
{
    if (!mlp) return;
    (void)hipSetDevice(mlp->device);
    if (mlp->stream) (void)hipStreamSynchronize(mlp->stream);
    if (mlp->P) (void)hipFree(mlp->P);
    if (mlp->m) (void)hipFree(mlp->m);
    if (mlp->v) (void)hipFree(mlp->v);
    if (mlp->wbf) (void)hipFree(mlp->wbf);
    if (mlp->norm) (void)hipFree(mlp->norm);
    if (mlp->stream) (void)hipStreamDestroy(mlp->stream);
    delete mlp;
}

extern "C" int mgr_mlp_set_params(mgr_mlp *mlp, const float *params)
{
    if (!mlp || !params) return MGR_ERR_ARGUMENT;
    MLP_HIP(hipSetDevice(mlp->device));
    MLP_HIP(hipMemcpy(mlp->P, params, NPAR * sizeof(float), hipMemcpyHostToDevice));
    MLP_HIP(hipMemset(mlp->m, 0, NPAR * sizeof(float)));
    MLP_HIP(hipMemset(mlp->v, 0, NPAR * sizeof(float)));
    mlp->step = 0;
    int rc = mlp_pack(mlp);
    if (rc) return rc;
    MLP_HIP(hipStreamSynchronize(mlp->stream));
    return MGR_OK;
}

extern "C" int mgr_mlp_get_params(mgr_mlp *mlp, float *params)
{
    if (!mlp || !params) return MGR_ERR_ARGUMENT;
    MLP_HIP(hipSetDevice(mlp->device));
    MLP_HIP(hipStreamSynchronize(mlp->stream));
    MLP_HIP(hipMemcpy(params, mlp->P, NPAR * sizeof(float), hipMemcpyDeviceToHost));
    return MGR_OK;
}

extern "C" int mgr_mlp_set_normalisation(mgr_mlp *mlp, const float *x_mean, const float *x_std, const float *y_mean,
                                         const float *y_std)
{
    if (!mlp || !x_mean || !x_std || !y_mean || !y_std) return MGR_ERR_ARGUMENT;
    for (int i = 0; i < IN; i++)
        if (!(x_std[i] > 0.0f)) return mlp->fail(MGR_ERR_ARGUMENT, "x_std must be positive");
    for (int i = 0; i < OUT; i++)
        if (!(y_std[i] > 0.0f)) return mlp->fail(MGR_ERR_ARGUMENT, "y_std must be positive");
    std::memcpy(mlp->h_norm.xm, x_mean, sizeof(mlp->h_norm.xm));
    std::memcpy(mlp->h_norm.xs, x_std, sizeof(mlp->h_norm.xs));
    std::memcpy(mlp->h_norm.ym, y_mean, sizeof(mlp->h_norm.ym));
    std::memcpy(mlp->h_norm.ys, y_std, sizeof(mlp->h_norm.ys));
    MLP_HIP(hipSetDevice(mlp->device));
    MLP_HIP(hipMemcpy(mlp->norm, &mlp->h_norm, sizeof(Norm), hipMemcpyHostToDevice));
    return MGR_OK;
}

// Workgroups for n rows: one per tile up to `most`.  The gradient kernel fills
// a CU with one workgroup, and each costs 74 KB of partial gradients: more
// than one per CU only adds to both (400000 rows: the reduction takes 6 us
// after 256 workgroups, 40 after 1024).
constexpr int GRAD_GROUPS = 256;
static int grid_for_rows(int64_t n, int most)
{
    const int64_t tiles = (n + ROWS - 1) / ROWS;
    return (int)std::min<int64_t>(std::max<int64_t>(tiles, 1), most);
}

extern "C" int mgr_mlp_forward(mgr_mlp *mlp, const float *X, int64_t n, float *Y)
{
    if (!mlp || !X || !Y || n < 0) return MGR_ERR_ARGUMENT;
    if (n == 0) return MGR_OK;
    MLP_HIP(hipSetDevice(mlp->device));
    float *dX = nullptr, *dY = nullptr;
    MLP_HIP(mgr::device_malloc(&dX, n * IN * sizeof(float)));
    if (mgr::device_malloc(&dY, n * OUT * sizeof(float)) != hipSuccess) {
        (void)hipFree(dX);
        return mlp->fail(MGR_ERR_NOMEM, "forward: output allocation");
    }
    int rc = MGR_OK;
    if (hipMemcpy(dX, X, n * IN * sizeof(float), hipMemcpyHostToDevice) != hipSuccess) rc = MGR_ERR_DEVICE;
    if (!rc) {
        hipLaunchKernelGGL(k_mlp_forward, dim3(grid_for_rows(n, 1024)), dim3(THREADS), LDS_FORWARD, mlp->stream, dX, n,
                           mlp->wbf, mlp->P, mlp->norm, dY, (const double *)nullptr, (double *)nullptr);
        if (hipGetLastError() != hipSuccess || hipStreamSynchronize(mlp->stream) != hipSuccess) rc = MGR_ERR_DEVICE;
    }
    if (!rc && hipMemcpy(Y, dY, n * OUT * sizeof(float), hipMemcpyDeviceToHost) != hipSuccess) rc = MGR_ERR_DEVICE;
    (void)hipFree(dX);
    (void)hipFree(dY);
    if (rc) return mlp->fail(rc, "forward failed");
    return MGR_OK;
}

// one gradient evaluation of rows [0, n) of device-resident X/T (no Adam step)
static int mlp_grad_device(mgr_mlp *mlp, const float *dX, const float *dT, int64_t n, float *dpart, int G,
                           float *dgrad)
{
    hipLaunchKernelGGL(k_mlp_grad, dim3(G), dim3(GRAD_THREADS), LDS_TRAIN, mlp->stream, dX, dT,
                       (const TrainState *)nullptr, (const int64_t *)nullptr, (int64_t)0, n, n, mlp->wbf, mlp->P,
                       mlp->norm, dpart);
    MLP_HIP(hipGetLastError());
    hipLaunchKernelGGL(k_mlp_reduce_adam, dim3((NPAR + 1 + RED_P - 1) / RED_P), dim3(RED_P * RED_W), 0, mlp->stream,
                       dpart, G, dgrad, mlp->P, mlp->m, mlp->v, (uint16_t *)nullptr, 0, 0.0f, 1.0f, 1.0f,
                       (const TrainState *)nullptr, (int64_t)0, (int64_t)0, (int64_t)0, (float *)nullptr);
    MLP_HIP(hipGetLastError());
    return MGR_OK;
}

extern "C" int mgr_mlp_loss_grad(mgr_mlp *mlp, const float *X, const float *T, int64_t n, float *loss, float *grad)
{
    if (!mlp || !X || !T || n <= 0) return MGR_ERR_ARGUMENT;
    MLP_HIP(hipSetDevice(mlp->device));
    const int G = grid_for_rows(n, GRAD_GROUPS);
    float *dX = nullptr, *dT = nullptr, *dpart = nullptr, *dgrad = nullptr;
    int rc = MGR_OK;
    if (mgr::device_malloc(&dX, n * IN * sizeof(float)) != hipSuccess || mgr::device_malloc(&dT, n * OUT * sizeof(float)) != hipSuccess ||
        mgr::device_malloc(&dpart, (size_t)G * (NPAR + 1) * sizeof(float)) != hipSuccess ||
        mgr::device_malloc(&dgrad, (NPAR + 1) * sizeof(float)) != hipSuccess)
        rc = MGR_ERR_NOMEM;
    if (!rc && (hipMemcpy(dX, X, n * IN * sizeof(float), hipMemcpyHostToDevice) != hipSuccess ||
                hipMemcpy(dT, T, n * OUT * sizeof(float), hipMemcpyHostToDevice) != hipSuccess))
        rc = MGR_ERR_DEVICE;
    if (!rc) rc = mlp_grad_device(mlp, dX, dT, n, dpart, G, dgrad);
    std::vector<float> h(NPAR + 1);
    if (!rc && (hipStreamSynchronize(mlp->stream) != hipSuccess ||
                hipMemcpy(h.data(), dgrad, (NPAR + 1) * sizeof(float), hipMemcpyDeviceToHost) != hipSuccess))
        rc = MGR_ERR_DEVICE;
    (void)hipFree(dX); (void)hipFree(dT); (void)hipFree(dpart); (void)hipFree(dgrad);
    if (rc) return mlp->fail(rc, "loss_grad failed");
    if (grad) std::memcpy(grad, h.data(), NPAR * sizeof(float));
    if (loss) *loss = h[NPAR] / (float)(n * OUT);
    return MGR_OK;
}

// One epoch = minibatches b0 = 0, batch, 2 batch, ... of the epoch's row
// permutation, each a gradient and an Adam step with the bf16 repack; captured
// once as a hipGraph and replayed per epoch, with no host synchronisation
// until the end.
extern "C" int mgr_mlp_train(mgr_mlp *mlp, const float *X, const float *T, int64_t n, int64_t epochs, int64_t batch,
                             float lr, uint64_t seed, float *loss_per_epoch)
{
    if (!mlp || !X || !T || n <= 0 || epochs <= 0 || batch <= 0 || !(lr > 0.0f)) return MGR_ERR_ARGUMENT;
    if (n > (int64_t)1 << 31) return mlp->fail(MGR_ERR_ARGUMENT, "more than 2^31 training rows");
    MLP_HIP(hipSetDevice(mlp->device));
    const int64_t nbatch = (n + batch - 1) / batch;
    const int Gmax = grid_for_rows(std::min(batch, n), GRAD_GROUPS);
    float *dX = nullptr, *dT = nullptr, *dpart = nullptr, *dloss = nullptr;
    TrainState *dst = nullptr;
    int rc = MGR_OK;
    if (mgr::device_malloc(&dX, n * IN * sizeof(float)) != hipSuccess || mgr::device_malloc(&dT, n * OUT * sizeof(float)) != hipSuccess ||
        mgr::device_malloc(&dpart, (size_t)Gmax * (NPAR + 1) * sizeof(float)) != hipSuccess ||
        mgr::device_malloc(&dloss, epochs * sizeof(float)) != hipSuccess || mgr::device_malloc(&dst, sizeof(TrainState)) != hipSuccess)
        rc = MGR_ERR_NOMEM;
    TrainState h{};
    h.epoch = -1;
    h.seed = seed * 0x9E3779B97F4A7C15ull + 0x632BE59BD9B4E019ull;
    h.n = (uint32_t)n;
    int bits = 2;
    while (((int64_t)1 << bits) < n) bits += 2;
    h.half = bits / 2;
    h.mask = (1u << h.half) - 1u;
    if (!rc && (hipMemcpy(dX, X, n * IN * sizeof(float), hipMemcpyHostToDevice) != hipSuccess ||
                hipMemcpy(dT, T, n * OUT * sizeof(float), hipMemcpyHostToDevice) != hipSuccess ||
                hipMemcpy(dst, &h, sizeof(h), hipMemcpyHostToDevice) != hipSuccess ||
                hipMemset(dloss, 0, epochs * sizeof(float)) != hipSuccess))
        rc = MGR_ERR_DEVICE;
    hipGraph_t graph = nullptr;
    hipGraphExec_t exec = nullptr;
    if (!rc && hipStreamBeginCapture(mlp->stream, hipStreamCaptureModeThreadLocal) != hipSuccess) rc = MGR_ERR_DEVICE;
    if (!rc) {
        hipLaunchKernelGGL(k_epoch_begin, dim3(1), dim3(1), 0, mlp->stream, dst);
        for (int64_t b = 0; b < nbatch; b++) {
            const int64_t b0 = b * batch, nb = std::min(batch, n - b0);
            const int G = grid_for_rows(nb, GRAD_GROUPS);
            hipLaunchKernelGGL(k_mlp_grad, dim3(G), dim3(GRAD_THREADS), LDS_TRAIN, mlp->stream, dX, dT,
                               (const TrainState *)dst, (const int64_t *)nullptr, b0, nb, nb, mlp->wbf, mlp->P,
                               mlp->norm, dpart);
            hipLaunchKernelGGL(k_mlp_reduce_adam, dim3((NPAR + 1 + RED_P - 1) / RED_P), dim3(RED_P * RED_W), 0,
                               mlp->stream, dpart, G, (float *)nullptr, mlp->P, mlp->m, mlp->v, mlp->wbf, 1, lr, 1.0f,
                               1.0f, (const TrainState *)dst, mlp->step, nbatch, b, dloss);
        }
        const hipError_t le = hipGetLastError();
        const hipError_t ce = hipStreamEndCapture(mlp->stream, &graph);
        if (le != hipSuccess || ce != hipSuccess ||
            hipGraphInstantiate(&exec, graph, nullptr, nullptr, 0) != hipSuccess)
            rc = MGR_ERR_DEVICE;
    }
    for (int64_t e = 0; !rc && e < epochs; e++)
        if (hipGraphLaunch(exec, mlp->stream) != hipSuccess) rc = MGR_ERR_DEVICE;
    if (!rc && hipStreamSynchronize(mlp->stream) != hipSuccess) rc = MGR_ERR_DEVICE;
    if (!rc) mlp->step += epochs * nbatch;
    if (!rc && loss_per_epoch) {
        std::vector<float> l(epochs);
        if (hipMemcpy(l.data(), dloss, epochs * sizeof(float), hipMemcpyDeviceToHost) != hipSuccess) rc = MGR_ERR_DEVICE;
        for (int64_t e = 0; !rc && e < epochs; e++) loss_per_epoch[e] = (float)((double)l[e] / ((double)n * OUT));
    }
    if (exec) (void)hipGraphExecDestroy(exec);
    if (graph) (void)hipGraphDestroy(graph);
    (void)hipFree(dX); (void)hipFree(dT); (void)hipFree(dpart); (void)hipFree(dloss); (void)hipFree(dst);
    if (rc) return mlp->fail(rc, "train failed");
    return MGR_OK;
}

// ---- context side: features and warm start -----------------------------------

namespace mgr {
int launch_features(mgr_ctx *ctx, float *dX, bool jlin);
}

int mgr::launch_features(mgr_ctx *ctx, float *dX, bool jlin)
{
    const int partner = ctx->h_cp_num.empty() ? -1 : (int)ctx->h_cp_num[0];
    hipLaunchKernelGGL(k_features, dim3((unsigned)((ctx->N + 255) / 256)), dim3(256), 0, ctx->stream, ctx->N,
                       (int)ctx->L, (int)ctx->nspecs, (int)ctx->num, partner, ctx->abundance, ctx->temperature,
                       ctx->pos, ctx->vel, ctx->nb_off, ctx->nb, ctx->frequency, jlin ? ctx->Jlin : nullptr, dX);
    MGR_LAUNCH_CHECK();
    return MGR_OK;
}

extern "C" int mgr_features(mgr_ctx *ctx, float *X)
{
    if (!ctx || !X) return MGR_ERR_ARGUMENT;
    if (ctx->S > 1) return ctx->fail(MGR_ERR_UNSUPPORTED, "the warm-start features are defined for one line-producing species");
    MGR_HIP(hipSetDevice(ctx->device));
    float *dX = nullptr;
    MGR_HIP(mgr::device_malloc(&dX, ctx->N * IN * sizeof(float)));
    int rc = mgr::launch_features(ctx, dX, ctx->J_set);   // before any radiation field the J inputs are 0
    if (!rc && (hipStreamSynchronize(ctx->stream) != hipSuccess ||
                hipMemcpy(X, dX, ctx->N * IN * sizeof(float), hipMemcpyDeviceToHost) != hipSuccess))
        rc = ctx->fail(MGR_ERR_DEVICE, "features copy failed");
    (void)hipFree(dX);
    return rc;
}

extern "C" int mgr_warm_start(mgr_ctx *ctx, mgr_mlp *mlp)
{
    if (!ctx || !mlp) return MGR_ERR_ARGUMENT;
    if (ctx->V != OUT || ctx->S > 1)
        return ctx->fail(MGR_ERR_UNSUPPORTED, "the warm-start network predicts the 7 levels of one species");
    if (mlp->jlin_inputs && !ctx->J_set)
        return ctx->fail(MGR_ERR_STATE, "warm start needs a radiation field and J_eff first (the network reads J)");
    if (ctx->device != mlp->device) return ctx->fail(MGR_ERR_ARGUMENT, "context and network on different devices");
    MGR_HIP(hipSetDevice(ctx->device));
    MGR_HIP(hipStreamSynchronize(mlp->stream));
    ctx->warm_fallbacks = 0;
    float *dX = nullptr;
    double *dPrev = nullptr;
    unsigned long long *dCount = nullptr;
    const size_t npop = (size_t)ctx->N * OUT;
    if (mgr::device_malloc(&dX, ctx->N * IN * sizeof(float)) != hipSuccess ||
        mgr::device_malloc(&dPrev, npop * sizeof(double)) != hipSuccess ||
        mgr::device_malloc(&dCount, sizeof(unsigned long long)) != hipSuccess) {
        (void)hipFree(dX);
        (void)hipFree(dPrev);
        return ctx->fail(MGR_ERR_NOMEM, "warm start: device allocation failed");
    }
    int rc = mgr::launch_features(ctx, dX, mlp->jlin_inputs);
    if (!rc && (hipMemcpyAsync(dPrev, ctx->pop, npop * sizeof(double), hipMemcpyDeviceToDevice, ctx->stream) != hipSuccess ||
                hipMemsetAsync(dCount, 0, sizeof(unsigned long long), ctx->stream) != hipSuccess))
        rc = ctx->fail(MGR_ERR_DEVICE, "warm start: copy failed");
    if (!rc) {
        hipLaunchKernelGGL(k_mlp_forward, dim3(grid_for_rows(ctx->N, 1024)), dim3(THREADS), LDS_FORWARD, ctx->stream, dX,
                           ctx->N, mlp->wbf, mlp->P, mlp->norm, (float *)nullptr, ctx->pop_tot, ctx->pop);
        hipLaunchKernelGGL(k_warm_guard, dim3((unsigned)((ctx->N + 255) / 256)), dim3(256), 0, ctx->stream, ctx->N,
                           (int)OUT, (int)ctx->L, ctx->irad, ctx->jrad, ctx->Ba, ctx->Bs, dPrev, ctx->pop, dCount,
                           ctx->near_bad);
        if (hipGetLastError() != hipSuccess) rc = ctx->fail(MGR_ERR_DEVICE, "warm-start launch failed");
    }
    if (!rc) rc = launch_emissivity_opacity(ctx);
    unsigned long long nfb = 0;
    if (!rc && (hipMemcpyAsync(&nfb, dCount, sizeof(nfb), hipMemcpyDeviceToHost, ctx->stream) != hipSuccess ||
                hipStreamSynchronize(ctx->stream) != hipSuccess))
        rc = ctx->fail(MGR_ERR_DEVICE, "warm start failed");
    (void)hipFree(dX);
    (void)hipFree(dPrev);
    (void)hipFree(dCount);
    if (!rc) {
        ctx->warm_fallbacks = (int64_t)nfb;
        ctx->pops_set = true;
    }
    return rc;
}

extern "C" int mgr_mlp_set_jlin_inputs(mgr_mlp *mlp, int use)
{
    if (!mlp) return MGR_ERR_ARGUMENT;
    mlp->jlin_inputs = use != 0;
    return MGR_OK;
}

extern "C" int mgr_warm_start_fallbacks(const mgr_ctx *ctx, int64_t *cells)
{
    if (!ctx || !cells) return MGR_ERR_ARGUMENT;
    *cells = ctx->warm_fallbacks;
    return MGR_OK;
}
