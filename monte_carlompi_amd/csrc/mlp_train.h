// mlp_train.h -- training step of 256-wide networks: forward, loss and backward of a row block in one kernel, all
// weight gradients in one, Adam with the gradient reduction in one (part of mlp.hip's translation unit)
#pragma once

namespace mlp {

typedef float f32x4 __attribute__((ext_vector_type(4)));

// ---- bf16 weights as MFMA operands.  The 64 lanes' operands of one
// v_mfma_f32_16x16x32_bf16 (16 outputs x 32 inputs: lane l holds output l % 16,
// inputs 8 (l / 16) .. + 8) are 1 KB in a row, so a wave's operand load is one
// contiguous read instead of 16 or 32 rows' pieces.  tile_pos: place of element
// (o, i) of an operand matrix with `in` inputs (a multiple of 32).
__host__ __device__ __forceinline__ size_t tile_pos(int o, int i, int in)
{
    return ((size_t)((o >> 4) * (in >> 5) + (i >> 5)) << 9) + (size_t)((((i & 31) >> 3) * 16 + (o & 15)) * 8 + (i & 7));
}

constexpr int TR_ROWS = 16, TR_WAVES = 8, TR_H = 256;
constexpr int TR_MAX_LAYERS = 8, TR_MAX_NP = 1024, TR_TILES = TR_MAX_NP / (16 * TR_WAVES);
constexpr int LD_PAD = 64;   // between the rows of the transposed arrays (no power-of-two stride)
constexpr int TR_PITCH = TR_H + 8, TR_PITCH_Y = TR_MAX_NP + 8, TR_PITCH_X = K0 + 8;
static_assert(TR_H / 32 == TR_WAVES, "two 16-column tiles of a hidden layer per wave");

struct TrainArgs {
    const float *x, *t;         // dataset [n][n_in], [n][n_out]
    const int32_t *idx;         // rows of the batch (null: 0, 1, ...)
    int64_t n_data;
    int n_in, n_out, np, batch;
    int ld;                     // batch elements between the rows of the transposed arrays below
    const float *p, *w;         // parameters (biases at boff[l]); output weights, zero beyond n_out
    const bf16 *wf, *wt;        // weights by tile_pos: (output, input), and (input, output)
    size_t woff[TR_MAX_LAYERS + 1], boff[TR_MAX_LAYERS + 1];
    bf16 *xt;                   // [K0][ld] inputs
    bf16 *at[TR_MAX_LAYERS];    // [H][ld] activations of layer l
    bf16 *dzt[TR_MAX_LAYERS];   // [H][ld] loss gradient at layer l's pre-activations
    bf16 *dyt;                  // [np][ld] ... at the outputs
    float *lpart;               // per block: sum w (y - t)^2
};

// Workgroups go to the 8 XCDs, each with its own L2, round-robin by id: block
// `b` of `n` takes the place that gives each XCD one contiguous run.
__device__ __forceinline__ int xcd_run(int b, int n)
{
    const int x = b & 7, q = n >> 3, r = n & 7;
    return x * q + min(x, r) + (b >> 3);
}

__device__ __forceinline__ bf16x8 tile_load(const bf16 *W, int tile, int lane)
{
    return *reinterpret_cast<const bf16x8 *>(W + ((size_t)tile << 9) + lane * 8);
}

// a wave's two column tiles of a hidden layer, K = 32 KT inputs, from LDS rows
template <int KT>
__device__ __forceinline__ void tr_mma(f32x4 (&acc)[2], const bf16 *rows, int pitch, const bf16x8 (&w)[2][KT], int lane)
{
    const bf16 *a = rows + (lane & 15) * pitch + (lane >> 4) * 8;
#pragma unroll
    for (int k = 0; k < KT; ++k) {
        const bf16x8 v = *reinterpret_cast<const bf16x8 *>(a + k * 32);
        acc[0] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(v, w[0][k], acc[0], 0, 0, 0);
        acc[1] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(v, w[1][k], acc[1], 0, 0, 0);
    }
}

// store a tile's values v (rows 4 (lane / 16) .. + 4 of column col): bf16 into LDS rows and, transposed, to HBM
__device__ __forceinline__ void tr_store(const float (&v)[4], int col, bf16 *rows, int pitch, bf16 *tr, int ld, int r0,
                                         int lane)
{
    bf16x4 o;
    const int q = (lane >> 4) * 4;
#pragma unroll
    for (int r = 0; r < 4; ++r) {
        o[r] = (bf16)v[r];
        rows[(q + r) * pitch + col] = o[r];
    }
    *reinterpret_cast<bf16x4 *>(tr + (size_t)col * ld + r0 + q) = o;
}

// Forward, loss and backward of TR_ROWS batch rows: inputs gathered from the
// dataset; activations and pre-activation gradients pass from layer to layer
// through LDS in bf16, the pre-activations of every layer stay in the registers
// of the lane that will need them (FP32, the accumulator's layout, since dA's
// tiles are the layer's own), and the outputs are never stored: each wave turns
// its output tiles into loss and dY at once.  What the weight gradients need
// (inputs, activations, gradients) is written transposed, [feature][row], for
// k_train_dw to read along the batch.  16-row blocks put a batch of 4096 on
// all 256 CUs.  What bounds it: the step's weights (2 x 0.75 MB for the
// surrogate) stream from L2 through every CU at 64 B a cycle, ~10 us for 32
// rows as for 16 (a layer's operands are requested once the layer before is
// multiplied; two sets of them, kept two layers ahead, spilled and took 36 us
// instead of 27), and the transposed stores are 22 MB a step (5 us).
template <int L>
__global__ void __launch_bounds__(TR_WAVES * 64) __attribute__((amdgpu_waves_per_eu(2))) k_train_rows(const TrainArgs g)
{
    __shared__ __attribute__((aligned(16))) bf16 X0[TR_ROWS * TR_PITCH_X];
    __shared__ __attribute__((aligned(16))) bf16 Act[2][TR_ROWS * TR_PITCH];
    __shared__ __attribute__((aligned(16))) bf16 dY[TR_ROWS * TR_PITCH_Y];
    __shared__ float red[TR_WAVES];
    const int t = threadIdx.x, lane = t & 63, wave = t >> 6, l16 = lane & 15, q = (lane >> 4) * 4;
    const int rb = xcd_run(blockIdx.x, gridDim.x), r0 = rb * TR_ROWS;
    const auto source = [&](int r) {
        const int64_t s = g.idx ? g.idx[r0 + r] : r0 + r;
        return s < 0 || s >= g.n_data ? (int64_t)0 : s;
    };
    const int64_t xrow = source(l16);
    int64_t trow[4];
#pragma unroll
    for (int r = 0; r < 4; ++r) trow[r] = source(q + r);
    bf16x8 w0[2][1], w[2][8];
#pragma unroll
    for (int j = 0; j < 2; ++j) w0[j][0] = tile_load(g.wf + g.woff[0], wave * 2 + j, lane);
    const auto request = [&](const bf16 *W) {             // a 256-input layer's operands
#pragma unroll
        for (int j = 0; j < 2; ++j)
#pragma unroll
            for (int k = 0; k < 8; ++k) w[j][k] = tile_load(W, (wave * 2 + j) * 8 + k, lane);
    };
    if (L > 1) request(g.wf + g.woff[1]);
    {
        const int c = t >> 4;                             // one input per thread, row t % 16
        const bf16 v = (bf16)(c < g.n_in ? g.x[xrow * g.n_in + c] : 0.f);
        X0[l16 * TR_PITCH_X + c] = v;
        g.xt[(size_t)c * g.ld + r0 + l16] = v;
    }
    // the targets of the wave's output tiles, wave + 8 i: they come from HBM
    const int tiles = g.np >> 4;
    float tv[TR_TILES][4];
#pragma unroll
    for (int i = 0; i < TR_TILES; ++i) {
        const int c = (wave + TR_WAVES * i) * 16 + l16;
#pragma unroll
        for (int r = 0; r < 4; ++r) tv[i][r] = c < g.n_out ? g.t[trow[r] * g.n_out + c] : 0.f;
    }
    __syncthreads();
    const int col0 = wave * 32 + l16;
    float zs[L][2][4];                                    // pre-activations
#pragma unroll
    for (int l = 0; l < L; ++l) {
        f32x4 acc[2] = {};
        if (l == 0) {
            tr_mma<1>(acc, X0, TR_PITCH_X, w0, lane);
        } else {
            tr_mma<8>(acc, Act[(l - 1) & 1], TR_PITCH, w, lane);
            if (l + 1 < L) request(g.wf + g.woff[l + 1]);
        }
#pragma unroll
        for (int j = 0; j < 2; ++j) {
            const float b = g.p[g.boff[l] + col0 + 16 * j];
            float a[4];
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const float z = acc[j][r] + b;
                a[r] = z * sigm(z);
                zs[l][j][r] = z;
            }
            tr_store(a, col0 + 16 * j, Act[l & 1], TR_PITCH, g.at[l], g.ld, r0, lane);
        }
        __syncthreads();
    }
    // ---- outputs: loss and dY
    float lacc = 0.f;
    {
        const float inv = 1.f / g.batch;
        const bf16 *W = g.wf + g.woff[L];
        const float *bias = g.p + g.boff[L];
        const bf16 *a = Act[(L - 1) & 1] + l16 * TR_PITCH + (lane >> 4) * 8;
        bf16x8 av[8];
#pragma unroll
        for (int k = 0; k < 8; ++k) av[k] = *reinterpret_cast<const bf16x8 *>(a + k * 32);
        bf16x8 u[2][8];                                   // a tile's operands, two tiles ahead
        const auto ask = [&](int i) {
            const int nt = min(wave + TR_WAVES * i, tiles - 1);
#pragma unroll
            for (int k = 0; k < 8; ++k) u[i & 1][k] = tile_load(W, nt * 8 + k, lane);
        };
        ask(0);
        ask(1);
#pragma unroll
        for (int i = 0; i < TR_TILES; ++i) {
            const int nt = wave + TR_WAVES * i;
            if (nt >= tiles) break;
            f32x4 acc = {};
#pragma unroll
            for (int k = 0; k < 8; ++k) acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(av[k], u[i & 1][k], acc, 0, 0, 0);
            if (i + 2 < TR_TILES) ask(i + 2);
            const int c = nt * 16 + l16;
            const float b = c < g.n_out ? bias[c] : 0.f, wc = g.w[c];
            float d[4];
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const float e = acc[r] + b - tv[i][r];
                lacc += wc * e * e;
                d[r] = 2.f * wc * e * inv;
            }
            tr_store(d, c, dY, TR_PITCH_Y, g.dyt, g.ld, r0, lane);
        }
    }
#pragma unroll
    for (int h = 32; h > 0; h >>= 1) lacc += __shfl_xor(lacc, h, 64);
    if (lane == 0) red[wave] = lacc;
    // ---- backward: dA = dZ W, dZ = dA SiLU'
    const bf16 *WT = g.wt + g.woff[L];
    const int nk = g.np >> 5;
    // the output layer's operands in groups of four steps of 32 outputs, two
    // groups in registers (np / 32 is even: the last group may hold two)
    const auto group = [&](int half, int k) {
#pragma unroll
        for (int j = 0; j < 2; ++j)
#pragma unroll
            for (int m = 0; m < 4; ++m)
                w[j][half * 4 + m] = tile_load(WT, (wave * 2 + j) * nk + min(k + m, nk - 1), lane);
    };
    group(0, 0);
    group(1, 4);
    __syncthreads();
    if (t == 0) {
        float s = 0.f;
        for (int k = 0; k < TR_WAVES; ++k) s += red[k];
        g.lpart[rb] = s;
    }
#pragma unroll
    for (int l = L - 1; l >= 0; --l) {
        f32x4 acc[2] = {};
        if (l == L - 1) {
            const bf16 *a = dY + l16 * TR_PITCH_Y + (lane >> 4) * 8;
            const auto use = [&](int half, int k) {
#pragma unroll
                for (int m = 0; m < 4; m += 2) {
                    if (k + m >= nk) break;
                    const bf16x8 v0 = *reinterpret_cast<const bf16x8 *>(a + (k + m) * 32);
                    const bf16x8 v1 = *reinterpret_cast<const bf16x8 *>(a + (k + m) * 32 + 32);
#pragma unroll
                    for (int j = 0; j < 2; ++j) {
                        acc[j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(v0, w[j][half * 4 + m], acc[j], 0, 0, 0);
                        acc[j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(v1, w[j][half * 4 + m + 1], acc[j], 0, 0, 0);
                    }
                }
                group(half, k + 8);
            };
            for (int k = 0; k < nk; k += 8) {
                use(0, k);
                use(1, k + 4);
            }
        } else {
            tr_mma<8>(acc, Act[(l + 1) & 1], TR_PITCH, w, lane);
        }
        if (l > 0) request(g.wt + g.woff[l]);
#pragma unroll
        for (int j = 0; j < 2; ++j) {
            float d[4];
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const float z = zs[l][j][r], s = sigm(z);
                d[r] = acc[j][r] * s * (1.f + z * (1.f - s));
            }
            tr_store(d, col0 + 16 * j, Act[l & 1], TR_PITCH, g.dzt[l], g.ld, r0, lane);
        }
        if (l > 0) __syncthreads();
    }
}

// Weight and bias gradients of every layer: dW_l = dZ_l^T A_{l-1} summed over
// the batch, both operands [feature][row] (k_train_rows), so tiles load along
// the batch.  64 x 64 tiles of all layers in one launch (96 for the surrogate).
// The addends of a weight's sum are those of the per-layer kernels: chunks of
// kc rows (split_k, another for each layer; the surrogate's at batch 4096: 32,
// 128, 352), each one chain of MFMAs from zero.  A block adds the chunks of its
// slice of the batch (dw_slices), one array of the padded parameter layout per
// slice; k_train_adam / k_train_reduce add the slices in FP64 (no atomics, no
// zeroing; the same result every time, and with two chunks the per-layer
// kernels' bit for bit).  A layer's blocks go over the XCDs by slice (xcd_run):
// with eight slices every XCD's L2 reads one (2.8 of the surrogate's 22 MB)
// instead of all, the one whose rows k_train_rows wrote there.  A chunk is staged 64
// rows at a time through two LDS buffers (32 and zeros at its end).  The tiles of
// a layer's first input column block also sum their gradient rows: the biases.
constexpr int DW_P = 64 + 8, DW_SLICES = 16;
struct DwArgs {
    int L, batch, ld;
    size_t n_pad;
    int block0[TR_MAX_LAYERS + 2];         // first block of layer l
    int chunks[TR_MAX_LAYERS + 1], kc[TR_MAX_LAYERS + 1], slices[TR_MAX_LAYERS + 1];
    int mtiles[TR_MAX_LAYERS + 1], cols[TR_MAX_LAYERS + 1];
    const bf16 *dz[TR_MAX_LAYERS + 1], *in[TR_MAX_LAYERS + 1];
    size_t woff[TR_MAX_LAYERS + 1], boff[TR_MAX_LAYERS + 1];
    float *part;
};

__global__ void __launch_bounds__(256) k_train_dw(const DwArgs g)
{
    __shared__ __attribute__((aligned(16))) bf16 As[2][64 * DW_P];
    __shared__ __attribute__((aligned(16))) bf16 Bs[2][64 * DW_P];
    int l = 0;
    while ((int)blockIdx.x >= g.block0[l + 1]) ++l;
    const int slices = g.slices[l], chunks = g.chunks[l], kc = g.kc[l], blocks = g.block0[l + 1] - g.block0[l];
    const int at = xcd_run(blockIdx.x - g.block0[l], blocks), tiles = blocks / slices, slice = at / tiles, tile = at % tiles;
    const int m0 = (tile % g.mtiles[l]) * 64, n0 = (tile / g.mtiles[l]) * 64;
    const int cols = g.cols[l];
    const int t = threadIdx.x, lane = t & 63, wave = t >> 6, wm = wave >> 1, wn = wave & 1;
    const int kb = slice * chunks / slices * kc, ke = min(g.batch, (slice + 1) * chunks / slices * kc);
    // each thread moves 2 x 16 B of either operand per stage: rows t / 8 and + 32
    const int lr = t >> 3, lk = (t & 7) * 8;
    const bf16 *A = g.dz[l] + (size_t)(m0 + lr) * g.ld + lk;
    const size_t half = (size_t)32 * g.ld;
    const bf16 *B = g.in[l] + (size_t)(n0 + lr) * g.ld + lk;
    const bf16 *B1 = n0 + lr + 32 < cols ? B + half : B;   // (columns past the input's are not stored)
    const bf16 *A1 = A + half;
    bf16x8 ra0 = *reinterpret_cast<const bf16x8 *>(A + kb), ra1 = *reinterpret_cast<const bf16x8 *>(A1 + kb);
    bf16x8 rb0 = *reinterpret_cast<const bf16x8 *>(B + kb), rb1 = *reinterpret_cast<const bf16x8 *>(B1 + kb);
    bf16 *const sa = &As[0][lr * DW_P + lk], *const sb = &Bs[0][lr * DW_P + lk];
    double bs0 = 0.0, bs1 = 0.0;
    const bool bias = n0 == 0;
    f32x16 acc = {}, sum = {};
    for (int k = kb, ce = min(ke, kb + kc), buf = 0;; buf ^= 1) {   // ce: the chunk's end
        // stage k's rows; this buffer was read last before the barrier of the turn between
        const int rows = ce - k;           // 32 left of the chunk (a multiple of 32): the others as zeros
        if (rows < 64 && lk >= rows) ra0 = ra1 = rb0 = rb1 = bf16x8{};
        const int o = buf * 64 * DW_P;
        *reinterpret_cast<bf16x8 *>(sa + o) = ra0;
        *reinterpret_cast<bf16x8 *>(sa + o + 32 * DW_P) = ra1;
        *reinterpret_cast<bf16x8 *>(sb + o) = rb0;
        *reinterpret_cast<bf16x8 *>(sb + o + 32 * DW_P) = rb1;
        if (bias) {
            float s0 = 0.f, s1 = 0.f;
#pragma unroll
            for (int j = 0; j < 8; ++j) {
                s0 += (float)ra0[j];
                s1 += (float)ra1[j];
            }
            bs0 += (double)s0;
            bs1 += (double)s1;
        }
        const int kn = min(k + 64, ce);
        const bool more = kn < ke;
        {
            // (rows past the chunk's or the batch's end may be among them: the next
            // chunk's or the arrays' pad)
            const int kl = more ? kn : k;
            ra0 = *reinterpret_cast<const bf16x8 *>(A + kl);
            ra1 = *reinterpret_cast<const bf16x8 *>(A1 + kl);
            rb0 = *reinterpret_cast<const bf16x8 *>(B + kl);
            rb1 = *reinterpret_cast<const bf16x8 *>(B1 + kl);
        }
        __syncthreads();
        const bf16 *a = &As[buf][(wm * 32 + (lane & 31)) * DW_P + (lane >> 5) * 8];
        const bf16 *b = &Bs[buf][(wn * 32 + (lane & 31)) * DW_P + (lane >> 5) * 8];
#pragma unroll
        for (int s = 0; s < 4; ++s)
            acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(*reinterpret_cast<const bf16x8 *>(a + 16 * s),
                                                          *reinterpret_cast<const bf16x8 *>(b + 16 * s), acc, 0, 0, 0);
        if (kn == ce) {                    // the chunk is complete
            sum += acc;
            acc = f32x16{};
            ce = min(ke, ce + kc);
        }
        if (!more) break;
        k = kn;
    }
    float *out = g.part + (size_t)slice * g.n_pad;
    const int n = n0 + wn * 32 + (lane & 31);
    if (n < cols) {
        float *o = out + g.woff[l] + n;
#pragma unroll
        for (int r = 0; r < 16; ++r)
            o[(size_t)(m0 + wm * 32 + (r >> 2) * 8 + (lane >> 5) * 4 + (r & 3)) * cols] = sum[r];
    }
    if (bias) {
#pragma unroll
        for (int d = 1; d < 8; d <<= 1) {
            bs0 += __shfl_xor(bs0, d, 64);
            bs1 += __shfl_xor(bs1, d, 64);
        }
        if ((t & 7) == 0) {
            out[g.boff[l] + m0 + lr] = (float)bs0;
            out[g.boff[l] + m0 + lr + 32] = (float)bs1;
        }
    }
}

// Padded parameter layout, for kernels that go over all parameters: layer of
// index i, whether it is a weight (row, column) and not padding.
struct ParamMap {
    int L;
    size_t n_pad;
    size_t woff[TR_MAX_LAYERS + 1], boff[TR_MAX_LAYERS + 1], wboff[TR_MAX_LAYERS + 1];
    int rows[TR_MAX_LAYERS + 1], cols[TR_MAX_LAYERS + 1], prow[TR_MAX_LAYERS + 1], lgcol[TR_MAX_LAYERS + 1];
};
struct ParamAt {
    int l, r, c;
    bool weight, real;
};
__device__ __forceinline__ ParamAt param_at(const ParamMap &m, size_t i)
{
    ParamAt a;
    a.l = 0;
    while (a.l < m.L && i >= m.woff[a.l + 1]) ++a.l;
    a.weight = i < m.boff[a.l];
    if (a.weight) {
        const uint32_t k = (uint32_t)(i - m.woff[a.l]);
        a.r = (int)(k >> m.lgcol[a.l]);
        a.c = (int)(k & ((1u << m.lgcol[a.l]) - 1u));
        a.real = a.r < m.rows[a.l] && a.c < m.cols[a.l];
    } else {
        a.r = (int)(i - m.boff[a.l]);
        a.c = 0;
        a.real = a.r < m.rows[a.l];
    }
    return a;
}

// the bf16 operand copies of the weights: by tile_pos both ways round
__device__ __forceinline__ void put_tiles(const ParamMap &m, const ParamAt &a, float v, bf16 *wf, bf16 *wt)
{
    wf[m.wboff[a.l] + tile_pos(a.r, a.c, 1 << m.lgcol[a.l])] = (bf16)v;
    wt[m.wboff[a.l] + tile_pos(a.c, a.r, m.prow[a.l])] = (bf16)v;
}

// *loss = sum of the row blocks' parts / rows (one block of 256)
__device__ __forceinline__ void loss_of(const float *lpart, int nb, int rows, float *loss)
{
    __shared__ float red[256];
    float s = 0.f;
    for (int b = threadIdx.x; b < nb; b += 256) s += lpart[b];
    red[threadIdx.x] = s;
    __syncthreads();
    for (int h = 128; h > 0; h >>= 1) {
        if ((int)threadIdx.x < h) red[threadIdx.x] += red[threadIdx.x + h];
        __syncthreads();
    }
    if (threadIdx.x == 0) *loss = red[0] / rows;
}

// The slices' partial sums (k_train_dw)
struct GradParts {
    const float *part;                     // [slice][n_pad]
    int slices[TR_MAX_LAYERS + 1];
};
__device__ __forceinline__ float grad_sum(const GradParts &gp, size_t n_pad, int l, size_t i)
{
    double g = 0.0;
#pragma unroll 4
    for (int s = 0; s < gp.slices[l]; ++s) g += (double)gp.part[(size_t)s * n_pad + i];
    return (float)g;
}

// Gradient = sum of the slices' partial sums, then Adam (decoupled weight
// decay) on the FP32 parameters and the bf16 operand copies.  A block takes a
// 32 x 32 patch of a layer's weights, four columns per thread, and turns it in
// LDS so that both copies are written in whole 16-byte pieces (2-byte stores of
// the transposed copy: 8.8 us a step for the surrogate); blocks past the
// patches take 256 biases each.  The first block also writes the step's loss.
struct AdamArgs {
    ParamMap m;
    int patch0[TR_MAX_LAYERS + 2];         // first patch of layer l; [L + 1]: number of patches
    int bias0[TR_MAX_LAYERS + 2];          // first bias block of layer l
    GradParts g;
    float *p, *mo, *vo;
    AdamCoef c;
    bf16 *wf, *wt;
    const float *lpart;
    int nb, rows;
    float *loss;
};

__global__ void __launch_bounds__(256) k_train_adam(const AdamArgs a)
{
    __shared__ __attribute__((aligned(16))) bf16 patch[32][32 + 8];
    if (blockIdx.x == 0) loss_of(a.lpart, a.nb, a.rows, a.loss);
    const ParamMap &m = a.m;
    const int t = threadIdx.x, b = blockIdx.x;
    int l = 0;
    if (b >= a.patch0[m.L + 1]) {
        const int k = b - a.patch0[m.L + 1];
        while (k >= a.bias0[l + 1]) ++l;
        const int r = (k - a.bias0[l]) * 256 + t;
        if (r >= m.rows[l]) return;
        const size_t i = m.boff[l] + r;
        const float g = grad_sum(a.g, m.n_pad, l, i);
        float p = a.p[i], mi = a.mo[i], vi = a.vo[i];
        adam_step(a.c, g, p, mi, vi);
        a.p[i] = p; a.mo[i] = mi; a.vo[i] = vi;
        return;
    }
    while (b >= a.patch0[l + 1]) ++l;
    const int lg = m.lgcol[l] - 5;                        // column patches: 2^lg
    const int k = b - a.patch0[l], pr = k >> lg, pc = k & ((1 << lg) - 1);
    const int r = t >> 3, c = (t & 7) * 4;                // this thread's row and columns of the patch
    const int row = pr * 32 + r, col = pc * 32 + c;
    const size_t i = m.woff[l] + ((size_t)row << m.lgcol[l]) + col;
    double gx = 0.0, gy = 0.0, gz = 0.0, gw = 0.0;
#pragma unroll 4
    for (int s = 0; s < a.g.slices[l]; ++s) {
        const float4 d = *reinterpret_cast<const float4 *>(a.g.part + (size_t)s * m.n_pad + i);
        gx += (double)d.x; gy += (double)d.y; gz += (double)d.z; gw += (double)d.w;
    }
    const float4 g = make_float4((float)gx, (float)gy, (float)gz, (float)gw);
    float4 p = *reinterpret_cast<float4 *>(a.p + i), mi = *reinterpret_cast<float4 *>(a.mo + i),
           vi = *reinterpret_cast<float4 *>(a.vo + i);
    // padding rows and columns stay zero
    const bool in = row < m.rows[l];
    if (in && col < m.cols[l]) adam_step(a.c, g.x, p.x, mi.x, vi.x);
    if (in && col + 1 < m.cols[l]) adam_step(a.c, g.y, p.y, mi.y, vi.y);
    if (in && col + 2 < m.cols[l]) adam_step(a.c, g.z, p.z, mi.z, vi.z);
    if (in && col + 3 < m.cols[l]) adam_step(a.c, g.w, p.w, mi.w, vi.w);
    *reinterpret_cast<float4 *>(a.p + i) = p;
    *reinterpret_cast<float4 *>(a.mo + i) = mi;
    *reinterpret_cast<float4 *>(a.vo + i) = vi;
    bf16x4 o;
    o[0] = (bf16)p.x; o[1] = (bf16)p.y; o[2] = (bf16)p.z; o[3] = (bf16)p.w;
    *reinterpret_cast<bf16x4 *>(&patch[r][c]) = o;
    __syncthreads();
    // two 16 x 32 tiles of either copy, 64 pieces of 8 elements each
    const int tile = (t >> 6) & 1, lane = t & 63, u = tile * 16 + (lane & 15), v = (lane >> 4) * 8;
    bf16x8 e;
    if (t < 128) {
        e = *reinterpret_cast<const bf16x8 *>(&patch[u][v]);
        *reinterpret_cast<bf16x8 *>(a.wf + m.wboff[l] + tile_pos(pr * 32 + u, pc * 32 + v, 1 << m.lgcol[l])) = e;
    } else {
#pragma unroll
        for (int j = 0; j < 8; ++j) e[j] = patch[v + j][u];
        *reinterpret_cast<bf16x8 *>(a.wt + m.wboff[l] + tile_pos(pc * 32 + u, pr * 32 + v, m.prow[l])) = e;
    }
}

// gradient array and loss without an update
__global__ void __launch_bounds__(256) k_train_reduce(const ParamMap m, const GradParts gp, float *gr, const float *lpart, int nb, int rows, float *loss)
{
    if (blockIdx.x == 0) loss_of(lpart, nb, rows, loss);
    const size_t i = blockIdx.x * (size_t)256 + threadIdx.x;
    if (i >= m.n_pad) return;
    const ParamAt a = param_at(m, i);
    gr[i] = a.real ? grad_sum(gp, m.n_pad, a.l, i) : 0.f;
}

// the bf16 operand copies of the weights from the FP32 parameters
__global__ void __launch_bounds__(256) k_pack_weights(const ParamMap m, const float *p, bf16 *wf, bf16 *wt)
{
    const size_t i = blockIdx.x * (size_t)256 + threadIdx.x;
    if (i >= m.n_pad) return;
    const ParamAt a = param_at(m, i);
    if (!a.weight) return;
    put_tiles(m, a, p[i], wf, wt);
}

}  // namespace mlp
