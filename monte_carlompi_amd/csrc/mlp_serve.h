// mlp_serve.h -- inference of 256-wide networks: input features, every layer and the output transform in one kernel
// (part of mlp.hip's translation unit)
#pragma once

namespace mlp {

// bf16 weights as operands of v_mfma_f32_32x32x16_bf16: the 64 lanes' operands
// (32 outputs x 16 inputs: lane l holds output l % 32, inputs 8 (l / 32) .. + 8)
// are 1 KB in a row, a 32-output tile's steps one after the other (16 KB for
// 256 inputs).  Place of element (o, i) of a layer with `in` inputs:
__host__ __device__ __forceinline__ size_t serve_pos(int o, int i, int in)
{
    return ((size_t)((o >> 5) * (in >> 4) + (i >> 4)) << 9) + (size_t)((((i & 15) >> 3) * 32 + (o & 31)) * 8 + (i & 7));
}

constexpr int SV_H = 256, SV_WAVES = 8, SV_PITCH = SV_H + 8, SV_PITCH_X = K0 + 8, SV_MAX_LAYERS = 16;
struct ServeArgs {
    const float *x;             // [rows][5 raw case inputs] (snow) or [rows][n_in]
    int64_t rows;
    int snow, n_in, L, n_out, np;
    const float *fmu, *fsd;     // standardisation of the snow features
    const bf16 *w;              // weights by serve_pos, layer l at woff[l]
    const float *p;             // FP32 parameters (biases at boff[l])
    size_t woff[SV_MAX_LAYERS + 1], boff[SV_MAX_LAYERS + 1];
    float *y;                   // [rows][n_out]
    const float *oscale, *oshift, *ooff;   // output transform
};

// RT 32-row tiles per block, eight waves of one 32-column tile of a hidden
// layer each (and every eighth of the output layer), PF steps of 16 inputs of
// weight operands in registers ahead, built for EU waves per SIMD.  Activations
// stay in LDS (one buffer: a layer's tiles are computed into registers and,
// after a barrier, written over its input; the input features share it).
// Weights come from L2 straight into MFMA operands: the register of a step is
// loaded again, PF steps ahead, as soon as its products are issued, over the
// ends of tiles and layers.  Hidden layers multiply weights by activations, so
// that a lane holds four neighbouring features of a row (8-byte LDS writes); the
// output layer the other way round, a lane holding one column (128 contiguous
// bytes of a row per store, through a buffer descriptor: one 32-bit add per
// store).  Operands, k order and epilogues are those of k_gemm_fwd, so the
// results are the same bit for bit.  What bounds a large batch is the stores: 1e6
// rows take 1.27 ms, 0.84 without them (870 TFLOP/s); the answers' rows are
// 2,604 bytes apart, so every store straddles lines, and the operand loads
// behind a tile's stores wait for them.  Tried: 64 columns a wave and two waves
// per SIMD 1.40 ms, 64-row blocks 1.35, 16-byte stores of four columns of 32
// rows 2.1, non-temporal stores 1.7 - 2.5.
template <int RT, int PF, int EU, bool EXP>
__global__ void __launch_bounds__(SV_WAVES * 64) __attribute__((amdgpu_waves_per_eu(EU))) k_mlp_serve(const ServeArgs g)
{
    static_assert(SV_WAVES * 32 == SV_H && 16 % PF == 0, "a hidden tile per wave; the operand ring");
    constexpr int R = RT * 32;
    __shared__ __attribute__((aligned(16))) bf16 Act[R * SV_PITCH];
    const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
    const int64_t r0 = (int64_t)blockIdx.x * R;
    const int tiles = g.np >> 5;
    const auto hidden = [&](int l) { return g.w + g.woff[l] + ((size_t)wave << 13); };
    const auto outer = [&](int nt) { return g.w + g.woff[g.L] + ((size_t)min(nt, tiles - 1) << 13); };
    bf16x8 w[PF];
    const auto fetch = [&](int slot, const bf16 *W, int k) {
        w[slot] = *reinterpret_cast<const bf16x8 *>(W + (k << 9) + lane * 8);
    };
    // layer 0's operands (two steps), then the first of what follows it
    bf16x8 w0[2];
#pragma unroll
    for (int k = 0; k < 2; ++k)
        w0[k] = *reinterpret_cast<const bf16x8 *>(g.w + g.woff[0] + ((size_t)(wave * 2 + k) << 9) + lane * 8);
    {
        const bf16 *W = g.L > 1 ? hidden(1) : outer(wave);
#pragma unroll
        for (int k = 0; k < PF; ++k) fetch(k, W, k);
    }
    // ---- input rows (zero past the last) into Act, pitch SV_PITCH_X
    if (g.snow) {
        constexpr int SUBS = SV_WAVES * 64 / R;              // threads per row, each every SUBS-th feature
        const int row = t % R, sub = t / R;
        const bool in = r0 + row < g.rows;
        const float *q = g.x + (in ? r0 + row : 0) * 5;
        const SnowInputs s = snow_inputs(q);
        for (int k = sub; k < K0; k += SUBS)
            Act[row * SV_PITCH_X + k] = k < SNOW_FEATURES && in ? snow_feature(s, k, g.fmu, g.fsd) : (bf16)0.f;
    } else {
        for (int i = t; i < R * K0; i += SV_WAVES * 64) {
            const int row = i / K0, c = i % K0;
            const bool in = r0 + row < g.rows && c < g.n_in;
            Act[row * SV_PITCH_X + c] = (bf16)(in ? g.x[(r0 + row) * g.n_in + c] : 0.f);
        }
    }
    __syncthreads();
    const int l32 = lane & 31, hi = lane >> 5;
    const bf16 *const a0 = Act + l32 * SV_PITCH + hi * 8;
    // ---- hidden layers
    for (int l = 0; l < g.L; ++l) {
        f32x16 acc[RT] = {};
        if (l == 0) {
#pragma unroll
            for (int k = 0; k < 2; ++k)
#pragma unroll
                for (int i = 0; i < RT; ++i) {
                    const bf16x8 a = *reinterpret_cast<const bf16x8 *>(Act + (i * 32 + l32) * SV_PITCH_X + k * 16 + hi * 8);
                    acc[i] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(w0[k], a, acc[i], 0, 0, 0);
                }
        } else {
            const bf16 *W = hidden(l), *next = l + 1 < g.L ? hidden(l + 1) : outer(wave);
            // (turns of PF steps: unrolled whole, the compiler reads all of the
            // layer's rows ahead and spills)
#pragma unroll 1
            for (int kb = 0; kb < 16; kb += PF) {
                const bf16 *ahead = kb + PF < 16 ? W + ((kb + PF) << 9) : next;
#pragma unroll
                for (int k = 0; k < PF; ++k) {
#pragma unroll
                    for (int i = 0; i < RT; ++i) {
                        const bf16x8 a = *reinterpret_cast<const bf16x8 *>(a0 + i * 32 * SV_PITCH + (kb + k) * 16);
                        acc[i] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(w[k], a, acc[i], 0, 0, 0);
                    }
                    fetch(k, ahead, k);
                }
            }
        }
        __syncthreads();   // every wave has read this layer's input
        const float *bias = g.p + g.boff[l] + wave * 32 + hi * 4;
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            const float4 b = *reinterpret_cast<const float4 *>(bias + q * 8);
            const float bv[4] = {b.x, b.y, b.z, b.w};
#pragma unroll
            for (int i = 0; i < RT; ++i) {
                bf16x4 o;
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    const float v = acc[i][q * 4 + r] + bv[r];
                    o[r] = (bf16)(v * sigm(v));
                }
                *reinterpret_cast<bf16x4 *>(Act + (i * 32 + l32) * SV_PITCH + wave * 32 + q * 8 + hi * 4) = o;
            }
        }
        __syncthreads();
    }
    // ---- output layer
    const float *bias = g.p + g.boff[g.L];
    const int left = (int)min<int64_t>(R, g.rows - r0);
    const uint32_t row1 = (uint32_t)g.n_out * 4u, row5 = row1 * 5u;
    const auto ybuf = __builtin_amdgcn_make_buffer_rsrc(g.y + (size_t)r0 * g.n_out, 0, left * (int)row1, 0x00027000);
    for (int nt = wave; nt < tiles; nt += SV_WAVES) {
        f32x16 acc[RT] = {};
        const bf16 *W = outer(nt), *next = outer(nt + SV_WAVES);
#pragma unroll 1
        for (int kb = 0; kb < 16; kb += PF) {
            const bf16 *ahead = kb + PF < 16 ? W + ((kb + PF) << 9) : next;
#pragma unroll
            for (int k = 0; k < PF; ++k) {
#pragma unroll
                for (int i = 0; i < RT; ++i) {
                    const bf16x8 a = *reinterpret_cast<const bf16x8 *>(a0 + i * 32 * SV_PITCH + (kb + k) * 16);
                    acc[i] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, w[k], acc[i], 0, 0, 0);
                }
                fetch(k, ahead, k);
            }
        }
        const int n = nt * 32 + l32;
        if (n >= g.n_out) continue;
        const float b = bias[n];
        float osc = 1.f, osh = 0.f, oof = 0.f;
        if (EXP) { osc = g.oscale[n]; osh = g.oshift[n]; oof = g.ooff[n]; }
        // rows 8 q + 4 (lane / 32) + r of a tile; the buffer ends with the last
        // row, so stores past it are dropped
        uint32_t off = (uint32_t)(hi * 4 * g.n_out + n) * 4u;
#pragma unroll
        for (int i = 0; i < RT; ++i)
#pragma unroll
            for (int r = 0; r < 16; ++r) {
                const float v = acc[i][r] + b;
                const float o = EXP ? __builtin_amdgcn_exp2f(fmaf(osc, v, osh)) - oof : v;
                __builtin_amdgcn_raw_buffer_store_b32(__float_as_uint(o), ybuf, off, 0, 0);
                off += (r & 3) == 3 ? row5 : row1;
            }
    }
}

// weights by serve_pos from the FP32 parameters
struct ServePack {
    int L;
    size_t poff[SV_MAX_LAYERS + 1], woff[SV_MAX_LAYERS + 1];
    int prow[SV_MAX_LAYERS + 1], lgcol[SV_MAX_LAYERS + 1];
    int block0[SV_MAX_LAYERS + 2];
};
__global__ void __launch_bounds__(256) k_pack_serve(const ServePack s, const float *p, bf16 *w)
{
    int l = 0;
    while ((int)blockIdx.x >= s.block0[l + 1]) ++l;
    const int i = (blockIdx.x - s.block0[l]) * 256 + threadIdx.x;   // prow * pcol is a multiple of 256
    const int r = i >> s.lgcol[l], c = i & ((1 << s.lgcol[l]) - 1);
    w[s.woff[l] + serve_pos(r, c, 1 << s.lgcol[l])] = (bf16)p[s.poff[l] + i];
}

}  // namespace mlp
