// An encoder layer of the speaker-embedding models (models/PCF_NATransformer.py:228-265, models/MFA_NATransformer.py:
// 224-261) in training, forward and backward, on token-major activations: batch norms with batch statistics, projections,
// GELU, residuals and weight gradients around the attention kernels.
//
// A layer of 128 x 100 tokens, 256 channels, fp16, forward and backward: 24 launches of 225 us together and 38 us of torch's
// statistics, where the modules took some 80 launches and 800 us (torch's batch norm with its copies, bias gradients as
// reductions of their own, weight gradients through 16-bit sums of chunks).  The pooling behind the layers has its backward
// here too.  Everything else than the batch statistics is launched from native code, so the
// host keeps ahead.  The forward rounds where the modules round and is theirs to the bit wherever the library sums a product in
// the order of its inputs (at 3 x 50 tokens it does not: 1 to 3 of 38400 values differ): training amplifies a difference
// anywhere in it, by way of the rounding of sixteen layers, to what 16 bits give (1.2e-3 of the embeddings, 3 % of the
// gradients).  The backward's gradients are within 4e-4 of the modules', and nearer to 64 bits than they are.
#include "na1d_encoder.h"

namespace na1d {
namespace train {

using namespace enc;

// =============================================================================
// Batch norm over the rows of [M, C]
// =============================================================================
// The sums of the forward are torch's (batch_norm_update_stats on [N, C, T]), to the bit.
// What uses the statistics, and the backward, is bound by memory: a pass over 12800 x 256 16-bit values is 6.5 MB.  A
// workgroup takes 64 channels (whole 128-byte lines) of a chunk of rows; in the backward there are up to 64 chunks, and the kernel that uses the
// sums adds them up itself (from L2) instead of waiting for a third launch, with 16 waves, since with few its workgroups are one to a CU
// (8.9 -> 7.5 us; more workgroups read the sums more often: 9.7).  The forward, which reads none, has up to 256 chunks (6.0 -> 4.8).
// 12800 x 256 backward, where torch took 54 us, and 13 us for each change of layout: 7.5 us behind the product that sums.
constexpr int kBnCols = 64, kBnThreads = 256, kBnLanes = kBnThreads / 8, kBnApplyThreads = 1024;
constexpr int kBnChunks = 64, kBnForwardChunks = 256, kBnParts = 256;         // kBnParts: rows of sums that the workspace holds
static_assert(kBnChunks <= kBnParts, "a row of sums to a chunk");
struct Chunks {
    int rows, count;          // rows of a chunk (the last may have fewer), chunks
};
inline Chunks bn_chunks(int64_t M, int most) {
    const int64_t rows = std::max<int64_t>((M + most - 1) / most, kBnLanes);
    return Chunks{(int)rows, (int)((M + rows - 1) / rows)};
}
template <class DT> __device__ inline void unpack(u32x4 w, float (&v)[8]) {
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const f32x2 p = widen<DT>(w[i]);
        v[2 * i] = p.x;
        v[2 * i + 1] = p.y;
    }
}
// Sums round where the modules round: a projection's output before the residual takes it, a norm's gradient before the
// residual's.
template <class DT> __device__ inline f32x4 rounded(f32x4 v) { return widen4<DT>(narrow4<DT>(v)); }
template <class DT> __device__ inline u32x4 repack(const float (&v)[8]) {
    return u32x4{Mma<DT>::pack(v[0], v[1]), Mma<DT>::pack(v[2], v[3]), Mma<DT>::pack(v[4], v[5]), Mma<DT>::pack(v[6], v[7])};
}
// Sums over the 32 row lanes: a[channel of this thread's eight] -> total of channel `threadIdx.x & 63`, in threads below 64.
__device__ inline void meet(float (*part)[kBnCols + 1], float (*quarter)[kBnCols], const float (&v)[8], float &total) {
    const int c = threadIdx.x & 7, r = threadIdx.x >> 3, ch = threadIdx.x & 63, q = threadIdx.x >> 6;
    __syncthreads();
#pragma unroll
    for (int i = 0; i < 8; ++i) part[r][8 * c + i] = v[i];
    __syncthreads();
    float s = 0.f;
#pragma unroll
    for (int k = 0; k < kBnLanes / 4; ++k) s += part[q * (kBnLanes / 4) + k][ch];
    quarter[q][ch] = s;
    __syncthreads();
    total = quarter[0][ch] + quarter[1][ch] + (quarter[2][ch] + quarter[3][ch]);
}
// [N, T, C] -> [N, C, T], 64 x 64 at a time through LDS: the layout in which torch sums the statistics.
__global__ void __launch_bounds__(256)
to_channels_kernel(uint16_t *__restrict__ out, const char *__restrict__ x, int T, int C) {
    __shared__ uint16_t tile[64][64 + 2];
    const int t0 = blockIdx.x * 64, c0 = blockIdx.y * 64;
    const char *src = x + ((int64_t)blockIdx.z * T * C + c0) * 2;
    uint16_t *dst = out + ((int64_t)blockIdx.z * C + c0) * T;
#pragma unroll
    for (int i = 0; i < 2; ++i) {
        const int u = i * 256 + threadIdx.x, t = u >> 3, c = (u & 7) * 8;
        if (t0 + t < T) {
            const u32x4 v = *reinterpret_cast<const u32x4 *>(src + ((int64_t)(t0 + t) * C + c) * 2);
#pragma unroll
            for (int k = 0; k < 4; ++k) {
                tile[t][c + 2 * k] = (uint16_t)v[k];
                tile[t][c + 2 * k + 1] = (uint16_t)(v[k] >> 16);
            }
        }
    }
    __syncthreads();
    const int t = threadIdx.x & 63;
    if (t0 + t >= T) return;
#pragma unroll 4
    for (int c = threadIdx.x >> 6; c < 64; c += 4) dst[(int64_t)c * T + t0 + t] = tile[t][c];
}

// weight * (x - mean) * rstd + bias of two channels, each rounded once (as torch's kernel rounds: fp16 through the mixed
// multiply-add, which rounds its exact result).
template <class DT> __device__ inline uint32_t normal_pair(const float *x, const float *m, const float *w, const float *r, const float *b);
template <> __device__ inline uint32_t normal_pair<FP16>(const float *x, const float *m, const float *w, const float *r, const float *b) {
    uint32_t v;
    const float lo = w[0] * (x[0] - m[0]), hi = w[1] * (x[1] - m[1]);
    asm("v_fma_mixlo_f16 %0, %1, %2, %3" : "=v"(v) : "v"(lo), "v"(r[0]), "v"(b[0]));
    asm("v_fma_mixhi_f16 %0, %1, %2, %3" : "+v"(v) : "v"(hi), "v"(r[1]), "v"(b[1]));
    return v;
}
template <> __device__ inline uint32_t normal_pair<BF16>(const float *x, const float *m, const float *w, const float *r, const float *b) {
    return Mma<BF16>::pack(__builtin_fmaf(w[0] * (x[0] - m[0]), r[0], b[0]), __builtin_fmaf(w[1] * (x[1] - m[1]), r[1], b[1]));
}
struct BnApply {
    char *y;
    const char *x;
    const float *batch_mean, *batch_var, *weight, *bias;
    float *mean, *rstd;                        // for the backward
    int64_t *batches;                          // counts the calls, as torch's module does
    float eps;
    int M, C, rows;
    const char *add;                           // 16-bit [T, C], added to every sample's rows, or NULL
    int T;
};
template <class DT>
__global__ void __launch_bounds__(kBnThreads)
bn_apply_kernel(BnApply a) {
    const int c = threadIdx.x & 7, c0 = blockIdx.x * kBnCols + 8 * c, r0 = blockIdx.y * a.rows, r1 = min(a.M, r0 + a.rows);
    float m[8], w[8], b[8], r[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) {
        m[i] = a.batch_mean[c0 + i], w[i] = a.weight[c0 + i], b[i] = a.bias[c0 + i];
        r[i] = __builtin_amdgcn_rsqf(a.batch_var[c0 + i] + a.eps);
    }
    if (blockIdx.y == 0 && threadIdx.x < 8) {
#pragma unroll
        for (int i = 0; i < 8; ++i) a.mean[c0 + i] = m[i], a.rstd[c0 + i] = r[i];
        if (c0 == 0) *a.batches += 1;
    }
    const int64_t pitch = 2 * (int64_t)a.C, at = 2 * (int64_t)c0;
#pragma unroll 4
    for (int t = r0 + (threadIdx.x >> 3); t < r1; t += kBnLanes) {
        float v[8];
        unpack<DT>(*reinterpret_cast<const u32x4 *>(a.x + t * pitch + at), v);
        u32x4 y;
#pragma unroll
        for (int i = 0; i < 4; ++i) y[i] = normal_pair<DT>(v + 2 * i, m + 2 * i, w + 2 * i, r + 2 * i, b + 2 * i);
        if (a.add) {
            float e[8];
            unpack<DT>(y, v);
            unpack<DT>(*reinterpret_cast<const u32x4 *>(a.add + t % a.T * pitch + at), e);
#pragma unroll
            for (int i = 0; i < 8; ++i) v[i] += e[i];
            y = repack<DT>(v);
        }
        *reinterpret_cast<u32x4 *>(a.y + t * pitch + at) = y;
    }
}

// Backward: sums of dy and of dy * (x - mean) over a chunk's rows (behind the product that makes dy, where it is few enough
// blocks of rows: see launch_gemm), then
// dx = weight * rstd * (dy - sum(dy) / M - (x - mean) * rstd^2 * sum(dy (x - mean)) / M) + `add`.
template <class DT>
__global__ void __launch_bounds__(kBnThreads)
bn_bwd_sums_kernel(float *__restrict__ part_dy, float *__restrict__ part_dyx, const char *__restrict__ dy, const char *__restrict__ x,
                   const float *__restrict__ mean, int M, int C, int rows) {
    __shared__ float part[kBnLanes][kBnCols + 1], quarter[4][kBnCols];
    const int c = threadIdx.x & 7, r = threadIdx.x >> 3, c0 = blockIdx.x * kBnCols, r0 = blockIdx.y * rows, r1 = min(M, r0 + rows);
    const int64_t pitch = 2 * (int64_t)C, at = 2 * (int64_t)(c0 + 8 * c);
    float m[8], s1[8], s2[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) {
        m[i] = mean[c0 + 8 * c + i];
        s1[i] = s2[i] = 0.f;
    }
#pragma unroll 4
    for (int t = r0 + r; t < r1; t += kBnLanes) {
        float v[8], d[8];
        unpack<DT>(*reinterpret_cast<const u32x4 *>(x + t * pitch + at), v);
        unpack<DT>(*reinterpret_cast<const u32x4 *>(dy + t * pitch + at), d);
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            s1[i] += d[i];
            s2[i] = __builtin_fmaf(d[i], v[i] - m[i], s2[i]);
        }
    }
    float a, b;
    meet(part, quarter, s1, a);
    meet(part, quarter, s2, b);
    if (threadIdx.x >= kBnCols) return;
    part_dy[(int64_t)blockIdx.y * C + c0 + threadIdx.x] = a;
    part_dyx[(int64_t)blockIdx.y * C + c0 + threadIdx.x] = b;
}
struct BnBackward {
    char *dx;
    const char *dy, *x, *add;
    const float *part_dy, *part_dyx, *weight, *mean, *rstd;
    float *dweight, *dbias;
    int M, C, rows, chunks;
};
template <class DT>
__global__ void __launch_bounds__(kBnApplyThreads)
bn_bwd_apply_kernel(BnBackward a) {
    constexpr int kLanes = kBnApplyThreads / (kBnCols / 4);            // chunks side by side, four channels to a thread
    __shared__ float met[2][kLanes][kBnCols], s_k1[kBnCols], s_k2[kBnCols], s_a[kBnCols];
    const int c0 = blockIdx.x * kBnCols, ch = threadIdx.x & 63;
    {
        const int lane = threadIdx.x / (kBnCols / 4), at = c0 + 4 * (threadIdx.x % (kBnCols / 4));
        f32x4 s1 = {0.f, 0.f, 0.f, 0.f}, s2 = s1;
#pragma unroll 8
        for (int k = lane; k < a.chunks; k += kLanes) {
            s1 += *reinterpret_cast<const f32x4 *>(a.part_dy + (int64_t)k * a.C + at);
            s2 += *reinterpret_cast<const f32x4 *>(a.part_dyx + (int64_t)k * a.C + at);
        }
#pragma unroll
        for (int r = 0; r < 4; ++r) met[0][lane][at - c0 + r] = s1[r], met[1][lane][at - c0 + r] = s2[r];
        __syncthreads();
    }
    float s1 = 0.f, s2 = 0.f;
    if (threadIdx.x < kBnCols)
#pragma unroll
        for (int k = 0; k < kLanes; ++k) s1 += met[0][k][ch], s2 += met[1][k][ch];
    if (threadIdx.x < kBnCols) {
        const float rstd = a.rstd[c0 + ch];
        s_a[ch] = a.weight[c0 + ch] * rstd;
        s_k1[ch] = s1 / (float)a.M;
        s_k2[ch] = s2 * rstd * rstd / (float)a.M;
        if (blockIdx.y == 0) {
            a.dweight[c0 + ch] = s2 * rstd;
            a.dbias[c0 + ch] = s1;
        }
    }
    __syncthreads();
    const int c = threadIdx.x & 7, r0 = blockIdx.y * a.rows, r1 = min(a.M, r0 + a.rows);
    float m[8], k1[8], k2[8], f[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) m[i] = a.mean[c0 + 8 * c + i], k1[i] = s_k1[8 * c + i], k2[i] = s_k2[8 * c + i], f[i] = s_a[8 * c + i];
    const int64_t pitch = 2 * (int64_t)a.C, at = 2 * (int64_t)(c0 + 8 * c);
#pragma unroll 4
    for (int t = r0 + (threadIdx.x >> 3); t < r1; t += kBnApplyThreads / 8) {
        float v[8], d[8], e[8];
        unpack<DT>(*reinterpret_cast<const u32x4 *>(a.x + t * pitch + at), v);
        unpack<DT>(*reinterpret_cast<const u32x4 *>(a.dy + t * pitch + at), d);
        unpack<DT>(*reinterpret_cast<const u32x4 *>(a.add + t * pitch + at), e);
#pragma unroll
        for (int i = 0; i < 8; ++i) v[i] = f[i] * (d[i] - k1[i] - (v[i] - m[i]) * k2[i]);
        unpack<DT>(repack<DT>(v), v);
#pragma unroll
        for (int i = 0; i < 8; ++i) v[i] += e[i];
        *reinterpret_cast<u32x4 *>(a.dx + t * pitch + at) = repack<DT>(v);
    }
}

// =============================================================================
// Weights of a projection, packed
// =============================================================================
// A projection's weight lies in memory as [outputs, inputs / groups] (a linear layer or a grouped 1x1 convolution) and is
// used as the dense [outputs, inputs] matrix with the groups' blocks on its diagonal.  Row r of a qkv projection of a
// channels-first model is output channel ((f % per) * groups + f / per) * 3 + which, r = which * C + f, per = C / groups.
struct Weight {
    const float *w, *b;           // parameters
    float *dw, *db;               // and their gradients
    int outputs, inputs, groups, ordered;
    __host__ __device__ inline int row(int r) const {
        if (!ordered) return r;
        const int C = outputs / 3, per = C / groups, which = r / C, f = r - which * C;
        return ((f % per) * groups + f / per) * 3 + which;
    }
    // place of element (row r, input i) in the parameter, -1 off the diagonal
    __host__ __device__ inline int64_t at(int r, int i) const {
        const int o = row(r), in = inputs / groups, i0 = o / (outputs / groups) * in;
        return i < i0 || i >= i0 + in ? -1 : (int64_t)o * in + (i - i0);
    }
};
constexpr int kWeights = 5;       // qkv, proj, fc1, fc2; linear_pos of dense layers, otherwise empty
struct Pack {
    Weight w[kWeights];
    char *plain[kWeights], *turned[kWeights];   // in fragment order: [outputs, inputs] and its transpose
    float *bias[kWeights];                      // in the rows' order
    int first[kWeights + 1];                    // blocks of 32 x 32 before each
};
template <class DT>
__global__ void __launch_bounds__(256)
pack_kernel(Pack p) {
    __shared__ float tile[32][33];
    int j = 0;
    while (j < kWeights - 1 && (int)blockIdx.x >= p.first[j + 1]) ++j;
    const Weight &w = p.w[j];
    const int block = (int)blockIdx.x - p.first[j], cols = w.inputs / 32, o0 = block / cols * 32, i0 = block % cols * 32;
    {
        const int r = threadIdx.x >> 3, c = (threadIdx.x & 7) * 4;
        const int64_t at = w.at(o0 + r, i0 + c);           // groups have multiples of 32 inputs: four of a row are in or out together
        const f32x4 v = at < 0 ? f32x4{0.f, 0.f, 0.f, 0.f} : *reinterpret_cast<const f32x4 *>(w.w + at);
#pragma unroll
        for (int k = 0; k < 4; ++k) tile[r][c + k] = v[k];
        if (w.b && i0 == 0 && c == 0) p.bias[j][o0 + r] = widen<DT>(Mma<DT>::pack(w.b[w.row(o0 + r)], 0.f)).x;     // autocast's
    }
    __syncthreads();
    const int half = threadIdx.x >> 7, t = threadIdx.x & 127, frag = t >> 6, lane = t & 63, n = lane & 15, g = lane >> 4;
    float v[8];
    if (half == 0) {
#pragma unroll
        for (int k = 0; k < 8; ++k) v[k] = tile[16 * frag + n][8 * g + k];
        *reinterpret_cast<u32x4 *>(p.plain[j] + ((int64_t)(o0 / 16 + frag) * (w.inputs / 32) + i0 / 32) * kFrag + lane * 16) = repack<DT>(v);
    } else if (p.turned[j]) {
#pragma unroll
        for (int k = 0; k < 8; ++k) v[k] = tile[8 * g + k][16 * frag + n];
        *reinterpret_cast<u32x4 *>(p.turned[j] + ((int64_t)(i0 / 16 + frag) * (w.outputs / 32) + o0 / 32) * kFrag + lane * 16) = repack<DT>(v);
    }
}

// =============================================================================
// Products over all tokens
// =============================================================================
enum GemmEnd {
    kStore,           // out = v
    kBias,            // out = v + bias
    kResidual,        // out = aux + sample_scale * (v + bias)
    kGelu,            // out2 = v + bias, out = gelu(out2)
    kGeluBack,        // out = v * gelu'(aux)
    kNormBack,        // out = v, and for the norm whose input aux is, sums of v and of v * (aux - mean) over the block's rows
};
struct Gemm {
    const char *x, *w;
    char *out, *out2;
    const char *aux;
    const float *bias, *sample_scale;      // one factor per sample of T rows, or NULL
    const float *mean;                     // kNormBack ...
    float *part_dy, *part_dyx;             // ... [blocks of rows, outputs]
    int inputs, outputs, M, T;
    uint32_t T_magic;
    int late;                              // the sum is rounded before the bias is added (a product and an addition in torch)
};
__device__ inline float over_row(float x) {                       // sum over 16 lanes
    x += __uint_as_float(__builtin_amdgcn_mov_dpp(__float_as_uint(x), 0xb1, 0xf, 0xf, true));
    x += __uint_as_float(__builtin_amdgcn_mov_dpp(__float_as_uint(x), 0x4e, 0xf, 0xf, true));
    x += __uint_as_float(__builtin_amdgcn_mov_dpp(__float_as_uint(x), 0x141, 0xf, 0xf, true));
    return x + __uint_as_float(__builtin_amdgcn_mov_dpp(__float_as_uint(x), 0x140, 0xf, 0xf, true));
}
// Phi(x) and x's density, the former by formula 7.1.26 of Abramowitz and Stegun's handbook (error below 1.5e-7); infinities
// come out as x * Phi(x) gives them.
__device__ inline void normal_of(float x, float &cdf, float &pdf) {
    const float t = __builtin_amdgcn_rcpf(__builtin_fmaf(__builtin_fabsf(x), 0.3275911f * 0.70710678f, 1.f));
    float e = __builtin_fmaf(t, 0.5f * 1.061405429f, 0.5f * -1.453152027f);
    e = __builtin_fmaf(t, e, 0.5f * 1.421413741f);
    e = __builtin_fmaf(t, e, 0.5f * -0.284496736f);
    e = __builtin_fmaf(t, e, 0.5f * 0.254829592f);
    const float ex = __builtin_amdgcn_exp2f(x * x * -0.72134752f), tail = t * e * ex;
    cdf = x < 0.f ? tail : 1.f - tail;
    pdf = ex * 0.3989422804f;
}
template <class DT, int MT, int NTW, GemmEnd END>
__global__ void __launch_bounds__(kThreads, 2)
gemm_kernel(Gemm a, int col_blocks) {
    constexpr int PF = 4, NW = kWaves;
    extern __shared__ __attribute__((aligned(16))) char smem[];
    LDS_PTR(char) lds = (LDS_PTR(char))smem;
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), n = lane & 15, g = lane >> 4;
    const uint32_t item = xcd_item(blockIdx.x, gridDim.x);           // neighbours share their rows' lines
    const uint32_t row_block = item / (uint32_t)col_blocks;
    const int64_t m0 = (int64_t)row_block * (16 * MT);
    const int rows = (int)min((int64_t)(16 * MT), a.M - m0), x_pitch = 2 * a.inputs, pitch = 2 * a.outputs;
    const int tile0 = ((int)(item - row_block * col_blocks) * NW + wave) * NTW;
    const Rsrc xs = make_rsrc(a.x + m0 * x_pitch, rows * x_pitch), ws = weight_rsrc(a.w, a.outputs, a.inputs);
    const int steps = a.inputs / 32, pieces = a.inputs / 256;
    auto stage = [&](int piece) {
        constexpr int kChunks = 16 * MT * kRow / kChunk;
#pragma unroll
        for (int j = 0; j < kChunks / NW; ++j) {
            const int c = j * NW + wave, row = 2 * c + (lane >> 5);
            load_to_lds<16, kReadShared>(xs, lds + (piece & 1) * (16 * MT * kRow) + c * kChunk, row * x_pitch + piece * kRow + ((lane & 31) ^ (row & 15)) * 16);
        }
    };
    stage(0);
    f32x4 acc[NTW][MT];
    clear(acc);
    Ring<NTW, PF> ring;
    using P = Product<NTW, 8>;
    const int lane16 = lane * 16;
    ring.begin(P{ws, tile0 * steps, steps, 0}, lane16);
#pragma unroll 1
    for (int p = 0; p < pieces; ++p) {
        wait_direct();
        barrier_lds();
        if (p + 1 < pieces) stage(p + 1);
        const P now{ws, tile0 * steps + 8 * p, steps, 0}, next{ws, tile0 * steps + 8 * min(p + 1, pieces - 1), steps, 0};
        multiply<DT, MT>(acc, ring, now, next, lds + (p & 1) * (16 * MT * kRow), n, g, lane16);
    }
    const Rsrc os = make_rsrc(a.out + m0 * pitch, rows * pitch);
    f32x4 bias[NTW];
    if constexpr (END == kBias || END == kResidual || END == kGelu) {
#pragma unroll
        for (int j = 0; j < NTW; ++j) bias[j] = *reinterpret_cast<const f32x4 *>(a.bias + 16 * (tile0 + j) + 4 * g);
    }
    f32x4 mean[NTW], s1[NTW], s2[NTW];
    if constexpr (END == kNormBack) {
#pragma unroll
        for (int j = 0; j < NTW; ++j) mean[j] = *reinterpret_cast<const f32x4 *>(a.mean + 16 * (tile0 + j) + 4 * g), s1[j] = s2[j] = f32x4{0.f, 0.f, 0.f, 0.f};
    }
    // What an end reads of every output, all at once and store_tile backwards: 16 bytes to a lane, 64 of a row together (GELU's
    // derivative over 12800 x 1024: 29.0 -> 23.6 us, 27.1 with a row tile's behind the other).
    u32x4 aux16[MT][NTW / 2];
    if constexpr (END == kResidual || END == kGeluBack || END == kNormBack) {
        const Rsrc as = make_rsrc(a.aux + m0 * pitch, rows * pitch);
#pragma unroll
        for (int i = 0; i < MT; ++i)
#pragma unroll
            for (int p = 0; p < NTW / 2; ++p)
                aux16[i][p] = __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(as, (16 * i + n) * pitch + 32 * tile0 + (2 * p + (g & 1)) * 32 + (g >> 1) * 16, 0, 0));
    }
#pragma unroll
    for (int i = 0; i < MT; ++i) {
        u32x2 o[NTW];
        const int row_byte = (16 * i + n) * pitch + 32 * tile0;
        f32x4 aux[NTW];
        if constexpr (END == kResidual || END == kGeluBack || END == kNormBack) {
#pragma unroll
            for (int p = 0; p < NTW / 2; ++p) {
                const u32x4 v = aux16[i][p];
                const u32x2 lo = __builtin_amdgcn_permlane16_swap(v.x, v.z, false, false), hi = __builtin_amdgcn_permlane16_swap(v.y, v.w, false, false);
                aux[2 * p] = widen4<DT>(u32x2{lo.x, hi.x});
                aux[2 * p + 1] = widen4<DT>(u32x2{lo.y, hi.y});
            }
        }
        float f = 1.f;
        if constexpr (END == kResidual)
            if (a.sample_scale) {
                const uint32_t m = (uint32_t)min(m0 + 16 * i + n, (int64_t)a.M - 1);
                f = a.sample_scale[div_by(m, a.T, a.T_magic)];
            }
        if constexpr (END == kGelu) {
            u32x2 h[NTW];
#pragma unroll
            for (int j = 0; j < NTW; ++j) {
                h[j] = narrow4<DT>((a.late ? rounded<DT>(acc[j][i]) : acc[j][i]) + bias[j]);
                f32x4 v = widen4<DT>(h[j]);                  // of the value that the backward sees
#pragma unroll
                for (int r = 0; r < 4; ++r) v[r] = v[r] * 0.5f * (1.f + erff(v[r] * 0.70710678118654752f));
                o[j] = narrow4<DT>(v);
            }
            store_tile<16 * NTW, 0>(make_rsrc(a.out2 + m0 * pitch, rows * pitch), row_byte, h, g, 32 * NTW);
        } else {
#pragma unroll
            for (int j = 0; j < NTW; ++j) {
                f32x4 v = acc[j][i];
                if constexpr (END == kBias) v = (a.late ? rounded<DT>(v) : v) + bias[j];
                if constexpr (END == kResidual) v = aux[j] + rounded<DT>(f * rounded<DT>((a.late ? rounded<DT>(v) : v) + bias[j]));
                if constexpr (END == kGeluBack) {
                    v = rounded<DT>(v);
#pragma unroll
                    for (int r = 0; r < 4; ++r) {
                        float cdf, pdf;
                        normal_of(aux[j][r], cdf, pdf);
                        v[r] *= __builtin_fmaf(aux[j][r], pdf, cdf);
                    }
                }
                o[j] = narrow4<DT>(v);
                if constexpr (END == kNormBack) {            // of what is stored; rows behind the last are zeros
                    const f32x4 d = widen4<DT>(o[j]);
                    s1[j] += d;
                    s2[j] += d * (aux[j] - mean[j]);
                }
            }
        }
        store_tile<16 * NTW, 0>(os, row_byte, o, g, 32 * NTW);
    }
    if constexpr (END == kNormBack) {
#pragma unroll
        for (int j = 0; j < NTW; ++j) {
#pragma unroll
            for (int r = 0; r < 4; ++r) s1[j][r] = over_row(s1[j][r]), s2[j][r] = over_row(s2[j][r]);
            const int64_t at = (int64_t)row_block * a.outputs + 16 * (tile0 + j) + 4 * g;
            if (n == 0) *reinterpret_cast<f32x4 *>(a.part_dy + at) = s1[j], *reinterpret_cast<f32x4 *>(a.part_dyx + at) = s2[j];
        }
    }
}

// out[m, :] = x[m, :] * sample_scale[m / T]
template <class DT>
__global__ void __launch_bounds__(256)
scale_kernel(char *__restrict__ out, const char *__restrict__ x, const float *__restrict__ sample_scale, int64_t units, int units_per_sample) {
    for (int64_t u = (int64_t)blockIdx.x * 256 + threadIdx.x; u < units; u += (int64_t)gridDim.x * 256) {
        float v[8];
        unpack<DT>(*reinterpret_cast<const u32x4 *>(x + u * 16), v);
        const float f = sample_scale[u / units_per_sample];
#pragma unroll
        for (int i = 0; i < 8; ++i) v[i] *= f;
        *reinterpret_cast<u32x4 *>(out + u * 16) = repack<DT>(v);
    }
}

// out[t, :] = sum over the samples of x[n, t, :]: 32 units of eight channels to a workgroup, a sample to each of its eight lanes.
template <class DT>
__global__ void __launch_bounds__(256)
sum_samples_kernel(char *__restrict__ out, const char *__restrict__ x, int N, int64_t units) {
    __shared__ float part[8][32][9];
    const int k = threadIdx.x & 31, lane = threadIdx.x >> 5;
    const int64_t u = (int64_t)blockIdx.x * 32 + k;
    float s[8] = {};
    if (u < units)
#pragma unroll 4
        for (int n = lane; n < N; n += 8) {
            float v[8];
            unpack<DT>(*reinterpret_cast<const u32x4 *>(x + (n * units + u) * 16), v);
#pragma unroll
            for (int i = 0; i < 8; ++i) s[i] += v[i];
        }
#pragma unroll
    for (int i = 0; i < 8; ++i) part[lane][k][i] = s[i];
    __syncthreads();
    if (lane || u >= units) return;
#pragma unroll
    for (int l = 1; l < 8; ++l)
#pragma unroll
        for (int i = 0; i < 8; ++i) s[i] += part[l][k][i];
    *reinterpret_cast<u32x4 *>(out + u * 16) = repack<DT>(s);
}

// =============================================================================
// Weight gradients of the layer's projections in one launch
// =============================================================================
// dW[o, i] = sum over rows of dY[m, o] X[m, i], db[o] = sum of dY[m, o].  The contraction runs along the rows of both
// operands, so both come out of LDS transposed (ds_read_b64_tr_b16).  A workgroup computes a 128 x 128 block of one dW
// (each wave 64 x 64) over one of `splits` ranges of rows, 64 rows at a time, double buffered; the ranges' sums (fp32) are
// folded in a fixed order by a second kernel, which also undoes the row order and drops what is off the diagonal.
// 12800 tokens, 256 channels, 1024 hidden (20 GFLOP): 32 us, 620 TFLOP/s, and 7 us to fold ten ranges; as four library
// products of chunks with four sums over the chunks and four bias sums it was 200 us.
constexpr int kGradTile = 128, kGradRows = 64;
struct GradJob {
    const char *dy, *x;
    int outputs, inputs, M, first;       // M: rows; first: blocks of 128 x 128 before
    int64_t part;                        // floats before: dW, then db
};
struct Grads {
    GradJob job[kWeights];
    float *partial;
    int64_t stride;                      // floats of one range
    int rows, blocks;                    // rows of a range (a multiple of 64)
};
template <class DT>
__global__ void __launch_bounds__(kThreads, 2)
grad_kernel(Grads a) {
    using L = Lds<kGradTile>;
    constexpr int kPart = kGradRows * L::kRowBytes;            // 16 KB of dY, then of X
    extern __shared__ __attribute__((aligned(16))) char smem[];
    LDS_PTR(char) lds = (LDS_PTR(char))smem;
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), n = lane & 15, g = lane >> 4;
    const uint32_t item = xcd_item(blockIdx.x, gridDim.x);     // the blocks of a range read the same rows
    const int split = (int)(item / (uint32_t)a.blocks), block = (int)item - split * a.blocks;
    int jn = 0;
    while (jn < kWeights - 1 && block >= a.job[jn + 1].first) ++jn;
    const GradJob &job = a.job[jn];
    const int cols = job.inputs / kGradTile, o0 = (block - job.first) / cols * kGradTile, i0 = (block - job.first) % cols * kGradTile;
    const int64_t m0 = (int64_t)split * a.rows;
    const int rows = (int)max((int64_t)0, min((int64_t)a.rows, job.M - m0)), pieces = (rows + kGradRows - 1) / kGradRows;
    const int y_pitch = 2 * job.outputs, x_pitch = 2 * job.inputs;
    const Rsrc ys = make_rsrc(job.dy + m0 * y_pitch, rows * y_pitch), xs = make_rsrc(job.x + m0 * x_pitch, rows * x_pitch);
    const int wo = wave & 1, wi = wave >> 1;
    auto stage = [&](int piece) {
        LDS_PTR(char) to = lds + (piece & 1) * (2 * kPart);
#pragma unroll
        for (int j = 0; j < kPart / kChunk / kWaves; ++j) {
            const int c = j * kWaves + wave, r = 4 * c + (lane >> 4), unit = ((lane & 15) ^ (r & 15)) * 16, row = piece * kGradRows + r;
            load_to_lds<16, kReadShared>(ys, to + c * kChunk, row * y_pitch + 2 * o0 + unit);
            load_to_lds<16, kReadShared>(xs, to + kPart + c * kChunk, row * x_pitch + 2 * i0 + unit);
        }
    };
    // byte of this lane's piece of channel tile t, rows 0 .. 15; tiles of 16 rows follow each other
    int yo[4], xo[4];
#pragma unroll
    for (int t = 0; t < 4; ++t) {
        yo[t] = L::addr(4 * g + (n >> 2), 128 * wo + 32 * t + 8 * (n & 3));
        xo[t] = kPart + L::addr(4 * g + (n >> 2), 128 * wi + 32 * t + 8 * (n & 3));
    }
    const bool sums = i0 == 0 && wi == 0;
    const uint32_t one = Mma<DT>::pack(1.f, 1.f);
    const u32x4 ones = {one, one, one, one};
    f32x4 acc[4][4], db[4];                                    // [o tile][i tile]
    clear(acc);
#pragma unroll
    for (int t = 0; t < 4; ++t) db[t] = f32x4{0.f, 0.f, 0.f, 0.f};
    if (pieces) stage(0);                                      // a projection of few rows has ranges without any: zeros
#pragma unroll 1
    for (int p = 0; p < pieces; ++p) {
        wait_direct();
        barrier_lds();
        if (p + 1 < pieces) stage(p + 1);
        LDS_PTR(char) from = lds + (p & 1) * (2 * kPart);
#pragma unroll
        for (int s = 0; s < kGradRows / 32; ++s) {
            u32x4 y[4], x[4];
#pragma unroll
            for (int t = 0; t < 4; ++t) {
                const u32x2 y0 = read_tr(from + 2 * s * L::kTileBytes + yo[t]), y1 = read_tr(from + (2 * s + 1) * L::kTileBytes + yo[t]);
                const u32x2 x0 = read_tr(from + 2 * s * L::kTileBytes + xo[t]), x1 = read_tr(from + (2 * s + 1) * L::kTileBytes + xo[t]);
                y[t] = u32x4{y0.x, y0.y, y1.x, y1.y};
                x[t] = u32x4{x0.x, x0.y, x1.x, x1.y};
            }
#pragma unroll
            for (int t = 0; t < 4; ++t)
#pragma unroll
                for (int u = 0; u < 4; ++u) acc[t][u] = Mma<DT>::k32(x[u], y[t], acc[t][u]);
            if (sums)
#pragma unroll
                for (int t = 0; t < 4; ++t) db[t] = Mma<DT>::k32(ones, y[t], db[t]);
        }
    }
    float *part = a.partial + (int64_t)split * a.stride + job.part;
#pragma unroll
    for (int t = 0; t < 4; ++t) {
        const int o = o0 + 64 * wo + 16 * t + n;
#pragma unroll
        for (int u = 0; u < 4; ++u) *reinterpret_cast<f32x4 *>(part + (int64_t)o * job.inputs + i0 + 64 * wi + 16 * u + 4 * g) = acc[t][u];
        if (sums && g == 0) part[(int64_t)job.outputs * job.inputs + o] = db[t][0];
    }
}
struct Fold {
    Weight w[kWeights];
    int64_t part[kWeights + 1];          // floats before each projection's dW
    const float *partial;
    int64_t stride;
    int splits;
};
__global__ void __launch_bounds__(256)
grad_fold_kernel(Fold a) {
    const int64_t e = ((int64_t)blockIdx.x * 256 + threadIdx.x) * 4;
    if (e >= a.part[kWeights]) return;
    int j = 0;
    while (j < kWeights - 1 && e >= a.part[j + 1]) ++j;
    const Weight &w = a.w[j];
    const int64_t k = e - a.part[j], nw = (int64_t)w.outputs * w.inputs;
    const int r = (int)(k / w.inputs), i = (int)(k - (int64_t)r * w.inputs);
    const int64_t at = k < nw ? w.at(r, i) : 0;
    if (at < 0) return;
    f32x4 s = *reinterpret_cast<const f32x4 *>(a.partial + e);
#pragma unroll 4
    for (int p = 1; p < a.splits; ++p) s += *reinterpret_cast<const f32x4 *>(a.partial + p * a.stride + e);
    if (k < nw) {
        *reinterpret_cast<f32x4 *>(w.dw + at) = s;
    } else if (w.db) {
#pragma unroll
        for (int q = 0; q < 4; ++q) w.db[w.row((int)(k - nw) + q)] = s[q];
    }
}

// =============================================================================
// Attentive statistics pooling, backward, on [N, C, T]
// =============================================================================
// Rows of T values lie one behind the other, so R rows (a multiple of eight) are whole 16-byte units in memory whatever T is:
// they come to LDS and leave it as such, and 16 lanes work on a row.  Bound by memory.  128 x 1536 rows of 100 values, fp16: 48
// and 47 us (157 and 197 MB), where torch took some thirty kernels of 440 and 330 us.  A training step, which its host paces by
// then: 10.1-10.3 -> 9.5-9.7 ms.
constexpr int kPoolLanes = 16, kPoolThreads = 256;
__device__ inline float max_over_row(float x) {
    x = __builtin_fmaxf(x, __uint_as_float(__builtin_amdgcn_mov_dpp(__float_as_uint(x), 0xb1, 0xf, 0xf, true)));
    x = __builtin_fmaxf(x, __uint_as_float(__builtin_amdgcn_mov_dpp(__float_as_uint(x), 0x4e, 0xf, 0xf, true)));
    x = __builtin_fmaxf(x, __uint_as_float(__builtin_amdgcn_mov_dpp(__float_as_uint(x), 0x141, 0xf, 0xf, true)));
    return __builtin_fmaxf(x, __uint_as_float(__builtin_amdgcn_mov_dpp(__float_as_uint(x), 0x140, 0xf, 0xf, true)));
}
template <class DT> __device__ inline float value_of(uint16_t v) { return widen<DT>((uint32_t)v).x; }
template <class DT> __device__ inline uint16_t bits_of(float v) { return (uint16_t)Mma<DT>::pack(v, 0.f); }
struct RowBlock {
    int rows, C, T;                     // rows of a block; channels of a sample
    float eps;
};
// Gradients of mean = sum of w x and std = sqrt(max(sum of w (x - mean)^2, eps)), w = softmax(logits), by logits and x.
template <class DT>
__global__ void __launch_bounds__(kPoolThreads)
pool_backward_kernel(char *__restrict__ dlogits, char *__restrict__ dx, const char *__restrict__ logits, const char *__restrict__ x,
                     const float *__restrict__ pooled, const float *__restrict__ dpooled, int64_t all, RowBlock a) {
    extern __shared__ __attribute__((aligned(16))) char smem[];
    const int64_t row0 = (int64_t)blockIdx.x * a.rows;
    const int rows = (int)min((int64_t)a.rows, all - row0), units = rows * a.T / 8;
    u32x4 *zs = reinterpret_cast<u32x4 *>(smem), *xs = zs + a.rows * a.T / 8;
    const int64_t at = row0 * a.T / 8;
    for (int u = threadIdx.x; u < units; u += kPoolThreads) {
        zs[u] = reinterpret_cast<const u32x4 *>(logits)[at + u];
        xs[u] = reinterpret_cast<const u32x4 *>(x)[at + u];
    }
    __syncthreads();
    const int lane = threadIdx.x % kPoolLanes;
    for (int r = threadIdx.x / kPoolLanes; r < rows; r += kPoolThreads / kPoolLanes) {
        const uint32_t row = (uint32_t)(row0 + r), n = row / (uint32_t)a.C;
        const int64_t o = (int64_t)row + (int64_t)n * a.C;              // of [N, 2 C]
        uint16_t *z = reinterpret_cast<uint16_t *>(zs) + r * a.T, *v = reinterpret_cast<uint16_t *>(xs) + r * a.T;
        const float mean = pooled[o], std = pooled[o + a.C], gm = dpooled[o], gs = dpooled[o + a.C];
        float top = kNegInf, s0 = 0.f, s1 = 0.f, s2 = 0.f;
        for (int t = lane; t < a.T; t += kPoolLanes) top = __builtin_fmaxf(top, value_of<DT>(z[t]));
        top = max_over_row(top);
        for (int t = lane; t < a.T; t += kPoolLanes) {
            const float e = __builtin_amdgcn_exp2f((value_of<DT>(z[t]) - top) * kLog2e), d = value_of<DT>(v[t]) - mean;
            s0 += e;
            s1 = __builtin_fmaf(e, d, s1);
            s2 = __builtin_fmaf(e * d, d, s2);
        }
        const float inv = 1.f / over_row(s0), off = over_row(s1) * inv, var = over_row(s2) * inv;
        const float gv = var >= a.eps ? gs / (2.f * std) : 0.f;         // by the variance, and through it by the mean
        const float g1 = __builtin_fmaf(-2.f * gv, off, gm), base = __builtin_fmaf(g1, off, gv * var);
        for (int t = lane; t < a.T; t += kPoolLanes) {
            const float w = __builtin_amdgcn_exp2f((value_of<DT>(z[t]) - top) * kLog2e) * inv, d = value_of<DT>(v[t]) - mean;
            z[t] = bits_of<DT>(w * (__builtin_fmaf(__builtin_fmaf(gv, d, g1), d, -base)));
            v[t] = bits_of<DT>(w * __builtin_fmaf(2.f * gv, d, g1));
        }
    }
    __syncthreads();
    for (int u = threadIdx.x; u < units; u += kPoolThreads) {
        reinterpret_cast<u32x4 *>(dlogits)[at + u] = zs[u];
        reinterpret_cast<u32x4 *>(dx)[at + u] = xs[u];
    }
}
// [x, mean, std] along the channels, the latter two repeated along T (8 at least, so that a unit of eight values has two rows).
// A unit of each part to a thread.  128 x 1536 rows of 100 values: 24 us (157 MB); torch's concatenation of expanded tensors 103.
__global__ void __launch_bounds__(kPoolThreads)
context_kernel(u32x4 *__restrict__ out, const u32x4 *__restrict__ x, const uint16_t *__restrict__ mean, const uint16_t *__restrict__ std, int C, int T,
               uint32_t T_magic) {
    const uint32_t u = blockIdx.x * kPoolThreads + threadIdx.x, units = (uint32_t)C * T / 8;
    if (u >= units) return;
    const int64_t n = blockIdx.y;
    u32x4 *to = out + n * 3 * units + u;
    const uint32_t row = div_by(8 * u, T, T_magic), left = (row + 1) * T - 8 * u, next = min(row + 1, (uint32_t)C - 1);
    auto repeat = [&](const uint16_t *v) {
        const uint32_t a = v[n * C + row], b = v[n * C + next];
        u32x4 w;
#pragma unroll
        for (uint32_t k = 0; k < 4; ++k) w[k] = (2 * k < left ? a : b) | (2 * k + 1 < left ? a : b) << 16;
        return w;
    };
    const u32x4 m = repeat(mean), s = repeat(std);
    __builtin_nontemporal_store(x[n * units + u], to);
    __builtin_nontemporal_store(m, to + units);
    __builtin_nontemporal_store(s, to + 2 * (int64_t)units);
}
// Gradient of [x, mean over T, std over T] (the latter two along all of T) by x.
template <class DT>
__global__ void __launch_bounds__(kPoolThreads)
context_backward_kernel(char *__restrict__ dx, const char *__restrict__ dctx, const char *__restrict__ x, const uint16_t *__restrict__ var,
                        const uint16_t *__restrict__ std, RowBlock a) {
    extern __shared__ __attribute__((aligned(16))) char smem[];
    const int n = blockIdx.y, c0 = blockIdx.x * a.rows, rows = min(a.rows, a.C - c0), units = rows * a.T / 8, stride = a.rows * a.T / 8;
    u32x4 *lds = reinterpret_cast<u32x4 *>(smem);                      // x, and the gradient's three parts
    const u32x4 *gs = reinterpret_cast<const u32x4 *>(dctx) + ((int64_t)n * 3 * a.C + c0) * a.T / 8;
    const int64_t at = ((int64_t)n * a.C + c0) * a.T / 8, part = (int64_t)a.C * a.T / 8;
    for (int u = threadIdx.x; u < units; u += kPoolThreads) {
        lds[u] = reinterpret_cast<const u32x4 *>(x)[at + u];
#pragma unroll
        for (int k = 0; k < 3; ++k) lds[(k + 1) * stride + u] = gs[k * part + u];
    }
    __syncthreads();
    const int lane = threadIdx.x % kPoolLanes;
    const float per = 1.f / (float)a.T;
    for (int r = threadIdx.x / kPoolLanes; r < rows; r += kPoolThreads / kPoolLanes) {
        uint16_t *v = reinterpret_cast<uint16_t *>(lds) + r * a.T;
        const uint16_t *g = v + 8 * stride, *g_mean = g + 8 * stride, *g_std = g_mean + 8 * stride;
        float sx = 0.f, sm = 0.f, ss = 0.f;
        for (int t = lane; t < a.T; t += kPoolLanes) {
            sx += value_of<DT>(v[t]);
            sm += value_of<DT>(g_mean[t]);
            ss += value_of<DT>(g_std[t]);
        }
        const int64_t o = (int64_t)n * a.C + c0 + r;
        const float mean = over_row(sx) * per, add = over_row(sm) * per, by_std = over_row(ss);
        const float f = value_of<DT>(var[o]) >= a.eps ? by_std / (value_of<DT>(std[o]) * (float)(a.T - 1)) : 0.f;
        for (int t = lane; t < a.T; t += kPoolLanes) v[t] = bits_of<DT>(value_of<DT>(g[t]) + __builtin_fmaf(value_of<DT>(v[t]) - mean, f, add));
    }
    __syncthreads();
    for (int u = threadIdx.x; u < units; u += kPoolThreads) reinterpret_cast<u32x4 *>(dx)[at + u] = lds[u];
}
// Rows to a block of `tensors` tensors in LDS: some 32 KB, and eight rows at least.
inline int pool_rows(int64_t T, int tensors) { return (int)std::max<int64_t>(8, (32 << 10) / (2 * T * tensors) / 8 * 8); }
template <class DT>
int pool_backward(void *dlogits, void *dx, const void *logits, const void *x, const float *pooled, const float *dpooled, int64_t N, int64_t C, int64_t T,
                  float eps, hipStream_t s) {
    const int rows = pool_rows(T, 2);
    const size_t lds = (size_t)rows * T * 4;
    if (!allow_lds(pool_backward_kernel<DT>, lds)) return NA1D_ERR_LAUNCH;
    pool_backward_kernel<DT><<<(unsigned)((N * C + rows - 1) / rows), kPoolThreads, lds, s>>>(
        (char *)dlogits, (char *)dx, (const char *)logits, (const char *)x, pooled, dpooled, N * C, RowBlock{rows, (int)C, (int)T, eps});
    return launch_status();
}
template <class DT>
int context_backward(void *dx, const void *dctx, const void *x, const void *var, const void *std, int64_t N, int64_t C, int64_t T, float eps, hipStream_t s) {
    const int rows = (int)std::min<int64_t>(pool_rows(T, 4), C);
    const size_t lds = (size_t)rows * T * 8;
    if (!allow_lds(context_backward_kernel<DT>, lds)) return NA1D_ERR_LAUNCH;
    context_backward_kernel<DT><<<dim3((unsigned)((C + rows - 1) / rows), (unsigned)N), kPoolThreads, lds, s>>>(
        (char *)dx, (const char *)dctx, (const char *)x, (const uint16_t *)var, (const uint16_t *)std, RowBlock{rows, (int)C, (int)T, eps});
    return launch_status();
}
bool pool_ok(int64_t N, int64_t C, int64_t T) { return N >= 1 && N <= 65535 && C >= 8 && C % 8 == 0 && C <= (1 << 16) && T >= 2 && T <= 2048 && N * C < (1ll << 31); }
int run_pool_backward(void *dlogits, void *dx, const void *logits, const void *x, const float *pooled, const float *dpooled, int64_t N, int64_t C, int64_t T,
                      float eps, int dtype, hipStream_t s) {
    return dtype == NA1D_BF16 ? pool_backward<BF16>(dlogits, dx, logits, x, pooled, dpooled, N, C, T, eps, s)
                              : pool_backward<FP16>(dlogits, dx, logits, x, pooled, dpooled, N, C, T, eps, s);
}
int run_context(void *out, const void *x, const void *mean, const void *std, int64_t N, int64_t C, int64_t T, hipStream_t s) {
    if (T < 8 || C * T * T >= (1ll << 32)) return NA1D_ERR_UNSUPPORTED;            // what div_by takes
    const int64_t blocks = (C * T / 8 + kPoolThreads - 1) / kPoolThreads;
    context_kernel<<<dim3((unsigned)blocks, (unsigned)N), kPoolThreads, 0, s>>>((u32x4 *)out, (const u32x4 *)x, (const uint16_t *)mean, (const uint16_t *)std, (int)C, (int)T,
                                                                                div_magic(T));
    return launch_status();
}
int run_context_backward(void *dx, const void *dctx, const void *x, const void *var, const void *std, int64_t N, int64_t C, int64_t T, float eps, int dtype,
                         hipStream_t s) {
    return dtype == NA1D_BF16 ? context_backward<BF16>(dx, dctx, x, var, std, N, C, T, eps, s) : context_backward<FP16>(dx, dctx, x, var, std, N, C, T, eps, s);
}

// ----------------------------------------------------------------------------- the layer
inline Weight weight_of(const na1d_train_layer &l, int j) {
    const int C = l.dim, outputs[kWeights] = {3 * C, C, l.hidden, C, l.window ? 0 : C}, inputs[kWeights] = {C, C, C, l.hidden, C};
    return Weight{l.w[j], l.b[j], l.dw[j], l.db[j], outputs[j], inputs[j], l.groups, j == 0 && l.ordered};
}
struct Buffers {
    int64_t bytes = 0;
    int64_t take(int64_t n) {
        const int64_t at = bytes;
        bytes += (n + 255) / 256 * 256;
        return at;
    }
};
// What the forward leaves for the backward.
struct Saved : Buffers {
    int64_t y1, qkv, lse, attn, x1, y2, h, g, stats[4], turned[4];
    Saved(const na1d_train_layer &l, int64_t N, int64_t T) {
        const int64_t M = N * T, row = M * l.dim * 2;
        y1 = take(row), qkv = take(3 * row), lse = take(M * l.heads * 4), attn = take(row), x1 = take(row), y2 = take(row);
        h = take(M * l.hidden * 2), g = take(M * l.hidden * 2);
        for (int64_t &s : stats) s = take(l.dim * 4);
        for (int j = 0; j < 4; ++j) {
            const Weight w = weight_of(l, j);
            turned[j] = take((int64_t)w.outputs * w.inputs * 2);
        }
    }
};
struct ForwardScratch : Buffers {
    int64_t plain[kWeights], bias[kWeights], pos;
    ForwardScratch(const na1d_train_layer &l, int64_t T) {
        pos = take(l.window ? 0 : T * l.dim * 2);
        for (int j = 0; j < kWeights; ++j) {
            const Weight w = weight_of(l, j);
            plain[j] = take((int64_t)w.outputs * w.inputs * 2);
            bias[j] = take(w.outputs * 4);
        }
    }
};
struct GradPlan {
    int blocks = 0, splits, rows, first[kWeights];
    int64_t part[kWeights + 1] = {};
    GradPlan(const na1d_train_layer &l, int64_t M) {
        for (int j = 0; j < kWeights; ++j) {
            const Weight w = weight_of(l, j);
            first[j] = blocks;
            blocks += (w.outputs / kGradTile) * (w.inputs / kGradTile);
            part[j + 1] = part[j] + (int64_t)w.outputs * w.inputs + w.outputs;
        }
        // two workgroups on each CU; a range is worth a few pieces, and stays in the reach of 31-bit offsets
        int64_t want = std::max<int64_t>(1, std::min<int64_t>(512 / blocks, (M + 255) / 256));
        want = std::max(want, M * 2 * std::max(3 * l.dim, l.hidden) / (1 << 29) + 1);
        rows = (int)(((M + want - 1) / want + kGradRows - 1) / kGradRows * kGradRows);
        splits = (int)((M + rows - 1) / rows);
    }
};
struct BackwardScratch : Buffers {
    int64_t dz, dh, dy, dx1, ds, dattn, dqkv, part, grads, delta, dpos;
    BackwardScratch(const na1d_train_layer &l, int64_t N, int64_t T) {
        const int64_t M = N * T, row = M * l.dim * 2;
        const GradPlan p(l, M);
        dz = take(l.scale_mlp ? row : 0), dh = take(M * l.hidden * 2), dy = take(row), dx1 = take(row), ds = take(l.scale_attn ? row : 0);
        dattn = take(row), dqkv = take(3 * row), part = take((int64_t)2 * kBnParts * l.dim * 4);
        grads = take(p.splits * p.part[kWeights] * 4);
        delta = take(l.window ? 0 : M * l.heads * 4), dpos = take(l.window ? 0 : T * l.dim * 2);
    }
};

#define NA1D_TRY(...)                       \
    do {                                    \
        const int st_ = (__VA_ARGS__);      \
        if (st_ != NA1D_OK) return st_;     \
    } while (0)

inline int gemm_rows(int64_t M, int outputs) { return (M + 63) / 64 * (outputs / 256) >= 128 ? 64 : 32; }
// 64 rows x 128 outputs (a hundred registers: four workgroups on a CU); fewer rows where that leaves CUs idle.  Twice the
// outputs halve the rows' reads but two workgroups on a CU do not hide the ends: GELU's 28 instead of 22 us at 12800 rows.
template <class DT, GemmEnd END> int launch_gemm(const Gemm &a, hipStream_t s) {
    auto go = [&](auto kern, int mt, int ntw) {
        const size_t lds = (size_t)(a.inputs > 256 ? 2 : 1) * 16 * mt * kRow;
        if (!allow_lds(kern, lds)) return (int)NA1D_ERR_LAUNCH;
        const int cols = a.outputs / (64 * ntw);
        kern<<<(unsigned)((a.M + 16 * mt - 1) / (16 * mt) * cols), kThreads, lds, s>>>(a, cols);
        return launch_status();
    };
    if (gemm_rows(a.M, a.outputs) == 64) return go(gemm_kernel<DT, 4, 2, END>, 4, 2);
    return go(gemm_kernel<DT, 2, 2, END>, 2, 2);
}
template <class DT> int scale_rows(char *out, const char *x, const float *f, int64_t N, int64_t T, int dim, hipStream_t s) {
    const int64_t units = N * T * dim / 8;
    scale_kernel<DT><<<(unsigned)std::min<int64_t>((units + 255) / 256, 4096), 256, 0, s>>>(out, x, f, units, (int)(T * dim / 8));
    return launch_status();
}
inline Geom attention_geom(const na1d_train_layer &l, int64_t N, int64_t T, Layout &in, Layout &out) {
    Geom g;
    const int64_t C = l.dim;
    g.B = N * l.heads, g.T = T, g.H = l.heads, g.C = l.dim / l.heads, g.W = l.window ? l.window : 1, g.L = l.window ? l.left : 0;
    in = Layout{T * 3 * C, g.C, 3 * C}, out = Layout{T * C, g.C, C};
    if (l.window) set_dilation(g, l.dilation);
    in.row *= g.dilation, out.row *= g.dilation;
    return g;
}

template <class DT> int norm_apply(const na1d_train_layer &l, int which, char *y, const char *x, float *mean, float *rstd, int64_t M, const char *add, int64_t T, hipStream_t s) {
    const Chunks c = bn_chunks(M, kBnForwardChunks);
    const na1d_train_norm &n = l.norm[which];
    bn_apply_kernel<DT><<<dim3((unsigned)(l.dim / kBnCols), (unsigned)c.count), kBnThreads, 0, s>>>(
        BnApply{y, x, n.batch_mean, n.batch_var, n.weight, n.bias, mean, rstd, n.batches, n.eps, (int)M, l.dim, c.rows, add, (int)T});
    return launch_status();
}
int to_channels(const na1d_train_layer &l, void *out, const void *x, int64_t N, int64_t T, hipStream_t s) {
    to_channels_kernel<<<dim3((unsigned)((T + 63) / 64), (unsigned)(l.dim / 64), (unsigned)N), 256, 0, s>>>((uint16_t *)out, (const char *)x, (int)T, l.dim);
    return launch_status();
}
// The product a.x . W, which is the gradient dy of a norm's output (in a.out), and the norm's backward.
// The product's ends sum up what the norm needs, a row of sums for every block of 64 or 32 tokens, which the kernel behind adds up
// again (up to kBnParts of them: 0.5 MB from L2); with more blocks of rows a kernel of its own does.
// 12800 tokens, us: products of 12.5 and sums of 7.8 -> products of 14.9; a step of MFA 4x4 at 128 x 2 s 9070 -> 8700.
template <class DT>
int product_and_norm_backward(Gemm a, const na1d_train_layer &l, int which, char *dx, const char *x, const char *add, const float *mean, const float *rstd, float *part,
                              hipStream_t s) {
    const Chunks c = bn_chunks(a.M, kBnChunks);
    const dim3 grid((unsigned)(l.dim / kBnCols), (unsigned)c.count);
    float *part_dyx = part + (int64_t)kBnParts * l.dim;
    const int rows = gemm_rows(a.M, a.outputs);
    int chunks = (a.M + rows - 1) / rows;
    if (chunks <= kBnParts) {
        a.aux = x, a.mean = mean, a.part_dy = part, a.part_dyx = part_dyx;
        NA1D_TRY(launch_gemm<DT, kNormBack>(a, s));
    } else {
        NA1D_TRY(launch_gemm<DT, kStore>(a, s));
        bn_bwd_sums_kernel<DT><<<grid, kBnThreads, 0, s>>>(part, part_dyx, a.out, x, mean, a.M, l.dim, c.rows);
        NA1D_TRY(launch_status());
        chunks = c.count;
    }
    const na1d_train_norm &n = l.norm[which];
    bn_bwd_apply_kernel<DT><<<grid, kBnApplyThreads, 0, s>>>(BnBackward{dx, a.out, x, add, part, part_dyx, n.weight, mean, rstd, n.dweight, n.dbias, a.M, l.dim, c.rows, chunks});
    return launch_status();
}

// part 0: up to x1, which also goes to `out` as [N, dim, T]; part 1: from x1 and its statistics on
template <class DT> int forward(const na1d_train_layer &l, int half, char *out, const char *x, char *saved, char *ws, int64_t N, int64_t T, hipStream_t s) {
    const int64_t M = N * T;
    const Saved o(l, N, T);
    const ForwardScratch f(l, T);
    auto stat = [&](int i) { return reinterpret_cast<float *>(saved + o.stats[i]); };
    Pack p{};
    for (int j = 0; j < kWeights; ++j) {
        p.w[j] = weight_of(l, j);
        p.plain[j] = ws + f.plain[j], p.turned[j] = j < 4 ? saved + o.turned[j] : nullptr, p.bias[j] = reinterpret_cast<float *>(ws + f.bias[j]);
        p.first[j + 1] = p.first[j] + p.w[j].outputs / 32 * (p.w[j].inputs / 32);
    }
    Gemm a{};
    a.M = (int)M, a.T = (int)T, a.T_magic = div_magic(T);
    auto product = [&](int j, const char *in, char *to) {
        a.x = in, a.w = p.plain[j], a.bias = p.bias[j], a.out = to, a.inputs = p.w[j].inputs, a.outputs = p.w[j].outputs;
        a.late = l.ordered || (l.late && j % 2 == 0);
    };
    if (half) {
        NA1D_TRY(norm_apply<DT>(l, 1, saved + o.y2, saved + o.x1, stat(2), stat(3), M, nullptr, T, s));
        product(2, saved + o.y2, saved + o.g);
        a.out2 = saved + o.h;
        NA1D_TRY(launch_gemm<DT, kGelu>(a, s));
        product(3, saved + o.g, out);
        a.aux = saved + o.x1, a.sample_scale = l.scale_mlp;
        return launch_gemm<DT, kResidual>(a, s);
    }
    pack_kernel<DT><<<(unsigned)p.first[kWeights], 256, 0, s>>>(p);
    NA1D_TRY(launch_status());
    if (!l.window) {
        a.M = (int)T;
        product(4, (const char *)l.pos, ws + f.pos);
        NA1D_TRY(launch_gemm<DT, kStore>(a, s));
        a.M = (int)M;
    }
    NA1D_TRY(norm_apply<DT>(l, 0, saved + o.y1, x, stat(0), stat(1), M, l.window ? nullptr : ws + f.pos, T, s));
    product(0, saved + o.y1, saved + o.qkv);
    NA1D_TRY(launch_gemm<DT, kBias>(a, s));
    Layout in, outl;
    const Geom g = attention_geom(l, N, T, in, outl);
    const char *q = saved + o.qkv, *k = q + 2 * l.dim, *v = k + 2 * l.dim;
    float *lse = reinterpret_cast<float *>(saved + o.lse);
    int st = !l.window ? global_fwd(saved + o.attn, lse, q, k, v, nullptr, g, in, outl, l.scale, DT::tag, s)
                       : fused_fwd(saved + o.attn, lse, q, k, v, l.rpb, nullptr, g, in, outl, l.scale, DT::tag, s);
    if (st == NA1D_ERR_UNSUPPORTED && l.window) st = wide_fwd(saved + o.attn, lse, q, k, v, l.rpb, nullptr, g, in, outl, l.scale, DT::tag, s);
    NA1D_TRY(st);
    product(1, saved + o.attn, saved + o.x1);
    a.aux = x, a.sample_scale = l.scale_attn;
    NA1D_TRY(launch_gemm<DT, kResidual>(a, s));
    return to_channels(l, out, saved + o.x1, N, T, s);
}

template <class DT>
int backward(const na1d_train_layer &l, char *dx, const char *dout, const char *x, const char *saved, char *ws, int64_t N, int64_t T, hipStream_t s) {
    const int64_t M = N * T;
    const Saved o(l, N, T);
    const BackwardScratch b(l, N, T);
    auto stat = [&](int i) { return reinterpret_cast<const float *>(saved + o.stats[i]); };
    float *part = reinterpret_cast<float *>(ws + b.part);
    Gemm a{};
    a.M = (int)M, a.T = (int)T, a.T_magic = div_magic(T);
    auto turned = [&](int j, const char *dy, char *to) {
        const Weight w = weight_of(l, j);
        a.x = dy, a.w = saved + o.turned[j], a.out = to, a.inputs = w.outputs, a.outputs = w.inputs;
    };
    const char *dz = dout;
    if (l.scale_mlp) {
        NA1D_TRY(scale_rows<DT>(ws + b.dz, dout, l.scale_mlp, N, T, l.dim, s));
        dz = ws + b.dz;
    }
    turned(3, dz, ws + b.dh);
    a.aux = saved + o.h;
    NA1D_TRY(launch_gemm<DT, kGeluBack>(a, s));
    turned(2, ws + b.dh, ws + b.dy);
    NA1D_TRY(product_and_norm_backward<DT>(a, l, 1, ws + b.dx1, saved + o.x1, dout, stat(2), stat(3), part, s));
    const char *ds = ws + b.dx1;
    if (l.scale_attn) {
        NA1D_TRY(scale_rows<DT>(ws + b.ds, ds, l.scale_attn, N, T, l.dim, s));
        ds = ws + b.ds;
    }
    turned(1, ds, ws + b.dattn);
    NA1D_TRY(launch_gemm<DT, kStore>(a, s));
    Layout in, outl;
    const Geom g = attention_geom(l, N, T, in, outl);
    const int64_t step = 2 * l.dim;
    const char *q = saved + o.qkv;
    char *dq = ws + b.dqkv;
    const float *lse = reinterpret_cast<const float *>(saved + o.lse);
    int st = !l.window ? global_bwd(dq, dq + step, dq + 2 * step, reinterpret_cast<float *>(ws + b.delta), q, q + step, q + 2 * step, saved + o.attn, ws + b.dattn,
                                    lse, nullptr, g, in, outl, l.scale, DT::tag, s)
                       : fused_bwd(dq, dq + step, dq + 2 * step, l.drpb, q, q + step, q + 2 * step, nullptr, ws + b.dattn, lse, l.rpb, nullptr, g, in, outl, l.scale, DT::tag,
                       nullptr, 0, s);
    if (st == NA1D_ERR_UNSUPPORTED && l.window)
        st = wide_bwd(dq, dq + step, dq + 2 * step, l.drpb, q, q + step, q + 2 * step, ws + b.dattn, lse, l.rpb, nullptr, g, in, outl, l.scale, DT::tag, nullptr, 0, s);
    NA1D_TRY(st);
    turned(0, ws + b.dqkv, ws + b.dy);
    NA1D_TRY(product_and_norm_backward<DT>(a, l, 0, dx, x, ws + b.dx1, stat(0), stat(1), part, s));
    if (!l.window) {
        const int64_t units = T * l.dim / 8;
        sum_samples_kernel<DT><<<(unsigned)((units + 31) / 32), 256, 0, s>>>(ws + b.dpos, ws + b.dy, (int)N, units);
        NA1D_TRY(launch_status());
    }
    const GradPlan plan(l, M);
    Grads ga{};
    Fold fo{};
    const char *dys[kWeights] = {ws + b.dqkv, ds, ws + b.dh, dz, ws + b.dpos};
    const char *xs[kWeights] = {saved + o.y1, saved + o.attn, saved + o.y2, saved + o.g, (const char *)l.pos};
    for (int j = 0; j < kWeights; ++j) {
        fo.w[j] = weight_of(l, j);
        ga.job[j] = GradJob{dys[j], xs[j], fo.w[j].outputs, fo.w[j].inputs, (int)(j < 4 ? M : T), plan.first[j], plan.part[j]};
        fo.part[j + 1] = plan.part[j + 1];
    }
    ga.partial = reinterpret_cast<float *>(ws + b.grads);
    ga.stride = fo.stride = plan.part[kWeights];
    ga.rows = plan.rows, ga.blocks = plan.blocks;
    fo.partial = ga.partial, fo.splits = plan.splits;
    const size_t lds = (size_t)4 * kGradRows * kGradTile * 2;
    if (!allow_lds(grad_kernel<DT>, lds)) return NA1D_ERR_LAUNCH;
    grad_kernel<DT><<<(unsigned)(plan.blocks * plan.splits), kThreads, lds, s>>>(ga);
    NA1D_TRY(launch_status());
    grad_fold_kernel<<<(unsigned)((plan.part[kWeights] / 4 + 255) / 256), 256, 0, s>>>(fo);
    return launch_status();
}

bool layer_ok(const na1d_train_layer &l, int64_t N, int64_t T) {
    if (l.dim < 256 || l.dim % 256 || l.dim > 2048 || l.hidden < 256 || l.hidden % 256 || l.hidden > 8192) return false;
    if (l.heads < 1 || l.dim % l.heads || l.dim / l.heads % 8 || l.dim / l.heads > 128) return false;
    if (l.groups < 1 || l.dim % l.groups || l.dim / l.groups % 32 || l.hidden % l.groups || l.hidden / l.groups % 32) return false;
    if (l.window < 0 || l.window > NA1D_MAX_WINDOW || (l.window && (l.left < 0 || l.left >= l.window)) || l.dilation < 1 || (!l.window && l.dilation > 1)) return false;
    // offsets inside an utterance, and what the attention kernels' launches count, stay in the reach of 32 bits
    if (N < 1 || T < 1 || N > 65535 || T > (1 << 16) || N * T > (1 << 20)) return false;     // samples: a grid's third dimension
    const int64_t M = N * T, most = 1ll << 31;
    if (T * 3 * l.dim > (1 << 29) || M * T >= most || l.dilation > 64) return false;
    if (l.heads * M * l.heads >= most || l.heads * M * (T / 32 + 1) >= most || l.heads * M * l.dilation >= most) return false;
    return N * T >= 2;          // variance of one row
}
int64_t saved_bytes(const na1d_train_layer &l, int64_t N, int64_t T) { return Saved(l, N, T).bytes; }
int64_t scratch_bytes(const na1d_train_layer &l, int64_t N, int64_t T, bool backward) {
    return backward ? BackwardScratch(l, N, T).bytes : ForwardScratch(l, T).bytes;
}
int run_forward(const na1d_train_layer &l, int half, void *out, const void *x, void *saved, void *ws, int64_t N, int64_t T, hipStream_t s) {
    return l.dtype == NA1D_BF16 ? forward<BF16>(l, half, (char *)out, (const char *)x, (char *)saved, (char *)ws, N, T, s)
                                : forward<FP16>(l, half, (char *)out, (const char *)x, (char *)saved, (char *)ws, N, T, s);
}
int run_backward(const na1d_train_layer &l, void *dx, const void *dout, const void *x, const void *saved, void *ws, int64_t N, int64_t T, hipStream_t s) {
    return l.dtype == NA1D_BF16 ? backward<BF16>(l, (char *)dx, (const char *)dout, (const char *)x, (const char *)saved, (char *)ws, N, T, s)
                                : backward<FP16>(l, (char *)dx, (const char *)dout, (const char *)x, (const char *)saved, (char *)ws, N, T, s);
}

}  // namespace train
}  // namespace na1d
