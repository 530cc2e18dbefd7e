// What the token-local kernels of the speaker-embedding models share: everything of an encoder layer that is not
// attention works on one token at a time, so a workgroup that holds a few tokens in LDS can run a layer's output
// projection, its MLP and the next layer's qkv projection without touching memory in between.
#pragma once

#include "na1d_mfma_core.h"

namespace na1d {
namespace enc {

using namespace mfma;

constexpr int kDim = 256;            // channels of a token
constexpr int kHidden = 1024;        // channels of the MLP's hidden layer
constexpr int kRow = 2 * kDim;       // bytes of a token's row in LDS: the staged tiles are all this wide
constexpr int kFrag = 1024;          // bytes of a weight fragment: 16 outputs x 32 inputs, in the order of the lanes

// A tile of token rows in LDS: 512 bytes a row, its 16-byte units XOR-swizzled with the row's place in a 16-row tile
// (the rows an operand read touches land in distinct banks, and the swizzle is the same for every tile).
__device__ inline int tile_addr(int row, int unit) { return row * kRow + ((unit ^ (row & 15)) << 4); }

// A lane's place in such a tile, as the operand of a product (unit g of row n) and for four channels of its results (channels
// 4g .. 4g+3); the units that a step or a tile of outputs lies further on only turn bits over: one instruction by a constant.
__device__ inline int operand_lane(int n, int g) { return n * kRow + ((g ^ n) << 4); }
__device__ inline int result_lane(int n, int g) { return n * kRow + (((g >> 1) ^ n) << 4) + (g & 1) * 8; }

// Copy `rows` (a multiple of 16) token rows of `width` bytes, `pitch` bytes apart, into such a tile with loads that write
// LDS directly; the resource ends behind the last row there is, and bytes past a row's width arrive as zeros.
template <int ROWS, int NW, int AUX>
__device__ inline void stage_tokens(Rsrc src, LDS_PTR(char) tile, int pitch, int width, int wave, int lane) {
    constexpr int kChunks = ROWS * kRow / kChunk;          // two rows each
#pragma unroll
    for (int j = 0; j < (kChunks + NW - 1) / NW; ++j) {
        const int c = j * NW + wave, row = 2 * c + (lane >> 5);
        const int at = ((lane & 31) ^ (row & 15)) * 16;
        if (kChunks % NW == 0 || c < kChunks) load_to_lds<16, AUX>(src, tile + c * kChunk, at < width ? row * pitch + at : kNowhere);
    }
}

// Where a product's operands are: step s of output tile j of this wave multiplies weight fragment
// first + j * stride + skip(j) + s by the tokens' 32 channels number x0 + skip(j) + s.  `skip` is there for grouped
// projections (block-diagonal weights), whose output tiles start at inputs of their own: SKIP = 0: all at the same,
// 1: two steps later from tile to tile, 2: odd tiles four steps later.
template <int TILES, int STEPS, int SKIP = 0> struct Product {
    static constexpr int kTiles = TILES, kSteps = STEPS, kSkip = SKIP;
    Rsrc w;
    int first, stride, x0;               // wave-uniform, in fragments / steps
    static __device__ constexpr int skip(int j) { return SKIP == 1 ? 2 * j : SKIP == 2 ? 4 * (j & 1) : 0; }
    __device__ inline u32x4 load(int j, int s, int lane16) const {
        return __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(w, lane16, (first + j * stride + skip(j) + s) * kFrag, 0));
    }
};
__device__ inline Rsrc weight_rsrc(const char *w, int outputs, int inputs) { return make_rsrc(w, outputs * inputs * 2); }

// The weight fragments on their way: they come straight from memory into registers (packed so that a fragment is one
// contiguous kilobyte; every workgroup reads the same ones, so they sit in the L2s), PF steps ahead of their use, also
// across the border of two products: while one runs out its slots fill with the next one's first steps.
template <int NTW, int PF> struct Ring {
    u32x4 w[PF][NTW];
    template <class P> __device__ inline void fill(const P &p, int slot, int s, int lane16) {
#pragma unroll
        for (int j = 0; j < P::kTiles; ++j) w[slot][j] = p.load(j, s, lane16);
    }
    template <class P> __device__ inline void begin(const P &p, int lane16) {
#pragma unroll
        for (int s = 0; s < PF; ++s)
            if (s < P::kSteps) fill(p, s, s, lane16);
    }
};

// acc[j][i] += W[tile j of this wave] . X[token tile i]^T; lane (n, g) ends up with outputs 4g .. 4g+3 of each tile for
// token n of each token tile.  The ring holds this product's first PF steps on entry and `next`'s on exit.
template <class DT, int MT, int NTW, int PF, class P, class Q>
__device__ inline void multiply(f32x4 (&acc)[P::kTiles][MT], Ring<NTW, PF> &ring, const P &p, const Q &next, LDS_PTR(char) tile,
                                int n, int g, int lane16) {
    static_assert(P::kSteps % PF == 0 || P::kSteps < PF, "slots of a product");
    if constexpr (P::kSteps < PF) {
#pragma unroll
        for (int s = P::kSteps; s < PF; ++s)
            if (s < Q::kSteps) ring.fill(next, s, s, lane16);
    }
    // Rows are read one turn (a step, or a tile of it where tiles differ in their inputs) ahead and no further: left to itself
    // the scheduler reads a whole product's rows at its start, which takes the registers of the waves that would hide the rest.
    // The products stay in their turn too, so that a slot's next weights set out as soon as it is free: with products that pass
    // the barrier the loads collect behind them, down to a wait right behind a load (dense layers of 64000 tokens 131 -> 113 us,
    // 25600: 60 -> 55, 16 rows to a workgroup as before).
    constexpr int kPerStep = P::kSkip ? P::kTiles : 1, kTurns = P::kSteps * kPerStep;
    const int x_lane = operand_lane(n, g);
    u32x4 x[2][MT];
    auto read = [&](int turn) {
        LDS_PTR(char) at = tile + (x_lane ^ 64 * (p.x0 + P::skip(turn % kPerStep) + turn / kPerStep));
#pragma unroll
        for (int i = 0; i < MT; ++i) x[turn & 1][i] = *reinterpret_cast<LDS_PTR(u32x4)>(at + i * 16 * kRow);
    };
    read(0);
#pragma unroll
    for (int turn = 0; turn < kTurns; ++turn) {
        const int s = turn / kPerStep, j0 = turn % kPerStep;
        if (turn + 1 < kTurns) read(turn + 1);
        __builtin_amdgcn_sched_barrier(0x406);       // only other arithmetic passes
#pragma unroll
        for (int j = j0; j < (P::kSkip ? j0 + 1 : P::kTiles); ++j)
#pragma unroll
            for (int i = 0; i < MT; ++i) acc[j][i] = Mma<DT>::k32(ring.w[s % PF][j], x[turn & 1][i], acc[j][i]);
        if (j0 + 1 < kPerStep) continue;
        if (s + PF < P::kSteps) {
            ring.fill(p, s % PF, s + PF, lane16);
        } else {
            const int t = P::kSteps < PF ? s : s + PF - P::kSteps;
            if (t < Q::kSteps) ring.fill(next, s % PF, t, lane16);
        }
    }
}
// The same over a number of steps known at run time, from LDS rows that are still on their way: the first weights set out
// before the wait for the rows.
template <class DT, int MT, int NTW, int PF, class P>
__device__ inline void multiply_all(f32x4 (&acc)[NTW][MT], Ring<NTW, PF> &ring, const P &p, int steps, LDS_PTR(char) tile, int n, int g, int lane16) {
#pragma unroll
    for (int u = 0; u < PF; ++u)
        if (u < steps) ring.fill(p, u, u, lane16);
    wait_direct();
    barrier_lds();
    const int x_lane = operand_lane(n, g);
#pragma unroll 1
    for (int s0 = 0; s0 < steps; s0 += PF) {
#pragma unroll
        for (int u = 0; u < PF; ++u) {
            const int s = s0 + u;
            if (s >= steps) break;
            LDS_PTR(char) at = tile + (x_lane ^ 64 * (p.x0 + s));
            u32x4 x[MT];
#pragma unroll
            for (int i = 0; i < MT; ++i) x[i] = *reinterpret_cast<LDS_PTR(u32x4)>(at + i * 16 * kRow);
#pragma unroll
            for (int j = 0; j < NTW; ++j)
#pragma unroll
                for (int i = 0; i < MT; ++i) acc[j][i] = Mma<DT>::k32(ring.w[u][j], x[i], acc[j][i]);
            if (s + PF < steps) ring.fill(p, u, s + PF, lane16);
        }
    }
}
template <int NTW, int MT> __device__ inline void clear(f32x4 (&acc)[NTW][MT]) {
#pragma unroll
    for (int j = 0; j < NTW; ++j)
#pragma unroll
        for (int i = 0; i < MT; ++i) acc[j][i] = f32x4{0.f, 0.f, 0.f, 0.f};
}

// Two 16-bit values of a register as floats.
template <class DT> __device__ inline f32x2 widen(uint32_t w);
template <> __device__ inline f32x2 widen<BF16>(uint32_t w) {
    return f32x2{__uint_as_float(w << 16), __uint_as_float(w & 0xffff0000u)};
}
template <> __device__ inline f32x2 widen<FP16>(uint32_t w) {
    return __builtin_convertvector(__builtin_bit_cast(f16x2, w), f32x2);
}
template <class DT> __device__ inline f32x4 widen4(u32x2 w) {
    const f32x2 a = widen<DT>(w.x), b = widen<DT>(w.y);
    return f32x4{a.x, a.y, b.x, b.y};
}
template <class DT> __device__ inline u32x2 narrow4(f32x4 v) { return u32x2{Mma<DT>::pack(v[0], v[1]), Mma<DT>::pack(v[2], v[3])}; }

// x * Phi(x), the exact (erf) GELU, as max(x, 0) - |x| Phi(-|x|) for either sign.  The base-2 logarithm of Phi(-a) is a smooth
// function that a polynomial of degree 8 follows: -1 at 0 exactly, so that small values keep their digits, beyond that least
// maximum of the error times max(a Phi(-a), 0.8 exp(-(a / 0.8)^2)); its leading coefficient is negative, so the tail vanishes.
// Error at fp32 against 64 bits, and in brackets by formula 7.1.26 of Abramowitz and Stegun's handbook, which takes a reciprocal
// too: 2.8e-7 at most (3.3e-7), most of it the result's own rounding; 2.4e-7 of the value below 0.1 (5.7e-7); rms for
// arguments of deviation 0.1, 0.3, 1 and 4: 3.9e-9, 1.3e-8, 4.7e-8, 6.9e-8 (7.4e-9, 2.0e-8, 5.4e-8, 9.9e-8).  Degree 7, with a
// constant of -0.9999923, saves 0.5 to 1 % of a pass and is off by 5.4e-6 of every small value.
constexpr float kGelu[] = {-1.f, -1.1511104e+00f, -4.5914903e-01f, -5.2711148e-02f, 7.413445e-03f, -4.2505088e-04f, -6.2449646e-05f, 1.3129477e-05f, -6.7946235e-07f};
__device__ inline float gelu(float x) {
    constexpr int kDegree = sizeof(kGelu) / sizeof(float) - 1;
    const float a = __builtin_fabsf(x);
    float p = kGelu[kDegree];
#pragma unroll
    for (int k = kDegree - 1; k >= 0; --k) p = __builtin_fmaf(a, p, kGelu[k]);
    // The larger of x and 0 as a median: a maximum takes a second instruction that quiets signalling NaN (which the product does
    // here); with the compiler's two a pass over 25600 tokens is 1.5 % longer.
    return __builtin_fmaf(-a, __builtin_amdgcn_exp2f(p), __builtin_amdgcn_fmed3f(x, 0.f, 3.402823466e38f));
}

}  // namespace enc
}  // namespace na1d
