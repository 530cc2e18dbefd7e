// The token-local part of the speaker-embedding models (models/PCF_NATransformer.py, models/MFA_NATransformer.py) in
// inference on the matrix cores: projections, MLPs, residuals, patch embeddings.
#include "na1d_encoder.h"

namespace na1d {
namespace enc {

// Four floats that a caller may have put on any float.
__device__ inline f32x4 load4(const float *p) {
    typedef float on_any_float __attribute__((ext_vector_type(4), aligned(4)));
    return *reinterpret_cast<const on_any_float *>(p);
}

// What a batch norm with running statistics multiplies channels c .. c+3 by.  The few norms that no weight has been folded
// with are read as the module holds them, so that the next call sees what a program writes there.
__device__ inline f32x4 norm_gain(const na1d_encoder_norm &n, int c) {
    const f32x4 w = load4(n.weight + c), v = load4(n.var + c);
    f32x4 gain;
#pragma unroll
    for (int r = 0; r < 4; ++r) gain[r] = w[r] * __builtin_amdgcn_rsqf(v[r] + n.eps);
    return gain;
}

// =============================================================================
// Between two attentions
// =============================================================================
// One workgroup takes 16 * MT tokens through everything between the attention of one layer and that of the next:
//   x1 = x + proj(attention),  x2 = x1 + fc2(gelu(fc1(x1)))          the rest of the layer before   (`attn` != null)
//   x2 += embed(patches)                                             where a block takes its own embedding
//   qkv = x2 . Wqkv^T + b                                            the head of the next layer     (`qkv` != null)
// with batch norms folded into the projections behind them.  Tokens sit in two LDS tiles; the hidden layer passes
// through one of them 256 channels at a time and never exists in memory; the weights of a layer (1.6 MB) stream from L2.
struct LayerArgs {
    const char *attn, *x_in;
    const char *w_proj, *w_fc1, *w_fc2;
    const float *b_proj, *b_fc1, *b_fc2;
    char *block_out;                  // the layer's output where a block ends
    const char *patches, *w_embed;
    const float *b_embed;
    char *x_out;                      // the residual stream the next layer reads
    const char *w_qkv;
    const float *b_qkv;
    char *qkv;
    na1d_encoder_norm norm;           // dense layers: qkv of x * gain(norm) + posb[token's place] (posb != null)
    const float *posb;
    int x_in_pitch, block_pitch, patch_width, M, T;
    uint32_t T_magic;
    int tail_groups, head_groups;     // block-diagonal weights: 8, 4, 2; otherwise 1
    int large;                        // layer_kernel with three row tiles: the first so many workgroups have them, the others two
    char *x1;                         // split layers (part_kernel): [M, 256] ...
    float *parts;                     // ... and what each quarter of the hidden channels adds, [4, M, 256]
};

// Grouped projections (PCF-NAT: blocks of 8, 4, 2 and 1 groups) have block-diagonal weights; which 32-input steps of an
// output tile are not zero follows from the number of groups G alone (any other number: all of them, as with one group):
//   output projection, fc1   outputs of a group see the 256 / G inputs of the same group
//   fc2                      256 hidden channels (chunk c) reach kOut outputs, from kOut * (c * kOut / 256 ...) on
//   qkv                      output f (head-major order, see _qkv_channel_order) sees group (f mod 256/G) / (256/G^2)
template <int G, int NW> struct Groups {
    static constexpr int kSize = kDim / G;                             // channels of a group
    static constexpr int NTW = 16 / NW, CW = 16 * NTW;                 // output tiles / channels a wave has of 256
    static constexpr int kProj = (kSize > CW ? kSize : CW) / 32;       // steps of the output projection (CW channels may touch several groups)
    static constexpr int kFc1 = kSize / 32;
    static constexpr int kOutTiles = G == 1 ? 16 : G == 2 ? 8 : 4;     // output tiles a chunk of 256 hidden channels reaches
    static constexpr int kSets = 16 / kOutTiles;                       // different ones
    static constexpr int kPer = kOutTiles >= NW ? kOutTiles / NW : 1;  // of them to a wave
    static constexpr int kActive = kOutTiles < NW ? kOutTiles : NW;    // waves that have any
    static constexpr int kFc2 = G == 8 ? 4 : 8;
    static constexpr int kEach = 4 / kSets;                            // chunks that reach the same ones
    static constexpr int kQkv = G == 1 ? 8 : G == 4 ? 2 : 4;
    static constexpr int kQkvSkip = G == 4 ? 1 : G == 8 ? 2 : 0;
    using Proj = Product<NTW, kProj>;
    using Fc1 = Product<NTW, kFc1>;
    using Fc2 = Product<kPer, kFc2>;
    using Qkv = Product<NTW, kQkv, kQkvSkip>;
    static __device__ inline Proj proj(Rsrc w, int wave) {
        const int k0 = wave * CW / (32 * kProj) * kProj;
        return Proj{w, wave * NTW * 8 + k0, 8, k0};
    }
    static __device__ inline Fc1 fc1(Rsrc w, int c, int wave) {
        const int k0 = (256 * c + wave * CW) / (kHidden / G) * kFc1;
        return Fc1{w, (16 * c + wave * NTW) * 8 + k0, 8, k0};
    }
    static __device__ inline Fc2 fc2(Rsrc w, int c, int wave) {
        const int set = c * kSets / 4, tile = set * kOutTiles + wave * kPer;
        const int k0 = G == 8 ? wave / 2 * 4 : 0;
        return Fc2{w, tile * (kHidden / 32) + 8 * c + k0, kHidden / 32, k0};
    }
    static __device__ inline Qkv qkv(Rsrc w, int which, int wave) {
        const int k0 = G == 2 ? wave * CW % 128 / 64 * 4 : G == 4 ? wave * NTW % 4 * 2 : 0;
        return Qkv{w, (16 * which + wave * NTW) * 8 + k0, 8, k0};
    }
};

// Places of the biases in LDS, in floats.
constexpr int kBiasFc1 = 0, kBiasProj = kHidden, kBiasFc2 = kBiasProj + kDim, kBiasQkv = kBiasFc2 + kDim, kBias = kBiasQkv + 3 * kDim;
template <int MT> constexpr size_t layer_lds() { return (size_t)2 * 16 * MT * kRow + kBias * sizeof(float); }

// The number of groups as the kernels know it: every switch over it and every sum over its parts starts from this.
inline int known_groups(int groups) { return groups == 2 || groups == 4 || groups == 8 ? groups : 1; }

template <class DT, int MT, int NW, int PF, bool SPLIT, int QKV_AUX> struct LayerWave {
    static constexpr int NTW = 16 / NW, CW = 16 * NTW;
    const LayerArgs &a;
    LDS_PTR(char) p_lds;
    LDS_PTR(char) q_lds;
    LDS_PTR(float) b_lds;             // the projections' biases, kBias floats
    int wave, lane, n, g, lane16;
    Ring<NTW, PF> ring;

    // LDS place of channels c + 4g .. + 3 of token n (c: a multiple of 16, wave-uniform)
    __device__ inline LDS_PTR(u32x2) at(LDS_PTR(char) tile, int c, int i) const {
        return reinterpret_cast<LDS_PTR(u32x2)>(tile + (result_lane(n, g) ^ 2 * c) + i * 16 * kRow);
    }
    __device__ inline f32x4 bias(const float *b, int c) const { return load4(b + c + 4 * g); }
    __device__ inline f32x4 staged_bias(int c) const { return *reinterpret_cast<LDS_PTR(f32x4)>(b_lds + c + 4 * g); }

    // Biases come through LDS, and sums start at them: read from memory behind a product, a bias would have to wait for every
    // weight of the next product that is on its way (loads return in order).
    // The caller's own parameters may lie on any float (views of one flat buffer); those go a float to a lane.
    __device__ inline void stage_bias(const float *b, int count, int to) const {
        const Rsrc bs = make_rsrc(b, 4 * count);
        if ((uintptr_t)b & 15u) {
            for (int k = wave; k < count / 64; k += NW) load_to_lds<4, 0>(bs, (LDS_PTR(char))(b_lds + to + 64 * k), 256 * k + 4 * lane);
        } else {
            for (int k = wave; k < count / 256; k += NW) load_to_lds<16, kReadShared>(bs, (LDS_PTR(char))(b_lds + to + 256 * k), 1024 * k + lane16);
        }
    }
    __device__ inline void stage_tail_biases() const {
        stage_bias(a.b_proj, kDim, kBiasProj);
        stage_bias(a.b_fc1, kHidden, kBiasFc1);
        stage_bias(a.b_fc2, kDim, kBiasFc2);
    }
    __device__ inline void stage_qkv_bias() const {
        if (a.qkv) stage_bias(a.b_qkv, 3 * kDim, kBiasQkv);
    }
    template <int NTILES> __device__ inline void begin_sums(f32x4 (&acc)[NTILES][MT], int c) const {
#pragma unroll
        for (int j = 0; j < NTILES; ++j) {
            const f32x4 b = staged_bias(c + 16 * j);
#pragma unroll
            for (int i = 0; i < MT; ++i) acc[j][i] = b;
        }
    }

    // attention rows in p_lds, x in q_lds (on their way) -> x1 in q_lds; the ring holds the start of fc1's chunk c
    template <int G> __device__ inline void project(Rsrc w1, int first_chunk) {
        using S = Groups<G, NW>;
        const auto proj = S::proj(weight_rsrc(a.w_proj, kDim, kDim), wave);
        ring.begin(proj, lane16);
        f32x4 hid[NTW][MT];
        wait_direct();
        barrier_lds();
        begin_sums(hid, kBiasProj + CW * wave);
        multiply<DT, MT>(hid, ring, proj, S::fc1(w1, first_chunk, wave), p_lds, n, g, lane16);
#pragma unroll
        for (int j = 0; j < NTW; ++j) {
            const int c = CW * wave + 16 * j;
#pragma unroll
            for (int i = 0; i < MT; ++i) *at(q_lds, c, i) = narrow4<DT>(hid[j][i] + widen4<DT>(*at(q_lds, c, i)));
        }
    }
    // 256 hidden channels: x1 in q_lds -> their share of the output in acc
    template <int G, int NA> __device__ inline void chunk(f32x4 (&acc)[NA][MT], Rsrc w1, Rsrc w2, int c, bool last) {
        using S = Groups<G, NW>;
        f32x4 hid[NTW][MT];
        begin_sums(hid, kBiasFc1 + 256 * c + CW * wave);
        barrier_lds();                           // x1 is whole (first round); every wave is done with the hidden channels before
        multiply<DT, MT>(hid, ring, S::fc1(w1, c, wave), S::fc2(w2, c, wave), q_lds, n, g, lane16);
#pragma unroll
        for (int j = 0; j < NTW; ++j) {
            const int ch = CW * wave + 16 * j;
#pragma unroll
            for (int i = 0; i < MT; ++i) {
                f32x4 h = hid[j][i];
#pragma unroll
                for (int r = 0; r < 4; ++r) h[r] = gelu(h[r]);
                *at(p_lds, ch, i) = narrow4<DT>(h);
            }
        }
        barrier_lds();
        if (S::kActive == NW || wave < S::kActive)
            multiply<DT, MT>(acc, ring, S::fc2(w2, c, wave), S::fc1(w1, last ? 0 : c + 1, wave), p_lds, n, g, lane16);
        else
            ring.begin(S::fc1(w1, last ? 0 : c + 1, wave), lane16);
    }
    // The rest of a layer of 8 or 4 groups, whose channels never meet before the next projection: a group is one wave's, or two
    // waves' that halve the tokens, from the output projection to x2, without a barrier.  Of every 32 hidden channels lane
    // (n, g) of two tiles' sums gets channels 8g .. 8g+3 and 8g+4 .. 8g+7 of token n (fc1's rows are taken in that order),
    // which rounded are the next product's operand as they stand.  Four groups' weights are read by two waves each, 0.6 MB
    // for 64 tokens, in the shadow of GELU, which bounds it (64 tokens alone on a CU: the layer's rest 15.6 -> 9 us).  In chunks of 256
    // hidden channels through LDS, all waves together: 16400 tokens 32.8 -> 30.7 us with 8 groups, 38.9 -> 35.2 with 4; 64000: 69.6 -> 65.8,
    // 81.4 -> 76.8.
    template <int G, int kTok> __device__ inline void tail_of_groups(int i0) {
        static_assert(NW == 8 && (G == 8 || G == 4), "a group to a wave, or to two");
        constexpr int kOut = G == 8 ? 2 : 4, kSteps = kOut / 2, kBlocks = 2 * kOut;     // tiles and steps of a group's channels; its hidden channels in blocks of 32
        constexpr int kAhead = MT > 2 ? 1 : G == 8 ? 4 : 2;                // blocks whose weights are on their way
        const int group = G == 8 ? wave : wave >> 1;
        const Rsrc wp = weight_rsrc(a.w_proj, kDim, kDim), w1 = weight_rsrc(a.w_fc1, kHidden, kDim), w2 = weight_rsrc(a.w_fc2, kDim, kHidden);
        auto load = [](Rsrc w, int at, int frag) { return __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(w, at, frag * kFrag, 0)); };
        int hidden_lane[2];                      // a lane's place in the two fragments of 32 rows of fc1
#pragma unroll
        for (int t = 0; t < 2; ++t) {
            const int row = 8 * (n >> 2) + (n & 3) + 4 * t;
            hidden_lane[t] = (row >> 4) * (kDim / 32) * kFrag + (g * 16 + (row & 15)) * 16;
        }
        u32x4 p_w[kSteps][kOut], fc1_w[kAhead][kSteps][2], fc2_w[kAhead][kOut];
        auto fill1 = [&](int slot, int b) {
#pragma unroll
            for (int s = 0; s < kSteps; ++s)
#pragma unroll
                for (int t = 0; t < 2; ++t) fc1_w[slot][s][t] = load(w1, hidden_lane[t], (2 * kBlocks * group + 2 * b) * (kDim / 32) + kSteps * group + s);
        };
        auto fill2 = [&](int slot, int b) {
#pragma unroll
            for (int j = 0; j < kOut; ++j) fc2_w[slot][j] = load(w2, lane16, (kOut * group + j) * (kHidden / 32) + kBlocks * group + b);
        };
#pragma unroll
        for (int s = 0; s < kSteps; ++s)
#pragma unroll
            for (int j = 0; j < kOut; ++j) p_w[s][j] = load(wp, lane16, (kOut * group + j) * (kDim / 32) + kSteps * group + s);
#pragma unroll
        for (int u = 0; u < kAhead; ++u) fill1(u, u), fill2(u, u);
        wait_direct();
        barrier_lds();
        const int x_lane = operand_lane(n, g);
        u32x4 x[kSteps][kTok];
        auto read = [&](LDS_PTR(char) tile) {
#pragma unroll
            for (int s = 0; s < kSteps; ++s)
#pragma unroll
                for (int i = 0; i < kTok; ++i) x[s][i] = *reinterpret_cast<LDS_PTR(u32x4)>(tile + (x_lane ^ 64 * (kSteps * group + s)) + (i0 + i) * 16 * kRow);
        };
        f32x4 acc[kOut][kTok];
        auto begin = [&](int bias_at) {
#pragma unroll
            for (int j = 0; j < kOut; ++j) {
                const f32x4 b = staged_bias(bias_at + 16 * (kOut * group + j));
#pragma unroll
                for (int i = 0; i < kTok; ++i) acc[j][i] = b;
            }
        };
        auto add_to_x = [&] {
#pragma unroll
            for (int j = 0; j < kOut; ++j)
#pragma unroll
                for (int i = 0; i < kTok; ++i) {
                    LDS_PTR(u32x2) to = at(q_lds, 16 * (kOut * group + j), i0 + i);
                    *to = narrow4<DT>(acc[j][i] + widen4<DT>(*to));
                }
        };
        read(p_lds);
        begin(kBiasProj);
#pragma unroll
        for (int s = 0; s < kSteps; ++s)
#pragma unroll
            for (int j = 0; j < kOut; ++j)
#pragma unroll
                for (int i = 0; i < kTok; ++i) acc[j][i] = Mma<DT>::k32(p_w[s][j], x[s][i], acc[j][i]);
        add_to_x();
        read(q_lds);                             // a wave's LDS operations keep their order
        begin(kBiasFc2);
#pragma unroll 1
        for (int b0 = 0; b0 < kBlocks; b0 += kAhead) {
#pragma unroll
            for (int u = 0; u < kAhead; ++u) {
                const int b = b0 + u, next = min(b + kAhead, kBlocks - 1);
                f32x4 hid[2][kTok];
#pragma unroll
                for (int t = 0; t < 2; ++t) {
                    const f32x4 from = *reinterpret_cast<LDS_PTR(f32x4)>(b_lds + kBiasFc1 + 32 * (kBlocks * group + b) + 8 * g + 4 * t);
#pragma unroll
                    for (int i = 0; i < kTok; ++i) hid[t][i] = from;
                }
#pragma unroll
                for (int s = 0; s < kSteps; ++s)
#pragma unroll
                    for (int t = 0; t < 2; ++t)
#pragma unroll
                        for (int i = 0; i < kTok; ++i) hid[t][i] = Mma<DT>::k32(fc1_w[u][s][t], x[s][i], hid[t][i]);
                fill1(u, next);
                __builtin_amdgcn_sched_barrier(0x406);       // see multiply()
                u32x4 h[kTok];
#pragma unroll
                for (int i = 0; i < kTok; ++i) {
#pragma unroll
                    for (int t = 0; t < 2; ++t)
#pragma unroll
                        for (int r = 0; r < 4; ++r) hid[t][i][r] = gelu(hid[t][i][r]);
                    const u32x2 lo = narrow4<DT>(hid[0][i]), hi = narrow4<DT>(hid[1][i]);
                    h[i] = u32x4{lo.x, lo.y, hi.x, hi.y};
                }
#pragma unroll
                for (int j = 0; j < kOut; ++j)
#pragma unroll
                    for (int i = 0; i < kTok; ++i) acc[j][i] = Mma<DT>::k32(fc2_w[u][j], h[i], acc[j][i]);
                fill2(u, next);
                __builtin_amdgcn_sched_barrier(0x406);
            }
        }
        add_to_x();
    }
    // the rest of the layer: -> x2 in q_lds
    template <int G> __device__ inline void tail() {
        if constexpr (G == 8)
            tail_of_groups<8, MT>(0);
        else if constexpr (G == 4 && MT % 2 == 0)
            tail_of_groups<4, MT / 2>((wave & 1) * MT / 2);
        else if constexpr (G == 4 && MT == 3) {  // two and one; waves w and w + 4 share a SIMD
            if ((wave ^ wave >> 2) & 1)
                tail_of_groups<4, 1>(2);
            else
                tail_of_groups<4, 2>(0);
        } else {
            tail_in_chunks<G>();
        }
    }
    // through LDS, 256 hidden channels at a time
    template <int G> __device__ inline void tail_in_chunks() {
        using S = Groups<G, NW>;
        const Rsrc w1 = weight_rsrc(a.w_fc1, kHidden, kDim), w2 = weight_rsrc(a.w_fc2, kDim, kHidden);
        project<G>(w1, 0);
        // Outputs that a later chunk adds nothing to are written at once, over x1: the chunks behind read other channels.
#pragma unroll 1
        for (int set = 0; set < S::kSets; ++set) {
            const int first = 16 * (set * S::kOutTiles + wave * S::kPer);
            f32x4 acc[S::kPer][MT];
            if (S::kActive == NW || wave < S::kActive) begin_sums(acc, kBiasFc2 + first);
#pragma unroll 1
            for (int k = 0; k < S::kEach; ++k) {
                const int c = set * S::kEach + k;
                chunk<G>(acc, w1, w2, c, c == 3);
            }
            if (S::kActive == NW || wave < S::kActive) {
#pragma unroll
                for (int t = 0; t < S::kPer; ++t)
#pragma unroll
                    for (int i = 0; i < MT; ++i) {
                        LDS_PTR(u32x2) x = at(q_lds, first + 16 * t, i);
                        *x = narrow4<DT>(acc[t][i] + widen4<DT>(*x));
                    }
            }
        }
    }

    // a quarter of it: x1 to memory (the first quarter's), the hidden channels' share of the output to `parts`
    template <int G> __device__ inline void tail_part(int c, int64_t m0, int rows) {
        using S = Groups<G, NW>;
        const Rsrc w1 = weight_rsrc(a.w_fc1, kHidden, kDim), w2 = weight_rsrc(a.w_fc2, kDim, kHidden);
        project<G>(w1, c);
        f32x4 acc[S::kPer][MT];
        clear(acc);
        chunk<G>(acc, w1, w2, c, true);
        const Rsrc d = make_rsrc(a.parts + ((int64_t)c * a.M + m0) * kDim, rows * kDim * 4);
        if (wave < S::kActive) {
#pragma unroll
            for (int t = 0; t < S::kPer; ++t) {
                const int ch = 16 * (c * S::kSets / 4 * S::kOutTiles + wave * S::kPer + t) + 4 * g;
#pragma unroll
                for (int i = 0; i < MT; ++i)
                    __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u32x4, acc[t][i]), d, (16 * i + n) * kDim * 4 + ch * 4, 0, 0);
            }
        }
        if (c == 0) write_rows(a.x1, m0, rows, kRow);
    }
    // and the quarters put together: -> x2 in q_lds.  A quarter reaches all outputs (one group), half of them (two) or its own
    // quarter; the PER that reach an output are fetched together.  (One after the other a dense layer's four took 2.8 of a
    // launch's 5.2 us.)
    __device__ inline void join(int64_t m0) {
        static_assert(Groups<8, NW>::kEach == 1 && Groups<4, NW>::kEach == 1 && Groups<2, NW>::kEach == 2 && Groups<1, NW>::kEach == 4, "quarters of an output");
        if (a.tail_groups >= 4)
            join_of<1>(m0);
        else if (a.tail_groups == 2)
            join_of<2>(m0);
        else
            join_of<4>(m0);
    }
    template <int PER> __device__ inline void join_of(int64_t m0) {
        const Rsrc xs = make_rsrc(a.x1, a.M * kRow), ps = make_rsrc(a.parts, 4 * a.M * (4 * kDim));
        u32x2 x[NTW][MT];
        f32x4 part[NTW][MT][PER], b[NTW];
#pragma unroll
        for (int j = 0; j < NTW; ++j) {
            const int c = CW * wave + 16 * j, first = c / (64 * PER) * PER;
#pragma unroll
            for (int i = 0; i < MT; ++i) {
                const int row = (int)m0 + 16 * i + n;                    // rows behind the last are not stored
                x[j][i] = __builtin_bit_cast(u32x2, __builtin_amdgcn_raw_buffer_load_b64(xs, row * kRow + 2 * c + 8 * g, 0, 0));
#pragma unroll
                for (int k = 0; k < PER; ++k)
                    part[j][i][k] = __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(ps, row * (4 * kDim) + 4 * c + 16 * g, (first + k) * a.M * (4 * kDim), 0));
            }
            b[j] = bias(a.b_fc2, c);
        }
#pragma unroll
        for (int j = 0; j < NTW; ++j)
#pragma unroll
            for (int i = 0; i < MT; ++i) {
                f32x4 v = part[j][i][0];
#pragma unroll
                for (int k = 1; k < PER; ++k) v += part[j][i][k];
                *at(q_lds, CW * wave + 16 * j, i) = narrow4<DT>(v + b[j] + widen4<DT>(x[j][i]));
            }
    }

    // QKV_AUX: how a head's rows go to memory.  A launch that is one round of workgroups writes them all at its end and then waits for what
    // the L2s still hold; streamed, they leave at once (five layers and their attentions, us in a trace: 4000 tokens 127 -> 124,
    // 6400: 141 -> 132, 10000: 198 -> 192, 12800: 205 -> 204, 16300: 233 -> 234).  With more tokens the attention behind loses what
    // it would find there (25600: 11 -> 12.8 each), and of few nothing is left to wait for.
    template <int G> __device__ inline void head(int64_t m0, int rows, int from, int to) {
        using S = Groups<G, NW>;
        const Rsrc w = weight_rsrc(a.w_qkv, 3 * kDim, kDim);
        ring.begin(S::qkv(w, from, wave), lane16);
        barrier_lds();
        const Rsrc qs = make_rsrc(a.qkv + m0 * (3 * kRow), rows * (3 * kRow));
#pragma unroll 1
        for (int which = from; which < to; ++which) {
            f32x4 acc[NTW][MT];
            begin_sums(acc, kBiasQkv + which * kDim + CW * wave);
            multiply<DT, MT>(acc, ring, S::qkv(w, which, wave), S::qkv(w, min(which + 1, 2), wave), q_lds, n, g, lane16);
            u32x2 o[MT][NTW];
#pragma unroll
            for (int j = 0; j < NTW; ++j)
#pragma unroll
                for (int i = 0; i < MT; ++i) o[i][j] = narrow4<DT>(acc[j][i]);
#pragma unroll
            for (int i = 0; i < MT; ++i)
                store_tile<CW, QKV_AUX>(qs, (16 * i + n) * (3 * kRow) + which * kRow + 2 * CW * wave, o[i], g, 2 * CW);
        }
    }

    // rows of q_lds to memory, whole
    __device__ inline void write_rows(char *dst, int64_t m0, int rows, int pitch) const {
        const Rsrc d = make_rsrc(dst + m0 * pitch, rows * pitch);
#pragma unroll
        for (int r = 0; r < 16 * MT * 32 / (64 * NW); ++r) {
            const int u = r * 64 * NW + wave * 64 + lane, row = u >> 5, unit = u & 31;
            const u32x4 v = *reinterpret_cast<LDS_PTR(u32x4)>(q_lds + tile_addr(row, unit));
            __builtin_amdgcn_raw_buffer_store_b128(v, d, row * pitch + unit * 16, 0, 0);
        }
    }
};

// Few tokens: a layer's weights (up to 1.6 MB) take a CU 21 us to read, so each 16 tokens go to four workgroups, one for
// every 256 hidden channels (each works out the output projection), and then to three, one each for q, k and v
// (layer_kernel with SPLIT, which puts the quarters together).  One 3 s utterance through MFA 4x4: 429 -> 313 us.
template <class DT, int NW, int PF>
__global__ void __launch_bounds__(64 * NW, 2)
part_kernel(LayerArgs a) {
    using W = LayerWave<DT, 1, NW, PF, true, 0>;
    extern __shared__ __attribute__((aligned(16))) char smem[];
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    W w{a, (LDS_PTR(char))smem, (LDS_PTR(char))smem + 16 * kRow, (LDS_PTR(float))(smem + 32 * kRow), wave, lane, lane & 15, lane >> 4, lane * 16};
    const int c = (int)(blockIdx.x & 3);
    const int64_t m0 = (int64_t)(blockIdx.x >> 2) * 16;
    const int rows = (int)min((int64_t)16, a.M - m0);
    const Rsrc as = make_rsrc(a.attn + m0 * kRow, rows * kRow), xs = make_rsrc(a.x_in + m0 * a.x_in_pitch, rows * a.x_in_pitch);
    stage_tokens<16, NW, kReadShared>(as, w.p_lds, kRow, kRow, wave, lane);
    stage_tokens<16, NW, kReadShared>(xs, w.q_lds, a.x_in_pitch, kRow, wave, lane);
    w.stage_bias(a.b_proj, kDim, kBiasProj);
    w.stage_bias(a.b_fc1 + 256 * c, 256, kBiasFc1 + 256 * c);
    switch (a.tail_groups) {
        case 8: w.template tail_part<8>(c, m0, rows); break;
        case 4: w.template tail_part<4>(c, m0, rows); break;
        case 2: w.template tail_part<2>(c, m0, rows); break;
        default: w.template tail_part<1>(c, m0, rows);
    }
}

// Waves on a SIMD.  SPARSE (blocks of 4 or 8 groups before the tile) and dense layers are kernels of their own, so that the
// former, whose sums never span chunks, run 64 tokens with eight waves of 128 registers: a layer of 64000 tokens 75 -> 70 us,
// its qkv projection 9 -> 4.5 of a workgroup's 35 us.  Dense layers need the registers for weights that set out four steps
// ahead (145 -> 134 us); with eight waves of 128 registers they spill 55 and a whole pass takes 3.72 instead of 3.37 ms.
constexpr int layer_waves(int MT, int NW) { return MT == 2 || (MT > 2 && NW == 8) ? 4 : 2; }

// SPLIT: one workgroup to each of q, k and v of a tile (or one where there is no projection behind); the layer before
// comes in quarters
template <class DT, int MT, int NW, int PF, bool SPLIT, bool SPARSE, int QKV_AUX>
__device__ inline void layer_tile(const LayerArgs &a, char *smem, int64_t m0, int mine, int each) {
    using W = LayerWave<DT, MT, NW, PF, SPLIT, QKV_AUX>;
    constexpr int NTW = W::NTW, CW = W::CW;
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    // p_lds: attention rows, then 256 hidden channels at a time, then patches; q_lds: x, then x1, then x2
    W w{a, (LDS_PTR(char))smem, (LDS_PTR(char))smem + 16 * MT * kRow, (LDS_PTR(float))(smem + 32 * MT * kRow), wave, lane, lane & 15, lane >> 4, lane * 16};
    const int rows = (int)min((int64_t)(16 * MT), a.M - m0);
    w.stage_qkv_bias();
    if (SPLIT && a.attn) {
        w.join(m0);
        wait_direct();                               // qkv's biases
        if (a.block_out && mine == 0) {
            barrier_lds();
            w.write_rows(a.block_out, m0, rows, a.block_pitch);
        }
    } else if (a.attn) {
        const Rsrc as = make_rsrc(a.attn + m0 * kRow, rows * kRow), xs = make_rsrc(a.x_in + m0 * a.x_in_pitch, rows * a.x_in_pitch);
        stage_tokens<16 * MT, NW, kReadOnce>(as, w.p_lds, kRow, kRow, wave, lane);
        stage_tokens<16 * MT, NW, kReadOnce>(xs, w.q_lds, a.x_in_pitch, kRow, wave, lane);
        w.stage_tail_biases();
        if constexpr (SPARSE) {
            if (a.tail_groups == 8)
                w.template tail<8>();
            else
                w.template tail<4>();
        } else {
            if (a.tail_groups == 2)
                w.template tail<2>();
            else
                w.template tail<1>();
        }
        if (a.block_out) {
            barrier_lds();
            w.write_rows(a.block_out, m0, rows, a.block_pitch);
        }
    }
    if (!a.qkv) return;
    if (a.patches) {
        if (a.attn && !SPLIT) barrier_lds();         // every wave is done with the hidden channels
        const Rsrc es = make_rsrc(a.patches + m0 * a.patch_width, rows * a.patch_width);
        stage_tokens<16 * MT, NW, kReadShared>(es, w.p_lds, a.patch_width, a.patch_width, wave, lane);
        const int ks_all = a.patch_width / 64;       // steps of 32 inputs
        const Rsrc we = weight_rsrc(a.w_embed, kDim, a.patch_width / 2);
        f32x4 acc[NTW][MT];
#pragma unroll
        for (int j = 0; j < NTW; ++j) {
            const int c = CW * wave + 16 * j;
            const f32x4 b = w.bias(a.b_embed, c);
#pragma unroll
            for (int i = 0; i < MT; ++i) acc[j][i] = a.attn ? widen4<DT>(*w.at(w.q_lds, c, i)) + b : b;
        }
        multiply_all<DT, MT>(acc, w.ring, Product<NTW, 1>{we, wave * NTW * ks_all, ks_all, 0}, ks_all, w.p_lds, w.n, w.g, w.lane16);
#pragma unroll
        for (int j = 0; j < NTW; ++j)
#pragma unroll
            for (int i = 0; i < MT; ++i) *w.at(w.q_lds, CW * wave + 16 * j, i) = narrow4<DT>(acc[j][i]);
    }
    if (a.x_out && mine == 0) {
        barrier_lds();
        w.write_rows(a.x_out, m0, rows, kRow);
    }
    if (a.posb) {
        f32x4 gain[NTW];
#pragma unroll
        for (int j = 0; j < NTW; ++j) gain[j] = norm_gain(a.norm, CW * wave + 16 * j + 4 * w.g);
        barrier_lds();
        const uint32_t first = (uint32_t)m0 % (uint32_t)a.T;     // place of the tile's first token in its utterance
#pragma unroll
        for (int i = 0; i < MT; ++i) {
            const uint32_t m = first + 16 * i + w.n;             // below T + 64
            const uint32_t t = m - div_by(m, a.T, a.T_magic) * a.T;
            const float *pos = a.posb + (int64_t)t * kDim;
#pragma unroll
            for (int j = 0; j < NTW; ++j) {
                const int c = CW * wave + 16 * j;
                *w.at(w.q_lds, c, i) = narrow4<DT>(widen4<DT>(*w.at(w.q_lds, c, i)) * gain[j] + w.bias(pos, c));
            }
        }
    }
    switch (a.head_groups) {
        case 8: w.template head<8>(m0, rows, mine, each == 3 ? mine + 1 : 3); break;
        case 4: w.template head<4>(m0, rows, mine, each == 3 ? mine + 1 : 3); break;
        case 2: w.template head<2>(m0, rows, mine, each == 3 ? mine + 1 : 3); break;
        default: w.template head<1>(m0, rows, mine, each == 3 ? mine + 1 : 3);
    }
}
template <class DT, int MT, int NW, int PF, bool SPLIT, bool SPARSE>
__global__ void __launch_bounds__(64 * NW, layer_waves(MT, NW))
layer_kernel(LayerArgs a) {
    extern __shared__ __attribute__((aligned(16))) char smem[];
    const int each = SPLIT && a.qkv ? 3 : 1, mine = each == 3 ? (int)(blockIdx.x % 3u) : 0;
    const int tile = (int)(blockIdx.x / (uint32_t)each);
    if constexpr (MT == 3)
        if (tile >= a.large) return layer_tile<DT, 2, NW, PF, SPLIT, SPARSE, 0>(a, smem, (int64_t)16 * (2 * tile + a.large), mine, each);
    layer_tile<DT, MT, NW, PF, SPLIT, SPARSE, !SPLIT && MT <= 2 ? kStoreAux : 0>(a, smem, (int64_t)16 * MT * tile, mine, each);
}

// tanh(x) = 1 - 2 / (1 + exp(2x)); its series where that would cancel
__device__ inline float tanh_of(float x) {
    const float t = 1.f - 2.f * __builtin_amdgcn_rcpf(1.f + __builtin_amdgcn_exp2f(x * (2.f * kLog2e)));
    const float u = x * x;
    return __builtin_fabsf(x) < 0.0625f ? x * __builtin_fmaf(u, __builtin_fmaf(u, 2.f / 15.f, -1.f / 3.f), 1.f) : t;
}

// =============================================================================
// Plain projections: out[m, o] = f(X[m, :] . W[o, :])
// =============================================================================
enum LinearEnd {
    kAffine,          // + bias, as fp32
    kShift,           // + what a norm adds, as fp32
    kEmbedding,       // + bias, 16-bit
    kReluNorm,        // relu(. + bias) * scale + offset, 16-bit
    kTanhNorm,        // tanh(relu(. + add[m / T]) * scale + offset), 16-bit
};
struct LinearArgs {
    const char *x, *w;
    char *out;
    const float *bias, *scale, *offset;
    int x_pitch, out_pitch, inputs, outputs, M, T;      // T: rows that share a row of `bias` (kTanhNorm)
    na1d_encoder_norm norm;                             // kShift
};
template <class DT, LinearEnd END>
__device__ inline f32x4 ended(const LinearArgs &a, int64_t m, int c, f32x4 v) {
    if constexpr (END == kTanhNorm) {
        const uint32_t u = (uint32_t)m / (uint32_t)a.T;
        v += load4(a.bias + (int64_t)u * a.outputs + c);
    } else if constexpr (END == kShift) {
        v += load4(a.norm.bias + c) - load4(a.norm.mean + c) * norm_gain(a.norm, c);
    } else {
        v += load4(a.bias + c);
    }
    if constexpr (END == kReluNorm || END == kTanhNorm) {
        const f32x4 sc = load4(a.scale + c), of = load4(a.offset + c);
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            v[r] = __builtin_fmaf(v[r] < 0.f ? 0.f : v[r], sc[r], of[r]);        // NaN stays
            if constexpr (END == kTanhNorm) v[r] = tanh_of(v[r]);
        }
    }
    return v;
}
template <class DT, LinearEnd END>
__device__ inline void finish(const LinearArgs &a, Rsrc out, int64_t m0, int row, int c, f32x4 v) {
    v = ended<DT, END>(a, m0 + row, c, v);
    if constexpr (END == kAffine || END == kShift)
        __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u32x4, v), out, row * a.out_pitch + 4 * c, 0, 0);
    else
        __builtin_amdgcn_raw_buffer_store_b64(narrow4<DT>(v), out, row * a.out_pitch + 2 * c, 0, 0);
}

// Many rows: a workgroup of four waves computes 16 * MT rows x 64 * NTW outputs.  The rows come through LDS 256 inputs at
// a time, the next piece on its way while this one is multiplied; the weights stream from L2 into registers as above.
template <class DT, int MT, int NTW, LinearEnd END>
__global__ void __launch_bounds__(kThreads, 2)
linear_kernel(LinearArgs a, int col_blocks) {
    constexpr int PF = 4, NW = kWaves;
    extern __shared__ __attribute__((aligned(16))) char smem[];
    LDS_PTR(char) lds = (LDS_PTR(char))smem;
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), n = lane & 15, g = lane >> 4;
    const uint32_t item = xcd_item(blockIdx.x, gridDim.x);           // neighbours share their rows' lines
    const uint32_t row_block = item / (uint32_t)col_blocks;
    const int64_t m0 = (int64_t)row_block * (16 * MT);
    const int rows = (int)min((int64_t)(16 * MT), a.M - m0);
    const int tile0 = ((int)(item - row_block * col_blocks) * NW + wave) * NTW;
    const Rsrc xs = make_rsrc(a.x + m0 * a.x_pitch, rows * a.x_pitch), ws = weight_rsrc(a.w, a.outputs, a.inputs);
    const int steps = a.inputs / 32, pieces = a.inputs / 256;
    auto stage = [&](int piece) {
        constexpr int kChunks = 16 * MT * kRow / kChunk;
#pragma unroll
        for (int j = 0; j < kChunks / NW; ++j) {
            const int c = j * NW + wave, row = 2 * c + (lane >> 5);
            load_to_lds<16, kReadShared>(xs, lds + (piece & 1) * (16 * MT * kRow) + c * kChunk, row * a.x_pitch + piece * kRow + ((lane & 31) ^ (row & 15)) * 16);
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
    const Rsrc os = make_rsrc(a.out + m0 * a.out_pitch, rows * a.out_pitch);
#pragma unroll
    for (int i = 0; i < MT; ++i)
#pragma unroll
        for (int j = 0; j < NTW; ++j) finish<DT, END>(a, os, m0, 16 * i + n, 16 * (tile0 + j) + 4 * g, acc[j][i]);
}

// Very many rows, outputs in hundreds: 128 rows x 256 outputs to a workgroup of four waves.  A wave's 128 x 64 outputs use each
// weight eight times and each row's operand four times, which halves what the CU's path to L2 carries per product (64 rows ask
// for its 64 bytes a clock at the matrix cores' full rate); rows come 128 inputs at a time, so two workgroups share a CU.
// 1024 inputs, 1536 outputs, this and 64 rows, us in a trace: 8200 rows 35 and 54, 10000: 36 and 57, 25600: 85 and 132 (0.95
// PFLOP/s), 40000: 133 and 209.  Below the limit linear_kernel's 32 rows x 128 outputs: 2048: 24 and 16, 4000: 24.6 and 27.4 (one
// round of its workgroups more from 4096 on: 30.1), 6400: 34.9 and 41.0, 8000: 35.4 and 48.1.
template <class DT, LinearEnd END>
__global__ void __launch_bounds__(kThreads, 2)
linear_wide_kernel(LinearArgs a, int col_blocks) {
    constexpr int MT = 8, NTW = 4, PF = 4, NW = kWaves, kSteps = 4, kPiece = 64 * kSteps;     // bytes of a row's piece
    extern __shared__ __attribute__((aligned(16))) char smem[];
    LDS_PTR(char) lds = (LDS_PTR(char))smem;
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), n = lane & 15, g = lane >> 4;
    const uint32_t item = xcd_item(blockIdx.x, gridDim.x);           // neighbours share their rows' lines
    const uint32_t row_block = item / (uint32_t)col_blocks;
    const int64_t m0 = (int64_t)row_block * (16 * MT);
    const int rows = (int)min((int64_t)(16 * MT), a.M - m0);
    const int tile0 = ((int)(item - row_block * col_blocks) * NW + wave) * NTW;
    const Rsrc xs = make_rsrc(a.x + m0 * a.x_pitch, rows * a.x_pitch), ws = weight_rsrc(a.w, a.outputs, a.inputs);
    const int steps = a.inputs / 32, pieces = steps / kSteps, lane16 = lane * 16;
    auto stage = [&](int piece) {                                    // four rows to a load, their 16-byte units swizzled by the row
#pragma unroll
        for (int j = 0; j < 16 * MT * kPiece / kChunk / NW; ++j) {
            const int c = j * NW + wave, row = 4 * c + (lane >> 4);
            load_to_lds<16, kReadShared>(xs, lds + (piece & 1) * (16 * MT * kPiece) + c * kChunk, row * a.x_pitch + piece * kPiece + ((lane & 15) ^ (row & 15)) * 16);
        }
    };
    stage(0);
    f32x4 acc[NTW][MT];
    clear(acc);
    u32x4 w[PF][NTW];
    auto fill = [&](int slot, int step) {
#pragma unroll
        for (int j = 0; j < NTW; ++j)
            w[slot][j] = __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(ws, lane16, ((tile0 + j) * steps + step) * kFrag, 0));
    };
#pragma unroll
    for (int s = 0; s < PF; ++s) fill(s, s);
    const int x_lane = n * kPiece + ((g ^ n) << 4);
#pragma unroll 1
    for (int p = 0; p < pieces; ++p) {
        wait_direct();
        barrier_lds();
        if (p + 1 < pieces) stage(p + 1);
        LDS_PTR(char) from = lds + (p & 1) * (16 * MT * kPiece);
        u32x4 x[2][4];
        auto read = [&](int turn) {                                  // four of the row tiles of a step
            LDS_PTR(char) at = from + (x_lane ^ 64 * (turn >> 1)) + (turn & 1) * (64 * kPiece);
#pragma unroll
            for (int i = 0; i < 4; ++i) x[turn & 1][i] = *reinterpret_cast<LDS_PTR(u32x4)>(at + i * 16 * kPiece);
        };
        read(0);
#pragma unroll
        for (int turn = 0; turn < 2 * kSteps; ++turn) {
            const int s = turn >> 1, i0 = 4 * (turn & 1);
            if (turn + 1 < 2 * kSteps) read(turn + 1);
            __builtin_amdgcn_sched_barrier(0x27f);                   // see multiply()
#pragma unroll
            for (int j = 0; j < NTW; ++j)
#pragma unroll
                for (int i = 0; i < 4; ++i) acc[j][i0 + i] = Mma<DT>::k32(w[s % PF][j], x[turn & 1][i], acc[j][i0 + i]);
            if (turn & 1) fill(s % PF, min(kSteps * p + s + PF, steps - 1));
        }
    }
    const Rsrc os = make_rsrc(a.out + m0 * a.out_pitch, rows * a.out_pitch);
#pragma unroll
    for (int i = 0; i < MT; ++i) {
        u32x2 o[NTW];
#pragma unroll
        for (int j = 0; j < NTW; ++j) o[j] = narrow4<DT>(ended<DT, END>(a, m0 + 16 * i + n, 16 * (tile0 + j) + 4 * g, acc[j][i]));
        store_tile<16 * NTW, 0>(os, (16 * i + n) * a.out_pitch + 32 * tile0, o, g, 32 * NTW);
    }
}

// Few rows: the inputs are split over the eight waves of a workgroup that computes 16 rows x 16 * NT outputs; rows and
// weights go from memory straight into the operands' registers and the waves' sums meet in LDS.
template <class DT, int NT, LinearEnd END>
__global__ void __launch_bounds__(512)
linear_small_kernel(LinearArgs a, int col_blocks) {
    constexpr int NW = 8, U = 4;
    __shared__ __attribute__((aligned(16))) f32x4 sums[NW][NT][64];
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), n = lane & 15, g = lane >> 4;
    const int row_block = (int)(blockIdx.x / (uint32_t)col_blocks), tile0 = ((int)blockIdx.x - row_block * col_blocks) * NT;
    const int64_t m0 = (int64_t)row_block * 16;
    const int rows = (int)min((int64_t)16, a.M - m0);
    const Rsrc xs = make_rsrc(a.x + m0 * a.x_pitch, rows * a.x_pitch), ws = weight_rsrc(a.w, a.outputs, a.inputs);
    const int steps = a.inputs / 32;
    f32x4 acc[NT];
#pragma unroll
    for (int j = 0; j < NT; ++j) acc[j] = f32x4{0.f, 0.f, 0.f, 0.f};
    for (int s0 = wave; s0 < steps; s0 += NW * U) {
        u32x4 x[U], w[U][NT];
#pragma unroll
        for (int u = 0; u < U; ++u) {                // steps past the end: zero rows (no resource reaches kNowhere)
            const int s = s0 + u * NW, at = s < steps ? n * a.x_pitch + 64 * s + 16 * g : kNowhere;
            x[u] = __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(xs, at, 0, 0));
#pragma unroll
            for (int j = 0; j < NT; ++j)
                w[u][j] = __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(ws, lane * 16, ((tile0 + j) * steps + min(s, steps - 1)) * kFrag, 0));
        }
#pragma unroll
        for (int u = 0; u < U; ++u)
#pragma unroll
            for (int j = 0; j < NT; ++j) acc[j] = Mma<DT>::k32(w[u][j], x[u], acc[j]);
    }
#pragma unroll
    for (int j = 0; j < NT; ++j) sums[wave][j][lane] = acc[j];
    __syncthreads();
    if (wave < NT) {
        f32x4 v = sums[0][wave][lane];
#pragma unroll
        for (int k = 1; k < NW; ++k) v += sums[k][wave][lane];
        const Rsrc os = make_rsrc(a.out + m0 * a.out_pitch, rows * a.out_pitch);
        finish<DT, END>(a, os, m0, n, 16 * (tile0 + wave) + 4 * g, v);
    }
}

// =============================================================================
// Around the encoder
// =============================================================================
// Valid tokens and frames-as-tokens counts from relative lengths (models/PCF_NATransformer.py:406-414, Pooling.py:30-35).
__global__ void lengths_kernel(int32_t *t_valid, float *count, const float *lens, int N, int frames, int patch, int T) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= N) return;
    const float len = lens[i], pad = floorf(((float)frames - rintf(len * (float)frames)) / (float)patch);
    t_valid[i] = T - (int)pad;
    count[i] = rintf(len * (float)T);
}

// [N, in_chans, frames] fp32 -> patch rows [N * T, in_chans * patch] of 16 bit, element (c, j) of token t = x[c][t * patch + j].
// kPatchTokens tokens of `chans` channels to a workgroup through LDS: a wave reads along the frames of a channel, the
// writes run along the rows.  Bound by memory; the work is split over the channels too, or a single utterance is a handful
// of workgroups (3 s: 19.5 us in three workgroups of whole rows that divided twice for every value).
// The launch's last slices bring the last layer's weight into fragment order and the pooled norm into an affine map, from
// the module's own tensors at each call: of a single utterance's 273 us that is 3, and as much again with the last product
// rounding the fp32 rows itself; kept from call to call, a write that no version counts would go unseen.
constexpr int kPatchTokens = 32;
struct Head {
    char *w;                        // 16-bit fragments of ...
    const float *w_fc;              // ... [emb, inputs]
    float *a_pool, *c_pool;         // [inputs]
    na1d_encoder_norm norm;         // weight NULL: none
    int emb, inputs, slices;        // slices of the launch before these
};
template <class DT>
__device__ inline void prepare_head(const Head &h) {
    const int lane = threadIdx.x & 63, n = lane & 15, g = lane >> 4;
    const int64_t blocks = (int64_t)(gridDim.z - h.slices) * gridDim.y * gridDim.x;
    const int64_t block = ((int64_t)(blockIdx.z - h.slices) * gridDim.y + blockIdx.y) * gridDim.x + blockIdx.x;
    const int steps = h.inputs / 32;
    for (int64_t f = 4 * block + (threadIdx.x >> 6); f < (int64_t)h.emb / 16 * steps; f += 4 * blocks) {
        const float *from = h.w_fc + (f / steps * 16 + n) * h.inputs + f % steps * 32 + 8 * g;
        u32x4 w;
#pragma unroll
        for (int k = 0; k < 4; ++k) w[k] = Mma<DT>::pack(from[2 * k], from[2 * k + 1]);
        *reinterpret_cast<u32x4 *>(h.w + f * kFrag + lane * 16) = w;
    }
    for (int64_t c = block * 256 + threadIdx.x; c < h.inputs; c += blocks * 256) {
        const float gain = h.norm.weight ? h.norm.weight[c] * __builtin_amdgcn_rsqf(h.norm.var[c] + h.norm.eps) : 1.f;
        h.a_pool[c] = gain;
        h.c_pool[c] = h.norm.weight ? __builtin_fmaf(-h.norm.mean[c], gain, h.norm.bias[c]) : 0.f;
    }
}
template <class DT>
__global__ void __launch_bounds__(256)
patch_kernel(uint32_t *__restrict__ out, const float *__restrict__ x, int in_chans, int chans, int frames, int patch, int T, uint32_t patch_magic,
             uint32_t width_magic, Head head) {
    if ((int)blockIdx.z >= head.slices) return prepare_head<DT>(head);
    extern __shared__ __attribute__((aligned(16))) char smem[];
    float *tile = reinterpret_cast<float *>(smem);               // [chans][kPatchTokens * patch + 1]
    const int span = kPatchTokens * patch, pitch = span + 1, t0 = blockIdx.x * kPatchTokens, nt = min(kPatchTokens, T - t0), c_first = blockIdx.z * chans;
    const float *src = x + ((int64_t)blockIdx.y * in_chans + c_first) * frames + (int64_t)t0 * patch;
#pragma unroll 4
    for (int c = threadIdx.x >> 6; c < chans; c += 4)
        for (int f = threadIdx.x & 63; f < nt * patch; f += 64) tile[c * pitch + f] = src[(int64_t)c * frames + f];
    __syncthreads();
    const int half = chans * patch / 2, row = in_chans * patch / 2;                // pairs of a row here and in all
    uint32_t *dst = out + ((int64_t)blockIdx.y * T + t0) * row + c_first * patch / 2;
    for (int i = threadIdx.x; i < nt * half; i += 256) {
        const int t = div_by(i, half, width_magic), k = i - t * half, e = 2 * k;
        const int c0 = div_by(e, patch, patch_magic), j0 = e - c0 * patch, c1 = div_by(e + 1, patch, patch_magic), j1 = e + 1 - c1 * patch;
        dst[(int64_t)t * row + k] = Mma<DT>::pack(tile[c0 * pitch + t * patch + j0], tile[c1 * pitch + t * patch + j1]);
    }
}

// Mean and standard deviation over an utterance's tokens of 64 channels: one pass over the rows, sums of the differences
// to the first row (fp32; the first row is a sample, so nothing cancels).  Written as fp32 for the pooling's sums and in
// 16 bit for the product with the context's weights.
template <class DT>
__global__ void __launch_bounds__(256)
stats_kernel(float *__restrict__ mean_std, char *__restrict__ rounded, const char *__restrict__ h, const float *__restrict__ count,
             int T, int wide) {
    __shared__ float part[2][32][64 + 1];
    const int c = threadIdx.x & 7, r = threadIdx.x >> 3, n = blockIdx.y, c0 = blockIdx.x * 64 + c * 8;
    const int pitch = 2 * wide, valid = count ? max(0, min(T, (int)count[n])) : T;
    const char *src = h + (int64_t)n * T * pitch + 2 * c0;
    float first[8], s1[8], s2[8];
    auto row = [&](int t, float (&v)[8]) {
        const u32x4 w = *reinterpret_cast<const u32x4 *>(src + (int64_t)t * pitch);
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const f32x2 p = widen<DT>(w[i]);
            v[2 * i] = p.x;
            v[2 * i + 1] = p.y;
        }
    };
    row(0, first);
#pragma unroll
    for (int i = 0; i < 8; ++i) s1[i] = s2[i] = 0.f;
#pragma unroll 4
    for (int t = r; t < valid; t += 32) {
        float v[8];
        row(t, v);
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            const float d = v[i] - first[i];
            s1[i] += d;
            s2[i] = __builtin_fmaf(d, d, s2[i]);
        }
    }
#pragma unroll
    for (int i = 0; i < 8; ++i) {
        part[0][r][c * 8 + i] = s1[i];
        part[1][r][c * 8 + i] = s2[i];
    }
    __syncthreads();
    if (threadIdx.x >= 64) return;
    const int ch = threadIdx.x;
    float a = 0.f, b = 0.f;
#pragma unroll 8
    for (int k = 0; k < 32; ++k) {
        a += part[0][k][ch];
        b += part[1][k][ch];
    }
    const float x0 = (float)widen<DT>((uint32_t)*reinterpret_cast<const uint16_t *>(h + (int64_t)n * T * pitch + 2 * (blockIdx.x * 64 + ch))).x;
    const float cnt = count ? count[n] : (float)T, m = a / cnt;
    float var = (b - a * m) / (count ? cnt : cnt - 1.f);
    var = var < 1e-12f ? 1e-12f : var;                          // NaN stays
    const float mean = x0 + m, std = sqrtf(var);
    const int64_t at = (int64_t)n * 2 * wide + blockIdx.x * 64 + ch;
    mean_std[at] = mean;
    mean_std[at + wide] = std;
    reinterpret_cast<uint16_t *>(rounded)[at] = (uint16_t)Mma<DT>::pack(mean, 0.f);
    reinterpret_cast<uint16_t *>(rounded)[at + wide] = (uint16_t)Mma<DT>::pack(std, 0.f);
}

// Attentive statistics pooling: logits = W . hidden[t] on the matrix core, softmax over the tokens and the weighted mean and
// deviation in one pass over the rows, the logits never written.  Lane (n, g) sees channels 8g .. 8g+7 of each 32 (two tiles
// of the product, whose rows are taken in that order) for every 16th token, keeps its own running maximum (moved only when
// outgrown by 2^8) and sums of p, p d, p d^2 (d = difference to the plain mean), and the lanes meet at the end.  A wave takes
// 64 channels; the TS of four waves that have the same ones share an utterance's tokens (one_wave below).  Bound by the latency
// of a wave's few turns and, at 100 tokens, by its two ends (16 weights to fetch, 256 steps across lanes).  256 utterances of
// 100 tokens: 42 us; 64 of 1000: 76 us.  With loads of 8 bytes in the tiles' own order and none ahead of its turn 82 and 92.
// Half the channels and twice the waves to a SIMD: 56 and 121.
struct PoolArgs {
    const char *h, *hidden, *w;
    const float *count, *mean_std, *a_pool, *c_pool;
    char *out;                      // [N, 2 * wide], the next product's operand
    int T, wide;
};
// Over the 16 lanes of a row, in all of them, without LDS: by neighbours, by pairs, then mirrored within 8 and 16 lanes
// (whose quarters are equal by then).  256 of these steps close a wave's work; as shuffles through LDS they were half of
// the kernel's time at 100 tokens.
template <int CTRL> __device__ inline float row_step(float x) {
    return __uint_as_float(__builtin_amdgcn_mov_dpp(__float_as_uint(x), CTRL, 0xf, 0xf, true));
}
__device__ inline float row16_max(float x) {
    x = __builtin_fmaxf(x, row_step<0xb1>(x));
    x = __builtin_fmaxf(x, row_step<0x4e>(x));
    x = __builtin_fmaxf(x, row_step<0x141>(x));
    return __builtin_fmaxf(x, row_step<0x140>(x));
}
__device__ inline float row16_sum(float x) {
    x += row_step<0xb1>(x);
    x += row_step<0x4e>(x);
    x += row_step<0x141>(x);
    return x + row_step<0x140>(x);
}
template <class DT, int TS>
__global__ void __launch_bounds__(kThreads, 2)
pool_kernel(PoolArgs a) {
    constexpr int CT = 4, kSlack = 8, kChannels = 16 * CT * kWaves / TS;         // tiles of a wave, channels of a workgroup
    __shared__ float meet[TS][kChannels][4];
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), n = lane & 15, g = lane >> 4;
    const int part = wave % TS, mine = 16 * CT * (wave / TS);                    // tokens and channels of this wave
    const int utt = blockIdx.y, c0 = blockIdx.x * kChannels, pitch = 2 * a.wide;
    const Rsrc hs = make_rsrc(a.h + (int64_t)utt * a.T * pitch, a.T * pitch), ds = make_rsrc(a.hidden + (int64_t)utt * a.T * 256, a.T * 256);
    const Rsrc ws = weight_rsrc(a.w, a.wide, 128);
    const int valid = a.count ? max(0, min(a.T, (int)a.count[utt])) : a.T;
    u32x4 w[CT][4];
#pragma unroll
    for (int j = 0; j < CT; ++j)
#pragma unroll
        for (int s = 0; s < 4; ++s)
            w[j][s] = __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(
                ws, (n >> 3) * (4 * kFrag) + ((8 * (n >> 2) + 4 * (j & 1) + (n & 3)) % 16 + 16 * g) * 16, (((c0 + mine) / 16 + (j & ~1)) * 4 + s) * kFrag, 0));
    f32x4 mu[CT], m[CT], s0[CT], s1[CT], s2[CT];
#pragma unroll
    for (int j = 0; j < CT; ++j) {
        mu[j] = *reinterpret_cast<const f32x4 *>(a.mean_std + (int64_t)utt * 2 * a.wide + c0 + mine + 32 * (j / 2) + 8 * g + 4 * (j & 1));
        m[j] = f32x4{-1e30f, -1e30f, -1e30f, -1e30f};
        s0[j] = s1[j] = s2[j] = f32x4{0.f, 0.f, 0.f, 0.f};
    }
    const int tiles = (valid + 15) >> 4;
    u32x4 d[4], xr[CT / 2], d_next[4], x_next[CT / 2];
    auto fetch = [&](int t) {                                // rows past the utterance come as zeros
        const int row = 16 * t + n;
#pragma unroll
        for (int s = 0; s < 4; ++s) d_next[s] = __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(ds, row * 256 + 64 * s + 16 * g, 0, 0));
#pragma unroll
        for (int j = 0; j < CT / 2; ++j)
            x_next[j] = __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(hs, row * pitch + 2 * (c0 + mine + 32 * j + 8 * g), 0, 0));
    };
    fetch(part);
    for (int t = part; t < tiles; t += TS) {
        const int row = 16 * t + n;
#pragma unroll
        for (int s = 0; s < 4; ++s) d[s] = d_next[s];
#pragma unroll
        for (int j = 0; j < CT / 2; ++j) xr[j] = x_next[j];
        if (t + TS < tiles) fetch(t + TS);
        f32x4 z[CT], e[CT];                                  // logits, and how far they lie above the maximum
#pragma unroll
        for (int j = 0; j < CT; ++j) {
            z[j] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int s = 0; s < 4; ++s) z[j] = Mma<DT>::k32(w[j][s], d[s], z[j]);
        }
        if (16 * t + 16 > valid) {
#pragma unroll
            for (int j = 0; j < CT; ++j)
#pragma unroll
                for (int r = 0; r < 4; ++r) z[j][r] = row < valid ? z[j][r] : kNegInf;
        }
        float most = kNegInf;
#pragma unroll
        for (int j = 0; j < CT; ++j)
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                e[j][r] = __builtin_fmaf(z[j][r], kLog2e, -m[j][r]);
                most = __builtin_fmaxf(most, e[j][r]);
            }
        if (__builtin_amdgcn_ballot_w64(most > kSlack)) {
#pragma unroll
            for (int j = 0; j < CT; ++j)
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    const float up = __builtin_fmaxf(m[j][r], z[j][r] * kLog2e), f = __builtin_amdgcn_exp2f(m[j][r] - up);
                    m[j][r] = up;
                    s0[j][r] *= f;
                    s1[j][r] *= f;
                    s2[j][r] *= f;
                    e[j][r] = __builtin_fmaf(z[j][r], kLog2e, -up);
                }
        }
#pragma unroll
        for (int j = 0; j < CT; ++j) {
            const f32x4 v = widen4<DT>(j & 1 ? u32x2{xr[j / 2].z, xr[j / 2].w} : u32x2{xr[j / 2].x, xr[j / 2].y});
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const float p = __builtin_amdgcn_exp2f(e[j][r]), dx = v[r] - mu[j][r], pd = p * dx;
                s0[j][r] += p;
                s1[j][r] += pd;
                s2[j][r] = __builtin_fmaf(pd, dx, s2[j][r]);
            }
        }
    }
#pragma unroll
    for (int j = 0; j < CT; ++j)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const float top = row16_max(m[j][r]), f = __builtin_amdgcn_exp2f(m[j][r] - top);
            const float a0 = row16_sum(s0[j][r] * f), a1 = row16_sum(s1[j][r] * f), a2 = row16_sum(s2[j][r] * f);
            if (n == 0) {
                float *at = meet[part][mine + 32 * (j / 2) + 8 * g + 4 * (j & 1) + r];
                at[0] = top;
                at[1] = a0;
                at[2] = a1;
                at[3] = a2;
            }
        }
    __syncthreads();
    if (threadIdx.x >= kChannels) return;
    const int ch = threadIdx.x;
    float top = meet[0][ch][0], a0 = 0.f, a1 = 0.f, a2 = 0.f;
#pragma unroll
    for (int k = 1; k < TS; ++k) top = __builtin_fmaxf(top, meet[k][ch][0]);
#pragma unroll
    for (int k = 0; k < TS; ++k) {
        const float f = __builtin_amdgcn_exp2f(meet[k][ch][0] - top);
        a0 = __builtin_fmaf(f, meet[k][ch][1], a0);
        a1 = __builtin_fmaf(f, meet[k][ch][2], a1);
        a2 = __builtin_fmaf(f, meet[k][ch][3], a2);
    }
    const int64_t row = (int64_t)utt * 2 * a.wide;
    const int c = c0 + ch;
    const float dm = a1 / a0, mean = a.mean_std[row + c] + dm;
    float var = a2 / a0 - dm * dm;
    var = var < 1e-12f ? 1e-12f : var;
    uint16_t *out = reinterpret_cast<uint16_t *>(a.out) + row;
    out[c] = (uint16_t)Mma<DT>::pack(__builtin_fmaf(mean, a.a_pool[c], a.c_pool[c]), 0.f);
    out[c + a.wide] = (uint16_t)Mma<DT>::pack(__builtin_fmaf(sqrtf(var), a.a_pool[c + a.wide], a.c_pool[c + a.wide]), 0.f);
}

// ----------------------------------------------------------------------------- launchers
// Whether a wave takes all of an utterance's tokens.  Such workgroups last as long as the utterance is and two fit a CU, so what
// counts is how full the last 512 are; four waves to an utterance even that out, at the price of four times the ends.  1536
// channels, one and four waves, us: 100 tokens: 24 utterances 11.0 13.5, 32: 11.5 13.0, 96: 24.4 29.2; 200 tokens: 16: 16.2 11.3,
// 32: 16.4 16.8, 64: 24.0 28.8, 96: 37.4 41.6; 300 tokens: 32: 21.9 20.0, 48: 31.6 29.5, 64: 33.8 36.7, 96: 51.3 50.7, 112: 51.5
// 60.3; 500 tokens: 64: 47.3 45.3, 85: 47.6 59.4, 96: 76.4 67.3, 112: 76.8 80.4; 1000 tokens: 64: 87.0 75.8, 85: 87.9 102,
// 86: 151 116, 128: 158 159, 170: 176 210; 2000 tokens: 64: 167 143, 85: 170 191, 128: 313 292.
inline bool one_wave(int64_t N, int64_t T, int wide) {
    const int64_t blocks = N * (wide / 256), room = (blocks + 511) / 512 * 512;
    return T <= 200 ? blocks >= 192 : T <= 500 ? 8 * blocks >= 5 * room : 5 * blocks >= 4 * room;
}

// Two workgroups of two and more row tiles share a CU.  Up to 48 tokens to each of these places all of them get a workgroup and the
// row tiles are dealt out, three and two: in tiles of 64, some CUs have two and others one.  20000 tokens, us in a trace, layers
// of 8, 4, 2 and 1 groups: 33.1 -> 29.9, 37.6 -> 35.0, 46.5 -> 41.4, 50.1 -> 50.2 (weights bound these, and every workgroup reads
// them); dealt out in fours and threes, 25600 tokens gain nothing (240 us for five layers either way) and 30000 lose (259 -> 273).
constexpr int kLayerPlaces = 512;
template <class DT, int MT, int NW, int PF, bool SPARSE>
int launch_layer_mt(const LayerArgs &a, hipStream_t s) {
    auto kern = layer_kernel<DT, MT, NW, PF, false, SPARSE>;
    const size_t lds = layer_lds<MT>();
    if (!allow_lds(kern, lds)) return NA1D_ERR_LAUNCH;
    const int64_t tiles = (a.M + 15) / 16;
    int64_t wgs = (tiles + MT - 1) / MT;
    LayerArgs args = a;
    if (MT == 3) wgs = kLayerPlaces, args.large = (int)(tiles - 2 * wgs);
    kern<<<(unsigned)wgs, 64 * NW, lds, s>>>(args);
    return launch_status();
}

// Up to this many tokens the four quarters of every tile find a CU of their own.  A PCF 4x4 pass with and without:
// 500 tokens 290 and 335 us, 1000: 325 and 351; 1500: 416 and 363, 3000: 548 and 415.
constexpr int64_t kSplitTokens = 16 * 64;
template <class DT> int launch_layer_split(const LayerArgs &a, hipStream_t s) {
    const size_t lds = layer_lds<1>();
    const unsigned tiles = (unsigned)((a.M + 15) / 16);
    if (a.attn) {
        part_kernel<DT, 8, 8><<<4 * tiles, 512, lds, s>>>(a);
        const int st = launch_status();
        if (st != NA1D_OK) return st;
    }
    layer_kernel<DT, 1, 8, 8, true, false><<<(a.qkv ? 3 : 1) * tiles, 512, lds, s>>>(a);
    return launch_status();
}

template <class DT> int launch_layer(const LayerArgs &a, hipStream_t s) {
    if (a.M <= kSplitTokens) return launch_layer_split<DT>(a, s);
    // Fewer, larger tiles read the layer's weights fewer times; smaller ones spread few tokens over more CUs.  PCF 4x4 passes
    // with tiles of 16, 32 and 64 tokens: 4000 tokens 450, 494 and 653 us; 6000: 623, 539, 694; 16000: 1101, 884, 879;
    // 20000: 1319, 1083, 1055; 25600: 1668, 1291, 1166; MFA 4x4: 6000: 832, 629, 888; 16000: 1494, 1033, 1075; 25600: 2380,
    // 1614, 1399.  (Measured before the present loops; the lines have been the same since, but for 48 tokens, see above.)
    const bool sparse = a.tail_groups >= 4;
    if (a.M <= 16 * 256) return sparse ? launch_layer_mt<DT, 1, 8, 8, true>(a, s) : launch_layer_mt<DT, 1, 8, 8, false>(a, s);
    if (a.M <= 32 * 512) return sparse ? launch_layer_mt<DT, 2, 8, 4, true>(a, s) : launch_layer_mt<DT, 2, 8, 4, false>(a, s);
    if (a.M <= 48 * kLayerPlaces) return sparse ? launch_layer_mt<DT, 3, 8, 4, true>(a, s) : launch_layer_mt<DT, 3, 4, 4, false>(a, s);
    return sparse ? launch_layer_mt<DT, 4, 8, 4, true>(a, s) : launch_layer_mt<DT, 4, 4, 4, false>(a, s);
}

template <class DT, LinearEnd END> int launch_linear(const LinearArgs &a, hipStream_t s) {
    if (a.inputs % 256 == 0 && a.M > 512) {
        auto go = [&](auto kern, int mt, int ntw, int row = kRow) {
            const size_t lds = (size_t)2 * 16 * mt * row;
            if (!allow_lds(kern, lds)) return (int)NA1D_ERR_LAUNCH;
            const int cols = a.outputs / (64 * ntw);
            kern<<<(unsigned)((a.M + 16 * mt - 1) / (16 * mt) * cols), kThreads, lds, s>>>(a, cols);
            return launch_status();
        };
        if constexpr (END == kReluNorm)
            if (a.M > 4096) return go(linear_wide_kernel<DT, END>, 8, 4, 256);                      // outputs in 256s: encoder_ok
        if (a.M > 8192) {
            if constexpr (END == kShift || END == kEmbedding)                                       // the pooling's are 128
                if (a.outputs % 256 == 0) return go(linear_kernel<DT, 4, 4, END>, 4, 4);
            if constexpr (END != kReluNorm)
                if (a.outputs % 128 == 0) return go(linear_kernel<DT, 4, 2, END>, 4, 2);
        } else if (a.outputs % 128 == 0) {
            return go(linear_kernel<DT, 2, 2, END>, 2, 2);
        }
    }
    const int nt = a.outputs % 32 == 0 ? 2 : 1, cols = a.outputs / (16 * nt);
    const unsigned wgs = (unsigned)((a.M + 15) / 16 * cols);
    if (nt == 2)
        linear_small_kernel<DT, 2, END><<<wgs, 512, 0, s>>>(a, cols);
    else
        linear_small_kernel<DT, 1, END><<<wgs, 512, 0, s>>>(a, cols);
    return launch_status();
}

// The workspace's tensors, one behind the other.
struct Buffers {
    int64_t bytes = 0;
    int64_t x, qkv, attn, blocks, patches, pos, h, hidden, stats, rounded, context, pooled, t_valid, count, x1, parts, w_fc, pool_map;
    int64_t take(int64_t n) {
        const int64_t at = bytes;
        bytes += (n + 255) / 256 * 256;
        return at;
    }
    Buffers(const na1d_encoder &e, int64_t N, int64_t T, int dense) {
        const int64_t M = N * T;
        x = take(M * kRow);
        qkv = take(M * 3 * kRow);
        attn = take(M * kRow);
        blocks = take(M * e.blocks * kRow);
        patches = take(M * e.in_chans * e.patch * 2);
        pos = take(dense * T * kDim * 4);
        h = take(M * e.wide * 2);
        hidden = take(M * 256);
        stats = take(N * 2 * e.wide * 4);
        rounded = take(N * 2 * e.wide * 2);
        context = take(N * 128 * 4);
        pooled = take(N * 2 * e.wide * 2);
        t_valid = take(N * 4);
        count = take(N * 4);
        x1 = take(M <= kSplitTokens ? M * kRow : 0);
        parts = take(M <= kSplitTokens ? 4 * M * kDim * 4 : 0);
        w_fc = take((int64_t)e.emb * 2 * e.wide * 2);
        pool_map = take((int64_t)2 * 2 * e.wide * 4);
    }
};
inline int dense_layers(const na1d_encoder &e) {
    int n = 0;
    for (int i = 0; i < e.layers; ++i) n += e.layer[i].window == 0;
    return n;
}

#define NA1D_TRY(...)                       \
    do {                                    \
        const int st_ = (__VA_ARGS__);      \
        if (st_ != NA1D_OK) return st_;     \
    } while (0)

template <class DT>
int encode(const na1d_encoder &e, char *out, const float *x, const float *lens, int64_t N, int64_t frames, char *ws, hipStream_t s) {
    const int64_t T = (frames - e.patch) / e.patch + 1, M = N * T;
    const int patch_width = 2 * e.in_chans * e.patch;
    const Buffers b(e, N, T, dense_layers(e));
    int32_t *t_valid = nullptr;
    float *count = nullptr;
    if (lens) {
        t_valid = reinterpret_cast<int32_t *>(ws + b.t_valid);
        count = reinterpret_cast<float *>(ws + b.count);
        lengths_kernel<<<(unsigned)((N + 255) / 256), 256, 0, s>>>(t_valid, count, lens, (int)N, (int)frames, e.patch, (int)T);
        NA1D_TRY(launch_status());
    }
    {
        const int chans = e.in_chans % 16 == 0 ? 16 : e.in_chans, half = chans * e.patch / 2;
        const size_t lds = (size_t)chans * (kPatchTokens * e.patch + 1) * sizeof(float);
        if (!allow_lds(patch_kernel<DT>, lds)) return NA1D_ERR_LAUNCH;
        const int slices = e.in_chans / chans, inputs = 2 * e.wide;
        const int64_t x_blocks = (T + kPatchTokens - 1) / kPatchTokens, packing = ((int64_t)e.emb / 16 * (inputs / 32) + 3) / 4;     // a fragment to a wave
        const unsigned more = (unsigned)std::min<int64_t>(1024, (packing + x_blocks * N - 1) / (x_blocks * N));
        patch_kernel<DT><<<dim3((unsigned)x_blocks, (unsigned)N, slices + more), 256, lds, s>>>(
            reinterpret_cast<uint32_t *>(ws + b.patches), x, e.in_chans, chans, (int)frames, e.patch, (int)T, div_magic(e.patch), div_magic(half),
            Head{ws + b.w_fc, e.w_fc, reinterpret_cast<float *>(ws + b.pool_map), reinterpret_cast<float *>(ws + b.pool_map) + inputs, e.pool_norm, e.emb, inputs, slices});
        NA1D_TRY(launch_status());
    }
    int dense = 0;
    for (int i = 0; i < e.layers; ++i) {
        const na1d_encoder_layer &l = e.layer[i];
        if (l.window) continue;
        LinearArgs a{};
        a.x = (const char *)e.pos;
        a.w = (const char *)l.w_pos;
        a.out = ws + b.pos + dense++ * T * kDim * 4;
        a.norm = l.norm;
        a.x_pitch = kRow;
        a.out_pitch = 4 * kDim;
        a.inputs = a.outputs = kDim;
        a.M = (int)T;
        NA1D_TRY(launch_linear<DT, kShift>(a, s));
    }
    dense = 0;
    int block = 0;
    const char *x_in = nullptr;               // the residual stream of the layer before
    int x_in_pitch = kRow;
    for (int i = 0; i <= e.layers; ++i) {
        LayerArgs a{};
        a.M = (int)M;
        a.T = (int)T;
        a.T_magic = div_magic(T);
        a.tail_groups = a.head_groups = 1;
        a.x1 = ws + b.x1;
        a.parts = reinterpret_cast<float *>(ws + b.parts);
        if (i > 0) {
            const na1d_encoder_layer &l = e.layer[i - 1];
            a.attn = ws + b.attn;
            a.x_in = x_in;
            a.x_in_pitch = x_in_pitch;
            a.w_proj = (const char *)l.w_proj, a.w_fc1 = (const char *)l.w_fc1, a.w_fc2 = (const char *)l.w_fc2;
            a.b_proj = l.b_proj, a.b_fc1 = l.b_fc1, a.b_fc2 = l.b_fc2;
            a.tail_groups = known_groups(l.groups);
            if (l.block_end) {
                a.block_pitch = e.blocks * kRow;
                a.block_out = ws + b.blocks + block++ * kRow;
            }
        }
        if (i < e.layers) {
            const na1d_encoder_layer &l = e.layer[i];
            if (l.embeds) {
                a.patches = ws + b.patches;
                a.patch_width = patch_width;
                a.w_embed = (const char *)l.w_embed;
                a.b_embed = l.b_embed;
            }
            if (a.block_out && !l.embeds) {   // the block's output is the next layer's input as it is
                x_in = a.block_out;
                x_in_pitch = a.block_pitch;
            } else {
                a.x_out = ws + b.x;
                x_in = a.x_out;
                x_in_pitch = kRow;
            }
            a.qkv = ws + b.qkv;
            a.w_qkv = (const char *)l.w_qkv;
            a.b_qkv = l.b_qkv;
            a.head_groups = known_groups(l.groups);
            if (!l.window) {
                a.norm = l.norm;
                a.posb = reinterpret_cast<const float *>(ws + b.pos + dense++ * T * kDim * 4);
            }
        }
        NA1D_TRY(launch_layer<DT>(a, s));
        if (i == e.layers) break;
        const na1d_encoder_layer &l = e.layer[i];
        Geom g;
        g.B = N * l.heads;
        g.T = T;
        g.H = l.heads;
        g.C = kDim / l.heads;
        g.W = l.window ? l.window : 1;
        g.L = l.window ? l.left : 0;
        Layout in{T * 3 * kDim, g.C, 3 * kDim}, outl{T * kDim, g.C, kDim};
        const char *q = ws + b.qkv, *k = q + kRow, *v = k + kRow;
        if (l.window) {
            set_dilation(g, l.dilation);
            in.row *= g.dilation;
            outl.row *= g.dilation;
            int st = fused_fwd(ws + b.attn, nullptr, q, k, v, l.rpb, t_valid, g, in, outl, l.scale, DT::tag, s);
            if (st == NA1D_ERR_UNSUPPORTED) st = wide_fwd(ws + b.attn, nullptr, q, k, v, l.rpb, t_valid, g, in, outl, l.scale, DT::tag, s);
            NA1D_TRY(st);
        } else {
            NA1D_TRY(global_fwd(ws + b.attn, nullptr, q, k, v, t_valid, g, in, outl, l.scale, DT::tag, s));
        }
    }
    LinearArgs a{};
    a.x = ws + b.blocks, a.x_pitch = e.blocks * kRow, a.inputs = e.blocks * kDim, a.M = (int)M, a.T = (int)T;
    a.w = (const char *)e.w_wide, a.bias = e.b_wide, a.scale = e.a_wide, a.offset = e.c_wide;
    a.out = ws + b.h, a.out_pitch = 2 * e.wide, a.outputs = e.wide;
    NA1D_TRY(launch_linear<DT, kReluNorm>(a, s));
    stats_kernel<DT><<<dim3((unsigned)(e.wide / 64), (unsigned)N), 256, 0, s>>>(reinterpret_cast<float *>(ws + b.stats), ws + b.rounded,
                                                                              ws + b.h, count, (int)T, e.wide);
    NA1D_TRY(launch_status());
    LinearArgs c{};
    c.x = ws + b.rounded, c.x_pitch = 4 * e.wide, c.inputs = 2 * e.wide, c.M = (int)N;
    c.w = (const char *)e.w_ctx, c.bias = e.b_att, c.out = ws + b.context, c.out_pitch = 4 * 128, c.outputs = 128;
    NA1D_TRY(launch_linear<DT, kAffine>(c, s));
    LinearArgs d{};
    d.x = ws + b.h, d.x_pitch = 2 * e.wide, d.inputs = e.wide, d.M = (int)M, d.T = (int)T;
    d.w = (const char *)e.w_att, d.bias = reinterpret_cast<const float *>(ws + b.context), d.scale = e.a_att, d.offset = e.c_att;
    d.out = ws + b.hidden, d.out_pitch = 256, d.outputs = 128;
    NA1D_TRY(launch_linear<DT, kTanhNorm>(d, s));
    PoolArgs p{ws + b.h, ws + b.hidden, (const char *)e.w_logit, count, reinterpret_cast<const float *>(ws + b.stats),
               reinterpret_cast<const float *>(ws + b.pool_map), reinterpret_cast<const float *>(ws + b.pool_map) + 2 * e.wide, ws + b.pooled, (int)T, e.wide};
    if (one_wave(N, T, e.wide))
        pool_kernel<DT, 1><<<dim3((unsigned)(e.wide / 256), (unsigned)N), kThreads, 0, s>>>(p);
    else
        pool_kernel<DT, 4><<<dim3((unsigned)(e.wide / 64), (unsigned)N), kThreads, 0, s>>>(p);
    NA1D_TRY(launch_status());
    LinearArgs f{};
    f.x = ws + b.pooled, f.x_pitch = 4 * e.wide, f.inputs = 2 * e.wide, f.M = (int)N;
    f.w = ws + b.w_fc, f.bias = e.b_fc, f.out = out, f.out_pitch = 2 * e.emb, f.outputs = e.emb;
    return launch_linear<DT, kEmbedding>(f, s);
}

inline bool norm_whole(const na1d_encoder_norm &n) { return n.weight && n.bias && n.mean && n.var; }
// Sizes the kernels take (everything else is the caller's to run another way).
bool encoder_ok(const na1d_encoder &e, int64_t N, int64_t frames) {
    if (e.layers < 1 || e.blocks < 1 || e.patch < 1 || e.in_chans < 1 || e.wide < 256 || e.emb < 16 || frames < e.patch) return false;
    if (e.in_chans > 4096 || e.patch > 256 || e.in_chans * e.patch % 32 || e.in_chans * e.patch > kDim || e.wide % 256 || e.emb % 16 || e.wide > (1 << 16) || e.emb > (1 << 16)) return false;
    if ((size_t)e.in_chans * (64 * e.patch + 1) * sizeof(float) > 160 * 1024) return false;
    // a weight's bytes are counted in 31 bits
    if ((int64_t)e.emb * e.wide >= (1 << 29) || (int64_t)e.blocks * e.wide >= (1 << 22)) return false;
    const int64_t T = (frames - e.patch) / e.patch + 1;
    // rows of an utterance stay in the reach of 31-bit offsets (the widest are those of the projection), launches of 31-bit ids
    if (T > (1 << 29) / e.wide || N > 65535 || N * T > (1ll << 26) || frames > (1 << 24)) return false;
    int blocks = 0;
    for (int i = 0; i < e.layers; ++i) {
        const na1d_encoder_layer &l = e.layer[i];
        if (l.heads < 1 || kDim % l.heads || kDim / l.heads % 8 || kDim / l.heads > 128 || l.window < 0 || l.window > NA1D_MAX_WINDOW) return false;
        if (l.window && (l.left < 0 || l.left >= l.window || l.dilation < 1)) return false;
        if (!l.window && (!e.pos || e.pos_rows < T || !norm_whole(l.norm) || !l.w_pos)) return false;
        if (!l.w_qkv || !l.w_proj || !l.w_fc1 || !l.w_fc2 || (l.embeds && !l.w_embed)) return false;
        blocks += l.block_end != 0;
    }
    if (e.pool_norm.weight && !norm_whole(e.pool_norm)) return false;
    return blocks == e.blocks && e.layer[0].embeds && e.layer[e.layers - 1].block_end;
}
int64_t workspace_bytes(const na1d_encoder &e, int64_t N, int64_t frames) {
    return Buffers(e, N, (frames - e.patch) / e.patch + 1, dense_layers(e)).bytes;
}
int run(const na1d_encoder &e, void *out, const float *x, const float *lens, int64_t N, int64_t frames, void *ws, hipStream_t s) {
    return e.dtype == NA1D_BF16 ? encode<BF16>(e, (char *)out, x, lens, N, frames, (char *)ws, s)
                                : encode<FP16>(e, (char *)out, x, lens, N, frames, (char *)ws, s);
}

}  // namespace enc
}  // namespace na1d

