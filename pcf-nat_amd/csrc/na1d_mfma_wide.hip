// Fused NA1D forward and backward on the matrix cores for windows that the two- and
// three-block kernels of na1d_mfma.hip do not cover: W up to 80, or more than 16 keys
// on one side.  Same tiling, LDS layout and operand conventions (na1d_mfma_core.h),
// with NBV = ceil((15 + W) / 16) <= 6 virtual key blocks per query tile and no merging
// of blocks: lane (n, g) carries 4*NBV score slots, slot j = 16*vb + 4g + r - shift - n + L.
#include "na1d_mfma_core.h"

namespace na1d {
namespace mfma {

constexpr int kBiasSlots = 96;   // W <= 80, padded

// Blocks and shift of a wide window; 0 blocks if the shape is not covered.
struct WideCover {
    int nbv, shift;
};
inline WideCover wide_cover(const Geom &g) {
    WideCover c{0, 0};
    if (g.C > 128) return c;             // head_dim is run at the next of 16, 32, 64, 128, zero-padded
    if (g.T > (1 << 29) / g.C || g.W > NA1D_MAX_WINDOW) return c;
    c.nbv = (15 + g.W + 15) / 16;
    if (c.nbv < 3) c.nbv = 3;
    // any shift in [L, 16*NBV - 16 - R] covers the window; prefer one that puts key blocks on 128-byte lines
    const int R = g.W - 1 - g.L, rows = std::max(1, 128 / (2 * g.C));
    const int hi = 16 * c.nbv - 16 - R, s16 = (g.L + 15) / 16 * 16, s = (g.L + rows - 1) / rows * rows;
    c.shift = s16 <= hi ? s16 : s <= hi ? s : g.L;      // whole tiles, else whole lines, else the first key
    return c;
}

// rpb row of this head times log2(e) in LDS slots [0, W); -inf is applied at the read
__device__ inline void stage_bias(LDS_PTR(float) bias_lds, const float *rpb_h, int W, int tid) {
    if (tid < kBiasSlots) bias_lds[tid] = (rpb_h && tid < W) ? rpb_h[tid] * kLog2e : 0.f;
}
__device__ inline float bias_at(LDS_PTR(float) bias_lds, int j, int W) {
    const float val = bias_lds[min(max(j, 0), kBiasSlots - 1)];
    return (j >= 0 && j < W) ? val : kNegInf;
}

// =============================================================================
// Forward
// =============================================================================
template <class DT, int C, int NBV, bool DROP>
__global__ void __launch_bounds__(kThreads)
wide_fwd_kernel(char *__restrict__ out, float *__restrict__ lse, const char *__restrict__ q,
                const char *__restrict__ k, const char *__restrict__ v, const float *__restrict__ rpb,
                const int32_t *__restrict__ t_valid, uint32_t items, int T, int W, int L, int H, int tiles, int nt,
                int strips, float scale, uint32_t strips_magic, uint32_t heads_magic, Strides in, Strides outl,
                int shift, Dropout drop, Classes cls, float *__restrict__ clear) {
    using LL = Lds<C>;
    constexpr int CT = C / 16;
    constexpr int MT = Strip<C>::kMaxTiles;
    fetch_args_now(out, lse, q, k, v, rpb, t_valid, items, T, W, L, H, tiles, nt, strips, scale, strips_magic, heads_magic,
                   in.sample, in.head, in.pitch, in.width, outl.sample, outl.head, outl.pitch, outl.width, shift);
    if constexpr (DROP) fetch_args_now(drop.threshold, drop.seed_lo, drop.seed_hi, drop.inv_keep, drop.row_stride, drop.row_offset, drop.seq_rows);
    // dynamic LDS (launch_wide_fwd): K and V regions of kt tiles starting sb tiles before the strip, Q region of nt
    // tiles, kBiasSlots bias floats
    const int sb = (shift + 15) >> 4;                        // whole tiles in front of the strip
    const int kt = nt - 1 + NBV + ((shift & 15) ? 1 : 0);    // tiles a key-side region holds
    extern __shared__ __attribute__((aligned(16))) char smem[];
    const int key_region = region_bytes<C>(kt);
    LDS_PTR(char) k_lds = (LDS_PTR(char))smem;
    LDS_PTR(char) v_lds = k_lds + key_region;
    LDS_PTR(char) q_lds = v_lds + key_region;
    LDS_PTR(float) bias_lds = (LDS_PTR(float))(q_lds + region_bytes<C>(nt));

    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const WorkItem wi = work_item(blockIdx.x, items, strips, strips_magic, H, heads_magic);
    uint32_t sample = wi.sample;
    const uint32_t head = wi.head;
    int cr = 0;                                              // residue class of a dilated window
    if (cls.count > 1) {
        cr = split_class(sample, T, cls);
        if constexpr (DROP) drop.row_offset = (uint32_t)cr;
    }
    const uint32_t b = sample * H + head;
    const int i0 = wi.strip * nt, i1 = min(i0 + nt, tiles);
    const int g = lane >> 4, n = lane & 15;

    const int64_t in_off = sample * in.sample + head * in.head + (int64_t)(cr * cls.in_row);
    const int64_t out_off = sample * outl.sample + head * outl.head + (int64_t)(cr * cls.out_row);
    const int lse_pitch = 4 * cls.d;
    const int key_rows = max(0, min(T, 16 * (i0 - sb + kt)));
    const Rsrc qs = make_rsrc(q + in_off, min(T, 16 * i1) * in.pitch), ks = make_rsrc(k + in_off, key_rows * in.pitch);
    const Rsrc vs = make_rsrc(v + in_off, key_rows * in.pitch), os = make_rsrc(out + out_off, T * outl.pitch);
    const Rsrc ls = make_rsrc(lse ? lse + ((int64_t)b * cls.rows + cr) : nullptr, lse ? T * lse_pitch : 0);
    const bool out_whole_lines = stores_whole_lines(outl.pitch, C, 0);
    {
        const int lane_off = direct_lane_offset<C>(wave, lane, in.pitch, in.width);
        stage_direct<C, MT + NBV, kReadShared>(ks, 16 * (i0 - sb), k_lds, kt, wave, lane_off, in.pitch);
        stage_direct<C, MT, kReadShared>(qs, 16 * i0, q_lds, nt, wave, lane_off, in.pitch);
        stage_direct<C, MT + NBV, kReadShared>(vs, 16 * (i0 - sb), v_lds, kt, wave, lane_off, in.pitch);
        stage_bias(bias_lds, rpb ? rpb + head * W : nullptr, W, tid);
    }
    clear_sums<kThreads>(clear, H * W);

    int tv = T;
    if (t_valid) tv = max(0, min(T, cls.count > 1 ? class_valid(t_valid[sample], cr, cls) : t_valid[sample]));
    const float scale2 = scale * kLog2e;

    RowLane<C> k_lane, q_lane;
    TrLane<C> v_lane;
    k_lane.init(16 * sb - shift, lane);
    q_lane.init(0, lane);
    v_lane.init(16 * sb - shift, lane);

    wait_direct();
    barrier_lds();
    float bias[NBV][4];
#pragma unroll
    for (int vb = 0; vb < NBV; ++vb)
#pragma unroll
        for (int r = 0; r < 4; ++r) bias[vb][r] = bias_at(bias_lds, 16 * vb + 4 * g + r - shift - n + L, W);

    for (int i = i0 + wave; i < i1; i += kWaves) {
        const int tile_bytes = (i - i0) * LL::kTileBytes;
        RowOperand<C> qt;
        read_rows<C>(qt, q_lds + tile_bytes, q_lane);
        float z[NBV][4];
#pragma unroll
        for (int vb = 0; vb < NBV; ++vb) {
            RowOperand<C> kop;
            read_rows<C>(kop, k_lds + tile_bytes + vb * LL::kTileBytes, k_lane);
            const f32x4 s = dot_rows_mma<DT, C>(kop, qt);
#pragma unroll
            for (int r = 0; r < 4; ++r) z[vb][r] = __builtin_fmaf(s[r], scale2, bias[vb][r]);
        }
        const int s0 = 16 * i - shift;           // first row of the window
        const int qrow = 16 * i + n;
        if (s0 < 0 || s0 + 16 * NBV > tv) {      // the model's additive -100, only on tiles that touch an edge
            const bool row_masked = qrow >= tv;
#pragma unroll
            for (int vb = 0; vb < NBV; ++vb)
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    const uint32_t key = (uint32_t)(s0 + 16 * vb + 4 * g + r);   // unsigned: also key < 0
                    z[vb][r] += (key >= (uint32_t)tv || row_masked) ? kMaskValue * kLog2e : 0.f;
                }
        }
        float m = kNegInf;
#pragma unroll
        for (int vb = 0; vb < NBV; ++vb) m = max3(m, max2(z[vb][0], z[vb][1]), max2(z[vb][2], z[vb][3]));
        m = xor_max(m);
        float sum = 0.f;
        u32x2 pb[NBV];
        const uint32_t drop_key = DROP ? dropout_row_key(dropout_row(drop, b, T, qrow), drop) : 0u;
#pragma unroll
        for (int vb = 0; vb < NBV; ++vb) {
            float p[4];
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                p[r] = __builtin_amdgcn_exp2f(z[vb][r] - m);
                sum += p[r];
                // a dropped probability stays in the sum and leaves O
                if (DROP && !dropout_keeps(drop_key, 16 * vb + 4 * g + r - shift - n + L, drop)) p[r] = 0.f;
            }
            pb[vb] = u32x2{Mma<DT>::pack(p[0], p[1]), Mma<DT>::pack(p[2], p[3])};
        }
        sum = xor_sum(sum);
        const float inv = __builtin_amdgcn_rcpf(sum) * (DROP ? drop.inv_keep : 1.f);

        f32x4 o[CT];
#pragma unroll
        for (int ct = 0; ct < CT; ++ct) o[ct] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int vb = 0; vb < NBV; ++vb) {
            LDS_PTR(char) blk = v_lds + tile_bytes + vb * LL::kTileBytes;
#pragma unroll
            for (int ct = 0; ct < CT; ++ct) o[ct] = Mma<DT>::k16(read_tr(blk + v_lane.off[ct]), pb[vb], o[ct]);
        }
        u32x2 ow[CT];
#pragma unroll
        for (int ct = 0; ct < CT; ++ct) ow[ct] = pack_acc<DT>(o[ct], inv);
        store_tile<C>(os, qrow * outl.pitch, ow, g, out_whole_lines, outl.width);   // rows past T are dropped by the store
        if (g == 0)
            __builtin_amdgcn_raw_buffer_store_b32(
                __float_as_uint((m + __builtin_amdgcn_logf(sum)) * kLn2), ls, qrow * lse_pitch, 0, 0);
    }
}

template <class DT, int C, int NBV>
int launch_wide_fwd_n(void *out, float *lse, const void *q, const void *k, const void *v, const float *rpb,
                      const int32_t *t_valid, const Geom &g, const Layout &in, const Layout &outl, float scale,
                      int shift, hipStream_t s) {
    const Split sp = make_split(g.B * g.classes, g.T, Strip<C>::kMaxTiles);
    if (!items_ok(sp, g) || !strides_ok(in, g) || !strides_ok(outl, g)) return NA1D_ERR_UNSUPPORTED;
    auto kern = g.drop.threshold ? wide_fwd_kernel<DT, C, NBV, true> : wide_fwd_kernel<DT, C, NBV, false>;
    const int kt = sp.nt - 1 + NBV + ((shift & 15) ? 1 : 0);
    const size_t lds = (size_t)2 * region_bytes<C>(kt) + region_bytes<C>(sp.nt) + kBiasSlots * sizeof(float);
    if (!allow_lds(kern, lds)) return NA1D_ERR_LAUNCH;
    note_kernel("wide_fwd_kernel", DT::tag, C, NBV, g.drop.threshold != 0);
    launch_kernel(kern, (unsigned)sp.items, lds, s, (char *)out, lse, (const char *)q, (const char *)k, (const char *)v,
                  rpb, t_valid, (uint32_t)sp.items, (int)g.T, g.W, g.L, g.H, sp.tiles, sp.nt, sp.strips, scale,
                  div_magic(sp.strips), div_magic(g.H), byte_strides(in, g), byte_strides(outl, g), shift, g.drop,
                  classes_of(g, in, outl), g.clear);
    return launch_status();
}

template <class DT, int C>
int launch_wide_fwd(void *out, float *lse, const void *q, const void *k, const void *v, const float *rpb,
                    const int32_t *t_valid, const Geom &g, const Layout &in, const Layout &outl, float scale,
                    hipStream_t s) {
    const WideCover c = wide_cover(g);
    switch (c.nbv) {
        case 3: return launch_wide_fwd_n<DT, C, 3>(out, lse, q, k, v, rpb, t_valid, g, in, outl, scale, c.shift, s);
        case 4: return launch_wide_fwd_n<DT, C, 4>(out, lse, q, k, v, rpb, t_valid, g, in, outl, scale, c.shift, s);
        case 5: return launch_wide_fwd_n<DT, C, 5>(out, lse, q, k, v, rpb, t_valid, g, in, outl, scale, c.shift, s);
        case 6: return launch_wide_fwd_n<DT, C, 6>(out, lse, q, k, v, rpb, t_valid, g, in, outl, scale, c.shift, s);
    }
    return NA1D_ERR_UNSUPPORTED;
}

int wide_fwd(void *out, float *lse, const void *q, const void *k, const void *v, const float *rpb,
             const int32_t *t_valid, const Geom &g, const Layout &in, const Layout &outl, float scale, int dtype,
             hipStream_t s) {
    if (!wide_cover(g).nbv) return NA1D_ERR_UNSUPPORTED;
    NA1D_MFMA_DISPATCH(launch_wide_fwd, out, lse, q, k, v, rpb, t_valid, g, in, outl, scale, s);
}

// =============================================================================
// Backward
// =============================================================================
// Key block kp (rows 16*kp - shift ...) is virtual block vb of query tile kp - vb, so the key blocks that touch rows of the
// query tiles i0 .. i1 - 1 see HB = NBV - 1 - floor(shift / 16) query tiles before them and HA = ceil(shift / 16) behind.
// Two kernels: one that walks sequences, and one that has a strip of a sequence in LDS as a whole, for sequences that are one
// strip and for launches too small to walk.  Both take a key block's query tiles in their order: the sums of dK and dV are
// the same to the bit whichever runs, and however sequences are cut.
constexpr int kCuLds = 160 * 1024;
constexpr int kWideSlots = 128;          // d rpb slot sums per wave: slot + 32 indexes them

// d rpb.  Register (vb, r) of lane (n, g) holds key a = 4g + r of block vb against query n: slot
// 16*vb + a - n + L - shift.  A lane permutation lines the diagonals a - n = d (mod 16) up in lane d; members
// with a >= d have a - n = d, the others d - 16, i.e. the slot of the block before.  Lane d thus owns the
// slots d + L - shift + 16*k, k = -1 .. NBV-1; the four lane groups hold the same sums and share the stores.
template <int NBV> __device__ inline void slot_sums(LDS_PTR(float) rsum, const float (&racc)[NBV][4], int wave, int g, int n, int slot) {
    float up[NBV], lo[NBV];
#pragma unroll
    for (int vb = 0; vb < NBV; ++vb) up[vb] = lo[vb] = 0.f;
#pragma unroll
    for (int r = 0; r < 4; ++r) {
        const int a = 4 * g + r;
        const int from = (16 * g + ((a - n) & 15)) * 4;
        const bool upper = a >= n;
#pragma unroll
        for (int vb = 0; vb < NBV; ++vb) {
            const float y = __int_as_float(__builtin_amdgcn_ds_bpermute(from, __float_as_int(racc[vb][r])));
            up[vb] += upper ? y : 0.f;
            lo[vb] += upper ? 0.f : y;
        }
    }
    LDS_PTR(float) mine = rsum + wave * kWideSlots + 32 + slot;
#pragma unroll
    for (int kk = -1; kk < NBV; ++kk) {                 // slot n + L - shift + 16*kk
        float t = (kk >= 0 ? up[kk >= 0 ? kk : 0] : 0.f) + (kk + 1 < NBV ? lo[kk + 1 < NBV ? kk + 1 : 0] : 0.f);
        t = xor_sum(t);
        if (g == ((kk + 1) & 3)) mine[16 * kk] = t;
    }
}
// The workgroup's sums, [kWaves][kWideSlots], to its row of the workspace (folded by drpb_reduce_kernel) or to d rpb.
__device__ inline void add_slot_sums(LDS_PTR(float) rsum, float *drpb, float *drpb_partial, uint32_t item, uint32_t head, int W, int tid) {
    if (!drpb || tid >= W) return;
    float t = 0.f;
#pragma unroll
    for (int w = 0; w < kWaves; ++w) t += rsum[w * kWideSlots + 32 + tid];
    if (drpb_partial)
        drpb_partial[(size_t)item * kWidePartialStride + tid] = t;
    else
        atomicAdd(drpb + head * W + tid, t);
}

// ---- walking sequences -------------------------------------------------------------------
// A workgroup walks a segment of a sequence (all of it, where there are enough sequences) in steps of four query tiles, a
// tile to each wave.  A segment starts HB query tiles before its own rows and ends HA behind them; inside it no score is
// worked out twice.  A step:
//   pass 1, per query tile: S^T, dP^T -> P, delta, dS -> dQ; the rounded P and dS go to LDS as 16x16 tiles.
//   pass 2: of the key blocks that the four tiles see, wave w adds to those with kp % 4 == w, whose sums it keeps in
//     registers from step to step: exactly NBV products of a tile and a block for every wave.  Four blocks are
//     complete behind each step.
// K and V lie in rings of LDS, whose next four tiles are fetched behind pass 1, Q and dO in two buffers up to 32 channels
// (beyond, a second buffer would cost a workgroup of the CU).
// Bound by vector instructions, LDS reads and memory in turn.  In strips, with HB + HA query tiles worked out by the neighbours
// too (at 65 slots as many as a strip's own), and walking, us in a trace: 128 x 8 heads of 300 x 32, W = 65: 57.3 and 36.2
// (3.8 TB/s of what is read and written once), W = 33: 31.7 and 28.0, W = 80: 123 and 46; 16 x 4 of 2000 x 64, W = 65: 66 and
// 31; 16 x 8 of 1000 x 128: 111 and 67.
constexpr int kStep = kWaves;            // query tiles of a step
template <int NBV> constexpr int kRing = NBV <= 5 ? 8 : 12;            // key tiles that a step reads, in whole steps
template <int C> constexpr int kQueryBuffers = C <= 32 ? 2 : 1;
template <int C, int NBV> constexpr size_t wide_bwd_lds() {
    return (size_t)2 * region_bytes<C>(kRing<NBV>) + kStep * NBV * 2 * 512 + 2 * kQueryBuffers<C> * region_bytes<C>(kStep) + 2 * 64 * sizeof(float);
}
// Workgroups of a CU: what its LDS holds, and the registers with it (see the launch bounds; a fifth workgroup, of 16 channels and
// three blocks, is worth 2 to 9 % of a long launch; splits are planned with four).
template <int C, int NBV> constexpr int wide_bwd_fit() { return (int)(128 / ((wide_bwd_lds<C, NBV>() + 1279) / 1280)); }
template <int C, int NBV> constexpr int wide_bwd_places() { return std::min(wide_bwd_fit<C, NBV>(), 4); }
template <int C, int NBV, bool DROP> constexpr int wide_bwd_waves() {
    return DROP ? std::min(wide_bwd_places<C, NBV>(), NBV == 6 ? 2 : 3) : std::min(wide_bwd_fit<C, NBV>(), 5);
}

template <class DT, int C, int NBV, bool DROP>
__global__ void __launch_bounds__(kThreads, (wide_bwd_waves<C, NBV, DROP>()))
wide_bwd_kernel(char *__restrict__ dq, char *__restrict__ dk, char *__restrict__ dv, float *__restrict__ drpb,
                const char *__restrict__ q, const char *__restrict__ k, const char *__restrict__ v,
                const char *__restrict__ dout, const float *__restrict__ lse, const float *__restrict__ rpb,
                const int32_t *__restrict__ t_valid, uint32_t items, int T, int W, int L, int H, int tiles, int nt,
                int strips, float scale, float *__restrict__ drpb_partial, uint32_t strips_magic,
                uint32_t heads_magic, Strides in, Strides outl, int shift, Dropout drop, Classes cls) {
    using LL = Lds<C>;
    constexpr int CT = C / 16, R = kRing<NBV>, QB = kQueryBuffers<C>;
    constexpr int kSets = NBV <= 5 ? 2 : 3;                // key blocks of a wave that are not complete
    constexpr int kScoreTile = 16 * 16 * 2;                // one 16x16 tile of 16-bit scores
    constexpr int kGroup = kStep * LL::kTileBytes;         // the tiles of a step
    constexpr int kBuffer = region_bytes<C>(kStep);
    static_assert(kGroup == kBuffer, "whole chunks");
    fetch_args_now(dq, dk, dv, drpb, q, k, v, dout, lse, rpb, t_valid, items, T, W, L, H, tiles, nt, strips, scale,
                   drpb_partial, strips_magic, heads_magic, in.sample, in.head, in.pitch, in.width, outl.sample,
                   outl.head, outl.pitch, outl.width, shift);
    if constexpr (DROP) fetch_args_now(drop.threshold, drop.seed_lo, drop.seed_hi, drop.inv_keep, drop.row_stride, drop.row_offset, drop.seq_rows);
    // LDS (wide_bwd_lds): K and V rings; P and dS of a step's tiles [(tile * NBV + vb) * 2 + P/dS], which first hold each
    // wave's bias and at the end its d rpb sums; Q and dO of a step; lse of two steps
    extern __shared__ __attribute__((aligned(16))) char smem[];
    LDS_PTR(char) k_lds = (LDS_PTR(char))smem;
    LDS_PTR(char) v_lds = k_lds + R * LL::kTileBytes;
    LDS_PTR(char) sc_lds = v_lds + R * LL::kTileBytes;
    LDS_PTR(char) q_lds = sc_lds + kStep * NBV * 2 * kScoreTile;
    LDS_PTR(char) g_lds = q_lds + QB * kBuffer;             // dO
    LDS_PTR(float) lse_lds = (LDS_PTR(float))(g_lds + QB * kBuffer);

    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const WorkItem wi = work_item(blockIdx.x, items, strips, strips_magic, H, heads_magic);
    uint32_t sample = wi.sample;
    const uint32_t item = wi.item, head = wi.head;
    int cr = 0;                                              // residue class of a dilated window
    if (cls.count > 1) {
        cr = split_class(sample, T, cls);
        if constexpr (DROP) drop.row_offset = (uint32_t)cr;
    }
    const uint32_t b = sample * H + head;
    const int i0 = wi.strip * nt, i1 = min(i0 + nt, tiles);
    const int g = lane >> 4, n = lane & 15;
    const int hb = NBV - 1 - (shift >> 4), ha = (shift + 15) >> 4;
    const int q0 = max(0, i0 - hb), qtiles = min(tiles, i1 + ha) - q0;       // the query tiles of the walk
    const int ktiles = qtiles + NBV - 1, steps = (qtiles + kStep - 1) / kStep;

    const int64_t in_off = sample * in.sample + head * in.head + (int64_t)(cr * cls.in_row);
    const int64_t out_off = sample * outl.sample + head * outl.head + (int64_t)(cr * cls.out_row);
    const int lse_pitch = 4 * cls.d;
    const int key_rows = max(0, min(T, 16 * (q0 + ktiles) - shift)), qry_rows = max(0, min(T, 16 * (q0 + qtiles)));
    const Rsrc ks = make_rsrc(k + in_off, key_rows * in.pitch), vs = make_rsrc(v + in_off, key_rows * in.pitch);
    const Rsrc qs = make_rsrc(q + in_off, qry_rows * in.pitch), gs = make_rsrc(dout + out_off, qry_rows * outl.pitch);
    const Rsrc ls = make_rsrc(lse + ((int64_t)b * cls.rows + cr), T * lse_pitch);
    const int lane_off = direct_lane_offset<C>(wave, lane, in.pitch, in.width);
    const int lane_off_g = direct_lane_offset<C>(wave, lane, outl.pitch, outl.width);
    // the query side of a step: all of its tiles, so that those behind the walk's end are zeros
    auto stage_queries = [&](int step) {
        const int row = 16 * (q0 + kStep * step), buf = QB == 2 ? (step & 1) * kBuffer : 0;
        stage_direct<C, kStep, kReadShared>(qs, row, q_lds + buf, kStep, wave, lane_off, in.pitch);
        stage_direct<C, kStep, kReadShared>(gs, row, g_lds + buf, kStep, wave, lane_off_g, outl.pitch);
        if (wave == (step & 3)) load_to_lds<4, 0>(ls, (LDS_PTR(char))(lse_lds + (step & 1) * 64), (row + lane) * lse_pitch);
    };
    stage_direct<C, R, kReadShared>(ks, 16 * q0 - shift, k_lds, min(R, ktiles), wave, lane_off, in.pitch);
    stage_queries(0);
    stage_direct<C, R, kReadShared>(vs, 16 * q0 - shift, v_lds, min(R, ktiles), wave, lane_off, in.pitch);

    int tv = T;
    if (t_valid) tv = max(0, min(T, cls.count > 1 ? class_valid(t_valid[sample], cr, cls) : t_valid[sample]));
    const float scale2 = scale * kLog2e;
    const float mask2 = kMaskValue * kLog2e;

    RowLane<C> row_lane;                // row operands (virtual key blocks and query tiles are whole tiles)
    TrLane<C> tr_lane;                  // transposed operands of the same
    row_lane.init(0, lane);
    tr_lane.init(0, lane);

    // As the forward adds it, behind the product: rpb / scale, at which the sums could start, has no value for every scale.
    // Every wave has a table of its own, in the place of its scores.
    float bias[NBV][4];
    {
        LDS_PTR(float) mine = (LDS_PTR(float))(sc_lds + wave * (NBV * 2 * kScoreTile));
        const float *rpb_h = rpb ? rpb + head * W : nullptr;
        for (int j = lane; j < kBiasSlots; j += 64) mine[j] = rpb_h && j < W ? rpb_h[j] * kLog2e : 0.f;
#pragma unroll
        for (int vb = 0; vb < NBV; ++vb)
#pragma unroll
            for (int r = 0; r < 4; ++r) bias[vb][r] = bias_at(mine, 16 * vb + 4 * g + r - shift - n + L, W);
    }
    wait_direct();
    barrier_lds();

    float racc[NBV][4];
    f32x4 acck[kSets][CT], accv[kSets][CT];                 // of key blocks kStep * (step + set) + wave of the walk
#pragma unroll
    for (int vb = 0; vb < NBV; ++vb)
#pragma unroll
        for (int r = 0; r < 4; ++r) racc[vb][r] = 0.f;
#pragma unroll
    for (int set = 0; set < kSets; ++set)
#pragma unroll
        for (int ct = 0; ct < CT; ++ct) acck[set][ct] = accv[set][ct] = f32x4{0.f, 0.f, 0.f, 0.f};
    const Rsrc dqs = make_rsrc(dq + in_off, T * in.pitch);
    const bool dq_whole_lines = stores_whole_lines(in.pitch, C, 0);
    const int sc_lane = (4 * g + (n >> 2)) * 32 + (n & 3) * 8;       // transposed read of a score tile
    const int row_lo = 16 * i0, row_hi = min(T, 16 * i1);            // rows this segment owns
    const Rsrc dks = make_rsrc(dk + in_off + (int64_t)row_lo * in.pitch, (row_hi - row_lo) * in.pitch);
    const Rsrc dvs = make_rsrc(dv + in_off + (int64_t)row_lo * in.pitch, (row_hi - row_lo) * in.pitch);
    const bool whole_lines = stores_whole_lines(in.pitch, C, shift);
    const int kp_lo = i0 + (shift >> 4), kp_hi = i1 - 1 + ha;        // key blocks that touch them: complete within the walk
    // The first set's blocks, kStep * step + wave of the walk, to memory; the next sets move up.
    auto emit = [&](int step) {
        const int kp = q0 + kStep * step + wave;
        if (kp >= kp_lo && kp <= kp_hi) {
            const int row_off = (16 * (kp - i0) - shift + n) * in.pitch;    // outside the segment -> dropped
            u32x2 kw[CT], vw[CT];
#pragma unroll
            for (int ct = 0; ct < CT; ++ct) {
                kw[ct] = pack_acc<DT>(acck[0][ct], scale);
                vw[ct] = pack_acc<DT>(accv[0][ct], 1.f);
            }
            store_tile<C>(dks, row_off, kw, g, whole_lines, in.width);
            store_tile<C>(dvs, row_off, vw, g, whole_lines, in.width);
        }
#pragma unroll
        for (int set = 0; set < kSets; ++set)
#pragma unroll
            for (int ct = 0; ct < CT; ++ct) {
                acck[set][ct] = set + 1 < kSets ? acck[set + 1 < kSets ? set + 1 : 0][ct] : f32x4{0.f, 0.f, 0.f, 0.f};
                accv[set][ct] = set + 1 < kSets ? accv[set + 1 < kSets ? set + 1 : 0][ct] : f32x4{0.f, 0.f, 0.f, 0.f};
            }
    };

    int ring = 0;                                           // place of the step's first key tile
#pragma unroll 1
    for (int step = 0; step < steps; ++step) {
        if (step) emit(step - 1);                           // here the stores have the step to finish in
        if (QB == 2 && step + 1 < steps) stage_queries(step + 1);
        LDS_PTR(char) q_now = q_lds + (QB == 2 ? (step & 1) * kBuffer : 0);
        LDS_PTR(char) g_now = q_now + (g_lds - q_lds);
        // ---------------- pass 1: a query tile -> dQ, d rpb, score tiles ----------------
        const int qt = q0 + kStep * step + wave;
        LDS_PTR(char) mine = sc_lds + wave * (NBV * 2 * kScoreTile) + n * 32 + g * 8;     // tile[query n][key slots 4g..4g+3]
        if (kStep * step + wave < qtiles) {
            RowOperand<C> qop, gop;
            read_rows<C>(qop, q_now + wave * LL::kTileBytes, row_lane);
            read_rows<C>(gop, g_now + wave * LL::kTileBytes, row_lane);
            const float row_lse = lse_lds[(step & 1) * 64 + wave * 16 + n];
            const int s0 = 16 * qt - shift;
            const int qrow = 16 * qt + n;
            const bool edge = s0 < 0 || s0 + 16 * NBV > tv;
            const bool own = qt >= i0 && qt < i1;           // the others only contribute their scores
            auto key_tile = [&](int vb) {                   // byte of virtual block vb in the rings
                const int at = ring + wave + vb;
                return (at >= R ? at - R : at) * LL::kTileBytes;
            };
            float p[NBV][4], dp[NBV][4], part = 0.f;
            // With dropout mask D (0 or 1/(1-p)): O = (D*P) V, so dV takes D*P and dP = D * (dO . V^T).
            const uint32_t drop_key = DROP ? dropout_row_key(dropout_row(drop, b, T, qrow), drop) : 0u;
#pragma unroll
            for (int vb = 0; vb < NBV; ++vb) {
                RowOperand<C> kop, vop;
                const int off = key_tile(vb);
                read_rows<C>(kop, k_lds + off, row_lane);
                read_rows<C>(vop, v_lds + off, row_lane);
                const f32x4 s = dot_rows_mma<DT, C>(kop, qop);
                const f32x4 d = dot_rows_mma<DT, C>(vop, gop);
                float z[4];
#pragma unroll
                for (int r = 0; r < 4; ++r) z[r] = __builtin_fmaf(row_lse, -kLog2e, __builtin_fmaf(s[r], scale2, bias[vb][r]));
                if (edge) {
#pragma unroll
                    for (int r = 0; r < 4; ++r) {
                        const uint32_t key = (uint32_t)(s0 + 16 * vb + 4 * g + r);   // unsigned: also key < 0
                        z[r] += (key >= (uint32_t)tv || qrow >= tv) ? mask2 : 0.f;
                    }
                }
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    p[vb][r] = __builtin_amdgcn_exp2f(z[r]);
                    dp[vb][r] = d[r];
                    if constexpr (DROP)
                        dp[vb][r] *= dropout_keeps(drop_key, 16 * vb + 4 * g + r - shift - n + L, drop) ? drop.inv_keep : 0.f;
                    part = __builtin_fmaf(p[vb][r], dp[vb][r], part);
                }
            }
            const float delta = xor_sum(part);
            u32x2 sc[NBV];                                  // dS, rounded to 16 bit
#pragma unroll
            for (int vb = 0; vb < NBV; ++vb) {
                float ds[4];
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    ds[r] = p[vb][r] * (dp[vb][r] - delta);
                    if (own) racc[vb][r] += ds[r];
                    if constexpr (DROP)        // the probability as the forward used it
                        p[vb][r] *= dropout_keeps(drop_key, 16 * vb + 4 * g + r - shift - n + L, drop) ? drop.inv_keep : 0.f;
                }
                sc[vb] = u32x2{Mma<DT>::pack(ds[0], ds[1]), Mma<DT>::pack(ds[2], ds[3])};
                *reinterpret_cast<LDS_PTR(u32x2)>(mine + (2 * vb) * kScoreTile) = u32x2{Mma<DT>::pack(p[vb][0], p[vb][1]), Mma<DT>::pack(p[vb][2], p[vb][3])};
                *reinterpret_cast<LDS_PTR(u32x2)>(mine + (2 * vb + 1) * kScoreTile) = sc[vb];
            }
            if (own) {
                f32x4 acc[CT];
#pragma unroll
                for (int ct = 0; ct < CT; ++ct) acc[ct] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
                for (int vb = 0; vb < NBV; ++vb) {
                    LDS_PTR(char) blk = k_lds + key_tile(vb);
#pragma unroll
                    for (int ct = 0; ct < CT; ++ct) acc[ct] = Mma<DT>::k16(read_tr(blk + tr_lane.off[ct]), sc[vb], acc[ct]);
                }
                u32x2 qw[CT];
#pragma unroll
                for (int ct = 0; ct < CT; ++ct) qw[ct] = pack_acc<DT>(acc[ct], scale);
                store_tile<C>(dqs, qrow * in.pitch, qw, g, dq_whole_lines, in.width);
            }
        } else {
#pragma unroll
            for (int i = 0; i < 2 * NBV; ++i) *reinterpret_cast<LDS_PTR(u32x2)>(mine + i * kScoreTile) = u32x2{0u, 0u};
        }
        barrier_lds();                  // the scores are whole, and every wave is done with the step's first key tiles
        const int next = kStep * step + R;                  // the key tiles that take their place
        if (next < ktiles) {
            stage_direct<C, kStep, kReadShared>(ks, 16 * (q0 + next) - shift, k_lds + ring * LL::kTileBytes, min(kStep, ktiles - next), wave, lane_off, in.pitch);
            stage_direct<C, kStep, kReadShared>(vs, 16 * (q0 + next) - shift, v_lds + ring * LL::kTileBytes, min(kStep, ktiles - next), wave, lane_off, in.pitch);
        }
        ring = ring + kStep == R ? 0 : ring + kStep;
        // ---------------- pass 2: the step's tiles -> dK, dV ----------------
        // (a block's query tiles in their order, wherever its steps begin: the sums are the same however a sequence is cut)
#pragma unroll
        for (int vb = NBV - 1; vb >= 0; --vb) {
            const int tl = (wave - vb) & 3, set = (tl + vb - wave) >> 2;      // tile and block: kp % 4 == wave
            LDS_PTR(char) stile = sc_lds + (tl * NBV + vb) * 2 * kScoreTile + sc_lane;
            const u32x2 pb = read_tr(stile), db = read_tr(stile + kScoreTile);
            u32x2 gt[CT], qt_[CT];
#pragma unroll
            for (int ct = 0; ct < CT; ++ct) {
                gt[ct] = read_tr(g_now + tl * LL::kTileBytes + tr_lane.off[ct]);
                qt_[ct] = read_tr(q_now + tl * LL::kTileBytes + tr_lane.off[ct]);
            }
#pragma unroll
            for (int i = 0; i < kSets; ++i) {
                if (vb < 4 * i - 3 || vb > 4 * i + 3 || set != i) continue;
#pragma unroll
                for (int ct = 0; ct < CT; ++ct) {
                    accv[i][ct] = Mma<DT>::k16(gt[ct], pb, accv[i][ct]);
                    acck[i][ct] = Mma<DT>::k16(qt_[ct], db, acck[i][ct]);
                }
            }
        }
        if (QB == 1 && step + 1 < steps) {
            barrier_lds();
            stage_queries(step + 1);
        }
        wait_direct();
        barrier_lds();
    }
#pragma unroll
    for (int set = 0; set < kSets; ++set) emit(steps - 1 + set);

    LDS_PTR(float) rsum = (LDS_PTR(float))sc_lds;           // [kWaves][kWideSlots]; every wave is done with the scores
    if (drpb) slot_sums<NBV>(rsum, racc, wave, g, n, n + L - shift);
    barrier_lds();
    add_slot_sums(rsum, drpb, drpb_partial, item, head, W, tid);
}

// ---- strips -----------------------------------------------------------------------------
// The same two passes as the two/three-block backward (na1d_mfma.hip): a workgroup stages a strip with the HB + HA query tiles
// around it and all their keys, and nothing more is fetched.  At most kStripQueryTiles query tiles, so that a wave keeps the
// rounded P and dS of its two until the K/V regions can be reused for them; LDS is as large as the strip asks for.
constexpr int kStripQueryTiles = 8;
constexpr int kStripTPW = kStripQueryTiles / kWaves;
static_assert(kStripQueryTiles * 16 <= kThreads, "one lane per staged lse row");

struct StripShape {
    int hb, ha, mt;                      // halo query tiles before / after, strip length
    int kx;                              // key blocks that touch a strip's rows beyond one per tile: 1 unless shift % 16 == 0
};
inline StripShape strip_shape(const WideCover &c) {
    StripShape w;
    w.hb = c.nbv - 1 - (c.shift >> 4);
    w.ha = (c.shift + 15) >> 4;
    w.mt = kStripQueryTiles - w.hb - w.ha;
    w.kx = w.ha - (c.shift >> 4);
    return w;
}

template <class DT, int C, int NBV, bool DROP>
__global__ void __launch_bounds__(kThreads)
wide_bwd_strip_kernel(char *__restrict__ dq, char *__restrict__ dk, char *__restrict__ dv, float *__restrict__ drpb,
                const char *__restrict__ q, const char *__restrict__ k, const char *__restrict__ v,
                const char *__restrict__ dout, const float *__restrict__ lse, const float *__restrict__ rpb,
                const int32_t *__restrict__ t_valid, uint32_t items, int T, int W, int L, int H, int tiles, int nt,
                int strips, float scale, float *__restrict__ drpb_partial, int kv_bytes, uint32_t strips_magic,
                uint32_t heads_magic, Strides in, Strides outl, int shift, Dropout drop, Classes cls) {
    using LL = Lds<C>;
    constexpr int CT = C / 16;
    constexpr int kScoreTile = 16 * 16 * 2;                // one 16x16 tile of 16-bit scores
    fetch_args_now(dq, dk, dv, drpb, q, k, v, dout, lse, rpb, t_valid, items, T, W, L, H, tiles, nt, strips, scale,
                   drpb_partial, kv_bytes, strips_magic, heads_magic, in.sample, in.head, in.pitch, in.width, outl.sample,
                   outl.head, outl.pitch, outl.width, shift);
    if constexpr (DROP) fetch_args_now(drop.threshold, drop.seed_lo, drop.seed_hi, drop.inv_keep, drop.row_stride, drop.row_offset, drop.seq_rows);
    const int hb = NBV - 1 - (shift >> 4), ha = (shift + 15) >> 4;
    const int qtiles = nt + hb + ha;                        // query-side tiles, <= kStripQueryTiles
    const int ktiles = qtiles + NBV - 1;                    // key-side tiles: whole virtual blocks
    // dynamic LDS (strip_lds): [K region | V region] starting at the first key of query tile i0 - hb, reused
    // after pass 1 for the score tiles of the strip's key blocks [((kp - kp_lo) * NBV + vb) * 2 + P/dS] and padded to kv_bytes; Q, dO regions of qtiles
    // tiles; lse of the query-side rows; bias; d rpb slot sums per wave
    extern __shared__ __attribute__((aligned(16))) char smem[];
    const int key_region = region_bytes<C>(ktiles), qry_region = region_bytes<C>(qtiles);
    LDS_PTR(char) k_lds = (LDS_PTR(char))smem;
    LDS_PTR(char) v_lds = k_lds + key_region;
    LDS_PTR(char) sc_lds = k_lds;
    LDS_PTR(char) q_lds = k_lds + kv_bytes;
    LDS_PTR(char) g_lds = q_lds + qry_region;               // dO
    LDS_PTR(float) lse_lds = (LDS_PTR(float))(g_lds + qry_region);
    LDS_PTR(float) bias_lds = lse_lds + kThreads;
    LDS_PTR(float) rsum = bias_lds + kBiasSlots;            // [kWaves][kWideSlots]

    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const WorkItem wi = work_item(blockIdx.x, items, strips, strips_magic, H, heads_magic);
    uint32_t sample = wi.sample;
    const uint32_t item = wi.item, head = wi.head;
    int cr = 0;                                              // residue class of a dilated window
    if (cls.count > 1) {
        cr = split_class(sample, T, cls);
        if constexpr (DROP) drop.row_offset = (uint32_t)cr;
    }
    const uint32_t b = sample * H + head;
    const int i0 = wi.strip * nt, i1 = min(i0 + nt, tiles);
    const int g = lane >> 4, n = lane & 15;
    const int q0 = i0 - hb;                                 // first query-side tile

    const int64_t in_off = sample * in.sample + head * in.head + (int64_t)(cr * cls.in_row);
    const int64_t out_off = sample * outl.sample + head * outl.head + (int64_t)(cr * cls.out_row);
    const int lse_pitch = 4 * cls.d;
    {
        const int key_rows = max(0, min(T, 16 * (q0 + ktiles) - shift));
        const int qry_rows = max(0, min(T, 16 * (q0 + qtiles)));
        const Rsrc ks = make_rsrc(k + in_off, key_rows * in.pitch), vs = make_rsrc(v + in_off, key_rows * in.pitch);
        const Rsrc qs = make_rsrc(q + in_off, qry_rows * in.pitch), gs = make_rsrc(dout + out_off, qry_rows * outl.pitch);
        const Rsrc ls = make_rsrc(lse + ((int64_t)b * cls.rows + cr), T * lse_pitch);
        const int lane_off = direct_lane_offset<C>(wave, lane, in.pitch, in.width);
        const int lane_off_g = direct_lane_offset<C>(wave, lane, outl.pitch, outl.width);
        load_to_lds<4, 0>(ls, (LDS_PTR(char))(lse_lds + 64 * wave), (16 * q0 + tid) * lse_pitch);
        constexpr int KT = kStripQueryTiles + NBV - 1;
        stage_direct<C, KT, kReadShared>(ks, 16 * q0 - shift, k_lds, ktiles, wave, lane_off, in.pitch);
        stage_direct<C, kStripQueryTiles, kReadShared>(qs, 16 * q0, q_lds, qtiles, wave, lane_off, in.pitch);
        stage_direct<C, KT, kReadShared>(vs, 16 * q0 - shift, v_lds, ktiles, wave, lane_off, in.pitch);
        stage_direct<C, kStripQueryTiles, kReadShared>(gs, 16 * q0, g_lds, qtiles, wave, lane_off_g, outl.pitch);
        stage_bias(bias_lds, rpb ? rpb + head * W : nullptr, W, tid);
    }

    int tv = T;
    if (t_valid) tv = max(0, min(T, cls.count > 1 ? class_valid(t_valid[sample], cr, cls) : t_valid[sample]));
    const float scale2 = scale * kLog2e;
    const float mask2 = kMaskValue * kLog2e;

    RowLane<C> row_lane;                // row operands (virtual key blocks and query tiles are whole tiles)
    TrLane<C> tr_lane;                  // transposed operands of the same
    row_lane.init(0, lane);
    tr_lane.init(0, lane);

    wait_direct();
    barrier_lds();
    float bias[NBV][4];
#pragma unroll
    for (int vb = 0; vb < NBV; ++vb)
#pragma unroll
        for (int r = 0; r < 4; ++r) bias[vb][r] = bias_at(bias_lds, 16 * vb + 4 * g + r - shift - n + L, W);

    // ---------------- pass 1: query tiles q0 .. q0 + qtiles - 1 -> dQ, d rpb, score tiles ----------------
    float racc[NBV][4];
#pragma unroll
    for (int vb = 0; vb < NBV; ++vb)
#pragma unroll
        for (int r = 0; r < 4; ++r) racc[vb][r] = 0.f;
    const Rsrc dqs = make_rsrc(dq + in_off, T * in.pitch);
    const bool dq_whole_lines = stores_whole_lines(in.pitch, C, 0);
    u32x2 sc[kStripTPW][NBV][2];         // [tile of this wave][block][P / dS], rounded to 16 bit
#pragma unroll
    for (int jt = 0; jt < kStripTPW; ++jt) {
#pragma unroll
        for (int vb = 0; vb < NBV; ++vb) sc[jt][vb][0] = sc[jt][vb][1] = u32x2{0u, 0u};
        const int tq = wave + jt * kWaves;                  // tile index inside the query-side regions
        const int qt = q0 + tq;
        if (tq >= qtiles || qt < 0 || qt >= tiles) continue;   // nothing there: its scores stay zero
        RowOperand<C> qop, gop;
        read_rows<C>(qop, q_lds + tq * LL::kTileBytes, row_lane);
        read_rows<C>(gop, g_lds + tq * LL::kTileBytes, row_lane);
        const float row_lse = lse_lds[tq * 16 + n];
        const int s0 = 16 * qt - shift;
        const int qrow = 16 * qt + n;
        const bool edge = s0 < 0 || s0 + 16 * NBV > tv;
        float p[NBV][4], dp[NBV][4], part = 0.f;
        // With dropout mask D (0 or 1/(1-p)): O = (D*P) V, so dV takes D*P and dP = D * (dO . V^T).
        const uint32_t drop_key = DROP ? dropout_row_key(dropout_row(drop, b, T, qrow), drop) : 0u;
#pragma unroll
        for (int vb = 0; vb < NBV; ++vb) {
            RowOperand<C> kop, vop;
            const int off = (tq + vb) * LL::kTileBytes;
            read_rows<C>(kop, k_lds + off, row_lane);
            read_rows<C>(vop, v_lds + off, row_lane);
            const f32x4 s = dot_rows_mma<DT, C>(kop, qop);
            const f32x4 d = dot_rows_mma<DT, C>(vop, gop);
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                float z = __builtin_fmaf(row_lse, -kLog2e, __builtin_fmaf(s[r], scale2, bias[vb][r]));
                if (edge) {
                    const uint32_t key = (uint32_t)(s0 + 16 * vb + 4 * g + r);   // unsigned: also key < 0
                    z += (key >= (uint32_t)tv || qrow >= tv) ? mask2 : 0.f;
                }
                p[vb][r] = __builtin_amdgcn_exp2f(z);
                dp[vb][r] = d[r];
                if constexpr (DROP)
                    dp[vb][r] *= dropout_keeps(drop_key, 16 * vb + 4 * g + r - shift - n + L, drop) ? drop.inv_keep : 0.f;
                part = __builtin_fmaf(p[vb][r], dp[vb][r], part);
            }
        }
        const float delta = xor_sum(part);
        const bool own = qt >= i0 && qt < i1;               // halo tiles only contribute their scores
#pragma unroll
        for (int vb = 0; vb < NBV; ++vb) {
            float ds[4];
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                ds[r] = p[vb][r] * (dp[vb][r] - delta);
                if (own) racc[vb][r] += ds[r];
                if constexpr (DROP)        // the probability as the forward used it
                    p[vb][r] *= dropout_keeps(drop_key, 16 * vb + 4 * g + r - shift - n + L, drop) ? drop.inv_keep : 0.f;
            }
            sc[jt][vb][0] = u32x2{Mma<DT>::pack(p[vb][0], p[vb][1]), Mma<DT>::pack(p[vb][2], p[vb][3])};
            sc[jt][vb][1] = u32x2{Mma<DT>::pack(ds[0], ds[1]), Mma<DT>::pack(ds[2], ds[3])};
        }
        if (!own) continue;
        f32x4 acc[CT];
#pragma unroll
        for (int ct = 0; ct < CT; ++ct) acc[ct] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int vb = 0; vb < NBV; ++vb) {
            LDS_PTR(char) blk = k_lds + (tq + vb) * LL::kTileBytes;
#pragma unroll
            for (int ct = 0; ct < CT; ++ct) acc[ct] = Mma<DT>::k16(read_tr(blk + tr_lane.off[ct]), sc[jt][vb][1], acc[ct]);
        }
        u32x2 qw[CT];
#pragma unroll
        for (int ct = 0; ct < CT; ++ct) qw[ct] = pack_acc<DT>(acc[ct], scale);
        store_tile<C>(dqs, qrow * in.pitch, qw, g, dq_whole_lines, in.width);
    }

    if (drpb) slot_sums<NBV>(rsum, racc, wave, g, n, n + L - shift);

    // Pass 2 reads the score tiles of the key blocks that touch the strip's rows, kp_lo .. kp_hi: block vb of query
    // tile tq is key block q0 + tq + vb, and only those in the range are kept (about half of what pass 1 computed).
    const int kp_lo = i0 + (shift >> 4), kp_hi = i1 - 1 + ha;
    barrier_lds();                      // every wave is done with K and V: their regions become the score tiles
#pragma unroll
    for (int jt = 0; jt < kStripTPW; ++jt) {
        const int tq = wave + jt * kWaves;
        if (tq >= qtiles) continue;
        LDS_PTR(char) t = sc_lds + n * 32 + g * 8;          // tile[query n][key slots 4g..4g+3]
#pragma unroll
        for (int vb = 0; vb < NBV; ++vb) {
            const int kp = q0 + tq + vb;
            if (kp < kp_lo || kp > kp_hi) continue;
#pragma unroll
            for (int pd = 0; pd < 2; ++pd)
                *reinterpret_cast<LDS_PTR(u32x2)>(t + (((kp - kp_lo) * NBV + vb) * 2 + pd) * kScoreTile) = sc[jt][vb][pd];
        }
    }
    barrier_lds();

    // ---------------- pass 2: key blocks of the strip -> dK, dV ----------------
    const int sc_lane = (4 * g + (n >> 2)) * 32 + (n & 3) * 8;       // transposed read of a score tile
    const int row_lo = 16 * i0, row_hi = min(T, 16 * i1);            // rows this strip owns
    const Rsrc dks = make_rsrc(dk + in_off + (int64_t)row_lo * in.pitch, (row_hi - row_lo) * in.pitch);
    const Rsrc dvs = make_rsrc(dv + in_off + (int64_t)row_lo * in.pitch, (row_hi - row_lo) * in.pitch);
    const bool whole_lines = stores_whole_lines(in.pitch, C, shift);
    for (int kp = kp_lo + wave; kp <= kp_hi; kp += kWaves) {
        f32x4 acck[CT], accv[CT];
#pragma unroll
        for (int ct = 0; ct < CT; ++ct) acck[ct] = accv[ct] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int vb = NBV - 1; vb >= 0; --vb) {
            const int tq = kp - vb - q0;                    // in [0, qtiles) by the choice of hb and ha
            LDS_PTR(char) qtile = q_lds + tq * LL::kTileBytes;
            LDS_PTR(char) gtile = g_lds + tq * LL::kTileBytes;
            LDS_PTR(char) stile = sc_lds + ((kp - kp_lo) * NBV + vb) * 2 * kScoreTile + sc_lane;
            const u32x2 pb = read_tr(stile), db = read_tr(stile + kScoreTile);
#pragma unroll
            for (int ct = 0; ct < CT; ++ct) {
                accv[ct] = Mma<DT>::k16(read_tr(gtile + tr_lane.off[ct]), pb, accv[ct]);
                acck[ct] = Mma<DT>::k16(read_tr(qtile + tr_lane.off[ct]), db, acck[ct]);
            }
        }
        const int row_off = (16 * (kp - i0) - shift + n) * in.pitch;    // outside the strip -> dropped
        u32x2 kw[CT], vw[CT];
#pragma unroll
        for (int ct = 0; ct < CT; ++ct) {
            kw[ct] = pack_acc<DT>(acck[ct], scale);
            vw[ct] = pack_acc<DT>(accv[ct], 1.f);
        }
        store_tile<C>(dks, row_off, kw, g, whole_lines, in.width);
        store_tile<C>(dvs, row_off, vw, g, whole_lines, in.width);
    }

    add_slot_sums(rsum, drpb, drpb_partial, item, head, W, tid);      // complete at the barriers before pass 2
}

// LDS of a workgroup whose strip is nt tiles long, and the K/V part of it
template <int C>
inline size_t strip_lds(int nt, int nbv, const StripShape &w, int &kv_bytes) {
    const int qtiles = nt + w.hb + w.ha, ktiles = qtiles + nbv - 1;
    kv_bytes = std::max(2 * region_bytes<C>(ktiles), (nt + w.kx) * nbv * 2 * 512);    // K and V, later the score tiles pass 2 reads
    return (size_t)kv_bytes + (size_t)2 * region_bytes<C>(qtiles) +
           (kThreads + kBiasSlots + kWaves * kWideSlots) * sizeof(float);
}

// The split of a walking backward into workgroups: whole sequences where they fill the CUs' places, otherwise the segments of which
// all places are done first: a segment takes its steps and about one more to start, and a launch as many rounds of segments as its
// places ask for.
template <int C, int NBV, bool DROP>
inline Split walk_split(const Geom &g, const WideCover &c) {
    const int64_t B = g.B * g.classes, places = 256 * std::min(wide_bwd_waves<C, NBV, DROP>(), 4);
    const int halo = c.nbv - 1 + ((c.shift & 15) ? 1 : 0);
    Split best{};
    int64_t least = INT64_MAX;
    for (int want = 1, tiles = (int)((g.T + 15) / 16); want <= tiles; want += 1 + want / 8) {
        Split sp;
        sp.tiles = tiles, sp.nt = (tiles + want - 1) / want, sp.strips = (tiles + sp.nt - 1) / sp.nt, sp.items = B * sp.strips;
        const int64_t cost = (sp.items + places - 1) / places * ((std::min(tiles, sp.nt + halo) + kStep - 1) / kStep + 1);
        if (cost < least) least = cost, best = sp;
        if (B * sp.strips >= 4 * places) break;
    }
    return best;
}

// How a backward runs: in strips or walking.
struct WidePlan {
    Split sp;
    bool strips;
    int kv_bytes;
    size_t lds;
};
// Walking saves the halo and pays for it with one wave's work behind the other, LDS for four tiles of everything, and its rings.
// Below, us of launches one behind the other, walking and in strips, 8 heads:
//   - A sequence that is one strip has no halo, and a strip takes the LDS that it asks for: 976 x 32 rows x 32 channels, W = 65:
//     17.2 and 12.9; 3904 x 16 x 64, W = 80: 123 and 63; 976 x 64 x 64, W = 49: 18.3 and 18.6.  Not where fewer of its workgroups
//     fit a CU (976 x 64 x 64, W = 65: 29 and 34), nor where a wave would have two tiles (from five on) and CUs stay idle: 24 x 64
//     x 128, W = 49, in one strip and in four 10.5 and 9.0.
//   - While strips find a CU, or a place on one, for themselves, theirs is the shorter chain: a workgroup to a CU for 64 (with
//     three or four blocks one and a half) and 128 channels, three for fewer (d rpb's atomics of a head meet, hence by the
//     heads): 8 x 200 x 128, W = 65: 17.0 and 10.4; 32 of them 17.6 and 11.5, 152: 30.7 and 33; 104 x 300 x 32, W = 65: 13.7 and
//     11.3, 416: 19.6 and 28.
template <int C, int NBV, bool DROP>
inline WidePlan wide_bwd_plan(const Geom &g, const WideCover &c) {
    WidePlan p{};
    const StripShape w = strip_shape(c);
    const int64_t B = g.B * g.classes;
    const int few = C <= 32 ? 128 * std::min(g.H, 6) : C == 64 && NBV < 5 ? 384 : 256;
    int mt = w.mt;
    while (strip_lds<C>(mt, NBV, w, p.kv_bytes) > kCuLds) --mt;          // a strip of one tile always fits
    const Split spread = make_split(B, g.T, mt, 256), whole = make_split(B, g.T, mt, 0);
    const bool one = whole.strips == 1 && std::min<int64_t>(kCuLds / strip_lds<C>(whole.nt, NBV, w, p.kv_bytes), 4) >= wide_bwd_places<C, NBV>();
    p.strips = true;
    if (one && whole.tiles <= kWaves)
        p.sp = C >= 64 && spread.items <= 128 ? spread : whole;
    else if (spread.items <= few)
        p.sp = spread;
    else if (one)
        p.sp = whole;
    else
        p.strips = false, p.sp = walk_split<C, NBV, DROP>(g, c);
    p.lds = p.strips ? strip_lds<C>(p.sp.nt, NBV, w, p.kv_bytes) : wide_bwd_lds<C, NBV>();
    return p;
}

template <class DT, int C, int NBV>
int launch_wide_bwd_n(void *dq, void *dk, void *dv, float *drpb, const void *q, const void *k, const void *v,
                      const void *dout, const float *lse, const float *rpb, const int32_t *t_valid, const Geom &g,
                      const Layout &in, const Layout &outl, float scale, const WideCover &c, float *workspace,
                      int64_t workspace_bytes, hipStream_t s) {
    const WidePlan p = g.drop.threshold ? wide_bwd_plan<C, NBV, true>(g, c) : wide_bwd_plan<C, NBV, false>(g, c);
    const Split &sp = p.sp;
    static_assert(wide_bwd_lds<C, NBV>() <= kCuLds, "LDS of a CU");
    if (!items_ok(sp, g) || !strides_ok(in, g) || !strides_ok(outl, g)) return NA1D_ERR_UNSUPPORTED;
    float *partial = nullptr;          // as in the two/three-block backward: a workspace is used or refused
    if (drpb && workspace) {
        if (workspace_bytes < sp.items * kWidePartialStride * (int64_t)sizeof(float)) return NA1D_ERR_WORKSPACE;
        partial = workspace;
    }
    auto go = [&](auto kern, const char *name, auto... kv_bytes) {
        if (!allow_lds(kern, p.lds)) return (int)NA1D_ERR_LAUNCH;
        note_kernel(name, DT::tag, C, NBV, g.drop.threshold != 0);
        launch_kernel(kern, (unsigned)sp.items, p.lds, s, (char *)dq, (char *)dk, (char *)dv, drpb, (const char *)q,
                      (const char *)k, (const char *)v, (const char *)dout, lse, rpb, t_valid, (uint32_t)sp.items, (int)g.T,
                      g.W, g.L, g.H, sp.tiles, sp.nt, sp.strips, scale, partial, kv_bytes..., div_magic(sp.strips), div_magic(g.H),
                      byte_strides(in, g), byte_strides(outl, g), c.shift, g.drop, classes_of(g, in, outl));
        return (int)NA1D_OK;
    };
    const int st = p.strips ? go(g.drop.threshold ? wide_bwd_strip_kernel<DT, C, NBV, true> : wide_bwd_strip_kernel<DT, C, NBV, false>, "wide_bwd_strip_kernel", p.kv_bytes)
                            : go(g.drop.threshold ? wide_bwd_kernel<DT, C, NBV, true> : wide_bwd_kernel<DT, C, NBV, false>, "wide_bwd_kernel");
    if (st != NA1D_OK) return st;
    if (partial && drpb && !launch_events().refused)
        drpb_reduce_kernel<kWidePartialStride><<<(unsigned)(g.H * g.W), 128, 0, s>>>(drpb, partial, (int)(g.B / g.H * g.classes), g.H,
                                                                                     sp.strips, g.W);
    return launch_status();
}

template <class DT, int C>
int launch_wide_bwd(void *dq, void *dk, void *dv, float *drpb, const void *q, const void *k, const void *v,
                    const void *dout, const float *lse, const float *rpb, const int32_t *t_valid, const Geom &g,
                    const Layout &in, const Layout &outl, float scale, float *workspace, int64_t workspace_bytes,
                    hipStream_t s) {
    const WideCover c = wide_cover(g);
    switch (c.nbv) {
        case 3: return launch_wide_bwd_n<DT, C, 3>(dq, dk, dv, drpb, q, k, v, dout, lse, rpb, t_valid, g, in, outl, scale, c, workspace, workspace_bytes, s);
        case 4: return launch_wide_bwd_n<DT, C, 4>(dq, dk, dv, drpb, q, k, v, dout, lse, rpb, t_valid, g, in, outl, scale, c, workspace, workspace_bytes, s);
        case 5: return launch_wide_bwd_n<DT, C, 5>(dq, dk, dv, drpb, q, k, v, dout, lse, rpb, t_valid, g, in, outl, scale, c, workspace, workspace_bytes, s);
        case 6: return launch_wide_bwd_n<DT, C, 6>(dq, dk, dv, drpb, q, k, v, dout, lse, rpb, t_valid, g, in, outl, scale, c, workspace, workspace_bytes, s);
    }
    return NA1D_ERR_UNSUPPORTED;
}

// d rpb: float atomics, or - given a workspace of wide_bwd_workspace_bytes() - per-workgroup partial rows that a second
// kernel folds in a fixed order.
int wide_bwd(void *dq, void *dk, void *dv, float *drpb, const void *q, const void *k, const void *v, const void *dout,
             const float *lse, const float *rpb, const int32_t *t_valid, const Geom &g, const Layout &in,
             const Layout &outl, float scale, int dtype, float *workspace, int64_t workspace_bytes, hipStream_t s) {
    if (!wide_cover(g).nbv) return NA1D_ERR_UNSUPPORTED;
    NA1D_MFMA_DISPATCH(launch_wide_bwd, dq, dk, dv, drpb, q, k, v, dout, lse, rpb, t_valid, g, in, outl, scale, workspace,
                       workspace_bytes, s);
}

// For launches with dropout and without, whichever has more workgroups.
template <int C, int NBV> int64_t most_items(const Geom &g, const WideCover &c) {
    return std::max(wide_bwd_plan<C, NBV, false>(g, c).sp.items, wide_bwd_plan<C, NBV, true>(g, c).sp.items);
}
template <int C> int64_t wide_workspace(const Geom &g, const WideCover &c) {
    const int64_t items = c.nbv == 3 ? most_items<C, 3>(g, c) : c.nbv == 4 ? most_items<C, 4>(g, c) : c.nbv == 5 ? most_items<C, 5>(g, c) : most_items<C, 6>(g, c);
    return items * kWidePartialStride * (int64_t)sizeof(float);
}
int64_t wide_bwd_workspace_bytes(const Geom &g) {
    const WideCover c = wide_cover(g);
    if (!c.nbv) return 0;
    switch (padded_width(g.C)) {
        case 16: return wide_workspace<16>(g, c);
        case 32: return wide_workspace<32>(g, c);
        case 64: return wide_workspace<64>(g, c);
        case 128: return wide_workspace<128>(g, c);
    }
    return 0;
}

}  // namespace mfma
}  // namespace na1d
