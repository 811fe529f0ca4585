// The attention of several layers that cannot see each other's writes, a KV head at a time: the second form of
// llmi_hip_mha_decode_append_stack's one launch (the first, and how the layers are told to be independent, is in mha_stack.hip).
//
// The work is layers x KV heads, and with a dozen layers and more there are about as many of those as compute units: a workgroup
// takes a KV head of a layer whole. It walks the head's splits in rounds, one after the other or a few short ones side by side, the tiles of all
// of them (and of its next head) as one sequence through the LDS rings, and keeps a split's folded row in registers, so that nothing has to be handed
// over: no partial rows in memory, no records, no waits for anybody. The splits, the tiles of a split's wavefronts, the folds and
// the merge are those of one launch per layer, in the same order: same bits. What bounds it is the K/V stream.
//
// Where the heads do not come out even with the workgroups (288 of 36 layers on 256), the last ones are cut in `parts` at split
// boundaries. A part that is not the head's last one leaves its splits' rows and records in the workspace, the last one
// brings them into its registers and merges. Parts are handed out ahead of the whole heads, consecutive workgroups taking the
// parts of a head, the last part the highest: the only wait (bounded) is for workgroups that were started earlier and wait for nobody.
//
// us, this form : the stream by layers (mha_layers_kernel), 32 Q / 8 KV heads: 36 layers at 4096 + 1 positions 95 : 107 (6.4 TB/s), at
// 300 22 : 55, 64 layers at 1000 51 : 105; 28 layers of 16 Q heads at 1000 25 : 43. Against one launch per layer, 64 Q / 8 KV heads:
// 64 layers at 3000 135 : 413, 36 at 1000 36 : 199, at 1100 52 : 203, 8 at 300 11 : 44; single passes, 12 layers of 32 Q heads at 150 8 : 51.
// Short lengths are bound by instructions, one or two wavefronts to a SIMD, not by the tiles' way: four wavefronts 0.75 us per round and 0.57 per
// tile; eight, by the clock in the kernel (23 layers at 384, 64 at 250, 36 at 1000 and at 1100 positions), 0.02 - 0.2 us waiting for a tile, 0.5 - 0.9
// folding it, 0.5 - 0.8 from there to the barrier, 0.4 - 1.3 at it, 0.5, 0.8 or 1.7 folding two, four or eight splits.
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "mha_device_helpers.h"

namespace llmi {
namespace {

constexpr int kWaves = 8;
constexpr int kMaxSplitsKept = 32;  // splits of a head, at most: half of their rows in the registers of a folding wavefront, four per lane and row

// NW wavefronts (of eight) stream, with a ring of NSTAGE tiles each: as many as a split has in the launch this stands for. With four
// the others fold and bring in operands.
// P: splits at a time. Where a split has no more than NW / P tiles, P consecutive splits are taken side by side, T = NW / P wavefronts each, a tile or
// none to a wavefront: a round (its tile, the barrier, the folds) costs about the same whatever it holds, and with one split a round most
// wavefronts had nothing to do in it. A wavefront without a tile adds nothing to a fold (weight zero), so the bits are those of NW wavefronts.
// us, one split at a time : side by side, groups of 8 (eight wavefronts): 64 layers at 250 positions 56.2 : 25.6, 23 at 384 31.0 : 16.8, 64 at 900 62.0 : 48.3,
// 36 at 1100 71.5 : 52.1, 20 at 1900 59.9 : 43.9, 4 at 300 12.2 : 10.4; groups of 4 (four wavefronts) 36 at 300 29.5 : 21.8, 64 at 400 44.3 : 29.5, 20 at 200
// 13.7 : 10.2; groups of 2 28 at 500 21.7 : 15.8, 4 at 200 level.
template <int G, int NW, int NSTAGE, int P>
__global__ __launch_bounds__(kWaves * 64, 2) void mha_heads_kernel(HeadsArgs ha) {
    const KernelArgs& a = ha.st.a;
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    constexpr int T = NW / P;
    const int sub = P == 1 ? 0 : wave / T, tw = P == 1 ? wave : wave % T;  // streaming: which split of a round, which of its tiles first
    const int n16 = lane & 15;
    const int kg = lane >> 4;
    const int S = a.num_splits;
    const int cached_len = a.seq_len - 1;
    const int run = a.tiles_run, longer = a.tiles_longer;
    const int items = ha.items, stride = (int)gridDim.x;

    constexpr int kStageBytes = 8192;
    constexpr int kRingBytes = NW * NSTAGE * kStageBytes;
    constexpr int kQSlots = (G * 16 + 63) / 64;
    constexpr int kOperandBytes = (2 + kQSlots) * 1024;  // q_norm | k_norm | sin | cos, new K row | new V row, the query rows
    constexpr int kFoldRows = NW * G * kHeadDim * (int)sizeof(float);
    constexpr int kFoldBytes = kFoldRows + 2 * NW * G * (int)sizeof(float);
    constexpr int kPairs = G * kMaxSplitsKept;  // (head, split)
    constexpr int kSmemBytes = kRingBytes + 2 * kOperandBytes + 2 * kFoldBytes + 4 * kPairs * (int)sizeof(float) + G * kHeadDim * (int)sizeof(float);
    static_assert(kSmemBytes <= 160 * 1024, "LDS of one compute unit");
    static_assert(kFoldBytes % 16 == 0, "16-byte accesses");
    __shared__ __attribute__((aligned(1024))) char smem[kSmemBytes];
    char* operands = smem + kRingBytes;
    char* folds = operands + 2 * kOperandBytes;
    float* s_m = reinterpret_cast<float*>(folds + 2 * kFoldBytes);  // [G][kMaxSplitsKept]: the splits' maxima ...
    float* s_l = s_m + kPairs;                                      // ... sums ...
    float* s_w = s_l + kPairs;                                      // ... and weights (a copy for either half of the folding wavefronts)
    float* s_odd = s_w + 2 * kPairs;                                // [G][128]: the odd splits' weighted sum
    auto fold_o = [&](int set, int w, int h) { return reinterpret_cast<float*>(folds + set * kFoldBytes) + (w * G + h) * kHeadDim; };
    auto fold_m = [&](int set, int w, int h) { return reinterpret_cast<float*>(folds + set * kFoldBytes + kFoldRows) + w * G + h; };
    auto fold_l = [&](int set, int w, int h) { return fold_m(set, NW + w, h); };
    // This wavefront's LDS accesses are done, then all wavefronts meet. (Requests to memory stay in flight.)
    auto meet = [&]() {
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
    };

    // An item: splits lo .. hi-1 of a KV head of a layer; cut: the head's number among the cut ones, or -1.
    struct Item {
        int layer, kvh, lo, hi, cut;
    };
    const int cut_items = ha.cut_heads * ha.parts;
    auto item_at = [&](int i) {
        Item it;
        int head = i - cut_items;
        it.lo = 0;
        it.hi = S;
        it.cut = -1;
        if (i < cut_items) {
            it.cut = i / ha.parts;
            const int part = i - it.cut * ha.parts;
            it.lo = part * S / ha.parts;
            it.hi = (part + 1) * S / ha.parts;
            head = items - cut_items + it.cut;
        }
        it.layer = head / ha.n_kv;
        it.kvh = head - it.layer * ha.n_kv;
        return it;
    };
    struct Unit {
        int nrows, n_my;
    };
    auto unit_at = [&](int split) {
        Unit u;
        const int ntiles = run + (split < longer ? 1 : 0);
        u.nrows = min(ntiles * kTile, cached_len - (split * run + min(split, longer)) * kTile);
        u.n_my = tw < ntiles ? (ntiles - tw + T - 1) / T : 0;
        return u;
    };

    // ---- streaming: the tiles of all this workgroup's splits, as one sequence per wavefront ----
    const uint32_t rs = (uint32_t)a.row_stride * 2u;
    const uint32_t k_row = (uint32_t)kg * rs;
    const uint32_t k_col0 = (uint32_t)(n16 ^ kg) * 16u;
    const uint32_t k_col1 = (uint32_t)(n16 ^ (4 + kg)) * 16u;
    const uint32_t k_rd = (uint32_t)((n16 >> 2) * 1024 + (n16 & 3) * 256);
    const uint32_t k_rd0 = k_rd + (uint32_t)((kg ^ (n16 & 7)) * 16);
    const uint32_t k_rd1 = k_rd + (uint32_t)(((4 + kg) ^ (n16 & 7)) * 16);
    const uint32_t v_col = (uint32_t)n16 * 16u;
    char* my_ring = smem + (wave < NW ? wave : 0) * NSTAGE * kStageBytes;
    const uint32_t my_ring_lds = (uint32_t)(uintptr_t)my_ring;
    int is_item = (int)blockIdx.x, is_split = 0, is_tile = 0, is_stage = 0, in_flight = 0, rd_stage = 0;
    bool is_live = wave < NW;
    Item is_it = item_at(is_item);
    int is_begin = 0, is_nrows = 0, is_n = 0;  // the split's first position and rows, the wavefront's tiles of it
    const char *is_kb = nullptr, *is_vb = nullptr;
    auto open_item = [&]() {
        is_split = is_it.lo + sub;
        is_begin = (is_split * run + min(is_split, longer)) * kTile;
        const int64_t off = (int64_t)is_it.layer * ha.st.cache_stride + (int64_t)is_it.kvh * a.head_stride + (int64_t)is_begin * a.row_stride;
        is_kb = reinterpret_cast<const char*>(a.k + off);
        is_vb = reinterpret_cast<const char*>(a.v + off);
    };
    auto open_split = [&]() {
        const int ntiles = P > 1 && is_split >= is_it.hi ? 0 : run + (is_split < longer ? 1 : 0);
        is_nrows = min(ntiles * kTile, cached_len - is_begin);
        is_n = tw < ntiles ? (ntiles - tw + T - 1) / T : 0;
        is_tile = 0;
    };
    // To the wavefront's next split with a tile for it. (A head's splits follow one another in memory.)
    auto next_split = [&]() {
        do {
            // (rows of this split and the P - 1 behind it)
            const int rows = (P == 1 ? run + (is_split < longer ? 1 : 0) : P * run + min(is_split + P, longer) - min(is_split, longer)) * kTile;
            is_begin += rows;
            is_kb += (uint32_t)rows * rs;
            is_vb += (uint32_t)rows * rs;
            is_split += P;
            if (is_split >= is_it.hi) {
                is_item += stride;
                if (is_item >= items) {
                    is_live = false;
                    return;
                }
                is_it = item_at(is_item);
                open_item();
            }
            open_split();
        } while (is_n == 0);
    };
    auto issue_next = [&]() {
        if (!is_live) return;
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");  // the slot's previous contents have reached the VGPRs
        const uint32_t last_off = (uint32_t)(is_nrows - 1) * rs;  // (rows past the split's last one: masked out of the softmax)
        const uint32_t base = (uint32_t)(tw + is_tile * T) * (kTile * rs);
        const uint32_t slot = my_ring_lds + (uint32_t)is_stage * kStageBytes;
        if constexpr (P > 1) scalar_bases(is_kb, is_vb);  // (one split at a time they are scalar throughout)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const uint32_t ko = min(base + k_row + (uint32_t)(4 * i) * rs, last_off) + ((i & 1) ? k_col1 : k_col0);
            dma16(is_kb, ko, slot + i * 1024);
        }
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const uint32_t vo = min(base + k_row + (uint32_t)(4 * i) * rs, last_off) + v_col;
            dma16(is_vb, vo, slot + 4096 + i * 1024);
        }
        ++in_flight;
        is_stage = is_stage + 1 == NSTAGE ? 0 : is_stage + 1;
        if (++is_tile == is_n) next_split();
    };

    // ---- the small operands, two items' worth: one wavefront brings in an item's while the one before it streams ----
    constexpr int kOperandWave = kWaves - 1;
    const int c16 = lane & 15, which = lane >> 4;
    auto fetch_operands = [&](const Item& it, int set) {
        const uint32_t st = (uint32_t)(uintptr_t)(operands + set * kOperandBytes);
        const float* sin_row = a.sin_cache + (int64_t)cached_len * 64;
        const float* cos_row = a.cos_cache + (int64_t)cached_len * 64;
        const uint64_t w_base = reinterpret_cast<uint64_t>(a.norm_w + (int64_t)it.layer * ha.st.normw_stride) + (uint64_t)(which & 1) * 256u;
        const uint64_t t_base = reinterpret_cast<uint64_t>(which == 2 ? sin_row : cos_row);
        dma16_gather(reinterpret_cast<const void*>((which < 2 ? w_base : t_base) + (uint64_t)c16 * 16u), st);
        if (it.hi == S) {
            const uint16_t* kn = a.k_new + (int64_t)it.layer * ha.st.knew_stride;
            const uint16_t* vn = a.v_new + (int64_t)it.layer * ha.st.vnew_stride;
            const uint64_t p1 = reinterpret_cast<uint64_t>((which & 1) == 0 ? kn : vn) + (uint64_t)(it.kvh * kHeadDim * 2 + c16 * 16);
            dma16_gather(reinterpret_cast<const void*>(p1), st + 1024);
        }
#pragma unroll
        for (int i = 0; i < kQSlots; ++i) {
            const int head = min(which + 4 * i, a.group - 1);
            dma16_gather(a.q + (int64_t)it.layer * ha.st.q_stride + (int64_t)(it.kvh * a.group + head) * kHeadDim + c16 * 8,
                         st + (uint32_t)(2 + i) * 1024);
        }
    };
    // Normalises and rotates the query group and the new K row, files the new token's rows in the cache.
    auto prepare_operands = [&](const Item& it, int set) {
        char* ops = operands + set * kOperandBytes;
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
#pragma unroll
        for (int b4 = 0; b4 < kQSlots; ++b4) norm_rope_rows_lds<true>(ops + 2048, ops, ops + 512, ops + 768, 4 * b4 + kg, n16, a.eps);
        if (it.hi == S) {
            norm_rope_rows_lds<true>(ops + 1024, ops + 256, ops + 512, ops + 768, 0, n16, a.eps);
            asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
            const u32x4* rows = reinterpret_cast<const u32x4*>(ops + 1024);
            const int64_t row_off = (int64_t)it.layer * ha.st.cache_stride + (int64_t)cached_len * a.row_stride + it.kvh * a.slot_head_stride;
            uint16_t* dst = const_cast<uint16_t*>(which == 0 ? a.k : a.v) + row_off;
            if (which < 2) *reinterpret_cast<u32x4*>(dst + c16 * 8) = rows[which * 16 + c16];
        }
    };

    // ---- folding: one thread per (head, 16-byte column), for the even splits and for the odd ones; their rows in registers ----
    constexpr int kFoldBase = NW == 4 ? 4 : 0;
    constexpr int kFoldWaves = (G * (kHeadDim / 4) + 63) / 64;
    static_assert(kFoldBase + 2 * kFoldWaves <= kWaves, "");
    const bool folds_here = wave >= kFoldBase && wave < kFoldBase + 2 * kFoldWaves;
    const int parity = folds_here && wave >= kFoldBase + kFoldWaves ? 1 : 0;
    const int fw = wave - kFoldBase - parity * kFoldWaves;  // folds heads 2 * fw and 2 * fw + 1
    const int fu = fw * 64 + lane;
    const int fh = folds_here ? min(fu >> 5, a.group - 1) : 0, c4 = lane & 31;
    const bool f_active = folds_here && fu < a.group * (kHeadDim / 4);
    constexpr int kRows = kMaxSplitsKept / 2;
    f32x4 rows[kRows];  // of splits 2 * i + parity
#pragma unroll
    for (int i = 0; i < kRows; ++i) rows[i] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
    const uint32_t tag = 0x80000000u | (a.tag & 0x7fffffffu);
    // Workspace: per cut head and query head pub_splits rows; behind all of them the records (tag, max, tag, sum).
    const uint32_t cut_rows = (uint32_t)ha.cut_heads * (uint32_t)(a.group * ha.pub_splits);
    const __amdgpu_buffer_rsrc_t part_rsrc = __builtin_amdgcn_make_buffer_rsrc(a.ws, 0, (int)(cut_rows * (kHeadDim * 4u + 16u)), 0x00020000);
    auto row_number = [&](int cut, int h, int split) { return (uint32_t)((cut * a.group + h) * ha.pub_splits + split); };
    auto record_at = [&](uint32_t row) { return cut_rows * (kHeadDim * 4u) + row * 16u; };

    if (is_live) {
        open_item();
        open_split();
        if (is_n == 0) next_split();
        for (int s0 = 0; s0 < NSTAGE; ++s0) issue_next();
    }
    if (wave == kOperandWave) {
        const Item first = item_at((int)blockIdx.x);
        fetch_operands(first, 0);
        prepare_operands(first, 0);
    }
    meet();  // the first item's operands are in LDS

    // The query group as the streaming wavefronts' operand.
    u32x4 qb[4];
    auto read_query = [&](int set) {
        const u32x4* ops4 = reinterpret_cast<const u32x4*>(operands + set * kOperandBytes);
        const int hq_local = min(n16, a.group - 1);
        const bool live = n16 < a.group;
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const u32x4 qv = ops4[128 + hq_local * 16 + j * 4 + kg];
            qb[j] = live ? qv : u32x4{0u, 0u, 0u, 0u};
        }
    };
    // The wavefront's tiles of its split of the round, `round` the first one, folded, and its result left in LDS.
    auto stream_round = [&](const Item& it, int round, int op_set, int fold_set) {
        const int split = round + sub;
        if (P > 1 && split >= it.hi) return;  // (nobody folds it)
        const u32x4* ops4 = reinterpret_cast<const u32x4*>(operands + op_set * kOperandBytes);
        const Unit u = unit_at(split);
        float m_run = -INFINITY, l_run = 0.0f;
        f32x4 o[8];
#pragma unroll
        for (int j = 0; j < 8; ++j) o[j] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
        if (split == S - 1 && tw == 0) {
            u32x4 kf[4], vf;
            start_from_new_row(ops4 + 64, ops4 + 80, qb, kg, n16, a.scale_log2e, kf, vf, m_run, l_run, o);
        }
        for (int i = 0; i < u.n_my; ++i) {
            TileRegs r;
            // (other requests of this wavefront, an item's operands or results, only make this wait for more)
            wait_tiles_in_flight(in_flight - 1);
            const char* kp = my_ring + rd_stage * kStageBytes;
#pragma unroll
            for (int j = 0; j < 4; ++j)
                r.k[j] = *reinterpret_cast<const u32x4*>(kp + ((j & 1) ? k_rd1 : k_rd0) + (j >> 1) * 128);
#pragma unroll
            for (int e = 0; e < 4; ++e)
                r.v[e] = *reinterpret_cast<const u32x4*>(kp + 4096 + kg * 1024 + e * 256 + n16 * 16);
            rd_stage = rd_stage + 1 == NSTAGE ? 0 : rd_stage + 1;
            --in_flight;
            issue_next();
            fold_tile<G>(r, qb, (tw + i * T) * kTile + 4 * kg, u.nrows, a.scale_log2e, m_run, l_run, o);
        }
        l_run = rows_sum(l_run);
#pragma unroll
        for (int r4 = 0; r4 < 4; ++r4) {
            const int h = 4 * kg + r4;
            if (h < G) {
                float* dst = fold_o(fold_set, wave, h) + n16 * 8;
                *reinterpret_cast<f32x4*>(dst) = f32x4{o[0][r4], o[1][r4], o[2][r4], o[3][r4]};
                *reinterpret_cast<f32x4*>(dst + 4) = f32x4{o[4][r4], o[5][r4], o[6][r4], o[7][r4]};
            }
        }
        if (kg == 0 && n16 < G) {
            *fold_m(fold_set, wave, n16) = m_run;
            *fold_l(fold_set, wave, n16) = l_run;
        }
    };
    // The wavefronts' results of a split into one row.
    auto fold_split = [&](const Item& it, int round, int split, int fold_set) {
        const int w0 = P == 1 ? 0 : (split - round) * T;
        float mw[T], lw[T];
        f32x4 ow[T];
#pragma unroll
        for (int w = 0; w < T; ++w) {
            mw[w] = *fold_m(fold_set, w0 + w, fh);
            lw[w] = *fold_l(fold_set, w0 + w, fh);
            ow[w] = *reinterpret_cast<const f32x4*>(fold_o(fold_set, w0 + w, fh) + c4 * 4);
        }
        float mx = -INFINITY;
#pragma unroll
        for (int w = 0; w < T; ++w) mx = fmaxf(mx, mw[w]);
        f32x4 acc = {0.0f, 0.0f, 0.0f, 0.0f};
        float lsum = 0.0f;
#pragma unroll
        for (int w = 0; w < T; ++w) {
            const float f = (mw[w] == -INFINITY) ? 0.0f : fast_exp2(mw[w] - mx);
            acc += ow[w] * f;
            lsum += lw[w] * f;
        }
        if (f_active && c4 == 0) {
            s_m[fh * kMaxSplitsKept + split] = mx;
            s_l[fh * kMaxSplitsKept + split] = lsum;
        }
        if (it.hi == S) {
            // (the register number is fixed in the code: a branch to the four it may be, and a select of those)
#pragma unroll
            for (int g = 0; g < kRows; g += 4) {
                if (split >> 3 == g >> 2) {
#pragma unroll
                    for (int i = g; i < g + 4; ++i)
#pragma unroll
                        for (int e = 0; e < 4; ++e) rows[i][e] = split >> 1 == i ? acc[e] : rows[i][e];
                }
            }
        } else if (f_active) {
            __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u32x4, acc), part_rsrc,
                                                   row_number(it.cut, fh, split) * (kHeadDim * 4u) + (uint32_t)c4 * 16u, 0, kCacheDevice);
        }
    };
    // An item's end: what crosses between workgroups ...
    auto hand_over = [&](const Item& it) {
        if (folds_here && it.hi != S) {
            // A part that others merge: its records, once its rows are acknowledged.
            asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory");
#pragma unroll
            for (int hh = 0; hh < 2; ++hh) {
                const int h = 2 * fw + hh;
                if (h < a.group && lane >= it.lo && lane < it.hi && (lane & 1) == parity)
                    __builtin_amdgcn_raw_buffer_store_b128(u32x4{tag, __builtin_bit_cast(uint32_t, s_m[h * kMaxSplitsKept + lane]), tag,
                                                                 __builtin_bit_cast(uint32_t, s_l[h * kMaxSplitsKept + lane])},
                                                           part_rsrc, record_at(row_number(it.cut, h, lane)), 0, kCacheDevice);
            }
        } else if (folds_here && it.lo > parity) {
            // The other parts' splits of this wavefront's parity (a lane each, for both of its heads).
            u32x4 rec[2];
            bool arrived = false;
            const bool mine = lane < it.lo && (lane & 1) == parity;
            const int sp = mine ? lane : parity;
            for (int spin = 0; spin < a.max_polls && !arrived; ++spin) {
                bool here = true;
#pragma unroll
                for (int hh = 0; hh < 2; ++hh) {
                    const int h = min(2 * fw + hh, a.group - 1);
                    asm volatile("" ::: "memory");  // (a poll is a load of its own)
                    rec[hh] = __builtin_bit_cast(
                        u32x4, __builtin_amdgcn_raw_buffer_load_b128(part_rsrc, record_at(row_number(it.cut, h, sp)), 0, kCacheDevice));
                    here = here && rec[hh][0] == tag && rec[hh][2] == tag;
                }
                arrived = __all(here);
            }
            asm volatile("" ::: "memory");  // (the rows are asked for behind the last poll)
            if (__builtin_expect(!arrived, 0)) {
                if (lane == 0) atomicAdd(&g_poll_timeouts, 1u);
            } else {
#pragma unroll
                for (int i = 0; i < kRows; ++i)
                    if (2 * i + parity < it.lo)
                        rows[i] = __builtin_bit_cast(
                            f32x4, __builtin_amdgcn_raw_buffer_load_b128(
                                       part_rsrc, row_number(it.cut, fh, 2 * i + parity) * (kHeadDim * 4u) + (uint32_t)c4 * 16u, 0, kCacheDevice));
                // (a wait the compiler knows of: with loads that may be outstanding it would put one for everything, tiles too, in front
                // of every later write to these registers)
                __builtin_amdgcn_s_waitcnt(0x0f70);  // vmcnt(0)
            }
#pragma unroll
            for (int hh = 0; hh < 2; ++hh) {
                const int h = 2 * fw + hh;
                if (h < a.group && mine) {
                    const uint32_t m_bits = rec[hh][1], l_bits = rec[hh][3];
                    // (a wait that gave up makes the whole head NaN)
                    s_m[h * kMaxSplitsKept + lane] = arrived ? __builtin_bit_cast(float, m_bits) : 0.0f;
                    s_l[h * kMaxSplitsKept + lane] = arrived ? __builtin_bit_cast(float, l_bits) : __builtin_nanf("");
                    // (cleared: a replay of this launch carries the same tag)
                    __builtin_amdgcn_raw_buffer_store_b128(u32x4{0u, 0u, 0u, 0u}, part_rsrc, record_at(row_number(it.cut, h, lane)), 0,
                                                           kCacheDevice);
                }
            }
        }
    };
    // ... the weighted rows of the even and of the odd splits, once every split's (max, sum) is in LDS ...
    f32x4 sum = {0.0f, 0.0f, 0.0f, 0.0f};
    float den = 0.0f;
    auto weigh = [&](const Item& it) {
        sum = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
        if (folds_here && it.hi == S) {
            // Weights e^(m_s - M) and the denominator, lane = split; then this half's rows.
            float* w = s_w + parity * kPairs;
#pragma unroll
            for (int hh = 0; hh < 2; ++hh) {
                const int h = min(2 * fw + hh, a.group - 1);
                const float m_reg = lane < S ? s_m[h * kMaxSplitsKept + min(lane, S - 1)] : -INFINITY;
                const float l_reg = lane < S ? s_l[h * kMaxSplitsKept + min(lane, S - 1)] : 0.0f;
                const float mx = wave_max(m_reg);
                const float f = (m_reg == -INFINITY) ? 0.0f : fast_exp2(m_reg - mx);
                if (lane < S) w[h * kMaxSplitsKept + lane] = f;
                const float d = wave_sum(lane < S ? l_reg * f : 0.0f);
                if (hh == (lane >> 5)) den = d;
            }
            asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
            __builtin_amdgcn_wave_barrier();
#pragma unroll
            for (int i = 0; i < kRows; ++i)
                if (2 * i + parity < S) sum += rows[i] * w[fh * kMaxSplitsKept + 2 * i + parity];
            if (parity == 1 && f_active) *reinterpret_cast<f32x4*>(s_odd + fh * kHeadDim + c4 * 4) = sum;
        }
    };
    // ... and the result, once the odd ones' sum is there too.
    auto write_out = [&](const Item& it) {
        if (f_active && it.hi == S && parity == 0) {
            const f32x4 r = (sum + *reinterpret_cast<const f32x4*>(s_odd + fh * kHeadDim + c4 * 4)) * (1.0f / den);
            const int64_t off = (int64_t)it.layer * ha.st.out_stride + (int64_t)(it.kvh * a.group + fh) * kHeadDim + c4 * 4;
            *reinterpret_cast<uint2*>(a.out + off) = make_uint2(pack_bf16(r[0], r[1]), pack_bf16(r[2], r[3]));
            if (a.out_f32) {
#pragma unroll
                for (int e = 0; e < 4; ++e) a.out_f32[off + e] = r[e];  // (only 4-byte alignment is promised)
            }
        }
    };
    const int item0 = (int)blockIdx.x;
    int op_set = 0, fold_set = 0;
    if constexpr (NW == 4) {
        if (wave < NW) {
            for (int item = item0; item < items; item += stride) {
                const Item it = item_at(item);
                read_query(op_set);
                for (int round = it.lo; round < it.hi; round += P) {
                    stream_round(it, round, op_set, fold_set);
                    meet();
                    fold_set ^= 1;
                }
                meet();
                meet();
                op_set ^= 1;
            }
            return;
        }
    }
    for (int item = item0; item < items; item += stride) {
        const Item it = item_at(item);
        const bool more = item + stride < items;
        if (wave == kOperandWave && more) fetch_operands(item_at(item + stride), op_set ^ 1);
        if constexpr (NW == 8) read_query(op_set);
        for (int round = it.lo; round < it.hi; round += P) {
            if constexpr (NW == 8) stream_round(it, round, op_set, fold_set);
            if (wave == kOperandWave && more && round + P >= it.hi) prepare_operands(item_at(item + stride), op_set ^ 1);
            meet();
            if constexpr (P == 1) {
                if (folds_here && (round & 1) == parity) fold_split(it, round, round, fold_set);
            } else if (folds_here) {
                for (int split = round + ((round ^ parity) & 1); split < min(round + P, it.hi); split += 2) fold_split(it, round, split, fold_set);
            }
            fold_set ^= 1;
        }
        hand_over(it);
        meet();
        weigh(it);
        meet();
        write_out(it);
        op_set ^= 1;
    }
}

template <int G>
void launch_g(const HeadsArgs& ha, int grid, int waves, hipStream_t stream) {
    const int splits = ha.st.a.num_splits, most = ha.st.a.tiles_run + (ha.st.a.tiles_longer > 0 ? 1 : 0);  // tiles of a split, at most
    const int at_once = heads_splits_at_once(splits, most, waves);
    auto launch = [&](auto nw, auto stages, auto p) {
        hipLaunchKernelGGL((mha_heads_kernel<G, decltype(nw)::value, decltype(stages)::value, decltype(p)::value>), dim3(grid), dim3(kWaves * 64), 0, stream, ha);
    };
    const std::integral_constant<int, 1> one{};
    const std::integral_constant<int, 2> two{};
    const std::integral_constant<int, 4> four{};
    const std::integral_constant<int, 8> eight{};
    if constexpr (G <= 4) {
        // (eight wavefronts: a single pass)
        if (waves == 8) launch(eight, one, one);
        else if (at_once >= 4) launch(four, four, four);
        else if (at_once >= 2) launch(four, four, two);
        else launch(four, four, one);
    } else {
        if (at_once >= 8) launch(eight, one, eight);
        else if (at_once >= 4) launch(eight, one, four);
        else if (at_once >= 2) launch(eight, one, two);
        else launch(eight, one, one);
    }
}

}  // namespace

void launch_heads(const HeadsArgs& ha, int grid, int group_pad, int waves, hipStream_t stream) {
    switch (group_pad) {
        case 1: return launch_g<1>(ha, grid, waves, stream);
        case 2: return launch_g<2>(ha, grid, waves, stream);
        case 4: return launch_g<4>(ha, grid, waves, stream);
        default: return launch_g<8>(ha, grid, waves, stream);
    }
}

hipError_t poll_timeouts_heads(unsigned int* n) { return hipMemcpyFromSymbol(n, HIP_SYMBOL(g_poll_timeouts), sizeof(*n)); }

}  // namespace llmi
