// Decode-phase grouped-query attention for gfx950 (MI355X), batch 1: the kernel templates.
// Included by one translation unit per query-group size (mha_decode_group*.hip defines LLMI_GROUP first), which
// instantiates the kernels of that group; the host-side launcher is mha_decode.hip.
//
// One kernel template serves both paths of the reference's dispatcher
// (code/source/op/kernel/cuda/mha_kernel.cu:505-528):
//   * single pass  (num_splits == 1): the workgroup owns every position of one
//     KV head and writes the bf16 result itself;
//   * KV split     (num_splits  > 1): workgroup (split, kv_head) owns a
//     contiguous range of positions and leaves (o[128], m, l) per query head
//     in the fp32 workspace; either mha_combine_kernel merges them
//     (log-sum-exp, a second launch) or the workgroup of the last split does,
//     inside the same launch (fused combine).
// Three more template switches: APPEND folds the per-token QK-Norm + RoPE and the
// K/V cache append of the reference's layer loop into the launch (the new row
// enters the softmax from the workgroup's own LDS), DYN reads the position from device memory
// so that one captured launch serves every token, STAGGER makes the splits of the
// position-major layout walk their tiles from different starting points.
//
// Differences from the reference design, chosen for CDNA4:
//   * a workgroup serves ALL query heads of its KV head, so K and V are read
//     from HBM exactly once (the reference re-reads them once per query head,
//     mha_kernel.cu:67,104);
//   * K/V tiles stream through per-wave LDS rings filled by LDS-DMA loads, every
//     load instruction a run of whole 256-byte rows (1 KiB of contiguous memory
//     in the head-major layout); the query rows (and the append variant's operands)
//     take the same road, issued ahead of the tiles, so that every wait is a hand-placed vmcnt;
//   * q.K^T runs on the matrix cores: one v_mfma_f32_16x16x32_bf16 chain per
//     tile of 16 positions, K rows as the A operand (lane = row, no transpose
//     needed because the contraction over head_dim is order-free), the query
//     group as B;
//   * P^T.V runs on the matrix cores too (v_mfma_f32_16x16x16_bf16): the score
//     MFMA leaves a lane's four probabilities exactly where the A fragment of
//     that product wants them, the V fragment is packed from the lane's four
//     16-byte V rows with v_perm_b32; a probability enters as hi + lo bf16, so
//     the product is as accurate as an fp32 one;
//   * running max / sum are kept in the exp2 domain (scale*log2(e) folded in);
//   * 64-bit offsets throughout (the reference's int32 layer_offset,
//     mha_kernel.cu:488, overflows on large caches).
//
// Tile bookkeeping (T = 16 consecutive positions, r = row in tile, h = head in group):
//   QK  A  lane L: row r = L%16, dims (j*4 + L/16)*8 .. +8 for step j = 0..3
//   QK  B  lane L: head h = L%16 (the group's last head again for h >= group), same dims
//   QK  C  lane L: head h = L%16, rows r = 4*(L/16) + i in register i = 0..3
//   loads  lane L: K and V load i fetch rows 4i + L/16 whole (256 contiguous bytes over the row's 16 lanes;
//                  K with its 16-byte chunks swizzled by row & 7); the operands are read back from
//                  LDS in the layouts above and below
//   V oper lane L: rows r = 4*(L/16) + i (register i), columns (L%16)*8 .. +8
//   PV  A  lane L: head h = L%16, rows 4*(L/16) + i      (= QK C, as bf16)
//   PV  B  lane L: rows 4*(L/16) + i, column 8*(L%16) + j for product j = 0..7
//   PV  C  lane L: heads 4*(L/16) + i, column 8*(L%16) + j (accumulator o[j][i])

#ifndef LLMI_MHA_DECODE_KERNELS_H
#define LLMI_MHA_DECODE_KERNELS_H

#include <hip/hip_runtime.h>
#include <stdint.h>

#include <type_traits>

#include "mha_device_helpers.h"

namespace llmi {
namespace {

// Occupancy hint. Two waves per SIMD keep the register budget at 256, where the compiler picks
// VGPR-form MFMAs; with the whole file of 512 it keeps the accumulators in AGPRs and copies them to
// VGPRs and back around the rescaling of every tile. Groups of 16 heads cannot meet the hint in every
// shape; there it is 1.
template <int G, int NW>
constexpr int kWavesPerEu = (G >= 16 && NW != 2) ? 1 : LLMI_MIN_WAVES_PER_EU;

// Splits above which the wavefronts of a merging workgroup share a head's splits. (At 64 it is level: 6.50 -> 6.35 us with four
// wavefronts, 6.43 -> 6.86 with eight, 4001 positions. And the multi-layer kernels, which stand for launches of up to 64
// splits, add them up in one wavefront's order.)
#ifndef LLMI_WIDE_MERGE_MIN
#define LLMI_WIDE_MERGE_MIN 64
#endif
constexpr int kWideMergeMin = LLMI_WIDE_MERGE_MIN;

template <int G, int NW, int NSTAGE, bool APPEND, bool DYN, bool STAGGER, bool OPROJ, bool BYSIDE, bool EARLY = false>
__device__ __forceinline__ void mha_decode_body(const KernelArgs& a, OprojState& proj) {
    constexpr bool kSpreadMerge = LLMI_SPREAD_MERGE && !OPROJ;
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);  // scalar: loop control stays on the SALU
    const int n16 = lane & 15;  // MFMA column / DPP-row lane
    const int kg = lane >> 4;   // MFMA k-group / DPP row
    // Workgroups are handed to the eight XCDs (each with its own L2) in turn, in index order with x
    // fastest: with the KV head in x, the splits of a head land on one XCD whenever the number of
    // KV heads is a multiple of eight, and the combiners (last splits) spread over all of them
    // instead of sharing one. Nothing relies on that placement for correctness; it is worth
    // 0.1-0.35 us per call (32 query / 8 KV heads, 1K to 32K positions) against split-fastest.
    const int kvh = blockIdx.x;
    const int split = blockIdx.y;

    // Each wave streams its tiles through a private ring of NSTAGE LDS slots
    // (8 KiB each: 4 KiB of K rows, 4 KiB of V rows) filled by LDS-DMA loads,
    // so the bytes in flight cost no VGPRs. A load lands at offset 16*lane of its
    // 1 KiB block, i.e. as four whole rows; the operand reads pick their 16 bytes
    // out of those rows (K through a row-dependent swizzle, V directly), both free
    // of bank conflicts. Out-of-range rows of a ragged last
    // tile read the last valid row and are masked out of the softmax.
    constexpr int kStageBytes = 8192;
    constexpr int kRingBytes = NW * NSTAGE * kStageBytes;
    // Epilogue: a wave's G x 128 partial outputs go to the start of its own (drained) ring,
    // so no wave has to wait for another one's ring. Behind the rings: per-wave and merged
    // (max, sum) pairs, then the combine area (weights [G][kMaxSplits], denominators [G],
    // per-wave arrival flags [NW], one 16-byte partial sum per thread).
    constexpr int kWaveRingBytes = NSTAGE * kStageBytes;
    static_assert(G * kHeadDim * (int)sizeof(float) <= kWaveRingBytes, "a wave's partial outputs must fit its ring");
    constexpr int kMergeTail = (2 * NW * G + 2 * G) * (int)sizeof(float);
    constexpr int kCombineBase = kRingBytes + ((kMergeTail + 15) & ~15);
    constexpr int kCombineBytes = (G * kMaxSplits + G + NW) * (int)sizeof(float) + NW * 64 * 16;
    // Position on the device, groups of exactly eight on eight wavefronts: norm weights and raw query rows are asked for while the position
    // travels and the sines and cosines as soon as it is in, ahead of the splits' rule, so that all of a row's work but the rotation is done
    // when they land; and a long context branches past the rule's other lines. Everything behind the position, the rule in selects : so, 36 captured
    // layers of 64 Q / 8 KV heads, us: 195.1 : 195.9 at 200 positions, 203.8 : 206.4 at 300, 207.8 : 205.0 at 600, 211.4 : 208.0 at 1000, 229.6 :
    // 221.9 at 1700, 240.2 : 234.3 at 2500, 252.6 : 249.9 at 3500, 277.7 : 275.2 at 5000, a window of 160 positions 155.5 : 153.3. It is the three
    // together: at 1000, 2500 and 5000 positions without the branch 210.8, 242.2, 277.9, without the rows ahead 214.2, 232.3, 280.0, one wait for
    // rows and tables 213.8, 240.7, 275.4, the branch alone 212.3, 231.3, 290.8. Nobody else gains: 40 Q heads, not so : so, 204.0 : 207.7 at 300, 209.2 : 215.3
    // at 1000, 239.8 : 235.5 at 2500, 275.7 : 283.8 at 5000, 48 Q heads 211.0 : 217.0 at 1000; eight wavefronts for smaller groups, windows of 160
    // positions, 32 Q heads 153.0 : 155.5, 8 Q heads 144.8 : 146.8; four wavefronts, 32 Q heads 177.8 : 185.8 at 300, 187.5 : 195.9 at 1100.
    constexpr bool kEarlyRows = EARLY;
    static_assert(!EARLY || (G == 8 && NW == 8 && APPEND && DYN), "");
    // 1 KiB LDS-DMA slots for the small operands, rows of 256 bytes four to a slot. Plain variant: every wave fetches all
    // query rows of the group for itself. Append variant: the query rows, and in the
    // workgroup of the last split the new K and V rows behind them, are dealt to the waves two at a time, 32 lanes a row, the last wave
    // first (it has the fewest tiles); a wave fetches its own, raw, and leaves them normalised and rotated (V: as it is) behind the
    // slots, where all waves read them after a barrier. In front of the slots one that the workgroup shares, q_norm | k_norm | sin row | cos row
    // (every wave that works on rows fills it with the same bytes and waits only for its own loads); kEarlyRows: sin row | cos row, and a wave's
    // own slots begin with q_norm | k_norm. The slots
    // lie over the combine area, which nobody touches before the barrier of the epilogue, so they
    // cost no LDS: with more than 80 KiB per workgroup the compiler assumes one wave per SIMD, puts
    // the MFMA accumulators into AGPRs and copies all 32 of them to VGPRs and back around the
    // rescaling of every tile.
    constexpr int kRowPasses = (G + 2 + 2 * NW - 1) / (2 * NW);  // append variant: rows per half wavefront
    constexpr int kRowSlots = APPEND ? ((kEarlyRows ? 2 : 0) + 2 * kRowPasses + 3) / 4 : (G * 16 + 63) / 64;
    constexpr int kSharedSlots = APPEND ? 1 : 0;
    constexpr int kReadyBytes = APPEND ? (G + 2) * 256 : 0;  // the finished rows: G query rows, the new K row, the new V row
    constexpr int kStagingBase = (kCombineBase + 1023) & ~1023;
    constexpr int kStagingBytes = (kSharedSlots + NW * kRowSlots) * 1024 + kReadyBytes;
    constexpr int kSmemBytes =
        kCombineBase + kCombineBytes > kStagingBase + kStagingBytes ? kCombineBase + kCombineBytes : kStagingBase + kStagingBytes;
    __shared__ __attribute__((aligned(1024))) char smem[kSmemBytes];
    char* shared_staging = smem + kStagingBase;                                       // append variant only
    auto row_slots = [&]() { return smem + kStagingBase + (kSharedSlots + wave * kRowSlots) * 1024; };  // this wave's rows
    char* ready_rows = smem + kStagingBase + (kSharedSlots + NW * kRowSlots) * 1024;  // append variant only
    // Append variant: the rows of this workgroup -- the query heads, in the last split's the new K and V rows too -- are dealt to the waves in
    // pairs, the last wave first: the first pair of this one (the next is NW on).
    const int first_pair = NW - 1 - wave;
    const bool has_queries = APPEND && 2 * first_pair < a.group;
    // (early, wavefronts with nothing but the new K and V rows wait for the position all the same: they are the last split's business)
    // (one pass and one slot: the weights in lanes 0 to 31, where `row` lies in front of the first one and is not used, the pair behind them)
    static_assert(!kEarlyRows || (kRowPasses == 1 && kRowSlots == 1), "");
    auto issue_rows = [&]() {
        const int which = lane >> 4;
        const int row = 2 * (first_pair + NW * ((which >> 1) - 1)) + (which & 1);
        const uint64_t q_row = reinterpret_cast<uint64_t>(a.q) + (uint64_t)(uint32_t)((kvh * a.group + min(row, a.group - 1)) * 256);
        const uint64_t new_row = reinterpret_cast<uint64_t>(row == a.group ? a.k_new : a.v_new) + (uint64_t)(uint32_t)(kvh * 256);
        const uint64_t weights = reinterpret_cast<uint64_t>(a.norm_w) + (uint64_t)which * 256u;
        uint64_t src = row >= a.group ? new_row : q_row;  // (rows behind the last one repeat a row that is there and are not used)
        src = which < 2 ? weights : src;                  // (selects: with the weights' address in its arm this becomes a branch)
        dma16_gather(reinterpret_cast<const void*>(src + (uint64_t)n16 * 16u), (uint32_t)(uintptr_t)row_slots());
    };
    auto issue_sincos = [&](int seq_len) {
        const uint64_t row = reinterpret_cast<uint64_t>((lane & 16) ? a.cos_cache : a.sin_cache) + (uint64_t)(uint32_t)(seq_len - 1) * 256u;
        dma16_gather(reinterpret_cast<const void*>(row + (uint64_t)n16 * 16u), (uint32_t)(uintptr_t)shared_staging);
    };

    // A KV head's 16-position tiles are dealt to the splits in contiguous runs whose lengths
    // differ by at most one tile (the first tiles % S splits get the longer run), so every split
    // has work whenever there are at least S tiles and the last split -- the one that merges,
    // and in the append variant the one that holds the new token -- never has the longest run.
    // With a position read from device memory the grid was sized for the largest position:
    // the same rules are applied to the tiles there are -- a single pass, a quarter or half of the
    // splits or all of them, nearly as the host would have planned (dyn_split_rule) --, and the splits that are not needed leave at once.
    // 32 Q / 8 KV heads, append variant in a captured 36-layer step sized for 8192 positions, us per layer, all splits as far as
    // there are tiles : the rule: 5.58 : 4.02 at 60 positions, 5.51 : 5.33 at 170, 5.65 : 5.36 at 300, 5.73 : 5.40 at 600.
    // Append variant: the new token's row never comes from the cache (its K and V rows lie finished in LDS, where the running
    // softmax of one wave starts from them), so the tiles cover positions 0 .. pos-1.
    int seq_len = a.seq_len, n_active = a.num_splits;
    // (the host never asks for more splits than tiles; 0 tiles: 1 split). The division is done on
    // the host when the position is known there: it is 33 instructions in front of the first load.
    int run = a.tiles_run, longer = a.tiles_longer;  // splits 0 .. longer-1 take run + 1 tiles
    if constexpr (DYN) {
        // Everything on the way to the first request depends on the position, which takes a trip to memory of its own: the
        // arguments the prologue needs are therefore all asked for in one go in front of it (left to itself the compiler
        // asks for some where they are used, a trip each), and the division by the split count is a multiplication by
        // the host's reciprocal. With the rule
        // but without these two 5.84 us per layer at 1100 positions and 9.44 at 8000, with them 5.72 and 9.26 (5.58 and 9.18 with
        // the position known to the host).
        asm volatile("" ::"s"(a.q), "s"(a.k), "s"(a.v), "s"(a.row_stride), "s"(a.head_stride), "s"(a.group), "s"(a.num_splits), "s"(a.seq_len),
                     "s"(a.dyn_single), "s"(a.dyn_half), "s"(a.dyn_quarter), "s"(a.dyn_magic[0]), "s"(a.dyn_magic[1]), "s"(a.dyn_magic[2]));
        if constexpr (kEarlyRows) asm volatile("" ::"s"(a.dyn_full));
        if constexpr (APPEND) asm volatile("" ::"s"(a.norm_w), "s"(a.sin_cache), "s"(a.cos_cache), "s"(a.k_new), "s"(a.v_new), "s"(a.eps));
        // (constant address space: a scalar load, where the compiler, not knowing that nothing in the launch writes the position, takes a
        // vector one and its longer way: 36 layers 209.8 -> 205.5 us at 1100 positions, 194.5 -> 192.9 at 300, 64 layers of 64 Q heads at 5000
        // 532.0 -> 530.5. The heads' addresses ahead of its arrival: level.)
        const auto pos_dev = reinterpret_cast<const __attribute__((address_space(4))) int32_t*>(reinterpret_cast<uintptr_t>(a.pos_dev));
        const int32_t pos = *pos_dev;
        if (kEarlyRows && has_queries) issue_rows();
        seq_len = max(0, min(pos, a.seq_len - 1)) + 1;
        if (kEarlyRows && has_queries) issue_sincos(seq_len);
        const int tiles = (seq_len - (APPEND ? 1 : 0) + kTile - 1) / kTile;
        // (the rounded-up reciprocal is one too high at most, and only beyond 2^24 tiles)
        auto deal = [&](int count, uint32_t magic) {
            n_active = count;
            run = (int)(((uint64_t)(uint32_t)tiles * magic) >> 32);
            longer = tiles - run * count;
            if (longer < 0) {
                --run;
                longer += count;
            }
        };
        if (kEarlyRows && tiles > a.dyn_full) {
            deal(a.num_splits, a.dyn_magic[2]);
        } else {
            const bool few = tiles < a.dyn_half, medium = tiles <= 4 * a.dyn_half;
            deal(few ? a.dyn_quarter : medium ? a.dyn_half : a.num_splits, few ? a.dyn_magic[0] : medium ? a.dyn_magic[1] : a.dyn_magic[2]);
            if (tiles < n_active) {  // a tile each
                n_active = tiles;
                run = 1;
                longer = 0;
            }
            if (tiles <= a.dyn_single || n_active <= 1) {
                n_active = 1;
                run = tiles;
                longer = 0;
            }
        }
        if (split >= n_active) {
            if constexpr (kEarlyRows) asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // (what is on its way to this workgroup's LDS lands first)
            return;
        }
    }
    const int cached_len = seq_len - (APPEND ? 1 : 0);  // positions streamed from the cache
    const int ntiles = run + (split < longer ? 1 : 0);
    const int begin = (split * run + min(split, longer)) * kTile;
    const int nrows = min(ntiles * kTile, cached_len - begin);  // > 0 unless nothing is cached yet

    // Filled in below, once the first tiles are on their way.
    u32x4 qb[4];                       // query group, MFMA B operand
    // Append variant: wave 0 of the last split (the one with the shortest run) takes the new token.
    const bool holds_new_row = APPEND && split == n_active - 1 && wave == 0;
    // Append variant: with two waves on a SIMD those that have rows go first
    // until the rows are done: their requests would else queue behind the tiles of the others (64 Q / 8 KV heads, a layer of a captured step at
    // 1000 positions, without : with 6.49 : 6.32 us).
    const int work_rows = a.group + (split == n_active - 1 ? 2 : 0);
    const bool has_rows = APPEND && 2 * first_pair < work_rows;
    if (NW > 4 && has_rows) __builtin_amdgcn_s_setprio(3);
    if (kEarlyRows && has_rows && !has_queries) {
        issue_rows();
        issue_sincos(seq_len);
    }

    // Wave-uniform 64-bit bases of this split; lanes add 32-bit byte offsets
    // (scalar-base + vector-offset addressing, no 64-bit multiplies per load).
    const char* kb = reinterpret_cast<const char*>(a.k + (int64_t)kvh * a.head_stride + (int64_t)begin * a.row_stride);
    const char* vb = reinterpret_cast<const char*>(a.v + (int64_t)kvh * a.head_stride + (int64_t)begin * a.row_stride);
    const uint32_t rs = (uint32_t)a.row_stride * 2u;           // bytes per position step
    const uint32_t last_off = (uint32_t)(nrows - 1) * rs;      // rows past the range clamp to its last row
    // K load i of a tile fetches rows 4i .. 4i+3 whole (DPP row kg takes row 4i + kg, 256 contiguous
    // bytes across its 16 lanes): every request is a full cache line in either layout, and in the
    // head-major layout one instruction covers 1 KiB of contiguous memory. Lane p of the row fetches
    // 16-byte chunk p ^ (row & 7): the swizzle that lets the MFMA operand read below (lane = row,
    // 16 rows 256 bytes apart) spread over the LDS banks instead of hitting one.
    const uint32_t k_row = (uint32_t)kg * rs;
    const uint32_t k_col0 = (uint32_t)(n16 ^ kg) * 16u;        // rows 4i + kg with i even: (row & 7) = kg
    const uint32_t k_col1 = (uint32_t)(n16 ^ (4 + kg)) * 16u;  // i odd: (row & 7) = 4 + kg
    // Operand read: row n16 sits in load n16 / 4, at row slot n16 % 4; chunk c is at lane slot c ^ (n16 & 7).
    const uint32_t k_rd = (uint32_t)((n16 >> 2) * 1024 + (n16 & 3) * 256);
    const uint32_t k_rd0 = k_rd + (uint32_t)((kg ^ (n16 & 7)) * 16);        // chunks j*4 + kg, j even (+ 128 bytes for j = 2)
    const uint32_t k_rd1 = k_rd + (uint32_t)(((4 + kg) ^ (n16 & 7)) * 16);  // j odd (+ 128 bytes for j = 3)
    const uint32_t v_col = (uint32_t)n16 * 16u;

    float m_run = -INFINITY;  // running max, exp2 domain, per (head = n16)
    float l_run = 0.0f;       // running sum over this lane's rows
    // Output accumulators, MFMA C layout of P^T V: o[j][r] belongs to head 4*kg + r and
    // column 8*n16 + j, summed over all positions this wave has seen.
    f32x4 o[8];
#pragma unroll
    for (int j = 0; j < 8; ++j) o[j] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
#if LLMI_PV_VALU
    // Vector-ALU variant: ov[h][j] belongs to head h and column 8*n16 + j, summed over the rows
    // 4*kg .. 4*kg+3 of every tile this wave has seen; the four DPP rows are added up after the loop.
    float ov[G][8];
#pragma unroll
    for (int h = 0; h < G; ++h)
#pragma unroll
        for (int j = 0; j < 8; ++j) ov[h][j] = 0.0f;
#endif

    char* my_ring = smem + wave * (NSTAGE * kStageBytes);
    const uint32_t my_ring_lds = (uint32_t)(uintptr_t)my_ring;  // low 32 bits of a flat LDS address = LDS offset

    // (`refill`: the slot holds a tile whose contents must have reached the VGPRs first; a slot's first tile waits for nothing)
    auto issue_tile = [&](int t, int stage, auto refill) {
        if constexpr (decltype(refill)::value) asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
        const uint32_t base = (uint32_t)t * (kTile * rs);
        const uint32_t slot = my_ring_lds + (uint32_t)stage * kStageBytes;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const uint32_t ko = min(base + k_row + (uint32_t)(4 * i) * rs, last_off) + ((i & 1) ? k_col1 : k_col0);
            dma16(kb, ko, slot + i * 1024);
        }
        // V the same way: load i fetches rows 4i .. 4i+3 whole. The operand wants rows 4*kg + i in lane
        // (kg, n16): row r sits in load r / 4 at row slot r % 4, read back below without bank conflicts
        // (the 16 lanes of a DPP row read 256 consecutive bytes).
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const uint32_t vo = min(base + k_row + (uint32_t)(4 * i) * rs, last_off) + v_col;
            dma16(vb, vo, slot + 4096 + i * 1024);
        }
    };

    auto read_tile = [&](int stage, TileRegs& r) {
        const char* kp = my_ring + stage * kStageBytes;
#pragma unroll
        for (int j = 0; j < 4; ++j)
            r.k[j] = *reinterpret_cast<const u32x4*>(kp + ((j & 1) ? k_rd1 : k_rd0) + (j >> 1) * 128);
#pragma unroll
        for (int i = 0; i < 4; ++i)
            r.v[i] = *reinterpret_cast<const u32x4*>(kp + 4096 + kg * 1024 + i * 256 + n16 * 16);
    };

    auto compute_tile = [&](int t, const TileRegs& r) {
        const int row0 = t * kTile + 4 * kg;
#if !LLMI_PV_VALU
        fold_tile<G>(r, qb, row0, nrows, a.scale_log2e, m_run, l_run, o);
#else
        f32x4 c = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
        for (int j = 0; j < 4; ++j)
            c = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, r.k[j]),
                                                        __builtin_bit_cast(bf16x8, qb[j]), c, 0, 0, 0);
        float s[4];
        float tmax = -INFINITY;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            s[i] = (row0 + i < nrows) ? c[i] * a.scale_log2e : -INFINITY;
            tmax = fmaxf(tmax, s[i]);
        }
        tmax = rows_max(tmax);
        const float m_new = fmaxf(m_run, tmax);
        const float alpha = fast_exp2(m_run - m_new);
        float p[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) p[i] = fast_exp2(s[i] - m_new);
        const float psum = (p[0] + p[1]) + (p[2] + p[3]);
        l_run = l_run * alpha + psum;
        m_run = m_new;
        // Rescale only when some head's max moved (wave-uniform test); head h's factor sits in
        // lane h of every 16-lane row.
        if (__any(alpha != 1.0f)) {
            static_for<0, G>([&](auto h) {
                const float ah = row_bcast<h.value>(alpha);
#pragma unroll
                for (int j = 0; j < 8; ++j) ov[h.value][j] *= ah;
            });
        }
        float vf[4][8];
#pragma unroll
        for (int i = 0; i < 4; ++i)
#pragma unroll
            for (int j = 0; j < 8; ++j) {
                const uint32_t w = r.v[i][j >> 1];
                vf[i][j] = (j & 1) ? bf16_hi(w) : bf16_lo(w);
            }
        static_for<0, G>([&](auto h) {
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const float ph = row_bcast<h.value>(p[i]);  // probability of (head h, row 4*kg + i)
#pragma unroll
                for (int j = 0; j < 8; ++j) ov[h.value][j] = fmaf(ph, vf[i][j], ov[h.value][j]);
            }
        });
#endif
    };

    // Wave w owns tiles w, w+NW, ...: NSTAGE of them are in flight throughout the loop (append variant: one until the rows are done).
    const int n_my = wave < ntiles ? (ntiles - wave + NW - 1) / NW : 0;
    // STAGGER: the splits of a head walk their tiles from different starting points (split s starts
    // s & a.stagger tiles into its wave's sequence and wraps round), so that workgroups running in
    // step do not all sit at the same offset of their runs. Where the runs start a multiple of 512 KiB
    // apart, walking them in step keeps hitting the same few memory channels: position-major, 8192
    // positions, 1.7 us of 13.6; head-major, 131072 positions (runs of 1 MiB), up to 6 us of 86. Elsewhere it
    // gains nothing or loses, and the bookkeeping costs 0.08 us per call, so the host asks for it by
    // length and it is compiled in only where it is used.
    // (position read on the device: the host could only say that the rule may apply; what the length found asks for)
    int rot_mask = a.stagger;
    if constexpr (DYN && STAGGER)
        if (rot_mask == kStaggerByDevice) rot_mask = head_major_stagger_rule((long long)run * kTile * a.row_stride * 2);
    const int rot = STAGGER ? min(split & rot_mask, max(n_my - 1, 0)) : 0;
    auto tile_of = [&](int i) {
        if constexpr (!STAGGER) return wave + i * NW;
        int ii = i + rot;
        if (ii >= n_my) ii -= n_my;
        return wave + ii * NW;
    };
    // The query rows (and in the append variant the operands of the fused QK-Norm + RoPE) go to
    // LDS by DMA *ahead of* the first K/V tiles. Loads complete in order, so they are there
    // after one memory round trip: the normalisation runs while the tiles are still in flight,
    // and the first tile is worked on as soon as it lands. As ordinary loads their wait would be
    // placed by the compiler, which does not know about the DMA loads: it would also wait for
    // every tile issued before that point.
    if constexpr (OPROJ) {
        // The generation word moves once per launch, after every head's output is written. That needs
        // every combiner, each combiner needs the records of its splits, and those go out only after
        // every load of this wavefront has come back (the wait in front of the record stores): read
        // here, the word still holds the value of before, in every workgroup of the grid. Issued ahead of
        // the tiles, so that nothing near the end of the kernel has to wait for it.
        proj.gen_base = __hip_atomic_load(a.ready, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
    char* my_rows = row_slots();
    if constexpr (!kEarlyRows) {
        const uint32_t st = (uint32_t)(uintptr_t)shared_staging;
        const uint32_t st_rows = (uint32_t)(uintptr_t)my_rows;
        const int c16 = lane & 15, which = lane >> 4;
        if constexpr (APPEND) {
            if (has_rows) {
                const float* sin_row = a.sin_cache + (int64_t)(seq_len - 1) * 64;
                const float* cos_row = a.cos_cache + (int64_t)(seq_len - 1) * 64;
                // (integer selects: as pointer conditionals this becomes a chain of branches)
                const uint64_t w_base = reinterpret_cast<uint64_t>(a.norm_w) + (uint64_t)(which & 1) * 256u;
                const uint64_t t_base = reinterpret_cast<uint64_t>(which == 2 ? sin_row : cos_row);
                const uint64_t p0 = (which < 2 ? w_base : t_base) + (uint64_t)c16 * 16u;
                dma16_gather(reinterpret_cast<const void*>(p0), st);
            }
        }
#pragma unroll
        for (int i = 0; i < kRowSlots; ++i) {
            uint64_t src;
            if constexpr (APPEND) {
                const int pair = first_pair + 2 * NW * i;  // the slot holds this one and the one NW on
                if (2 * pair >= work_rows) continue;
                const int row = 2 * (pair + NW * (which >> 1)) + (which & 1);
                // (rows behind the last one repeat a row that is there and are not used)
                const uint64_t q_row = reinterpret_cast<uint64_t>(a.q) + (uint64_t)(uint32_t)((kvh * a.group + min(row, a.group - 1)) * 256);
                const uint64_t new_row = reinterpret_cast<uint64_t>(row == a.group ? a.k_new : a.v_new) + (uint64_t)(uint32_t)(kvh * 256);
                src = (row >= a.group && work_rows > a.group ? new_row : q_row) + (uint64_t)c16 * 16u;
            } else {
                const int head = min(which + 4 * i, a.group - 1);  // chunk lane + 64*i: head (lane + 64*i) / 16
                src = reinterpret_cast<uint64_t>(a.q + (int64_t)(kvh * a.group + head) * kHeadDim + c16 * 8);
            }
            dma16_gather(reinterpret_cast<const void*>(src), st_rows + i * 1024);
        }
    }
    // Append variant: one tile ahead of the rows' work, the others behind it. (32 Q / 8 KV heads, a layer of a captured step at 4000 positions, both
    // tiles of the ring ahead : one 7.42 : 7.21 us: a wave is held up by its requests once some 40 KiB of its compute unit's are on their way.)
    const int first_tiles = min(APPEND ? 1 : NSTAGE, n_my);
#pragma unroll
    for (int s0 = 0; s0 < (APPEND ? 1 : NSTAGE); ++s0)
        if (s0 < first_tiles) issue_tile(tile_of(s0), s0, std::false_type{});
    // What the end of the kernel needs to know about where its results go is worked out here, while the first tiles
    // are on their way and the wavefront has nothing else to do: behind the last tile every instruction is on the
    // path of whoever waits for this split (the empty asm statements keep the compiler from moving the work there).
    const bool fused = a.records != nullptr && n_active > 1;
    const int my_xs = package_side<BYSIDE>();  // wave-uniform: the side of the package this workgroup runs on
    // Who merges a query head's splits (log-sum-exp): with enough splits, and at least as many as heads in the group,
    // head h's splits are merged by the workgroup of split SA-1-h, so that the heads' read-backs (16 KiB each at 32
    // splits) run on different compute units at the same time instead of queueing at one; otherwise the workgroup of
    // the last split merges every head. For groups of 16 (four wavefronts per workgroup) the latter means four heads'
    // polls in turn and a shared read-back: 32 Q / 2 KV heads 10.9 -> 5.9 us at 500 positions, 27.3 -> 12.2 at 40001.
    const bool spread = kSpreadMerge && n_active >= a.spread_min && n_active >= a.group;
    const int merge_head = spread && n_active - 1 - split < a.group ? n_active - 1 - split : -1;
    const bool merges_any = spread ? merge_head >= 0 : split == n_active - 1;
    // (testing aid: pretend this split ran on the other side; never a merging one, whose own rows it reads itself)
    const int store_xs = my_xs ^ (int)(BYSIDE && !merges_any && (a.far_home == 1 || (a.far_home == 2 && (split & 1))));
    const int n_units = a.group * (kHeadDim / 4);
    const int64_t part_rows = BYSIDE ? 2 * (((int64_t)a.n_q * a.num_splits + 15) & ~(int64_t)15) : (int64_t)a.n_q * a.num_splits;
    int part_bytes = (int)(part_rows * kHeadDim * (int64_t)sizeof(float));
    asm volatile("" : "+s"(part_bytes));
    const __amdgpu_buffer_rsrc_t part_rsrc = __builtin_amdgcn_make_buffer_rsrc(a.ws, 0, part_bytes, 0x00020000);
    // A (head, 16-byte column) unit of the final merge: where its partial row and its record go.
    struct MergeUnit {
        int hq;
        int64_t po;               // element offset of the column in the partial array
        int64_t rec;              // index of the first word of the head's record of this split (fused combine)
    };
    auto merge_unit = [&](int u) {
        const int h = u >> 5, c4 = u & 31;
        MergeUnit m;
        m.hq = kvh * a.group + h;
        const WsHead wh = ws_head<BYSIDE>(a, m.hq);
        m.po = (fused ? (int64_t)ws_row<4>(wh, split, store_xs) : (int64_t)m.hq * a.num_splits + split) * kHeadDim + c4 * 4;
        m.rec = (int64_t)ws_row<9>(wh, split, store_xs) * 2;
        return m;
    };
    MergeUnit first_unit = merge_unit((int)threadIdx.x);
    asm volatile("" : "+v"(first_unit.hq), "+v"(first_unit.po), "+v"(first_unit.rec));
    // Query group as the MFMA B operand. Columns beyond the group repeat its last row: a column's scores, maximum and sum stay in
    // its lanes and its outputs in its own accumulators, and nobody reads those of a head that is not there. (Zeros in their place were 16 selects
    // between the query and the first score, on every launch's way to its first tile: a layer of a captured step, zeros : repeats, us, 32 Q / 8 KV
    // heads 4.27 : 4.18 at 100 positions, 5.07 : 4.96 at 300, 64 Q heads 6.36 : 6.28 at 1000, 7.37 : 7.22 at 2500.)
    {
        // Everything issued before the tiles has landed once only the tiles are in flight.
        // (the accumulators are cleared here, in front of the wait, not behind it)
#pragma unroll
        for (int j = 0; j < 8; ++j) asm volatile("" : "+v"(o[j]));
        if constexpr (!APPEND) wait_tiles_in_flight(first_tiles);
        const int hq_local = min(n16, a.group - 1);
        if constexpr (APPEND) {
            const int half = lane >> 5, p32 = lane & 31;
            // Two rows a wave, finished once for the workgroup. Every wave on its own took four rows at a time, 16 lanes each, groups of eight in two
            // passes, and the one with the new token another for its K row, which in the workgroup that merges was the launch's
            // longest way. A layer of a captured step, us, so : two rows a wave: 32 Q / 8 KV heads 4.89 : 4.27 at 100 positions, 5.33 : 5.13 at 300, 5.68 :
            // 5.47 at 1100, 7.38 : 7.21 at 4000; 64 Q heads 5.97 : 5.74 at 200, 6.52 : 6.32 at 1000, 8.25 : 8.06 at 5000.
            // (finished query rows: the 16-byte chunks swizzled by row & 7, so that the operand read below, one chunk of every row
            // at once, spreads over the LDS banks)
            if constexpr (!kEarlyRows) wait_tiles_in_flight(first_tiles);
            else if (has_rows) wait_loads_in_flight<1>(first_tiles);  // (all but the sin and cos rows and the tile)
#pragma unroll
            for (int j = 0; j < kRowPasses; ++j) {
                const int pair = first_pair + NW * j;
                if (2 * pair >= work_rows) continue;
                const int row = 2 * pair + half;
                const bool is_new = row >= a.group, is_v = row > a.group;
                uint32_t xl, xh, lo, hi;
                // (early: weights and rows are a wavefront's own, the tables the workgroup's)
                const char* raw = my_rows + (kEarlyRows ? 512 : 0) + (2 * j + half) * 256;
                const char* weights = (kEarlyRows ? my_rows : shared_staging) + (is_new ? 256 : 0);
                const char* tables = shared_staging + (kEarlyRows ? 0 : 512);
                norm_rope_row32<kEarlyRows>(raw, weights, tables, tables + 256, p32, a.eps, [&]() { wait_tiles_in_flight(first_tiles); }, xl, xh, lo, hi);
                lo = is_v ? xl : lo;
                hi = is_v ? xh : hi;
                if (row < work_rows) {
                    const int at = is_new ? (is_v ? G + 1 : G) * 256 + p32 * 4 : row * 256 + ((p32 >> 2) ^ (row & 7)) * 16 + (p32 & 3) * 4;
                    *reinterpret_cast<uint32_t*>(ready_rows + at) = lo;
                    *reinterpret_cast<uint32_t*>(ready_rows + at + 128) = hi;
                    if (is_new) {  // the new token's rows, filed in the cache
                        uint32_t* dst = reinterpret_cast<uint32_t*>(const_cast<uint16_t*>(is_v ? a.v : a.k) + (int64_t)(seq_len - 1) * a.row_stride +
                                                                    kvh * a.slot_head_stride);
                        dst[p32] = lo;
                        dst[p32 + 32] = hi;
                    }
                }
            }
            if (NW > 4 && has_rows) __builtin_amdgcn_s_setprio(0);
            if constexpr (kEarlyRows) wait_tiles_in_flight(first_tiles);  // (whatever was asked for and is not used has landed too: its place is the combine area's)
            asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
#pragma unroll
            for (int s0 = 1; s0 < NSTAGE; ++s0)
                if (s0 < n_my) issue_tile(tile_of(s0), s0, std::false_type{});
            const u32x4* rows4 = reinterpret_cast<const u32x4*>(ready_rows);
#pragma unroll
            for (int j = 0; j < 4; ++j) qb[j] = rows4[hq_local * 16 + ((j * 4 + kg) ^ (hq_local & 7))];
            // Fused append: this wave starts its running softmax from the new token's position -- score q.k, weight 1, output = the V
            // row -- while its first tiles are still on their way.
            if (holds_new_row) {
                u32x4 kf[4], vf;
                start_from_new_row(rows4 + G * 16, rows4 + G * 16 + 16, qb, kg, n16, a.scale_log2e, kf, vf, m_run, l_run, o);
#if LLMI_PV_VALU
#pragma unroll
                for (int h = 0; h < G; ++h)
#pragma unroll
                    for (int j = 0; j < 8; ++j) ov[h][j] = kg == 0 ? o[j][0] : 0.0f;
#endif
            }
        } else {
            const u32x4* rows4 = reinterpret_cast<const u32x4*>(my_rows);
#pragma unroll
            for (int j = 0; j < 4; ++j) qb[j] = rows4[hq_local * 16 + j * 4 + kg];
        }
    }

    int stage = 0;
#if LLMI_TIMING_BARRIER_PER_TILE
    // (measurement only: what a scheme in which the wavefronts of a workgroup share every tile would pay for having to
    // agree, tile by tile, that a slot may be refilled -- a workgroup barrier per tile, every wavefront the same number)
    for (int i = 0; i < (ntiles + NW - 1) / NW; ++i) {
        __syncthreads();
        if (i >= n_my) continue;
#else
    for (int i = 0; i < n_my; ++i) {
#endif
        TileRegs r;
        wait_tiles_in_flight(min(NSTAGE - 1, n_my - 1 - i));
        read_tile(stage, r);
        if (i + NSTAGE < n_my) issue_tile(tile_of(i + NSTAGE), stage, std::true_type{});
        compute_tile(tile_of(i), r);
        stage = (stage + 1 == NSTAGE) ? 0 : stage + 1;
    }

    // ---- epilogue: fold the workgroup's waves ----
    // The outputs are already summed over a wave's positions; the denominators are
    // per DPP row (kg) and share the running max of their head, so they add up plainly.
    l_run = rows_sum(l_run);
#if LLMI_PV_VALU
    // Into the layout the epilogue expects: o[j][r] of DPP row kg is head 4*kg + r.
    static_for<0, G>([&](auto h) {
#pragma unroll
        for (int j = 0; j < 8; ++j) {
            const float t = rows_sum(ov[h.value][j]);
            if (kg == h.value / 4) o[j][h.value % 4] = t;
        }
    });
#endif

    // This wave's ring is drained (every tile it issued was waited for and read).
    auto s_o = [&](int w, int h) { return reinterpret_cast<float*>(smem + w * kWaveRingBytes) + h * kHeadDim; };
    // [G][NW] maxima, then sums: a head's side by side, read 16 bytes at a time (one by one, wave by wave : so, us: 32 Q / 8 KV heads 4.94 : 4.87 at 1100
    // positions, 64 Q heads 5.24 : 5.15; a layer of a captured step 64 Q heads 5.68 : 5.59 at 300, 5.82 : 5.76 at 1000, 7.92 : 7.81 at 5000).
    float* s_m = reinterpret_cast<float*>(smem + kRingBytes);
    float* s_l = s_m + G * NW;
    float* s_fin = s_l + G * NW;  // [G][2]: merged (max, sum) per head
#pragma unroll
    for (int r = 0; r < 4; ++r) {
        const int h = 4 * kg + r;
        if (h < G) {
            float* dst = s_o(wave, h) + n16 * 8;
            *reinterpret_cast<f32x4*>(dst) = f32x4{o[0][r], o[1][r], o[2][r], o[3][r]};
            *reinterpret_cast<f32x4*>(dst + 4) = f32x4{o[4][r], o[5][r], o[6][r], o[7][r]};
        }
    }
    if (kg == 0 && n16 < G) {
        s_m[n16 * NW + wave] = m_run;
        s_l[n16 * NW + wave] = l_run;
    }
    __syncthreads();

    if constexpr (OPROJ) proj.worker = split != n_active - 1;
    // One thread per (head, 16-byte column): weights e^(m_w - M) of the waves, weighted sum.
    constexpr int kUnits = (G * (kHeadDim / 4) + NW * 64 - 1) / (NW * 64);  // columns per thread
    float unit_m[kUnits], unit_l[kUnits];
#pragma unroll
    for (int i = 0; i < kUnits; ++i) {
        const int u = (int)threadIdx.x + i * NW * 64;
        if (u >= n_units) break;
        const int h = u >> 5;
        const int c4 = u & 31;
        MergeUnit unit = first_unit;  // (worked out while the first tiles were on their way)
        if (i > 0) unit = merge_unit(u);
        // (all of a unit's LDS reads are requested before the first is used: one round trip, not two)
        float mw[NW], lw[NW];
        f32x4 ow[NW];
#pragma unroll
        for (int w = 0; w < NW; ++w) {
            mw[w] = s_m[h * NW + w];
            lw[w] = s_l[h * NW + w];
            ow[w] = *reinterpret_cast<const f32x4*>(s_o(w, h) + c4 * 4);
        }
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
        float mx = -INFINITY;
#pragma unroll
        for (int w = 0; w < NW; ++w) mx = fmaxf(mx, mw[w]);
        const float ref = mx == -INFINITY ? 0.0f : mx;  // (one select for a wave without a tile, not one per wave)
        f32x4 acc = {0.0f, 0.0f, 0.0f, 0.0f};
        float lsum = 0.0f;
#pragma unroll
        for (int w = 0; w < NW; ++w) {
            const float f = fast_exp2(mw[w] - ref);
            acc += ow[w] * f;
            lsum += lw[w] * f;
        }
        unit_m[i] = mx;
        unit_l[i] = lsum;
        const int hq = unit.hq;
        if (n_active == 1) {
            const f32x4 r = acc * (1.0f / lsum);  // (one division, like the fused combine's)
            *reinterpret_cast<uint2*>(a.out + (int64_t)hq * kHeadDim + c4 * 4) = make_uint2(pack_bf16(r[0], r[1]), pack_bf16(r[2], r[3]));
            if (a.out_f32) {
                float* of = a.out_f32 + (int64_t)hq * kHeadDim + c4 * 4;  // only 4-byte alignment is promised
#pragma unroll
                for (int e = 0; e < 4; ++e) of[e] = r[e];
            }
        } else {
            const int64_t S = a.num_splits;
            const int64_t po = unit.po;  // element offset in the workspace
            if (fused) {
                // Device-coherent store (cache policy sc1): it goes past this XCD's L2, so the
                // workgroup (possibly on another XCD) that does the combine can read it without
                // anyone flushing or invalidating a cache.
                __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u32x4, acc), part_rsrc,
                                                       (uint32_t)(po * (int64_t)sizeof(float)), 0, 16);
            } else {
                *reinterpret_cast<f32x4*>(a.ws + po) = acc;
                if (c4 == 0) {
                    a.ws[(int64_t)a.n_q * S * kHeadDim + (int64_t)hq * S + split] = mx;
                    a.ws[(int64_t)a.n_q * S * (kHeadDim + 1) + (int64_t)hq * S + split] = lsum;
                }
            }
        }
    }
    if (!fused) return;
    // The heads' records, once every column of this wavefront is acknowledged (one wait, however many heads it has).
#pragma unroll
    for (int i = 0; i < kUnits; ++i) {
        const int u = (int)threadIdx.x + i * NW * 64;
        if (u >= n_units) break;
        const int h = u >> 5;
        const int c4 = u & 31;
        if (spread ? h != merge_head : split != n_active - 1) {
            // Publish the head's record as soon as this wavefront's stores are acknowledged:
            // the 32 columns of a head are stored by one half of one wavefront, so no
            // workgroup barrier is needed.
            asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
            if (c4 == 0) {
                unsigned long long* rec = a.records + (i > 0 ? merge_unit(u).rec : first_unit.rec);
                const unsigned long long tag = a.tag;
                const unsigned long long m_bits = __builtin_bit_cast(uint32_t, unit_m[i]);
                const unsigned long long l_bits = __builtin_bit_cast(uint32_t, unit_l[i]);
                __hip_atomic_store(rec, tag | (m_bits << 32), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                __hip_atomic_store(rec + 1, tag | (l_bits << 32), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            }
        } else if (c4 == 0) {  // the workgroup that merges this head keeps its own pair in LDS
            s_fin[2 * h] = unit_m[i];
            s_fin[2 * h + 1] = unit_l[i];
        }
    }

    // ---- fused combine ----
    // The workgroup of the LAST split of this KV head merges the partials of its
    // query heads, or (spread) those of the last splits a head each, so no second launch is needed. Every split publishes, per
    // query head, a record {epoch | max} {epoch | sum} as soon as the head's partial outputs have
    // been acknowledged; who merges a head waits for all its records but its own (it
    // has its own pair in LDS and its own partials acknowledged). Workgroups are
    // dispatched in index order and those that merge nothing never wait for anything, so the workgroup of the last split
    // waits only for some that are running or done. The workgroups of a spread merge wait for each other too: the host asks for
    // it only where all of them fit the chip with room to spare (spread_merge_fits).
    // A record carries the epoch of the call that wrote it; anything else (an
    // uninitialised workspace, an earlier call) reads as "not arrived", so the
    // workspace needs no clearing. The combiner zeroes the records again so that a
    // graph replay of this very call (same epoch) starts clean.
    const int S = a.num_splits;  // layout stride of partials and records
    const int SA = n_active;     // splits that hold positions
    if (!merges_any) return;  // (its records went out above)
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // the combiner's own partial stores are acknowledged
    __syncthreads();                                  // ... and its (max, sum) pairs are in LDS

    float* s_w = reinterpret_cast<float*>(smem + kCombineBase);  // [G][kMaxSplits] weights
    float* s_den = s_w + G * kMaxSplits;                         // [G] denominators
    int* s_ok = reinterpret_cast<int*>(s_den + G);               // [NW] every record seen
    f32x4* s_part = reinterpret_cast<f32x4*>(s_ok + NW);         // [NW * 64] per-thread partial sums
    // Waits for the records of head h (one wavefront does); the (max, sum) pairs stay in the polling
    // lanes' registers. This workgroup's own pair comes straight from LDS: its record would be the
    // last one to become visible. Returns false if a record never came. A record only counts when
    // it carries this call's tag (never zero, which is what a cleared record holds).
    // (splits first .. first + count - 1: all of them, or a wavefront's share of a wide merge)
    auto wait_records = [&](int h, int first, int count, auto slots, float* m_reg, float* l_reg, bool* home) -> bool {
        constexpr int kSlots = decltype(slots)::value;  // splits per lane
#pragma unroll
        for (int j = 0; j < kSlots; ++j) {
            m_reg[j] = -INFINITY;
            l_reg[j] = 0.0f;
            home[j] = my_xs != 0;  // the side whose home a split's record was found in: its partial outputs are in that side's home too
        }
        bool ok = false;
        // Bounded wait: every wave leaves this loop even if a record never shows up
        // (the result is then poisoned below instead of hanging the GPU).
        const WsHead wh = ws_head<BYSIDE>(a, kvh * a.group + h);
        const unsigned long long* rec_near[kSlots];
#pragma unroll
        for (int j = 0; j < kSlots; ++j) rec_near[j] = a.records + (int64_t)ws_row<9>(wh, min(first + lane + 64 * j, SA - 1), my_xs) * 2;
        // One round of polls. BOTH: also look where a split that ran on the other side of the package would have put its
        // record (never needed when the workgroups of a KV head share an XCD, so the first rounds do without).
        auto poll_round = [&](auto both_tag) {
            constexpr bool kBoth = decltype(both_tag)::value;
            ok = true;
#pragma unroll
            for (int j = 0; j < kSlots; ++j) {
                const int sp = first + lane + 64 * j;
                m_reg[j] = -INFINITY;
                l_reg[j] = 0.0f;
                if (lane + 64 * j >= count) continue;
                if (sp != split) {
                    const unsigned long long* rec = rec_near[j];
                    unsigned long long r0 = __hip_atomic_load(rec, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                    unsigned long long r1 = __hip_atomic_load(rec + 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                    bool here = (uint32_t)r0 == a.tag && (uint32_t)r1 == a.tag;
                    if constexpr (kBoth) {
                        home[j] = my_xs != 0;
                        if (!here) {
                            rec = a.records + (int64_t)ws_row<9>(wh, sp, my_xs ^ 1) * 2;
                            r0 = __hip_atomic_load(rec, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                            r1 = __hip_atomic_load(rec + 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                            here = (uint32_t)r0 == a.tag && (uint32_t)r1 == a.tag;
                            home[j] = my_xs == 0;
                        }
                    }
                    ok = ok && here;
                    m_reg[j] = __builtin_bit_cast(float, (uint32_t)(r0 >> 32));
                    l_reg[j] = __builtin_bit_cast(float, (uint32_t)(r1 >> 32));
                } else {
                    m_reg[j] = s_fin[2 * h];
                    l_reg[j] = s_fin[2 * h + 1];
                }
            }
            return __all(ok);
        };
        // The first rounds poll the near home only (some ten microseconds: far beyond the spread of the splits).
        constexpr int kNearRounds = 16;
        const int near_rounds = BYSIDE ? min(a.max_polls, kNearRounds) : a.max_polls;
        bool all_in = false;
        // (back to back: a round is one round trip of the memory system; a pause between rounds only adds to the
        // wait -- 0.03-0.06 us per call with s_sleep 2, measured at every length)
        for (int spin = 0; spin < near_rounds && !all_in; ++spin) all_in = poll_round(std::false_type{});
        if constexpr (BYSIDE) {
            if (__builtin_expect(!all_in, 0)) {
                for (int spin = near_rounds; spin < a.max_polls && !all_in; ++spin) {
                    all_in = poll_round(std::true_type{});
                    if (!all_in) __builtin_amdgcn_s_sleep(2);
                }
            }
        }
        const bool arrived = __all(ok);
        // A give-up is counted where the host can read it (llmi_hip_poll_timeouts).
        if (__builtin_expect(!arrived, 0) && lane == 0) atomicAdd(&g_poll_timeouts, 1u);
        return arrived;
    };
    // From the polled (max, sum) pairs: M = max m_s, the weights e^(m_s - M) into the head's row
    // of s_w, the denominator sum l_s * weight; the records are zeroed for the next use.
    // (`alone`: nobody else writes weights of the head, so all 64 * kSlots places are written, zeros behind the last split: the sum of the
    // partial rows then reads them without a test for each)
    auto make_weights = [&](int h, int first, int count, auto slots, auto alone, const float* m_reg, const float* l_reg, const bool* home,
                            float& mx) -> float {
        constexpr int kSlots = decltype(slots)::value;
        const WsHead wh = ws_head<BYSIDE>(a, kvh * a.group + h);
        mx = -INFINITY;
#pragma unroll
        for (int j = 0; j < kSlots; ++j) mx = fmaxf(mx, m_reg[j]);
        mx = wave_max(mx);
        float den = 0.0f;
#pragma unroll
        for (int j = 0; j < kSlots; ++j) {
            const int sp = first + lane + 64 * j;
            if (decltype(alone)::value || lane + 64 * j < count) {  // (places without a split: weight and sum are zero)
                const float f = (m_reg[j] == -INFINITY) ? 0.0f : fast_exp2(m_reg[j] - mx);
                s_w[h * kMaxSplits + sp] = f;
                den += l_reg[j] * f;
                if (sp != split && lane + 64 * j < count) {
                    unsigned long long* rec = a.records + (int64_t)ws_row<9>(wh, sp, home[j] ? 1 : 0) * 2;
                    __hip_atomic_store(rec, 0ull, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                    __hip_atomic_store(rec + 1, 0ull, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                }
            }
        }
        return wave_sum(den);
    };
    auto poll_head_n = [&](int h, float& den_out, auto slots) -> bool {
        constexpr int kSlots = decltype(slots)::value;
        float m_reg[kSlots], l_reg[kSlots];
        bool home[kSlots];  // (plain layout on this path: one home)
        const bool arrived = wait_records(h, 0, SA, slots, m_reg, l_reg, home);
        float mx;
        den_out = make_weights(h, 0, SA, slots, std::true_type{}, m_reg, l_reg, home, mx);
        return arrived;
    };
    auto poll_head = [&](int h, float& den_out) -> bool {
        if (SA <= 64) return poll_head_n(h, den_out, std::integral_constant<int, 1>{});
        return poll_head_n(h, den_out, std::integral_constant<int, kMaxSplits / 64>{});
    };
    const __amdgpu_buffer_rsrc_t ws_rsrc = part_rsrc;
    constexpr int kCoherent = kCacheDevice;

    if (G <= NW || a.group <= NW || spread) {  // (G, the group rounded up, decides it at compile time where it can)
        // One wavefront per head, all the way: poll, then read the head's partials back and write
        // its 128 outputs, without a workgroup barrier (a wave whose records are in need not wait
        // for the others). Lane = (16-byte column, half of the splits); the two halves are added
        // with one lane swap. The partials of the other workgroups were acknowledged before
        // their records were written; they are read with device-coherent 16-byte loads, a
        // lane's loads all in flight at once.
        // With many splits (shapes of few KV heads: 64 to 256) the merging workgroup's wavefronts share them: each polls,
        // weighs and reads back its own contiguous part, and wavefront 0 adds the parts up. One wavefront would read
        // 32 rows per round trip, one round after the other: 16 Q / 2 KV heads (128 splits) 12.97 -> 11.68 us at 40001
        // positions, 8 Q / 1 KV head (256 splits) 11.2 -> 7.7 at 12001, 18.8 -> 15.2 at 120001.
        const bool wide = NW >= 4 && spread && SA > kWideMergeMin;
        if (spread ? wave != 0 && !wide : wave >= a.group) return;
        const int h = spread ? merge_head : wave;
        const int c4 = lane & 31;
        const int part = lane >> 5;
        const int hq = kvh * a.group + h;
        const WsHead wh = ws_head<BYSIDE>(a, hq);
        // Byte offset of split sp's partial row, in both layouts with the same few instructions: plain, it is
        // B = row * 512; by side, the row's pair of 8 KiB blocks starts at twice B's block start and the home adds 8 KiB
        // or not: B + (B & block_mask) + home, with block_mask = 0 and home = 0 in the plain layout.
        const uint32_t row0_bytes = (uint32_t)wh.rbase * (kHeadDim * 4u);
        const uint32_t block_mask = BYSIDE ? ~(uint32_t)(kSideBlockBytes - 1) : 0u;
        const uint32_t lane_bytes = (uint32_t)c4 * 16u;
        // The first batch of partials is requested as soon as the records are in and travels
        // while the weights are worked out (they need the maximum over all records first).
        auto run = [&](auto slots, auto batch, auto wide_tag) {
            constexpr int kSlots = decltype(slots)::value;
            constexpr int kBatch = decltype(batch)::value;
            constexpr bool kWide = decltype(wide_tag)::value;
            const int share = (SA + NW - 1) / NW;  // (at most 64: 256 splits, four wavefronts)
            const int first = kWide ? wave * share : 0;
            const int count = kWide ? max(0, min(share, SA - first)) : SA;
            const float* w = s_w + h * kMaxSplits + first;
            auto load_partial = [&](int sp, uint32_t home_bytes) {  // (sp counted from `first`)
                const int spc = first + min(sp, count - 1);  // in range, a row whose record is in; the weight drops the repeat
                const uint32_t B = row0_bytes + (uint32_t)spc * (kHeadDim * 4u);
                return __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(ws_rsrc, B + (B & block_mask) + home_bytes + lane_bytes, 0, kCoherent));
            };
            float m_reg[kSlots], l_reg[kSlots];
            bool home[kSlots];
            const bool arrived = wait_records(h, first, count, slots, m_reg, l_reg, home);
            // Which home each split's partial outputs are in: this side's, for all of them, when the workgroups of the KV
            // head share an XCD -- one constant. Otherwise (wave-uniform test) per split, from the polling lanes' flags.
            bool other = false;
#pragma unroll
            for (int j = 0; j < kSlots; ++j) other = other || home[j] != (my_xs != 0);
            const bool mixed = BYSIDE && __any(other);
            const uint32_t near_bytes = BYSIDE ? (uint32_t)(wh.ppar ^ my_xs) * kSideBlockBytes : 0u;
            float den = 0.0f, mx = -INFINITY, inv = 0.0f;
            // The read-back, once for the usual case (every split in this side's home: one constant, nothing between the
            // loads) and once for the other one: two copies of the code rather than a test in front of every load.
            // Where the heads' rows start at whole blocks of 16 (the launch's split count is a multiple of it, as the dispatcher's usual ones are) and
            // the batch is full, a lane's rows lie at constant distances, which the loads carry as they are: five instructions less
            // each. With the weights read without a test each and the division made while the rows travel (some 200 instructions in
            // all, between the records' arrival and the output on the launch's last way), us, before : now: 32 Q / 8 KV heads 4.62 : 4.55 at 500 positions,
            // 5.09 : 4.95 at 1100, 8.11 : 7.95 at 6007 (position-major), 64 Q heads 5.38 : 5.25 at 1100; a layer of a captured step 5.26 : 5.09
            // at 1100, 7.19 : 7.03 at 4000, 64 Q heads 5.97 : 5.83 at 1000, 8.07 : 7.87 at 5000. (The rows' and the records' addresses ahead of
            // the waits: level.)
            const bool regular = !kWide && kSlots == 1 && (S & 15) == 0 && count >= 2 * kBatch;
            const uint32_t regular_base = (BYSIDE ? 2 * row0_bytes + near_bytes : row0_bytes) + (uint32_t)part * (kHeadDim * 4u) + lane_bytes;
            auto load_regular = [&](auto j_tag) {
                constexpr int j = decltype(j_tag)::value;
                constexpr uint32_t at = BYSIDE ? (j >> 3) * 2 * kSideBlockBytes + (j & 7) * 1024u : j * 1024u;
                return __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(ws_rsrc, regular_base + (at & 4095u), at & ~4095u, kCoherent));
            };
            auto gather = [&](auto mixed_tag, auto regular_tag) -> f32x4 {
                auto home_bytes = [&](int sp) -> uint32_t {
                    if constexpr (!decltype(mixed_tag)::value) return near_bytes;
                    // (the flag of split spc sits in lane spc % 64, slot spc / 64 of the polling layout: the slot's flags
                    // as a 64-bit lane mask, bit spc % 64 of it -- no shuffle, and no indexed array, which the compiler
                    // would put into scratch memory)
                    const int spc = min(sp, max(count - 1, 0));
                    int xs = 0;
#pragma unroll
                    for (int j = 0; j < kSlots; ++j) {
                        const unsigned long long flags = __ballot(home[j]);
                        const int f = (int)((flags >> (spc & 63)) & 1ull);
                        xs = (spc >> 6) == j ? f : xs;
                    }
                    return (uint32_t)(wh.ppar ^ xs) * kSideBlockBytes;
                };
                f32x4 v[kBatch];
                if constexpr (decltype(regular_tag)::value) {
                    static_for<0, kBatch>([&](auto j) { v[j.value] = load_regular(j); });
                } else {
#pragma unroll
                    for (int j = 0; j < kBatch; ++j) v[j] = load_partial(part + 2 * j, home_bytes(part + 2 * j));
                }
                den = make_weights(h, first, count, slots, std::bool_constant<!kWide>{}, m_reg, l_reg, home, mx);
                if constexpr (!kWide) {  // (the division while the rows travel)
                    inv = 1.0f / den;
                    asm volatile("" : "+v"(inv));
                }
                asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");  // the wave's own weights are in LDS
                __builtin_amdgcn_wave_barrier();
                f32x4 sum = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
                for (int j = 0; j < kBatch; ++j) {
                    const int sp = part + 2 * j;
                    sum += v[j] * (!kWide || sp < count ? w[sp] : 0.0f);
                }
                for (int s0 = part + 2 * kBatch; s0 < count; s0 += kBatch * 2) {
#pragma unroll
                    for (int j = 0; j < kBatch; ++j) v[j] = load_partial(s0 + 2 * j, home_bytes(s0 + 2 * j));
#pragma unroll
                    for (int j = 0; j < kBatch; ++j) {
                        const int sp = s0 + 2 * j;
                        sum += v[j] * (!kWide || sp < count ? w[sp] : 0.0f);
                    }
                }
                return sum;
            };
            f32x4 acc = {0.0f, 0.0f, 0.0f, 0.0f};
            if (kWide && count == 0) {
                // (fewer splits than the shares have room for: nothing to read)
            } else if (BYSIDE && __builtin_expect(mixed, 0)) {
                acc = gather(std::bool_constant<BYSIDE>{}, std::false_type{});
            } else if (!kWide && kSlots == 1 && regular) {
                acc = gather(std::false_type{}, std::bool_constant<!kWide && kSlots == 1>{});
            } else {
                acc = gather(std::false_type{}, std::false_type{});
            }
#pragma unroll
            for (int e = 0; e < 4; ++e) acc[e] = halves_sum(acc[e]);
            bool all_in = arrived;
            if constexpr (kWide) {
                // (the epilogue's per-wavefront pairs have been read: their place takes the parts' maxima and sums)
                if (part == 0) s_part[wave * 32 + c4] = acc;
                if (lane == 0) {
                    s_m[wave] = mx;
                    s_l[wave] = den;
                    s_ok[wave] = arrived ? 1 : 0;
                }
                __syncthreads();
                if (wave != 0) return;
                float top = -INFINITY;
#pragma unroll
                for (int x = 0; x < NW; ++x) top = fmaxf(top, s_m[x]);
                acc = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
                den = 0.0f;
#pragma unroll
                for (int x = 0; x < NW; ++x) {
                    const float mw = s_m[x];
                    const float f = (mw == -INFINITY) ? 0.0f : fast_exp2(mw - top);
                    acc += s_part[x * 32 + c4] * f;
                    den += s_l[x] * f;
                    all_in = all_in && s_ok[x] != 0;
                }
            }
            if (part == 0) {
                // A wait that ran out of patience poisons the output rather than returning a partial sum.
                if constexpr (kWide) inv = 1.0f / den;
                inv = all_in ? inv : __builtin_nanf("");
                const f32x4 r = acc * inv;
                const unsigned long long packed = (unsigned long long)pack_bf16(r[0], r[1]) | ((unsigned long long)pack_bf16(r[2], r[3]) << 32);
                unsigned long long* op = reinterpret_cast<unsigned long long*>(a.out + (int64_t)hq * kHeadDim + c4 * 4);
                if constexpr (OPROJ) __hip_atomic_store(op, packed, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);  // read by other workgroups in this launch
                else *op = packed;
                if (a.out_f32) {
                    float* of = a.out_f32 + (int64_t)hq * kHeadDim + c4 * 4;  // only 4-byte alignment is promised
#pragma unroll
                    for (int e = 0; e < 4; ++e) of[e] = r[e];
                }
            }
            if constexpr (OPROJ) {
                // The head's output is acknowledged: say so, with the generation this launch will end on.
                // (Every workgroup of the grid read the same generation word: it moves only after all
                // heads are done.) The workers wait for all heads' tags; one wavefront of the grid (head 0
                // of the last KV head, whose workgroup is dispatched last) does too and then moves the
                // word for the next launch -- also when its wait gives up, so that tags left behind by
                // this launch can never match the next one.
                asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
                uint32_t* done = a.ready + 4;
                const uint32_t target = proj.gen_base + 1u;
                if (lane == 0) __hip_atomic_store(done + hq, target, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                if (kvh == (int)gridDim.x - 1 && h == 0) {
                    bool all_done = false;
                    for (int spin = 0; spin < a.max_polls; ++spin) {
                        const uint32_t d0 = __hip_atomic_load(done + min(lane, a.n_q - 1), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                        const uint32_t d1 = __hip_atomic_load(done + min(lane + 64, a.n_q - 1), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                        all_done = __all(d0 == target && d1 == target);
                        if (all_done) break;
                        __builtin_amdgcn_s_sleep(8);
                    }
                    if (lane == 0) {
                        __hip_atomic_store(a.ready, target, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                        if (!all_done) atomicAdd(&g_poll_timeouts, 1u);
                    }
                }
            }
        };
        const std::integral_constant<int, 1> one{};
        const std::integral_constant<int, 8> eight{};
        const std::integral_constant<int, 16> sixteen{};
        // The wide merge is a copy of its own: with the shares' arithmetic in the path of the usual merges those took 0.04 - 0.08 us longer
        // (shared : apart, append 64 Q / 8 KV heads 5.93 : 5.87 us at 400 positions, 6.06 : 5.99 at 700, plain 40 Q heads 4.99 : 4.92 at 400,
        // 32 Q heads 4.87 : 4.83 at 700; the wide ones level).
        if constexpr (NW >= 4 && kSpreadMerge) {
            if (__builtin_expect(wide, 0)) {
                if (SA <= 16 * NW) run(one, eight, std::true_type{});
                else run(one, sixteen, std::true_type{});
                return;
            }
        }
        // (a lane polls one split unless a single wavefront has more than 64: a rare case, kept out of the way of the usual ones)
        if (__builtin_expect(SA > 64, 0)) run(std::integral_constant<int, kMaxSplits / 64>{}, sixteen, std::false_type{});
        else if (SA <= 16) run(one, eight, std::false_type{});
        else run(one, sixteen, std::false_type{});
        return;
    }

    // More heads than wavefronts: the waves take the heads in turn, then the whole workgroup
    // shares the read-back.
    bool wave_ok = true;
    for (int h = wave; h < a.group; h += NW) {
        float den;
        wave_ok = poll_head(h, den) && wave_ok;
        if (lane == 0) s_den[h] = den;
    }
    if (lane == 0) s_ok[wave] = wave_ok ? 1 : 0;
    __syncthreads();
    bool all_arrived = true;
#pragma unroll
    for (int w = 0; w < NW; ++w) all_arrived = all_arrived && s_ok[w] != 0;

    // Weighted sum of the partial outputs. Every other workgroup's partials were
    // acknowledged before its records were written; they are read with device-coherent
    // (L2-bypassing) 16-byte loads, a thread's loads all in flight at once, so that
    // the time does not depend on how the split count divides. A thread owns four
    // output columns of one head for every P-th split; the P partitions are added up
    // through LDS.
    constexpr int NT = NW * 64;
    const int units = a.group * (kHeadDim / 4);
    const int parts = units <= NT ? NT / units : 1;
    for (int u0 = 0; u0 < units; u0 += NT) {
        const int t = u0 + (int)threadIdx.x;
        const int u = t % units;
        const int part = units <= NT ? (int)threadIdx.x / units : 0;
        const bool active = (units <= NT) ? part < parts : t < units;
        const int h = u >> 5;
        const int c4 = u & 31;
        const int hq = kvh * a.group + h;
        const uint32_t base = (uint32_t)(((int64_t)hq * S * kHeadDim + c4 * 4) * (int64_t)sizeof(float));
        const float* w = s_w + h * kMaxSplits;
        f32x4 acc = {0.0f, 0.0f, 0.0f, 0.0f};
        // All of a batch's loads are issued before the first one is used; a short list
        // of splits takes the small batch so that it does not pay for repeats.
        auto gather = [&](auto batch) {
            constexpr int kBatch = decltype(batch)::value;
            for (int s0 = part; s0 < SA; s0 += kBatch * parts) {
                f32x4 v[kBatch];
                float wv[kBatch];
#pragma unroll
                for (int j = 0; j < kBatch; ++j) {
                    const int sp = s0 + j * parts;
                    const int spc = min(sp, SA - 1);  // in range; the weight below drops the repeat
                    v[j] = __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(
                                                         ws_rsrc, base + (uint32_t)spc * (kHeadDim * 4u), 0, kCoherent));
                    wv[j] = sp < SA ? w[sp] : 0.0f;
                }
#pragma unroll
                for (int j = 0; j < kBatch; ++j) acc += v[j] * wv[j];
            }
        };
        if (active) {
            if (SA <= 8 * parts) gather(std::integral_constant<int, 8>{});
            else gather(std::integral_constant<int, 16>{});
        }
        if (units <= NT && parts > 1) {
            s_part[threadIdx.x] = acc;
            __syncthreads();
            if (part == 0)
                for (int pp = 1; pp < parts; ++pp) acc += s_part[pp * units + u];
        }
        if (active && part == 0) {
            // A wait that ran out of patience poisons the output rather than returning a partial sum.
            const float inv = all_arrived ? 1.0f / s_den[h] : __builtin_nanf("");
            const f32x4 r = acc * inv;
            uint16_t* op = a.out + (int64_t)hq * kHeadDim + c4 * 4;
            *reinterpret_cast<uint2*>(op) = make_uint2(pack_bf16(r[0], r[1]), pack_bf16(r[2], r[3]));
            if (a.out_f32) {
                float* of = a.out_f32 + (int64_t)hq * kHeadDim + c4 * 4;  // only 4-byte alignment is promised
#pragma unroll
                for (int e = 0; e < 4; ++e) of[e] = r[e];
            }
        }
    }
}

template <int G, int NW, int NSTAGE, bool APPEND, bool DYN, bool STAGGER = false, bool BYSIDE = false, bool EARLY = false>
__global__ __launch_bounds__(NW * 64, (kWavesPerEu<G, NW>)) void mha_decode_kernel(KernelArgs a) {
    OprojState unused;
    mha_decode_body<G, NW, NSTAGE, APPEND, DYN, STAGGER, false, BYSIDE, EARLY>(a, unused);
}

// The attention launch with the layer's output projection and residual add behind it, in the same launch
// (role of the pair mha_kernel_cu + fused_gemv_add_kernel_cu, code/source/model/qwen3_fused.cpp:548-552).
// A workgroup that has handed its partial results over (every one but the combiners) is idle while the
// combine runs: it requests its share of the projection's weight rows -- they do not depend on the
// attention -- and holds them in registers, waits (bounded) for every head's tag of this launch, reads the
// attention output (ordinary loads: see below) and finishes its rows: dot products, residual add, one
// rounding. The weights stream while HBM would otherwise sit idle behind the attention's hand-over.
// Needs every workgroup of the grid resident at once (the launcher checks the grid against the CU count).
template <int G, int NW, int NSTAGE, bool BYSIDE>
__global__ __launch_bounds__(NW * 64, (kWavesPerEu<G, NW>)) void mha_oproj_kernel(KernelArgs a) {
    OprojState proj;
    mha_decode_body<G, NW, NSTAGE, true, false, false, true, BYSIDE>(a, proj);
    if (!proj.worker) return;
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int n_kv = gridDim.x;
    // Rows are dealt to the wavefronts of the workers in turn: wavefront w takes rows w, w + W, w + 2W.
    const int n_waves = n_kv * ((int)gridDim.y - 1) * NW;
    const int gw = ((int)blockIdx.y * n_kv + (int)blockIdx.x) * NW + wave;
    constexpr int kRows = kOprojRows, kSteps = kOprojSteps;
    const int k16 = a.n_q * (kHeadDim / 8);  // 16-byte chunks per weight row
    const int steps = k16 >> 6;
    const u32x4* w4 = reinterpret_cast<const u32x4*>(a.o_w);
    u32x4 wv[kRows][kSteps];
    int row[kRows];
#pragma unroll
    for (int i = 0; i < kRows; ++i) {
        row[i] = gw + i * n_waves;
        const u32x4* wr = w4 + (int64_t)min(row[i], a.o_n - 1) * k16 + lane;  // rows past the end repeat the last one and are not written
        if (i < LLMI_OPROJ_PREFETCH_ROWS) {
#pragma unroll
            for (int t = 0; t < kSteps; ++t)
                if (t < steps) wv[i][t] = __builtin_nontemporal_load(wr + t * 64);
        }
    }
    // (the residual values these rows are added to travel with the weights)
    float res_in[kRows];
#pragma unroll
    for (int i = 0; i < kRows; ++i) res_in[i] = bf16_lo((uint32_t)a.o_res[min(row[i], a.o_n - 1)]);
    // Bounded wait for the attention output: every head carries this launch's tag. One wavefront per
    // workgroup polls (a thousand wavefronts polling one line slow everything that shares its channel).
    __shared__ int s_seen;
    if (wave == 0) {
        const uint32_t* done = a.ready + 4;
        const uint32_t target = proj.gen_base + 1u;
        bool seen = false;
        for (int spin = 0; spin < a.max_polls; ++spin) {
            const uint32_t d0 = __hip_atomic_load(done + min(lane, a.n_q - 1), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            const uint32_t d1 = __hip_atomic_load(done + min(lane + 64, a.n_q - 1), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            seen = __all(d0 == target && d1 == target);
            if (seen) break;
            __builtin_amdgcn_s_sleep(4);
        }
        if (lane == 0) {
            s_seen = seen ? 1 : 0;
            if (!seen) atomicAdd(&g_poll_timeouts, 1u);
        }
    }
    __syncthreads();
    const bool ok = s_seen != 0;
    // (rows beyond the prefetch depth are fetched now)
#pragma unroll
    for (int i = LLMI_OPROJ_PREFETCH_ROWS; i < kRows; ++i) {
        const u32x4* wr = w4 + (int64_t)min(row[i], a.o_n - 1) * k16 + lane;
#pragma unroll
        for (int t = 0; t < kSteps; ++t)
            if (t < steps) wv[i][t] = __builtin_nontemporal_load(wr + t * 64);
    }
    // The attention output was written through to memory before the word moved, and no cache on this
    // side can hold an older copy: nothing in this launch has read it before, and caches do not keep
    // lines across launches. Ordinary loads, so that an XCD's L2 fetches the 8 KiB once for all its
    // workgroups (a thousand device-coherent reads of the same lines would queue at one memory channel).
    const u32x4* x4 = reinterpret_cast<const u32x4*>(a.out);
    u32x4 xv[kSteps];
#pragma unroll
    for (int t = 0; t < kSteps; ++t)
        if (t < steps) xv[t] = x4[t * 64 + lane];
#pragma unroll
    for (int i = 0; i < kRows; ++i) {
        float acc = 0.0f;
#pragma unroll
        for (int t = 0; t < kSteps; ++t)
            if (t < steps) acc = dot8_bf16(xv[t], wv[i][t], acc);
        acc = wave_sum(acc);
        // fp32 + fp32 -> bf16 once, like fused_gemv_add (matmul_kernel.cu:169-170). A wait that gave up leaves the row
        // as it was: the residual stream is updated in place, and a NaN stored there would destroy the layer's input
        // for good (the give-up is counted, and the combine's own give-up poisons the attention output).
        if (lane == 0 && row[i] < a.o_n && ok) a.o_res[row[i]] = f32_to_bf16(acc + res_in[i]);
    }
}

#ifndef LLMI_STAGES
#define LLMI_STAGES 2
#endif
#ifndef LLMI_RING_LIMIT
#define LLMI_RING_LIMIT 65536
#endif

// The layout by package side has instantiations for the wave counts the dispatcher picks itself; the planner asks
// for it nowhere else (by_side_variant).
template <int G, int NW>
constexpr bool kHasBySide = by_side_variant(G, NW);

template <int G, int NW>
void launch_decode(const KernelArgs& ka, int n_kv, bool append, hipStream_t stream) {
    // NW * NSTAGE * 8 KiB of ring must fit the LDS budget of one workgroup.
    constexpr int kStages = (NW * LLMI_STAGES * 8192 <= LLMI_RING_LIMIT) ? LLMI_STAGES : LLMI_RING_LIMIT / (NW * 8192);
    dim3 grid(n_kv, ka.num_splits);
    const bool dyn = ka.pos_dev != nullptr;  // position read at run time: its own instantiation, the static one pays nothing
    if constexpr (G == 8 && NW == 8) {
        if (append && dyn && ka.group == 8) {  // (kEarlyRows: only these)
            const bool stagger = ka.stagger && ka.num_splits > 1;
            if (ka.by_side && stagger) hipLaunchKernelGGL((mha_decode_kernel<8, 8, kStages, true, true, true, true, true>), grid, dim3(512), 0, stream, ka);
            else if (ka.by_side) hipLaunchKernelGGL((mha_decode_kernel<8, 8, kStages, true, true, false, true, true>), grid, dim3(512), 0, stream, ka);
            else if (stagger) hipLaunchKernelGGL((mha_decode_kernel<8, 8, kStages, true, true, true, false, true>), grid, dim3(512), 0, stream, ka);
            else hipLaunchKernelGGL((mha_decode_kernel<8, 8, kStages, true, true, false, false, true>), grid, dim3(512), 0, stream, ka);
            return;
        }
    }
    if constexpr (kHasBySide<G, NW>) {
        if (ka.by_side) {
            if (append) {
                if (dyn && ka.stagger)
                    hipLaunchKernelGGL((mha_decode_kernel<G, NW, kStages, true, true, true, true>), grid, dim3(NW * 64), 0, stream, ka);
                else if (dyn) hipLaunchKernelGGL((mha_decode_kernel<G, NW, kStages, true, true, false, true>), grid, dim3(NW * 64), 0, stream, ka);
                else if (ka.stagger)
                    hipLaunchKernelGGL((mha_decode_kernel<G, NW, kStages, true, false, true, true>), grid, dim3(NW * 64), 0, stream, ka);
                else hipLaunchKernelGGL((mha_decode_kernel<G, NW, kStages, true, false, false, true>), grid, dim3(NW * 64), 0, stream, ka);
            } else {
                if (dyn && ka.stagger)
                    hipLaunchKernelGGL((mha_decode_kernel<G, NW, kStages, false, true, true, true>), grid, dim3(NW * 64), 0, stream, ka);
                else if (dyn) hipLaunchKernelGGL((mha_decode_kernel<G, NW, kStages, false, true, false, true>), grid, dim3(NW * 64), 0, stream, ka);
                else if (ka.stagger)
                    hipLaunchKernelGGL((mha_decode_kernel<G, NW, kStages, false, false, true, true>), grid, dim3(NW * 64), 0, stream, ka);
                else hipLaunchKernelGGL((mha_decode_kernel<G, NW, kStages, false, false, false, true>), grid, dim3(NW * 64), 0, stream, ka);
            }
            return;
        }
    }
    if (append) {
        if (dyn && ka.stagger && ka.num_splits > 1)
            hipLaunchKernelGGL((mha_decode_kernel<G, NW, kStages, true, true, true>), grid, dim3(NW * 64), 0, stream, ka);
        else if (dyn) hipLaunchKernelGGL((mha_decode_kernel<G, NW, kStages, true, true>), grid, dim3(NW * 64), 0, stream, ka);
        else if (ka.stagger && ka.num_splits > 1)
            hipLaunchKernelGGL((mha_decode_kernel<G, NW, kStages, true, false, true>), grid, dim3(NW * 64), 0, stream, ka);
        else hipLaunchKernelGGL((mha_decode_kernel<G, NW, kStages, true, false>), grid, dim3(NW * 64), 0, stream, ka);
    } else {
        if (dyn && ka.stagger && ka.num_splits > 1)
            hipLaunchKernelGGL((mha_decode_kernel<G, NW, kStages, false, true, true>), grid, dim3(NW * 64), 0, stream, ka);
        else if (dyn) hipLaunchKernelGGL((mha_decode_kernel<G, NW, kStages, false, true>), grid, dim3(NW * 64), 0, stream, ka);
        else if (ka.stagger && ka.num_splits > 1)
            hipLaunchKernelGGL((mha_decode_kernel<G, NW, kStages, false, false, true>), grid, dim3(NW * 64), 0, stream, ka);
        else hipLaunchKernelGGL((mha_decode_kernel<G, NW, kStages, false, false>), grid, dim3(NW * 64), 0, stream, ka);
    }
}

template <int G>
bool launch_decode_nw(const KernelArgs& ka, int n_kv, int nw, bool append, hipStream_t stream) {
    switch (nw) {
        case 1: launch_decode<G, 1>(ka, n_kv, append, stream); return true;
        case 2: launch_decode<G, 2>(ka, n_kv, append, stream); return true;
        case 4: launch_decode<G, 4>(ka, n_kv, append, stream); return true;
        case 8:
            if constexpr (G <= 8) { launch_decode<G, 8>(ka, n_kv, append, stream); return true; }
            return false;
        default: return false;
    }
}

template <int G, int NW>
void launch_oproj(const KernelArgs& ka, int n_kv, hipStream_t stream) {
    constexpr int kStages = (NW * LLMI_STAGES * 8192 <= LLMI_RING_LIMIT) ? LLMI_STAGES : LLMI_RING_LIMIT / (NW * 8192);
    if constexpr (kHasBySide<G, NW>) {
        if (ka.by_side) {
            hipLaunchKernelGGL((mha_oproj_kernel<G, NW, kStages, true>), dim3(n_kv, ka.num_splits), dim3(NW * 64), 0, stream, ka);
            return;
        }
    }
    hipLaunchKernelGGL((mha_oproj_kernel<G, NW, kStages, false>), dim3(n_kv, ka.num_splits), dim3(NW * 64), 0, stream, ka);
}

}  // namespace

// ---- what this translation unit exports: the launchers of its group size ----
#ifndef LLMI_GROUP
#error "define LLMI_GROUP (1, 2, 4, 8 or 16) before including mha_decode_kernels.h"
#endif
#define LLMI_CAT2(a, b) a##b
#define LLMI_CAT(a, b) LLMI_CAT2(a, b)

bool LLMI_CAT(launch_decode_group, LLMI_GROUP)(const KernelArgs& ka, int n_kv, int nw, bool append, hipStream_t stream) {
    return launch_decode_nw<LLMI_GROUP>(ka, n_kv, nw, append, stream);
}

#if LLMI_GROUP <= 8
bool LLMI_CAT(launch_oproj_group, LLMI_GROUP)(const KernelArgs& ka, int n_kv, int nw, hipStream_t stream) {
    constexpr int kWaves = LLMI_GROUP == 8 ? 8 : 4;
    if (nw != kWaves) return false;
    launch_oproj<LLMI_GROUP, kWaves>(ka, n_kv, stream);
    return true;
}
#endif

hipError_t LLMI_CAT(poll_timeouts_group, LLMI_GROUP)(unsigned int* n) {
    return hipMemcpyFromSymbol(n, HIP_SYMBOL(g_poll_timeouts), sizeof(*n));
}

}  // namespace llmi

#endif
