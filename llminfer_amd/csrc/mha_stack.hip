// The attention of SEVERAL consecutive layers of one decode step in ONE launch, for gfx950 (MI355X):
// per layer the fused QK-Norm + RoPE, the K/V append and grouped-query attention over positions 0..pos --
// what the layer loop of the reference issues as one pair of kernels per layer
// (code/source/model/qwen3_fused.cpp:115-127 with :524-548; kernels rmsnorm_kernel.cu:205-290 and
// mha_kernel.cu:440-529), and what llmi_hip_mha_decode_append does per layer here.
//
// Why one launch: at 4096 positions a layer's K and V (16 MiB) stream in about 3 us, but a launch spends 2-3 us
// before its first byte arrives and as long again between its last byte and its result, with HBM idle. Here the
// grid stays resident and walks the layers itself:
//   * the grid is the split path's, one workgroup per (KV head, split) and at most one per compute unit; a wavefront
//     streams its tiles through its ring of LDS slots as one continuous sequence over all layers: the moment a tile
//     of layer l has been read out of its slot, the slot is refilled with the wavefront's next tile, which may
//     belong to layer l+1 -- K and V of the next layer do not depend on this layer's result;
//   * what does depend on it waits for it: layer l+1's query, new K row and new V row are loaded -- and its new row
//     is stored to the cache -- only after every query head of layer l has published its "done" tag, which the
//     merging wavefront of a head writes once the head's output is acknowledged by memory. In an engine the query
//     of layer l+1 is computed from the output of layer l; the launch honours that order also when the buffers
//     alias (a layer's query may BE the previous layer's output);
//   * within a layer everything is the split kernel's: online softmax over 16-position tiles on the matrix cores,
//     the merge of a workgroup's wavefronts through LDS, partial results and arrival records handed to the
//     workgroup of the head's last split, which merges them (log-sum-exp) and writes the bf16 output.
// That chain (mha_stack_kernel) costs 6.8 us per layer, six dependent trips through memory, with HBM idle two thirds of the
// time. It is needed only where a layer can see another layer's writes. Where the caller's buffers say that none can (no
// layer's inputs overlap anything a layer writes, see layers_are_independent in c_api.cpp), the layers may run in any order
// and mha_layers_kernel below runs them as one stream with nothing between a layer and the next
// (or, with enough of them, the kernel of mha_heads.hip, a KV head at a time).
// Every wait is bounded (llmi_hip_set_poll_limit): a wait that gives up is counted and poisons the outputs of its
// layer and the following ones with NaN instead of hanging the device; every wavefront reaches the end of the kernel.
// Needs every workgroup of the grid resident at once (the host checks the grid against the compute unit count).

#include <hip/hip_runtime.h>
#include <stdint.h>

#include "mha_device_helpers.h"

namespace llmi {
namespace {

#ifndef LLMI_STACK_PREFETCH_LATE
// 0: a ring slot is refilled with the wavefront's next tile (of the next layer, at the end of a layer) as soon as it
//    has been read; 1: tiles of the NEXT layer are requested only after the wavefront has handed this layer's
//    partial results over.
#define LLMI_STACK_PREFETCH_LATE 0
#endif

#ifndef LLMI_STACK_SPREAD_MERGE
#define LLMI_STACK_SPREAD_MERGE 1  // the heads of a KV head are merged by different workgroups (see `spread` below)
#endif
#ifndef LLMI_STACK_TIMING_NO_WAIT
// 1: timing-only build that does not wait for the previous layer's tags (wrong whenever a layer's inputs depend on the
// layer before): what the order between layers costs. Never the library's build.
#define LLMI_STACK_TIMING_NO_WAIT 0
#endif

#ifndef LLMI_STACK_STAMPS
// 1: diagnostic build that writes the 100 MHz clock at the phases of four layers (LLMI_STACK_STAMP_LAYER ..+3) into the
// caller's workspace, 4 MiB in (the workspace must be at least 4 MiB + 64 KiB + 16 * grid bytes): per layer and
// workgroup 16 words -- 0 tags seen, 1 operands landed, 2 tiles done, 3 partial results handed over, 4 records in,
// 5 partial rows read back, 6 output acknowledged and tag published (4-6: head 0 of a merging workgroup), 8..11 tiles
// done per wavefront. Never the library's build.
#define LLMI_STACK_STAMPS 0
#endif
#ifndef LLMI_STACK_STAMP_LAYER
#define LLMI_STACK_STAMP_LAYER 16
#endif
#if LLMI_STACK_STAMPS
#define LLMI_STAMP(slot, cond)                                                                                          \
    do {                                                                                                                 \
        const int stamp_l_ = layer - LLMI_STACK_STAMP_LAYER;                                                             \
        if (stamp_l_ >= 0 && stamp_l_ < 4 && lane == 0 && (cond)) {                                                      \
            const int stamp_wg_ = (int)blockIdx.y * (int)gridDim.x + (int)blockIdx.x;                                    \
            const int stamp_i_ = ((stamp_l_ * (int)(gridDim.x * gridDim.y) + stamp_wg_) * 16 + (slot)) & ((1 << 18) - 1); \
            reinterpret_cast<uint32_t*>(reinterpret_cast<char*>(a.ws) + (4u << 20))[stamp_i_] = (uint32_t)wall_clock64();   \
        }                                                                                                                \
    } while (0)
#else
#define LLMI_STAMP(slot, cond) do {} while (0)
#endif

// Copies of a head's done tag, each in a 256-byte line of its own: a workgroup polls copy
// (its index in the grid) % kDoneCopies, so that a line is polled by a few workgroups instead of all of them.
#ifndef LLMI_STACK_DONE_COPIES
#define LLMI_STACK_DONE_COPIES 16
#endif
constexpr int kDoneCopies = LLMI_STACK_DONE_COPIES;
static_assert(kDoneCopies >= 1 && kDoneCopies <= 64, "one lane of the merging wavefront writes each copy");
constexpr int kDoneLineWords = 64;  // 256 bytes: room for 64 heads' tags per copy (128 heads: two lines per copy)

template <int G, int NW, int NSTAGE, bool BYSIDE>
__global__ __launch_bounds__(NW * 64, 2) void mha_stack_kernel(StackArgs sa) {
    const KernelArgs& a = sa.a;
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int n16 = lane & 15;  // MFMA column / DPP-row lane
    const int kg = lane >> 4;   // MFMA k-group / DPP row
    const int kvh = blockIdx.x;  // (the KV head is the fastest grid index: a head's splits and its merging workgroup share an XCD)
    const int split = blockIdx.y;
    const int S = a.num_splits;  // every split holds positions: the host asks for no more splits than tiles

    // The same positions in every layer: tiles 0 .. pos-1 come from the cache, the new token's row from registers.
    const int seq_len = a.seq_len;
    const int cached_len = seq_len - 1;
    const int run = a.tiles_run, longer = a.tiles_longer;  // splits 0 .. longer-1 take run + 1 tiles
    const int ntiles = run + (split < longer ? 1 : 0);
    const int begin = (split * run + min(split, longer)) * kTile;
    const int nrows = min(ntiles * kTile, cached_len - begin);
    // Who merges a query head's splits (log-sum-exp): with at least as many splits as heads in the group, head h's are
    // merged by wavefront 0 of the workgroup of split S-1-h, so that the heads' read-backs run on different compute
    // units at the same time; else the workgroup of the last split merges every head, a wavefront each.
    const bool spread = LLMI_STACK_SPREAD_MERGE && S >= a.group;
    const int merge_head = spread ? (S - 1 - split < a.group ? S - 1 - split : -1) : -1;
    const bool merges_any = spread ? merge_head >= 0 : split == S - 1;
    const bool holds_new_row = split == S - 1 && wave == 0;  // this wavefront takes the new token

    const int64_t split_off = (int64_t)kvh * a.head_stride + (int64_t)begin * a.row_stride;
    const uint32_t rs = (uint32_t)a.row_stride * 2u;
    const uint32_t last_off = (uint32_t)(nrows - 1) * rs;
    const uint32_t k_row = (uint32_t)kg * rs;
    const uint32_t k_col0 = (uint32_t)(n16 ^ kg) * 16u;
    const uint32_t k_col1 = (uint32_t)(n16 ^ (4 + kg)) * 16u;
    const uint32_t k_rd = (uint32_t)((n16 >> 2) * 1024 + (n16 & 3) * 256);
    const uint32_t k_rd0 = k_rd + (uint32_t)((kg ^ (n16 & 7)) * 16);
    const uint32_t k_rd1 = k_rd + (uint32_t)(((4 + kg) ^ (n16 & 7)) * 16);
    const uint32_t v_col = (uint32_t)n16 * 16u;

    // LDS: the wavefronts' rings; the staging of a layer's small operands (norm weights, sin / cos row, new K and V
    // row, the wavefronts' query rows: 1 KiB slots filled by DMA); the wavefronts' partial outputs for the merge; the
    // per-wavefront and merged (max, sum) pairs, the weights of the log-sum-exp merge and the flag of the wait.
    // Just under 80 KiB for groups of four heads: above that the compiler assumes one wavefront per SIMD and moves the
    // accumulators of the matrix products into AGPRs.
    constexpr int kStageBytes = 8192;
    constexpr int kWaveRingBytes = NSTAGE * kStageBytes;
    constexpr int kRingBytes = NW * kWaveRingBytes;
    constexpr int kQSlots = (G * 16 + 63) / 64;
    constexpr int kStagingBytes = (2 + NW * kQSlots) * 1024;
    constexpr int kMergeBytes = NW * G * kHeadDim * (int)sizeof(float);
    constexpr int kTailFloats = 2 * NW * G + 2 * G + G * 64 + 4;
    constexpr int kSmemBytes = kRingBytes + kStagingBytes + kMergeBytes + kTailFloats * 4;
    static_assert(NW > 4 || kSmemBytes <= 80 * 1024, "two workgroups' worth of LDS per CU keeps the VGPR-form matrix instructions");
    static_assert(kSmemBytes <= 160 * 1024, "LDS of one compute unit");
    __shared__ __attribute__((aligned(1024))) char smem[kSmemBytes];
    char* my_ring = smem + wave * kWaveRingBytes;
    const uint32_t my_ring_lds = (uint32_t)(uintptr_t)my_ring;
    char* shared_staging = smem + kRingBytes;
    char* my_rows = shared_staging + (2 + wave * kQSlots) * 1024;
    char* merge_area = smem + kRingBytes + kStagingBytes;
    typedef float (*MergeS)[G];
    auto s_o = [&](int w, int h) { return reinterpret_cast<float*>(merge_area) + (w * G + h) * kHeadDim; };
    MergeS s_m = reinterpret_cast<MergeS>(merge_area + kMergeBytes);
    MergeS s_l = s_m + NW;
    float* s_fin = reinterpret_cast<float*>(s_l + NW);   // [G][2]: merged (max, sum) per head
    float* s_w = s_fin + 2 * G;                          // [G][64] weights of the merge
    int* s_flag = reinterpret_cast<int*>(s_w + G * 64);  // [0]: the previous layer's tags were all seen

    // ---- the stream: this wavefront's tiles of all layers, one sequence ----
    const int n_my = wave < ntiles ? (ntiles - wave + NW - 1) / NW : 0;  // tiles per layer
    int iss_layer = 0, iss_i = 0;  // the next tile to request: tile wave + iss_i * NW of layer iss_layer
    int in_flight = 0;             // tiles requested and not yet read out of their slot
    int iss_stage = 0;
    auto issue_next = [&]() {
        if (n_my == 0 || iss_layer >= sa.layers) return;
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");  // the slot's previous contents have reached the VGPRs
        const char* kb = reinterpret_cast<const char*>(a.k + (int64_t)iss_layer * sa.cache_stride + split_off);
        const char* vb = reinterpret_cast<const char*>(a.v + (int64_t)iss_layer * sa.cache_stride + split_off);
        const uint32_t base = (uint32_t)(wave + iss_i * NW) * (kTile * rs);
        const uint32_t slot = my_ring_lds + (uint32_t)iss_stage * kStageBytes;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const uint32_t ko = min(base + k_row + (uint32_t)(4 * i) * rs, last_off) + ((i & 1) ? k_col1 : k_col0);
            dma16(kb, ko, slot + i * 1024);
        }
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const uint32_t vo = min(base + k_row + (uint32_t)(4 * i) * rs, last_off) + v_col;
            dma16(vb, vo, slot + 4096 + i * 1024);
        }
        ++in_flight;
        iss_stage = (iss_stage + 1 == NSTAGE) ? 0 : iss_stage + 1;
        if (++iss_i == n_my) {
            iss_i = 0;
            ++iss_layer;
        }
    };
    // (a request may belong to the next layer: see LLMI_STACK_PREFETCH_LATE)
    auto issue_within = [&](int layer) {
        if (!LLMI_STACK_PREFETCH_LATE || iss_layer <= layer) issue_next();
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

    // Where this split's partial results and records go (the same rows in every layer: a layer's are consumed
    // before the next layer's are written, and a record names its layer by its tag).
    const int my_xs = package_side<BYSIDE>();
    const int store_xs = my_xs ^ (int)(BYSIDE && !merges_any && (a.far_home == 1 || (a.far_home == 2 && (split & 1))));
    const int64_t part_rows = BYSIDE ? 2 * (((int64_t)a.n_q * S + 15) & ~(int64_t)15) : (int64_t)a.n_q * S;
    const int part_bytes = (int)(part_rows * kHeadDim * (int64_t)sizeof(float));
    const __amdgpu_buffer_rsrc_t part_rsrc = __builtin_amdgcn_make_buffer_rsrc(a.ws, 0, part_bytes, 0x00020000);
    const int n_units = a.group * (kHeadDim / 4);
    // (NW * 64 threads cover G * 32 units: one unit per thread at most, since G <= NW)
    const int u_h = (int)threadIdx.x >> 5, u_c4 = (int)threadIdx.x & 31;
    const int u_hq = kvh * a.group + min(u_h, a.group - 1);
    const WsHead u_wh = ws_head<BYSIDE>(a, u_hq);
    const uint32_t u_po = (uint32_t)(((int64_t)ws_row<4>(u_wh, split, store_xs) * kHeadDim + u_c4 * 4) * (int64_t)sizeof(float));
    const int64_t u_rec = (int64_t)ws_row<9>(u_wh, split, store_xs) * 2;
    const bool u_own = spread ? merge_head == u_h : split == S - 1;  // this workgroup merges the unit's head itself

    // The done tags: copy c of head h at done[c * words_per_copy + h].
    const int words_per_copy = ((a.n_q + kDoneLineWords - 1) / kDoneLineWords) * kDoneLineWords;
    const uint32_t* my_done = sa.done + (size_t)(((int)blockIdx.y * (int)gridDim.x + (int)blockIdx.x) % kDoneCopies) * words_per_copy;

    int rd_stage = 0;       // the slot the wavefront's next tile is in
    bool poisoned = false;  // a wait gave up: this workgroup's results of this layer and the following are NaN
    for (int s0 = 0; s0 < NSTAGE; ++s0) issue_next();

    for (int layer = 0; layer < sa.layers; ++layer) {
        const uint32_t tag = 0x80000000u | ((a.tag + (uint32_t)layer) & 0x7fffffffu);
        // ---- (1) the previous layer is done: every query head carries its tag ----
        if (!LLMI_STACK_TIMING_NO_WAIT && layer > 0 && wave == 0 && !poisoned) {  // (after a give-up nothing is waited for any more: the rest is NaN anyway)
            const uint32_t want = 0x80000000u | ((a.tag + (uint32_t)layer - 1u) & 0x7fffffffu);
            bool seen = false;
            // (one poll at a time, back to back: two, four or eight polls in flight a fraction of a round trip apart see a
            // tag sooner on paper, and measured 0.06, 0.17 and 0.34 us per layer SLOWER -- polls are traffic on the lines
            // the tags have to reach)
            const uint32_t* tag_ptr = my_done + min(lane, a.n_q - 1);
            for (int spin = 0; spin < a.max_polls && !seen; ++spin)
                seen = __all(__hip_atomic_load(tag_ptr, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == want);
            if (lane == 0) {
                *s_flag = seen ? 1 : 0;
                if (!seen) atomicAdd(&g_poll_timeouts, 1u);
            }
        }
        // (also: every wavefront is through with the previous layer's merge area and staging slots)
        __syncthreads();
        if (!LLMI_STACK_TIMING_NO_WAIT && layer > 0 && *s_flag == 0) poisoned = true;
        LLMI_STAMP(0, wave == 0);

        // ---- (2) this layer's small operands, by DMA into the staging slots ----
        const uint16_t* q_l = a.q + (int64_t)layer * sa.q_stride;
        const int c16 = lane & 15, which = lane >> 4;
        {
            const uint32_t st = (uint32_t)(uintptr_t)shared_staging;
            const uint32_t st_rows = (uint32_t)(uintptr_t)my_rows;
            const float* sin_row = a.sin_cache + (int64_t)(seq_len - 1) * 64;
            const float* cos_row = a.cos_cache + (int64_t)(seq_len - 1) * 64;
            const uint64_t w_base = reinterpret_cast<uint64_t>(a.norm_w + (int64_t)layer * sa.normw_stride) + (uint64_t)(which & 1) * 256u;
            const uint64_t t_base = reinterpret_cast<uint64_t>(which == 2 ? sin_row : cos_row);
            const uint64_t p0 = (which < 2 ? w_base : t_base) + (uint64_t)c16 * 16u;
            dma16_gather(reinterpret_cast<const void*>(p0), st);
            if (holds_new_row) {
                const uint16_t* kn = a.k_new + (int64_t)layer * sa.knew_stride;
                const uint16_t* vn = a.v_new + (int64_t)layer * sa.vnew_stride;
                const uint64_t p1 = reinterpret_cast<uint64_t>((which & 1) == 0 ? kn : vn) + (uint64_t)(kvh * kHeadDim * 2 + c16 * 16);
                dma16_gather_coherent(reinterpret_cast<const void*>(p1), st + 1024);
            }
#pragma unroll
            for (int i = 0; i < kQSlots; ++i) {
                const int head = min(which + 4 * i, a.group - 1);
                dma16_gather_coherent(q_l + (int64_t)(kvh * a.group + head) * kHeadDim + c16 * 8, st_rows + i * 1024);
            }
        }
        // (loads complete in order: the tiles requested earlier are in their slots as well)
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        u32x4 qb[4];
        u32x4 new_k[4], new_v;  // the new token's K row (operand layout) and V row, in the wavefront that holds it
        LLMI_STAMP(1, wave == 0);
        float m_run = -INFINITY, l_run = 0.0f;
        f32x4 o[8];
#pragma unroll
        for (int j = 0; j < 8; ++j) o[j] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
        {
            const u32x4* sh4 = reinterpret_cast<const u32x4*>(shared_staging);
            const u32x4* rows4 = reinterpret_cast<const u32x4*>(my_rows);
#pragma unroll
            for (int b4 = 0; b4 < kQSlots; ++b4)
                norm_rope_rows_lds<false>(my_rows, shared_staging, shared_staging + 512, shared_staging + 768, 4 * b4 + kg, n16, a.eps);
            if (holds_new_row)
                norm_rope_rows_lds<false>(shared_staging + 1024, shared_staging + 256, shared_staging + 512, shared_staging + 768, 0, n16, a.eps);
            const int hq_local = min(n16, a.group - 1);
            const bool live = n16 < a.group;
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                const u32x4 qv = rows4[hq_local * 16 + j * 4 + kg];
                qb[j] = live ? qv : u32x4{0u, 0u, 0u, 0u};
            }
            // The new token's row starts the running softmax; it is filed in this layer's cache slot behind the tiles (the
            // stores' acknowledgement must not sit in front of a tile's wait).
            if (holds_new_row) start_from_new_row(sh4 + 64, sh4 + 80, qb, kg, n16, a.scale_log2e, new_k, new_v, m_run, l_run, o);
        }

        // ---- (3) this layer's tiles ----
        for (int i = 0; i < n_my; ++i) {
            TileRegs r;
            // tile i of this layer is the oldest request in flight: in_flight - 1 newer ones may still be travelling
            wait_tiles_in_flight(in_flight - 1);
            read_tile(rd_stage, r);
            rd_stage = (rd_stage + 1 == NSTAGE) ? 0 : rd_stage + 1;
            --in_flight;
            issue_within(layer);
            fold_tile<G>(r, qb, (wave + i * NW) * kTile + 4 * kg, nrows, a.scale_log2e, m_run, l_run, o);
        }

        if (holds_new_row) {
            const int64_t row_off = (int64_t)layer * sa.cache_stride + (int64_t)(seq_len - 1) * a.row_stride + kvh * a.slot_head_stride;
            if (n16 == 0) {
                uint16_t* kd = const_cast<uint16_t*>(a.k) + row_off;
#pragma unroll
                for (int j = 0; j < 4; ++j) *reinterpret_cast<u32x4*>(kd + (j * 4 + kg) * 8) = new_k[j];
            }
            if (kg == 0) *reinterpret_cast<u32x4*>(const_cast<uint16_t*>(a.v) + row_off + n16 * 8) = new_v;
        }
        LLMI_STAMP(2, wave == 0);
        LLMI_STAMP(8 + wave, true);
        // ---- (4) fold the workgroup's wavefronts, hand the split's partial results over ----
        l_run = rows_sum(l_run);
        if (kg == 0) {
#pragma unroll
            for (int r4 = 0; r4 < 4; ++r4) {
                if (r4 < G) {
                    float* dst = s_o(wave, r4) + n16 * 8;
                    *reinterpret_cast<f32x4*>(dst) = f32x4{o[0][r4], o[1][r4], o[2][r4], o[3][r4]};
                    *reinterpret_cast<f32x4*>(dst + 4) = f32x4{o[4][r4], o[5][r4], o[6][r4], o[7][r4]};
                }
            }
            if (n16 < G) {
                s_m[wave][n16] = m_run;
                s_l[wave][n16] = l_run;
            }
        }
        __syncthreads();
        if ((int)threadIdx.x < n_units) {
            float mw[NW], lw[NW];
            f32x4 ow[NW];
#pragma unroll
            for (int w = 0; w < NW; ++w) {
                mw[w] = s_m[w][u_h];
                lw[w] = s_l[w][u_h];
                ow[w] = *reinterpret_cast<const f32x4*>(s_o(w, u_h) + u_c4 * 4);
            }
            asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
            float mx = -INFINITY;
#pragma unroll
            for (int w = 0; w < NW; ++w) mx = fmaxf(mx, mw[w]);
            f32x4 acc = {0.0f, 0.0f, 0.0f, 0.0f};
            float lsum = 0.0f;
#pragma unroll
            for (int w = 0; w < NW; ++w) {
                const float f = (mw[w] == -INFINITY) ? 0.0f : fast_exp2(mw[w] - mx);
                acc += ow[w] * f;
                lsum += lw[w] * f;
            }
            if (poisoned) lsum = __builtin_nanf("");
            // (after a give-up the layer before may not have been read back: its rows stay, and the record's NaN is all of this one)
            else __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u32x4, acc), part_rsrc, u_po, 0, kCacheDevice);
            if (!u_own) {
                // the head's record goes out as soon as this wavefront's stores are acknowledged (the 32 columns of a
                // head are stored by one half of one wavefront)
                asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
                if (u_c4 == 0) {
                    unsigned long long* rec = a.records + u_rec;
                    const unsigned long long t64 = tag;
                    const unsigned long long m_bits = __builtin_bit_cast(uint32_t, mx);
                    const unsigned long long l_bits = __builtin_bit_cast(uint32_t, lsum);
                    __hip_atomic_store(rec, t64 | (m_bits << 32), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                    __hip_atomic_store(rec + 1, t64 | (l_bits << 32), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                }
            } else if (u_c4 == 0) {
                s_fin[2 * u_h] = mx;
                s_fin[2 * u_h + 1] = lsum;
            }
        }
        LLMI_STAMP(3, wave == 0);
        if (LLMI_STACK_PREFETCH_LATE) {
            while (in_flight < NSTAGE && iss_layer < sa.layers && n_my > 0) issue_next();
        }
        if (!merges_any) continue;

        // ---- (5) the log-sum-exp merge of a head's splits, one wavefront per head ----
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // its own partial stores are acknowledged
        __syncthreads();                                  // ... and its (max, sum) pairs are in LDS
        if (spread ? wave == 0 : wave < a.group) {
            const int h = spread ? merge_head : wave;
            const int c4 = lane & 31, part = lane >> 5;
            const int hq = kvh * a.group + h;
            const WsHead wh = ws_head<BYSIDE>(a, hq);
            // the records of the other splits, one per lane; this workgroup's own pair comes from LDS
            float m_reg = -INFINITY, l_reg = 0.0f;
            bool home = my_xs != 0;
            bool ok = false;
            const unsigned long long* rec_near = a.records + (int64_t)ws_row<9>(wh, min(lane, S - 1), my_xs) * 2;
            auto poll_round = [&](auto both_tag) {
                constexpr bool kBoth = decltype(both_tag)::value;
                ok = true;
                m_reg = -INFINITY;
                l_reg = 0.0f;
                if (lane < S && lane != split) {
                    const unsigned long long* rec = rec_near;
                    unsigned long long r0 = __hip_atomic_load(rec, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                    unsigned long long r1 = __hip_atomic_load(rec + 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                    bool here = (uint32_t)r0 == tag && (uint32_t)r1 == tag;
                    if constexpr (kBoth) {
                        home = my_xs != 0;
                        if (!here) {
                            rec = a.records + (int64_t)ws_row<9>(wh, lane, my_xs ^ 1) * 2;
                            r0 = __hip_atomic_load(rec, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                            r1 = __hip_atomic_load(rec + 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                            here = (uint32_t)r0 == tag && (uint32_t)r1 == tag;
                            home = my_xs == 0;
                        }
                    }
                    ok = here;
                    m_reg = __builtin_bit_cast(float, (uint32_t)(r0 >> 32));
                    l_reg = __builtin_bit_cast(float, (uint32_t)(r1 >> 32));
                } else if (lane == split) {
                    m_reg = s_fin[2 * h];
                    l_reg = s_fin[2 * h + 1];
                }
                return __all(ok);
            };
            constexpr int kNearRounds = 16;
            const int near_rounds = BYSIDE ? min(a.max_polls, kNearRounds) : a.max_polls;
            bool all_in = false;
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
            if (__builtin_expect(!arrived, 0) && lane == 0) atomicAdd(&g_poll_timeouts, 1u);
            LLMI_STAMP(4, wave == 0);

            const uint32_t row0_bytes = (uint32_t)wh.rbase * (kHeadDim * 4u);
            const uint32_t block_mask = BYSIDE ? ~(uint32_t)(kSideBlockBytes - 1) : 0u;
            const uint32_t lane_bytes = (uint32_t)c4 * 16u;
            const bool mixed = BYSIDE && __any(home != (my_xs != 0));
            const unsigned long long home_flags = __ballot(home);
            auto load_partial = [&](int sp) {
                const int spc = min(sp, S - 1);
                const uint32_t B = row0_bytes + (uint32_t)spc * (kHeadDim * 4u);
                uint32_t home_bytes = 0u;
                if constexpr (BYSIDE) {
                    const int xs = mixed ? (int)((home_flags >> spc) & 1ull) : my_xs;
                    home_bytes = (uint32_t)(wh.ppar ^ xs) * kSideBlockBytes;
                }
                return __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(part_rsrc, B + (B & block_mask) + home_bytes + lane_bytes, 0, kCacheDevice));
            };
            // lane = (16-byte column, half of the splits): all of a lane's partial rows requested at once, the weights
            // worked out while they travel
            constexpr int kBatch = 16;
            f32x4 v[kBatch];
#pragma unroll
            for (int j = 0; j < kBatch; ++j) v[j] = load_partial(part + 2 * j);
            float mx = wave_max(m_reg);
            const float f = (m_reg == -INFINITY) ? 0.0f : fast_exp2(m_reg - mx);
            float* w = s_w + h * 64;
            if (lane < S) {
                w[lane] = f;
                if (lane != split) {  // consumed: cleared, so that a replay of this launch (same tags) starts clean
                    unsigned long long* rec = a.records + (int64_t)ws_row<9>(wh, lane, home ? 1 : 0) * 2;
                    __hip_atomic_store(rec, 0ull, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                    __hip_atomic_store(rec + 1, 0ull, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                }
            }
            const float den = wave_sum(lane < S ? l_reg * f : 0.0f);
            asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
            __builtin_amdgcn_wave_barrier();
            f32x4 sum = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
            for (int j = 0; j < kBatch; ++j) {
                const int sp = part + 2 * j;
                sum += v[j] * (sp < S ? w[sp] : 0.0f);
            }
            for (int s0 = part + 2 * kBatch; s0 < S; s0 += 2 * kBatch) {
#pragma unroll
                for (int j = 0; j < kBatch; ++j) v[j] = load_partial(s0 + 2 * j);
#pragma unroll
                for (int j = 0; j < kBatch; ++j) {
                    const int sp = s0 + 2 * j;
                    sum += v[j] * (sp < S ? w[sp] : 0.0f);
                }
            }
#pragma unroll
            for (int e = 0; e < 4; ++e) sum[e] = halves_sum(sum[e]);
            LLMI_STAMP(5, wave == 0);
            if (part == 0) {
                const float inv = (arrived && !poisoned) ? 1.0f / den : __builtin_nanf("");
                const f32x4 r = sum * inv;
                const unsigned long long packed = (unsigned long long)pack_bf16(r[0], r[1]) | ((unsigned long long)pack_bf16(r[2], r[3]) << 32);
                unsigned long long* op = reinterpret_cast<unsigned long long*>(a.out + (int64_t)layer * sa.out_stride + (int64_t)hq * kHeadDim + c4 * 4);
                // (device scope: the next layer of this launch may read this row as its query, from any XCD)
                __hip_atomic_store(op, packed, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                if (a.out_f32) {
                    float* of = a.out_f32 + (int64_t)layer * sa.out_stride + (int64_t)hq * kHeadDim + c4 * 4;
#pragma unroll
                    for (int e = 0; e < 4; ++e) of[e] = r[e];
                }
            }
            // The head's output (and its cleared records) are acknowledged: every copy of its done tag says so.
            if (layer + 1 < sa.layers) {
                asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
                if (lane < kDoneCopies)
                    __hip_atomic_store(sa.done + (size_t)lane * words_per_copy + hq, tag, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            }
            LLMI_STAMP(6, wave == 0);
        }
    }
}

// ---- layers that cannot see each other's writes ----
// The same results as mha_stack_kernel and as one launch per layer, bit for bit (the same tiles per split and wavefront, the
// same folds in the same order), with nothing in front of a layer: what bounds it is the K/V stream. The grid is the same,
// one workgroup per (KV head, split) and compute unit, resident, walking the layers; its eight wavefronts have roles, and meet
// at one workgroup barrier per layer:
//   0-3  stream: tiles through a ring of kNStage LDS slots, one sequence over all layers, and fold them; four slots hold two
//        layers' tiles ahead at 4096 positions. They do nothing else: no wavefront that streams ever waits for a store;
//   4, 5 fold the four wavefronts' results of the layer before (one thread per head and 16-byte column) and store the split's
//        partial rows, while 0-3 are in the next layer; the records follow a layer later, when the rows' acknowledgement has
//        long arrived;
//   6    brings in a later layer's small operands, normalises and rotates the query group once for the workgroup (the
//        streaming wavefronts read operand fragments) and files the new token's rows in the cache;
//   7    merges a head's splits, a step per layer and nothing waited for in between: asks for the records two layers behind,
//        turns them into weights and asks for the partial rows three layers behind, sums them up four layers behind. A head's
//        merging workgroup moves on from layer to layer (merge_split), so that each takes part every num_splits / group layers.
// With the stream running a trip to memory takes 2 us and more, about as long as a layer's stream per workgroup (2.4 us at 4096
// positions): waiting for one anywhere in a layer costs the stream (records right behind their rows + 12 us, a merge in
// one piece + 10 us of 89 us over 36 layers).
// A layer's partial rows and records live in region layer % regions of the workspace; region reuse waits for the heads' done
// tags of the layer that had it before (set by 7 once the rows have been read back; normally long there).
// Layer j's tags are set while layer j + kMergeLag streams, so with more regions than that no wait is for anything later than
// its own layer and there is no cycle; with fewer (three or four) 7 takes its steps one after the other two layers behind.
// 32 Q / 8 KV heads, 36 layers at 4096 + 1 positions: 243 us as a chain (mha_stack_kernel) -> 107 us = 5.6 TB/s; at 300 positions
// 190 -> 54 us. The stream alone, with neither partial rows stored nor merges, is 89 us (6.8 TB/s): half a megabyte of stores per
// layer costs 10 us and reading it back 8, whatever their cache policy and however many layers' stores go out together --
// writes between a saturating stream of reads. Two, three or four ring slots: level.
constexpr int kLayersStage = 4;   // ring slots per streaming wavefront
constexpr int kLayersWaves = 8;
constexpr int kStreamWaves = 4;   // wavefronts per split, as in the per-layer launches
constexpr int kRecordLag = 2;     // layers behind the stream at which a merge asks for the records ...
constexpr int kMergeLag = 4;      // ... and finishes

// The workgroup (its split) that merges head h of the group in a layer.
__device__ __forceinline__ int merge_split(int layer, int h, int group, int S) {
    return S - 1 - (int)((uint32_t)(layer * group + h) % (uint32_t)S);
}

template <int G>
__global__ __launch_bounds__(kLayersWaves * 64, 2) void mha_layers_kernel(StackArgs sa) {
    static_assert(G <= 4, "two wavefronts fold a workgroup's G * 32 columns");
    const KernelArgs& a = sa.a;
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int n16 = lane & 15;
    const int kg = lane >> 4;
    const int kvh = blockIdx.x;
    const int split = blockIdx.y;
    const int S = a.num_splits, L = sa.layers;
    const int seq_len = a.seq_len, cached_len = seq_len - 1;
    const int run = a.tiles_run, longer = a.tiles_longer;
    const int ntiles = run + (split < longer ? 1 : 0);
    const int begin = (split * run + min(split, longer)) * kTile;
    const int nrows = min(ntiles * kTile, cached_len - begin);
    const bool holds_new_row = split == S - 1;

    // LDS: the rings; three layers' small operands (3 KiB each: q_norm | k_norm | sin | cos, new K row | new V row, the
    // query rows); two layers' results of the streaming wavefronts; the weights of a merge.
    constexpr int kStageBytes = 8192;
    constexpr int kRingBytes = kStreamWaves * kLayersStage * kStageBytes;
    constexpr int kOperandBytes = 3 * 1024, kOperandSets = 3;
    constexpr int kFoldRows = kStreamWaves * G * kHeadDim * (int)sizeof(float);
    constexpr int kFoldBytes = kFoldRows + 2 * kStreamWaves * G * (int)sizeof(float);
    constexpr int kSmemBytes = kRingBytes + kOperandSets * kOperandBytes + 2 * kFoldBytes + 64 * (int)sizeof(float);
    static_assert(kSmemBytes <= 160 * 1024, "LDS of one compute unit");
    static_assert(kFoldBytes % 16 == 0, "16-byte accesses");
    __shared__ __attribute__((aligned(1024))) char smem[kSmemBytes];
    char* operands = smem + kRingBytes;
    char* folds = operands + kOperandSets * kOperandBytes;
    float* s_w = reinterpret_cast<float*>(folds + 2 * kFoldBytes);
    auto fold_o = [&](int set, int w, int h) { return reinterpret_cast<float*>(folds + set * kFoldBytes) + (w * G + h) * kHeadDim; };
    auto fold_m = [&](int set, int w, int h) { return reinterpret_cast<float*>(folds + set * kFoldBytes + kFoldRows) + w * G + h; };
    auto fold_l = [&](int set, int w, int h) { return fold_m(set, kStreamWaves + w, h); };
    // This wavefront's LDS accesses are done, then all wavefronts meet. (Requests to memory stay in flight.)
    auto meet = [&]() {
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
    };
    auto layer_tag = [&](int layer) { return 0x80000000u | ((a.tag + (uint32_t)layer) & 0x7fffffffu); };
    // (a record: tag, max, tag, sum; behind the region's partial rows)
    auto record_offset = [&](int region, int hq, int sp) {
        return (uint32_t)region * (uint32_t)sa.region_bytes + (uint32_t)(a.n_q * S) * (kHeadDim * 4u) + (uint32_t)(hq * S + sp) * 16u;
    };
    const __amdgpu_buffer_rsrc_t part_rsrc =
        __builtin_amdgcn_make_buffer_rsrc(a.ws, 0, (int)(sa.regions * sa.region_bytes), 0x00020000);

    if (wave < kStreamWaves) {
        const int64_t split_off = (int64_t)kvh * a.head_stride + (int64_t)begin * a.row_stride;
        const uint32_t rs = (uint32_t)a.row_stride * 2u;
        const uint32_t last_off = (uint32_t)(nrows - 1) * rs;
        const uint32_t k_row = (uint32_t)kg * rs;
        const uint32_t k_col0 = (uint32_t)(n16 ^ kg) * 16u;
        const uint32_t k_col1 = (uint32_t)(n16 ^ (4 + kg)) * 16u;
        const uint32_t k_rd = (uint32_t)((n16 >> 2) * 1024 + (n16 & 3) * 256);
        const uint32_t k_rd0 = k_rd + (uint32_t)((kg ^ (n16 & 7)) * 16);
        const uint32_t k_rd1 = k_rd + (uint32_t)(((4 + kg) ^ (n16 & 7)) * 16);
        const uint32_t v_col = (uint32_t)n16 * 16u;
        char* my_ring = smem + wave * kLayersStage * kStageBytes;
        const uint32_t my_ring_lds = (uint32_t)(uintptr_t)my_ring;
        const int n_my = wave < ntiles ? (ntiles - wave + kStreamWaves - 1) / kStreamWaves : 0;
        int iss_layer = 0, iss_i = 0, iss_stage = 0, in_flight = 0, rd_stage = 0;
        auto issue_next = [&]() {
            if (n_my == 0 || iss_layer >= L) return;
            asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");  // the slot's previous contents have reached the VGPRs
            const char* kb = reinterpret_cast<const char*>(a.k + (int64_t)iss_layer * sa.cache_stride + split_off);
            const char* vb = reinterpret_cast<const char*>(a.v + (int64_t)iss_layer * sa.cache_stride + split_off);
            const uint32_t base = (uint32_t)(wave + iss_i * kStreamWaves) * (kTile * rs);
            const uint32_t slot = my_ring_lds + (uint32_t)iss_stage * kStageBytes;
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const uint32_t ko = min(base + k_row + (uint32_t)(4 * i) * rs, last_off) + ((i & 1) ? k_col1 : k_col0);
                dma16(kb, ko, slot + i * 1024);
            }
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const uint32_t vo = min(base + k_row + (uint32_t)(4 * i) * rs, last_off) + v_col;
                dma16(vb, vo, slot + 4096 + i * 1024);
            }
            ++in_flight;
            iss_stage = (iss_stage + 1 == kLayersStage) ? 0 : iss_stage + 1;
            if (++iss_i == n_my) {
                iss_i = 0;
                ++iss_layer;
            }
        };
        for (int s0 = 0; s0 < kLayersStage; ++s0) issue_next();
        meet();  // layer 0's query is in LDS
        int op_set = 0;
        for (int layer = 0; layer < L; ++layer) {
            const u32x4* ops4 = reinterpret_cast<const u32x4*>(operands + op_set * kOperandBytes);
            op_set = op_set + 1 == kOperandSets ? 0 : op_set + 1;
            const int hq_local = min(n16, a.group - 1);
            const bool live = n16 < a.group;
            u32x4 qb[4];
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                const u32x4 qv = ops4[128 + hq_local * 16 + j * 4 + kg];
                qb[j] = live ? qv : u32x4{0u, 0u, 0u, 0u};
            }
            float m_run = -INFINITY, l_run = 0.0f;
            f32x4 o[8];
#pragma unroll
            for (int j = 0; j < 8; ++j) o[j] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
            if (holds_new_row && wave == 0) {
                u32x4 kf[4], vf;
                start_from_new_row(ops4 + 64, ops4 + 80, qb, kg, n16, a.scale_log2e, kf, vf, m_run, l_run, o);
            }
            for (int i = 0; i < n_my; ++i) {
                TileRegs r;
                wait_tiles_in_flight(in_flight - 1);
                const char* kp = my_ring + rd_stage * kStageBytes;
#pragma unroll
                for (int j = 0; j < 4; ++j)
                    r.k[j] = *reinterpret_cast<const u32x4*>(kp + ((j & 1) ? k_rd1 : k_rd0) + (j >> 1) * 128);
#pragma unroll
                for (int e = 0; e < 4; ++e)
                    r.v[e] = *reinterpret_cast<const u32x4*>(kp + 4096 + kg * 1024 + e * 256 + n16 * 16);
                rd_stage = (rd_stage + 1 == kLayersStage) ? 0 : rd_stage + 1;
                --in_flight;
                issue_next();
                fold_tile<G>(r, qb, (wave + i * kStreamWaves) * kTile + 4 * kg, nrows, a.scale_log2e, m_run, l_run, o);
            }
            l_run = rows_sum(l_run);
            const int set = layer & 1;
            if (kg == 0) {
#pragma unroll
                for (int r4 = 0; r4 < 4; ++r4) {
                    if (r4 < G) {
                        float* dst = fold_o(set, wave, r4) + n16 * 8;
                        *reinterpret_cast<f32x4*>(dst) = f32x4{o[0][r4], o[1][r4], o[2][r4], o[3][r4]};
                        *reinterpret_cast<f32x4*>(dst + 4) = f32x4{o[4][r4], o[5][r4], o[6][r4], o[7][r4]};
                    }
                }
                if (n16 < G) {
                    *fold_m(set, wave, n16) = m_run;
                    *fold_l(set, wave, n16) = l_run;
                }
            }
            meet();
        }
    } else if (wave < 6) {
        const int u = (wave - kStreamWaves) * 64 + lane;
        const int h = min(u >> 5, a.group - 1), c4 = u & 31;
        const bool active = u < a.group * (kHeadDim / 4);
        const int hq = kvh * a.group + h;
        const uint32_t po = (uint32_t)(((int64_t)hq * S + split) * kHeadDim + c4 * 4) * (uint32_t)sizeof(float);
        // Region reuse: every `step` layers the tags of the `step` layers that had the next regions, one lane per layer and
        // head, asked for a layer ahead.
        const int step = max(1, min(8, sa.regions - kMergeLag - 2));
        int next_check = sa.regions;
        auto ask_done = [&](int layer) {
            const int k = min(lane >> 2, step - 1);
            return __hip_atomic_load(sa.done + ((layer + k) % sa.regions) * kDoneLineWords + kvh * a.group + min(lane & 3, a.group - 1),
                                     __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        };
        auto wanted = [&](int layer) { return layer_tag(layer - sa.regions + min(lane >> 2, step - 1)); };
        uint32_t seen = 0;
        bool poisoned = false;  // a wait gave up: this split's results of the layer and the following ones are NaN
        int region = 0, prev_region = 0;
        float prev_m = 0.0f, prev_l = 0.0f;
        // The records of a layer's partial rows, once those are acknowledged. (The 32 columns of a head are stored by one half
        // of one wavefront.)
        auto publish = [&](int layer) {
            asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
            // (one 16-byte store: either half carries the tag, so it does not matter if they arrive one after the other)
            if (active && c4 == 0)
                __builtin_amdgcn_raw_buffer_store_b128(
                    u32x4{layer_tag(layer), __builtin_bit_cast(uint32_t, prev_m), layer_tag(layer), __builtin_bit_cast(uint32_t, prev_l)},
                    part_rsrc, record_offset(prev_region, hq, split), 0, kCacheDevice);
        };
        meet();
        for (int layer = 0; layer < L; ++layer) {
            meet();
            const int set = layer & 1;
            float mw[kStreamWaves], lw[kStreamWaves];
            f32x4 ow[kStreamWaves];
#pragma unroll
            for (int w = 0; w < kStreamWaves; ++w) {
                mw[w] = *fold_m(set, w, h);
                lw[w] = *fold_l(set, w, h);
                ow[w] = *reinterpret_cast<const f32x4*>(fold_o(set, w, h) + c4 * 4);
            }
            if (layer > 0) publish(layer - 1);
            asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
            float mx = -INFINITY;
#pragma unroll
            for (int w = 0; w < kStreamWaves; ++w) mx = fmaxf(mx, mw[w]);
            f32x4 acc = {0.0f, 0.0f, 0.0f, 0.0f};
            float lsum = 0.0f;
#pragma unroll
            for (int w = 0; w < kStreamWaves; ++w) {
                const float f = (mw[w] == -INFINITY) ? 0.0f : fast_exp2(mw[w] - mx);
                acc += ow[w] * f;
                lsum += lw[w] * f;
            }
            if (layer == next_check && !poisoned) {
                bool free = a.max_polls > 0 && __all(seen == wanted(layer));
                for (int spin = 1; spin < a.max_polls && !free; ++spin) free = __all(ask_done(layer) == wanted(layer));
                if (__builtin_expect(!free, 0)) {
                    poisoned = true;
                    if (lane == 0) atomicAdd(&g_poll_timeouts, 1u);
                }
                next_check += step;
            }
            // (after a give-up the layer that had the region may not have been read back: its rows stay, and the record's NaN is all
            // of this one)
            if (active && !poisoned)
                __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u32x4, acc), part_rsrc,
                                                       po + (uint32_t)region * (uint32_t)sa.region_bytes, 0, kCacheDevice);
            prev_m = mx;
            prev_l = poisoned ? __builtin_nanf("") : lsum;
            prev_region = region;
            region = region + 1 == sa.regions ? 0 : region + 1;
            if (layer + 1 == next_check) seen = ask_done(layer + 1);
        }
        publish(L - 1);
    } else if (wave == 6) {
        const int c16 = lane & 15, which = lane >> 4;
        auto fetch = [&](int layer, int set) {
            const uint32_t st = (uint32_t)(uintptr_t)(operands + set * kOperandBytes);
            const float* sin_row = a.sin_cache + (int64_t)(seq_len - 1) * 64;
            const float* cos_row = a.cos_cache + (int64_t)(seq_len - 1) * 64;
            const uint64_t w_base = reinterpret_cast<uint64_t>(a.norm_w + (int64_t)layer * sa.normw_stride) + (uint64_t)(which & 1) * 256u;
            const uint64_t t_base = reinterpret_cast<uint64_t>(which == 2 ? sin_row : cos_row);
            dma16_gather(reinterpret_cast<const void*>((which < 2 ? w_base : t_base) + (uint64_t)c16 * 16u), st);
            if (holds_new_row) {
                const uint16_t* kn = a.k_new + (int64_t)layer * sa.knew_stride;
                const uint16_t* vn = a.v_new + (int64_t)layer * sa.vnew_stride;
                const uint64_t p1 = reinterpret_cast<uint64_t>((which & 1) == 0 ? kn : vn) + (uint64_t)(kvh * kHeadDim * 2 + c16 * 16);
                dma16_gather(reinterpret_cast<const void*>(p1), st + 1024);
            }
            const int head = min(which, a.group - 1);
            dma16_gather(a.q + (int64_t)layer * sa.q_stride + (int64_t)(kvh * a.group + head) * kHeadDim + c16 * 8, st + 2048);
        };
        // Layer p's operands are asked for a barrier ahead of their use here and handed over a barrier ahead of the layer.
        fetch(0, 0);
        int set = 0;
        for (int p = 0; p < L; ++p) {
            char* ops = operands + set * kOperandBytes;
            set = set + 1 == kOperandSets ? 0 : set + 1;
            asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
            if (p + 1 < L) fetch(p + 1, set);
            norm_rope_rows_lds<true>(ops + 2048, ops, ops + 512, ops + 768, kg, n16, a.eps);
            if (holds_new_row) {
                norm_rope_rows_lds<true>(ops + 1024, ops + 256, ops + 512, ops + 768, 0, n16, a.eps);
                asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
                const u32x4* rows = reinterpret_cast<const u32x4*>(ops + 1024);
                const int64_t row_off = (int64_t)p * sa.cache_stride + (int64_t)(seq_len - 1) * a.row_stride + kvh * a.slot_head_stride;
                uint16_t* dst = const_cast<uint16_t*>(which == 0 ? a.k : a.v) + row_off;
                if (which < 2) *reinterpret_cast<u32x4*>(dst + c16 * 8) = rows[which * 16 + c16];
            }
            meet();
        }
        meet();
    } else {
        const int c4 = lane & 31, part = lane >> 5;
        constexpr int kBatch = 16;
        // What a merge carries from step to step: the records, then the rows and what their weights need.
        u32x4 rec = {0u, 0u, 0u, 0u};
        f32x4 v[kBatch];
        float den = 0.0f;
        bool arrived = false;
        auto head_of = [&](int layer) {  // the head of the group this workgroup merges in the layer, or -1
            if (layer < 0 || layer >= L) return -1;
            int found = -1;
            for (int h = 0; h < a.group; ++h) found = merge_split(layer, h, a.group, S) == split ? h : found;
            return found;
        };
        auto load_record = [&](int layer, int hq) {
            return __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(
                                                 part_rsrc, record_offset(layer % sa.regions, hq, min(lane, S - 1)), 0, kCacheDevice));
        };
        auto load_partial = [&](int layer, int hq, int sp) {
            const uint32_t base = (uint32_t)(layer % sa.regions) * (uint32_t)sa.region_bytes + (uint32_t)hq * (uint32_t)S * (kHeadDim * 4u);
            return __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(
                                                 part_rsrc, base + (uint32_t)c4 * 16u + (uint32_t)min(sp, S - 1) * (kHeadDim * 4u), 0, kCacheDevice));
        };
        auto ask_records = [&](int layer) {
            const int h = head_of(layer);
            if (h < 0) return;
            asm volatile("" ::: "memory");
            rec = load_record(layer, kvh * a.group + h);
        };
        auto ask_rows = [&](int layer) {
            const int h = head_of(layer);
            if (h < 0) return;
            const int hq = kvh * a.group + h;
            const uint32_t tag = layer_tag(layer);
            arrived = a.max_polls > 0 && __all(rec[0] == tag && rec[2] == tag);
            for (int spin = 1; spin < a.max_polls && !arrived; ++spin) {
                asm volatile("" ::: "memory");  // (a poll is a load of its own ...)
                rec = load_record(layer, hq);
                arrived = __all(rec[0] == tag && rec[2] == tag);
            }
            asm volatile("" ::: "memory");  // (... and the rows are asked for behind the last one)
            if (__builtin_expect(!arrived, 0) && lane == 0) atomicAdd(&g_poll_timeouts, 1u);
#pragma unroll
            for (int j = 0; j < kBatch; ++j) v[j] = load_partial(layer, hq, part + 2 * j);
            const uint32_t m_bits = rec[1], l_bits = rec[3];
            const float m_reg = lane < S ? __builtin_bit_cast(float, m_bits) : -INFINITY;
            const float l_reg = lane < S ? __builtin_bit_cast(float, l_bits) : 0.0f;
            const float mx = wave_max(m_reg);
            const float f = (m_reg == -INFINITY) ? 0.0f : fast_exp2(m_reg - mx);
            if (lane < S) {
                s_w[lane] = f;
                // A record is cleared only where a replay of this launch (same tags) would find it again: in a region that
                // one layer has to itself. Elsewhere the region's other layers leave another layer's tag there.
                if (layer < sa.regions && layer + sa.regions >= L)
                    __builtin_amdgcn_raw_buffer_store_b128(u32x4{0u, 0u, 0u, 0u}, part_rsrc, record_offset(layer, hq, lane), 0, kCacheDevice);
            }
            den = wave_sum(lane < S ? l_reg * f : 0.0f);
        };
        auto finish = [&](int layer) {
            const int h = head_of(layer);
            if (h < 0) return;
            const int hq = kvh * a.group + h;
            asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
            __builtin_amdgcn_wave_barrier();
            f32x4 sum = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
            for (int j = 0; j < kBatch; ++j) {
                const int sp = part + 2 * j;
                sum += v[j] * (sp < S ? s_w[sp] : 0.0f);
            }
            for (int s0 = part + 2 * kBatch; s0 < S; s0 += 2 * kBatch) {
#pragma unroll
                for (int j = 0; j < kBatch; ++j) v[j] = load_partial(layer, hq, s0 + 2 * j);
#pragma unroll
                for (int j = 0; j < kBatch; ++j) {
                    const int sp = s0 + 2 * j;
                    sum += v[j] * (sp < S ? s_w[sp] : 0.0f);
                }
            }
#pragma unroll
            for (int e = 0; e < 4; ++e) sum[e] = halves_sum(sum[e]);
            // The rows have been read and the records are cleared (asked for a step ago): the region is free for this head.
            asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
            if (lane == 0)
                __hip_atomic_store(sa.done + (layer % sa.regions) * kDoneLineWords + hq, layer_tag(layer), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            if (part == 0) {
                const f32x4 r = sum * (arrived ? 1.0f / den : __builtin_nanf(""));
                const int64_t off = (int64_t)layer * sa.out_stride + (int64_t)hq * kHeadDim + c4 * 4;
                *reinterpret_cast<uint2*>(a.out + off) = make_uint2(pack_bf16(r[0], r[1]), pack_bf16(r[2], r[3]));
                if (a.out_f32) {
#pragma unroll
                    for (int e = 0; e < 4; ++e) a.out_f32[off + e] = r[e];  // (only 4-byte alignment is promised)
                }
            }
        };
        const bool in_steps = sa.regions > kMergeLag;
        meet();
        for (int layer = 0; layer < L + kMergeLag; ++layer) {
            if (layer < L) meet();
            if (in_steps) {
                finish(layer - kMergeLag);
                ask_rows(layer - kRecordLag - 1);
                ask_records(layer - kRecordLag);
            } else {
                ask_records(layer - kRecordLag);
                ask_rows(layer - kRecordLag);
                finish(layer - kRecordLag);
            }
        }
    }
}

template <int G>
bool launch_stack_g(const StackArgs& sa, int n_kv, hipStream_t stream) {
#ifndef LLMI_STACK_WAVES
#define LLMI_STACK_WAVES 4
#endif
    constexpr int NW = LLMI_STACK_WAVES, NSTAGE = 8 / NW;  // the rings hold eight tiles per workgroup either way
    const dim3 grid(n_kv, sa.a.num_splits), block(NW * 64);
    if (sa.regions > 0) {
        hipLaunchKernelGGL((mha_layers_kernel<G>), grid, dim3(kLayersWaves * 64), 0, stream, sa);
        return true;
    }
    if (sa.a.by_side) hipLaunchKernelGGL((mha_stack_kernel<G, NW, NSTAGE, true>), grid, block, 0, stream, sa);
    else hipLaunchKernelGGL((mha_stack_kernel<G, NW, NSTAGE, false>), grid, block, 0, stream, sa);
    return true;
}

}  // namespace

bool launch_stack(const StackArgs& sa, int n_kv, int group_pad, int waves, hipStream_t stream) {
    if (waves != 4) return false;  // (the plan's wave count; the kernel's own is LLMI_STACK_WAVES)
    switch (group_pad) {
        case 1: return launch_stack_g<1>(sa, n_kv, stream);
        case 2: return launch_stack_g<2>(sa, n_kv, stream);
        case 4: return launch_stack_g<4>(sa, n_kv, stream);
        default: return false;
    }
}

int stack_max_regions(int head_num) { return head_num <= kDoneLineWords ? kDoneCopies : 0; }

size_t stack_done_bytes(int head_num) {
    return (size_t)kDoneCopies * (size_t)((head_num + kDoneLineWords - 1) / kDoneLineWords) * kDoneLineWords * sizeof(uint32_t);
}

hipError_t poll_timeouts_stack(unsigned int* n) { return hipMemcpyFromSymbol(n, HIP_SYMBOL(g_poll_timeouts), sizeof(*n)); }

}  // namespace llmi
