// The per-token writers that feed decode attention on gfx950:
//   * fused per-head RMSNorm * weight + half-rotation RoPE on the query (in
//     place) and on the new K row, which lands in its cache slot in either
//     layout together with the new V row
//     (role of fused_qk_norm_rope_kernel, code/source/op/kernel/cuda/rmsnorm_kernel.cu:205-290,
//     plus the slot addressing of Model::slice_kv_cache, code/source/model/model.cpp:90-107);
//   * the sin/cos table (role of sin_cos_cache_kernel, code/source/op/kernel/cuda/rope_kernel.cu:6-21);
//   * a position-major -> head-major cache copy.
// One wavefront per head: lane i owns the rotation pair (i, i+64), the sum of
// squares is folded across the 64 lanes with DPP row steps and scalar reads, no LDS.

#include <hip/hip_runtime.h>
#include <stdint.h>

#include "llmi_internal.h"
#include "wave_ops.h"

namespace llmi {
namespace {

constexpr int kHeadDim = 128;
constexpr int kHalf = 64;

__device__ __forceinline__ float bf16_to_f32(uint16_t h) {
    return __builtin_bit_cast(float, (uint32_t)h << 16);
}

__device__ __forceinline__ uint16_t f32_to_bf16(float x) {
    uint32_t u = __builtin_bit_cast(uint32_t, x);
    if (x != x) return 0x7fc0;
    return (uint16_t)((u + 0x7fffu + ((u >> 16) & 1u)) >> 16);
}

struct AppendArgs {
    uint16_t* query;
    const uint16_t* query_src;
    const uint16_t* key_new;
    const uint16_t* value_new;
    uint16_t* key_slot;    // cache address of (layer, pos, kv_head 0)
    uint16_t* value_slot;
    const uint16_t* weight;
    const float* sin_row;
    const float* cos_row;
    int64_t slot_head_stride;  // elements between KV heads inside the slot
    int32_t head_num;
    int32_t n_kv;
    float eps;
};

__global__ __launch_bounds__(kHalf) void qk_norm_rope_append_kernel(AppendArgs a) {
    const int b = blockIdx.x;
    const int i = threadIdx.x;
    if (b >= a.head_num + a.n_kv) {
        // V row: plain copy into the slot, 4 bytes per lane.
        const int kh = b - a.head_num - a.n_kv;
        const uint32_t* src = reinterpret_cast<const uint32_t*>(a.value_new + kh * kHeadDim);
        uint32_t* dst = reinterpret_cast<uint32_t*>(a.value_slot + kh * a.slot_head_stride);
        dst[i] = src[i];
        return;
    }
    const uint16_t* src;
    uint16_t* dst;
    const uint16_t* w;
    if (b < a.head_num) {
        src = a.query_src + b * kHeadDim;
        dst = a.query + b * kHeadDim;
        w = a.weight;
    } else {
        const int kh = b - a.head_num;
        src = a.key_new + kh * kHeadDim;
        dst = a.key_slot + kh * a.slot_head_stride;
        w = a.weight + kHeadDim;
    }
    const float x0 = bf16_to_f32(src[i]);
    const float x1 = bf16_to_f32(src[i + kHalf]);
    float ss = x0 * x0 + x1 * x1;
    ss = wave_sum(ss);
    const float r = 1.0f / sqrtf(ss / (float)kHeadDim + a.eps);
    const float av = x0 * bf16_to_f32(w[i]) * r;
    const float bv = x1 * bf16_to_f32(w[i + kHalf]) * r;
    const float sn = a.sin_row[i];
    const float cs = a.cos_row[i];
    dst[i] = f32_to_bf16(av * cs - bv * sn);
    dst[i + kHalf] = f32_to_bf16(av * sn + bv * cs);
}

__global__ void sincos_table_kernel(float* __restrict__ sin_cache, float* __restrict__ cos_cache, int32_t half,
                                    int64_t total, float inv_head_dim, float ln_base) {
    const int64_t idx = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (idx >= total) return;
    const int32_t i = (int32_t)(idx % half);
    const int32_t pos = (int32_t)(idx / half);
    // Same expression as the reference's host table (cpu/rope_kernel.cpp:12):
    // the exponent is formed in double and the frequency stored as float.
    const float freq = (float)exp(-2.0 * i * (double)inv_head_dim * (double)ln_base);
    const float theta = (float)pos * freq;
    float s, c;
    sincosf(theta, &s, &c);
    sin_cache[idx] = s;
    cos_cache[idx] = c;
}

// Memory-bound, reading and writing in equal parts: 16 head rows (256 bytes each) per workgroup, contiguous in the source, a
// 16-byte chunk per thread, both ways past the caches (each byte is touched once). K and V, 8 KV heads, cached accesses and a 64-bit
// division for each of layer, position and head : this, us: 36 layers of 3777 positions 184.5 : 177.7 (6.3 TB/s; a copy by torch of the
// same bytes 207), 8 of 12000 135.6 : 128.7, 28 of 500 23.7 : 23.0, 60 of 100 14.6 : 12.8; a first pass on new buffers 223 : 191 and
// 169 : 142. Where both caches fit the 256 MB memory-side cache a conversion of the same buffers over again is slower for going past it (36 layers of 1000
// 21.9 : 24.1, 28 of 2000 32.8 : 36.7, 28 of 500 level) and so is a reader of the result right behind it (copy included, 36 of 1000 49 : 53, but 28 of 2000 92 : 79); with the
// source just written it is faster (30 : 23, 50 : 34). A prompt is converted once, out of buffers that its prefill wrote. Cached reads with such stores 180 (first pass 230); two, four and eight chunks per thread 181, 187 and 280; positions of one KV
// head per workgroup (whole runs on the writing side) 184 ... 215.
constexpr int kRestrideThreads = 256;
__global__ __launch_bounds__(kRestrideThreads) void kv_restride_kernel(const uint4* __restrict__ src, uint4* __restrict__ dst,
                                                                       int32_t max_seq_len, int32_t n_kv, int32_t num_pos, int32_t layers) {
    typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
    const uint32_t row = blockIdx.x * (kRestrideThreads / 16) + (threadIdx.x >> 4);
    const uint32_t t = row / (uint32_t)n_kv, kh = row - t * (uint32_t)n_kv;
    if (t >= (uint32_t)num_pos) return;
    const int c = (int)(threadIdx.x & 15);
    const int64_t layer_chunks = (int64_t)max_seq_len * n_kv * 16;
    const int64_t from = (int64_t)row * 16 + c, to = ((int64_t)kh * max_seq_len + t) * 16 + c;
    for (int64_t layer = blockIdx.y; layer < layers; layer += gridDim.y) {
        const u32x4 v = __builtin_nontemporal_load(reinterpret_cast<const u32x4*>(src) + layer * layer_chunks + from);
        __builtin_nontemporal_store(v, reinterpret_cast<u32x4*>(dst) + layer * layer_chunks + to);
    }
}

}  // namespace

int launch_qk_norm_rope_append(const llmi_qk_norm_rope_args& args) {
    const int n_kv = args.kv_dim / args.head_dim;
    const int64_t layer_off = (int64_t)args.layer_id * args.max_seq_len * args.kv_dim;
    int64_t slot_off, slot_head_stride;
    if (args.kv_layout == LLMI_KV_LAYOUT_POS_MAJOR) {
        slot_off = layer_off + (int64_t)args.pos * args.kv_dim;
        slot_head_stride = args.head_dim;
    } else {
        slot_off = layer_off + (int64_t)args.pos * args.head_dim;
        slot_head_stride = (int64_t)args.max_seq_len * args.head_dim;
    }
    AppendArgs a;
    a.query = static_cast<uint16_t*>(args.query);
    a.query_src = args.query_src ? static_cast<const uint16_t*>(args.query_src) : a.query;
    a.key_new = static_cast<const uint16_t*>(args.key_new);
    a.value_new = static_cast<const uint16_t*>(args.value_new);
    a.key_slot = static_cast<uint16_t*>(args.key_cache) + slot_off;
    a.value_slot = args.value_cache ? static_cast<uint16_t*>(args.value_cache) + slot_off : nullptr;
    a.weight = static_cast<const uint16_t*>(args.norm_weight);
    a.sin_row = args.sin_cache + (int64_t)args.pos * (args.head_dim / 2);
    a.cos_row = args.cos_cache + (int64_t)args.pos * (args.head_dim / 2);
    a.slot_head_stride = slot_head_stride;
    a.head_num = args.head_num;
    a.n_kv = n_kv;
    a.eps = args.eps;
    const int blocks = args.head_num + n_kv + (args.value_new ? n_kv : 0);
    hipLaunchKernelGGL(qk_norm_rope_append_kernel, dim3(blocks), dim3(kHalf), 0,
                       static_cast<hipStream_t>(args.stream), a);
    return check_launch();
}

int launch_sincos_table(float* sin_cache, float* cos_cache, int32_t head_dim, int32_t max_seq_len,
                        hipStream_t stream) {
    const int32_t half = head_dim / 2;
    const int64_t total = (int64_t)half * max_seq_len;
    const int threads = 256;
    const int64_t blocks = (total + threads - 1) / threads;
    hipLaunchKernelGGL(sincos_table_kernel, dim3((unsigned)blocks), dim3(threads), 0, stream, sin_cache, cos_cache,
                       half, total, 1.0f / (float)head_dim, logf(1000000.0f));
    return check_launch();
}

int launch_kv_restride(const void* src, void* dst, int32_t layer_num, int32_t max_seq_len, int32_t kv_dim,
                       int32_t head_dim, int32_t num_pos, hipStream_t stream) {
    const int n_kv = kv_dim / head_dim;
    if (layer_num == 0 || num_pos == 0) return LLMI_OK;
    constexpr int rows = kRestrideThreads / 16;
    const int64_t blocks = ((int64_t)num_pos * n_kv + rows - 1) / rows;
    const dim3 grid((unsigned)blocks, (unsigned)(layer_num < 65535 ? layer_num : 65535));
    hipLaunchKernelGGL(kv_restride_kernel, grid, dim3(kRestrideThreads), 0, stream, static_cast<const uint4*>(src), static_cast<uint4*>(dst),
                       max_seq_len, n_kv, num_pos, layer_num);
    return check_launch();
}

}  // namespace llmi
