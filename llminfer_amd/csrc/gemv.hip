// The bf16 GEMVs that sit either side of decode attention in the layer loop, on
// gfx950: the packed QKV projection that produces the new token's raw q/k/v rows
// (role of fused_qkv_gemv_bf16x8_kernel, code/source/op/kernel/cuda/matmul_kernel.cu:211-246),
// the plain projection with bf16 or fp32 output (gemv_bf16x8_{bf16,fp32}_kernel, :38-98)
// and the output projection with the residual add folded in
// (fused_gemv_add_bf16x8_kernel, :143-172).
//
// HBM-bound weight streams: every weight byte is read once, with non-temporal 16-byte loads, one row per wavefront
// (64 lanes x 8 bf16 per step of 512 elements). A kernel per step count, unrolled: rows of up to 8 steps are asked for at once,
// in longer ones the weights and the input run six steps ahead of the sum, each request taking the place of a step that has
// been added. (In batches of four steps, each waited for, a row of 5120 was four trips to memory.) Graph replays over distinct
// matrices, batches of four : the window, us and TB/s of the latter:
//   6144 x 2560    6.95 : 6.65 (4.7)      2560 x 4096   5.17 : 5.16 (4.1)     10240 x 5120   17.7 : 16.6 (6.3)
//   5120 x 8192    15.5 : 14.9 (5.6)      2560 x 9728   9.58 : 9.13 (5.5)    152000 x 2560  110.1 : 109.0 (7.1)
// That is the stream: the bytes at 7.1 TB/s and 1.7 us for the launch, within a tenth. Measured and not taken: whole rows of ten
// steps and more at once, weights ahead of the input 18.9 at 10240 x 5120 and the input ahead of the weights 18.4 (the order of the
// requests counts: side by side is best); windows of 3, 4, 5 and 8 (level to 4 % slower); two or four rows per wavefront (level to
// 5 % slower); workgroups that stay and walk the rows (4-12 % slower); fewer of them in flight by LDS (level). K split
// over the wavefronts of a workgroup is level, 3 % faster at 8192, 3 % slower at 9728. Products are formed in fp32 by
// v_dot2_f32_bf16 (two bf16 pairs per instruction, fp32 accumulate), the 64 lanes fold with DPP row steps and four scalar
// reads, lane 0 rounds once and writes.

#include <hip/hip_runtime.h>
#include <stdint.h>

#include "llmi_internal.h"
#include "wave_ops.h"

namespace llmi {
namespace {

typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));

constexpr int kMaxSteps = 20;  // longest row, in steps, with a kernel of its own
constexpr int kWindow = 6;     // steps ahead in longer rows than 8 steps

__device__ __forceinline__ float bf16_to_f32(uint16_t h) { return __builtin_bit_cast(float, (uint32_t)h << 16); }

__device__ __forceinline__ uint16_t f32_to_bf16(float x) {
    uint32_t u = __builtin_bit_cast(uint32_t, x);
    if (x != x) return 0x7fc0;
    return (uint16_t)((u + 0x7fffu + ((u >> 16) & 1u)) >> 16);
}

struct GemvArgs {
    const uint16_t* x;   // [k]
    const uint16_t* w;   // [n][k]
    void* out[3];        // row segments (one for the plain GEMV, query/key/value for the packed one)
    int32_t seg_end[3];  // exclusive end row of each segment
    int32_t n;
    int32_t k8;          // k / 8
    int32_t mode;        // LLMI_GEMV_*
};

__device__ __forceinline__ void write_row(const GemvArgs& a, int row, float sum) {
    const int seg = row < a.seg_end[0] ? 0 : (row < a.seg_end[1] ? 1 : 2);
    const int local = row - (seg == 0 ? 0 : a.seg_end[seg - 1]);
    if (a.mode == LLMI_GEMV_OUT_F32) {
        static_cast<float*>(a.out[seg])[local] = sum;
    } else {
        uint16_t* o = static_cast<uint16_t*>(a.out[seg]) + local;
        if (a.mode == LLMI_GEMV_ADD_BF16) sum += bf16_to_f32(*o);  // fp32 + fp32 -> bf16 (:169-170)
        *o = f32_to_bf16(sum);
    }
}

// Rows of (S - 1, S] steps, W wavefronts per workgroup: kWindow steps (weights and input) ahead of the one being added.
template <int S, int W>
__global__ __launch_bounds__(W * 64) void gemv_row_kernel(GemvArgs a) {
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int row = blockIdx.x * W + wave;
    if (row >= a.n) return;
    const u32x4* x4 = reinterpret_cast<const u32x4*>(a.x) + lane;
    const u32x4* w4 = reinterpret_cast<const u32x4*>(a.w) + (int64_t)row * a.k8 + lane;
    constexpr int kAhead = S <= kWindow + 2 ? S : kWindow;
    u32x4 wv[S], xv[S];
    auto request = [&](int s) {
        xv[s] = wv[s] = u32x4{0u, 0u, 0u, 0u};
        if (s < S - 1 || lane + 64 * (S - 1) < a.k8) {  // (the last step may be a part of one)
            xv[s] = x4[64 * s];
            wv[s] = __builtin_nontemporal_load(w4 + 64 * s);
        }
    };
    float acc = 0.0f;
    // (the empty asm statements keep the requests in this order and where they are)
#pragma unroll
    for (int s = 0; s < kAhead; ++s) {
        request(s);
        asm volatile("" ::: "memory");
    }
#pragma unroll
    for (int s = 0; s < S; ++s) {
        acc = dot8_bf16(xv[s], wv[s], acc);
        if (s + kAhead < S) {
            asm volatile("" : "+v"(acc)::"memory");
            request(s + kAhead);
            asm volatile("" ::: "memory");
        }
    }
    acc = wave_sum(acc);
    if (lane == 0) write_row(a, row, acc);
}

// Longer rows, of any step count: the same window, its steps in a ring of registers. Graph replays over distinct matrices, batches
// of four steps (each waited for) : twenty at a time and the rest one by one : the ring, us and TB/s of the latter:
//   2560 x 12288   11.3 : 13.1 : 11.4 (5.5)   5120 x 13824   24.8 : 25.5 : 23.0 (6.2)   5120 x 17408  30.6 : 32.2 : 29.4 (6.1)
//   5120 x 25600   44.1 : 46.1 : 41.7 (6.3)   8192 x 28672   73.6 : 82.5 : 70.0 (6.7)   1000 x 11008  7.39 : 7.73 : 6.20 (3.6)
//   500 x 53248    18.8 : 20.7 : 12.8 (4.2)   16384 x 16384  82.7 : 84.5 : 80.4 (6.7)
template <int W>
__global__ __launch_bounds__(W * 64) void gemv_long_row_kernel(GemvArgs a) {
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int row = blockIdx.x * W + wave;
    if (row >= a.n) return;
    const u32x4* x4 = reinterpret_cast<const u32x4*>(a.x) + lane;
    const u32x4* w4 = reinterpret_cast<const u32x4*>(a.w) + (int64_t)row * a.k8 + lane;
    const int whole = a.k8 >> 6;  // steps all lanes have (kMaxSteps or more)
    u32x4 wv[kWindow], xv[kWindow];
    auto request = [&](int u) {  // (the first of the steps not asked for yet, into place u)
        xv[u] = *x4;
        wv[u] = __builtin_nontemporal_load(w4);
        x4 += 64;
        w4 += 64;
    };
    float acc = 0.0f;
#pragma unroll
    for (int u = 0; u < kWindow; ++u) {
        request(u);
        asm volatile("" ::: "memory");
    }
    int asked = kWindow;
    for (; asked + kWindow <= whole; asked += kWindow) {
#pragma unroll
        for (int u = 0; u < kWindow; ++u) {
            acc = dot8_bf16(xv[u], wv[u], acc);
            asm volatile("" : "+v"(acc)::"memory");
            request(u);
            asm volatile("" ::: "memory");
        }
    }
    // What is left to ask for: fewer whole steps than places, and a part of one.
    const int left = whole - asked;
    const bool part = lane < (a.k8 & 63);
#pragma unroll
    for (int u = 0; u < kWindow; ++u) {
        acc = dot8_bf16(xv[u], wv[u], acc);
        asm volatile("" : "+v"(acc)::"memory");
        xv[u] = wv[u] = u32x4{0u, 0u, 0u, 0u};
        if (u < left || (u == left && part)) request(u);
        asm volatile("" ::: "memory");
    }
#pragma unroll
    for (int u = 0; u < kWindow; ++u) acc = dot8_bf16(xv[u], wv[u], acc);
    acc = wave_sum(acc);
    if (lane == 0) write_row(a, row, acc);
}

// Four wavefronts per workgroup where there are six rows or more for each of the chip's 1024 SIMDs (half the workgroup
// starts), two below (a row's wavefront leaves as soon as it is done). Two : four wavefronts, us: 16.56 : 16.25 at 10240 x 5120,
// 109.9 : 109.5 at 152000 x 2560, level at 6144 x 2560; 4.83 : 5.09 at 2560 x 4096, 9.13 : 9.54 at 2560 x 9728, 14.0 : 14.3 at 5120 x 8192.
constexpr int kRowsForFour = 6144;

template <int W>
void launch_rows(const GemvArgs& a, hipStream_t stream) {
    const dim3 grid((a.n + W - 1) / W), block(W * 64);
    switch ((a.k8 + 63) / 64) {
#define LLMI_GEMV_STEPS(S) \
    case S: hipLaunchKernelGGL((gemv_row_kernel<S, W>), grid, block, 0, stream, a); break;
        LLMI_GEMV_STEPS(1) LLMI_GEMV_STEPS(2) LLMI_GEMV_STEPS(3) LLMI_GEMV_STEPS(4) LLMI_GEMV_STEPS(5)
        LLMI_GEMV_STEPS(6) LLMI_GEMV_STEPS(7) LLMI_GEMV_STEPS(8) LLMI_GEMV_STEPS(9) LLMI_GEMV_STEPS(10)
        LLMI_GEMV_STEPS(11) LLMI_GEMV_STEPS(12) LLMI_GEMV_STEPS(13) LLMI_GEMV_STEPS(14) LLMI_GEMV_STEPS(15)
        LLMI_GEMV_STEPS(16) LLMI_GEMV_STEPS(17) LLMI_GEMV_STEPS(18) LLMI_GEMV_STEPS(19) LLMI_GEMV_STEPS(20)
#undef LLMI_GEMV_STEPS
        default: hipLaunchKernelGGL((gemv_long_row_kernel<W>), grid, block, 0, stream, a);
    }
}

}  // namespace

int launch_gemv(const void* input, const void* weight, void* const out[3], const int32_t seg_end[3], int32_t n,
                int32_t k, int32_t mode, hipStream_t stream) {
    GemvArgs a;
    a.x = static_cast<const uint16_t*>(input);
    a.w = static_cast<const uint16_t*>(weight);
    for (int i = 0; i < 3; ++i) {
        a.out[i] = out[i];
        a.seg_end[i] = seg_end[i];
    }
    a.n = n;
    a.k8 = k / 8;
    a.mode = mode;
    if (n >= kRowsForFour) launch_rows<4>(a, stream);
    else launch_rows<2>(a, stream);
    return check_launch();
}

}  // namespace llmi
