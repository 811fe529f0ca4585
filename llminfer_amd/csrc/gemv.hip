// The bf16 GEMVs that sit either side of decode attention in the layer loop, on
// gfx950: the packed QKV projection that produces the new token's raw q/k/v rows
// (role of fused_qkv_gemv_bf16x8_kernel, code/source/op/kernel/cuda/matmul_kernel.cu:211-246),
// the plain projection with bf16 or fp32 output (gemv_bf16x8_{bf16,fp32}_kernel, :38-98)
// and the output projection with the residual add folded in
// (fused_gemv_add_bf16x8_kernel, :143-172).
//
// HBM-bound weight streams: every weight byte is read once, with non-temporal 16-byte loads, one row per wavefront
// (64 lanes x 8 bf16 per step of 512 elements). A kernel per step count up to 20, unrolled: rows of up to 8 steps are asked for at once,
// in longer ones the weights and the input run a window of steps ahead of the sum, each request taking the place of a step that has
// been added; six steps, but where launch_rows says otherwise. Longer rows keep the window in a ring. (In batches of four steps, each waited for, a row of 5120 was four trips to memory.) Graph replays over distinct
// matrices, batches of four : the window, us and TB/s of the latter:
//   6144 x 2560    6.95 : 6.65 (4.7)      2560 x 4096   5.17 : 5.16 (4.1)     10240 x 5120   17.7 : 16.6 (6.3)
//   5120 x 8192    15.5 : 14.9 (5.6)      2560 x 9728   9.58 : 9.13 (5.5)    152000 x 2560  110.1 : 109.0 (7.1)
// That is the stream: the bytes at 7.1 TB/s and 1.7 us for the launch, within a tenth. Measured and not taken: whole rows of ten
// steps and more at once, weights ahead of the input 18.9 at 10240 x 5120 and the input ahead of the weights 18.4 (the order of the
// requests counts: side by side is best); windows of 3, 4, 5 and 8 (level to 4 % slower); two or four rows per wavefront (level to
// 5 % slower); workgroups that stay and walk the rows (4-12 % slower); fewer of them in flight by LDS (level). K split
// over the wavefronts of a workgroup is level, 3 % faster at 8192, 3 % slower at 9728. Products are formed in fp32 by
// v_dot2_f32_bf16 (two bf16 pairs per instruction, fp32 accumulate), the 64 lanes fold with DPP row steps and four scalar
// reads, lane 0 rounds once and writes. All forms add a lane's steps in the same order: the same bits.

#include <hip/hip_runtime.h>
#include <stdint.h>

#include "llmi_internal.h"
#include "wave_ops.h"

namespace llmi {
namespace {

typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));

constexpr int kMaxSteps = 20;  // longest row, in steps, with a kernel of its own
constexpr int kWindow = 6;     // steps ahead in longer rows than 8 steps, unless launch_rows says otherwise

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

// Rows of (S - 1, S] steps, W wavefronts per workgroup: WINDOW steps (weights and input) ahead of the one being added.
template <int S, int W, int WINDOW>
__global__ __launch_bounds__(W * 64) void gemv_row_kernel(GemvArgs a) {
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int row = blockIdx.x * W + wave;
    if (row >= a.n) return;
    const u32x4* x4 = reinterpret_cast<const u32x4*>(a.x) + lane;
    const u32x4* w4 = reinterpret_cast<const u32x4*>(a.w) + (int64_t)row * a.k8 + lane;
    constexpr int kAhead = S <= WINDOW + 2 ? S : WINDOW;
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

// More than two and up to five workgroups of two rows on each of 256 compute units is where the window gains least, and where rows start
// a multiple of 4 KiB apart it loses: k a multiple of 2048, at which batches of four have no remainder. us, batches of four : windows
// of 4 : 6 : 10:
//   1000 x 6144  4.27 : 4.05 : 3.89 : 3.93    1000 x 8192   4.92 : 4.65 : 4.43 : 4.70    1000 x 10240  5.61 : 5.23 : 5.12 : 5.26
//   1500 x 6144  4.69 : 4.65 : 4.86 : 4.70    1500 x 10240  6.35 : 6.29 : 6.45 : 6.52    1500 x 7000   5.82 : 5.23 : 5.36 : 5.40
//   2560 x 6144  6.49 : 6.71 : 6.69 : 6.52    2560 x 10240  9.56 : 10.03 : 9.73 : 9.49   2560 x 12288 (ring) 10.8 : - : 11.5
//   2600 x 6144, of the batches' time, 0.94 : 0.92 : 0.88     4000 x 10240  14.5 : 13.9 : 13.6 : 13.6
// So batches there, but for sixteen steps up to 2048 rows, where six ahead is level or better (1500 x 8192 5.80 : 5.71 : 5.66 : 5.73, but 2300 x
// 8192, of the batches' time, 1.05 : 1.03 : 1.02). With three wavefronts on a SIMD (from 2049 rows on) the other lengths want ten steps ahead: 2560 x 8704 8.84 : 8.92 :
// 8.99 : 8.55, 2300 x 9728, of the batches' time, 1.00 : 0.97 : 0.94.
constexpr int kRowsOfTwo = 1024, kRowsOfFour = 2048, kRowsOfFive = 2560;
// Eight steps, otherwise asked for at once (71 registers: a wavefront less per SIMD than the window of four's 44), are a window of four where
// rows start 4 KiB apart and are many. Batches : window of 4 : at once, us: 151936 x 4096 175.3 : 174.7 : 178.2, 60000 rows 69.9 : 69.6 : 70.7,
// 20000 25.1 : 24.9 : 24.8.
constexpr int kManyRows = 24576;

// Rows of whole batches of four steps, each batch waited for before the next is asked for (when: see launch_rows).
__global__ __launch_bounds__(2 * 64) void gemv_batch_kernel(GemvArgs a) {
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int row = blockIdx.x * 2 + wave;
    if (row >= a.n) return;
    const u32x4* x4 = reinterpret_cast<const u32x4*>(a.x);
    const u32x4* w4 = reinterpret_cast<const u32x4*>(a.w) + (int64_t)row * a.k8;
    float acc = 0.0f;
    for (int c = lane; c < a.k8; c += 64 * 4) {
        u32x4 xv[4], wv[4];
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            xv[u] = x4[c + 64 * u];
            wv[u] = __builtin_nontemporal_load(w4 + c + 64 * u);
        }
#pragma unroll
        for (int u = 0; u < 4; ++u) acc = dot8_bf16(xv[u], wv[u], acc);
    }
    acc = wave_sum(acc);
    if (lane == 0) write_row(a, row, acc);
}

template <int S, int W, int WINDOW>
void launch_row_kernel(const GemvArgs& a, hipStream_t stream) {
    hipLaunchKernelGGL((gemv_row_kernel<S, W, WINDOW>), dim3((a.n + W - 1) / W), dim3(W * 64), 0, stream, a);
}

#define LLMI_GEMV_STEPS(S, WINDOW) \
    case S: return launch_row_kernel<S, W, WINDOW>(a, stream);

template <int W>
void launch_rows(const GemvArgs& a, hipStream_t stream) {
    const int steps = (a.k8 + 63) / 64;
    const bool apart_4k = a.k8 % 256 == 0;
    if constexpr (W == 2) {
        if (apart_4k && steps > 8 && a.n > kRowsOfTwo && a.n <= kRowsOfFive && !(steps == 16 && a.n <= kRowsOfFour)) {
            hipLaunchKernelGGL(gemv_batch_kernel, dim3((a.n + 1) / 2), dim3(2 * 64), 0, stream, a);
            return;
        }
        if (a.n > kRowsOfFour && a.n <= kRowsOfFive) {
            switch (steps) {
                LLMI_GEMV_STEPS(9, 10) LLMI_GEMV_STEPS(10, 10) LLMI_GEMV_STEPS(11, 10) LLMI_GEMV_STEPS(12, 10) LLMI_GEMV_STEPS(13, 10)
                LLMI_GEMV_STEPS(14, 10) LLMI_GEMV_STEPS(15, 10) LLMI_GEMV_STEPS(16, 10) LLMI_GEMV_STEPS(17, 10) LLMI_GEMV_STEPS(18, 10)
                LLMI_GEMV_STEPS(19, 10) LLMI_GEMV_STEPS(20, 10)
            }
        }
    } else if (apart_4k && steps == 8 && a.n >= kManyRows) {
        return launch_row_kernel<8, W, 4>(a, stream);
    }
    switch (steps) {
        LLMI_GEMV_STEPS(1, kWindow) LLMI_GEMV_STEPS(2, kWindow) LLMI_GEMV_STEPS(3, kWindow) LLMI_GEMV_STEPS(4, kWindow)
        LLMI_GEMV_STEPS(5, kWindow) LLMI_GEMV_STEPS(6, kWindow) LLMI_GEMV_STEPS(7, kWindow) LLMI_GEMV_STEPS(8, kWindow)
        LLMI_GEMV_STEPS(9, kWindow) LLMI_GEMV_STEPS(10, kWindow) LLMI_GEMV_STEPS(11, kWindow) LLMI_GEMV_STEPS(12, kWindow)
        LLMI_GEMV_STEPS(13, kWindow) LLMI_GEMV_STEPS(14, kWindow) LLMI_GEMV_STEPS(15, kWindow) LLMI_GEMV_STEPS(16, kWindow)
        LLMI_GEMV_STEPS(17, kWindow) LLMI_GEMV_STEPS(18, kWindow) LLMI_GEMV_STEPS(19, kWindow) LLMI_GEMV_STEPS(20, kWindow)
        default: hipLaunchKernelGGL((gemv_long_row_kernel<W>), dim3((a.n + W - 1) / W), dim3(W * 64), 0, stream, a);
    }
}
#undef LLMI_GEMV_STEPS

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
