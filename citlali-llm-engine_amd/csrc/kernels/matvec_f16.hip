// matvec_f16.hip -- GEMV over fp16 weight rows (kernels.cu:27-35, 381-412 of
// the reference) of the lengths that the streaming kernels of
// matvec_kquant.hip have no instantiation for.  Products and sums in fp32
// (v_dot2_f32_f16), fp16 outputs rounded nearest-even.
//
// gfx950 design of the ring kernel (multiples of 8)
//  * A wave takes one row at a time and copies it 1 KB per instruction (512
//    values, lane l the 16 bytes at 16 l of the step), whole cache lines,
//    nontemporal, into four LDS slots of its own, the ring running on over the
//    wave's rows.  (A ring of registers had its waits merged at the loop edge:
//    every turn drained it.)
//  * x is staged in LDS in its own order, padded with zeros to whole steps;
//    in a partial last step the lanes past the row end re-read its last
//    values and count them as zero.
//  * A row's sum: per lane short fp32 chains (see one_chain), then the wave sum.
// Bound by HBM.  Against the walk over 256-value blocks of four rows that
// served these lengths before (us, rotated weights): 5120 x 17408 39.5 -> 28.8
// (6.2 TB/s), 18944 x 3584 25.5 -> 22.1, 300 x 19968 16.3 -> 10.1.  The
// streaming kernels' own lengths stay with them: large matrices would gain
// (100000 x 2560 with the norm 85 -> 77), short launches lose (4096 x 4096 6.9
// -> 7.5, grouped q/k/v 6144 x 2560 7.1 -> 7.8), and all launch forms of a
// length have to give the same bits.
#include <algorithm>

#include "citlali_hip.h"
#include "device_common.hpp"
#include "launch.hpp"

namespace citlali::hip {
namespace {

constexpr int kBlock = 256;
constexpr int kWaves = kBlock / kWave;
constexpr int kStepValues = kWave * 8;
constexpr int kStepBytes = kStepValues * 2;
constexpr int kDepth = 4;   // steps in flight per wave; eight measured no faster
constexpr int kFlush = 4;   // steps between additions to a lane's total

__host__ __device__ constexpr int steps_of(int K) { return (K + kStepValues - 1) / kStepValues; }
constexpr int lds_bytes(int K) { return (steps_of(K) + kWaves * kDepth) * kStepBytes; }

// One wave per row, x and the row straight into registers: K not a multiple of
// 8 or longer than the ring kernel stages, and launches too small for it.
template <bool kF32>
__global__ __launch_bounds__(kBlock) void matvec_f16_kernel(const uint16_t* __restrict__ w,
                                                          const uint16_t* __restrict__ x, void* __restrict__ y,
                                                          int K, int N) {
    const int lane = threadIdx.x & (kWave - 1);
    const int row = blockIdx.x * (kBlock / kWave) + threadIdx.x / kWave;
    if (row >= N) return;
    const uint16_t* r = w + (size_t)row * K;
    float a = 0.f;
    if ((K & 7) == 0) {
        for (int k = lane * 8; k < K; k += kWave * 8) {
            const u32x4 wv = *reinterpret_cast<const u32x4*>(r + k);
            const u32x4 xv = *reinterpret_cast<const u32x4*>(x + k);
            a = dot2(wv.x, xv.x, a);
            a = dot2(wv.y, xv.y, a);
            a = dot2(wv.z, xv.z, a);
            a = dot2(wv.w, xv.w, a);
        }
    } else {
        for (int k = lane; k < K; k += kWave) a = fmaf(h2f(r[k]), h2f(x[k]), a);
    }
    a = wave_sum(a);
    if (lane == 0) {
        if constexpr (kF32) static_cast<float*>(y)[row] = a;
        else static_cast<uint16_t*>(y)[row] = f2h_rne(a);
    }
}

// A lane's sums run as one chain over its words in order (the order of
// matvec_f16_kernel, so the two give the same bits), or, for long rows of whole
// blocks, as four, one per weight word, that are added to a total every kFlush
// steps, with what the addition rounds off kept beside it (Knuth's two-sum):
// chains over the whole row were up to 1.3 times further from 64-bit sums than
// the walk over 256-value blocks that served these lengths before.
__host__ __device__ constexpr bool one_chain(int K) { return K % 256 != 0 || K <= 1536; }

template <bool kF32, bool kOneChain>
__global__ __launch_bounds__(kBlock, 2) void f16_rows_kernel(const uint16_t* __restrict__ w,
                                                             const uint16_t* __restrict__ x, void* __restrict__ y,
                                                             int K, int n) {
    extern __shared__ __align__(16) uint8_t smem[];
    const int tid = (int)threadIdx.x, lane = tid & (kWave - 1);
    const int wave = __builtin_amdgcn_readfirstlane(tid / kWave);
    const int T = steps_of(K);
    const bool ragged = K % kStepValues != 0;
    const int lane_at = lane * 16, last_at = K * 2 - 16;
    const int first = blockIdx.x * kWaves + wave, stride = gridDim.x * kWaves;
    int my_rows = 0;
    for (int r = first; r < n; r += stride) ++my_rows;
    const int S = my_rows * T;   // steps of this wave

    // x, then the first steps.  These copies are unconditional (a wave without
    // rows copies the last one), so the number behind x's is known.
    const int runs = K >> 3;
    for (int r0 = wave * kWave; r0 < runs; r0 += kBlock)
        if (r0 + lane < runs) copy16_to_lds(reinterpret_cast<const uint8_t*>(x) + (size_t)(r0 + lane) * 16, smem + r0 * 16);
    for (int i = runs + tid; i < T * kWave; i += kBlock) reinterpret_cast<u32x4*>(smem)[i] = u32x4{0u, 0u, 0u, 0u};
    uint8_t* ring = smem + (T + wave * kDepth) * kStepBytes;
    int head = first, ht = 0;   // row and step of the next copy
    const uint8_t* base = reinterpret_cast<const uint8_t*>(w + (size_t)min(head, n - 1) * K);
    auto copy = [&](int slot) {
        copy16_to_lds<true>(base + (uint32_t)min(ht * kStepBytes + lane_at, last_at), ring + slot * kStepBytes);
        if (++ht == T) {   // wave-uniform
            ht = 0;
            head += stride;
            base = reinterpret_cast<const uint8_t*>(w + (size_t)min(head, n - 1) * K);
        }
    };
#pragma unroll
    for (int d = 0; d < kDepth; ++d) copy(d);
    wait_vm<kDepth>();   // x is in LDS
    lds_only_barrier();

    float a0 = 0.f, a1 = 0.f, a2 = 0.f, a3 = 0.f, total = 0.f, lost = 0.f;
    int row = first, t = 0, slot = 0, issued = kDepth;
    for (int c = 0; c < S; ++c) {
        const int later = issued - c - 1;   // steps in flight behind this one
        if (later >= 3) wait_vm<3>();
        else if (later == 2) wait_vm<2>();
        else if (later == 1) wait_vm<1>();
        else wait_vm<0>();
        u32x4 b = *reinterpret_cast<const u32x4*>(ring + slot * kStepBytes + lane_at);
        const u32x4 xv = *reinterpret_cast<const u32x4*>(smem + t * kStepBytes + lane_at);
        wait_lds();
        __builtin_amdgcn_sched_barrier(0);
        if (issued < S) {   // the slot is read: refill it
            copy(slot);
            ++issued;
        }
        __builtin_amdgcn_sched_barrier(0);
        slot = (slot + 1) & (kDepth - 1);
        if (ragged && t == T - 1) {   // wave-uniform
            const uint32_t keep = t * kStepBytes + lane_at <= last_at ? 0xffffffffu : 0u;
            b = b & u32x4{keep, keep, keep, keep};
        }
        if constexpr (kOneChain) {
            a0 = dot2(b.w, xv.w, dot2(b.z, xv.z, dot2(b.y, xv.y, dot2(b.x, xv.x, a0))));
        } else {
            a0 = dot2(b.x, xv.x, a0);
            a1 = dot2(b.y, xv.y, a1);
            a2 = dot2(b.z, xv.z, a2);
            a3 = dot2(b.w, xv.w, a3);
        }
        ++t;
        if (!kOneChain && (t % kFlush == 0 || t == T)) {   // wave-uniform
            const float p = (a0 + a1) + (a2 + a3), sum = total + p, z = sum - total;
            lost += (total - (sum - z)) + (p - z);
            total = sum;
            a0 = a1 = a2 = a3 = 0.f;
        }
        if (t == T) {   // wave-uniform
            // (an infinite total stays what it is)
            const float s = wave_sum(kOneChain ? a0 : fabsf(lost) < INFINITY ? total + lost : total);
            if (lane == 0) {
                if constexpr (kF32) static_cast<float*>(y)[row] = s;
                else static_cast<uint16_t*>(y)[row] = f2h_rne(s);
            }
            a0 = total = lost = 0.f;
            t = 0;
            row += stride;
        }
    }
    wait_vm<0>();   // no copy outlives the workgroup's LDS
}

template <bool kF32, bool kOneChain>
hipError_t launch_ring(const uint16_t* w, const uint16_t* x, void* y, int K, int n, hipStream_t s) {
    // three workgroups per CU where their LDS fits (5120 x 17408: 30.1 us with
    // two, 28.8 with three, 31.5 with four)
    const int lds = lds_bytes(K), per_cu = std::max(1, std::min(3, 160 * 1024 / lds));
    const int grid = std::min((n + kWaves - 1) / kWaves, per_cu * device_cus());
    constexpr auto kernel = f16_rows_kernel<kF32, kOneChain>;
    const hipError_t e = allow_lds<kernel>(lds);
    if (e != hipSuccess) return e;
    launch_kernel(kernel, dim3(grid), dim3(kBlock), (size_t)lds, s, w, x, y, K, n);
    return hipGetLastError();
}

// Launches for which the ring kernel's set-up (x and zeros to LDS, the rings
// filled) costs more than it gains, among the one-chain lengths, where both
// kernels give the same bits.  us, wave per row / ring: 12000 x 8 3.0 / 4.1,
// 3584 x 200 2.8 / 3.9, 12000 x 200 4.3 / 4.5 (40000: 8.1 / 7.9), 3584 x 1000 3.8
// / 4.2 (12000: 6.8 / 6.6); longer rows, whose loads a wave waits for in turn,
// 200 x 1800 2.6 / 3.2 (1024: 4.3 / 3.4), 128 x 2504 2.6 / 3.4 (200: 3.9 / 3.4),
// 64 x 5000 3.1 / 4.1 (128: 6.1 / 4.1), 32 x 19000 6.5 / 8.6 (64: 19.6 / 8.5).
bool small_launch(int K, int n) {
    return one_chain(K) && ((long long)K * n < (K <= 1024 ? 8 << 20 : 480 << 10) || n <= (K <= 9216 ? 64 : 32));
}

template <bool kF32>
hipError_t launch(const uint16_t* w, const uint16_t* x, void* y, int K, int n, hipStream_t s) {
    if (K % 8 != 0 || K > CITLALI_MAX_IN_FEATURES || small_launch(K, n)) {
        launch_kernel(matvec_f16_kernel<kF32>, dim3((n + kWaves - 1) / kWaves), dim3(kBlock), 0, s, w, x, y, K, n);
        return hipGetLastError();
    }
    return one_chain(K) ? launch_ring<kF32, true>(w, x, y, K, n, s) : launch_ring<kF32, false>(w, x, y, K, n, s);
}

}  // namespace

hipError_t launch_matvec_f16_rows(const uint16_t* w, const uint16_t* x, void* y, bool f32_out, int K, int N,
                                  hipStream_t s) {
    return f32_out ? launch<true>(w, x, y, K, N, s) : launch<false>(w, x, y, K, N, s);
}

}  // namespace citlali::hip
