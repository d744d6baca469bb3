// dequant.hip -- Q6_K embedding gather and whole-tensor Q4_K / Q6_K -> fp16.
//
// Values are the exact fp32 dequantised weights of kernels.cu:134-186
// (== weight_loader.cpp:147-323 before rounding).  The two entry points round
// them the way their reference counterparts do, and the reference is not
// consistent on exact ties:
//  * embed_q6k follows the reference kernel (kernels.cu:340-378), whose
//    store_half is __float2half: nearest-even.
//  * the whole-tensor dequant follows the host loader (dequant_q4_k /
//    dequant_q6_k with float_to_half_bits, dtype.cpp:136-176): nearest, ties
//    away from zero, so its output equals the host routines bit for bit.
#include "device_common.hpp"
#include "launch.hpp"

namespace citlali::hip {
namespace {

__device__ __forceinline__ float blk_half(const uint8_t* p) {
    return h2f((uint16_t)(p[0] | (p[1] << 8)));
}

// The host routines run on x86-64, where a NaN operand propagates with its
// sign (the first operand's when both are NaN) and an invalid operation
// (Inf * 0, Inf - Inf) yields the negative default NaN; the host fp16 rule
// then keeps that sign on the resulting infinity.  AMD hardware makes
// positive default NaNs, so NaN results get their host sign explicitly.
// (Only reachable when a block's d or dmin is Inf or NaN.)
__device__ __forceinline__ float host_nan(bool negative) {
    return __builtin_bit_cast(float, negative ? 0xffc00000u : 0x7fc00000u);
}

// element e of a Q4_K block (kernels.cu:209-230)
__device__ __forceinline__ float q4k_value(const uint8_t* blk, int e) {
    const int j = e >> 6, hi = (e & 63) >= 32;
    const int g = 2 * j + hi;
    const uint8_t* s = blk + 4;
    int sc, m;
    if (g < 4) {
        sc = s[g] & 63;
        m = s[g + 4] & 63;
    } else {
        sc = (s[g + 4] & 0x0f) | ((s[g - 4] >> 6) << 4);
        m = (s[g + 4] >> 4) | ((s[g] >> 6) << 4);
    }
    const uint8_t b = blk[16 + 32 * j + (e & 31)];
    const int q = hi ? (b >> 4) : (b & 0x0f);
    const float d = blk_half(blk), dmin = blk_half(blk + 2);
    const float v = d * (float)sc * (float)q - dmin * (float)m;
    if (!__builtin_isnan(v)) return v;
    // host order: (d*sc)*q - dmin*m
    if (__builtin_isnan(d)) return host_nan(__builtin_signbit(d));
    if (__builtin_isinf(d) && (sc == 0 || q == 0)) return host_nan(true);
    if (__builtin_isnan(dmin)) return host_nan(__builtin_signbit(dmin));
    return host_nan(true);   // dmin*0 with dmin = Inf, or Inf - Inf
}

// element e of a Q6_K block (kernels.cu:134-172)
__device__ __forceinline__ float q6k_value(const uint8_t* blk, int e) {
    const int h = e >> 7, part = (e & 127) >> 5, i = e & 31;
    const uint8_t lb = blk[64 * h + 32 * (part & 1) + i];
    const int lo = part < 2 ? (lb & 0x0f) : (lb >> 4);
    const int hi2 = (blk[128 + 32 * h + i] >> (2 * part)) & 3;
    const int q = (lo | (hi2 << 4)) - 32;
    const int8_t sc = (int8_t)blk[192 + 8 * h + i / 16 + 2 * part];
    const float d = blk_half(blk + 208);
    const float v = d * (float)sc * (float)q;
    if (!__builtin_isnan(v)) return v;
    return host_nan(__builtin_isnan(d) ? __builtin_signbit(d) : true);   // NaN d, or Inf * 0
}

// The token comes from `token_at` (device memory) when that is not null; a
// token there outside [0, vocab) yields a zero row instead of a read past
// the table (the host validates the scalar form).
__global__ void embed_q6k_kernel(const uint8_t* __restrict__ table, int32_t token_id,
                                 const int32_t* __restrict__ token_at, int vocab, uint16_t* __restrict__ out,
                                 int hidden) {
    const int idx = blockIdx.x * blockDim.x + threadIdx.x;
    if (idx >= hidden) return;
    if (token_at) {
        token_id = *token_at;
        if (token_id < 0 || token_id >= vocab) {
            out[idx] = 0;
            return;
        }
    }
    const size_t nb = (size_t)hidden / kQK;
    const uint8_t* row = table + (size_t)token_id * nb * kQ6KBytes;
    out[idx] = f2h_rne(q6k_value(row + (size_t)(idx / kQK) * kQ6KBytes, idx % kQK));
}

// Vectors at any byte alignment (gfx950 global loads and stores take
// unaligned addresses); `out` holds fp16 values, so 2 bytes there.
typedef u32x2 u32x2_a1 __attribute__((aligned(1)));
typedef u32x4 u32x4_a1 __attribute__((aligned(1)));

// Two dequantised values of magnitude below 65504 to fp16, the host rule
// (nearest, ties away from zero): half an fp16 ulp of the value's binade is
// added away from zero, then the conversion truncates.  The fp32 sum is exact
// within the binade, and above it only loses bits far below the fp16
// spacing, so the truncation sees the right side of every tie.  A value is a
// multiple of 2^-24 (fp16 scales times integers), so those below 2^-14 are
// fp16 numbers already and the truncation returns them.
__device__ __forceinline__ float add_half_ulp(float v) {
    const float binade = __builtin_bit_cast(float, __builtin_bit_cast(uint32_t, v) & 0xff800000u);   // with v's sign
    return fmaf(binade, 0x1p-11f, v);
}
__device__ __forceinline__ uint32_t f2h2_ties_away(float a, float b) {
    return __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_pkrtz(add_half_ulp(a), add_half_ulp(b)));
}

// Eight consecutive values of a block, value(code) of the codes in the bytes of
// c0, c1.
template <typename Value>
__device__ __forceinline__ void values_of_codes(uint32_t c0, uint32_t c1, Value value, float (&v)[8]) {
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        v[i] = value((float)((c0 >> (8 * i)) & 0xffu));
        v[4 + i] = value((float)((c1 >> (8 * i)) & 0xffu));
    }
}

// The share of a block that one thread dequantises, from wide loads that no
// other thread repeats: kRuns runs of eight values, run k being values
// first(r) + k * kApart .. + 7.  Q4_K: both nibbles of 8 quant bytes (two
// runs, 16 threads a block); Q6_K: the four parts of 8 positions (four runs,
// 8 threads a block).  load() is false when a value could leave the range of
// f2h2_ties_away: the scales bound every value, and an Inf or NaN scale fails
// the comparison.
struct DequantQ4K {
    static constexpr int kBytes = kQ4KBytes, kThreads = 16, kRuns = 2, kApart = 32;
    u32x2 w;
    float s[2], m[2];
    __device__ __forceinline__ static int first(int r) { return 64 * (r >> 2) + 8 * (r & 3); }
    __device__ __forceinline__ static float value(const uint8_t* blk, int e) { return q4k_value(blk, e); }
    __device__ __forceinline__ bool load(const uint8_t* blk, int r) {
        const u32x4 hdr = *reinterpret_cast<const u32x4_a1*>(blk);
        const int j = r >> 2;   // groups 2j, 2j + 1
        w = *reinterpret_cast<const u32x2_a1*>(blk + 16 + 32 * j + 8 * (r & 3));
        const uint32_t sh = (uint32_t)((2 * j) & 3) * 8u;
        const uint32_t a = (hdr.y >> sh) & 0xffffu, b = (hdr.z >> sh) & 0xffffu, c = (hdr.w >> sh) & 0xffffu;
        const uint32_t sc = j < 2 ? a & 0x3f3fu : (c & 0x0f0fu) | ((a >> 2) & 0x3030u);
        const uint32_t mn = j < 2 ? b & 0x3f3fu : ((c >> 4) & 0x0f0fu) | ((b >> 2) & 0x3030u);
        const float d = h2f(hdr.x & 0xffffu), dmin = h2f(hdr.x >> 16);
        s[0] = d * (float)(sc & 0xffu);
        s[1] = d * (float)(sc >> 8);
        m[0] = dmin * (float)(mn & 0xffu);
        m[1] = dmin * (float)(mn >> 8);
        return fabsf(d) * 945.f + fabsf(dmin) * 63.f < 65000.f;
    }
    // s, m and s * code are exact in fp32: one rounding, as on the host
    __device__ __forceinline__ void run(int k, float (&v)[8]) const {
        values_of_codes((w.x >> (4 * k)) & 0x0f0f0f0fu, (w.y >> (4 * k)) & 0x0f0f0f0fu,
                        [&](float q) { return fmaf(s[k], q, -m[k]); }, v);
    }
};
struct DequantQ6K {
    static constexpr int kBytes = kQ6KBytes, kThreads = 8, kRuns = 4, kApart = 32;
    u32x2 l[2], u;
    float s[4];
    __device__ __forceinline__ static int first(int r) { return 128 * (r >> 2) + 8 * (r & 3); }
    __device__ __forceinline__ static float value(const uint8_t* blk, int e) { return q6k_value(blk, e); }
    __device__ __forceinline__ bool load(const uint8_t* blk, int r) {
        const int h = r >> 2, i = 8 * (r & 3);
        l[0] = *reinterpret_cast<const u32x2_a1*>(blk + 64 * h + i);
        l[1] = *reinterpret_cast<const u32x2_a1*>(blk + 64 * h + 32 + i);
        u = *reinterpret_cast<const u32x2_a1*>(blk + 128 + 32 * h + i);
        const u32x2 sc = *reinterpret_cast<const u32x2_a1*>(blk + 192 + 8 * h);   // scale i/16 + 2 part
        const float d = blk_half(blk + 208);
        const uint32_t sh = (uint32_t)(i >> 4) * 8u;
        s[0] = d * (float)(int8_t)(sc.x >> sh);   // exact, and every product too
        s[1] = d * (float)(int8_t)(sc.x >> (sh + 16u));
        s[2] = d * (float)(int8_t)(sc.y >> sh);
        s[3] = d * (float)(int8_t)(sc.y >> (sh + 16u));
        return fabsf(d) * 4096.f < 65000.f;
    }
    __device__ __forceinline__ void run(int k, float (&v)[8]) const {
        const u32x2 lo = l[k & 1];
        const int nib = 4 * (k >> 1);
        values_of_codes(((lo.x >> nib) & 0x0f0f0f0fu) | (((u.x >> (2 * k)) & 0x03030303u) << 4),
                        ((lo.y >> nib) & 0x0f0f0f0fu) | (((u.y >> (2 * k)) & 0x03030303u) << 4),
                        [&](float q) { return s[k] * (q - 32.f); }, v);
    }
};

// Whole-tensor dequant.  Bound by memory: per 256 values 144 / 210 bytes in
// and 512 out.  50.3M values of each type on MI355X: Q4_K 27.7 us, Q6_K 28.7
// us, 4.8 TB/s over both (a 1 GiB copy moves 5.2 TB/s).  With one value per
// thread, byte loads and a branching conversion, bound by instruction issue,
// they took 129 and 97 us; with eight values per thread and plain stores 34
// and 44; with the shares above and plain stores 29.6 and 35.5 -- the output
// is not read again soon, so it is stored nontemporal.  A partial last block
// takes the same steps but stores its last run value by value (100,000 values:
// 3.4 us; going back to the bytes value by value 7.6 and 10.3).  Values that
// could overflow are converted one by one by the exact host rule, a run with a
// NaN from the bytes.
template <class QT>
__global__ __launch_bounds__(256) void dequant_kernel(const uint8_t* __restrict__ w, uint64_t count,
                                                      uint16_t* __restrict__ out) {
    const uint64_t n = (count + kQK - 1) / kQK * QT::kThreads, stride = (uint64_t)gridDim.x * blockDim.x;
    for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += stride) {
        const uint64_t b = i / QT::kThreads;
        const uint8_t* blk = w + b * QT::kBytes;
        const int r = (int)(i % QT::kThreads);
        const uint64_t e0 = b * kQK + QT::first(r);
        QT t;
        const bool in_range = t.load(blk, r), whole = b * kQK + kQK <= count;
        float v[8];
        if (in_range) {
#pragma unroll
            for (int k = 0; k < QT::kRuns; ++k) {
                t.run(k, v);
                const u32x4 h{f2h2_ties_away(v[0], v[1]), f2h2_ties_away(v[2], v[3]), f2h2_ties_away(v[4], v[5]),
                              f2h2_ties_away(v[6], v[7])};
                const uint64_t at = e0 + k * QT::kApart;
                if (whole || at + 8 <= count) {
                    __builtin_nontemporal_store(h, reinterpret_cast<u32x4_a2*>(out + at));
                } else {
#pragma unroll
                    for (int e = 0; e < 8; ++e)
                        if (at + e < count) out[at + e] = (uint16_t)(h[e >> 1] >> (16 * (e & 1)));
                }
            }
        } else {
#pragma unroll
            for (int k = 0; k < QT::kRuns; ++k) {
                const uint64_t at = e0 + k * QT::kApart;
                if (at >= count) break;
                const int n = count - at < 8 ? (int)(count - at) : 8;
                t.run(k, v);
                bool nan = false;
#pragma unroll
                for (int e = 0; e < 8; ++e) nan |= __builtin_isnan(v[e]);
                if (!nan) {
#pragma unroll
                    for (int e = 0; e < 8; ++e)
                        if (e < n) out[at + e] = f2h_ties_away(v[e]);
                } else {
#pragma unroll 1
                    for (int e = 0; e < n; ++e)
                        out[at + e] = f2h_ties_away(QT::value(blk, QT::first(r) + k * QT::kApart + e));
                }
            }
        }
    }
}

}  // namespace

hipError_t launch_embed_q6k(const uint8_t* table, int32_t token_id, const int32_t* token_at, int vocab,
                            uint16_t* out, int hidden, hipStream_t s) {
    const int block = 256;
    launch_kernel(embed_q6k_kernel, dim3((hidden + block - 1) / block), dim3(block), 0, s, table, token_id,
                  token_at, vocab, out, hidden);
    return hipGetLastError();
}

namespace {
template <class QT>
hipError_t launch_dequant(const uint8_t* w, uint64_t count, uint16_t* out, hipStream_t s) {
    uint64_t blocks = ((count + kQK - 1) / kQK * QT::kThreads + 255) / 256;
    if (blocks > 1u << 20) blocks = 1u << 20;
    launch_kernel(dequant_kernel<QT>, dim3((unsigned)blocks), dim3(256), 0, s, w, count, out);
    return hipGetLastError();
}
}  // namespace

hipError_t launch_dequant_q4k_f16(const uint8_t* w, uint64_t count, uint16_t* out, hipStream_t s) {
    return launch_dequant<DequantQ4K>(w, count, out, s);
}

hipError_t launch_dequant_q6k_f16(const uint8_t* w, uint64_t count, uint16_t* out, hipStream_t s) {
    return launch_dequant<DequantQ6K>(w, count, out, s);
}

}  // namespace citlali::hip
