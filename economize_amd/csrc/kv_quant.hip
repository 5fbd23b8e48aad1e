// FP8 / bf16 quantize-and-append into the paged KV cache, and per-head absmax scales (gfx950).
//
// Append follows the reference's fp8 encode (techniques/kv_quant/fp8.py:81-86, FP8Cache.transform_update
// fp8.py:161-176): x.float() / scale with IEEE division, clamp to the format's finite maximum, cast with
// round-to-nearest-even (f32_to_fp8 in common.hpp), written at the token's slot (vLLM-style slot mapping: slot =
// page * 16 + position; a negative slot is padding and writes nothing, like the trash slot of
// modules/kv_cache.py:13-27). The per-head scale is the reference's static_scales rule (fp8.py:130-133) over each
// KV head's absolute maximum.
//
// Layout of the caches: see paged_attention.hip. One workgroup per new token; a thread encodes 8 consecutive
// channels of one head, so the key write is one 8-byte (fp8) or 16-byte (bf16) store into the token's 16-byte run,
// and the value write scatters the 8 channels into their channel rows.

#include "common.hpp"
#include "kv_quant.hpp"
#include "quest_page.hpp"

namespace eco {

namespace {

constexpr int PAGE = 16;

__device__ inline float load_elem(const void* base, int64_t offset, int format) {
    if (format == BF16) return bf16_to_f32(static_cast<const uint16_t*>(base)[offset]);
    if (format == FP16) return static_cast<float>(static_cast<const _Float16*>(base)[offset]);
    return static_cast<const float*>(base)[offset];
}

template <int FMT>
__device__ inline uint8_t encode(float x, float scale, bool scaled) {
    float w = scaled ? __fdiv_rn(x, scale) : x;
    if (w != w) return f32_to_fp8<FMT>(x != x ? x : w);  // NaN stays NaN (fminf/fmaxf would drop it)
    return f32_to_fp8<FMT>(fminf(fmaxf(w, -fp8_max<FMT>()), fp8_max<FMT>()));
}

// ---- encoding four values at a time -------------------------------------------------------------------------------
//
// What encode() computes, for bf16 and fp16 inputs: x / s as corrected_quotient and the hardware's round-to-nearest-even
// conversion of two values per instruction, about 6 operations per value instead of 30. The quotient is IEEE division's for every 8- or 11-bit
// significand of x and every fp32 significand of s (checked exhaustively) while nothing under- or overflows, which
// kScaleMin <= s <= kScaleMax and |x| < 2^60 ensure down to |x| = 2^-64; a smaller |x| gives a quotient below 2^-23, a zero
// of x's sign in both formats either way. The conversion equals f32_to_fp8 on every fp32 value up to the format's maximum
// (checked on all of them). Values outside these limits (and NaN) take encode().
constexpr float kScaleMin = 0x1p-40f, kScaleMax = 0x1p60f;

template <int FMT>
__device__ __forceinline__ uint32_t fp8_pack4(float a, float b, float c, float d) {
    if constexpr (FMT == FP8_E4M3)
        return static_cast<uint32_t>(
            __builtin_amdgcn_cvt_pk_fp8_f32(c, d, __builtin_amdgcn_cvt_pk_fp8_f32(a, b, 0, false), true));
    else
        return static_cast<uint32_t>(
            __builtin_amdgcn_cvt_pk_bf8_f32(c, d, __builtin_amdgcn_cvt_pk_bf8_f32(a, b, 0, false), true));
}

// Codes of four values. FAST: within the limits above; CLAMP: quotients may pass the format's maximum (they do not with
// the scale of their own largest value, whose quotient is at most an ulp beyond it).
template <int FMT, bool FAST, bool CLAMP>
__device__ __forceinline__ uint32_t encode4(float a, float b, float c, float d, float s, float r) {
    if constexpr (FAST) {
        const auto one = [&](float x) __attribute__((always_inline)) {
            const float q = corrected_quotient(x, s, r);
            return CLAMP ? __builtin_amdgcn_fmed3f(q, -fp8_max<FMT>(), fp8_max<FMT>()) : q;
        };
        return fp8_pack4<FMT>(one(a), one(b), one(c), one(d));
    }
    return encode<FMT>(a, s, true) | encode<FMT>(b, s, true) << 8 | encode<FMT>(c, s, true) << 16 |
           static_cast<uint32_t>(encode<FMT>(d, s, true)) << 24;
}

typedef unsigned short u16x2 __attribute__((ext_vector_type(2)));

// The larger of two pairs of 16-bit magnitudes.
__device__ __forceinline__ uint32_t max_pair(uint32_t a, uint32_t b) {
    return __builtin_bit_cast(uint32_t, __builtin_elementwise_max(__builtin_bit_cast(u16x2, a), __builtin_bit_cast(u16x2, b)));
}

// The largest magnitude's bits in the four words' eight values, in the low half.
__device__ __forceinline__ uint32_t max_magnitude8(const uint4& w) {
    constexpr uint32_t M = 0x7FFF7FFFu;
    const uint32_t m = max_pair(max_pair(w.x & M, w.y & M), max_pair(w.z & M, w.w & M));
    return max_pair(m, m >> 16) & 0xFFFFu;
}

template <int IN>
__device__ __forceinline__ bool magnitude_within(uint32_t bits) {  // below 2^60 (fp16: finite)
    return bits < (IN == BF16 ? 0x5D80u : 0x7C00u);
}

// New token t into its slot, by one workgroup.
template <int FMT>
__device__ inline void append_token(const AppendParams& p, int t) {
    constexpr int ES = FMT == BF16 ? 2 : 1;
    constexpr int E = 16 / ES;  // channels per 16-byte run of the key layout
    const int slot = p.slots[t];
    if (slot < 0 || slot / PAGE >= p.num_pages) return;
    const int page = slot / PAGE;
    const int pos = slot % PAGE;
    const int runs = p.head_dim / 8;
    for (int item = threadIdx.x; item < p.kv_heads * runs; item += blockDim.x) {
        const int h = item / runs;
        const int d0 = (item % runs) * 8;
        const float ks = p.k_scale ? p.k_scale[h] : 1.0f;
        const float vs = p.v_scale ? p.v_scale[h] : 1.0f;
        float k[8], v[8];
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            k[i] = load_elem(p.k_new, t * p.sk_t + h * p.sk_h + d0 + i, p.in_format);
            v[i] = load_elem(p.v_new, t * p.sv_t + h * p.sv_h + d0 + i, p.in_format);
        }
        uint8_t* kp = p.k_cache + static_cast<int64_t>(page) * p.kc_page + h * p.kc_head;
        uint8_t* vp = p.v_cache + static_cast<int64_t>(page) * p.vc_page + h * p.vc_head;
        const int64_t k_off = ((d0 / E) * PAGE + pos) * 16 + (d0 % E) * ES;
        if constexpr (FMT == BF16) {
            uint4 w;
            w.x = f32_to_bf16(k[0]) | (static_cast<uint32_t>(f32_to_bf16(k[1])) << 16);
            w.y = f32_to_bf16(k[2]) | (static_cast<uint32_t>(f32_to_bf16(k[3])) << 16);
            w.z = f32_to_bf16(k[4]) | (static_cast<uint32_t>(f32_to_bf16(k[5])) << 16);
            w.w = f32_to_bf16(k[6]) | (static_cast<uint32_t>(f32_to_bf16(k[7])) << 16);
            *reinterpret_cast<uint4*>(kp + k_off) = w;
#pragma unroll
            for (int i = 0; i < 8; ++i)
                *reinterpret_cast<uint16_t*>(vp + ((d0 + i) * PAGE + pos) * 2) = f32_to_bf16(v[i]);
        } else {
            const bool scaled = p.k_scale != nullptr;
            uint32_t lo = 0, hi = 0;
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                lo |= static_cast<uint32_t>(encode<FMT>(k[i], ks, scaled)) << (8 * i);
                hi |= static_cast<uint32_t>(encode<FMT>(k[i + 4], ks, scaled)) << (8 * i);
            }
            *reinterpret_cast<uint2*>(kp + k_off) = make_uint2(lo, hi);
            const bool vscaled = p.v_scale != nullptr;
#pragma unroll
            for (int i = 0; i < 8; ++i) vp[(d0 + i) * PAGE + pos] = encode<FMT>(v[i], vs, vscaled);
        }
    }
}

template <int FMT>
__global__ __launch_bounds__(256) void paged_append_kernel(AppendParams p) {
    append_token<FMT>(p, blockIdx.x);
}

// The append with Quest's metadata kept on the device, in one launch: workgroups below `tokens` append a token each;
// the others are four waves each of the refresh, kRefreshWaves waves per (row, KV head) taking equal parts of the Quest
// pages from valid to the row's committed ones (the bounds of pages that became committed, quest_refresh_kernel's
// work). The last of a row's waves to finish (a counter per row, agent-scope atomics; every
// wave has read valid before it counts itself) advances valid and writes done, then leaves the counter zero. The
// tokens appended lie at or past the committed ones, so no page this launch refreshes is written by it.
constexpr int kRefreshWaves = 8;

template <int FMT, int D>
__global__ __launch_bounds__(256) void paged_append_quest_kernel(AppendParams p, BoundsParams q, int32_t* counters) {
    if (static_cast<int>(blockIdx.x) < p.tokens) {
        append_token<FMT>(p, blockIdx.x);
        return;
    }
    const int wave = (static_cast<int>(blockIdx.x) - p.tokens) * 4 + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int lane = static_cast<int>(threadIdx.x & 63);
    if (wave >= q.batch * q.kv_heads * kRefreshWaves) return;
    const int row = wave / kRefreshWaves, y = wave % kRefreshWaves;
    const int b = row / q.kv_heads, kvh = row % q.kv_heads;
    const int last = min(max(q.committed[b], 0) / (16 * q.span), q.page_cap);
    const int from = q.valid[row];
    const int each = (last - from + kRefreshWaves - 1) / kRefreshWaves;
    const int q0 = from + y * each;
    quest_bounds_range<FMT, D>(q, b, kvh, q0, min(q0 + each, last), lane);
    int prev = 0;
    if (lane == 0) prev = __hip_atomic_fetch_add(counters + row, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    if (__shfl(prev, 0) != kRefreshWaves - 1) return;
    if (lane == 0) {
        q.valid[row] = max(from, last);
        if (q.done && kvh == 0) q.done[b] = last;
        __hip_atomic_store(counters + row, 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
}

// Dense encode (fp8_encode of fp8.py:81-86 over a [B, H, T, D] block, the fused fp8 cache's dense buffers of
// kv_fp8_fused/fused.py:56-63): one wave per (b, h, t) row, each lane a few channels. The per-token mode computes the
// row's scale as token_scale does (fp8.py:95-97: absmax / format max with IEEE division, at least 1e-12), writes it
// and encodes with it; the per-head mode divides by head_scale[h]; with neither the values are cast directly.
template <int FMT>
__global__ __launch_bounds__(256) void fp8_encode_kernel(EncodeParams p) {
    const int lane = threadIdx.x & 63;
    const int64_t rows = static_cast<int64_t>(p.batch) * p.heads * p.tokens;
    for (int64_t row = blockIdx.x * 4LL + (threadIdx.x >> 6); row < rows; row += static_cast<int64_t>(gridDim.x) * 4) {
        const int t = static_cast<int>(row % p.tokens);
        const int h = static_cast<int>((row / p.tokens) % p.heads);
        const int b = static_cast<int>(row / (static_cast<int64_t>(p.tokens) * p.heads));
        const int64_t src = b * p.ss_b + h * p.ss_h + t * p.ss_t;
        uint8_t* dst = p.dst + b * p.sd_b + h * p.sd_h + t * p.sd_t;
        float x[8];  // channels lane, lane + 64, .. (head dims up to 512)
        float amax = 0.0f;
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            const int d = lane + 64 * i;
            x[i] = d < p.head_dim ? load_elem(p.src, src + d, p.in_format) : 0.0f;
            amax = fmaxf(amax, fabsf(x[i]));
        }
        float scale = 1.0f;
        bool scaled = false;
        if (p.token_scale) {
            bool nan = false;  // torch's amax propagates NaN, and so does the scale then
#pragma unroll
            for (int i = 0; i < 8; ++i) nan |= x[i] != x[i];
            for (int off = 32; off > 0; off >>= 1) amax = fmaxf(amax, __shfl_xor(amax, off));
            scale = __ballot(nan) ? __builtin_nanf("") : fmaxf(__fdiv_rn(amax, fp8_max<FMT>()), 1e-12f);
            scaled = true;
            if (lane == 0) p.token_scale[b * p.st_b + h * p.st_h + t * p.st_t] = scale;
        } else if (p.head_scale) {
            scale = p.head_scale[h];
            scaled = true;
        }
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            const int d = lane + 64 * i;
            if (d < p.head_dim) dst[d] = encode<FMT>(x[i], scale, scaled);
        }
    }
}

// The dense encode of bf16 and fp16 rows whose 8-channel runs are 16-byte loads and 8-byte stores: L lanes per row (D / 8
// rounded up to a power of two), kEncodeRows rows per lane with all their loads in flight. Bound by reading x and writing
// the codes; fp8_encode_kernel, which takes everything else, is bound by its instructions: 2-byte loads, three 64-bit
// divisions per row, the IEEE divisions and the bitwise encoder. 8 x 8 x 4096 rows of D = 128, bf16 with a
// scale per token (101 MB): 133 us there, 19.4 us here (5.2 TB/s).
constexpr int kEncodeRows = 4;

template <int FMT, int IN, int L>
__global__ __launch_bounds__(256) void fp8_encode_rows_kernel(EncodeParams p) {
    constexpr int R = 256 / L;  // rows per workgroup and step
    const int c = threadIdx.x % L;
    const int b = blockIdx.y / p.heads, h = blockIdx.y % p.heads;
    const int t0 = blockIdx.x * (R * kEncodeRows) + threadIdx.x / L;
    const bool lane_used = 8 * c < p.head_dim;
    const uint16_t* src = static_cast<const uint16_t*>(p.src) + b * p.ss_b + h * p.ss_h + 8 * c;
    uint8_t* dst = p.dst + b * p.sd_b + h * p.sd_h + 8 * c;
    uint4 raw[kEncodeRows];
#pragma unroll
    for (int i = 0; i < kEncodeRows; ++i) {
        const int t = t0 + i * R;
        raw[i] = lane_used && t < p.tokens ? stream_load16(src + t * p.ss_t) : make_uint4(0, 0, 0, 0);
    }
    const bool per_token = p.token_scale != nullptr;
    const float head = p.head_scale ? p.head_scale[h] : 1.0f;
#pragma unroll
    for (int i = 0; i < kEncodeRows; ++i) {
        const int t = t0 + i * R;
        if (blockIdx.x * (R * kEncodeRows) + i * R >= p.tokens) break;
        uint32_t m = max_magnitude8(raw[i]);
        float s = head;
        if (per_token) {
            m = max(m, dpp<0xB1>(m));   // quad_perm 1 0 3 2
            m = max(m, dpp<0x4E>(m));   // quad_perm 2 3 0 1
            m = max(m, dpp<0x141>(m));  // row_half_mirror
            if constexpr (L > 8) m = max(m, dpp<0x140>(m));  // row_mirror
            if constexpr (L > 16) m = max(m, static_cast<uint32_t>(__shfl_xor(static_cast<int>(m), 16)));
            if constexpr (L > 32) m = max(m, static_cast<uint32_t>(__shfl_xor(static_cast<int>(m), 32)));
            const float amax = IN == BF16 ? bits_f32(m << 16)
                                          : static_cast<float>(__builtin_bit_cast(_Float16, static_cast<uint16_t>(m)));
            // a NaN's magnitude is the largest: the row's scale is then NaN, as torch's amax propagates it
            s = amax == amax ? fmaxf(__fdiv_rn(amax, fp8_max<FMT>()), 1e-12f) : __builtin_nanf("");
            if (c == 0 && t < p.tokens) p.token_scale[b * p.st_b + h * p.st_h + t * p.st_t] = s;
        }
        const bool ok = magnitude_within<IN>(m) && s >= kScaleMin && s <= kScaleMax;
        const float r = __fdiv_rn(1.0f, s);
        float x[8];
        unpack8<IN>(raw[i], x);
        uint2 codes;
        const auto encode8 = [&](auto fast, auto clamp) __attribute__((always_inline)) {
            constexpr bool F = decltype(fast)::value, K = decltype(clamp)::value;
            codes.x = encode4<FMT, F, K>(x[0], x[1], x[2], x[3], s, r);
            codes.y = encode4<FMT, F, K>(x[4], x[5], x[6], x[7], s, r);
        };
        if (__ballot(!ok) != 0) encode8(std::false_type{}, std::true_type{});
        else if (per_token) encode8(std::true_type{}, std::false_type{});
        else encode8(std::true_type{}, std::true_type{});
        if (lane_used && t < p.tokens) *reinterpret_cast<uint2*>(dst + t * p.sd_t) = codes;
    }
}

// Whether fp8_encode_rows_kernel takes a call: its loads and stores aligned, its grid within the limits.
bool encode_rows(const EncodeParams& p) {
    return (p.in_format == BF16 || p.in_format == FP16) && p.head_dim % 8 == 0 &&
           static_cast<int64_t>(p.batch) * p.heads <= 65535 && ((p.ss_b | p.ss_h | p.ss_t) & 7) == 0 &&
           ((p.sd_b | p.sd_h | p.sd_t) & 7) == 0 && (reinterpret_cast<uintptr_t>(p.src) & 15) == 0 &&
           (reinterpret_cast<uintptr_t>(p.dst) & 7) == 0;
}

template <int FMT, int IN>
void launch_encode_rows(const EncodeParams& p, hipStream_t stream) {
    const auto launch = [&](auto lanes) {
        constexpr int L = decltype(lanes)::value;
        const dim3 grid(ceil_div(p.tokens, 256 / L * kEncodeRows), p.batch * p.heads);
        hipLaunchKernelGGL((fp8_encode_rows_kernel<FMT, IN, L>), grid, dim3(256), 0, stream, p);
    };
    if (p.head_dim <= 64) launch(std::integral_constant<int, 8>{});
    else if (p.head_dim <= 128) launch(std::integral_constant<int, 16>{});
    else if (p.head_dim <= 256) launch(std::integral_constant<int, 32>{});
    else launch(std::integral_constant<int, 64>{});
}

// absmax[h] = max |x[a, h, s, d]| as float bits (non-negative floats order like their bit patterns).
__global__ __launch_bounds__(256) void head_absmax_kernel(AbsmaxParams p) {
    const int h = blockIdx.y;
    const int64_t total = static_cast<int64_t>(p.a) * p.s * p.d;
    float m = 0.0f;
    for (int64_t idx = blockIdx.x * static_cast<int64_t>(blockDim.x) + threadIdx.x; idx < total;
         idx += static_cast<int64_t>(gridDim.x) * blockDim.x) {
        const int64_t a = idx / (static_cast<int64_t>(p.s) * p.d);
        const int64_t s = (idx / p.d) % p.s;
        const int64_t d = idx % p.d;
        const float x = load_elem(p.x, a * p.sa + h * p.sh + s * p.ss + d * p.sd, p.in_format);
        m = fmaxf(m, fabsf(x));
    }
    for (int off = 32; off > 0; off >>= 1) m = fmaxf(m, __shfl_xor(m, off));
    if ((threadIdx.x & 63) == 0) atomicMax(p.absmax_bits + h, f32_bits(m));
}

// static_scales (fp8.py:130-133): absmax / format max with IEEE division, 1 where that is not positive.
__global__ void scales_from_absmax_kernel(const uint32_t* absmax_bits, int heads, float format_max, float* scales) {
    const int h = blockIdx.x * blockDim.x + threadIdx.x;
    if (h < heads) {
        const float s = __fdiv_rn(bits_f32(absmax_bits[h]), format_max);
        scales[h] = s > 0.0f ? s : 1.0f;
    }
}

}  // namespace

int paged_append(const AppendParams& p, hipStream_t stream) {
    if (p.tokens == 0) return 0;
    dim3 grid(p.tokens);
    switch (p.cache_format) {
        case BF16: hipLaunchKernelGGL(paged_append_kernel<BF16>, grid, dim3(256), 0, stream, p); break;
        case FP8_E4M3: hipLaunchKernelGGL(paged_append_kernel<FP8_E4M3>, grid, dim3(256), 0, stream, p); break;
        case FP8_E5M2: hipLaunchKernelGGL(paged_append_kernel<FP8_E5M2>, grid, dim3(256), 0, stream, p); break;
        default: return fail("paged append: cache format must be bf16, fp8 e4m3 or fp8 e5m2");
    }
    return check_launch("paged_append_kernel");
}

int paged_append_quest(const AppendParams& p, const BoundsParams& q, int32_t* counters, hipStream_t stream) {
    const int refresh = (q.batch * q.kv_heads * kRefreshWaves + 3) / 4;
    dim3 grid(p.tokens + refresh);
    if (!quest_bounds_dispatch(p.cache_format, q.head_dim, [&](auto fmt, auto dim) {
            hipLaunchKernelGGL((paged_append_quest_kernel<fmt.value, dim.value>), grid, dim3(256), 0, stream, p, q,
                               counters);
        }))
        return fail("paged append: cache format must be bf16, fp8 e4m3 or fp8 e5m2");
    return check_launch("paged_append_quest_kernel");
}

int fp8_encode(const EncodeParams& p, hipStream_t stream) {
    const int64_t rows = static_cast<int64_t>(p.batch) * p.heads * p.tokens;
    if (rows == 0) return 0;
    if (encode_rows(p) && (p.out_format == FP8_E4M3 || p.out_format == FP8_E5M2)) {
        const bool bf16 = p.in_format == BF16, e4m3 = p.out_format == FP8_E4M3;
        if (bf16) e4m3 ? launch_encode_rows<FP8_E4M3, BF16>(p, stream) : launch_encode_rows<FP8_E5M2, BF16>(p, stream);
        else e4m3 ? launch_encode_rows<FP8_E4M3, FP16>(p, stream) : launch_encode_rows<FP8_E5M2, FP16>(p, stream);
        return check_launch("fp8_encode_rows_kernel");
    }
    const int blocks = static_cast<int>((rows + 3) / 4 < 65535 ? (rows + 3) / 4 : 65535);
    switch (p.out_format) {
        case FP8_E4M3: hipLaunchKernelGGL(fp8_encode_kernel<FP8_E4M3>, dim3(blocks), dim3(256), 0, stream, p); break;
        case FP8_E5M2: hipLaunchKernelGGL(fp8_encode_kernel<FP8_E5M2>, dim3(blocks), dim3(256), 0, stream, p); break;
        default: return fail("fp8 encode: the output format must be fp8 e4m3 or e5m2");
    }
    return check_launch("fp8_encode_kernel");
}

int head_absmax(const AbsmaxParams& p, hipStream_t stream) {
    const int64_t total = static_cast<int64_t>(p.a) * p.s * p.d;
    int blocks = static_cast<int>((total + 256 * 16 - 1) / (256 * 16));
    blocks = blocks < 1 ? 1 : (blocks > 1024 ? 1024 : blocks);
    hipLaunchKernelGGL(head_absmax_kernel, dim3(blocks, p.h), dim3(256), 0, stream, p);
    return check_launch("head_absmax_kernel");
}

int scales_from_absmax(const uint32_t* absmax_bits, int heads, int format, float* scales, hipStream_t stream) {
    const float fmax = format == FP8_E4M3 ? 448.0f : 57344.0f;
    hipLaunchKernelGGL(scales_from_absmax_kernel, dim3((heads + 63) / 64), dim3(64), 0, stream, absmax_bits, heads,
                       fmax, scales);
    return check_launch("scales_from_absmax_kernel");
}

}  // namespace eco
