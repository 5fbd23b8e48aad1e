// FP8 / bf16 quantize-and-append into the paged KV cache, and per-head absmax scales (gfx950).
//
// Append follows the reference's fp8 encode (techniques/kv_quant/fp8.py:81-86, FP8Cache.transform_update
// fp8.py:161-176): x.float() / scale with IEEE division, clamp to the format's finite maximum, cast with
// round-to-nearest-even (f32_to_fp8 in common.hpp), written at the token's slot (vLLM-style slot mapping: slot =
// page * 16 + position; a negative slot is padding and writes nothing, like the trash slot of
// modules/kv_cache.py:13-27). The per-head scale is the reference's static_scales rule (fp8.py:130-133) over each
// KV head's absolute maximum.
//
// Layout of the caches: see paged_attention.hip. 16-bit states with aligned channels are appended by windows of 16 tokens
// (paged_append_window_kernel); any others, and an append that keeps Quest's metadata, by one workgroup per new token: a
// thread encodes 8 consecutive channels of one head, so the key write is one 8-byte (fp8) or 16-byte (bf16) store into
// the token's 16-byte run, and the value write scatters the 8 channels into their channel rows.

#include "common.hpp"
#include "kv_quant.hpp"
#include "quest_page.hpp"
#include "token_window.hpp"

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
// conversion of two values per instruction, about 6 operations per value instead of 30. The quotient is IEEE
// division's for every 8- or 11-bit significand of x and every fp32 significand of s (its CPU test compares them all)
// while nothing under- or overflows, which kScaleMin <= s <= kScaleMax and |x| < 2^60 ensure down to |x| = 2^-64; a
// smaller |x| gives a quotient below 2^-23, a zero of x's sign in both formats either way. The conversion rounds as
// f32_to_fp8 does up to the format's maximum (the GPU test compares the two kernels on every 16-bit input, the ties of
// both formats and their neighbours among them, at twelve scales). Values outside these limits (and NaN) take encode().
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

// The append by windows of 16 tokens (token_window.hpp) and units of 128 channels over the KV heads, one wave each. Bound
// by reading the states and writing the codes; the workgroup-per-token kernel is bound by its value stores, one byte of
// every 16-byte run from each of 16 workgroups, and by its encoder. Keys: lane (n, g) encodes a 16-byte run of token n
// (any slots), 64 lanes writing 1 KB in a row for consecutive slots. Values: a lane holds two channels of the run's 16
// tokens and packs each channel's run in registers, no exchange between lanes; a wave writes 2 KB in a row. Tokens outside
// runs (decode steps, the ends of prompts) are stored alone, their loads in flight together. 32768 tokens x 8 KV heads, D
// = 128, bf16 to e4m3 (201 MB): 250 us by token, 38.7 us by windows (5.2 TB/s).
template <int FMT, int IN>
__global__ __launch_bounds__(256) void paged_append_window_kernel(AppendParams p) {
    constexpr int ES = FMT == BF16 ? 2 : 1;
    constexpr int E = 16 / ES;           // channels per 16-byte run of the key layout
    constexpr int KR = 128 / E / 4;      // key runs per lane
    constexpr int KL = FMT == BF16 ? 1 : 2;  // 16-byte loads per key run
    const int lane = threadIdx.x & 63;
    const int first = first_of_window();
    if (first >= p.tokens) return;
    const unsigned channels = static_cast<unsigned>(p.kv_heads) * p.head_dim;
    TokenWindow w = token_window(first, p.tokens, lane, [&](int t) {
        const int slot = p.slots[t];
        return slot / PAGE < p.num_pages ? slot : -1;
    });
    const uint16_t* k_new = static_cast<const uint16_t*>(p.k_new);
    const uint16_t* v_new = static_cast<const uint16_t*>(p.v_new);

    const unsigned vc = blockIdx.y * 128 + 2 * lane;  // the lane's value channels: vc, vc + 1
    const bool v_used = vc < channels;
    const int vh = v_used ? vc / p.head_dim : 0, vd = v_used ? vc % p.head_dim : 0;
    const uint16_t* v_src = v_new + vh * p.sv_h + vd;
    uint8_t* v_dst = p.v_cache + vh * p.vc_head + vd * (PAGE * ES);
    uint32_t v[PAGE];
    const auto load_rest = [&]() __attribute__((always_inline)) {
#pragma unroll
        for (int j = 0; j < PAGE; ++j) {
            v[j] = 0;
            if (w.rest >> j & 1) v[j] = *reinterpret_cast<const uint32_t*>(v_src + (first + j) * p.sv_t);
        }
    };
    if (!takes_values()) {
        w.run = -1;
        w.rest = 0;
    }
    if (w.run >= 0) {
#pragma unroll
        for (int j = 0; j < PAGE; ++j)
            v[j] = __builtin_nontemporal_load(reinterpret_cast<const uint32_t*>(v_src + (w.run + j) * p.sv_t));
    } else {
        load_rest();
    }

    if (takes_keys()) {
        const int n = lane & 15, g = lane >> 4;
        const int slot = w.slot(first + n, first);
        const int page = slot / PAGE, pos = slot % PAGE;
        uint4 raw[KR][KL];
        int h[KR], d0[KR];
        bool used[KR];
#pragma unroll
        for (int i = 0; i < KR; ++i) {
            const unsigned ch = blockIdx.y * 128 + (4 * i + g) * E;
            used[i] = ch < channels && slot >= 0;
            h[i] = used[i] ? ch / p.head_dim : 0;
            d0[i] = used[i] ? ch % p.head_dim : 0;
            const uint16_t* src = k_new + (used[i] ? (first + n) * p.sk_t : 0) + h[i] * p.sk_h + d0[i];
#pragma unroll
            for (int u = 0; u < KL; ++u) raw[i][u] = used[i] ? stream_load16(src + 8 * u) : make_uint4(0, 0, 0, 0);
        }
#pragma unroll
        for (int i = 0; i < KR; ++i) {
            uint4 out = raw[i][0];
            if constexpr (FMT == BF16) {
                if (__ballot(max_magnitude8(out) > 0x7F80u) != 0)
                    out = make_uint4(quiet_pair(out.x), quiet_pair(out.y), quiet_pair(out.z), quiet_pair(out.w));
            } else {
                const float s = p.k_scale ? p.k_scale[h[i]] : 1.0f;
                const bool ok = magnitude_within<IN>(max(max_magnitude8(raw[i][0]), max_magnitude8(raw[i][KL - 1]))) &&
                                s >= kScaleMin && s <= kScaleMax;
                const float r = __fdiv_rn(1.0f, s);
                float x[8], y[8];
                unpack8<IN>(raw[i][0], x);
                unpack8<IN>(raw[i][KL - 1], y);
                const auto run = [&](auto fast) __attribute__((always_inline)) {
                    constexpr bool F = decltype(fast)::value;
                    out.x = encode4<FMT, F, true>(x[0], x[1], x[2], x[3], s, r);
                    out.y = encode4<FMT, F, true>(x[4], x[5], x[6], x[7], s, r);
                    out.z = encode4<FMT, F, true>(y[0], y[1], y[2], y[3], s, r);
                    out.w = encode4<FMT, F, true>(y[4], y[5], y[6], y[7], s, r);
                };
                if (__ballot(!ok) == 0) run(std::true_type{});
                else run(std::false_type{});
            }
            if (used[i])
                *reinterpret_cast<uint4*>(p.k_cache + page * p.kc_page + h[i] * p.kc_head +
                                          ((d0[i] / E) * PAGE + pos) * 16) = out;
        }
    }

    const float s = FMT != BF16 && p.v_scale ? p.v_scale[vh] : 1.0f;
    const float r = FMT != BF16 ? __fdiv_rn(1.0f, s) : 1.0f;
    const bool scale_ok = s >= kScaleMin && s <= kScaleMax;
    // One token's two values to its slot.
    const auto store_alone = [&](uint32_t x, int slot, bool fast) __attribute__((always_inline)) {
        uint8_t* dst = v_dst + (slot / PAGE) * p.vc_page + (slot % PAGE) * ES;
        if constexpr (FMT == BF16) {
            *reinterpret_cast<uint16_t*>(dst) = static_cast<uint16_t>(x);
            *reinterpret_cast<uint16_t*>(dst + PAGE * ES) = static_cast<uint16_t>(x >> 16);
        } else {
            float a, b;
            unpack_pair<IN>(x, a, b);
            const uint32_t codes = fast ? encode4<FMT, true, true>(a, b, 0.0f, 0.0f, s, r)
                                        : encode<FMT>(a, s, true) | encode<FMT>(b, s, true) << 8;
            dst[0] = static_cast<uint8_t>(codes);
            dst[PAGE] = static_cast<uint8_t>(codes >> 8);
        }
    };
    if (w.run >= 0) {
        const int slot = __builtin_amdgcn_readfirstlane(w.slot(w.run, first));
        uint8_t* dst = v_dst + (slot / PAGE) * p.vc_page;
        if constexpr (FMT == BF16) {
            quiet_pairs(v);
            uint32_t lo[8], hi[8];
#pragma unroll
            for (int j = 0; j < 8; ++j) {
                lo[j] = __builtin_amdgcn_perm(v[2 * j + 1], v[2 * j], 0x05040100u);
                hi[j] = __builtin_amdgcn_perm(v[2 * j + 1], v[2 * j], 0x07060302u);
            }
            if (v_used) {
                uint4* to = reinterpret_cast<uint4*>(dst);
                to[0] = make_uint4(lo[0], lo[1], lo[2], lo[3]);
                to[1] = make_uint4(lo[4], lo[5], lo[6], lo[7]);
                to[2] = make_uint4(hi[0], hi[1], hi[2], hi[3]);
                to[3] = make_uint4(hi[4], hi[5], hi[6], hi[7]);
            }
        } else {
            uint32_t m = 0;
#pragma unroll
            for (int j = 0; j < PAGE; ++j) m = max_pair(m, v[j] & 0x7FFF7FFFu);
            const bool ok = scale_ok && magnitude_within<IN>(max(m & 0xFFFFu, m >> 16));
            if (__ballot(!ok) == 0) {
                uint32_t lo[4], hi[4];
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    float a[4], b[4];
#pragma unroll
                    for (int i = 0; i < 4; ++i) unpack_pair<IN>(v[4 * j + i], a[i], b[i]);
                    lo[j] = encode4<FMT, true, true>(a[0], a[1], a[2], a[3], s, r);
                    hi[j] = encode4<FMT, true, true>(b[0], b[1], b[2], b[3], s, r);
                }
                if (v_used) {
                    uint4* to = reinterpret_cast<uint4*>(dst);
                    to[0] = make_uint4(lo[0], lo[1], lo[2], lo[3]);
                    to[1] = make_uint4(hi[0], hi[1], hi[2], hi[3]);
                }
            } else if (v_used) {
                for (int j = 0; j < PAGE; ++j)
                    store_alone(*reinterpret_cast<const uint32_t*>(v_src + (w.run + j) * p.sv_t), slot + j, false);
            }
        }
    }
    if (w.rest != 0) {
        uint32_t m = 0;
        if (w.run >= 0) load_rest();
        if constexpr (FMT == BF16) quiet_pairs(v);
#pragma unroll
        for (int j = 0; j < PAGE; ++j) m = max_pair(m, v[j] & 0x7FFF7FFFu);
        const bool ok = scale_ok && magnitude_within<IN>(max(m & 0xFFFFu, m >> 16));
        if (FMT == BF16 || __ballot(!ok) == 0) {
#pragma unroll
            for (int j = 0; j < PAGE; ++j) {
                const int slot = __builtin_amdgcn_readlane(w.slots, j + 15);
                if ((w.rest >> j & 1) && v_used) store_alone(v[j], slot, true);
            }
        } else if (v_used) {
            for (int j = 0; j < PAGE; ++j) {
                const int slot = __builtin_amdgcn_readlane(w.slots, j + 15);
                if (w.rest >> j & 1)
                    store_alone(*reinterpret_cast<const uint32_t*>(v_src + (first + j) * p.sv_t), slot, false);
            }
        }
    }
}

// Whether paged_append_window_kernel takes a call: 16-byte loads of the states, and a format it has an instance for.
bool append_windows(const AppendParams& p) {
    const bool formats = p.cache_format == BF16 ? p.in_format == BF16 : p.in_format == BF16 || p.in_format == FP16;
    return formats && static_cast<int64_t>(p.kv_heads) * p.head_dim <= 65535 * 128 &&
           ((p.sk_t | p.sk_h | p.sv_t | p.sv_h) & 7) == 0 &&
           ((reinterpret_cast<uintptr_t>(p.k_new) | reinterpret_cast<uintptr_t>(p.v_new) |
             reinterpret_cast<uintptr_t>(p.k_cache) | reinterpret_cast<uintptr_t>(p.v_cache)) & 15) == 0;
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
    if (append_windows(p)) {
        dim3 grid, block;
        window_launch(p.tokens, static_cast<int64_t>(p.kv_heads) * p.head_dim, grid, block);
        const auto launch = [&](auto fmt, auto in) {
            hipLaunchKernelGGL((paged_append_window_kernel<fmt.value, in.value>), grid, block, 0, stream, p);
        };
        const std::integral_constant<int, BF16> bf16;
        const std::integral_constant<int, FP16> fp16;
        const std::integral_constant<int, FP8_E4M3> e4m3;
        const std::integral_constant<int, FP8_E5M2> e5m2;
        if (p.cache_format == BF16) launch(bf16, bf16);
        else if (p.cache_format == FP8_E4M3) p.in_format == BF16 ? launch(e4m3, bf16) : launch(e4m3, fp16);
        else p.in_format == BF16 ? launch(e5m2, bf16) : launch(e5m2, fp16);
        return check_launch("paged_append_window_kernel");
    }
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
