// KIVI (Liu et al., ICML 2024) on gfx950: the quantization schedule, the full-precision residual ring, and
// quantize-and-append into 32-token pages (the attention over them: kivi.hip).
//
// Quantization follows the reference's quantize (techniques/kv_quant/kivi.py:121-140): fp32 min and max along the
// group; scale = fp16r((high - low) / levels) and low = fp16r(low), fp16r rounding to nearest even where fp16 holds
// the value; codes = round_half_even((x - low) / safe) clamped to [0, levels], safe = scale or 1 where the scale is 0.
// Both divisions are IEEE divisions (__fdiv_rn), the CPU semantics of torch's tensor / int and tensor / tensor (GPU
// torch multiplies by a reciprocal instead; the parity oracle is the CPU definition). Keys are quantized per channel
// over a 32-token group (one page), values per token over 32-channel groups. The schedule is the reference's
// (kivi.py:230-243): with c committed tokens, keys below (c / R) * R and values below max(0, c - R) are quantized.
//
// Page block: see kivi.hip. Pages of bf16 and fp16 sources with contiguous, aligned channels are quantized by one wave
// each (quantize_keys_wave, quantize_values_wave); any other source (fp32, the token-contiguous value ring, odd
// strides) by one workgroup per page (kivi_quant_keys_kernel, kivi_quant_values_kernel).

#include "common.hpp"
#include "kivi.hpp"
#include "kivi_math.hpp"
#include "token_window.hpp"

namespace eco {

namespace {

constexpr int KPAGE = KiviParams::kPage;  // 32 tokens

__device__ inline float load_elem(const void* base, int64_t offset, int format) {
    if (format == BF16) return bf16_to_f32(static_cast<const uint16_t*>(base)[offset]);
    if (format == FP16) return static_cast<float>(static_cast<const _Float16*>(base)[offset]);
    return static_cast<const float*>(base)[offset];
}

__device__ inline uint16_t f16_bits(float x) {
    return __builtin_bit_cast(uint16_t, static_cast<_Float16>(x));
}

// ---- schedule --------------------------------------------------------------------------------------------------

// ranges [4][B]: keys [from, to), values [from, to) to quantize now; the counts advance to their new values.
__global__ void kivi_schedule_kernel(const int32_t* committed, int residual, int32_t* kq, int32_t* vq,
                                     int32_t* ranges, int batch) {
    const int b = blockIdx.x * blockDim.x + threadIdx.x;
    if (b >= batch) return;
    const int c = max(committed[b], 0);
    const int k_to = max(kq[b], (c / residual) * residual);
    const int v_to = max(vq[b], c - residual);
    ranges[b] = kq[b];
    ranges[batch + b] = k_to;
    ranges[2 * batch + b] = vq[b];
    ranges[3 * batch + b] = v_to;
    kq[b] = k_to;
    vq[b] = v_to;
}

// ---- residual ring ------------------------------------------------------------------------------------------

// One workgroup per new token: keys to slot t % W of [B, Hkv, W, D], values to [B, Hkv, D, W], rounded to bf16.
__global__ __launch_bounds__(256) void kivi_ring_kernel(KiviRingParams p) {
    const int t = blockIdx.x;
    const int pos = p.positions[t];
    const int b = p.rows[t];
    if (pos < 0 || b < 0 || b >= p.batch) return;
    const int slot = pos % p.ring;
    for (int i = threadIdx.x; i < p.kv_heads * p.head_dim; i += blockDim.x) {
        const int h = i / p.head_dim, d = i % p.head_dim;
        const float k = load_elem(p.k_new, t * p.sk_t + h * p.sk_h + d, p.in_format);
        const float v = load_elem(p.v_new, t * p.sv_t + h * p.sv_h + d, p.in_format);
        const int64_t row = static_cast<int64_t>(b) * p.kv_heads + h;
        p.k_ring[(row * p.ring + slot) * p.head_dim + d] = f32_to_bf16(k);
        p.v_ring[(row * p.head_dim + d) * p.ring + slot] = f32_to_bf16(v);
    }
}

// The same for bf16 states with aligned 8-channel runs, by windows of 16 tokens (token_window.hpp; a token's slot here is
// its row's ring and its place in it) and units of 128 channels over the KV heads, one wave each. Bound by moving the
// states; the workgroup-per-token kernel is bound by its value stores, 2 bytes each at the ring's stride. Keys are copied
// 16 bytes at a time; for values a lane holds two channels of a run's 16 tokens and stores 32 bytes of each; the four
// waves of a workgroup take successive windows, so that they fill a value line together. 8 rows' 384 tokens x 8 KV
// heads, D = 128 (25 MB): 33 us by token, 8 us by windows.
__global__ __launch_bounds__(256) void kivi_ring_window_kernel(KiviRingParams p) {
    const int lane = threadIdx.x & 63;
    const int first = first_of_window();
    if (first >= p.tokens) return;
    const unsigned channels = static_cast<unsigned>(p.kv_heads) * p.head_dim;
    TokenWindow w = token_window(first, p.tokens, lane, [&](int t) {
        const int pos = p.positions[t], b = p.rows[t];
        return pos < 0 || b < 0 || b >= p.batch ? -1 : b * p.ring + pos % p.ring;
    });

    const unsigned vc = blockIdx.y * 128 + 2 * lane;  // the lane's value channels: vc, vc + 1
    const bool v_used = vc < channels;
    const int vh = v_used ? vc / p.head_dim : 0, vd = v_used ? vc % p.head_dim : 0;
    const uint16_t* v_src = static_cast<const uint16_t*>(p.v_new) + vh * p.sv_h + vd;
    // the slots' rows and places, divided in the lanes that hold them
    const int slot_row = w.slots / p.ring, slot_at = w.slots - slot_row * p.ring;
    const auto v_dst = [&](int l) {
        const int64_t head = static_cast<int64_t>(__builtin_amdgcn_readlane(slot_row, l)) * p.kv_heads + vh;
        return p.v_ring + (head * p.head_dim + vd) * p.ring + __builtin_amdgcn_readlane(slot_at, l);
    };
    uint32_t v[16];
    const auto load_rest = [&]() __attribute__((always_inline)) {
#pragma unroll
        for (int j = 0; j < 16; ++j) {
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
        for (int j = 0; j < 16; ++j) v[j] = *reinterpret_cast<const uint32_t*>(v_src + (w.run + j) * p.sv_t);
    } else {
        load_rest();
    }

    if (takes_keys()) {
        const unsigned kc = blockIdx.y * 128 + 8 * (lane & 15);  // the lane's key channels: kc .. kc + 7
        const int kh = kc < channels ? kc / p.head_dim : 0, kd = kc < channels ? kc % p.head_dim : 0;
        const uint16_t* k_src = static_cast<const uint16_t*>(p.k_new) + kh * p.sk_h + kd;
        uint4 k[4];
        int slots[4], k_row[4], k_at[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int t = first + 4 * i + (lane >> 4);
            slots[i] = w.slot(t, first);
            k_row[i] = __shfl(slot_row, t - first + 15);
            k_at[i] = __shfl(slot_at, t - first + 15);
            if (kc >= channels) slots[i] = -1;
            k[i] = slots[i] >= 0 ? *reinterpret_cast<const uint4*>(k_src + t * p.sk_t) : make_uint4(0, 0, 0, 0);
        }
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            uint32_t x[4] = {k[i].x, k[i].y, k[i].z, k[i].w};
            quiet_pairs(x);
            if (slots[i] < 0) continue;
            const int64_t head = static_cast<int64_t>(k_row[i]) * p.kv_heads + kh;
            *reinterpret_cast<uint4*>(p.k_ring + (head * p.ring + k_at[i]) * p.head_dim + kd) =
                make_uint4(x[0], x[1], x[2], x[3]);
        }
    }

    if (w.run >= 0) {
        quiet_pairs(v);
        uint32_t lo[8], hi[8];
#pragma unroll
        for (int j = 0; j < 8; ++j) {
            lo[j] = __builtin_amdgcn_perm(v[2 * j + 1], v[2 * j], 0x05040100u);
            hi[j] = __builtin_amdgcn_perm(v[2 * j + 1], v[2 * j], 0x07060302u);
        }
        uint16_t* dst = v_dst(w.run - first + 15);
        if (v_used) {
            uint4* to = reinterpret_cast<uint4*>(dst);
            to[0] = make_uint4(lo[0], lo[1], lo[2], lo[3]);
            to[1] = make_uint4(lo[4], lo[5], lo[6], lo[7]);
            to = reinterpret_cast<uint4*>(dst + p.ring);
            to[0] = make_uint4(hi[0], hi[1], hi[2], hi[3]);
            to[1] = make_uint4(hi[4], hi[5], hi[6], hi[7]);
        }
    }
    if (w.rest != 0) {
        if (w.run >= 0) load_rest();
        quiet_pairs(v);
#pragma unroll
        for (int j = 0; j < 16; ++j) {
            uint16_t* dst = v_dst(j + 15);
            if ((w.rest >> j & 1) && v_used) {
                dst[0] = static_cast<uint16_t>(v[j]);
                dst[p.ring] = static_cast<uint16_t>(v[j] >> 16);
            }
        }
    }
}

// Whether kivi_ring_window_kernel takes a call: bf16 states as 16-byte runs, ring slots whose multiples of 16 are aligned.
bool ring_windows(const KiviRingParams& p) {
    return p.in_format == BF16 && p.head_dim % 8 == 0 && p.ring % 16 == 0 &&
           ((p.sk_t | p.sk_h | p.sv_t | p.sv_h) & 7) == 0 &&
           static_cast<int64_t>(p.batch) * p.ring <= INT32_MAX &&
           static_cast<int64_t>(p.kv_heads) * p.head_dim <= 65535 * 128 &&
           ((reinterpret_cast<uintptr_t>(p.k_new) | reinterpret_cast<uintptr_t>(p.v_new) |
             reinterpret_cast<uintptr_t>(p.k_ring) | reinterpret_cast<uintptr_t>(p.v_ring)) & 15) == 0;
}

// ---- quantize-and-append ----------------------------------------------------------------------------------------

__device__ inline float src_elem(const KiviQuantParams& p, int b, int h, int t, int d) {
    const int slot = p.src_ring > 0 ? t % p.src_ring : t - p.src_start;
    return load_elem(p.src, b * p.ss_b + h * p.ss_h + static_cast<int64_t>(slot) * p.ss_t + d * p.ss_d,
                     p.src_format);
}

__device__ inline uint8_t* page_block(const KiviQuantParams& p, int b, int h, int page) {
    if (page >= p.bt_cols) return nullptr;
    const int phys = p.block_table[b * p.bt_stride + page];
    if (phys < 0 || phys >= p.num_pages) return nullptr;
    return p.blocks + static_cast<int64_t>(phys) * p.blk_page + h * p.blk_head;
}

// Keys: one workgroup per (row, KV head) and 32-token group in [from, to) (multiples of 32).
__global__ __launch_bounds__(256) void kivi_quant_keys_kernel(KiviQuantParams p) {
    __shared__ float s_low[256], s_safe[256];
    const int row = blockIdx.x;
    const int b = row / p.kv_heads, h = row % p.kv_heads;
    const int page = p.from[b] / KPAGE + static_cast<int>(blockIdx.y);
    const int t0 = page * KPAGE;
    if (t0 + KPAGE > p.to[b]) return;
    uint8_t* blk = page_block(p, b, h, page);
    if (!blk) return;
    const KiviLayout L{p.head_dim, p.bits};
    const int levels = (1 << p.bits) - 1;
    for (int d = threadIdx.x; d < p.head_dim; d += blockDim.x) {
        float lo = INFINITY, hi = -INFINITY;
        for (int t = 0; t < KPAGE; ++t) {
            const float x = src_elem(p, b, h, t0 + t, d);
            lo = fminf(lo, x);
            hi = fmaxf(hi, x);
        }
        const Quant q = make_quant(lo, hi, levels, p.overflow);
        s_low[d] = q.low;
        s_safe[d] = q.safe;
        reinterpret_cast<uint16_t*>(blk + L.k_scale())[d] = f16_bits(q.scale);
        reinterpret_cast<uint16_t*>(blk + L.k_zero())[d] = f16_bits(q.low);
    }
    __syncthreads();
    const int per_word = 32 / p.bits;
    const int words = p.head_dim / per_word;  // per token
    for (int item = threadIdx.x; item < KPAGE * words; item += blockDim.x) {
        const int t = item / words, w = item % words;
        uint32_t word = 0;
        for (int e = 0; e < per_word; ++e) {
            const int d = w * per_word + e;
            const Quant q{0.0f, s_low[d], s_safe[d]};
            word |= code_of(src_elem(p, b, h, t0 + t, d), q, levels) << (8 * (e & 3) + (e >> 2) * p.bits);
        }
        reinterpret_cast<uint32_t*>(blk + L.k_codes() + t * (p.head_dim * p.bits / 8))[w] = word;
    }
}

// Values: one workgroup per (row, KV head) and page overlapping [from, to); the page's other tokens keep their codes.
__global__ __launch_bounds__(256) void kivi_quant_values_kernel(KiviQuantParams p) {
    __shared__ float s_low[KPAGE][8], s_safe[KPAGE][8];
    const int row = blockIdx.x;
    const int b = row / p.kv_heads, h = row % p.kv_heads;
    const int page = p.from[b] / KPAGE + static_cast<int>(blockIdx.y);
    const int t0 = page * KPAGE;
    const int lo_t = max(p.from[b], t0), hi_t = min(p.to[b], t0 + KPAGE);
    if (lo_t >= hi_t) return;
    uint8_t* blk = page_block(p, b, h, page);
    if (!blk) return;
    const KiviLayout L{p.head_dim, p.bits};
    const int levels = (1 << p.bits) - 1;
    const int groups = p.head_dim / 32;
    for (int item = threadIdx.x; item < (hi_t - lo_t) * groups; item += blockDim.x) {
        const int t = lo_t + item / groups, grp = item % groups;
        float lo = INFINITY, hi = -INFINITY;
        for (int d = 32 * grp; d < 32 * grp + 32; ++d) {
            const float x = src_elem(p, b, h, t, d);
            lo = fminf(lo, x);
            hi = fmaxf(hi, x);
        }
        const Quant q = make_quant(lo, hi, levels, p.overflow);
        s_low[t - t0][grp] = q.low;
        s_safe[t - t0][grp] = q.safe;
        reinterpret_cast<uint16_t*>(blk + L.v_scale())[grp * KPAGE + (t - t0)] = f16_bits(q.scale);
        reinterpret_cast<uint16_t*>(blk + L.v_zero())[grp * KPAGE + (t - t0)] = f16_bits(q.low);
    }
    __syncthreads();
    const int per_word = 32 / p.bits;  // tokens per word
    const int nd_count = p.head_dim / 16;
    uint32_t* words = reinterpret_cast<uint32_t*>(blk + L.v_codes());
    for (int item = threadIdx.x; item < p.bits * 16 * nd_count; item += blockDim.x) {
        const int u = item / (16 * nd_count);
        const int n = (item / nd_count) % 16;
        const int nd = item % nd_count;
        const int d = 16 * nd + n;
        const int w0 = t0 + u * per_word;  // first token of the word
        if (w0 + per_word <= lo_t || w0 >= hi_t) continue;
        uint32_t word = words[item];
        for (int e = 0; e < per_word; ++e) {
            const int t = w0 + e;
            if (t < lo_t || t >= hi_t) continue;
            const int shift = 8 * (e & 3) + (e >> 2) * p.bits;
            const Quant q{0.0f, s_low[t - t0][d / 32], s_safe[t - t0][d / 32]};
            word = (word & ~(static_cast<uint32_t>(levels) << shift)) | (code_of(src_elem(p, b, h, t, d), q, levels) << shift);
        }
        words[item] = word;
    }
}

// ---- quantize-and-append, one wave per page ---------------------------------------------------------------------
//
// Bound by reading the source once. A lane holds 8 channels (one 16-byte load) of D / 16 tokens of the page, so all of
// a page's loads are in flight together and its elements stay in registers for both passes (minimum and maximum, then
// codes); the workgroup-per-page kernels read every element twice with 2-byte loads, 32 in a serial chain per thread,
// and divide each by IEEE division. Here the quotient (x - low) / safe is one correction step on a reciprocal, which
// gives the same codes (page_code). 8 rows x 4096 tokens x 8 KV heads, D = 128, 4 bits, bf16 (88 and 85 MB): keys 119 and
// values 120 us by workgroups, 19.4 and 24.8 us by waves. The keys' 88 MB move at 4.5 TB/s; the values' code stores, 4 bytes
// of every 32, reach memory as 36.5 MB where the bytes are 20.3, 102 MB in all at 4.1 TB/s.

// A group's quantization with what its codes need.
struct PageQuant {
    float scale, low, safe, rcp;
};

// make_quant of a group whose values are finite, |low| <= 65504 and (high - low) / levels <= 65504: (high - low) /
// levels by one correction step on the rounded reciprocal, which is the IEEE quotient for every fp32 numerator (checked
// over all 2^23 significands for 3 and 15; a numerator too small for the step to be exact rounds to a zero scale either
// way). False (in any lane) leaves the group to make_quant.
template <int BITS>
__device__ __forceinline__ bool page_quant(float lo, float hi, PageQuant& q) {
    constexpr float L = static_cast<float>((1 << BITS) - 1);
    constexpr float R = 1.0f / L;
    const float n = hi - lo;
    const float s = corrected_quotient(n, L, R);
    q.scale = static_cast<float>(static_cast<_Float16>(s));
    q.low = static_cast<float>(static_cast<_Float16>(lo));
    q.safe = q.scale > 0.0f ? q.scale : 1.0f;
    q.rcp = __builtin_amdgcn_rcpf(q.safe);
    return fabsf(lo) <= 65504.0f && n <= 65504.0f * L;  // false for NaN and infinities
}

// A word whose low byte is code_of(x, q, levels), for a q of page_quant. The code is the quotient rounded half to even,
// so only the side of a half integer h <= 14.5 it lies on matters. safe has an 11-bit significand: h * safe is an fp32
// value, so the fp32 numerator n either equals it or differs by an ulp, and then n / safe differs from h by more than
// (1 + 2^-11) half ulps of h: the IEEE quotient and the corrected one (relative error below 2^-44 before its rounding,
// the remainder being exact) lie on the same side, and both equal h when n = h * safe. The largest code and zero bound
// the rest; adding 2^23 rounds half to even and leaves the code in the low byte. NaN does not reach this.
template <int BITS>
__device__ __forceinline__ uint32_t page_code(float x, const PageQuant& q) {
    const float c = corrected_quotient(x - q.low, q.safe, q.rcp);
    return f32_bits(__builtin_amdgcn_fmed3f(c, 0.0f, static_cast<float>((1 << BITS) - 1)) + 8388608.0f);
}

template <int BITS>
__device__ __forceinline__ uint32_t element_code(float x, const PageQuant& q, bool fast) {
    if (fast) return page_code<BITS>(x, q);
    return code_of(x, Quant{q.scale, q.low, q.safe}, (1 << BITS) - 1);
}

// The low bytes of four words as one.
__device__ __forceinline__ uint32_t low_bytes(uint32_t a, uint32_t b, uint32_t c, uint32_t d) {
    return __builtin_amdgcn_perm(b, a, 0x0C0C0400u) | __builtin_amdgcn_perm(d, c, 0x04000C0Cu);
}

__device__ __forceinline__ uint32_t pack_halves(float a, float b) {
    return f16_bits(a) | static_cast<uint32_t>(f16_bits(b)) << 16;
}

// x of lane l ^ STRIDE, for the strides between the lane groups of a wave.
template <int STRIDE>
__device__ __forceinline__ uint32_t lane_xor(uint32_t x) {
    if constexpr (STRIDE == 1) return dpp<0xB1>(x);   // quad_perm 1 0 3 2
    if constexpr (STRIDE == 2) return dpp<0x4E>(x);   // quad_perm 2 3 0 1
    if constexpr (STRIDE == 8) return dpp<0x128>(x);  // row_ror:8
    return static_cast<uint32_t>(__shfl_xor(static_cast<int>(x), STRIDE));
}

// Minimum and maximum with lane l ^ STRIDE, NaN if either is (NAN_WINS) or ignoring NaN. The halves and the odd and even
// rows of the wave come from a lane swap of the value with itself: both results hold one side each in every lane.
template <int STRIDE, bool NAN_WINS>
__device__ __forceinline__ void fold_min_max(float& lo, float& hi) {
    float lo2, hi2, lo1 = lo, hi1 = hi;
    if constexpr (STRIDE >= 16) {
        const auto swap = [](uint32_t x) {
            if constexpr (STRIDE == 32) return __builtin_amdgcn_permlane32_swap(x, x, false, false);
            else return __builtin_amdgcn_permlane16_swap(x, x, false, false);
        };
        const auto a = swap(f32_bits(lo)), b = swap(f32_bits(hi));
        lo1 = bits_f32(a[0]);
        lo2 = bits_f32(a[1]);
        hi1 = bits_f32(b[0]);
        hi2 = bits_f32(b[1]);
    } else {
        lo2 = bits_f32(lane_xor<STRIDE>(f32_bits(lo)));
        hi2 = bits_f32(lane_xor<STRIDE>(f32_bits(hi)));
    }
    lo = NAN_WINS ? min_nan(lo1, lo2) : fminf(lo1, lo2);
    hi = NAN_WINS ? max_nan(hi1, hi2) : fmaxf(hi1, hi2);
}

// Codes of one page's keys by one wave: lane (c, g) = (l % C, l / C) holds channels 8 c .. 8 c + 7 of tokens i T + g,
// so the codes of a load's tokens are contiguous over the wave. The channels' extremes fold over the lane groups.
template <int D, int BITS, int FMT>
__device__ __forceinline__ void quantize_keys_wave(const KiviQuantParams& p, const uint16_t* src, uint8_t* blk,
                                                   int lane) {
    constexpr int C = D / 8, T = 64 / C, N = KPAGE / T;
    constexpr KiviLayout L{D, BITS};
    const int c = lane % C, g = lane / C;
    uint4 raw[N];
#pragma unroll
    for (int i = 0; i < N; ++i) raw[i] = stream_load16(src + (i * T + g) * p.ss_t + 8 * c);
    float lo[8], hi[8];
    PageQuant q[8];
    const auto extremes = [&](auto nan_wins) __attribute__((always_inline)) {
        constexpr bool NW = decltype(nan_wins)::value;
#pragma unroll
        for (int i = 0; i < N; ++i) {
            float x[8];
            unpack8<FMT>(raw[i], x);
#pragma unroll
            for (int k = 0; k < 8; ++k) {
                lo[k] = i == 0 ? x[k] : (NW ? min_nan(lo[k], x[k]) : fminf(lo[k], x[k]));
                hi[k] = i == 0 ? x[k] : (NW ? max_nan(hi[k], x[k]) : fmaxf(hi[k], x[k]));
            }
        }
#pragma unroll
        for (int k = 0; k < 8; ++k) {
            if constexpr (C <= 8) fold_min_max<8, NW>(lo[k], hi[k]);
            fold_min_max<16, NW>(lo[k], hi[k]);
            fold_min_max<32, NW>(lo[k], hi[k]);
        }
    };
    extremes(std::true_type{});
    bool ok = true;
#pragma unroll
    for (int k = 0; k < 8; ++k) ok &= page_quant<BITS>(lo[k], hi[k], q[k]);
    const bool fast = __ballot(!ok) == 0;
    if (!fast) {
        extremes(std::false_type{});
#pragma unroll
        for (int k = 0; k < 8; ++k) {
            // fminf of one NaN alone keeps it: an all-NaN channel has the extremes of no element
            const Quant e = make_quant(lo[k] == lo[k] ? lo[k] : INFINITY, hi[k] == hi[k] ? hi[k] : -INFINITY,
                                       (1 << BITS) - 1, p.overflow);
            q[k] = PageQuant{e.scale, e.low, e.safe, 0.0f};
        }
    }
    if (g == 0)
        *reinterpret_cast<uint4*>(blk + L.k_scale() + 16 * c) =
            make_uint4(pack_halves(q[0].scale, q[1].scale), pack_halves(q[2].scale, q[3].scale),
                       pack_halves(q[4].scale, q[5].scale), pack_halves(q[6].scale, q[7].scale));
    else if (g == 1)
        *reinterpret_cast<uint4*>(blk + L.k_zero() + 16 * c) =
            make_uint4(pack_halves(q[0].low, q[1].low), pack_halves(q[2].low, q[3].low),
                       pack_halves(q[4].low, q[5].low), pack_halves(q[6].low, q[7].low));
    uint32_t word[N];
    const auto encode = [&](auto is_fast) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < N; ++i) {
            float x[8];
            unpack8<FMT>(raw[i], x);
            uint32_t t[4];
#pragma unroll
            for (int k = 0; k < 4; ++k)
                t[k] = element_code<BITS>(x[k + 4], q[k + 4], decltype(is_fast)::value) << BITS |
                       element_code<BITS>(x[k], q[k], decltype(is_fast)::value);
            word[i] = low_bytes(t[0], t[1], t[2], t[3]);
        }
    };
    if (fast) encode(std::true_type{});
    else encode(std::false_type{});
    uint32_t* codes = reinterpret_cast<uint32_t*>(blk + L.k_codes());
    if constexpr (BITS == 4) {
#pragma unroll
        for (int i = 0; i < N; ++i) codes[(i * T + g) * (D / 8) + c] = word[i];
    } else {
        // a word holds 16 channels, two lanes' worth: the even lane writes the first half of the tokens, the odd lane
        // the others
        const bool odd = c & 1;
#pragma unroll
        for (int i = 0; i < N / 2; ++i) {
            const uint32_t mine = odd ? word[i + N / 2] : word[i];
            const uint32_t theirs = lane_xor<1>(odd ? word[i] : word[i + N / 2]);
            codes[((i + (odd ? N / 2 : 0)) * T + g) * (D / 16) + c / 2] = odd ? theirs | mine << 4 : mine | theirs << 4;
        }
    }
}

// Codes of tokens [lo_t, hi_t) of one page's values (of page token 0 at src) by one wave: lane (c, g) holds channels 8 c
// .. 8 c + 7 of the N consecutive tokens g N .., so a word's tokens of a channel lie in one lane or in LW lanes of
// stride C, and a token's 32-channel group in four neighbouring lanes. The page's other tokens keep their codes.
template <int D, int BITS, int FMT>
__device__ __forceinline__ void quantize_values_wave(const KiviQuantParams& p, const uint16_t* src, uint8_t* blk,
                                                     int lane, int lo_t, int hi_t) {
    constexpr int C = D / 8, N = KPAGE * C / 64, LW = 32 / BITS / N;
    constexpr int SUB = BITS * N / 4;  // bits per byte of a lane's share of a word
    constexpr KiviLayout L{D, BITS};
    const int c = lane % C, g = lane / C;
    uint4 raw[N];
#pragma unroll
    for (int i = 0; i < N; ++i)
        raw[i] = stream_load16(src + min(max(g * N + i, lo_t), hi_t - 1) * p.ss_t + 8 * c);
    PageQuant q[N];
    const auto quantize = [&](auto nan_wins) __attribute__((always_inline)) {
        constexpr bool NW = decltype(nan_wins)::value;
        bool ok = true;
#pragma unroll
        for (int i = 0; i < N; ++i) {
            float x[8];
            unpack8<FMT>(raw[i], x);
            float lo = x[0], hi = x[0];
#pragma unroll
            for (int k = 1; k < 8; ++k) {
                lo = NW ? min_nan(lo, x[k]) : fminf(lo, x[k]);
                hi = NW ? max_nan(hi, x[k]) : fmaxf(hi, x[k]);
            }
            fold_min_max<1, NW>(lo, hi);
            fold_min_max<2, NW>(lo, hi);
            if constexpr (NW) {
                ok &= page_quant<BITS>(lo, hi, q[i]);
            } else {
                const Quant e = make_quant(lo == lo ? lo : INFINITY, hi == hi ? hi : -INFINITY, (1 << BITS) - 1,
                                           p.overflow);
                q[i] = PageQuant{e.scale, e.low, e.safe, 0.0f};
            }
        }
        return ok;
    };
    const bool fast = __ballot(!quantize(std::true_type{})) == 0;
    if (!fast) quantize(std::false_type{});
    uint32_t word[8];
    const auto encode = [&](auto is_fast) __attribute__((always_inline)) {
        uint32_t t[8][4];
#pragma unroll
        for (int i = 0; i < N; ++i) {
            float x[8];
            unpack8<FMT>(raw[i], x);
#pragma unroll
            for (int k = 0; k < 8; ++k) {
                const uint32_t code = element_code<BITS>(x[k], q[i], decltype(is_fast)::value);
                if (i < 4) t[k][i] = code;
                else t[k][i & 3] |= code << BITS;
            }
        }
#pragma unroll
        for (int k = 0; k < 8; ++k) word[k] = low_bytes(t[k][0], t[k][1], t[k][2], t[k][3]);
    };
    if (fast) encode(std::true_type{});
    else encode(std::false_type{});
    const int part = g % LW;  // which of a word's lanes this is: it writes channels 8 / LW part ..
    if constexpr (LW > 1) {
#pragma unroll
        for (int k = 0; k < 8; ++k) word[k] <<= SUB * part;
        if constexpr (LW == 4) {
#pragma unroll
            for (int k = 0; k < 8; ++k) word[k] |= lane_xor<C>(word[k]);
#pragma unroll
            for (int k = 0; k < 8; ++k) word[k] |= lane_xor<2 * C>(word[k]);
        } else {
#pragma unroll
            for (int k = 0; k < 8; ++k) word[k] |= lane_xor<C>(word[k]);
        }
    }
    const int first = g * N;  // the lane's tokens
    constexpr int W = 8 / LW;
    uint32_t* codes = reinterpret_cast<uint32_t*>(blk + L.v_codes()) +
                      ((g / LW) * 16 + 8 * (c & 1) + W * part) * (D / 16) + c / 2;
    uint16_t* params = reinterpret_cast<uint16_t*>(blk + (c & 1 ? L.v_zero() : L.v_scale())) + c / 4 * KPAGE + first;
    uint32_t mine[W];
#pragma unroll
    for (int k = 0; k < W; ++k) {
        mine[k] = word[k];
#pragma unroll
        for (int j = 1; j < LW; ++j) mine[k] = part == j ? word[W * j + k] : mine[k];
    }
    if (lo_t == 0 && hi_t == KPAGE) {
#pragma unroll
        for (int k = 0; k < W; ++k) codes[k * (D / 16)] = mine[k];
        if ((c & 3) < 2) {
            uint32_t h[N / 2];
#pragma unroll
            for (int i = 0; i < N / 2; ++i)
                h[i] = c & 1 ? pack_halves(q[2 * i].low, q[2 * i + 1].low)
                             : pack_halves(q[2 * i].scale, q[2 * i + 1].scale);
            if constexpr (N == 8) *reinterpret_cast<uint4*>(params) = make_uint4(h[0], h[1], h[2], h[3]);
            else *reinterpret_cast<uint2*>(params) = make_uint2(h[0], h[1]);
        }
        return;
    }
    uint32_t keep = 0;  // bits of the word's tokens outside the range
    const int word_first = g / LW * LW * N;
#pragma unroll
    for (int e = 0; e < 32 / BITS; ++e)
        if (word_first + e < lo_t || word_first + e >= hi_t)
            keep |= ((1u << BITS) - 1) << (8 * (e & 3) + (e >> 2) * BITS);
    if (keep != 0xFFFFFFFFu) {
#pragma unroll
        for (int k = 0; k < W; ++k) codes[k * (D / 16)] = (codes[k * (D / 16)] & keep) | (mine[k] & ~keep);
    }
    if ((c & 3) < 2) {
#pragma unroll
        for (int i = 0; i < N; ++i)
            if (first + i >= lo_t && first + i < hi_t) params[i] = f16_bits(c & 1 ? q[i].low : q[i].scale);
    }
}

// Four waves per workgroup, each one page of (row, KV head) blockIdx.x.
template <int D, int BITS, int FMT, bool KEYS>
__global__ __launch_bounds__(256) void kivi_quant_pages_kernel(KiviQuantParams p) {
    const int row = blockIdx.x;
    const int b = row / p.kv_heads, h = row % p.kv_heads;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int from = p.from[b], to = p.to[b];
    const int page = from / KPAGE + static_cast<int>(blockIdx.y) * 4 + wave;
    const int t0 = page * KPAGE;
    const int lo_t = max(from - t0, 0), hi_t = min(to - t0, KPAGE);
    if (KEYS ? t0 + KPAGE > to : lo_t >= hi_t) return;
    uint8_t* blk = page_block(p, b, h, page);
    if (!blk) return;
    const int slot = p.src_ring > 0 ? t0 % p.src_ring : t0 - p.src_start;
    const uint16_t* src = static_cast<const uint16_t*>(p.src) + b * p.ss_b + h * p.ss_h + slot * p.ss_t;
    const int lane = threadIdx.x & 63;
    if constexpr (KEYS) quantize_keys_wave<D, BITS, FMT>(p, src, blk, lane);
    else quantize_values_wave<D, BITS, FMT>(p, src, blk, lane, lo_t, hi_t);
}

// Whether a page can be read as 16-byte loads of 8 channels and its tokens lie in one run of the source.
bool wave_pages(const KiviQuantParams& p) {
    return (p.src_format == BF16 || p.src_format == FP16) && p.ss_d == 1 &&
           ((p.ss_b | p.ss_h | p.ss_t) & 7) == 0 && (reinterpret_cast<uintptr_t>(p.src) & 15) == 0 &&
           (reinterpret_cast<uintptr_t>(p.blocks) & 15) == 0 && p.src_ring % KPAGE == 0;
}

template <bool KEYS>
void launch_wave_pages(const KiviQuantParams& p, dim3 grid, hipStream_t stream) {
    const auto by_format = [&](auto dim, auto bits) {
        if (p.src_format == BF16)
            hipLaunchKernelGGL((kivi_quant_pages_kernel<dim.value, bits.value, BF16, KEYS>), grid, dim3(256), 0, stream, p);
        else
            hipLaunchKernelGGL((kivi_quant_pages_kernel<dim.value, bits.value, FP16, KEYS>), grid, dim3(256), 0, stream, p);
    };
    const auto by_bits = [&](auto dim) {
        if (p.bits == 2) by_format(dim, std::integral_constant<int, 2>{});
        else by_format(dim, std::integral_constant<int, 4>{});
    };
    if (p.head_dim == 64) by_bits(std::integral_constant<int, 64>{});
    else by_bits(std::integral_constant<int, 128>{});
}

}  // namespace

int kivi_schedule(const int32_t* committed, int residual, int32_t* keys_quantized, int32_t* values_quantized,
                  int32_t* ranges, int batch, hipStream_t stream) {
    hipLaunchKernelGGL(kivi_schedule_kernel, dim3((batch + 255) / 256), dim3(256), 0, stream, committed, residual,
                       keys_quantized, values_quantized, ranges, batch);
    return check_launch("kivi_schedule_kernel");
}

int kivi_ring_write(const KiviRingParams& p, hipStream_t stream) {
    if (p.tokens == 0) return 0;
    if (ring_windows(p)) {
        dim3 grid, block;
        window_launch(p.tokens, static_cast<int64_t>(p.kv_heads) * p.head_dim, grid, block);
        hipLaunchKernelGGL(kivi_ring_window_kernel, grid, block, 0, stream, p);
        return check_launch("kivi_ring_window_kernel");
    }
    hipLaunchKernelGGL(kivi_ring_kernel, dim3(p.tokens), dim3(256), 0, stream, p);
    return check_launch("kivi_ring_kernel");
}

int kivi_quantize(const KiviQuantParams& p, int kind, int max_tokens, hipStream_t stream) {
    const int pages = (max_tokens + KPAGE - 1) / KPAGE + 1;  // a range need not start at a page boundary
    if (wave_pages(p)) {
        const dim3 grid(p.batch * p.kv_heads, (pages + 3) / 4);
        if (kind == 0) launch_wave_pages<true>(p, grid, stream);
        else launch_wave_pages<false>(p, grid, stream);
        return check_launch("kivi_quant_pages_kernel");
    }
    dim3 grid(p.batch * p.kv_heads, pages);
    if (kind == 0)
        hipLaunchKernelGGL(kivi_quant_keys_kernel, grid, dim3(256), 0, stream, p);
    else
        hipLaunchKernelGGL(kivi_quant_values_kernel, grid, dim3(256), 0, stream, p);
    return check_launch(kind == 0 ? "kivi_quant_keys_kernel" : "kivi_quant_values_kernel");
}

}  // namespace eco
