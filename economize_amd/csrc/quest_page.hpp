// The bounds of Quest pages of the paged key cache, by one wave (shared by the Quest kernels and the append that keeps
// the bounds up to date): the channel-wise smallest and largest stored key over a page's tokens, fp8 decoded exactly,
// written as bf16 (attention/quest.py:54-65).
#pragma once

#include <type_traits>

#include "common.hpp"
#include "quest.hpp"

namespace eco {

template <int FMT>
__device__ inline float quest_decode_elem(const uint8_t* p, int i) {
    if constexpr (FMT == BF16) {
        return bf16_to_f32(reinterpret_cast<const uint16_t*>(p)[i]);
    } else {
        // exact fp8 value, through the hardware converter (scale 1)
        const uint32_t word = p[i];
        if constexpr (FMT == FP8_E4M3)
            return __builtin_amdgcn_cvt_scalef32_f32_fp8(word, 1.0f, 0);
        else
            return __builtin_amdgcn_cvt_scalef32_f32_bf8(word, 1.0f, 0);
    }
}

// The bounds of Quest page qp of (row b, KV head kvh) by one wave, any head dim, alignment and values: lane l holds
// token l % 16 of the runs l / 16, l / 16 + 4, ... of every cache page of the Quest page; the 16 lanes of a run then
// reduce over the tokens.
template <int FMT>
__device__ inline void quest_bounds_of_page(const BoundsParams& p, int b, int qp, int kvh, int lane) {
    constexpr int ES = FMT == BF16 ? 2 : 1;
    constexpr int X = 16 / ES;  // channels per 16-byte run
    const int runs = p.head_dim / X;
    const int token = lane & 15;
    // every cache page of the Quest page must be held (a missing one leaves the bounds untouched)
    for (int s = 0; s < p.span; ++s) {
        const int lp = qp * p.span + s;
        if (lp >= p.bt_cols) return;
        const int phys = p.block_table[b * p.bt_stride + lp];
        if (phys < 0 || phys >= p.num_pages) return;
    }
    for (int r0 = 0; r0 < runs; r0 += 4) {
        const int run = r0 + (lane >> 4);
        float lo[X], hi[X];
#pragma unroll
        for (int i = 0; i < X; ++i) {
            lo[i] = INFINITY;
            hi[i] = -INFINITY;
        }
        if (run < runs) {
            for (int s = 0; s < p.span; ++s) {
                const int phys = p.block_table[b * p.bt_stride + qp * p.span + s];
                const uint8_t* src = p.k_cache + static_cast<int64_t>(phys) * p.kc_page + kvh * p.kc_head +
                                     (run * 16 + token) * 16;
                uint8_t raw[16];
                *reinterpret_cast<uint4*>(raw) = *reinterpret_cast<const uint4*>(src);
#pragma unroll
                for (int i = 0; i < X; ++i) {
                    const float v = quest_decode_elem<FMT>(raw, i);
                    lo[i] = fminf(lo[i], v);
                    hi[i] = fmaxf(hi[i], v);
                }
            }
        }
#pragma unroll
        for (int off = 1; off < 16; off <<= 1)
#pragma unroll
            for (int i = 0; i < X; ++i) {
                lo[i] = fminf(lo[i], __shfl_xor(lo[i], off));
                hi[i] = fmaxf(hi[i], __shfl_xor(hi[i], off));
            }
        if (run < runs && token == 0) {
            const int64_t at = b * p.sb_b + kvh * p.sb_h + qp * p.sb_p + run * X;
#pragma unroll
            for (int i = 0; i < X; ++i) {
                p.kmin[at + i] = f32_to_bf16(lo[i]);
                p.kmax[at + i] = f32_to_bf16(hi[i]);
            }
        }
    }
}

// ---- head dims 64, 128 and 256: packed minima and maxima ----------------------------------------------------------

typedef short i16x2 __attribute__((ext_vector_type(2)));

__device__ inline i16x2 as_i16x2(uint32_t x) { return __builtin_bit_cast(i16x2, x); }
__device__ inline uint32_t as_u32(i16x2 x) { return __builtin_bit_cast(uint32_t, x); }

// Two bf16 values as two int16 in the order of the floats (-0 below +0, a NaN beyond the infinity of its sign), and
// back: the map is its own inverse.
__device__ inline i16x2 ordered_bf16(i16x2 x) {
    const i16x2 sign = x >> static_cast<short>(15);
    return x ^ (sign & static_cast<short>(0x7FFF));
}

// Halves v[0 .. 2 N): the lane keeps the half its `upper` names, sends the other to its partner (a lane permutation
// that is its own inverse and pairs lanes of different `upper`) and takes the minimum with what the partner sent.
template <int CTRL, int N>
__device__ __forceinline__ void fold_min(const i16x2* v, bool upper, i16x2 (&out)[N]) {
#pragma unroll
    for (int i = 0; i < N; ++i) {
        const uint32_t a = as_u32(v[i]), b = as_u32(v[N + i]);
        const uint32_t received = dpp<CTRL>(upper ? a : b);
        out[i] = __builtin_elementwise_min(as_i16x2(upper ? b : a), as_i16x2(received));
    }
}

// Whether quest_bounds_pages takes this call: the bounds are stored as 4-byte pairs, and a Quest page's cache pages fit
// the window of 64 block-table entries.
__device__ inline bool quest_bounds_packed(const BoundsParams& p) {
    return p.span <= 64 && ((reinterpret_cast<uintptr_t>(p.kmin) | reinterpret_cast<uintptr_t>(p.kmax)) & 3) == 0 &&
           ((p.sb_b | p.sb_h | p.sb_p) & 1) == 0;
}

// The bounds of Quest pages [q0, q1) of (row b, KV head kvh) by one wave. Bound by reading the keys once; what kept a
// wave from that is the reduction over the 16 tokens of a page, which the lanes of a row of 16 hold. Two bf16 channels
// share a register as order-preserving int16 (one instruction per minimum or maximum of two channels), and the
// reduction halves the values a lane holds at every step instead of reducing each over all 16 lanes: the lower 8
// lanes of a row take the minima and the upper 8 the maxima (as minima of the complement), then each of three more
// steps keeps half of the channels (DPP lane exchanges), so that every lane ends with D / 64 finished pairs and the
// wave writes the page's bounds with contiguous stores. The next cache page's loads are in flight while a page is
// reduced, and the block table comes 64 entries per load. A page with a NaN (an extreme beyond infinity) is redone by
// quest_bounds_of_page, whose fp32 minimum and maximum ignore NaN. 32,768 tokens of 64 (row, KV head) pairs, bf16, D =
// 128 (604 MB): 121 us (5.0 TB/s), against 2123 us with a page reduced by 256 lane shuffles after dependent loads, in
// eight waves per (row, KV head).
template <int FMT, int D>
__device__ __forceinline__ void quest_bounds_pages(const BoundsParams& p, int b, int kvh, int q0, int q1, int lane) {
    constexpr int ES = FMT == BF16 ? 2 : 1;
    constexpr int NL = D * ES / 64;     // 16-byte loads per lane and cache page: run 4 u + lane / 16 of token lane % 16
    constexpr int DPL = 8 / ES;         // bf16 pairs per load
    constexpr int V = NL * DPL;         // pairs a lane holds: D / 8
    constexpr int F = V / 8;            // finished pairs per lane
    const int token = lane & 15, g = lane >> 4;
    const bool kind = token & 8;        // maxima
    const bool b2 = token & 4, b1 = token & 2, b0 = token & 1;
    const int steps = (q1 - q0) * p.span;  // cache pages
    if (steps <= 0) return;
    const uint8_t* keys = p.k_cache + kvh * p.kc_head + (g * 16 + token) * 16;
    const int32_t* table = p.block_table + b * p.bt_stride;
    int wbase = 0, window = -1;  // lane i: the cache page of table entry wbase + i, -1 for none
    auto load_window = [&](int first) __attribute__((always_inline)) {
        wbase = first;
        const int lp = first + lane;
        const int phys = lp < p.bt_cols && lp < q1 * p.span ? table[lp] : -1;
        window = phys < p.num_pages ? phys : -1;
    };
    auto issue = [&](int lp, uint4 (&raw)[NL]) __attribute__((always_inline)) {
        const int phys = __builtin_amdgcn_readlane(window, lp - wbase);
        const uint8_t* src = keys + static_cast<int64_t>(max(phys, 0)) * p.kc_page;
#pragma unroll
        for (int u = 0; u < NL; ++u) raw[u] = stream_load16(src + u * 1024);
    };
    load_window(q0 * p.span);
    uint4 next[NL];
    issue(wbase, next);
    i16x2 lo[V], hi[V];
    int s = 0;  // cache page within the Quest page
    bool held = true;
    for (int i = 0; i < steps; ++i) {
        const int lp = q0 * p.span + i;
        held = held && __builtin_amdgcn_readlane(window, lp - wbase) >= 0;
        uint4 raw[NL];
#pragma unroll
        for (int u = 0; u < NL; ++u) raw[u] = next[u];
        if (i + 1 < steps) {
            if (lp + 1 - wbase >= 64) load_window(lp + 1);
            issue(lp + 1, next);
        }
#pragma unroll
        for (int u = 0; u < NL; ++u) {
            const uint32_t w[4] = {raw[u].x, raw[u].y, raw[u].z, raw[u].w};
#pragma unroll
            for (int j = 0; j < DPL; ++j) {
                uint32_t pair;
                if constexpr (FMT == BF16) {
                    pair = w[j];
                } else {
                    bf16x2 x;
                    if constexpr (FMT == FP8_E4M3)
                        x = (j & 1) ? __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(w[j / 2], 1.0f, true)
                                    : __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(w[j / 2], 1.0f, false);
                    else
                        x = (j & 1) ? __builtin_amdgcn_cvt_scalef32_pk_bf16_bf8(w[j / 2], 1.0f, true)
                                    : __builtin_amdgcn_cvt_scalef32_pk_bf16_bf8(w[j / 2], 1.0f, false);
                    pair = __builtin_bit_cast(uint32_t, x);
                }
                const i16x2 x = ordered_bf16(as_i16x2(pair));
                i16x2 &l = lo[u * DPL + j], &h = hi[u * DPL + j];
                l = s == 0 ? x : __builtin_elementwise_min(l, x);
                h = s == 0 ? x : __builtin_elementwise_max(h, x);
            }
        }
        if (++s < p.span) continue;
        s = 0;
        i16x2 v8[V], v4[V / 2], v2[V / 4], v1[F];
#pragma unroll
        for (int j = 0; j < V; ++j) {
            const uint32_t keep = kind ? ~as_u32(hi[j]) : as_u32(lo[j]);
            const uint32_t sent = kind ? as_u32(lo[j]) : ~as_u32(hi[j]);
            v8[j] = __builtin_elementwise_min(as_i16x2(keep), as_i16x2(dpp<0x128>(sent)));  // row_ror:8
        }
        fold_min<0x141, V / 2>(v8, b2, v4);  // row_half_mirror: lane i of 8 with 7 - i
        fold_min<0x1B, V / 4>(v4, b1, v2);   // quad_perm 3 2 1 0
        fold_min<0xB1, F>(v2, b0, v1);       // quad_perm 1 0 3 2
        const int qp = q0 + i / p.span;
        bool nan = false;
        i16x2 x[F];  // ordered bf16 pairs
#pragma unroll
        for (int j = 0; j < F; ++j) {
            x[j] = as_i16x2(kind ? ~as_u32(v1[j]) : as_u32(v1[j]));
            nan |= kind ? x[j][0] > 0x7F80 || x[j][1] > 0x7F80 : x[j][0] < -0x7F81 || x[j][1] < -0x7F81;
        }
        // (one of the two writes the page: the other's lanes would store to the same bounds in no stated order)
        if (held && __ballot(nan) != 0) {
            quest_bounds_of_page<FMT>(p, b, qp, kvh, lane);
        } else if (held) {
            uint16_t* out = (kind ? p.kmax : p.kmin) + b * p.sb_b + kvh * p.sb_h + qp * p.sb_p;
            const int first = (b2 * 4 + b1 * 2 + b0) * F;
#pragma unroll
            for (int j = 0; j < F; ++j) {
                const int v = first + j;
                const int channel = (4 * (v / DPL) + g) * (2 * DPL) + 2 * (v % DPL);
                *reinterpret_cast<uint32_t*>(out + channel) = as_u32(ordered_bf16(x[j]));
            }
        }
        held = true;
    }
}

// The bounds of Quest pages [q0, q1) of (row b, KV head kvh): D the head dim of the packed form, 0 for any other.
template <int FMT, int D>
__device__ __forceinline__ void quest_bounds_range(const BoundsParams& p, int b, int kvh, int q0, int q1, int lane) {
    if constexpr (D > 0) {
        if (quest_bounds_packed(p)) {
            quest_bounds_pages<FMT, D>(p, b, kvh, q0, q1, lane);
            return;
        }
    }
    for (int qp = q0; qp < q1; ++qp) quest_bounds_of_page<FMT>(p, b, qp, kvh, lane);
}

// Calls f(format, dim) with the instance of a call: dim 64, 128 or 256, 0 for any other head dim. False for a format
// that holds no keys.
template <typename F>
bool quest_bounds_dispatch(int format, int head_dim, const F& f) {
    auto by_dim = [&](auto fmt) {
        switch (head_dim) {
            case 64: f(fmt, std::integral_constant<int, 64>{}); break;
            case 128: f(fmt, std::integral_constant<int, 128>{}); break;
            case 256: f(fmt, std::integral_constant<int, 256>{}); break;
            default: f(fmt, std::integral_constant<int, 0>{}); break;
        }
        return true;
    };
    switch (format) {
        case BF16: return by_dim(std::integral_constant<int, BF16>{});
        case FP8_E4M3: return by_dim(std::integral_constant<int, FP8_E4M3>{});
        case FP8_E5M2: return by_dim(std::integral_constant<int, FP8_E5M2>{});
        default: return false;
    }
}

}  // namespace eco
