// Windows of 16 tokens of a call that writes every token to a slot of its own (the paged append, the KIVI rings), where
// values are stored token-contiguous: a token alone is scattered over D short stores, 16 tokens in consecutive slots from
// a multiple of 16 on are 16- or 32-byte runs.
#pragma once

#include "common.hpp"

namespace eco {

// What one wave takes for tokens [first, first + 16): the run of 16 tokens in consecutive slots whose first token lies in
// the window (it may end in the next one), and the window's other tokens that lie in no such run. Every token with a
// slot is so taken by exactly one wave.
struct TokenWindow {
    int slots;      // lane l < 47: slot of token first - 15 + l, -1 for none
    int run;        // first token of the run, -1 for none
    uint32_t rest;  // bit j: token first + j, alone
    __device__ int slot(int token, int first) const { return __shfl(slots, token - first + 15); }
};

// slot_of(t): the slot of token t of the call, negative for none.
template <typename F>
__device__ __forceinline__ TokenWindow token_window(int first, int tokens, int lane, const F& slot_of) {
    const int t = first - 15 + lane;
    const int slot = lane < 47 && t >= 0 && t < tokens ? slot_of(t) : -1;
    const uint64_t held = __ballot(slot >= 0);
    // bit l: the token after lane l's takes the next slot
    const uint64_t link = __ballot(__shfl_down(slot, 1) == slot + 1 && lane < 46) & held;
    uint64_t chain = link & link >> 1;  // 2, 4, 8, then 15 links in a row
    chain &= chain >> 2;
    chain &= chain >> 4;
    chain &= chain >> 7;
    const uint64_t from = __ballot((slot & 15) == 0) & chain;
    uint64_t covered = from | from << 1;
    covered |= covered << 2;
    covered |= covered << 4;
    covered |= covered << 8;
    const uint32_t own = static_cast<uint32_t>(from >> 15) & 0xFFFFu;
    return {slot, own ? first + __builtin_ctz(own) : -1,
            static_cast<uint32_t>((held & ~covered) >> 15) & 0xFFFFu};
}

// The first token of the calling wave, and the launch: windows over x, one per wave, units of 128 channels over y. Tokens
// alone cost a wave up to 64 store requests each, so a call that does not fill the chip takes one wave per workgroup, and
// so more compute units (128 tokens of different pages, 8 KV heads of 128 channels, fp8 pages / rings: 8.6 / 10.2 us by four
// waves per workgroup, 6.0 / 6.2 by one, 4.7 / 5.4 with keys and values apart; 6.4 / 5.5 by the kernels of one workgroup
// per token); longer ones take four, whose windows are successive. By tokens (8 heads of 128, fp8 pages, us): one wave and
// two passes, four waves, the kernel of one workgroup per token, for tokens alone in their pages, prompts of 30, prompts
// of whole pages:
//     512   alone   6.5  10.3   9.3    30   5.4   7.0   8.8    pages   4.1   5.1   8.8
//    2048   alone  13.7  14.6  22.0    30   8.8   7.9  20.1    pages   5.0   5.7  19.7
//    8192   alone  44.5  45.3  62.5    30  22.2  19.5  60.4    pages  12.6  12.1  60.6
//   32768   alone   413   439   440    30  70.8  67.0   207    pages  41.2  40.5   206
// and rings in runs of 64 at 32768: 99.5, 63.9, 417. The two forms cross between 2048 and 8192 tokens (1024 and 4096 waves).
__device__ __forceinline__ int first_of_window() {
    return (blockIdx.x * (blockDim.x >> 6) + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6)) * 16;
}

__device__ __forceinline__ bool takes_keys() { return gridDim.z == 1 || blockIdx.z == 0; }
__device__ __forceinline__ bool takes_values() { return gridDim.z == 1 || blockIdx.z == 1; }

inline void window_launch(int tokens, int64_t channels, dim3& grid, dim3& block) {
    const int windows = (tokens + 15) / 16;
    const unsigned units = static_cast<unsigned>((channels + 127) / 128);
    const int waves = static_cast<int64_t>(windows) * units <= 1024 ? 1 : 4;
    grid = dim3(ceil_div(windows, waves), units, waves == 1 ? 2 : 1);
    block = dim3(64 * waves);
}

}  // namespace eco
