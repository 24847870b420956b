// Which sequence and which of its query tiles a workgroup of prompt-portion attention has.
#pragma once

#include "common.h"

struct QueryTile {
    int b, tile, q_begin, q_len;       // (b < 0: a surplus workgroup)
};

// Number `place` of `places` where the sequences are handed out one after the other, the last tiles of TILE rows (a query is `rows` of them) first.
template <int TILE>
__device__ __forceinline__ QueryTile next_tile(const int* __restrict__ cu_q, int n_seqs, int rows, int place, int places) {
    int tile = places - 1 - place;
    for (int b = 0; b < n_seqs; ++b) {
        const int q_begin = cu_q[b], q_len = cu_q[b + 1] - q_begin, n = (q_len * rows + TILE - 1) / TILE;
        if (tile < n) return {b, tile, q_begin, q_len};
        tile -= n;
    }
    return {-1, 0, 0, 0};
}

// Number `place` where those that see most keys come first over all sequences: a causal tile's work grows with its position and
// workgroups start in the order of their numbers (on the compute units in turn, on the first again when all have one), so the long ones
// start first, and what shares a unit with them or starts behind them is short. Pairs of neighbouring tiles of a sequence, which see as
// many tiles of 128 keys, stay together. Handed out sequence by sequence, long tiles of some sequences start last: 64 queries a tile,
// 12 heads of 64 in bfloat16, 8 x 512 tokens 23.8 > 20.7 us, 4 x 512 with 25 heads 24.6 > 21.0. (Single tiles instead of pairs: 18.8 us for
// 17.4 at 2 x 1,024; with the second round's order turned around, so that the longest share with the shortest, slower than either.)
// A lane has a sequence (at most 64): all of a wavefront has to be here.
template <int TILE>
__device__ __forceinline__ QueryTile longest_tile(const int* __restrict__ cu_q, const int* __restrict__ ctx_len, int n_seqs, int rows, int place) {
    // The tiles of the lane's sequence have the numbers first, first + 1, ... up to `end`: as many tiles as would hold the rows in front of
    // them. Their pairs are counted through from the highest, so that the longest tiles know soonest; many of them are halved first.
    const int lane = threadIdx.x % MLLM_WAVE, b = min(lane, n_seqs - 1);
    const int q_begin = cu_q[b], q_len = cu_q[b + 1] - q_begin, n = lane < n_seqs ? (q_len * rows + TILE - 1) / TILE : 0;
    const int first = static_cast<int>(static_cast<long long>(ctx_len[b] - q_len) * rows / TILE), end = n > 0 ? first + n : 0;
    int high = (static_cast<int>(wave_max(static_cast<float>(end))) + 1) / 2;
    const bool many = high > 32;
    for (int low = 0; high - low > 32;) {
        const int middle = (low + high) / 2;
        if (static_cast<int>(wave_sum(static_cast<float>(min(n, max(end - 2 * middle, 0))))) > place) low = middle;      // (the tiles from it on)
        else high = middle;
    }
    if (many) place -= static_cast<int>(wave_sum(static_cast<float>(min(n, max(end - 2 * high, 0)))));
    auto below = [](unsigned long long lanes) {        // how many of them are in front of this one
        return static_cast<int>(__builtin_amdgcn_mbcnt_hi(static_cast<unsigned>(lanes >> 32), __builtin_amdgcn_mbcnt_lo(static_cast<unsigned>(lanes), 0)));
    };
    for (int pair = high - 1; pair >= 0; --pair) {
        const int last = min(end, 2 * pair + 2) - 1, here = max(0, last + 1 - max(first, 2 * pair));      // the lane's tiles of this pair
        const unsigned long long any = __ballot(here > 0), both = __ballot(here > 1);
        const int count = __popcll(any) + __popcll(both);
        if (place < count) {
            const int mine = place - below(any) - below(both);
            const int owner = __ffsll(static_cast<long long>(__ballot(mine >= 0 && mine < here))) - 1;
            return {owner, __builtin_amdgcn_readlane(last - first - mine, owner), __builtin_amdgcn_readlane(q_begin, owner), __builtin_amdgcn_readlane(q_len, owner)};
        }
        place -= count;
    }
    return {-1, 0, 0, 0};
}

// Whether the longest come first. With as many workgroups as compute units all start at once and the order is of no use, and finding it takes
// 0.1 to 0.5 us longer than a walk over few sequences; a walk over many is the longer way. From eight sequences on, and below from `from` on where
// a unit gets more than one workgroup. Longest first / in turn, us: bfloat16, 12 heads of 64, 8 portions of 37 to 177 tokens 7.3 / 7.7, 5 of 37 to 203
// 7.4 / 7.0, 25 heads 4 x 512 22.2 / 26.8, 2 x 512 16.1 / 15.7 (from four there); 32-bit, 12 heads of 64, 2 x 1,024 66 / 80, 3 x 512
// 33.2 / 35.5, 200 + 250 16.1 / 15.9; latent, 12 heads of 256 + 32, 2 x 1,024 59 / 61, 3 x 512 31.0 / 31.9, 200 + 250 16.9 / 16.3; 8 heads of 96, which run
// on the kernel for any head, the same within 3 % in either.
__host__ __device__ inline bool longest_first(int n_seqs, int from, long long workgroups) {
    return n_seqs <= MLLM_WAVE && (n_seqs >= 8 || (n_seqs >= from && workgroups > 256));
}

// Either, where the kernel decides.
template <int TILE>
__device__ __forceinline__ QueryTile query_tile(const int* __restrict__ cu_q, const int* __restrict__ ctx_len, int n_seqs, int rows, int place, int places) {
    return longest_first(n_seqs, 2, static_cast<long long>(gridDim.x) * gridDim.y) ? longest_tile<TILE>(cu_q, ctx_len, n_seqs, rows, place)
                                                                                   : next_tile<TILE>(cu_q, n_seqs, rows, place, places);
}
