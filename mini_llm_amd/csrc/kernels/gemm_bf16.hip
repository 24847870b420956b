// bf16 matrix products on the MFMA units of gfx950, fp32 accumulation:
//   C[M,N] = A[M,K] * W[N,K]^T + bias, with the epilogues of common.h fused
// (bias, GELU, residual add into the fp32 stream, fp32 store for logits).
// Both operands are k-contiguous, so each lane feeds v_mfma_f32_32x32x16_bf16 with one
// 16-byte LDS read per operand. Many rows: tiles of both matrices in stages of LDS, loaded
// several k tiles ahead; few rows: the weights streamed once (each described below).
//
// It stands where the reference has its tiled SGEMM with fused store path
// (/root/reference/src/kernels/gemm.cu:394-580, epilogue :534-564).
// Requires K % 8 == 0 and 16-byte aligned rows; any M and N.
#include "common.h"
#include "lds_loads.h"

#include <algorithm>
#include <type_traits>

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x16 __attribute__((ext_vector_type(16)));

#define N_XCD 8       // accelerator dies of an MI355X, each with its own L2

// ---------------------------------------------------------------------------------------------
// Many rows (prefill): WM x WN wavefronts, each TM x TN MFMA tiles of 32x32. A k tile of both matrices lies in one of STAGES stages of
// LDS, which loads fill without passing through registers (STAGES - 1 tiles ahead; one barrier a k tile); what an LDS read needs to be free of
// bank conflicts is in the choice of the piece a lane asks for. For a long K two such groups of wavefronts may share a workgroup's
// tile, each on half of a twice as wide k tile. The weight fragment is the MFMA's A operand, so a lane's accumulator registers hold 4
// consecutive columns of one output row; the epilogue turns that, through LDS, into stores of whole rows.
// Bound by the rate at which a compute unit takes tiles from its L2 and by what the matrix units wait around the barriers: at 2,048 x
// 2,304 x 3,072 the products alone take 24.8 us, the loads alone 25.6, both 30.5. (With tiles loaded into registers and written to LDS from there,
// at 78 bytes a clock, 37.5. us, so / now, alone with weights and rows that no cache holds: 2,048 x 2,304 x 768 14.9 / 12.7, 2,048 x 3,072
// x 768 15.7 / 14.0, 2,048 x 4,800 x 1,600 42.1 / 36.5, 2,048 x 6,400 x 1,600 53.8 / 45.9, 560 x 3,072 x 768 7.9 / 7.3, 256 x 3,072 x 768 6.4 /
// 6.2; in a step of 2,048 rows, where a kernel before wrote the rows, 18.3 / 15.4, 18.2 / 17.1, 52.9 / 40.3, 64.6 / 50.9. Long sums in
// halves gain in a step only: 2,048 x 1,600 x 6,400 55.2 / 57.8 alone, 64.3 / 59.3 there.)
// ---------------------------------------------------------------------------------------------
// Optional second destination of a plain bf16 store: columns [q_cols, q_cols + kv_dim) of output row
// m also go to row slots[m] of the key pages and the next kv_dim columns to the value pages (the
// fused QKV product writes a step's keys and values where attention reads them;
// /root/reference/src/kernels/prefill/append_kv.cu:28-46 is a kernel of its own). slots == nullptr: off.
struct KvScatter {
    const int* slots;
    bf16_t* k_pages;
    bf16_t* v_pages;
    int q_cols, kv_dim;
};

// Two maps of one input whose results meet in a gated activation (EPI_GATED): W holds the gate's rows, `up` the other's (row
// stride and count alike), and what leaves the kernel is g sigmoid(alpha g) (u + 1) with g = min(gate, limit) and
// u = clamp(up, -limit, limit), from the fp32 sums.
struct GatedPair {
    const bf16_t* up;
    float limit, alpha;
};
__device__ __forceinline__ float gated_value(float g, float u, const GatedPair& p) {
    g = fminf(g, p.limit);
    u = fminf(fmaxf(u, -p.limit), p.limit);
    return g * __builtin_amdgcn_rcpf(1.f + __expf(-p.alpha * g)) * (u + 1.f);
}

// What a kernel of one mode takes beside its matrices.
template <int MODE> struct TiledExtra { typedef KvScatter type; };
template <> struct TiledExtra<EPI_GATED> { typedef GatedPair type; };
template <> struct TiledExtra<EPI_THROUGH> { typedef MllmStreamAdd type; };

// EPI_THROUGH for 4 consecutive columns of one row: the stream's row at x, columns n..n+3 of which n_left exist.
__device__ __forceinline__ void through4(float* x, size_t idx, int n, const float (&v)[4], bool vec, int n_left, const MllmStreamAdd& add) {
    const bool has = add.norm.weight != nullptr, has_next = add.next.weight != nullptr;
    const float alpha = has ? add.norm.alpha[0] : 0.f, alpha2 = has_next ? add.next.alpha[0] : 0.f;
    bf16_t* copy = static_cast<bf16_t*>(add.copy);          // (rows as far apart as the stream's)
    if (vec && n_left >= 4) {
        const float4 old = *reinterpret_cast<const float4*>(x + idx);
        float w[4] = {1.f, 1.f, 1.f, 1.f}, b[4] = {0.f, 0.f, 0.f, 0.f};
        if (has) {
            const float4 w4 = *reinterpret_cast<const float4*>(add.norm.weight + n), b4 = *reinterpret_cast<const float4*>(add.norm.bias + n);
            w[0] = w4.x; w[1] = w4.y; w[2] = w4.z; w[3] = w4.w; b[0] = b4.x; b[1] = b4.y; b[2] = b4.z; b[3] = b4.w;
        }
        float o[4] = {old.x, old.y, old.z, old.w};
#pragma unroll
        for (int e = 0; e < 4; ++e) o[e] += mllm_norm_column(v[e], has, alpha, {w[e], b[e]});
        *reinterpret_cast<float4*>(x + idx) = make_float4(o[0], o[1], o[2], o[3]);
        if (copy == nullptr) return;
        if (has_next) {
            const float4 w4 = *reinterpret_cast<const float4*>(add.next.weight + n), b4 = *reinterpret_cast<const float4*>(add.next.bias + n);
            o[0] = mllm_norm_column(o[0], true, alpha2, {w4.x, b4.x}); o[1] = mllm_norm_column(o[1], true, alpha2, {w4.y, b4.y});
            o[2] = mllm_norm_column(o[2], true, alpha2, {w4.z, b4.z}); o[3] = mllm_norm_column(o[3], true, alpha2, {w4.w, b4.w});
        }
        *reinterpret_cast<uint2*>(copy + idx) = make_uint2(pack_bf16x2(o[0], o[1]), pack_bf16x2(o[2], o[3]));
    } else {
        for (int e = 0; e < n_left; ++e) {
            float o = x[idx + e] + mllm_norm_column(v[e], has, alpha, {has ? add.norm.weight[n + e] : 1.f, has ? add.norm.bias[n + e] : 0.f});
            x[idx + e] = o;
            if (copy == nullptr) continue;
            if (has_next) o = mllm_norm_column(o, true, alpha2, {add.next.weight[n + e], add.next.bias[n + e]});
            copy[idx + e] = float_to_bf16(o);
        }
    }
}

template <int MODE>
__device__ __forceinline__ float activated(float v) {
    return MODE == EPI_GELU_TANH ? gelu_tanh(v) : MODE == EPI_GELU_ERF ? gelu_erf(v) : MODE == EPI_RELU2 ? relu2(v) : v;
}
template <int MODE>
__device__ __forceinline__ void store4(void* C, size_t idx, const float (&v)[4], bool vec, int n_left) {
    // v: 4 consecutive columns of one row, bias already added; n_left: columns that exist (1..4)
    float o[4];
#pragma unroll
    for (int e = 0; e < 4; ++e)
        o[e] = activated<MODE>(v[e]);
    if (MODE == EPI_ADD_RESIDUAL || MODE == EPI_STORE_F32) {
        float* c = static_cast<float*>(C) + idx;
        if (vec && n_left >= 4) {
            float4 r = make_float4(o[0], o[1], o[2], o[3]);
            if (MODE == EPI_ADD_RESIDUAL) {
                const float4 old = *reinterpret_cast<const float4*>(c);
                r.x += old.x; r.y += old.y; r.z += old.z; r.w += old.w;
            }
            *reinterpret_cast<float4*>(c) = r;
        } else {
            for (int e = 0; e < n_left; ++e) c[e] = (MODE == EPI_ADD_RESIDUAL ? c[e] : 0.f) + o[e];
        }
    } else {
        bf16_t* c = static_cast<bf16_t*>(C) + idx;
        if (vec && n_left >= 4) {
            uint2 pk;
            pk.x = pack_bf16x2(o[0], o[1]);
            pk.y = pack_bf16x2(o[2], o[3]);
            *reinterpret_cast<uint2*>(c) = pk;
        } else {
            for (int e = 0; e < n_left; ++e) c[e] = float_to_bf16(o[e]);
        }
    }
}

// How far apart (in elements) the rows of a matrix may lie for the 32-bit byte offsets from a tile's first row to the other 255 and a
// k tile's pieces. Beyond it (FAR) a lane forms 64-bit addresses, which only one shape of tile for either order of sums does: rows over 16 MiB
// apart have nothing else in common with what the prices know.
#define NEAR_ROWS (1 << 23)

template <int WM, int WN, int TM, int TN, int BK, int STAGES, int KG, bool HALVES, bool FAR, bool EDGE, int MODE>
__global__ void __launch_bounds__(WM * WN * KG * 64)
gemm_bf16_mfma(// The first 14 dwords arrive in registers with the wavefront: all that the first tiles' loads need. (K, the tile counts and their split
               // among the XCDs lay behind them and came from memory, 0.7 us in front of the first load.)
               const bf16_t* __restrict__ A, const bf16_t* __restrict__ W,
               const void* __restrict__ bias_or_up,        // (EPI_GATED: the second map)
               int lda, int ldw, int M, int N, int K, int xm_bits,
               void* __restrict__ C, int ldc, typename TiledExtra<MODE>::type kv) {
    // EPI_GATED: of a wavefront's TN column sub-tiles the even ones are the gate's and the odd ones the same 32 columns of the up
    // map, so that both values of an output lie in one register of one lane; N and the tile's columns count outputs.
    constexpr bool GATED = MODE == EPI_GATED, F32_OUT = MODE == EPI_ADD_RESIDUAL || MODE == EPI_STORE_F32 || MODE == EPI_THROUGH;
    static_assert(!GATED || TN % 2 == 0, "a wavefront holds whole pairs of sub-tiles");
    constexpr int PAIR = GATED ? 2 : 1;
    const float* bias = GATED ? nullptr : static_cast<const float*>(bias_or_up);
    // KG groups of WM x WN wavefronts share the tile: group g multiplies the g-th part of every k tile; their sums meet in LDS.
    constexpr int NW = WM * WN * KG, BM = WM * TM * 32, BN = WN * TN * 32, ROWS = BM + BN;
    constexpr int ROW_BYTES = BK * 2, PIECES = BK / 8;         // 16-byte pieces of a row of the k tile
    constexpr int ROWS_PER_LOAD = 64 / PIECES;
    constexpr int LOADS = ROWS / ROWS_PER_LOAD / NW;           // of a wavefront and k tile
    static_assert(LOADS * ROWS_PER_LOAD * NW == ROWS && BM % ROWS_PER_LOAD == 0 && (PIECES == 8 || PIECES == 16), "whole loads");
    static_assert(!GATED || 32 % ROWS_PER_LOAD == 0, "a load's rows belong to one map");
    constexpr int KS = BK / 16 / KG;                           // MFMA k steps of a group and k tile
    // HALVES: the 64-column blocks of K are summed in turn into two sums that are added at the end, as two groups (of 64 columns of a k
    // tile of 128 each) do: which products do is a matter of their sizes alone (the dispatch), and so is every result's rounding.
    static_assert(!HALVES || (KG == 1 && BK == 64), "one block a k tile");
    static_assert(KG == 1 || (KG == 2 && BK == 128), "a group, a block of 64");
    static_assert(KS % 2 == 0 && STAGES >= 3, "the k loop alternates two fragment sets and asks two tiles ahead");
    constexpr int STAGE_BYTES = ROWS * ROW_BYTES;
    constexpr bool APART = GATED && KG > 1;                    // both maps' sums go through LDS, as the groups' are still to be added
    constexpr int EC = TN / PAIR * 32, EPI_STRIDE = EC * (APART ? 2 : 1) + 4;    // columns a wavefront stores; floats between their rows in LDS
    constexpr int EPI_BYTES = NW * 32 * EPI_STRIDE * 4;
    constexpr int V = F32_OUT ? 4 : 8, PER_ROW = EC / V, STEPS = 32 / KG * PER_ROW / 64;      // columns a lane stores at a time
    static_assert(STEPS >= 1 && (KG == 1 || TM == 1), "two groups store half of the rows each");
    __shared__ __attribute__((aligned(16))) unsigned char smem[STAGES * STAGE_BYTES > EPI_BYTES ? STAGES * STAGE_BYTES : EPI_BYTES];
    __shared__ __attribute__((aligned(16))) float bias_s[BN];
    __shared__ int slot_s[BM];
    static_assert(NW * 64 >= BN && NW * 64 >= BM, "a thread a column's bias, a thread a row's slot");

    const int tid = threadIdx.x, lane = tid % 64;
    const int wid = __builtin_amdgcn_readfirstlane(tid / 64);
    const int kg = wid / (WM * WN), wave = wid % (WM * WN);    // k group; wavefront within it
    const int wm = wave / WN, wn = wave % WN;
    // Workgroups are handed to the 8 XCDs round-robin and every XCD has an L2 of its own, so the
    // tiles of one XCD (workgroup id % 8) form one compact rectangle of the output: the rows of A
    // and W it needs then fit in its L2 instead of every XCD streaming both matrices.
    const int xcd = blockIdx.x % N_XCD, local = blockIdx.x / N_XCD;
    const int tiles_m = (M + BM - 1) / BM, tiles_n = (N + BN / PAIR - 1) / (BN / PAIR);
    const int xn_bits = 3 - xm_bits;           // (8 XCDs)
    const int rect_m = (tiles_m + (1 << xm_bits) - 1) >> xm_bits, rect_n = (tiles_n + (1 << xn_bits) - 1) >> xn_bits;
    const int down = uniform_quotient(local, rect_n);
    const int tm = (xcd >> xn_bits) * rect_m + down, tn = (xcd & ((1 << xn_bits) - 1)) * rect_n + local - down * rect_n;
    if (local >= rect_m * rect_n || tm >= tiles_m || tn >= tiles_n) return;      // padding of the grid
    const int m0 = tm * BM, n0 = tn * (BN / PAIR);

    // A k tile in LDS is its rows one behind the other (A's, then W's), without gaps, as the loads leave it: a load covers
    // ROWS_PER_LOAD whole rows. Piece p of row r stands in place p ^ swizzle(r), so that the 16 lanes an LDS read serves at a time (16
    // rows, one piece) fall on 16 different groups of banks; a lane asks for the piece whose place is its own.
    auto swizzle = [](int row) { return PIECES == 8 ? (row >> 1) & 7 : row & 15; };
    const unsigned char* base[LOADS];      // (uniform: a wavefront's load lies in one matrix)
    typedef typename std::conditional<FAR, size_t, unsigned>::type Offset;
    Offset offset[LOADS];
#pragma unroll
    for (int q = 0; q < LOADS; ++q) {
        const int first = (wid * LOADS + q) * ROWS_PER_LOAD, row = first + lane / PIECES;
        // (rows beyond the matrices: the last one; what is computed from it is never stored)
        if (first < BM) {
            base[q] = reinterpret_cast<const unsigned char*>(A + static_cast<size_t>(m0) * lda);
            offset[q] = static_cast<Offset>(min(row, M - 1 - m0)) * lda * 2;
        } else {
            const int w_row = row - BM, n = GATED ? w_row / 64 * 32 + w_row % 32 : w_row;
            const bf16_t* map = W;
            if constexpr (GATED) map = (first - BM) / 32 % 2 ? static_cast<const bf16_t*>(bias_or_up) : W;
            base[q] = reinterpret_cast<const unsigned char*>(map + static_cast<size_t>(n0) * ldw);
            offset[q] = static_cast<Offset>(min(n, N - 1 - n0)) * ldw * 2;
        }
        offset[q] += (lane % PIECES ^ swizzle(row)) * 16;
    }
    const unsigned lds0 = static_cast<unsigned>(reinterpret_cast<uintptr_t>((__attribute__((address_space(3))) unsigned char*)smem));
    const int nk = (K + BK - 1) / BK, rest = K - (nk - 1) * BK;      // k tiles; columns of the last
    auto fetch = [&](int q, int t, int stage) {
        Offset at = offset[q];
        if (EDGE && t == nk - 1) {
            // (pieces beyond K: the row's last one, against zeros)
            const int piece = (lane % PIECES ^ swizzle((wid * LOADS + q) * ROWS_PER_LOAD + lane / PIECES)) * 16;
            at += min(piece, rest * 2 - 16) - piece;
        }
        load_to_lds(base[q] + static_cast<size_t>(t) * ROW_BYTES, at, lds0 + stage * STAGE_BYTES + (wid * LOADS + q) * 1024);
    };
    // What the epilogue adds, asked for first and put into LDS behind the k loop.
    float bias_r = 0.f;
    int slot_r = -1;
    if (bias != nullptr && tid < BN) bias_r = bias[min(n0 + tid, N - 1)];
    if constexpr (MODE == EPI_STORE)
        if (kv.slots != nullptr && tid < BM) slot_r = kv.slots[min(m0 + tid, M - 1)];
    // The stream's old values: here too, unless registers are short, otherwise all of 32 rows together in the epilogue.
    constexpr bool EARLY = MODE == EPI_ADD_RESIDUAL && !(HALVES && TM > 1);
    const bool vec = (ldc % 4 == 0) && ((reinterpret_cast<uintptr_t>(C) & 15) == 0), vec8 = vec && ldc % 8 == 0;
    float4 old[MODE == EPI_ADD_RESIDUAL ? (EARLY ? TM : 1) : 1][MODE == EPI_ADD_RESIDUAL ? STEPS : 1];
    auto fetch_old = [&](int i) {
#pragma unroll
        for (int it = 0; it < (MODE == EPI_ADD_RESIDUAL ? STEPS : 0); ++it) {
            const int idx = it * 64 + lane, m = m0 + (wm * TM + i) * 32 + 32 / KG * kg + idx / PER_ROW, n = n0 + wn * EC + idx % PER_ROW * V;
            float4& o = old[EARLY ? i : 0][it];
            o = make_float4(0.f, 0.f, 0.f, 0.f);
            if (vec && m < M && n + 4 <= N) o = *reinterpret_cast<const float4*>(static_cast<const float*>(C) + static_cast<size_t>(m) * ldc + n);
        }
    };
    if constexpr (EARLY) {
#pragma unroll
        for (int i = 0; i < TM; ++i) fetch_old(i);
    }
#pragma unroll
    for (int s = 0; s < STAGES - 1; ++s) {
        if (s >= nk) break;
#pragma unroll
        for (int q = 0; q < LOADS; ++q) fetch(q, s, s);
    }

    f32x16 acc[TM][TN], acc2[TM][TN];      // (acc2: only with HALVES)
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j)
#pragma unroll
            for (int r = 0; r < 16; ++r) acc[i][j][r] = acc2[i][j][r] = 0.f;
    // two sets of MFMA operands: the fragments of k step ks+1 are read while step ks multiplies. A lane reads 8 elements of row
    // lane % 32 of a sub-tile, from element 8 (lane / 32) of the k step on. (32 rows on the swizzle is the same.)
    const int a_row = wm * TM * 32 + lane % 32, w_row = BM + wn * TN * 32 + lane % 32;
    int a_at[KS], w_at[KS];
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) {
        const int piece = 2 * (kg * KS + ks) + lane / 32;
        a_at[ks] = a_row * ROW_BYTES + (piece ^ swizzle(a_row)) * 16;
        w_at[ks] = w_row * ROW_BYTES + (piece ^ swizzle(w_row)) * 16;
    }
    bf16x8 fa[2][TM], fb[2][TN];
    auto read_frags = [&](int stage_at, int ks, int set) {
#pragma unroll
        for (int i = 0; i < TM; ++i) fa[set][i] = *reinterpret_cast<const bf16x8*>(smem + stage_at + a_at[ks] + i * 32 * ROW_BYTES);
#pragma unroll
        for (int j = 0; j < TN; ++j) fb[set][j] = *reinterpret_cast<const bf16x8*>(smem + stage_at + w_at[ks] + j * 32 * ROW_BYTES);
    };
    auto mma = [&](int set, f32x16 (&sum)[TM][TN]) {
#pragma unroll
        for (int i = 0; i < TM; ++i)
#pragma unroll
            for (int j = 0; j < TN; ++j)
                sum[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(fb[set][j], fa[set][i], sum[i][j], 0, 0, 0);
    };
    auto zero_beyond = [&](int set, int ks) {                       // EDGE: the last tile's pieces beyond K
        const bf16x8 zero = {0, 0, 0, 0, 0, 0, 0, 0};
        if ((2 * (kg * KS + ks) + lane / 32) * 8 >= rest) {
#pragma unroll
            for (int i = 0; i < TM; ++i) fa[set][i] = zero;
#pragma unroll
            for (int j = 0; j < TN; ++j) fb[set][j] = zero;
        }
    };

    // Tile t is in stage t % STAGES, the tiles up to t + STAGES - 2 are on their way. Every k step issues its share of the loads
    // of tile t + STAGES - 1 (into the stage that tile t - 1 left: all wavefronts had read it when they last met), the fragment
    // reads of the next k step and its MFMAs; the scheduling barriers keep that order. In front of the last step's MFMAs the
    // wavefronts wait for tile t + 1 and meet, and read its first fragments: met behind them instead, all wavefronts would stand at the
    // barrier and then for these reads with idle matrix units (36.5 > 31.4 us at 2,048 x 2,304 x 3,072). The last STAGES - 1 tiles ask
    // for nothing and wait for fewer and fewer loads. (Asking for the last tile again there, so that one loop did for all, cost short
    // sums most: 2,048 x 2,048 x 512 12.0 > 8.9 us, 4,096 x 2,048 x 256 16.5 > 11.2, 8,192 x 3,072 x 192 34.6 > 24.4.)
    wait_tiles_and_meet<STAGES - 2, LOADS>(nk - 1);
    read_frags(0, 0, 0);
    int stage_at = 0, fetch_stage = STAGES - 1;
    auto step = [&](auto fetches, int t, f32x16 (&sum)[TM][TN]) {
        constexpr bool FETCHES = decltype(fetches)::value;
        const int next_at = stage_at == (STAGES - 1) * STAGE_BYTES ? 0 : stage_at + STAGE_BYTES;
#pragma unroll
        for (int ks = 0; ks < KS; ++ks) {
#pragma unroll
            for (int q = 0; q < LOADS; ++q)
                if (FETCHES && q * KS / LOADS == ks) fetch(q, t + STAGES - 1, fetch_stage);
            if (ks + 1 < KS) {
                read_frags(stage_at, ks + 1, (ks + 1) & 1);
            } else if (FETCHES) {
                wait_loads_and_meet<(STAGES - 2) * LOADS>();
                read_frags(next_at, 0, 0);
            } else if (t + 1 < nk) {
                wait_tiles_and_meet<STAGES - 3, LOADS>(nk - 2 - t);
                read_frags(next_at, 0, 0);
            }
            if (EDGE && !FETCHES && t == nk - 1) zero_beyond(ks & 1, ks);
            mma(ks & 1, sum);
            __builtin_amdgcn_sched_barrier(0);
        }
        stage_at = next_at;
        fetch_stage = fetch_stage == STAGES - 1 ? 0 : fetch_stage + 1;
    };
    // (Loops of their own: a choice of both in one loop has every sum twice in registers, and moves them.)
    const std::true_type asking;
    const std::false_type done;
    int t = 0;
    if constexpr (HALVES) {
        for (; t + STAGES < nk; t += 2) {
            step(asking, t, acc);
            step(asking, t + 1, acc2);
        }
        if (t + STAGES - 1 < nk) {
            step(asking, t, acc);
            step(done, t + 1, acc2);
            t += 2;
        }
        for (; t < nk; t += 2) {
            step(done, t, acc);
            if (t + 1 < nk) step(done, t + 1, acc2);
        }
#pragma unroll
        for (int i = 0; i < TM; ++i)
#pragma unroll
            for (int j = 0; j < TN; ++j) acc[i][j] += acc2[i][j];
    } else {
        for (; t + STAGES - 1 < nk; ++t) step(asking, t, acc);
        for (; t < nk; ++t) step(done, t, acc);
    }
    wait_loads_and_meet<0>();          // (nothing of the tiles is on its way or read any more)
    if (tid < BN) bias_s[tid] = bias_r;
    if (MODE == EPI_STORE && tid < BM) slot_s[tid] = slot_r;

    // With the weights as the A operand, register r of lane l holds output row l%32 and column
    // 8*(r/4) + 4*(l/32) + r%4 of a 32x32 sub-tile. Stored from there, one instruction would touch
    // 16 bytes in each of 32 rows. So the wavefront's 32 rows go through its own region of LDS: written as the MFMA left them,
    // read back as whole rows, 16 bytes of output a lane.
    // Two groups write both their sums, and each adds and stores half of the rows.
    lds_barrier();                     // bias and slots
    float* epi = reinterpret_cast<float*>(smem) + wid * (32 * EPI_STRIDE);
    const float* other = KG > 1 ? reinterpret_cast<const float*>(smem) + wave * (32 * EPI_STRIDE) : epi;      // group 0's
    const float* second = reinterpret_cast<const float*>(smem) + (WM * WN + wave) * (32 * EPI_STRIDE);        // group 1's
    bool kv8 = false;                  // eight columns lie in one of the two parts and in 16 bytes
    if constexpr (MODE == EPI_STORE) kv8 = kv.q_cols % 8 == 0 && kv.kv_dim % 8 == 0 && ((reinterpret_cast<uintptr_t>(kv.k_pages) | reinterpret_cast<uintptr_t>(kv.v_pages)) & 15) == 0;
    // 16-bit rows that start anywhere are stored a column a lane, so that an instruction still covers whole lines (eight columns a
    // lane, one behind the other: 2,048 x 50,257 x 256 158 us so, 246 with; 8,192 x 1,001 x 768 20.4, 29.4; 560 x 3,001 x 768 9.1, 10.2).
    bool single = false;
    if constexpr (!F32_OUT) {
        single = !vec;
        if constexpr (MODE == EPI_STORE) single = single && kv.slots == nullptr;
    }
#pragma unroll
    for (int i = 0; i < TM; ++i) {
        const int mb = m0 + (wm * TM + i) * 32, cb = wn * EC;      // first row; first column within the tile
        if constexpr (MODE == EPI_ADD_RESIDUAL && !EARLY) fetch_old(i);
        wave_lds_sync();          // the reads of the rows before are done
#pragma unroll
        for (int j = 0; j < TN; j += APART ? 1 : PAIR) {
            if constexpr (GATED && !APART) {
#pragma unroll
                for (int r = 0; r < 16; ++r) acc[i][j][r] = gated_value(acc[i][j][r], acc[i][j + 1][r], kv);
            }
            const int column = APART ? j % 2 * EC + j / 2 * 32 : j / PAIR * 32;
#pragma unroll
            for (int g = 0; g < 4; ++g)
                *reinterpret_cast<float4*>(&epi[(lane % 32) * EPI_STRIDE + column + 8 * g + 4 * (lane / 32)]) =
                    make_float4(acc[i][j][4 * g], acc[i][j][4 * g + 1], acc[i][j][4 * g + 2], acc[i][j][4 * g + 3]);
        }
        if constexpr (KG > 1) lds_barrier(); else wave_lds_sync();
        if constexpr (!F32_OUT) if (single) {
#pragma unroll 4
            for (int idx = lane; idx < 32 / KG * EC; idx += 64) {
                const int r = 32 / KG * kg + idx / EC, c = idx % EC, m = mb + r, n = n0 + cb + c;
                if (m >= M || n >= N) continue;
                float v = other[r * EPI_STRIDE + c];
                if constexpr (KG > 1) v += second[r * EPI_STRIDE + c];
                if constexpr (APART) v = gated_value(v, other[r * EPI_STRIDE + EC + c] + second[r * EPI_STRIDE + EC + c], kv);
                if constexpr (!GATED) v += bias_s[cb + c];
                static_cast<bf16_t*>(C)[static_cast<size_t>(m) * ldc + n] = float_to_bf16(activated<MODE>(v));
            }
            continue;
        }
#pragma unroll
        for (int it = 0; it < STEPS; ++it) {
            const int idx = it * 64 + lane, r = 32 / KG * kg + idx / PER_ROW, c = idx % PER_ROW * V;
            const int m = mb + r, n = n0 + cb + c;
            if (m >= M || n >= N) continue;
            float v[V / 4][4];
#pragma unroll
            for (int h = 0; h < V / 4; ++h) {
                const float4 t = *reinterpret_cast<const float4*>(&other[r * EPI_STRIDE + c + 4 * h]);
                v[h][0] = t.x; v[h][1] = t.y; v[h][2] = t.z; v[h][3] = t.w;
                if constexpr (KG > 1) {
                    const float4 u = *reinterpret_cast<const float4*>(&second[r * EPI_STRIDE + c + 4 * h]);
                    v[h][0] += u.x; v[h][1] += u.y; v[h][2] += u.z; v[h][3] += u.w;
                }
                if constexpr (GATED && KG > 1) {
                    // (the up map's columns stand behind the gate's)
                    const float4 a = *reinterpret_cast<const float4*>(&other[r * EPI_STRIDE + EC + c + 4 * h]), b = *reinterpret_cast<const float4*>(&second[r * EPI_STRIDE + EC + c + 4 * h]);
                    v[h][0] = gated_value(v[h][0], a.x + b.x, kv); v[h][1] = gated_value(v[h][1], a.y + b.y, kv);
                    v[h][2] = gated_value(v[h][2], a.z + b.z, kv); v[h][3] = gated_value(v[h][3], a.w + b.w, kv);
                }
                if constexpr (!GATED) {
                    const float4 b = *reinterpret_cast<const float4*>(&bias_s[cb + c + 4 * h]);
                    v[h][0] += b.x; v[h][1] += b.y; v[h][2] += b.z; v[h][3] += b.w;
                }
            }
            const size_t at = static_cast<size_t>(m) * ldc + n;
            if constexpr (MODE == EPI_THROUGH) {
                through4(static_cast<float*>(C), at, n, v[0], vec, min(4, N - n), kv);
            } else if constexpr (MODE == EPI_ADD_RESIDUAL) {
                if (vec && n + 4 <= N)
                    *reinterpret_cast<float4*>(static_cast<float*>(C) + at) = make_float4(old[EARLY ? i : 0][it].x + v[0][0], old[EARLY ? i : 0][it].y + v[0][1], old[EARLY ? i : 0][it].z + v[0][2], old[EARLY ? i : 0][it].w + v[0][3]);
                else store4<MODE>(C, at, v[0], vec, min(4, N - n));
            } else if constexpr (MODE == EPI_STORE_F32) {
                store4<MODE>(C, at, v[0], vec, min(4, N - n));
            } else if (vec8 && n + 8 <= N) {
                uint4 pk;
                pk.x = pack_bf16x2(activated<MODE>(v[0][0]), activated<MODE>(v[0][1])); pk.y = pack_bf16x2(activated<MODE>(v[0][2]), activated<MODE>(v[0][3]));
                pk.z = pack_bf16x2(activated<MODE>(v[1][0]), activated<MODE>(v[1][1])); pk.w = pack_bf16x2(activated<MODE>(v[1][2]), activated<MODE>(v[1][3]));
                *reinterpret_cast<uint4*>(static_cast<bf16_t*>(C) + at) = pk;
            } else {
#pragma unroll
                for (int h = 0; h < 2; ++h)
                    if (n + 4 * h < N) store4<MODE>(C, at + 4 * h, v[h], vec, min(4, N - n - 4 * h));
            }
            if constexpr (MODE == EPI_STORE) if (kv.slots != nullptr && n + 7 >= kv.q_cols) {
                const int slot = slot_s[mb - m0 + r];
                const int col8 = n - kv.q_cols;
                if (kv8 && n + 8 <= N) {
                    bf16_t* dst = (col8 < kv.kv_dim ? kv.k_pages + col8 : kv.v_pages + (col8 - kv.kv_dim)) + static_cast<size_t>(max(slot, 0)) * kv.kv_dim;
                    if (slot >= 0) *reinterpret_cast<uint4*>(dst) = make_uint4(pack_bf16x2(v[0][0], v[0][1]), pack_bf16x2(v[0][2], v[0][3]), pack_bf16x2(v[1][0], v[1][1]), pack_bf16x2(v[1][2], v[1][3]));
                    continue;
                }
#pragma unroll
                for (int h = 0; h < 2; ++h) {
                    // q_cols and kv_dim are multiples of 4: four columns lie in one of the two parts
                    const int col = n + 4 * h - kv.q_cols;
                    if (slot < 0 || col < 0 || n + 4 * h >= N) continue;
                    bf16_t* dst = (col < kv.kv_dim ? kv.k_pages + col : kv.v_pages + (col - kv.kv_dim)) + static_cast<size_t>(slot) * kv.kv_dim;
                    if (n + 4 * h + 4 <= N) {
                        *reinterpret_cast<uint2*>(dst) = make_uint2(pack_bf16x2(v[h][0], v[h][1]), pack_bf16x2(v[h][2], v[h][3]));
                    } else {
                        for (int e = 0; e < N - n - 4 * h; ++e) dst[e] = float_to_bf16(v[h][e]);
                    }
                }
            }
        }
    }
}

// split of the output among the XCDs (xm x xn = 8) that keeps the A rows plus W rows of one XCD smallest; returns its grid
static int split_among_xcds(int tiles_m, int tiles_n, int bm, int bn, int& xm, int& xn) {
    xm = 1, xn = N_XCD;
    double best = 1e300;
    for (int cand = 1; cand <= N_XCD; cand *= 2) {
        const int cm = cand, cn = N_XCD / cand;
        const double rows = static_cast<double>((tiles_m + cm - 1) / cm) * bm + static_cast<double>((tiles_n + cn - 1) / cn) * bn;
        if (rows < best) { best = rows; xm = cm; xn = cn; }
    }
    return ((tiles_m + xm - 1) / xm) * ((tiles_n + xn - 1) / xn) * N_XCD;
}

template <int WM, int WN, int TM, int TN, int BK, int STAGES, int KG = 1, bool HALVES = false, bool FAR = false>
static void launch_tiled_gated(const bf16_t* a, int lda, const bf16_t* w, int ldw, void* C, int ldc, int M, int N, int K,
                               const GatedPair& pair, hipStream_t stream) {
    constexpr int BM = WM * TM * 32, BN = WN * TN * 32;
    const int tiles_m = (M + BM - 1) / BM, tiles_n = (N + BN / 2 - 1) / (BN / 2);
    int xm, xn;
    const dim3 grid(split_among_xcds(tiles_m, tiles_n, BM, BN, xm, xn)), block(WM * WN * KG * 64);
#define TILED(E) gemm_bf16_mfma<WM, WN, TM, TN, BK, STAGES, KG, HALVES, FAR, E, EPI_GATED><<<grid, block, 0, stream>>>(a, w, pair.up, lda, ldw, M, N, K, __builtin_ctz(xm), C, ldc, pair)
    if (FAR || K % BK != 0) TILED(true); else if constexpr (!FAR) TILED(false);
#undef TILED
}

template <int WM, int WN, int TM, int TN, int BK, int STAGES, int KG = 1, bool HALVES = false, bool FAR = false>
static void launch_tiled(const bf16_t* a, int lda, const bf16_t* w, int ldw, const float* bias, void* C, int ldc,
                         int M, int N, int K, int mode, hipStream_t stream, KvScatter kv = KvScatter{},
                         const MllmStreamAdd* through = nullptr) {
    constexpr int BM = WM * TM * 32, BN = WN * TN * 32;
    const int tiles_m = (M + BM - 1) / BM, tiles_n = (N + BN - 1) / BN;
    int xm, xn;
    const dim3 grid(split_among_xcds(tiles_m, tiles_n, BM, BN, xm, xn)), block(WM * WN * KG * 64);
    const bool edge = FAR || K % BK != 0;      // rows and columns beyond the matrices need no other kernel
#define TILED(E, MD) gemm_bf16_mfma<WM, WN, TM, TN, BK, STAGES, KG, HALVES, FAR, E, MD><<<grid, block, 0, stream>>>(a, w, bias, lda, ldw, M, N, K, __builtin_ctz(xm), C, ldc, extra)
    if (mode == EPI_THROUGH) {
        const MllmStreamAdd extra = *through;
        if (edge) TILED(true, EPI_THROUGH); else if constexpr (!FAR) TILED(false, EPI_THROUGH);
        return;
    }
    const KvScatter extra = kv;
#define TILED_MODE(MD) case MD: if (edge) TILED(true, MD); else if constexpr (!FAR) TILED(false, MD); break;
    switch (mode) {
        TILED_MODE(EPI_STORE) TILED_MODE(EPI_GELU_TANH) TILED_MODE(EPI_GELU_ERF) TILED_MODE(EPI_RELU2) TILED_MODE(EPI_ADD_RESIDUAL)
        default: if (edge) TILED(true, EPI_STORE_F32); else if constexpr (!FAR) TILED(false, EPI_STORE_F32); break;
    }
#undef TILED_MODE
#undef TILED
}

// ---------------------------------------------------------------------------------------------
// Few rows (decode; up to 16 rows and, of the widest products, 64 always; up to 256 where it is priced
// lower than the tiles, see the dispatch). The product is bound by streaming W once, and how fast a compute
// unit streams depends on the shape of a wavefront's load: 8 consecutive lanes take one 128-byte
// line (8 weight rows x 1 line per load) at up to 90 GB/s per unit, but the MFMA operand layout
// (consecutive lanes = consecutive weight rows, 4 lines per 4 lanes) at under 40 (measured). So
// the loads use the first shape and the 16-byte pieces change lanes through a region of LDS
// private to the wavefront (2 KB per weight tile and k block, up to two k blocks at a time; no
// barrier: LDS serves a wavefront's requests in order), swizzled so that neither the writes nor
// the reads conflict. A workgroup owns 16 rows of the output (more
// rows: more workgroups per column range, placed on the same XCD so that the weights they share
// come from its L2).
//   SPLIT_K:  one workgroup per 16-column tile, its wavefronts split K (wavefront w takes the
//             64-element k blocks w, w+NW, ...) and their partial sums are added in LDS in a fixed
//             order: for the narrow products, where tiles alone are too few to fill the chip.
//             With k_parts > 1 several workgroups share a tile as well (blockIdx.y is the part):
//             each writes its sum to a workspace, and the last one to arrive, found through a
//             counter per tile, adds the parts in the order of their index and runs the
//             epilogue. For products whose tiles alone use a fraction of the compute units and
//             whose K is long (the second product of the feed-forward).
//   !SPLIT_K: one wavefront per tile over the whole of K (wide products such as the logits head).
// The activations come from global memory (A_GLOBAL: a few KB, shared by all workgroups, read
// from L2), are copied into LDS once per workgroup (A_STAGED: wide products), or are normalised
// from the fp32 stream into LDS first (A_NORMED): LayerNorm
// (/root/reference/src/kernels/layernorm.cu:32-49) fused into the product that follows it.
// A_MERGED: A is the output of decode attention that split every (token, head) pair's keys over
// several workgroups and left their states in a workspace (attention_decode.hip, partial_out): a lane
// that would load 8 elements of a row loads those elements of every split's unnormalised output and
// the splits' maxima and sums instead, and merges them in registers. The attention kernel then
// needs no pass that waits for its last workgroup, and more workgroups stream the keys.
// At up to 16 rows a launch is a chain of latencies, not a stream: of the 3.6 us that the norm and a 2,304 x 768 product took from their
// first wavefront's start, 1.3 passed before the first row was asked for (an argument loaded from memory, integer divisions). With
// what the first loads need in the preloaded arguments and an instance for every number of a lane's columns it takes 2.4 (back to back
// 4.3 > 3.1 us at 1 row, 4.5 > 3.3 at 8; a token of GPT-2 small alone 0.344 > 0.317 ms, of eight 0.407 > 0.377).
// ---------------------------------------------------------------------------------------------
typedef float f32x4 __attribute__((ext_vector_type(4)));

enum { A_GLOBAL = 0, A_NORMED = 1, A_STAGED = 2, A_MERGED = 3 };
#define MERGE_MAX_SPLITS 4      // splits of a pair that the merging load takes (registers: 10 per split and load)

// The states of MS splits for 8 consecutive elements of one head of one token.
template <int MS> struct SplitStates {
    float2 ml[MS];          // maximum (base 2), sum
    float4 o[MS][2];        // 8 elements of the unnormalised output
};

template <int MT, int ASRC, bool SPLIT_K, int U, bool A_TWO = true, int NT = 1, bool THROUGH = false, int MS = MERGE_MAX_SPLITS,
          bool ONE = false, bool GATED = false, int NU = 8, int WC = 16, int KP = 1, bool IN_TURN = false>
__global__ void __launch_bounds__(ASRC == A_NORMED ? 512 : (ASRC == A_GLOBAL || ASRC == A_MERGED ? 768 : 1024))
gemm_bf16_skinny(// The first 14 dwords arrive in registers with the wavefront, and hold everything that the first loads need: an argument
                 // behind them comes with a load of its own from memory that no cache holds (as does blockDim), 0.6 to 0.8 us
                 // before which no row and no weight could be asked for.
                 const bf16_t* __restrict__ W,
                 // A_MERGED: the outputs of the attention's MS splits (layout: attention_decode.hip); otherwise A
                 const void* __restrict__ Ain,
                 // A_NORMED: scale and shift (GATED: the second map's weights). A_MERGED: the splits' maxima and sums, bias.
                 // Otherwise bias and C.
                 const void* __restrict__ p2, const void* __restrict__ p3,
                 int ldw, unsigned columns, unsigned shape, int K_or_ldc,
                 // A_MERGED: C; otherwise A's row stride and, in the upper half, C's
                 void* __restrict__ C_or_strides,
                 // the rest is loaded by the kernel and needed later
                 const float* __restrict__ late_bias, void* __restrict__ late_C, const int* __restrict__ late_rows, float eps,
                 float* __restrict__ part_sums, int* __restrict__ part_counters,
                 // THROUGH (mode EPI_THROUGH): the norms the result passes and the copy it leaves; GATED: the second map and the
                 // activation; otherwise (plain store of a split-K kernel) the pages that its key and value columns go to as well
                 typename std::conditional<THROUGH, MllmStreamAdd, typename std::conditional<GATED, GatedPair, KvScatter>::type>::type add = {}) {
    static_assert(!THROUGH || (SPLIT_K && MT == 1 && ASRC == A_GLOBAL), "results through norms: split-K kernels of one row tile");
    // NT > 1 (SPLIT_K, MT == 1): the workgroup owns cols_per_wg <= 16 NT columns, NT tiles that share
    // the rows of A, the last one possibly narrower: for products with more than 256 tiles, whose
    // columns are dealt out evenly to 256 workgroups (one per compute unit; a kernel of this size
    // keeps one workgroup per unit, so 400 one-tile workgroups would take two rounds).
    // GATED: the two tiles are the same 16 columns of the gate's map and of the up map, and one value leaves for both.
    static_assert(!GATED || (NT == 2 && ASRC == A_NORMED), "gated pairs: two tiles behind the norm");
    static_assert(NT == 1 || (MT == 1 && SPLIT_K), "column tiles per workgroup: split-K kernels of one row tile");
    // KP == 2: the two parts of K that two workgroups would take, one behind the other in every wavefront, with sums of their own that
    // are added at the end as the workgroups' would be: the same bits without the exchange through memory (the launcher's k_parts).
    static_assert(KP == 1 || (KP == 2 && ONE && SPLIT_K && MT == 1 && NT == 1 && ASRC == A_GLOBAL), "parts of K in one workgroup: kernels of one chunk");
    // IN_TURN: the rows of A are asked for block by block beside the weights, else all of a chunk's in front of them. What comes first is used
    // first: with a few blocks the rows, which come from L2 and are short behind weights; over a longer stretch of K the blocks,
    // whose weights the products then need not wait for (see the launcher).
    static_assert(!IN_TURN || (ASRC == A_GLOBAL && NT == 1 && WC == 16), "rows in turn: whole column tiles");
    constexpr int T = MT * NT;      // accumulators: row tiles (NT == 1) or column tiles (MT == 1)
    constexpr int REDUCED = ASRC == A_NORMED ? 8 : 12;      // wavefronts whose sums meet, at most (SPLIT_K)
    extern __shared__ __attribute__((aligned(16))) unsigned char smem_raw[];
    __shared__ int sm_last;
    constexpr bool LN_FUSED = ASRC == A_NORMED;
    constexpr bool IN_LDS = ASRC == A_NORMED || ASRC == A_STAGED;
    constexpr bool A_REGS = !IN_LDS;      // the rows of A travel through registers and the wavefront's LDS region
    // (the word as few_row_shape packs it)
    const int M = shape & 511, cols_per_wg = shape >> 9 & 63, k_parts = shape >> 15 & 15, mode = shape >> 19 & 15, row_blocks = ((M + 15) / 16 + MT - 1) / MT;
    const int nw = ASRC == A_NORMED ? 8 : shape >> 23 & 31;
    const bool rms = shape >> 28 & 1, scatters = shape >> 29 & 1, gathers = shape >> 30 & 1;
    const int N = ASRC == A_MERGED ? columns & 0x3fff : columns;
    const int a_head_dim = (columns >> 14 & 511) * 8, a_heads = columns >> 23;              // A_MERGED
    const int K = ASRC == A_MERGED ? a_heads * a_head_dim : K_or_ldc;
    const int lda = static_cast<int>(reinterpret_cast<uintptr_t>(C_or_strides));            // not A_MERGED
    const float* gamma = static_cast<const float*>(p2);                                     // A_NORMED
    const float* beta = GATED ? nullptr : static_cast<const float*>(p3);
    const float* split_o = static_cast<const float*>(Ain);                                  // A_MERGED
    const float* split_ml = static_cast<const float*>(p2);
    const float* bias = ASRC == A_NORMED ? late_bias : static_cast<const float*>(ASRC == A_MERGED ? p3 : p2);
    void* C = ASRC == A_NORMED ? late_C : ASRC == A_MERGED ? C_or_strides : const_cast<void*>(p3);
    const int ldc = ASRC == A_MERGED ? K_or_ldc : static_cast<int>(reinterpret_cast<uintptr_t>(C_or_strides) >> 32);
    // The wavefront's index as a scalar: what depends on it alone (its k blocks, whether it has a
    // whole chunk, whether it owns outputs) then branches for real. Derived from threadIdx it would
    // count as divergent, both sides of every such condition would run one after the other under
    // masks, and loads pending from one side would be waited for on the other.
    const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid / 64), lane = tid % 64;
    const int row16 = lane % 16, kq = lane / 16;
    // workgroup id -> (column block, row block): the row blocks of one column block have ids that
    // agree modulo 8, i.e. run on one XCD
    int cb = blockIdx.x, rb = 0;
    if (row_blocks > 1) {
        const int g = blockIdx.x;
        cb = (g / (N_XCD * row_blocks)) * N_XCD + g % N_XCD;
        rb = (g / N_XCD) % row_blocks;
    }
    if (cb * (SPLIT_K ? cols_per_wg : nw * 16) >= N) return;
    const int m_base = rb * 16 * MT;
    const int n0 = SPLIT_K ? cb * cols_per_wg : (cb * nw + wave) * 16;
    // K is dealt out in blocks of 64 elements, one 128-byte line of a weight row. In the MFMAs
    // lane group kq takes elements 16*kq .. 16*kq+15 of a block, the first 8 in one MFMA and the
    // rest in the next (the k index of an MFMA may be permuted as long as both operands agree).
    // (with k_parts workgroups on the tile, over all their wavefronts alike)
    const int part = SPLIT_K ? blockIdx.y : 0;
    const int k_first = SPLIT_K ? (part * nw + wave) * 64 : 0;      // first k block of this wavefront
    const int k_stride = SPLIT_K ? nw * k_parts * 64 : 64;         // distance between its k blocks
    const size_t red_bytes = SPLIT_K ? static_cast<size_t>(nw) * T * KP * 256 * sizeof(float) : 0;
    // per wavefront: SB k blocks at a time change lanes through LDS, each NT weight tiles (+ the A block)
    constexpr int SB = (ASRC == A_STAGED || (A_REGS && NT > 1) || U < 4) ? 1 : 2;
    constexpr int STAGE_BYTES = SB * (NT * 2048 + (A_REGS ? 2048 : 0));
    float* red = reinterpret_cast<float*>(smem_raw);                       // [nw][T][256]
    bf16x8* stage_w = reinterpret_cast<bf16x8*>(smem_raw + red_bytes + static_cast<size_t>(wave) * STAGE_BYTES);
    bf16x8* stage_a = stage_w + SB * NT * 128;                             // (A_GLOBAL only)
    bf16_t* a_s = reinterpret_cast<bf16_t*>(smem_raw + red_bytes + static_cast<size_t>(nw) * STAGE_BYTES);   // [16*MT][K+8]
    const int a_stride = K + 8;
    // (fused norm only) the scale and shift vectors, loaded once per workgroup: [2][K] fp32
    float4* gb_s = reinterpret_cast<float4*>(a_s + static_cast<size_t>(16) * MT * a_stride);
    const int n = n0 + row16;
    const bool n_ok = n < N;
    const bf16x8 zero = {0, 0, 0, 0, 0, 0, 0, 0};
    // Loads: lane -> (row lr = lane / 8 of 8, 16-byte piece lane % 8 of the row's 128-byte line);
    // two loads cover the tile's 16 rows. The piece a lane fetches is its slot number XORed with a
    // swizzle of the row (the row modulo 8, its lowest bit flipped for rows 8..15), so that slot s
    // of row r, written to LDS lane-linearly, holds piece s ^ swizzle(r): then the 16 lanes of an
    // operand read (rows 0..15, one piece number) fall on 16 different 16-byte bank groups.
    // WC: the columns that a workgroup has, at most: two loads cover 16 of a k block, one 8, and one 4 of two blocks. (768 x 3,072 on 192
    // workgroups of 4 columns: of what two loads asked for three quarters were the last column again, and a compute unit takes 64 bytes a
    // clock: 3.9 > 3.3 us from the first wavefront's start at 1 and 8 rows, with rows beyond M not asked for either.)
    const int lr = lane / 8;
    const int piece[2] = {(lane % 8) ^ lr, (lane % 8) ^ lr ^ 1};
    static_assert(WC == 16 || (SPLIT_K && NT == 1 && U % 4 == 0 && U >= 4), "narrow column tiles: whole pairs of k blocks");
    // (columns beyond the workgroup's or the matrix's: the last valid one, never stored)
    const bf16_t* wrow[NT][2];
#pragma unroll
    for (int t = 0; t < NT; ++t)
#pragma unroll
        for (int j = 0; j < 2; ++j) {
            if constexpr (GATED) wrow[t][j] = (t ? static_cast<const bf16_t*>(p3) : W) + static_cast<size_t>(min(n0 + lr + 8 * j, N - 1)) * ldw;
            else wrow[t][j] = W + static_cast<size_t>(min(n0 + min(16 * t + lr + 8 * j, cols_per_wg - 1), N - 1)) * ldw;
        }
    const bf16_t* wrow4 = W + static_cast<size_t>(min(n0 + min(lr % 4, cols_per_wg - 1), N - 1)) * ldw;     // (WC == 4)
    const int piece4 = (lane % 8) ^ (lr % 4);
    // reads: this lane's MFMA row/column is row16; for MFMA step `half` it wants piece 2*kq + half
    const int rd_swz = row16 < 8 ? row16 : ((row16 - 8) ^ 1);

    f32x4 acc[T];
#pragma unroll
    for (int i = 0; i < T; ++i) acc[i] = f32x4{0.f, 0.f, 0.f, 0.f};

    // Split-K epilogue operands (thread tid < 256 owns output element tid of the 16x16 tile, in
    // accumulator order): requested with the first loads so that their latency hides behind the product.
    bool ep_ok[NT];
    size_t ep_idx[NT];
    int ep_col[NT], ep_slot = -1;
    float ep_bias[NT], ep_old[NT];
    MllmNormColumn ep_norm[NT], ep_next[NT];
    float ep_alpha = 0.f, ep_alpha2 = 0.f;
#pragma unroll
    for (int t = 0; t < NT; ++t) { ep_ok[t] = false; ep_idx[t] = 0; ep_col[t] = 0; ep_bias[t] = 0.f; ep_old[t] = 0.f; }
    auto epilogue_loads = [&]() {
        if (!(SPLIT_K && MT == 1) || wave >= 4) return;
        // (loads without a per-lane condition: outputs beyond M or N read the last row or column)
        const int m = m_base + 4 * (lane / 16) + wave;
#pragma unroll
        for (int t = 0; t < (GATED ? 1 : NT); ++t) {
            const int ct = 16 * t + lane % 16, nn = n0 + ct;
            ep_ok[t] = m < M && nn < N && ct < cols_per_wg;
            ep_col[t] = nn;
            ep_idx[t] = static_cast<size_t>(min(m, M - 1)) * ldc + min(nn, N - 1);
            if (bias) ep_bias[t] = bias[min(nn, N - 1)];
            if (THROUGH || mode == EPI_ADD_RESIDUAL) ep_old[t] = static_cast<const float*>(C)[ep_idx[t]];
            if constexpr (THROUGH) {
                const int nc = min(nn, N - 1);
                if (add.norm.weight != nullptr) ep_norm[t] = {add.norm.weight[nc], add.norm.bias[nc]};
                if (add.next.weight != nullptr) ep_next[t] = {add.next.weight[nc], add.next.bias[nc]};
            }
        }
        if constexpr (THROUGH) {
            if (add.norm.weight != nullptr) ep_alpha = add.norm.alpha[0];
            if (add.next.weight != nullptr) ep_alpha2 = add.next.alpha[0];
        } else if constexpr (!GATED) {
            if (scatters) ep_slot = add.slots[min(m, M - 1)];
        }
    };
    // (behind the fused norm what they need comes late, and so do they: they are asked for behind the first loads there)
    if (!LN_FUSED) epilogue_loads();

    // A wavefront takes its k blocks in chunks of H = U/2. All loads of a chunk are issued
    // together and without a condition inside (a load under a condition makes the compiler wait
    // for every load in flight); the conditions that decide whether a chunk is loaded at all are
    // uniform over the wavefront. No load goes to a line that another load may still have in
    // flight: loads that hit such a line queue up behind it in the vector cache. Two chunks
    // alternate so that one is in flight while the other is multiplied; the first is requested
    // before the norm or the copy of A, so that its latency overlaps them. Blocks left over
    // (fewer than H) follow one by one. Only the last block of K can be short: its lanes beyond K
    // load the row's last 16 bytes and their weight fragment is zeroed.
    constexpr int H = U / 2;
    static_assert(U % 2 == 0, "whole k blocks per chunk");
    const bf16_t* A = static_cast<const bf16_t*>(Ain);
    // A_GLOBAL: the rows of A travel like the weights (rows beyond M: the last one, never stored);
    // a workgroup with at most 8 rows needs one load per k block
    const bf16_t* arow[2] = {A, A};
    int arow_idx[2] = {0, 0};
    // (A_TWO false: the launcher knows that M <= 8, and the chunks keep half the registers for A)
    const bool a_two = A_TWO && M - m_base > 8;
    if (A_REGS) {
#pragma unroll
        for (int j = 0; j < 2; ++j) {
            arow_idx[j] = min(m_base + lr + 8 * j, M - 1);
            arow[j] = A + static_cast<size_t>(arow_idx[j]) * lda;
        }
    }
    // (Lanes of rows beyond M ask for nothing: what they multiply reaches only outputs that are not stored. Where rows stand in turn with
    // weights, or splits are merged, for more than 8 rows they ask for the last row again: under a condition those kernels kept up to
    // 70 registers more in scratch memory, 5 heads of 256, 12 rows of four splits 25.0 us against 22.9.)
    constexpr bool EVERY_ROW = A_TWO && (IN_TURN || ASRC == A_MERGED);
    const bool row_exists[2] = {EVERY_ROW || m_base + lr < M, EVERY_ROW || m_base + lr + 8 < M};
    // A_MERGED: requests the splits' states for the 8 elements from k on of row `row` (all loads together; n_splits is MS),
    // and merges them later
    auto fetch_splits = [&](SplitStates<MS>& st, int row, int k) {
        // (k / head size in eighths, exact: both are small whole numbers, and half an eighth is further from the next
        // quotient than the reciprocal's error)
        const int h = static_cast<int>((static_cast<float>(k / 8) + 0.5f) * __builtin_amdgcn_rcpf(static_cast<float>(a_head_dim / 8)));
        const int e = k - h * a_head_dim;
        const size_t pair = static_cast<size_t>(row) * a_heads + h;
        typedef float f32x4_of_8 __attribute__((ext_vector_type(4), aligned(8)));
#pragma unroll
        for (int sidx = 0; sidx + 1 < MS; sidx += 2) {
            const f32x4_of_8 two = *reinterpret_cast<const f32x4_of_8*>(split_ml + (pair * MS + sidx) * 2);
            st.ml[sidx] = make_float2(two.x, two.y);
            st.ml[sidx + 1] = make_float2(two.z, two.w);
        }
        if constexpr (MS % 2 == 1) st.ml[MS - 1] = *reinterpret_cast<const float2*>(split_ml + (pair * MS + MS - 1) * 2);
#pragma unroll
        for (int sidx = 0; sidx < MS; ++sidx) {
            const size_t slot = pair * MS + sidx;
            const float4* src = reinterpret_cast<const float4*>(split_o + slot * a_head_dim + e);
            st.o[sidx][0] = src[0];
            st.o[sidx][1] = src[1];
        }
    };
    auto merge_splits = [&](const SplitStates<MS>& st) -> bf16x8 {
        float mx = st.ml[0].x;
#pragma unroll
        for (int sidx = 1; sidx < MS; ++sidx) mx = fmaxf(mx, st.ml[sidx].x);
        float l = 0.f, o[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int sidx = 0; sidx < MS; ++sidx) {
            const float w = fast_exp2(st.ml[sidx].x - mx);
            l = fmaf(w, st.ml[sidx].y, l);
            o[0] = fmaf(w, st.o[sidx][0].x, o[0]); o[1] = fmaf(w, st.o[sidx][0].y, o[1]);
            o[2] = fmaf(w, st.o[sidx][0].z, o[2]); o[3] = fmaf(w, st.o[sidx][0].w, o[3]);
            o[4] = fmaf(w, st.o[sidx][1].x, o[4]); o[5] = fmaf(w, st.o[sidx][1].y, o[5]);
            o[6] = fmaf(w, st.o[sidx][1].z, o[6]); o[7] = fmaf(w, st.o[sidx][1].w, o[7]);
        }
        const float inv = 1.0f / l;
        union { uint32_t w[4]; bf16x8 v; } pk;
#pragma unroll
        for (int i = 0; i < 4; ++i) pk.w[i] = pack_bf16x2(o[2 * i] * inv, o[2 * i + 1] * inv);
        return pk.v;
    };
    // blocks of this wavefront: those behind its first, divided by the wavefronts on the tile
    int n_blocks = (K + 63) / 64;
    if (SPLIT_K) {
        const int from = n_blocks - 1 - (part * nw + wave);
        n_blocks = from < 0 ? 0 : 1 + small_quotient(from, nw * k_parts);
    }
    const int n_chunks = n_blocks / H;
    struct Chunk {
        bf16x8 b[NT][U * WC / 16];
        bf16x8 a[A_REGS ? (A_TWO ? U : U / 2) : 1];
    };
    // (A_MERGED) the states requested for a chunk's blocks, rows 0..7 and 8..15
    SplitStates<MS> pending[ASRC == A_MERGED ? U / 2 : 1][ASRC == A_MERGED && A_TWO ? 2 : 1];
    auto fetch_block_splits = [&](int h, int k0) {
        if (ASRC != A_MERGED) return;
#pragma unroll
        for (int j = 0; j < (A_TWO ? 2 : 1); ++j)
            if ((j == 0 || a_two) && row_exists[j]) fetch_splits(pending[h][j], arow_idx[j], min(k0 + 8 * piece[j], K - 8));
    };
    auto merge_block_splits = [&](Chunk& c, int h) {
        if (ASRC != A_MERGED) return;
#pragma unroll
        for (int j = 0; j < (A_TWO ? 2 : 1); ++j)
            if (j == 0 || a_two) c.a[A_TWO ? 2 * h + j : h] = merge_splits(pending[h][j]);
    };
    // Weights that one workgroup alone reads (one row block: at most 8 rows, or the fused norm's 16) and the wide product's (the logits
    // head, as large as all the layers') are requested with streaming loads: read once a step, they would only displace what is read
    // again (activations, scale and shift vectors, biases) from the caches. With several row blocks the later ones find the weights
    // in L2 and plain loads are kept.
    auto load_piece = [&](const bf16_t* from) -> bf16x8 {
        constexpr bool STREAM = ASRC != A_GLOBAL || !A_TWO;
        const bf16x8* src = reinterpret_cast<const bf16x8*>(from);
        return STREAM ? __builtin_nontemporal_load(src) : *src;
    };
    auto load_steps = [&](Chunk& c, int u0, int k0) {      // weights of the k block at k0 (columns 0..7, columns 8..15) into slots u0, u0+1
#pragma unroll
        for (int j = 0; j < (WC == 16 ? 2 : WC / 8); ++j) {
            const int k = min(k0 + 8 * piece[j], K - 8);
#pragma unroll
            for (int t = 0; t < NT; ++t) c.b[t][WC == 16 ? u0 + j : u0 / 2] = load_piece(wrow[t][j] + k);
            if (IN_TURN && (j == 0 || a_two) && row_exists[j]) c.a[A_TWO ? u0 + j : u0 / 2] = *reinterpret_cast<const bf16x8*>(arow[j] + k);
        }
    };
    auto load_rows = [&](Chunk& c, int count, auto k_of) {      // rows of A for the first `count` blocks of a chunk, block h at k_of(h)
        if (ASRC != A_GLOBAL || IN_TURN) return;       // (A_MERGED: the splits' states were requested before and are merged after the weights)
#pragma unroll
        for (int j = 0; j < 2; ++j) {
            if ((j == 1 && !a_two) || !row_exists[j]) continue;
#pragma unroll
            for (int h = 0; h < H; ++h)
                if (h < count) c.a[A_TWO ? 2 * h + j : h] = *reinterpret_cast<const bf16x8*>(arow[j] + min(k_of(h) + 8 * piece[j], K - 8));
        }
    };
    auto load_pairs = [&](Chunk& c, auto k_of) {           // (WC == 4) weights of all blocks of a chunk, two to a load
        if constexpr (WC == 4) {
#pragma unroll
            for (int i = 0; i < U / 4; ++i) c.b[0][i] = load_piece(wrow4 + min((lane < 32 ? k_of(2 * i) : k_of(2 * i + 1)) + 8 * piece4, K - 8));
        }
    };
    auto wave_lds_order = [&]() {       // orders the wavefront's own LDS writes and reads (no instruction)
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    };
    // CNT (1 or 2) consecutive k blocks of a chunk, slots u0.., first k index k0: all their pieces go
    // through the wavefront's LDS region in one round trip (writes, then reads, then the MFMAs)
    auto mma_blocks = [&](const Chunk& c, int u0, int k0, auto cnt_tag) {
        constexpr int CNT = decltype(cnt_tag)::value;
        static_assert(CNT <= SB, "staging room");
#pragma unroll
        for (int i = 0; i < CNT; ++i) {
            if (A_REGS) {
                stage_a[i * 128 + lane] = c.a[A_TWO ? u0 + 2 * i : (u0 + 2 * i) / 2];
                if (a_two) stage_a[i * 128 + 64 + lane] = c.a[A_TWO ? u0 + 2 * i + 1 : 0];
            }
#pragma unroll
            for (int t = 0; t < NT; ++t) {
                if (WC > 4) stage_w[(i * NT + t) * 128 + lane] = c.b[t][WC == 16 ? u0 + 2 * i : u0 / 2 + i];
                if (WC == 16) stage_w[(i * NT + t) * 128 + 64 + lane] = c.b[t][u0 + 2 * i + 1];
            }
        }
        if (WC == 4) stage_w[(lane / 32) * 128 + lane % 32] = c.b[0][u0 / 4];       // (both blocks of the pair, columns 0..3)
        wave_lds_order();
        bf16x8 af[CNT][2], bf[CNT][NT][2];
#pragma unroll
        for (int i = 0; i < CNT; ++i)
#pragma unroll
            for (int half = 0; half < 2; ++half) {
                const int slot = row16 * 8 + ((2 * kq + half) ^ rd_swz);
                if (A_REGS) af[i][half] = stage_a[i * 128 + slot];
#pragma unroll
                for (int t = 0; t < NT; ++t) bf[i][t][half] = stage_w[(i * NT + t) * 128 + slot];
            }
        wave_lds_order();
#pragma unroll
        for (int i = 0; i < CNT; ++i)
#pragma unroll
            for (int half = 0; half < 2; ++half) {
                const int k = k0 + i * k_stride + 16 * kq + 8 * half;
                const int kc = min(k, K - 8);
                // (uniform over the wavefront; where the rows are in registers too, a branch costs them more than the comparison)
                const bool whole = IN_LDS && k0 + i * k_stride + 64 <= K;
#pragma unroll
                for (int mi = 0; mi < MT; ++mi) {
                    bf16x8 a;
                    if (IN_LDS) a = *reinterpret_cast<const bf16x8*>(a_s + static_cast<size_t>(mi * 16 + row16) * a_stride + kc);
                    else a = af[i][half];
#pragma unroll
                    for (int t = 0; t < NT; ++t) {
                        const bf16x8 b = whole || k < K ? bf[i][t][half] : zero;
                        acc[mi * NT + t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, acc[mi * NT + t], 0, 0, 0);
                    }
                }
            }
    };
    // `count` of the blocks in slots 0, 2, 4, ... of a chunk (count is uniform over the wavefront), k
    // indices from k0 on
    auto mma_some = [&](const Chunk& c, int count, int k0) {
#pragma unroll
        for (int h = 0; h < H; h += SB) {
            if (SB == 2 && h + 1 < H && h + 1 < count)
                mma_blocks(c, 2 * h, k0 + h * k_stride, std::integral_constant<int, SB>{});
            else if (h < count)
                mma_blocks(c, 2 * h, k0 + h * k_stride, std::integral_constant<int, 1>{});
        }
    };
    auto load_chunk = [&](Chunk& c, int chunk) {            // chunk index within this wavefront's blocks
        if (ASRC == A_MERGED) {
#pragma unroll
            for (int h = 0; h < H; ++h) fetch_block_splits(h, k_first + (chunk * H + h) * k_stride);
            __builtin_amdgcn_sched_barrier(0);
        }
        auto k_of = [&](int h) { return k_first + (chunk * H + h) * k_stride; };
        load_rows(c, H, k_of);
        if (WC == 4) load_pairs(c, k_of);
        else
#pragma unroll
            for (int h = 0; h < H; ++h) load_steps(c, 2 * h, k_of(h));
        // the instruction scheduler must not sink these loads towards their uses: they are issued
        // here to be in flight together
        __builtin_amdgcn_sched_barrier(0);
        if (ASRC == A_MERGED) {
#pragma unroll
            for (int h = 0; h < H; ++h) merge_block_splits(c, h);
        }
    };
    auto mma_chunk = [&](const Chunk& c, int chunk) { mma_some(c, H, k_first + chunk * H * k_stride); };
    // rows of the fp32 stream that this wavefront normalises (read before the weights are
    // requested: loads complete in order, and the row addresses depend on these)
    int src_row[2] = {0, 0};
    if (LN_FUSED) {
#pragma unroll
        for (int j = 0; j < 2; ++j) src_row[j] = min(m_base + wave + 8 * j, M - 1);      // 8 wavefronts, rows wave and wave + 8
        if (gathers) {
            src_row[0] = late_rows[src_row[0]];
            src_row[1] = late_rows[src_row[1]];
            // (waited for in here, not where the launches without a gather pass too)
            asm volatile("" : "+s"(src_row[0]), "+s"(src_row[1]));
        }
    }
    Chunk c0, c1;
    auto load_left = [&]() {                                // the blocks after the last whole chunk
        const int first = n_chunks * H, left = n_blocks - first;
        if (ASRC == A_MERGED) {
#pragma unroll
            for (int h = 0; h < H - 1; ++h)
                if (h < left) fetch_block_splits(h, k_first + (first + h) * k_stride);
            __builtin_amdgcn_sched_barrier(0);
        }
        auto k_of = [&](int h) { return k_first + min(first + h, n_blocks - 1) * k_stride; };
        load_rows(c1, left, k_of);
        if (WC == 4) load_pairs(c1, k_of);
        else
#pragma unroll
            for (int h = 0; h < H - 1; ++h)
                if (h < left) load_steps(c1, 2 * h, k_of(h));
        __builtin_amdgcn_sched_barrier(0);
        if (ASRC == A_MERGED) {
#pragma unroll
            for (int h = 0; h < H - 1; ++h)
                if (h < left) merge_block_splits(c1, h);
        }
    };
    // The first loads are one whole chunk for every wavefront, without a condition: a wavefront
    // with fewer blocks than a chunk takes its last block again (its own line, requested a moment
    // earlier) and leaves it unused. (Whole chunk or leftovers, decided by a branch, would hand the
    // norm that follows registers that count as pending on one side of the branch, and it would
    // wait for the weights.)
    const int last_block = n_blocks > 0 ? n_blocks - 1 : 0;
    int n_second = 0, k_second = 0;             // (KP == 2: this wavefront's blocks of the second part)
    if (KP == 2) {
        const int from = (K + 63) / 64 - 1 - (nw + wave);
        n_second = from < 0 ? 0 : 1 + small_quotient(from, nw * KP);
        k_second = (nw + wave) * 64;
    }
    auto first_loads = [&]() {
        if (ASRC == A_MERGED) {
#pragma unroll
            for (int h = 0; h < H; ++h) fetch_block_splits(h, k_first + min(h, last_block) * k_stride);
            __builtin_amdgcn_sched_barrier(0);
        }
        auto ask = [&](Chunk& c, auto k_of) {
            load_rows(c, H, k_of);
            if (WC == 4) load_pairs(c, k_of);
            else
#pragma unroll
                for (int h = 0; h < H; ++h) load_steps(c, 2 * h, k_of(h));
            __builtin_amdgcn_sched_barrier(0);
        };
        ask(c0, [&](int h) { return k_first + min(h, last_block) * k_stride; });
        if (KP == 2) ask(c1, [&](int h) { return k_second + min(h, max(n_second - 1, 0)) * k_stride; });
        if (ASRC == A_MERGED) {
#pragma unroll
            for (int h = 0; h < H; ++h) merge_block_splits(c0, h);
        }
    };
    // The fused norm's operands are requested before the weights: loads return in the order of
    // their requests, so the norm (whose rows come from L2) can be computed while the weights are
    // still on their way from memory, which it could not if it had to wait for them first.
    // (NU: float4 of a row per lane, so that nothing but the last is asked whether it exists: with 8 and a condition at each the
    // kernel had 2,140 instructions, most of a short launch's time)
    const int nq = K / 4;       // float4 per row
    constexpr int GB_ROUNDS = NU > 4 ? 2 : 1;       // rounds of 512 threads over scale and shift
    float4 gb_piece[GB_ROUNDS], v[2][NU];
    // whether this wavefront's two rows exist is uniform over it: rows beyond M are not read
    const bool row_ok[2] = {m_base + wave < M, m_base + wave + 8 < M};
    if (LN_FUSED) {
        const float* x = static_cast<const float*>(Ain);
        const float4* g4 = reinterpret_cast<const float4*>(gamma);
        const float4* b4 = reinterpret_cast<const float4*>(beta);
        // (the rows first: they come from L2, and their mean and variance need nothing else)
#pragma unroll
        for (int j = 0; j < 2; ++j) {
            if (!row_ok[j]) continue;
            const float4* row = reinterpret_cast<const float4*>(x + static_cast<size_t>(src_row[j]) * lda);
#pragma unroll
            for (int u = 0; u < NU; ++u) v[j][u] = row[u < NU - 1 ? lane + 64 * u : min(lane + 64 * u, nq - 1)];
        }
        __builtin_amdgcn_sched_barrier(0);
        // scale and shift: 2 K / 4 pieces of 16 bytes over the workgroup's 512 threads (K <= 2048:
        // at most two each), shared through LDS instead of every wavefront loading all of both
#pragma unroll
        for (int r = 0; r < GB_ROUNDS; ++r) {
            const int i = min(tid + 512 * r, 2 * nq - 1);
            const float4* src = i < nq ? g4 + i : (beta ? b4 + (i - nq) : g4);
            gb_piece[r] = *src;
        }
        __builtin_amdgcn_sched_barrier(0);
    }
    first_loads();
    if (LN_FUSED) epilogue_loads();
    if (ASRC == A_STAGED) {
        // the workgroup's rows of A, copied once into LDS for all its wavefronts
        // (four 16-byte pieces per thread requested together, then written)
        const int kv = K / 8, total = 16 * MT * kv;
        for (int base = tid; base < total; base += 4 * nw * 64) {
            bf16x8 v[4];
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                const int idx = min(base + j * nw * 64, total - 1);
                const int m = idx / kv, c = idx - m * kv;
                v[j] = *reinterpret_cast<const bf16x8*>(A + static_cast<size_t>(min(m_base + m, M - 1)) * lda + 8 * c);
            }
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                const int idx = base + j * nw * 64;
                const int m = idx / kv, c = idx - m * kv;
                if (idx < total)
                    *reinterpret_cast<bf16x8*>(a_s + static_cast<size_t>(m) * a_stride + 8 * c) =
                        (m_base + m < M) ? v[j] : zero;
            }
        }
        __syncthreads();
    }
    if (LN_FUSED) {
        // 8 wavefronts, two rows each; a row lives in registers (K <= 2048, K % 4 == 0): mean,
        // then variance of the centred values, all in fp32.
        float mean[2] = {0.f, 0.f}, inv[2] = {0.f, 0.f};
#pragma unroll
        for (int j = 0; j < 2; ++j) {
            if (!row_ok[j]) continue;
            float sum = 0.f;
#pragma unroll
            for (int u = 0; u < NU; ++u)
                if (u < NU - 1 || lane + 64 * u < nq) sum += (v[j][u].x + v[j][u].y) + (v[j][u].z + v[j][u].w);
            mean[j] = rms ? 0.f : wave_sum(sum) / static_cast<float>(K);
            float q = 0.f;
#pragma unroll
            for (int u = 0; u < NU; ++u) {
                if (u < NU - 1 || lane + 64 * u < nq) {
                    q += squares_sum(v[j][u].x - mean[j], v[j][u].y - mean[j], v[j][u].z - mean[j], v[j][u].w - mean[j]);
                }
            }
            inv[j] = 1.0f / sqrtf(wave_sum(q) / static_cast<float>(K) + eps);
        }
#pragma unroll
        for (int r = 0; r < GB_ROUNDS; ++r) {
            const int i = tid + 512 * r;
            if (i < 2 * nq) gb_s[i] = (i >= nq && !beta) ? make_float4(0.f, 0.f, 0.f, 0.f) : gb_piece[r];
        }
        lds_barrier();                 // scale and shift are in LDS (the weights stay in flight)
#pragma unroll
        for (int j = 0; j < 2; ++j) {
            const int m = wave + 8 * j;
            bf16_t* dst = a_s + static_cast<size_t>(m) * a_stride;
            if (!row_ok[j]) continue;      // (what its place in LDS holds goes into its own row of the products alone, which is not stored)
#pragma unroll
            for (int u = 0; u < NU; ++u) {
                const int i = lane + 64 * u;
                if (u < NU - 1 || i < nq) {
                    const float4 g = gb_s[i], b = gb_s[nq + i];
                    uint2 pk;
                    pk.x = pack_bf16x2((v[j][u].x - mean[j]) * inv[j] * g.x + b.x, (v[j][u].y - mean[j]) * inv[j] * g.y + b.y);
                    pk.y = pack_bf16x2((v[j][u].z - mean[j]) * inv[j] * g.z + b.z, (v[j][u].w - mean[j]) * inv[j] * g.w + b.w);
                    *reinterpret_cast<uint2*>(dst + 4 * i) = pk;
                }
            }
        }
        lds_barrier();
    }

    // ONE: the launcher knows that a chunk holds all of a wavefront's blocks, and a second one takes no registers. (With it the
    // kernels of four blocks a wavefront, and those that merge splits, kept 76 to 1,220 bytes a lane in scratch memory.)
    constexpr bool SINGLE = ONE || ASRC == A_MERGED;
    f32x4 of_first = {0.f, 0.f, 0.f, 0.f};      // (KP == 2: the first part's sums)
    if constexpr (KP == 2) {
        mma_some(c0, n_blocks, k_first);
        of_first = acc[0];
        acc[0] = f32x4{0.f, 0.f, 0.f, 0.f};
        mma_some(c1, n_second, k_second);
    } else if (n_chunks == 0) {
        mma_some(c0, n_blocks, k_first);
    } else if (SINGLE || n_chunks == 1) {
        mma_chunk(c0, 0);
    } else if (n_chunks > 1) {
        // past the last chunk the prefetch takes chunk 0 again (long since arrived, never used)
        for (int ci = 0; ci < n_chunks; ci += 2) {
            load_chunk(c1, ci + 1 < n_chunks ? ci + 1 : 0);
            mma_chunk(c0, ci);
            load_chunk(c0, ci + 2 < n_chunks ? ci + 2 : 0);
            if (ci + 1 < n_chunks) mma_chunk(c1, ci + 1);
        }
    }
    if (!SINGLE) {
        // blocks left over: fewer than H, loaded together
        const int first = n_chunks * H, left = n_chunks > 0 ? n_blocks - first : 0;
        if (left > 0) load_left();
        mma_some(c1, left, k_first + first * k_stride);
    }
    // (Arguments that the kernel loads itself stay where they are put until here: registers taken up again earlier are waited for, with the
    // loads into them still in flight, in front of the first rows and weights.)
    if constexpr (!THROUGH && !GATED) asm volatile("" ::"s"(add.slots), "s"(add.k_pages), "s"(add.v_pages), "s"(add.q_cols), "s"(add.kv_dim));
    asm volatile("" ::"s"(late_bias), "s"(late_C), "s"(part_sums), "s"(part_counters));
    // accumulator layout of the 16x16 tile: register r of lane l holds row 4*(l/16) + r, column l%16
    if (!SPLIT_K) {
        if (!n_ok) return;
        const float bv = bias ? bias[n] : 0.f;
#pragma unroll
        for (int i = 0; i < MT; ++i)
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const int m = m_base + i * 16 + 4 * kq + r;
                if (m < M) epilogue<bf16_t>(mode, acc[i][r], bv, C, static_cast<size_t>(m) * ldc + n);
            }
        return;
    }
#pragma unroll
    for (int i = 0; i < T; ++i)
#pragma unroll
        for (int r = 0; r < 4; ++r) red[(static_cast<size_t>(wave) * T * KP + i) * 256 + r * 64 + lane] = KP == 2 ? of_first[r] : acc[i][r];
    if (KP == 2)
#pragma unroll
        for (int r = 0; r < 4; ++r) red[(wave * KP + 1) * 256 + r * 64 + lane] = acc[0][r];
    __syncthreads();
    if (MT == 1) {
        // one output per tile and thread (the first 256); its bias and old residual value were
        // requested before the MFMA loop
        float vt[NT];
#pragma unroll
        for (int t = 0; t < NT; ++t) {
            vt[t] = 0.f;
            if (wave < 4) {
                // (all reads at once, then the sum in the order of the wavefronts; parts one by one)
                float of_wave[KP][REDUCED];
#pragma unroll
                for (int p = 0; p < KP; ++p)
#pragma unroll
                    for (int w = 0; w < REDUCED; ++w) of_wave[p][w] = red[(min(w, nw - 1) * NT * KP + t + p) * 256 + tid];
#pragma unroll
                for (int p = 0; p < KP; ++p) {
                    float sum = 0.f;
#pragma unroll
                    for (int w = 0; w < REDUCED; ++w)
                        if (w < nw) sum += of_wave[p][w];
                    vt[t] = p == 0 ? sum : vt[t] + sum;
                }
            }
        }
        float& v = vt[0];
        if (NT == 1 && KP == 1 && k_parts > 1) {
            // The parts of a tile meet in the workspace. Stores and loads of it are at device scope
            // (workgroups of one tile may run on different XCDs, whose L2 caches do not see each
            // other's lines); one thread's fences order them around the counter (a fence in every
            // thread costs tens of microseconds here, one about 1.5). The last workgroup leaves the
            // counter at zero for the next launch.
            const int tile = cb * row_blocks + rb;
            float* sums = part_sums + static_cast<size_t>(tile) * k_parts * 256;
            if (tid < 256) __hip_atomic_store(&sums[part * 256 + tid], v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            __syncthreads();
            if (tid == 0) {
                __builtin_amdgcn_fence(__ATOMIC_RELEASE, "agent");      // after the barrier: covers every thread's stores
                const int arrived = __hip_atomic_fetch_add(&part_counters[tile], 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                sm_last = (arrived == k_parts - 1) ? 1 : 0;
                if (sm_last) {
                    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "agent");
                    __hip_atomic_store(&part_counters[tile], 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                }
            }
            __syncthreads();
            if (!sm_last) return;
            v = 0.f;
            if (tid < 256)
                for (int p = 0; p < k_parts; ++p)
                    v += __hip_atomic_load(&sums[p * 256 + tid], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        }
        if constexpr (GATED) {
            if (ep_ok[0]) static_cast<bf16_t*>(C)[ep_idx[0]] = float_to_bf16(gated_value(vt[0], vt[1], add));
            return;
        }
#pragma unroll
        for (int t = 0; t < NT; ++t) {
            if (ep_ok[t]) {
                const float r = vt[t] + ep_bias[t];
                if constexpr (THROUGH) {
                    const float x = ep_old[t] + mllm_norm_column(r, add.norm.weight != nullptr, ep_alpha, ep_norm[t]);
                    static_cast<float*>(C)[ep_idx[t]] = x;
                    if (add.copy != nullptr)
                        static_cast<bf16_t*>(add.copy)[ep_idx[t]] = float_to_bf16(mllm_norm_column(x, add.next.weight != nullptr, ep_alpha2, ep_next[t]));
                } else if (mode == EPI_ADD_RESIDUAL) static_cast<float*>(C)[ep_idx[t]] = ep_old[t] + r;
                else if constexpr (!GATED) {
                    epilogue<bf16_t>(mode, r, 0.f, C, ep_idx[t]);
                    if (ep_slot >= 0 && ep_col[t] >= add.q_cols) {      // (only with slots: the row's place in the pages)
                        const int c = ep_col[t] - add.q_cols;
                        bf16_t* dst = c < add.kv_dim ? add.k_pages + c : add.v_pages + (c - add.kv_dim);
                        dst[static_cast<size_t>(ep_slot) * add.kv_dim] = float_to_bf16(r);
                    }
                }
            }
        }
        return;
    }
    for (int idx = tid; idx < MT * 256; idx += nw * 64) {
        const int i = idx / 256, r = (idx % 256) / 64, l = idx % 64;
        const int m = m_base + i * 16 + 4 * (l / 16) + r, nn = n0 + l % 16;
        if (m >= M || nn >= N) continue;
        const float bv = bias ? bias[nn] : 0.f;
        float v = 0.f;
        for (int w = 0; w < nw; ++w) v += red[(static_cast<size_t>(w) * MT + i) * 256 + r * 64 + l];
        epilogue<bf16_t>(mode, v, bv, C, static_cast<size_t>(m) * ldc + nn);
    }
}

constexpr int MAX_DYNAMIC_LDS = 160 * 1024 - 1024;      // the unit's LDS less the kernel's static variables
constexpr int SPLIT_COUNTERS = 4096;      // tiles that may be shared by several workgroups
constexpr int SPLIT_MAX_PARTS = 8;
constexpr int SPLIT_MIN_K_BLOCKS = 12;    // k blocks of 64 elements that every part keeps at least
constexpr int SPLIT_FROM_K_BLOCKS = 80;   // shorter K: the fences cost more than the parallelism gains (measured)

// What the few-row kernel is told in one word: rows of A (9 bits), columns a workgroup (6), parts of K (4), epilogue (4; one that does not
// exist stores nothing), wavefronts (5), an RMS norm, page slots, gathered rows.
static unsigned few_row_shape(int M, int cols_per_wg, int k_parts, int mode, int nw, bool rms, bool scatters, bool gathers) {
    return static_cast<unsigned>(M) | cols_per_wg << 9 | k_parts << 15 | (mode < 0 || mode > 15 ? 15 : mode) << 19 | nw << 23 |
           (rms ? 1u << 28 : 0u) | (scatters ? 1u << 29 : 0u) | (gathers ? 1u << 30 : 0u);
}

struct MergedA {        // A_MERGED: where the attention splits' states lie
    const float* split_o = nullptr;
    const float* split_ml = nullptr;
    int n_splits = 1, heads = 1, head_dim = 8;
};

template <bool LN_FUSED, bool MERGED = false>
static int launch_skinny(const void* A, int lda, const bf16_t* W, int ldw, const float* bias, void* C, int ldc,
                         int M, int N, int K, int mode, const float* gamma, const float* beta, float eps,
                         const int* rows, hipStream_t stream, void* workspace = nullptr, size_t workspace_bytes = 0,
                         MergedA merged = MergedA{}, int rms = 0, const MllmStreamAdd* through = nullptr,
                         KvScatter kv = KvScatter{}, const GatedPair* gated = nullptr) {
    static_assert(!(LN_FUSED && MERGED), "one source of A");
    const int tiles = (N + 15) / 16;
    const bool split_k = tiles < 1024;
    if (through != nullptr && (LN_FUSED || MERGED || !split_k)) return -2;
    if (gated != nullptr && (!LN_FUSED || !split_k)) return -2;
    if (kv.slots != nullptr && (through != nullptr || !split_k || mode != EPI_STORE)) return -2;
    // Narrow products: 16 rows per workgroup and one workgroup per 16 rows (more workgroups, each
    // reading only its rows). Wide products: every wavefront keeps all rows of its tile in
    // registers (up to 4 accumulators), so the weights are streamed once.
    int row_blocks = split_k ? (M + 15) / 16 : 1;
    int mt = split_k ? 1 : (M + 15) / 16;
    // Wide products without the fused norm: every wavefront needs all rows of A for its tile, as
    // many bytes as the tile's weights or more, so the workgroup copies its rows into LDS once
    // (at most 160 KB: more rows than fit are split over row blocks).
    const bool staged = !LN_FUSED && !split_k;
    size_t staged_bytes = 0;
    if (staged) {
        const size_t row16_bytes = static_cast<size_t>(16) * (K + 8) * sizeof(bf16_t);
        int fit = static_cast<int>((160 - 32) * 1024 / row16_bytes);      // 32 KB: the wavefronts' transposition regions
        if (fit < 1) return -2;
        if (fit > 4) fit = 4;
        row_blocks = (mt + fit - 1) / fit;
        mt = (mt + row_blocks - 1) / row_blocks;
        row_blocks = ((M + 15) / 16 + mt - 1) / mt;         // (as the kernel has it)
        staged_bytes = row16_bytes * mt;
    }
    int nw;
    int k_blocks = (K + 63) / 64;
    // Narrow products with a long K (from SPLIT_FROM_K_BLOCKS blocks): k_parts workgroups per tile,
    // as many as fit one round over the 256 compute units while each keeps at least
    // SPLIT_MIN_K_BLOCKS k blocks. Needs the workspace: SPLIT_COUNTERS counters, then 256 floats
    // per tile and part.
    int k_parts = 1;
    if (MERGED && (!split_k || M > 16 || merged.n_splits < 1 || merged.n_splits > MERGE_MAX_SPLITS ||
                   merged.head_dim % 8 != 0 || merged.heads * merged.head_dim != K))
        return -2;
    if (split_k && !LN_FUSED && !MERGED && workspace != nullptr && k_blocks >= SPLIT_FROM_K_BLOCKS) {
        const int wgs = tiles * row_blocks;
        k_parts = std::min(std::min(256 / std::max(wgs, 1), k_blocks / SPLIT_MIN_K_BLOCKS), SPLIT_MAX_PARTS);
        if (k_parts < 2 || wgs > SPLIT_COUNTERS ||
            workspace_bytes < SPLIT_COUNTERS * sizeof(int) + static_cast<size_t>(wgs) * k_parts * 256 * sizeof(float))
            k_parts = 1;
        k_blocks = (k_blocks + k_parts - 1) / k_parts;      // per workgroup from here on
    }
    // Two parts and at most 8 rows: one workgroup takes both, and the columns are dealt out to 256 workgroups (6 to 8 each) instead. What
    // it saves is the exchange of the parts' sums (stores, fences, a counter: about 2 us). 1,600 x 6,400 7.9 > 6.5 us at 1 row, 8.7 > 7.5 at
    // 8 (a chunk of five blocks with the exchange as it was: 7.6 and 8.4).
    const bool parts_inside = k_parts == 2 && M <= 8 && (N + 255) / 256 <= 8 && (k_blocks + 11) / 12 <= 6;
    int* part_counters = static_cast<int*>(workspace);
    float* part_sums = reinterpret_cast<float*>(static_cast<char*>(workspace) + SPLIT_COUNTERS * sizeof(int));
    if (split_k) {
        // the wavefront count (at least 4: one thread per output of the tile) that leaves every
        // wavefront the fewest k blocks; among equals the smallest, which has the least to add up
        // (the fused norm is written for 8 wavefronts, two rows each)
        // (at most 12: two chunks of loads in flight per wavefront need more than the 128 registers
        // that 16 wavefronts would leave each)
        nw = 4;
        for (int cand = 5; cand <= 12; ++cand)
            if ((k_blocks + cand - 1) / cand < (k_blocks + nw - 1) / nw) nw = cand;
        if (LN_FUSED) nw = 8;
    } else {
        // one round of workgroups over the 256 compute units, each wavefront one tile
        nw = (tiles * row_blocks + 255) / 256;
        nw = nw < 4 ? 4 : (nw > 16 ? 16 : nw);
    }
    // The LDS of a workgroup: the sums of its one or two tiles, the wavefronts' transposition regions (two k blocks at a time where the kernel
    // stages two), behind the fused norm its 16 normalised rows and the norm's vectors. (Two tiles fit up to K = 2,016 there.)
    const auto lds_bytes = [&](bool two) {
        size_t bytes = split_k ? static_cast<size_t>(nw) * mt * (two ? 2 : 1) * 256 * sizeof(float) : 0;
        bytes += static_cast<size_t>(nw) * (staged ? 2048 : LN_FUSED ? (two ? 8192 : 4096) : (two ? 6144 : 8192));
        return LN_FUSED ? bytes + static_cast<size_t>(16) * mt * (K + 8) * sizeof(bf16_t) + static_cast<size_t>(2) * K * sizeof(float) : bytes;
    };
    const bool two_fit = lds_bytes(true) <= MAX_DYNAMIC_LDS;
    // More than 256 tiles (and one row block): two tiles per workgroup, the columns dealt out evenly
    // to 256 workgroups.
    int cols_per_wg = 16;
    const bool dealt_out = !MERGED && gated == nullptr && split_k && row_blocks == 1 && k_parts == 1 && tiles > 256 && tiles <= 512 &&
                           (LN_FUSED || M <= 8) && two_fit;
    // The same behind the fused norm with 17 to 32 rows, 128 workgroups a row block: every workgroup normalises its 16 rows again, and more
    // than 256 of them share compute units. One and two tiles a workgroup, 32 rows, us: 2,304 x 768 7.4 > 6.6, 3,072 x 1,024 10.9 > 7.3,
    // 4,096 x 1,024 11.3 > 7.6, 3,600 x 1,600 14.7 > 9.2; two rounds of them pay only for a long K: 6,400 x 1,600 27.4 > 16.5, 5,120 x
    // 1,280 17.5 > 14.7, but 4,112 x 768 10.0 / 11.7, 10,000 x 768 15.4 / 17.2. (Norm and product apart: see norm_inside_pays of
    // the engine's ops.)
    const bool dealt_out_2 = gated == nullptr && split_k && LN_FUSED && row_blocks == 2 && tiles > 128 && (tiles <= 256 || K > 1024) && two_fit;
    const bool two_tiles = dealt_out || dealt_out_2 || gated != nullptr;      // (a gated pair: a tile of either map)
    if (dealt_out) cols_per_wg = (N + 255) / 256;
    if (dealt_out_2) {
        const int rounds = (tiles + 255) / 256;      // of 128 workgroups a row block, two tiles each
        cols_per_wg = (N + 128 * rounds - 1) / (128 * rounds);
    }
    // Fewer than 256 tiles, one row block and a long K (the second product of the feed-forward):
    // narrower tiles, down to 4 columns, so that more compute units share the weights. (Short K, or
    // the fused norm: the kernel's time is latency, not bytes, and nothing is gained; measured.)
    if (split_k && !LN_FUSED && !MERGED && row_blocks == 1 && (k_parts == 1 || parts_inside) && tiles < 256 && k_blocks >= (parts_inside ? 0 : 48))
        cols_per_wg = std::min(16, std::max((N + 255) / 256, 4));
    const int col_blocks = split_k ? (N + cols_per_wg - 1) / cols_per_wg : (tiles + nw - 1) / nw;
    // (what the words do not hold; K beyond 2^20: see the kernel's count of a wavefront's blocks)
    if (M > 511 || K > 1 << 20 || (MERGED && (N > 0x3fff || merged.heads > 511 || merged.head_dim > 511 * 8))) return -2;
    const unsigned shape = few_row_shape(M, cols_per_wg, k_parts, mode, nw, rms, kv.slots != nullptr, rows != nullptr);
    const unsigned columns = MERGED ? N | merged.head_dim / 8 << 14 | static_cast<unsigned>(merged.heads) << 23 : N;
    void* const strides = reinterpret_cast<void*>(static_cast<uintptr_t>(static_cast<unsigned>(lda)) | static_cast<uintptr_t>(static_cast<unsigned>(ldc)) << 32);
    const dim3 grid((col_blocks + N_XCD - 1) / N_XCD * N_XCD * row_blocks, parts_inside ? 1 : k_parts), block(nw * 64);
    const size_t smem = lds_bytes(two_tiles) + (parts_inside ? static_cast<size_t>(nw) * 256 * sizeof(float) : 0);
    if (staged) {
        staged_bytes += smem;
#define SKINNY_STAGED(MTV)                                                                             \
    case MTV: {                                                                                        \
        auto kernel = gemm_bf16_skinny<MTV, A_STAGED, false, 4>;                                        \
        hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(kernel),                      \
                                           hipFuncAttributeMaxDynamicSharedMemorySize,                 \
                                           static_cast<int>(staged_bytes));                            \
        if (e != hipSuccess) return static_cast<int>(e);                                               \
        kernel<<<grid, block, staged_bytes, stream>>>(W, A, bias, C, ldw, columns, shape, K, strides, nullptr, nullptr, nullptr, 0.f, \
                                                      nullptr, nullptr, KvScatter{});                  \
        break;                                                                                         \
    }
        switch (mt) {
            SKINNY_STAGED(1) SKINNY_STAGED(2) SKINNY_STAGED(3) SKINNY_STAGED(4)
            default: return -2;
        }
#undef SKINNY_STAGED
        return 0;
    }
    if (LN_FUSED) {
        if (K > 2048 || (reinterpret_cast<uintptr_t>(A) & 15) || lda % 4 != 0 ||
            (reinterpret_cast<uintptr_t>(gamma) & 15) || (reinterpret_cast<uintptr_t>(beta) & 15))
            return -2;
    }
    if (smem > MAX_DYNAMIC_LDS) return -2;
    constexpr int ASRC = LN_FUSED ? A_NORMED : (MERGED ? A_MERGED : A_GLOBAL);
    const void* p2 = LN_FUSED ? gamma : MERGED ? merged.split_ml : bias;
    const void* p3 = LN_FUSED ? (gated != nullptr ? static_cast<const void*>(gated->up) : beta) : MERGED ? static_cast<const void*>(bias) : C;
#define SKINNY_KERNEL(SPLIT, UV, A2, NTV, THROUGH, MSV, ONE, ...) SKINNY_ANY(SPLIT, UV, A2, NTV, THROUGH, MSV, ONE, false, 8, 16, __VA_ARGS__)
#define SKINNY_ANY(SPLIT, UV, A2, NTV, THROUGH, MSV, ONE, GATED, NUV, WCV, ...) SKINNY_PARTS(SPLIT, UV, A2, NTV, THROUGH, MSV, ONE, GATED, NUV, WCV, 1, false, __VA_ARGS__)
#define SKINNY_PARTS(SPLIT, UV, A2, NTV, THROUGH, MSV, ONE, GATED, NUV, WCV, KPV, TURN, ...)           \
    do {                                                                                               \
        auto kernel = gemm_bf16_skinny<1, ASRC, SPLIT, UV, A2, NTV, THROUGH, MSV, ONE, GATED, NUV, WCV, KPV, TURN>; \
        static bool lds_allowed = false;      /* more than 64 KB of dynamic LDS has to be asked for once */ \
        if (!lds_allowed) {                                                                            \
            hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(kernel),                  \
                                               hipFuncAttributeMaxDynamicSharedMemorySize, MAX_DYNAMIC_LDS); \
            if (e != hipSuccess) return static_cast<int>(e);                                           \
            lds_allowed = true;                                                                        \
        }                                                                                              \
        kernel<<<grid, block, smem, stream>>>(W, MERGED ? merged.split_o : A, p2, p3, ldw, columns, shape, MERGED ? ldc : K, \
                                              MERGED ? C : strides, bias, C, rows, eps, part_sums, part_counters, __VA_ARGS__); \
    } while (0)
#define SKINNY_TURNED(SPLIT, UV, A2, NTV, ONE, TURN)                                                   \
    do {                                                                                               \
        if constexpr (ASRC == A_GLOBAL) {                                                              \
            if (through != nullptr) { SKINNY_PARTS(SPLIT, UV, A2, NTV, true, MERGE_MAX_SPLITS, ONE, false, 8, 16, 1, TURN, *through); break; } \
        }                                                                                              \
        SKINNY_PARTS(SPLIT, UV, A2, NTV, false, MERGE_MAX_SPLITS, ONE, false, 8, 16, 1, TURN, kv);     \
    } while (0)
#define SKINNY_LAUNCH(SPLIT, UV, A2, NTV, ONE) SKINNY_TURNED(SPLIT, UV, A2, NTV, ONE, false)
// one chunk of UV / 2 blocks, or several
#define SKINNY_CHUNKS(UV, A2, NTV, TURN)                                                               \
    do {                                                                                               \
        if (per_wave <= UV / 2) SKINNY_TURNED(true, UV, A2, NTV, true, TURN);                          \
        else SKINNY_TURNED(true, UV, A2, NTV, false, TURN);                                            \
    } while (0)
// the same with narrow column tiles: chunks of four blocks
#define SKINNY_NARROW(WCV)                                                                              \
    do {                                                                                               \
        if (through != nullptr) {                                                                      \
            if (per_wave <= 4) SKINNY_ANY(true, 8, false, 1, true, MERGE_MAX_SPLITS, true, false, 8, WCV, *through); \
            else SKINNY_ANY(true, 8, false, 1, true, MERGE_MAX_SPLITS, false, false, 8, WCV, *through); \
        } else if (per_wave <= 4) SKINNY_ANY(true, 8, false, 1, false, MERGE_MAX_SPLITS, true, false, 8, WCV, kv); \
        else if (per_wave <= 6) SKINNY_ANY(true, 12, false, 1, false, MERGE_MAX_SPLITS, true, false, 8, WCV, kv); \
        else SKINNY_ANY(true, 8, false, 1, false, MERGE_MAX_SPLITS, false, false, 8, WCV, kv);          \
    } while (0)
    if (split_k) {
        // a chunk holds all k blocks of a wavefront when they are at most 3 (4 without the fused
        // norm and with at most 8 rows): whole chunks only, so nothing is requested twice, and
        // one chunk's registers are enough. (The largest chunks of the kernels without the norm spill a few registers
        // where a second one is in flight, and are still faster than smaller chunks.)
        const int per_wave = (k_blocks + nw - 1) / nw;
        if constexpr (MERGED) {
            // the splits' states of a whole chunk are in flight together: one chunk holds all of a
            // wavefront's k blocks, at most 3
            if (per_wave > 3) return -2;
#define SKINNY_MERGED(MSV)                                                                             \
    do {                                                                                               \
        if (M <= 8) {                                                                                  \
            switch (per_wave) {                                                                        \
                case 1: SKINNY_KERNEL(true, 2, false, 1, false, MSV, true, kv); break;                       \
                case 2: SKINNY_KERNEL(true, 4, false, 1, false, MSV, true, kv); break;                       \
                default: SKINNY_KERNEL(true, 6, false, 1, false, MSV, true, kv); break;                      \
            }                                                                                          \
        } else {                                                                                       \
            switch (per_wave) {                                                                        \
                case 1: SKINNY_KERNEL(true, 2, true, 1, false, MSV, true, kv); break;                        \
                case 2: SKINNY_KERNEL(true, 4, true, 1, false, MSV, true, kv); break;                        \
                default: SKINNY_KERNEL(true, 6, true, 1, false, MSV, true, kv); break;                       \
            }                                                                                          \
        }                                                                                              \
    } while (0)
            switch (merged.n_splits) {
                case 1: SKINNY_MERGED(1); break;
                case 2: SKINNY_MERGED(2); break;
                case 3: SKINNY_MERGED(3); break;
                default: SKINNY_MERGED(4); break;
            }
#undef SKINNY_MERGED
        } else if constexpr (LN_FUSED) {
            // (an instance for every count of a lane's float4s; two of them make one k block a wavefront. Two tiles take half the
            // blocks per chunk.)
#define SKINNY_NORMED(NUV)                                                                                                      \
    case NUV: {                                                                                                                 \
        constexpr int BLOCKS = (NUV + 1) / 2, U1 = BLOCKS > 3 ? 6 : 2 * BLOCKS, U2 = BLOCKS > 2 ? 4 : 2 * BLOCKS;                   \
        if (gated != nullptr) SKINNY_ANY(true, U2, false, 2, false, MERGE_MAX_SPLITS, BLOCKS <= U2 / 2, true, NUV, 16, *gated);         \
        else if (two_tiles) SKINNY_ANY(true, U2, false, 2, false, MERGE_MAX_SPLITS, BLOCKS <= U2 / 2, false, NUV, 16, kv);              \
        else SKINNY_ANY(true, U1, false, 1, false, MERGE_MAX_SPLITS, BLOCKS <= U1 / 2, false, NUV, 16, kv);                             \
        break;                                                                                                                  \
    }
            switch ((K + 255) / 256) {
                SKINNY_NORMED(1) SKINNY_NORMED(2) SKINNY_NORMED(3) SKINNY_NORMED(4)
                SKINNY_NORMED(5) SKINNY_NORMED(6) SKINNY_NORMED(7) SKINNY_NORMED(8)
                default: return -2;
            }
#undef SKINNY_NORMED
        } else if (two_tiles) {
            // (two tiles per chunk slot: half the blocks per chunk)
            SKINNY_CHUNKS(2, false, 2, false);
        } else if (M <= 8) {
            switch (std::min(per_wave, 4)) {
                case 1: SKINNY_LAUNCH(true, 2, false, 1, true); break;
                case 2: SKINNY_LAUNCH(true, 4, false, 1, true); break;
                case 3: SKINNY_LAUNCH(true, 6, false, 1, true); break;
                default:
                    if constexpr (ASRC == A_GLOBAL) {
                        if (parts_inside) {
#define SKINNY_INSIDE(UV)                                                                              \
    do {                                                                                               \
        if (through != nullptr) SKINNY_PARTS(true, UV, false, 1, true, MERGE_MAX_SPLITS, true, false, 8, 8, 2, false, *through); \
        else SKINNY_PARTS(true, UV, false, 1, false, MERGE_MAX_SPLITS, true, false, 8, 8, 2, false, kv);       \
    } while (0)
                            if (per_wave <= 4) SKINNY_INSIDE(8); else SKINNY_INSIDE(12);
#undef SKINNY_INSIDE
                            break;
                        }
                        if (cols_per_wg <= 4) { SKINNY_NARROW(4); break; }
                        if (cols_per_wg <= 8) { SKINNY_NARROW(8); break; }
                    }
                    // (rows in turn. 8 rows, in turn > in front: 2,304 x 3,072 5.6 > 5.8 us, 3,072 x 3,072 6.1 > 6.4; with up to three blocks
                    // 768 x 768 3.4 > 3.2, 1,600 x 1,600 4.4 > 4.1)
                    SKINNY_CHUNKS(8, false, 1, true);
                    break;
            }
        } else {
            switch (std::min(per_wave, 3)) {
                case 1: SKINNY_LAUNCH(true, 2, true, 1, true); break;
                case 2: SKINNY_LAUNCH(true, 4, true, 1, true); break;
                default:
                    // (In turn from two whole chunks on, in turn > in front: 16 rows of 1,024 x 4,096 13.1 > 13.5 us, 9 rows 12.5 > 13.0;
                    // with four and five blocks 3,072 x 3,072 7.0 > 6.9, 1,600 x 6,400 10.5 > 9.5, 32 rows of 2,304 x 3,072 11.4 > 11.0)
                    if (per_wave >= 6) SKINNY_TURNED(true, 6, true, 1, false, true);
                    else SKINNY_CHUNKS(6, true, 1, false);
                    break;
            }
        }
    } else {
        // wide products (the logits head): normalising the rows once in a kernel of its own and
        // staging them in LDS is faster than every workgroup normalising them again
        return -2;
    }
#undef SKINNY_NARROW
#undef SKINNY_CHUNKS
#undef SKINNY_LAUNCH
#undef SKINNY_TURNED
#undef SKINNY_KERNEL
#undef SKINNY_ANY
#undef SKINNY_PARTS
    return 0;
}


// Tile choice. A compute unit holds one workgroup at a time (its stages fill the LDS; of the six stages of plain 64x32 tiles it holds two, which their
// fitted numbers contain), so the workgroups of an XCD run in rounds of 32. A
// product is priced in microseconds as the launch, a round's start and end, and its k tiles, which take longer the more units load
// side by side. The numbers are fitted to 74 products of 96 to 8,000 rows, 768 to 6,400 columns and as many summed, each with rows that a
// kernel before it wrote and weights that no cache of an XCD holds, as a step has them: what is chosen takes 0.8 % more than the
// fastest of the tiles on average, where sums come in halves no more. (With rows and weights left in the caches 64x128 tiles beat
// 64x96 of two groups on the feed-forward's second product, 16.9 to 16.3 us; in a step they take 25.7 us and 22.3.)
// A K below the fitted ones is priced as their smallest, 768: for shorter sums the lines of the fit end in prices below zero (2,048 x 16,384
// x 64 83 us on 64x32, 25 on 128x256), and the results to store suit the same tiles as a k loop does: over 624 products of 33 to 8,192 rows,
// 64 to 50,257 columns and K of 32 to 512 0.6 % more than the fastest tile on average, 19 % at most.
struct TilePrice { int bm, bn; double launch, round, tile, load; };
static const TilePrice plain_tiles[] = {{128, 256, 4.15, -0.04, 0.583, 0.320}, {128, 192, 2.98, 0.89, 0.478, 0.232}, {128, 128, 2.39, 1.06, 0.362, 0.172},
                                        {64, 128, 1.57, 1.53, 0.290, 0.070},   {64, 64, 1.57, 1.55, 0.209, 0.051},   {64, 32, 3.80, -0.27, 0.138, 0.040}};
static const TilePrice halved_tiles[] = {{128, 256, 7.77, -5.49, 0.639, 0.299}, {128, 192, 4.61, -2.20, 0.522, 0.212}, {128, 128, 4.71, -2.01, 0.384, 0.182},
                                         {64, 128, 3.05, -0.29, 0.295, 0.085},  {64, 96, 2.08, 2.50, 0.215, 0.069},    {64, 64, 1.81, 1.69, 0.162, 0.071},
                                         {64, 32, 1.12, 2.01, 0.118, 0.044}};
static int cheapest_tile(const TilePrice* prices, int n, int M, int N, int K) {
    int best = 0;
    double best_price = 1e300;
    for (int c = 0; c < n; ++c) {
        const TilePrice& p = prices[c];
        const int tiles_m = (M + p.bm - 1) / p.bm, tiles_n = (N + p.bn - 1) / p.bn;
        int xm, xn;
        const int per_xcd = split_among_xcds(tiles_m, tiles_n, p.bm, p.bn, xm, xn) / N_XCD, rounds = (per_xcd + 31) / 32;
        const double k_tiles = std::max(12, (K + 63) / 64), blocks = static_cast<double>(tiles_m) * tiles_n;
        const double price = p.launch + rounds * (p.round + p.tile * k_tiles) + p.load * k_tiles * blocks / 256.0;
        if (price < best_price) { best_price = price; best = c; }
    }
    return best;
}

// Which products are summed in two halves (HALVES, or two groups of wavefronts). A rule of sizes alone, apart from the tile: the tile may change with
// what is measured, the order of the sums, and with it the last bit of every result, does not. Each of seven tile sizes is weighed as its
// rounds of 256 workgroups times its area over its efficiency, and the lightest says: 64x32, which is any product of up to 256 such tiles,
// halves; 64x64, 64x96 (results of up to 1,024 columns) and 128x128 halves from K = 2,048 on; the others never. (The efficiencies are
// those of the kernel that the rule was made for and price nothing any more. What it costs: by the prices 4 % of 2,048 x 1,600 x 6,400;
// few workgroups gain from halves, as two groups then share a tile's k loop.)
static bool sums_in_halves(int M, int N, int K) {
    struct Shape { int bm, bn; double efficiency; };
    static const Shape shapes[] = {{128, 256, 1.05}, {128, 192, 1.0}, {128, 128, 0.9}, {64, 128, 0.7},
                                   {64, 96, 0.65},   {64, 64, 0.55}, {64, 32, 0.4}};
    int best = 0;
    double best_cost = 1e300;
    for (int c = 0; c < 7; ++c) {
        if (c == 4 && N > 1024) continue;
        const long blocks = static_cast<long>((M + shapes[c].bm - 1) / shapes[c].bm) * ((N + shapes[c].bn - 1) / shapes[c].bn);
        const double cost = static_cast<double>((blocks + 255) / 256) * shapes[c].bm * shapes[c].bn / shapes[c].efficiency;
        if (cost < best_cost) { best_cost = cost; best = c; }
    }
    return best == 6 || (K >= 2048 && (best == 2 || best == 4 || best == 5));
}

static int gemm_bf16_dispatch(const void* A, int lda, const void* W, int ldw, const float* bias, void* C, int ldc,
                              int M, int N, int K, int mode, hipStream_t stream, KvScatter kv,
                              void* workspace = nullptr, size_t workspace_bytes = 0, const MllmStreamAdd* through = nullptr) {
    if (M <= 0 || N <= 0) return 0;
    if (K % 8 != 0 || lda % 8 != 0 || ldw % 8 != 0) return -1;
    if ((reinterpret_cast<uintptr_t>(A) & 15) || (reinterpret_cast<uintptr_t>(W) & 15)) return -1;
    const bf16_t* a = static_cast<const bf16_t*>(A);
    const bf16_t* w = static_cast<const bf16_t*>(W);
    // Which kernel for up to 256 rows. Up to 16 rows (one row block) and for the widest products (the
    // logits head) the weight-streaming kernel, always. In between both are priced, in microseconds,
    // by formulas fitted to measurements on the products of GPT-2 small to XL at 24 to 256 rows: the
    // weight-streaming kernel runs its 16-row by 16-column workgroups in rounds of 256 whose time
    // grows with K (steeply beyond 3072, where a wavefront's share of K no longer fits its chunks).
    // The tiles' formula is that of tiles loaded through registers and stays, as the two kernels add in another order and the line
    // between them is in every result's last bit. With today's tiles it still takes the faster kernel, within 5 %, for 108 of 120 products
    // of 20 to 256 rows of those models. The others (us, taken / the other kernel, operands cold): 20 to 32 rows of 4,800 and 6,400 x 1,600
    // 9.3 / 8.8 and 11.7 / 8.8, 40 and 48 of 2,304 x 768 5.5 / 4.6, 40 to 64 of 1,024 x 4,096 12.6 / 10.5, 96 and 128 of 768 x 768 5.1 / 4.5.
    const int col_tiles = (N + 15) / 16, row_blocks16 = (M + 15) / 16;
    auto streaming_is_faster = [&]() {
        const double rounds = static_cast<double>((static_cast<long>(col_tiles) * row_blocks16 + 255) / 256);
        const double streaming = 2.0 + rounds * (K <= 3072 ? 1.2 + 0.0008 * K : 0.0025 * K);
        const double blocks = static_cast<double>((M + 63) / 64) * ((N + 63) / 64);
        const bool ragged = K % 64 != 0;
        const double tiled = (blocks <= 128 ? 4.0 : 5.0) + 0.18 * (K / 64.0) * std::max(1.0, blocks / 256.0) + (ragged ? 2.0 : 0.0) +
                             (M <= 32 ? 4.0 : 0.0);       // (up to 32 rows the tiled kernel has one shape, 32x128)
        return streaming <= tiled;
    };
    const bool few_rows = M <= 16 || (M <= 64 && col_tiles >= 1024) || (M <= 256 && streaming_is_faster());
    // (Keys and values leave the weight-streaming kernel two bytes a lane, in rows of 32: up to 64 rows that costs less than the
    // copy it saves (a prompt of 7 tokens of GPT-2 small, with the norm inside as well: 443 -> 384 us), from 65 rows on the tiled
    // kernel's whole rows are faster again: 529 us a prompt of 65 tokens against 544.)
    if (few_rows && (kv.slots == nullptr || M <= 64) && launch_skinny<false>(A, lda, w, ldw, bias, C, ldc, M, N, K, mode, nullptr,
                                                                                nullptr, 0.f, nullptr, stream, workspace, workspace_bytes,
                                                                                MergedA{}, 0, through, kv) == 0) {
        // few rows: weight-streaming kernel
    } else {
#define TILE(...) launch_tiled<__VA_ARGS__>(a, lda, w, ldw, bias, C, ldc, M, N, K, mode, stream, kv, through)
        const bool far = lda > NEAR_ROWS || ldw > NEAR_ROWS, halves = M > 32 && sums_in_halves(M, N, K);
        if (far) {
            if (halves) TILE(2, 2, 1, 1, 128, 4, 2, false, true); else TILE(2, 2, 1, 1, 64, 6, 1, false, true);
        } else if (M <= 32) {
            TILE(1, 4, 1, 1, 64, 4);
        } else if (halves) {
            switch (cheapest_tile(halved_tiles, 7, M, N, K)) {
                case 0: TILE(2, 4, 2, 2, 64, 3, 1, true); break;
                case 1: TILE(4, 2, 1, 3, 64, 3, 1, true); break;
                case 2: TILE(4, 2, 1, 2, 64, 4, 1, true); break;
                case 3: TILE(2, 4, 1, 1, 64, 6, 1, true); break;
                case 4: TILE(2, 1, 1, 3, 128, 3, 2); break;
                case 5: TILE(2, 2, 1, 1, 128, 4, 2); break;
                default: TILE(2, 1, 1, 1, 128, 4, 2); break;
            }
        } else {
            switch (cheapest_tile(plain_tiles, 6, M, N, K)) {
                case 0: TILE(2, 4, 2, 2, 64, 3); break;
                case 1: TILE(4, 2, 1, 3, 64, 3); break;
                case 2: TILE(4, 2, 1, 2, 64, 4); break;
                case 3: TILE(2, 2, 1, 2, 64, 4); break;
                case 4: TILE(2, 2, 1, 1, 64, 6); break;
                default: TILE(2, 1, 1, 1, 64, 6); break;
            }
        }
#undef TILE
    }
    MLLM_LAUNCH_CHECK();
    return 0;
}

extern "C" {

// Returns 0, a HIP error code, or -1 when K or the row strides are not multiples of 8
// elements or a base pointer is not 16-byte aligned.
// `workspace` (optional; 4-byte aligned, zero when first handed over, never written by anyone else)
// lets narrow products of few rows and a long K share a tile among several workgroups: 16 KB of
// counters, then 1 KB per workgroup of such a launch (at most 256). Launches that use one
// workspace must not overlap.
int mllm_gemm_bf16(const void* A, int lda, const void* W, int ldw, const float* bias, void* C, int ldc,
                   int M, int N, int K, int mode, void* workspace, size_t workspace_bytes, hipStream_t stream) {
    return gemm_bf16_dispatch(A, lda, W, ldw, bias, C, ldc, M, N, K, mode, stream, KvScatter{}, workspace,
                              workspace_bytes);
}


// The product whose result is taken into the stream through norms (EPI_THROUGH): x [M, N] fp32 (row stride ldx), add.copy rows as
// far apart as x's. Workspace as above. -1: as above, or norms whose vectors are not 16-byte aligned.
int mllm_gemm_bf16_through(const void* A, int lda, const void* W, int ldw, const float* bias, float* x, int ldx, int M, int N, int K,
                           MllmStreamAdd add, void* workspace, size_t workspace_bytes, hipStream_t stream) {
    if (add.copy != nullptr && (add.ld_copy != ldx || (reinterpret_cast<uintptr_t>(add.copy) & 7))) return -1;
    for (const MllmTanhNorm* n : {&add.norm, &add.next})
        if (n->weight != nullptr && (n->alpha == nullptr || n->bias == nullptr || ((reinterpret_cast<uintptr_t>(n->weight) | reinterpret_cast<uintptr_t>(n->bias)) & 15))) return -1;
    return gemm_bf16_dispatch(A, lda, W, ldw, bias, x, ldx, M, N, K, EPI_THROUGH, stream, KvScatter{}, workspace, workspace_bytes, &add);
}

// The plain bf16 store (mode 0) with the key/value scatter of KvScatter fused: C = A W^T + bias, and
// columns [q_cols, q_cols + kv_dim) / [q_cols + kv_dim, q_cols + 2 kv_dim) of row m also go to row
// slots[m] (>= 0) of k_pages / v_pages ([rows, kv_dim] bf16). q_cols and kv_dim must be multiples
// of 4 and N == q_cols + 2 kv_dim; -1 otherwise or as mllm_gemm_bf16.
int mllm_gemm_bf16_kv(const void* A, int lda, const void* W, int ldw, const float* bias, void* C, int ldc,
                      int M, int N, int K, const int* slots, void* k_pages, void* v_pages, int q_cols, int kv_dim,
                      hipStream_t stream) {
    if (slots == nullptr || q_cols < 0 || kv_dim <= 0 || q_cols % 4 != 0 || kv_dim % 4 != 0 ||
        N != q_cols + 2 * kv_dim)
        return -1;
    KvScatter kv{slots, static_cast<bf16_t*>(k_pages), static_cast<bf16_t*>(v_pages), q_cols, kv_dim};
    return gemm_bf16_dispatch(A, lda, W, ldw, bias, C, ldc, M, N, K, EPI_STORE, stream, kv);
}

// The product whose A is the output of split decode attention, merged from the splits' states while it
// is loaded: C = epilogue(merge(states) W^T + bias) with A[m, h * head_dim + e] = sum_s w_s o_s[e] /
// sum_s w_s l_s, w_s = 2^(m_s - max m). M <= 16 tokens, n_splits <= 4, head_dim % 8 == 0, K = n_heads *
// head_dim <= 2304 or so. Returns 0, a HIP error code, -1 for misaligned operands, or -2 when the sizes
// are not ones this kernel takes (the caller then merges with mllm_merge_attention_splits and runs the
// ordinary product).
int mllm_gemm_bf16_merged(const float* split_o, const float* split_ml, int n_splits, int n_heads, int head_dim,
                          const void* W, int ldw, const float* bias, void* C, int ldc, int M, int N, int mode,
                          hipStream_t stream) {
    const int K = n_heads * head_dim;
    if (M <= 0 || N <= 0) return 0;
    if (K % 8 != 0 || ldw % 8 != 0 || (reinterpret_cast<uintptr_t>(W) & 15) ||
        (reinterpret_cast<uintptr_t>(split_o) & 15) || (reinterpret_cast<uintptr_t>(split_ml) & 7))
        return -1;
    MergedA merged{split_o, split_ml, n_splits, n_heads, head_dim};
    int rc = launch_skinny<false, true>(nullptr, K, static_cast<const bf16_t*>(W), ldw, bias, C, ldc, M, N, K, mode,
                                        nullptr, nullptr, 0.f, nullptr, stream, nullptr, 0, merged);
    if (rc != 0) return rc;
    MLLM_LAUNCH_CHECK();
    return 0;
}

// LayerNorm of the fp32 rows x[M,K] (row m taken from x[rows[m]] when `rows` is given) fused into the
// product with W[N,K]: C = epilogue(LN(x) W^T + bias).
// M <= 64, N < 16384. Returns 0, a HIP error code, -1 for misaligned operands, or -2 when M, N or K is too
// large for the fused kernel (the caller then runs the norm and the product separately).
int mllm_ln_gemm_bf16(const float* x, int ldx, const int* rows, const float* gamma, const float* beta, float eps,
                      const void* W, int ldw, const float* bias, void* C, int ldc, int M, int N, int K, int mode,
                      hipStream_t stream) {
    if (M <= 0 || N <= 0) return 0;
    if (K % 8 != 0 || ldw % 8 != 0 || (reinterpret_cast<uintptr_t>(W) & 15)) return -1;
    if (M > 64) return -2;
    int rc = launch_skinny<true>(x, ldx, static_cast<const bf16_t*>(W), ldw, bias, C, ldc, M, N, K, mode, gamma,
                                 beta, eps, rows, stream);
    if (rc != 0) return rc;
    MLLM_LAUNCH_CHECK();
    return 0;
}

// The norm and the product with the key/value scatter of mllm_gemm_bf16_kv (plain bf16 store, mode 0); return codes of both.
int mllm_ln_gemm_bf16_kv(const float* x, int ldx, const int* rows, const float* gamma, const float* beta, float eps, const void* W, int ldw,
                         const float* bias, void* C, int ldc, int M, int N, int K, const int* slots, void* k_pages, void* v_pages, int q_cols,
                         int kv_dim, hipStream_t stream) {
    if (M <= 0 || N <= 0) return 0;
    if (slots == nullptr || q_cols < 0 || kv_dim <= 0 || N != q_cols + 2 * kv_dim) return -1;
    if (K % 8 != 0 || ldw % 8 != 0 || (reinterpret_cast<uintptr_t>(W) & 15)) return -1;
    if (M > 64) return -2;
    const KvScatter kv{slots, static_cast<bf16_t*>(k_pages), static_cast<bf16_t*>(v_pages), q_cols, kv_dim};
    int rc = launch_skinny<true>(x, ldx, static_cast<const bf16_t*>(W), ldw, bias, C, ldc, M, N, K, EPI_STORE, gamma, beta, eps, rows, stream,
                                 nullptr, 0, MergedA{}, 0, nullptr, kv);
    if (rc != 0) return rc;
    MLLM_LAUNCH_CHECK();
    return 0;
}

// mllm_ln_gemm_bf16 with an RMS norm in front of the product: C = epilogue((x / sqrt(mean(x^2) + eps) * gamma) W^T + bias).
int mllm_rms_gemm_bf16(const float* x, int ldx, const int* rows, const float* gamma, float eps, const void* W, int ldw,
                       const float* bias, void* C, int ldc, int M, int N, int K, int mode, hipStream_t stream) {
    if (M <= 0 || N <= 0) return 0;
    if (K % 8 != 0 || ldw % 8 != 0 || (reinterpret_cast<uintptr_t>(W) & 15)) return -1;
    if (M > 64) return -2;
    int rc = launch_skinny<true>(x, ldx, static_cast<const bf16_t*>(W), ldw, bias, C, ldc, M, N, K, mode, gamma,
                                 nullptr, eps, rows, stream, nullptr, 0, MergedA{}, 1);
    if (rc != 0) return rc;
    MLLM_LAUNCH_CHECK();
    return 0;
}

// Gate and up map of a gated feed-forward in one product: out[m, n] = g sigmoid(alpha g) (u + 1) with g = min(a[m] . gate[n], limit)
// and u = clamp(a[m] . up[n], -limit, limit), bf16, both sums fp32. gate and up [N, K] with one row stride. Returns 0, a HIP
// error code or -1 as mllm_gemm_bf16. Two products and an activation each read or wrote the [M, N] values once more, in three
// launches; one product was faster at every size tried, 1 to 8192 rows (us, three launches > one): N 2048, K 768: 11.7 > 6.0 at
// 33 rows, 12.5 > 6.4 at 256, 35.2 > 17.6 at 2048, 106 > 70 at 8192; N 8192, K 3072: 24.3 > 16.9 at 1 row, 47 > 32 at 256,
// 979 > 829 at 8192. It is bound as the single product of 2 N columns is.
int mllm_gated_gemm_bf16(const void* A, int lda, const void* gate, const void* up, int ldw, float limit, float alpha, void* C, int ldc,
                         int M, int N, int K, hipStream_t stream) {
    if (M <= 0 || N <= 0) return 0;
    if (K % 8 != 0 || lda % 8 != 0 || ldw % 8 != 0) return -1;
    if ((reinterpret_cast<uintptr_t>(A) | reinterpret_cast<uintptr_t>(gate) | reinterpret_cast<uintptr_t>(up)) & 15) return -1;
    const bf16_t *a = static_cast<const bf16_t*>(A), *w = static_cast<const bf16_t*>(gate);
    const GatedPair pair{static_cast<const bf16_t*>(up), limit, alpha};
    // (the columns of both maps counted; few tiles of 64x64 are summed in halves, a rule that stays as sums_in_halves does)
    struct Shape { int bm, bn; double efficiency; };
    static const Shape shapes[] = {{128, 256, 1.05}, {128, 128, 0.9}, {64, 128, 0.7}, {64, 64, 0.55}};
    int best = 0;
    double best_cost = 1e300;
    for (int c = 0; c < 4; ++c) {
        const long blocks = static_cast<long>((M + shapes[c].bm - 1) / shapes[c].bm) * ((2L * N + shapes[c].bn - 1) / shapes[c].bn);
        const double cost = static_cast<double>((blocks + 255) / 256) * shapes[c].bm * shapes[c].bn / shapes[c].efficiency;
        if (cost < best_cost) { best_cost = cost; best = c; }
    }
    static const TilePrice gated_tiles[] = {plain_tiles[0], plain_tiles[2], plain_tiles[3]};
    const bool far = lda > NEAR_ROWS || ldw > NEAR_ROWS;
    if (best < 3) best = far ? 4 : cheapest_tile(gated_tiles, 3, M, 2 * N, K);
#define TILE(...) launch_tiled_gated<__VA_ARGS__>(a, lda, w, ldw, C, ldc, M, N, K, pair, stream)
    switch (best) {
        case 0: TILE(2, 4, 2, 2, 64, 3); break;
        case 1: TILE(4, 2, 1, 2, 64, 4); break;
        case 2: TILE(2, 2, 1, 2, 64, 4); break;
        case 3: if (far) TILE(2, 1, 1, 2, 128, 4, 2, false, true); else TILE(2, 1, 1, 2, 128, 4, 2); break;
        default: TILE(2, 2, 1, 2, 64, 4, 1, false, true); break;
    }
#undef TILE
    MLLM_LAUNCH_CHECK();
    return 0;
}

// The same behind the RMS norm of the fp32 rows x, normalised inside the product: M <= 64. Return codes of mllm_rms_gemm_bf16.
// Against two such products and the activation (us): N 2048, K 768: 11.3 > 4.8 at 8 rows, 12.8 > 5.7 at 32; N 6400, K 1600:
// 17.3 > 13.4 at 8 rows, 53 > 28 at 32.
int mllm_rms_gated_gemm_bf16(const float* x, int ldx, const float* gamma, float eps, const void* gate, const void* up, int ldw, float limit,
                             float alpha, void* C, int ldc, int M, int N, int K, hipStream_t stream) {
    if (M <= 0 || N <= 0) return 0;
    if (K % 8 != 0 || ldw % 8 != 0 || ((reinterpret_cast<uintptr_t>(gate) | reinterpret_cast<uintptr_t>(up)) & 15)) return -1;
    if (M > 64) return -2;
    const GatedPair pair{static_cast<const bf16_t*>(up), limit, alpha};
    int rc = launch_skinny<true>(x, ldx, static_cast<const bf16_t*>(gate), ldw, nullptr, C, ldc, M, N, K, EPI_STORE, gamma, nullptr, eps, nullptr,
                                 stream, nullptr, 0, MergedA{}, 1, nullptr, KvScatter{}, &pair);
    if (rc != 0) return rc;
    MLLM_LAUNCH_CHECK();
    return 0;
}

}  // extern "C"
