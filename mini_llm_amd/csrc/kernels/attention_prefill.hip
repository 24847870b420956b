// Prefill attention on the MFMA units of gfx950, bf16 with fp32 softmax: causal (optionally
// windowed) attention of a step's query rows over the paged cache. A workgroup takes 64
// consecutive queries of one sequence and one head; its four wavefronts take 16 queries each
// and walk the keys in tiles of 128, which are gathered through the block table into LDS (keys
// row-major, values transposed), so prompt portions that start anywhere read what earlier steps
// left in the pages. With eight wavefronts (head sizes 64 and 128) two wavefronts share 16 queries and
// take one half of every key tile each; their states are merged through LDS at the end. A launch lasts as
// long as its longest workgroup (the last 64 queries of the longest prompt, one key tile after the
// other), and halving a wavefront's share of a tile nearly halves that.
//
// Everything is computed transposed so that a lane owns ONE query:
//   S^T = K Q^T   (A = 16 keys x 32 dims from LDS, B = the lane's query fragment, held in registers)
//   O^T = V^T P^T (A = 16 dims x 32 keys from the transposed values, B = P^T straight from the S^T
//                  accumulators: the MFMA's k index may be permuted freely as long as both operands
//                  agree, so no shuffle or LDS round trip is needed)
// The running maximum and sum are then scalars per lane, merged over the four lane groups with two
// DPP steps. Recurrence: /root/reference/src/kernels/prefill/flashattention.cu:129-178, in base 2;
// the reference reads its keys from the step's own qkv buffer (:99-111) and so cannot continue a
// prompt from the cache.
#include "common.h"
#include "query_tiles.h"

#include <type_traits>

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x4 __attribute__((ext_vector_type(4)));

#define PF_BM 64
#define PF_BN 128
#define PF_TABLE_LDS 2048   // most block-table entries of a sequence (the table is staged in LDS)
#define PF_VT_STRIDE (PF_BN + 12)   // elements per transposed value row: 70 words, which spreads both the staging writes
                                    // (rows 8 apart) and the fragment reads (16 neighbouring rows, 4 word pairs each)
                                    // evenly over the banks (measured against 65, 66 and 68 words: 3 to 8 % of the kernel)

union Frag8 {
    bf16x8 v;
    uint4 q;
    uint32_t w[4];
    uint16_t h[8];
};

// (At most 2 wavefronts per SIMD: the compiler may then use 256 registers, and keeps both
// prefetched tiles in registers instead of private memory.)
// SHAPED: the scores are shaped before the softmax (score_shape.h: cap, distance bias), a chunked mask may stand in
// for the window, and the result may be multiplied by the sigmoid of a gate (fp32 rows, one value per output column).
// MODE 0: plain softmax; 1: shaped scores; 2: shaped scores whose weights are sigmoid(score + bias of the head), every
// visible key on its own: no running maximum, no sum, nothing to rescale, and the states of two wavefronts simply add.
// The weights are fp32 until they are packed for the second product, as the softmax's are.
template <int DH, int NW, int MODE, bool LONGEST_FIRST>
__global__ void __launch_bounds__(NW * 64) __attribute__((amdgpu_waves_per_eu(1, (DH >= 128 && NW == 4) ? 1 : 2)))
prefill_attention_kernel(// the first 14 dwords arrive in registers with the wavefront: what its tile, its queries and its table are found with
                         const int* __restrict__ cu_q, const int* __restrict__ ctx_len, const int* __restrict__ block_tables,
                         const bf16_t* __restrict__ q, int n_seqs, int places, int max_blocks, int q_stride,
                         const bf16_t* __restrict__ k_pages,
                         // the rest is loaded by the kernel
                         const bf16_t* __restrict__ v_pages, int kv_dim,
                         int n_heads, int n_kv_heads, int page_size, float scale_log2e, int window,
                         bf16_t* __restrict__ out, int out_stride, MllmScoreShape shape, float scale,
                         const float* __restrict__ gate, int ldg) {
    constexpr bool SHAPED = MODE != 0, SIGMOID = MODE == 2;
    constexpr int KS = DH / 32;            // k steps of S^T
    constexpr int DT = DH / 16;            // 16-dim tiles of O^T
    constexpr int KSTRIDE = DH + 8;
    constexpr int NTH = NW * 64;           // threads
    constexpr int KH = NW / 4;             // wavefronts per 16 queries: each takes 1/KH of a key tile
    constexpr int NT_PER = PF_BN / 16 / KH;      // 16-key groups of a tile per wavefront
    constexpr int SL_PER = PF_BN / 32 / KH;      // 32-key slabs of a tile per wavefront
    static_assert(NW == 4 || NW == 8, "one or two wavefronts per 16 queries");
    // two buffers of keys and of values: a tile is staged while the one before it is multiplied
    __shared__ __attribute__((aligned(16))) bf16_t Ks2[2][PF_BN * KSTRIDE];
    __shared__ __attribute__((aligned(16))) bf16_t Vt2[2][DH * PF_VT_STRIDE];
    extern __shared__ int sm_table[];          // the sequence's block table (max_blocks entries)

    // Heads vary fastest.
    const auto [b, tile, q_begin, q_len] = LONGEST_FIRST ? longest_tile<PF_BM>(cu_q, ctx_len, n_seqs, 1, blockIdx.y) : next_tile<PF_BM>(cu_q, n_seqs, 1, blockIdx.y, places);
    if (b < 0) return;                     // surplus workgroup; the whole workgroup leaves

    const int h = blockIdx.x;
    const int tid = threadIdx.x, lane = tid % 64;
    const int wave = __builtin_amdgcn_readfirstlane(tid / 64) % 4;      // which 16 queries
    const int kh = __builtin_amdgcn_readfirstlane(tid / 64) / 4;        // which part of every key tile
    const int G = lane / 16, c16 = lane % 16;
    // The sequence's block table goes to LDS first: the gathers below then depend on an LDS read, not on a global load that would have to be
    // waited for in front of every key load. Its whole row (the host passes at most PF_TABLE_LDS blocks, and rows are filled to their
    // end), so that neither it nor the queries wait for the context's length: one memory latency less in front of the first keys.
    const int* gtable = block_tables + static_cast<size_t>(b) * max_blocks;
    const int q0 = tile * PF_BM;
    const int qi = q0 + wave * 16 + c16;                  // this lane's query within the step's rows
    const int entry = gtable[min(tid, max_blocks - 1)];
    Frag8 qf[KS];
#pragma unroll
    for (int ks = 0; ks < KS; ++ks)      // a lane beyond the last query takes that query again; its scores are masked
        qf[ks].q = *reinterpret_cast<const uint4*>(q + static_cast<size_t>(q_begin + min(qi, q_len - 1)) * q_stride + h * DH + 32 * ks + 8 * G);
    const int start = ctx_len[b] - q_len;                 // position of the step's first query
    const int hk = n_heads == n_kv_heads ? h : small_quotient(h, small_quotient(n_heads, n_kv_heads));
    const bool q_ok = qi < q_len;
    const int p = start + qi;                             // its position
    const int p_first = start + q0;
    const int p_last = start + min(q0 + PF_BM, q_len) - 1;
    int k_lo = (window > 0 && p_first - window + 1 > 0) ? p_first - window + 1 : 0;
    const int chunk = SHAPED ? shape.chunk : 0;
    if (chunk > 0) k_lo = p_first - p_first % chunk;
    const float r1 = SHAPED ? mllm_bias_r1(shape, blockIdx.x) : 0.f, r2 = (SHAPED && shape.r1) ? shape.r2[blockIdx.x] : 0.f;
    const float sbias = (SIGMOID && shape.score_bias) ? shape.score_bias[blockIdx.x] : 0.f;
    // A window may keep the sequence's first kf positions visible. Key tiles that lie wholly in front of the window's
    // first tile and hold kept keys run first (n_head of them); the tiles are counted through, tile number vt being
    // key tile tile_of(vt). Their pages stay with the request, as the window's do.
    const int kf = (SHAPED && window > 0) ? shape.keep_first : 0;
    const int kt_first = k_lo / PF_BN, kt_last = p_last / PF_BN;
    const int n_head = kf > 0 ? min((kf + PF_BN - 1) / PF_BN, kt_first) : 0;
    const int vt_last = n_head + kt_last - kt_first;
    auto tile_of = [&](int vt) { return vt < n_head ? vt : vt - n_head + kt_first; };
    // (shaped scores are in base 2 already when they meet the exponent)
    const float sl = SHAPED ? 1.f : scale_log2e;
    const int shift = __ffs(page_size) - 1;       // (page sizes are powers of two)
    const int n_blocks_needed = (p_last >> shift) + 1;
    if (tid < max_blocks) sm_table[tid] = entry;
    for (int i = tid + NTH; i < n_blocks_needed; i += NTH) sm_table[i] = gtable[i];
    lds_barrier();        // (the queries stay in flight)
    auto page_row = [&](int j) -> size_t {
        return (static_cast<size_t>(sm_table[j >> shift]) << shift) + (j & (page_size - 1));
    };

    float m = -INFINITY, l = 0.f;
    f32x4 o[DT];
#pragma unroll
    for (int dt = 0; dt < DT; ++dt) o[dt] = f32x4{0.f, 0.f, 0.f, 0.f};
    const size_t kv_col = static_cast<size_t>(hk) * DH;

    // Tiles are fetched into registers ahead of their use, so the gather of the next keys and
    // values is in flight while the matrix cores work on the current ones. Every load of a fetch
    // is issued unconditionally, from a key clamped into [k_lo, p_last] (always a held page): a
    // load under a condition would make the compiler wait for all loads in flight. Keys outside
    // that range are masked in the scores, so what was loaded in their place never counts.
    // A thread takes KPT neighbouring keys (one group, inside one page) and 8 dims of them, keys
    // and values alike: one block-table lookup and one address per tile, the rest are constant
    // steps from it.
    constexpr int CH = DH / 8;                               // 16-byte chunks per row
    constexpr int KPT = PF_BN * CH / NTH;                    // keys per thread: 2, 4, 8 for head sizes 32, 64, 128 (half with 8 wavefronts)
    static_assert(KPT * NTH == PF_BN * CH && (KPT & (KPT - 1)) == 0 && KPT >= 2, "whole key groups per thread, keys in pairs");
    typedef unsigned int u32x4 __attribute__((ext_vector_type(4)));
    u32x4 ak[KPT], av[KPT];      // register set a: tiles of even order, in flight from memory
    u32x4 bk[KPT], bv[KPT];      // register set b: tiles of odd order
    const int ch = tid % CH, grp = tid / CH;
    const int g_lo = k_lo & ~(KPT - 1), g_hi = p_last & ~(KPT - 1);      // first keys of the groups that hold k_lo and p_last
    auto fetch = [&](u32x4 (&rk)[KPT], u32x4 (&rv)[KPT], int vt) {
        // (a group that holds a kept key lies in a page that is held: it is loaded where it is, its keys between the
        // kept ones and the window from the last kept key instead)
        const int G0 = tile_of(vt) * PF_BN + grp * KPT;
        const bool kept_grp = G0 < kf;
        const int g0 = min(kept_grp ? G0 : max(G0, g_lo), g_hi);
        const size_t base = page_row(g0) * kv_dim + kv_col + 8 * ch;
#pragma unroll
        for (int u = 0; u < KPT; ++u) {
            const int jj = g0 + u;
            const int jc = kept_grp ? (jj < kf ? jj : (jj < k_lo ? kf - 1 : jj)) : max(jj, k_lo);
            const int off = (min(jc, p_last) - g0) * kv_dim;     // stays inside the group
            rk[u] = *reinterpret_cast<const u32x4*>(k_pages + base + off);
            rv[u] = *reinterpret_cast<const u32x4*>(v_pages + base + off);
        }
    };
    auto stage = [&](const u32x4 (&rk)[KPT], const u32x4 (&rv)[KPT], int buf) {
        // keys row-major; values transposed: dim i of the thread's KPT keys becomes KPT/2 neighbouring words
        bf16_t* Ks = Ks2[buf];
        bf16_t* Vt = Vt2[buf];
#pragma unroll
        for (int u = 0; u < KPT; ++u)
            *reinterpret_cast<u32x4*>(Ks + (grp * KPT + u) * KSTRIDE + 8 * ch) = rk[u];
        Frag8 v[KPT];
#pragma unroll
        for (int u = 0; u < KPT; ++u) v[u].v = __builtin_bit_cast(bf16x8, rv[u]);
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            uint32_t w[KPT / 2];
#pragma unroll
            for (int u = 0; u < KPT; u += 2)
                w[u / 2] = static_cast<uint32_t>(v[u].h[i]) | (static_cast<uint32_t>(v[u + 1].h[i]) << 16);
            uint32_t* dst = reinterpret_cast<uint32_t*>(Vt + (8 * ch + i) * PF_VT_STRIDE + grp * KPT);
#pragma unroll
            for (int u = 0; u < KPT / 2; ++u) dst[u] = w[u];
        }
    };

    // Positions of this wavefront's first and last query: a key tile that every one of them sees
    // in full needs no mask.
    const int pw_min = start + q0 + wave * 16, pw_max = pw_min + 15;
    auto compute = [&](int vt, int buf, auto masked_tag) {
        constexpr bool MASKED = decltype(masked_tag)::value;
        const int j_base = tile_of(vt) * PF_BN;
        const bf16_t* Ks = Ks2[buf];
        const bf16_t* Vt = Vt2[buf];
        // S^T: s[nt][r] is the score of key j_base + 16*(nt0+nt) + 4*G + r with this lane's query
        const int nt0 = kh * NT_PER;
        float s[NT_PER][4];
        float tile_max = -INFINITY;
#pragma unroll
        for (int nt = 0; nt < NT_PER; ++nt) {
            f32x4 acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int ks = 0; ks < KS; ++ks) {
                const bf16x8 a = *reinterpret_cast<const bf16x8*>(Ks + (16 * (nt0 + nt) + c16) * KSTRIDE + 32 * ks + 8 * G);
                acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, qf[ks].v, acc, 0, 0, 0);
            }
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                s[nt][r] = acc[r];                   // raw dot product; the scale is applied with the exponent
                const int j = j_base + 16 * (nt0 + nt) + 4 * G + r;
                if constexpr (SIGMOID) {
                    const float z = mllm_shaped_score<true>(acc[r] * scale, shape, r1, r2, max(p - j, 0)) + sbias;
                    float w = __builtin_amdgcn_rcpf(1.f + fast_exp2(-z * MLLM_LOG2E));
                    if (MASKED) {
                        const bool seen = q_ok && j <= p && (window <= 0 || j > p - window || j < kf) && (chunk <= 0 || j >= p - p % chunk);
                        if (!seen) w = 0.f;
                    }
                    s[nt][r] = w;
                    continue;
                }
                if (SHAPED) s[nt][r] = mllm_shaped_score<true>(acc[r] * scale, shape, r1, r2, max(p - j, 0)) * MLLM_LOG2E;
                if (MASKED) {
                    const bool seen = q_ok && j <= p && (window <= 0 || j > p - window || j < kf) && (chunk <= 0 || j >= p - p % chunk);
                    if (!seen) s[nt][r] = -INFINITY;
                }
                tile_max = fmaxf(tile_max, s[nt][r]);
            }
        }
        if constexpr (!SIGMOID) {
        // the four lane groups of a query agree on the maximum
        tile_max = rows_max(tile_max);
        const float m_new = fmaxf(m, tile_max * sl);        // the scale is positive
        const float m_use = (m_new == -INFINITY) ? 0.f : m_new;      // nothing seen yet: all weights are 0
        const float alpha = fast_exp2(m - m_use);
        m = m_new;
        float psum = 0.f;
#pragma unroll
        for (int nt = 0; nt < NT_PER; ++nt)
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                s[nt][r] = fast_exp2(fmaf(s[nt][r], sl, -m_use));
                psum += s[nt][r];
            }
        l = l * alpha + psum;                 // this lane's share of the sum; merged over groups at the end
#pragma unroll
        for (int dt = 0; dt < DT; ++dt)
#pragma unroll
            for (int r = 0; r < 4; ++r) o[dt][r] *= alpha;
        }

        // O^T += V^T P^T over slabs of 32 keys. k slot i of lane group G stands for key
        // 32*slab + 4*G + i (i < 4) or 32*slab + 16 + 4*G + i - 4 (i >= 4) in both operands.
#pragma unroll
        for (int sl = 0; sl < SL_PER; ++sl) {
            const int slab = kh * SL_PER + sl;           // its place in the tile's transposed values
            Frag8 pf;
            pf.w[0] = pack_bf16x2(s[2 * sl][0], s[2 * sl][1]);
            pf.w[1] = pack_bf16x2(s[2 * sl][2], s[2 * sl][3]);
            pf.w[2] = pack_bf16x2(s[2 * sl + 1][0], s[2 * sl + 1][1]);
            pf.w[3] = pack_bf16x2(s[2 * sl + 1][2], s[2 * sl + 1][3]);
#pragma unroll
            for (int dt = 0; dt < DT; ++dt) {
                const uint32_t* vrow = reinterpret_cast<const uint32_t*>(Vt + (16 * dt + c16) * PF_VT_STRIDE);
                Frag8 vf;
                vf.w[0] = vrow[16 * slab + 2 * G];
                vf.w[1] = vrow[16 * slab + 2 * G + 1];
                vf.w[2] = vrow[16 * slab + 8 + 2 * G];
                vf.w[3] = vrow[16 * slab + 8 + 2 * G + 1];
                o[dt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(vf.v, pf.v, o[dt], 0, 0, 0);
            }
        }
    };

    auto run_tile = [&](int vt, int buf) {
        const int j_base = tile_of(vt) * PF_BN;
        const bool full = j_base + PF_BN - 1 <= pw_min && (window <= 0 || j_base > pw_max - window || j_base + PF_BN - 1 < kf) &&
                          (chunk <= 0 || j_base >= pw_max - pw_max % chunk);
        if (full) compute(vt, buf, std::false_type{}); else compute(vt, buf, std::true_type{});
    };

    // Tile t is multiplied from LDS buffer t % 2 while tile t+1 is written to the other buffer: one barrier
    // per tile. The loop body has no branch around a load; past the last tile the fetches repeat clamped
    // keys, which are staged and never multiplied.
    if constexpr (NW == 8) {
        // Two register sets, every tile requested two tiles ahead of its staging: with half a tile's
        // arithmetic per wavefront, one tile ahead is not enough and the loop runs at the latency of the
        // gather (measured).
        fetch(ak, av, 0);
        __builtin_amdgcn_sched_barrier(0);     // set a's loads stay the older ones, as on every later iteration
        fetch(bk, bv, 1);
        stage(ak, av, 0);
        fetch(ak, av, 2);
        lds_barrier();
        for (int vt = 0; vt <= vt_last; vt += 2) {
            stage(bk, bv, 1);                  // (its last readers passed the barrier that ended the tile before)
            fetch(bk, bv, vt + 3);
            run_tile(vt, 0);
            lds_barrier();
            stage(ak, av, 0);
            fetch(ak, av, vt + 4);
            if (vt + 1 <= vt_last) run_tile(vt + 1, 1);
            lds_barrier();
        }
    } else {
        // One register set, requested one tile ahead: a whole tile's arithmetic covers the gather, and the
        // registers saved keep more of the softmax's values out of the way (measured: 28.8 against 31.0 us
        // at 25 heads).
        fetch(ak, av, 0);
        stage(ak, av, 0);
        fetch(ak, av, 1);
        lds_barrier();
        for (int vt = 0; vt <= vt_last; ++vt) {
            const int buf = vt & 1;
            stage(ak, av, buf ^ 1);
            fetch(ak, av, vt + 2);
            run_tile(vt, buf);
            lds_barrier();
        }
    }
    if constexpr (KH == 2) {
        // The two wavefronts of a query group merge their states: the second leaves its maximum, its
        // share of the sum and its outputs in LDS (the tiles are done with), the first adds them.
        constexpr int STATE = 2 + 4 * DT;
        static_assert(sizeof(Ks2) >= 4 * 64 * STATE * sizeof(float), "the states fit the key buffers");
        float* state = reinterpret_cast<float*>(&Ks2[0][0]) + (wave * 64 + lane) * STATE;
        if (kh == 1) {
            state[0] = m;
            state[1] = l;
#pragma unroll
            for (int dt = 0; dt < DT; ++dt)
#pragma unroll
                for (int r = 0; r < 4; ++r) state[2 + 4 * dt + r] = o[dt][r];
        }
        lds_barrier();
        if (kh == 1) return;
        const float m1 = state[0];
        const float m_new = fmaxf(m, m1);
        const float m_use = (m_new == -INFINITY) ? 0.f : m_new;
        const float a0 = SIGMOID ? 1.f : fast_exp2(m - m_use), a1 = SIGMOID ? 1.f : fast_exp2(m1 - m_use);
        l = l * a0 + state[1] * a1;
#pragma unroll
        for (int dt = 0; dt < DT; ++dt)
#pragma unroll
            for (int r = 0; r < 4; ++r) o[dt][r] = o[dt][r] * a0 + state[2 + 4 * dt + r] * a1;
        m = m_new;                             // (what the sum and the outputs are now relative to: the sink below reads it)
    }
    l = rows_sum(l);
    if (!q_ok) return;
    if (SHAPED && !SIGMOID && shape.sink != nullptr) {
        // the sink: one more term of the denominator, exp(sink), without a value (the maximum is in base 2)
        const float sk = shape.sink[blockIdx.x] * MLLM_LOG2E, m_new = fmaxf(m, sk);
        const float a = fast_exp2(m - m_new);
        l = l * a + fast_exp2(sk - m_new);
#pragma unroll
        for (int dt = 0; dt < DT; ++dt)
#pragma unroll
            for (int r = 0; r < 4; ++r) o[dt][r] *= a;
    }
    const float inv = SIGMOID ? 1.f : 1.0f / l;
    const bool head_gate = SHAPED && gate != nullptr && shape.gate_per_head;
    const float hg = head_gate ? 1.f / (1.f + __expf(-gate[static_cast<size_t>(q_begin + qi) * ldg + blockIdx.x])) : 1.f;
    // o[dt][r] is dimension 16*dt + 4*G + r of this lane's query
    bf16_t* orow = out + static_cast<size_t>(q_begin + qi) * out_stride + h * DH;
#pragma unroll
    for (int dt = 0; dt < DT; ++dt) {
        float g4[4] = {1.f, 1.f, 1.f, 1.f};
        if (head_gate) {
            g4[0] = g4[1] = g4[2] = g4[3] = hg;
        } else if (SHAPED && gate != nullptr) {
            const float4 gv = *reinterpret_cast<const float4*>(gate + static_cast<size_t>(q_begin + qi) * ldg + blockIdx.x * DH + 16 * dt + 4 * G);
            g4[0] = 1.f / (1.f + __expf(-gv.x)); g4[1] = 1.f / (1.f + __expf(-gv.y));
            g4[2] = 1.f / (1.f + __expf(-gv.z)); g4[3] = 1.f / (1.f + __expf(-gv.w));
        }
        uint2 pk;
        pk.x = pack_bf16x2(o[dt][0] * inv * g4[0], o[dt][1] * inv * g4[1]);
        pk.y = pack_bf16x2(o[dt][2] * inv * g4[2], o[dt][3] * inv * g4[3]);
        *reinterpret_cast<uint2*>(orow + 16 * dt + 4 * G) = pk;
    }
}

extern "C" {

// n_tiles_upper: an upper bound of the number of 64-query tiles, sum over sequences of
// ceil(q_len / 64) (e.g. n_tokens / 64 + n_seqs); surplus workgroups leave at once.
// Returns 0, a HIP error code, or -1 when the head size is not 32, 64 or 128, the page size is no
// power of two or smaller than head_dim / 16 (a thread's group of keys must lie in one page), or a
// block table has more than PF_TABLE_LDS entries.
int mllm_prefill_attention_bf16(const void* q, int q_stride, int q_col, const void* k_pages, const void* v_pages,
                                int kv_dim, const int* block_tables, int max_blocks, const int* cu_q,
                                const int* ctx_len, int n_seqs, int n_tiles_upper, int n_heads, int n_kv_heads,
                                int head_dim, int page_size, float scale, int window, void* out, int out_stride,
                                hipStream_t stream, const MllmScoreShape* shape, const float* gate, int ldg) {
    if (n_seqs <= 0 || n_tiles_upper <= 0) return 0;
    // (the gate is read 16 bytes at a time)
    if (shape == nullptr && gate != nullptr) return -1;
    if (gate != nullptr && !shape->gate_per_head && (ldg % 4 != 0 || (reinterpret_cast<uintptr_t>(gate) & 15) != 0)) return -1;
    if (shape && window > 0 && shape->chunk > 0) return -1;
    const MllmScoreShape sh = shape ? *shape : MllmScoreShape{0.f, 0, nullptr, nullptr};
    if (n_heads % n_kv_heads != 0 || n_tiles_upper > 65535) return -1;
    if ((page_size & (page_size - 1)) != 0 || page_size < head_dim / 16 || max_blocks > PF_TABLE_LDS) return -1;
    const dim3 grid(n_heads, n_tiles_upper);
    const size_t table_bytes = static_cast<size_t>(max_blocks) * sizeof(int);
    const float sl2 = scale * 1.44269504088896340736f;
#define PF_LAUNCH_IN(D, W, S, L)                                                                                  \
    do {                                                                                                    \
        static bool lds_allowed = false;      /* static and dynamic LDS together pass 64 KB: asked for once */ \
        if (!lds_allowed) {                                                                                 \
            hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(prefill_attention_kernel<D, W, S, L>), \
                                               hipFuncAttributeMaxDynamicSharedMemorySize,                  \
                                               PF_TABLE_LDS * static_cast<int>(sizeof(int)));               \
            if (e != hipSuccess) return static_cast<int>(e);                                                \
            lds_allowed = true;                                                                             \
        }                                                                                                   \
        prefill_attention_kernel<D, W, S, L><<<grid, W * 64, table_bytes, stream>>>(                           \
            cu_q, ctx_len, block_tables, (const bf16_t*)q + q_col, n_seqs, n_tiles_upper, max_blocks, q_stride, (const bf16_t*)k_pages, \
            (const bf16_t*)v_pages, kv_dim, n_heads, n_kv_heads, page_size, sl2, window,                    \
            (bf16_t*)out, out_stride, sh, scale, gate, ldg);                                                \
    } while (0)
    const bool longest = longest_first(n_seqs, 4, static_cast<long long>(n_heads) * n_tiles_upper);
#define PF_LAUNCH(D, W, S) do { if (longest) PF_LAUNCH_IN(D, W, S, true); else PF_LAUNCH_IN(D, W, S, false); } while (0)
#define PF_CASE(D, W, KEY)                                                                                  \
    case KEY: {                                                                                             \
        if (shape && shape->sigmoid) PF_LAUNCH(D, W, 2);                                                    \
        else if (shape) PF_LAUNCH(D, W, 1);                                                                 \
        else PF_LAUNCH(D, W, 0);                                                                            \
        break;                                                                                              \
    }
    // Eight wavefronts (two per 16 queries, half a key tile each) shorten the longest workgroup's chain of
    // key tiles, which is what a launch of few workgroups lasts (2 x 1,024 tokens, 12 heads of 64: 384
    // workgroups, 20.6 -> 18.2 us); they also take a compute unit each, so launches of many workgroups, which
    // the units work off in rounds, keep four (25 heads, 800 workgroups: 28.5 us against 37.5). At head size
    // 128 a workgroup has a unit to itself either way.
    const bool eight = head_dim == 128 || (head_dim == 64 && static_cast<long>(n_heads) * n_tiles_upper <= 512);
    switch (head_dim * 2 + (eight ? 1 : 0)) {
        PF_CASE(32, 4, 64) PF_CASE(64, 4, 128) PF_CASE(64, 8, 129) PF_CASE(128, 8, 257)
        default: return -1;
    }
#undef PF_CASE
#undef PF_LAUNCH
#undef PF_LAUNCH_IN
    MLLM_LAUNCH_CHECK();
    return 0;
}

}  // extern "C"
