// Decode attention over the paged cache for gfx950: one query token per (token, head),
// its keys split over `nsplit` workgroups so that small batches still fill the chip.
//
// Inside a workgroup, LPK lanes share one key: each lane loads 16 bytes of the key row
// and of the value row (so a wavefront covers 64/LPK whole rows per load instruction),
// the LPK partial dot products are summed with DPP shuffles, and every lane keeps the
// running maximum, sum and its slice of the output for the keys of its lane group
// (recurrence of /root/reference/src/kernels/prefill/flashattention.cu:129-178, in base 2).
// Groups, wavefronts and splits are merged with the same (m, l, o) rule: within a wavefront every group is scaled to the largest
// maximum and the sums are scattered over the lanes, between the wavefronts a thread adds one element of all (exchanging whole states
// pairwise, twice, and scores as eight widened multiply-adds instead of four two-term ones cost 0.3 to 0.5 us more a launch: 192
// pairs 10.8 > 10.4 us, 384 15.4 > 15.1, 96 pairs in 32 bits 8.5 > 8.0, all inside a decode step). The splits of a
// (token, head) pair are merged either by the last workgroup to finish the pair, found through
// an atomic counter (no workgroup ever waits for another), or, with `partial_out`, not here at
// all: every workgroup leaves its state (maximum in base 2, sum, unnormalised output, fp32) in the
// workspace and the kernel that reads the attention output next merges them while it loads its
// operand (the few-row product of the output projection does), which costs no fence and no second
// pass here.
//
// It stands where the reference has its three-pass decode kernel
// (/root/reference/src/kernels/decode/paged_attention.cu:58-120); no 1e-6 is added to
// the denominator.
#include "common.h"

#define DEC_MAX_WAVES 16
#define DEC_TABLE_LDS 4096   // block-table entries staged in LDS: the most pages one workgroup's keys may span

// 16 bytes of a row: kept raw in registers while the load is in flight, widened to fp32 when used.
template <typename T> struct Vec16;
template <> struct Vec16<bf16_t> {
    static constexpr int N = 8;
    __device__ static void widen(const uint4& a, float (&v)[8]) {
        v[0] = __uint_as_float(a.x << 16); v[1] = __uint_as_float(a.x & 0xffff0000u);
        v[2] = __uint_as_float(a.y << 16); v[3] = __uint_as_float(a.y & 0xffff0000u);
        v[4] = __uint_as_float(a.z << 16); v[5] = __uint_as_float(a.z & 0xffff0000u);
        v[6] = __uint_as_float(a.w << 16); v[7] = __uint_as_float(a.w & 0xffff0000u);
    }
};
template <> struct Vec16<float> {
    static constexpr int N = 4;
    __device__ static void widen(const uint4& a, float (&v)[4]) {
        v[0] = __uint_as_float(a.x); v[1] = __uint_as_float(a.y);
        v[2] = __uint_as_float(a.z); v[3] = __uint_as_float(a.w);
    }
};
template <typename T>
__device__ __forceinline__ uint4 load_raw16(const T* p) { return *reinterpret_cast<const uint4*>(p); }
typedef unsigned int u32x4_nt __attribute__((ext_vector_type(4)));
template <typename T>
__device__ __forceinline__ uint4 load_stream16(const T* p) {
    const u32x4_nt v = __builtin_nontemporal_load(reinterpret_cast<const u32x4_nt*>(p));
    return make_uint4(v.x, v.y, v.z, v.w);
}

// A query's slice against 16 bytes of a key row: two bfloat16 products and their sum into fp32 in one instruction
// (v_dot2_f32_bf16), or four fp32 multiply-adds.
typedef __bf16 bf16x2_v __attribute__((ext_vector_type(2)));
__device__ __forceinline__ float dot_bf16x2(uint32_t a, uint32_t b, float acc) {
    return __builtin_amdgcn_fdot2_f32_bf16(__builtin_bit_cast(bf16x2_v, a), __builtin_bit_cast(bf16x2_v, b), acc, false);
}
template <typename T>
__device__ __forceinline__ float dot16(const uint4& q, const uint4& k) {
    if constexpr (sizeof(T) == 2) {
        return dot_bf16x2(q.w, k.w, dot_bf16x2(q.z, k.z, dot_bf16x2(q.y, k.y, dot_bf16x2(q.x, k.x, 0.f))));
    } else {
        float a[4], b[4];
        Vec16<float>::widen(q, a);
        Vec16<float>::widen(k, b);
        return fmaf(a[3], b[3], fmaf(a[2], b[2], fmaf(a[1], b[1], a[0] * b[0])));
    }
}

// Sums o over the wavefront's groups of LPK lanes; of the N sums a lane keeps N / (64 / LPK), at least one, from number
// group_kept<LPK, N>() on: at every step a lane hands half of what it still holds to its partner and takes the partner's share of
// the other half, so that 8 values over 8 groups take 7 additions and 7 exchanges instead of 24 of each.
template <int LPK, int N, int OFF = MLLM_WAVE / 2, int TOTAL = N>
__device__ __forceinline__ void group_scatter(float (&o)[TOTAL]) {
    if constexpr (OFF >= LPK) {
        if constexpr (N > 1) {
            constexpr int H = N / 2;
#pragma unroll
            for (int e = 0; e < H; ++e) {
                if constexpr (OFF >= 16) {
                    const unsigned a = __builtin_bit_cast(unsigned, o[e]), b = __builtin_bit_cast(unsigned, o[e + H]);
                    const auto r = OFF == 32 ? __builtin_amdgcn_permlane32_swap(a, b, false, false) : __builtin_amdgcn_permlane16_swap(a, b, false, false);
                    o[e] = __builtin_bit_cast(float, static_cast<unsigned>(r[0])) + __builtin_bit_cast(float, static_cast<unsigned>(r[1]));
                } else {
                    const bool high = threadIdx.x & OFF;
                    const float given = high ? o[e] : o[e + H], kept = high ? o[e + H] : o[e];
                    o[e] = kept + lane_xor(given, OFF);
                }
            }
            group_scatter<LPK, H, OFF / 2, TOTAL>(o);
        } else {
            o[0] += lane_xor(o[0], OFF);
            group_scatter<LPK, 1, OFF / 2, TOTAL>(o);
        }
    }
}
template <int LPK, int N, int OFF = MLLM_WAVE / 2>
__device__ __forceinline__ int group_kept() {
    if constexpr (OFF >= LPK && N > 1) return ((threadIdx.x & OFF) ? N / 2 : 0) + group_kept<LPK, N / 2, OFF / 2>();
    else return 0;
}
constexpr int group_share(int lpk, int n) { return n * lpk > MLLM_WAVE ? n * lpk / MLLM_WAVE : 1; }

// The states of a wavefront's lane groups (maximum, sum, slice of the output) as one, left in LDS: each is scaled to the largest
// maximum, and what is left are plain sums.
template <typename T, int LPK, int EPL>
__device__ __forceinline__ void wave_state(float m, float l, float (&o)[EPL], float* sm_m, float* sm_l, float* sm_o) {
    float mx = m;
#pragma unroll
    for (int off = LPK; off < MLLM_WAVE; off <<= 1) mx = fmaxf(mx, lane_xor(mx, off));
    const float f = exp2_for<T>(m - mx);
    l *= f;
#pragma unroll
    for (int off = LPK; off < MLLM_WAVE; off <<= 1) l += lane_xor(l, off);
#pragma unroll
    for (int e = 0; e < EPL; ++e) o[e] *= f;
    group_scatter<LPK, EPL>(o);
    const int lane = threadIdx.x % MLLM_WAVE, first = lane % LPK * EPL + group_kept<LPK, EPL>();
#pragma unroll
    for (int e = 0; e < group_share(LPK, EPL); ++e) sm_o[first + e] = o[e];
    if (lane == 0) { *sm_m = mx; *sm_l = l; }
}

template <typename T, int N>
__device__ __forceinline__ void merge_state(float& m, float& l, float (&o)[N], float m2, float l2,
                                            const float (&o2)[N]) {
    // empty states carry a large negative finite maximum and zero sums: their weight is 0 or
    // (both empty) irrelevant
    const float mn = fmaxf(m, m2);
    const float a = exp2_for<T>(m - mn), b = exp2_for<T>(m2 - mn);
    l = l * a + l2 * b;
#pragma unroll
    for (int e = 0; e < N; ++e) o[e] = o[e] * a + o2[e] * b;
    m = mn;
}

// SHAPED: the scores are shaped before the softmax and a chunked mask may stand in for the window (score_shape.h);
// the queries then come times the scale alone, and the shaped score goes to base 2 afterwards.
// MODE 0: plain softmax; 1: shaped scores; 2: shaped scores whose weights are sigmoid(score + bias of the head), every
// visible key on its own. The state keeps its form: the maximum stays 0 throughout, so every merge adds the outputs
// as they are, the sum is unused and nothing is divided at the end.
template <typename T, int LPK, int UNR, int MODE = 0>
__global__ void __launch_bounds__(UNR > 8 ? 512 : DEC_MAX_WAVES * MLLM_WAVE)
decode_attention_kernel(// the first 16 dwords arrive in registers with the wavefront: what the first loads need
                        const int* __restrict__ token_seq, const int* __restrict__ positions,
                        const int* __restrict__ block_tables, int max_blocks, int n_heads, int n_kv_heads,
                        int page_size, int window, int nsplit, const T* __restrict__ q, int q_stride, int q_col,
                        // the rest is loaded by the kernel
                        const T* __restrict__ k_pages, const T* __restrict__ v_pages, int kv_dim,
                        float scale_log2e, T* __restrict__ out, int out_stride,
                        float* __restrict__ ws_o, float* __restrict__ ws_ml, int* __restrict__ counters,
                        T* __restrict__ k_pages_w, T* __restrict__ v_pages_w, int k_col, int v_col,
                        const int* __restrict__ slots, int partial_out, MllmScoreShape shape,
                        const float* __restrict__ gate, int ldg) {
    constexpr bool SHAPED = MODE != 0, SIGMOID = MODE == 2;
    constexpr int EPL = Vec16<T>::N;        // elements per lane
    constexpr int DH = LPK * EPL;           // head size
    constexpr int KPW = MLLM_WAVE / LPK;    // keys per wavefront and load instruction
    __shared__ float sm_m[DEC_MAX_WAVES], sm_l[DEC_MAX_WAVES];
    __shared__ float sm_o[DEC_MAX_WAVES][DH];
    __shared__ int sm_last;
    __shared__ int sm_table[DEC_TABLE_LDS];
    const int n_waves = blockDim.x / MLLM_WAVE;

    const int pair = blockIdx.x, split = blockIdx.y;
    const int t = pair / n_heads, h = pair % n_heads;
    const int hk = h / (n_heads / n_kv_heads);
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / MLLM_WAVE), lane = threadIdx.x % MLLM_WAVE;
    const int c = lane % LPK, g = lane / LPK;
    // (token_seq == nullptr: every sequence brings one token, token t belongs to sequence t; the block
    // table can then be requested at once, beside the position, instead of after a load of its own)
    const int b = token_seq != nullptr ? token_seq[t] : t;
    const int* gtable_row = block_tables + static_cast<size_t>(b) * max_blocks;
    // Without a window the keys start at block 0 whatever the position is, and rows of the table are
    // filled to their end (zeros behind a sequence's last block): the whole row goes to LDS without
    // waiting for the position.
    const bool whole_row = window <= 0 && max_blocks <= DEC_TABLE_LDS;
    if (whole_row)
        for (int i = threadIdx.x; i < max_blocks; i += blockDim.x) sm_table[i] = gtable_row[i];
    const int p = positions[t];
    int lo = (window > 0 && p - window + 1 > 0) ? p - window + 1 : 0;
    if (SHAPED && shape.chunk > 0) lo = p - p % shape.chunk;
    const float r1 = SHAPED ? mllm_bias_r1(shape, h) : 0.f, r2 = (SHAPED && shape.r1) ? shape.r2[h] : 0.f;
    const float sbias = (SIGMOID && shape.score_bias) ? shape.score_bias[h] : 0.f;
    // The visible keys are counted through: first the kept first positions that lie in front of the window (none
    // without them), then the window's. Key number v stands at position key_at(v); kb, ke and the loops below count
    // in these numbers, so the splits share kept and window keys alike.
    const int kf = (SHAPED && window > 0 && shape.keep_first > 0) ? min(shape.keep_first, lo) : 0;
    const int shift_pos = lo - kf;
    auto key_at = [&](int v) { return v < kf ? v : v + shift_pos; };
    const int n_keys = p - lo + 1 + kf;
    const int per = (n_keys + nsplit - 1) / nsplit;
    const int kb = split * per;
    const int ke = min(n_keys, kb + per);
    // With `slots`, the token's own key and value are not in the pages yet: they are read from
    // its row of q (columns k_col, v_col), and written to the pages by the first query head of
    // each key/value head. That key is taken by one lane group after the loop over the pages.
    const bool append = slots != nullptr;
    const bool own_here = append && ke == n_keys && kb <= n_keys - 1;     // this workgroup's range holds the token itself
    const int ke_pages = own_here ? n_keys - 1 : ke;                      // keys [kb, ke_pages) come from the pages
    const size_t col = static_cast<size_t>(hk) * DH + c * EPL;
    const int shift = __ffs(page_size) - 1;                     // page sizes are powers of two

    // The block table entries of this workgroup's keys go to LDS first, so that no key load waits
    // for a table load.
    // (with kept first positions the keys of a range need not be neighbours: the table from block 0 on)
    const int first_blk = (whole_row || kf > 0) ? 0 : key_at(kb) >> shift;
    const int n_blk = ke_pages > kb ? (key_at(ke_pages - 1) >> shift) - first_blk + 1 : 0;
    if (!whole_row) {
        const int* gtable = gtable_row + first_blk;
        for (int i = threadIdx.x; i < n_blk; i += blockDim.x) sm_table[i] = gtable[i];
    }

    const uint4 qraw = load_raw16(q + static_cast<size_t>(t) * q_stride + q_col + h * DH + c * EPL);
    uint4 k_own = make_uint4(0, 0, 0, 0), v_own = make_uint4(0, 0, 0, 0);
    const bool own_lanes = own_here && wave == 0 && g == 0;
    if (own_lanes) {
        const T* src = q + static_cast<size_t>(t) * q_stride + col;
        k_own = load_raw16(src + k_col);
        v_own = load_raw16(src + v_col);
        const int slot = slots[t];
        if (slot >= 0 && h % (n_heads / n_kv_heads) == 0) {
            const size_t wrow = static_cast<size_t>(slot) * kv_dim + col;
            *reinterpret_cast<uint4*>(k_pages_w + wrow) = k_own;
            *reinterpret_cast<uint4*>(v_pages_w + wrow) = v_own;
        }
    }
    __syncthreads();       // the table is in LDS

    // Running state (maximum in base 2, sum, output slice). The maximum starts at a large
    // negative finite number, so that no difference of two of them is NaN.
    constexpr float NEG = -1.0e30f;
    constexpr float M0 = SIGMOID ? 0.f : NEG;       // an empty state's maximum
    float m = M0, l = 0.f, o[EPL];
#pragma unroll
    for (int e = 0; e < EPL; ++e) o[e] = 0.f;
    // A sink is one more term of the denominator, exp(sink), without a value: one lane group of the first split
    // starts from it instead of from nothing.
    if (SHAPED && !SIGMOID && shape.sink != nullptr && split == 0 && wave == 0 && g == 0) { m = shape.sink[h] * MLLM_LOG2E; l = 1.f; }

    // A wavefront takes UNR groups of 64/LPK keys at a time. All their loads are issued
    // first, unconditionally (a key beyond the range loads the last key of the range again and is
    // masked when used): a load under a condition, even one that is uniform over the wavefront,
    // makes every later use wait for all loads in flight (measured: 7.6 -> 8.4 us at 512 keys).
    const int mask = page_size - 1;
    const int group_keys = n_waves * KPW;                 // distance between a wavefront's groups
    for (int j0 = kb + wave * KPW; j0 < ke_pages; j0 += group_keys * UNR) {
        uint4 kraw[UNR], vraw[UNR];
#pragma unroll
        for (int u = 0; u < UNR; ++u) {
            const int j = key_at(min(j0 + u * group_keys + g, ke_pages - 1));
            const size_t row = (static_cast<size_t>(sm_table[(j >> shift) - first_blk]) << shift) + (j & mask);
            kraw[u] = load_stream16(k_pages + row * kv_dim + col);
            vraw[u] = load_stream16(v_pages + row * kv_dim + col);
        }
        float dot[UNR];
        float mx = NEG;
#pragma unroll
        for (int u = 0; u < UNR; ++u) {
            float d = group_sum<LPK>(dot16<T>(qraw, kraw[u])) * scale_log2e;
            const bool valid = j0 + u * group_keys + g < ke_pages;
            if (SHAPED) d = mllm_shaped_score<sizeof(T) == 2>(d, shape, r1, r2, valid ? p - key_at(j0 + u * group_keys + g) : 0) * MLLM_LOG2E;
            if (SIGMOID) {
                const float w = 1.f / (1.f + exp2_for<T>(-(d + sbias * MLLM_LOG2E)));
                dot[u] = valid ? w : 0.f;             // the weight itself
                continue;
            }
            dot[u] = valid ? d : NEG;
            mx = fmaxf(mx, dot[u]);
        }
        // one rescale of the state for the whole batch of keys
        const float mn = SIGMOID ? 0.f : fmaxf(m, mx);
        if (!SIGMOID) {
            const float a = exp2_for<T>(m - mn);
            l *= a;
#pragma unroll
            for (int e = 0; e < EPL; ++e) o[e] *= a;
        }
#pragma unroll
        for (int u = 0; u < UNR; ++u) {
            const float pj = SIGMOID ? dot[u] : dot[u] > NEG ? exp2_for<T>(dot[u] - mn) : 0.f;
            float vf[EPL];
            Vec16<T>::widen(vraw[u], vf);
            l += pj;
#pragma unroll
            for (int e = 0; e < EPL; ++e) o[e] = fmaf(pj, vf[e], o[e]);
        }
        m = mn;
    }
    if (own_lanes) {
        float vf[EPL];
        Vec16<T>::widen(v_own, vf);
        float d = group_sum<LPK>(dot16<T>(qraw, k_own)) * scale_log2e;
        if (SHAPED) d = mllm_shaped_score<sizeof(T) == 2>(d, shape, r1, r2, 0) * MLLM_LOG2E;
        const float mn = SIGMOID ? 0.f : fmaxf(m, d);
        const float a = SIGMOID ? 1.f : exp2_for<T>(m - mn);
        const float pj = SIGMOID ? 1.f / (1.f + exp2_for<T>(-(d + sbias * MLLM_LOG2E))) : exp2_for<T>(d - mn);
        l = l * a + pj;
#pragma unroll
        for (int e = 0; e < EPL; ++e) o[e] = o[e] * a + pj * vf[e];
        m = mn;
    }
    // Merges the states of all lane groups and wavefronts; `done` gets every element of the result (unnormalised) with the maximum and
    // the sum, each in a thread of its own.
    auto block_merge = [&](auto&& done) {
        wave_state<T, LPK, EPL>(m, l, o, &sm_m[wave], &sm_l[wave], sm_o[wave]);
        __syncthreads();
        for (int e = threadIdx.x; e < DH; e += blockDim.x) {
            float mx = sm_m[0];
            for (int w = 1; w < n_waves; ++w) mx = fmaxf(mx, sm_m[w]);
            float sum = 0.f, v = 0.f;
            for (int w = 0; w < n_waves; ++w) {
                const float f = exp2_for<T>(sm_m[w] - mx);
                sum = fmaf(f, sm_l[w], sum);
                v = fmaf(f, sm_o[w][e], v);
            }
            done(e, mx, sum, v);
        }
    };
    auto finish = [&](int e, float, float sum, float v) {
        float r = SIGMOID ? v : v / sum;
        if (SHAPED && gate != nullptr) r *= 1.f / (1.f + __expf(-gate[static_cast<size_t>(t) * ldg + (shape.gate_per_head ? h : h * DH + e)]));
        out[static_cast<size_t>(t) * out_stride + h * DH + e] = from_float<T>(r);
    };
    // (a split's state as it is: another kernel merges, or the last workgroup here)
    auto leave = [&](int e, float mx, float sum, float v) {
        const size_t slot = static_cast<size_t>(pair) * nsplit + split;
        ws_o[slot * DH + e] = v;
        if (e == 0) { ws_ml[slot * 2] = mx; ws_ml[slot * 2 + 1] = sum; }
    };
    if (nsplit == 1 && !partial_out) { block_merge(finish); return; }
    block_merge(leave);
    if (partial_out) return;
    // One thread's fences order the partial results around the counter (after the barrier its
    // release covers every thread's stores); a fence in every thread would write back and
    // invalidate the L2 once per wavefront, tens of microseconds in all.
    __syncthreads();
    if (threadIdx.x == 0) {
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "agent");
        const int arrived = __hip_atomic_fetch_add(&counters[pair], 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        sm_last = (arrived == nsplit - 1) ? 1 : 0;
        if (sm_last) __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "agent");
    }
    __syncthreads();
    if (!sm_last) return;
    // Last workgroup of this (token, head): lane group G takes split G (all loads in flight at
    // once), then the same merge as above.
    m = M0; l = 0.f;
#pragma unroll
    for (int e = 0; e < EPL; ++e) o[e] = 0.f;
    for (int s0 = 0; s0 < nsplit; s0 += n_waves * KPW) {
        const int sidx = s0 + wave * KPW + g;
        if (sidx < nsplit) {
            const size_t sl = static_cast<size_t>(pair) * nsplit + sidx;
            const float m2 = __hip_atomic_load(&ws_ml[sl * 2], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            const float l2 = __hip_atomic_load(&ws_ml[sl * 2 + 1], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            float o2[EPL];
#pragma unroll
            for (int e = 0; e < EPL; ++e)
                o2[e] = __hip_atomic_load(&ws_o[sl * DH + c * EPL + e], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            merge_state<T, EPL>(m, l, o, m2, l2, o2);
        }
    }
    block_merge(finish);
    if (threadIdx.x == 0) counters[pair] = 0;     // ready for the next launch
}

template <typename T>
static int launch_decode(int lpk, dim3 grid, int waves, hipStream_t stream, const T* q, int q_stride, int q_col,
                         const T* k_pages, const T* v_pages, int kv_dim, const int* block_tables,
                         int max_blocks, const int* token_seq, const int* positions, int n_heads,
                         int n_kv_heads, int page_size, float scale_log2e, int window, int nsplit, T* out,
                         int out_stride, float* ws_o, float* ws_ml, int* counters, T* k_pages_w, T* v_pages_w,
                         int k_col, int v_col, const int* slots, int partial_out, const MllmScoreShape* shape,
                         const float* gate, int ldg) {
    const MllmScoreShape sh = shape ? *shape : MllmScoreShape{0.f, 0, nullptr, nullptr};
#define DEC_ARGS token_seq, positions, block_tables, max_blocks, n_heads, n_kv_heads, page_size, window,  \
            nsplit, q, q_stride, q_col, k_pages, v_pages, kv_dim, scale_log2e, out, out_stride,        \
            ws_o, ws_ml, counters, k_pages_w, v_pages_w, k_col, v_col, slots, partial_out, sh, gate, ldg
#define DEC_CASE(L)                                                                                    \
    case L:                                                                                            \
        if (shape && shape->sigmoid) decode_attention_kernel<T, L, 8, 2><<<grid, waves * MLLM_WAVE, 0, stream>>>(DEC_ARGS); \
        else if (shape) decode_attention_kernel<T, L, 8, 1><<<grid, waves * MLLM_WAVE, 0, stream>>>(DEC_ARGS); \
        else decode_attention_kernel<T, L, 8, 0><<<grid, waves * MLLM_WAVE, 0, stream>>>(DEC_ARGS);      \
        return 0;
    switch (lpk) {
        DEC_CASE(2) DEC_CASE(4) DEC_CASE(8) DEC_CASE(16) DEC_CASE(32) DEC_CASE(64)
        default: return -1;
    }
#undef DEC_CASE
#undef DEC_ARGS
}

// Merges the splits' states that `partial_out` left in the workspace into the attention output, for readers of the output
// that do not merge while they load. One workgroup per (token, head): a thread takes 4 elements of every MERGE_THREADS /
// (head_dim / 4)-th split, whose states it asks for at once, and the threads' sums meet in LDS. Every split has one weight, against
// the maximum of all, and a lone state gets it where the sums are added: so many roundings as in one sum over all splits, or fewer.
// (One thread per 4 elements of all splits, in few workgroups, walked the splits one load after the other: 7.2 us for 12 heads of
// 64 in 15 splits, 3.0 us now.)
#define MERGE_THREADS 256
template <typename T>
__global__ void __launch_bounds__(MERGE_THREADS)
merge_splits_kernel(const float* __restrict__ ws_o, const float* __restrict__ ws_ml, int nsplit, int head_dim, int n_heads, T* __restrict__ out, int out_stride) {
    __shared__ __attribute__((aligned(16))) float4 o_s[MERGE_THREADS];
    __shared__ float2 wl_s[MERGE_THREADS];          // weight still to be applied, sum
    __shared__ float max_s[MERGE_THREADS / MLLM_WAVE];
    // (blockIdx.y: 4 MERGE_THREADS elements of heads wider than that)
    const int pair = blockIdx.x, quad0 = blockIdx.y * MERGE_THREADS, quads = min(head_dim / 4 - quad0, MERGE_THREADS), groups = MERGE_THREADS / quads;
    const int quad = threadIdx.x % quads, group = threadIdx.x / quads;
    const float* state = ws_ml + static_cast<size_t>(pair) * nsplit * 2;
    const float* values = ws_o + static_cast<size_t>(pair) * nsplit * head_dim + 4 * (quad0 + quad);
    // (surplus threads and groups take the last split along and drop it)
    int s = min(group, nsplit - 1);
    float2 ml = *reinterpret_cast<const float2*>(state + 2 * s);
    float4 v = *reinterpret_cast<const float4*>(values + static_cast<size_t>(s) * head_dim);
    float mx = ml.x;
    for (int i = threadIdx.x; i < nsplit; i += MERGE_THREADS) mx = fmaxf(mx, state[2 * i]);
    mx = wave_max(mx);
    if (threadIdx.x % MLLM_WAVE == 0) max_s[threadIdx.x / MLLM_WAVE] = mx;
    __syncthreads();
    mx = fmaxf(fmaxf(max_s[0], max_s[1]), fmaxf(max_s[2], max_s[3]));
    float w = exp2_for<T>(ml.x - mx), l = ml.y, o[4] = {v.x, v.y, v.z, v.w};
    if (group < groups) {
        if (s + groups < nsplit) {
            l *= w;
#pragma unroll
            for (int e = 0; e < 4; ++e) o[e] *= w;
            for (s += groups; s < nsplit; s += groups) {
                ml = *reinterpret_cast<const float2*>(state + 2 * s);
                v = *reinterpret_cast<const float4*>(values + static_cast<size_t>(s) * head_dim);
                w = exp2_for<T>(ml.x - mx);
                l += w * ml.y;
                o[0] += w * v.x; o[1] += w * v.y; o[2] += w * v.z; o[3] += w * v.w;
            }
            w = 1.f;
        }
        o_s[threadIdx.x] = make_float4(o[0], o[1], o[2], o[3]);
        wl_s[threadIdx.x] = make_float2(w, l);
    }
    __syncthreads();
    if (group > 0) return;
    l *= w;
#pragma unroll
    for (int e = 0; e < 4; ++e) o[e] *= w;
    for (int g = 1; g < min(groups, nsplit); ++g) {
        v = o_s[g * quads + quad];
        const float2 wl = wl_s[g * quads + quad];
        l += wl.x * wl.y;
        o[0] += wl.x * v.x; o[1] += wl.x * v.y; o[2] += wl.x * v.z; o[3] += wl.x * v.w;
    }
    const float inv = 1.0f / l;
    T* dst = out + static_cast<size_t>(pair / n_heads) * out_stride + (pair % n_heads) * head_dim + 4 * (quad0 + quad);
#pragma unroll
    for (int k = 0; k < 4; ++k) dst[k] = from_float<T>(o[k] * inv);
}

// ---------------------------------------------------------------------------------------------
// Norm, QKV product and decode attention of few tokens in one kernel (bfloat16, heads of 64, as many key/value heads as query
// heads, one token a sequence). At few rows the QKV product is a chain of latencies and so is the attention behind it, and between
// the two stands the boundary of dependent kernels. Here every workgroup of a (token, head, split) makes the head's query itself: the norm
// of the token's row, then 64 rows of the weights times it (98 KB at width 768, which the workgroups of a head share through
// their XCD's L2), while the keys and values of its range are on their way from the pages. The new key is made by split 0, the new
// value by split 1, and both go to the pages; nobody reads them back: the token's own key is a state of its own behind the
// splits' (maximum = its score, sum 1, output = its value), which split 0 and split 1 leave together, and whoever merges the
// states merges it like any other. One workgroup a pair makes all three, merges all itself and leaves the result. No workgroup waits
// for another. Query, key and value are rounded to bfloat16 as the product of its own would leave them.
// What bounds it is the chain launch, row, norm, product, scores, merge, and what a unit takes from its L2 (196 KB of weights and
// 98 KB of keys and values a workgroup at 8 tokens and 768 keys). Measured in a decode step of width 768, 12 heads, against product and
// attention as two kernels: 1 token at 130 keys 6.6 us (5.0 + 5.9), 8 tokens at 540 9.3 (5.2 + 7.6), 16 tokens of a queue 14.0 (6.1 + 10.4).
// A wavefront owns 8 of the head's 64 columns of each product: 8 lanes share a weight row, one 128-byte line of it a load, so
// that no sum crosses a wavefront. All of the first requests' weights are asked for behind the row and the norm's vectors, the
// keys and values behind the weights: loads complete in that order, and each is waited for only where it is used.
// ---------------------------------------------------------------------------------------------
#define QKV_WAVES 8
#define QKV_DH 64
#define QKV_MAX_K 2048         // a thread takes four columns of the row

struct QkvAttention {
    const int* token_blocks;      // [T, max_blocks]
    int max_blocks;
    const int* positions;
    int T, H, S;                  // tokens, heads, splits
    unsigned per_s, per_t;        // 2^32 / S and 2^32 / T, rounded up: quotients of small numbers by one multiplication
    const float* x;               // fp32 stream [T, K]
    int ldx, K;
    const float *gamma, *beta;
    float eps;
    const bf16_t* w;              // [3 H 64, K]
    int ldw;
    const float* bias;
    bf16_t *k_pages, *v_pages;
    int kv_dim, page_shift;
    const int* slots;
    float scale_log2e;
    float *ws_o, *ws_ml;          // states of the splits, or
    bf16_t* out;                  // the result
    int out_stride;
};

struct QkvShared {
    int table[DEC_TABLE_LDS];
    uint4 x[QKV_MAX_K / 8 + 32];                             // the normalised row, zeros behind it
    uint4 made[3][QKV_DH / 8];                               // query, and key and value where the workgroup makes them
    float m[QKV_WAVES + 1], l[QKV_WAVES + 1], o[QKV_WAVES + 1][QKV_DH];
    float sum[QKV_WAVES], sq[QKV_WAVES];
};

// CB: 128-byte lines of a weight row in one request, of which two are under way (TWO: they hold the whole row). UNR: groups of 64 keys
// whose loads are in flight together. MATS: 1 the query, 2 and a key (split 0) or a value (split 1), 3 all three, and with them the
// whole attention.
template <int CB, bool TWO, int UNR, int MATS>
__device__ __forceinline__ void qkv_attention_body(const QkvAttention& a, int t, int h, int split, QkvShared& sm) {
    const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid / 64), lane = tid % 64;
    const int c = lane % 8, g = lane / 8;
    const int K = a.K, nq = K / 4;
    const int* table = a.token_blocks + static_cast<size_t>(t) * a.max_blocks;
    // requested first: the table (every key's address hangs on it), the thread's own four columns of the row, the norm's vectors
    const int tab = table[min(tid, a.max_blocks - 1)];
    const int p = a.positions[t];
    const int own = min(tid, nq - 1);
    const float4 xt = reinterpret_cast<const float4*>(a.x + static_cast<size_t>(t) * a.ldx)[own], gt = reinterpret_cast<const float4*>(a.gamma)[own];
    float4 bt = reinterpret_cast<const float4*>(a.beta != nullptr ? a.beta : a.gamma)[own];
    if (a.beta == nullptr) bt = make_float4(0.f, 0.f, 0.f, 0.f);
    __builtin_amdgcn_sched_barrier(0);
    const int q_dim = a.H * QKV_DH, row = h * QKV_DH + wave * 8 + g;
    const bf16_t* w[MATS];
    float bias[MATS];
#pragma unroll
    for (int m = 0; m < MATS; ++m) {
        const int r = row + (MATS == 2 && m == 1 && split == 1 ? 2 : m) * q_dim;
        w[m] = a.w + static_cast<size_t>(r) * a.ldw;
        bias[m] = a.bias != nullptr ? a.bias[r] : 0.f;
    }
    uint4 w0[MATS][CB], w1[MATS][CB];
    auto load_weights = [&](uint4 (&wr)[MATS][CB], int chunk) {
#pragma unroll
        for (int i = 0; i < CB; ++i) {
            const int k = min((chunk * CB + i) * 64, K - 64) + 8 * c;       // (lines beyond the row: its last one, against zeros)
#pragma unroll
            for (int m = 0; m < MATS; ++m) wr[m][i] = load_raw16(w[m] + k);
        }
        __builtin_amdgcn_sched_barrier(0);
    };
    load_weights(w0, 0);
    load_weights(w1, 1);
    if (tid < a.max_blocks) sm.table[tid] = tab;
    for (int i = tid + 64 * QKV_WAVES; i < a.max_blocks; i += 64 * QKV_WAVES) sm.table[i] = table[i];
    // the norm: the mean first, then the variance of the centred values
    const float s = wave_sum(tid < nq ? (xt.x + xt.y) + (xt.z + xt.w) : 0.f);
    if (lane == 0) sm.sum[wave] = s;
    lds_barrier();

    // the split's keys: those in the pages, positions 0 to p - 1
    const int per = MATS == 3 ? p : (p + a.S - 1) / a.S, kb = split * per, ke = min(p, kb + per);
    const size_t col = static_cast<size_t>(h) * QKV_DH + 8 * c;
    const int mask = (1 << a.page_shift) - 1;
    uint4 kraw[UNR], vraw[UNR];
    auto load_keys = [&](int j0) {
#pragma unroll
        for (int u = 0; u < UNR; ++u) {
            // (beyond the range: its last key again, masked when used; without a key before the token: the token's own row, dropped)
            const int j = max(min(j0 + 64 * u + g, ke - 1), 0);
            const size_t r = (static_cast<size_t>(sm.table[j >> a.page_shift]) << a.page_shift) + (j & mask);
            kraw[u] = load_stream16(a.k_pages + r * a.kv_dim + col);
            vraw[u] = load_stream16(a.v_pages + r * a.kv_dim + col);
        }
        __builtin_amdgcn_sched_barrier(0);
    };
    load_keys(kb + 8 * wave);

    float mean = 0.f, var = 0.f;
#pragma unroll
    for (int i = 0; i < QKV_WAVES; ++i) mean += sm.sum[i];
    mean /= static_cast<float>(K);
    const float d0 = xt.x - mean, d1 = xt.y - mean, d2 = xt.z - mean, d3 = xt.w - mean;
    const float q2 = wave_sum(tid < nq ? (d0 * d0 + d1 * d1) + (d2 * d2 + d3 * d3) : 0.f);
    if (lane == 0) sm.sq[wave] = q2;
    lds_barrier();
#pragma unroll
    for (int i = 0; i < QKV_WAVES; ++i) var += sm.sq[i];
    const float inv = 1.0f / sqrtf(var / static_cast<float>(K) + a.eps);
    {
        uint2 pk = make_uint2(0, 0);           // (zeros behind the row, as far as whole requests of its weights reach)
        if (tid < nq) {
            pk.x = pack_bf16x2(d0 * inv * gt.x + bt.x, d1 * inv * gt.y + bt.y);
            pk.y = pack_bf16x2(d2 * inv * gt.z + bt.z, d3 * inv * gt.w + bt.w);
        }
        reinterpret_cast<uint2*>(sm.x)[tid] = pk;
        static_assert(64 * QKV_WAVES * 4 == QKV_MAX_K && (TWO ? 2 * CB : CB + 31) * 8 <= QKV_MAX_K / 8 + 32, "whole requests stay inside the row and its zeros");
        if (!TWO && tid < 64) reinterpret_cast<uint2*>(sm.x)[QKV_MAX_K / 4 + tid] = make_uint2(0, 0);
    }
    lds_barrier();
    float acc[MATS][2];
#pragma unroll
    for (int m = 0; m < MATS; ++m) acc[m][0] = acc[m][1] = 0.f;
    auto use_weights = [&](const uint4 (&wr)[MATS][CB], int chunk) {
#pragma unroll
        for (int i = 0; i < CB; ++i) {
            const uint4 xv = sm.x[(chunk * CB + i) * 8 + c];
#pragma unroll
            for (int m = 0; m < MATS; ++m) {
                acc[m][0] = dot_bf16x2(wr[m][i].x, xv.x, acc[m][0]);
                acc[m][1] = dot_bf16x2(wr[m][i].y, xv.y, acc[m][1]);
                acc[m][0] = dot_bf16x2(wr[m][i].z, xv.z, acc[m][0]);
                acc[m][1] = dot_bf16x2(wr[m][i].w, xv.w, acc[m][1]);
            }
        }
    };
    if constexpr (TWO) {
        use_weights(w0, 0);
        use_weights(w1, 1);
    } else {
        const int chunks = (K / 64 + CB - 1) / CB;
        for (int i = 0; i < chunks; i += 2) {
            // (past the end: the row's last line, long since arrived)
            use_weights(w0, i);
            load_weights(w0, i + 2);
            if (i + 1 < chunks) use_weights(w1, i + 1);
            load_weights(w1, i + 3);
        }
    }
#pragma unroll
    for (int m = 0; m < MATS; ++m) {
        const float v = group_sum<8>(acc[m][0] + acc[m][1]) + bias[m];
        if (c == 0) reinterpret_cast<bf16_t*>(sm.made[m])[wave * 8 + g] = float_to_bf16(v);
    }
    lds_barrier();

    const size_t pair = static_cast<size_t>(t) * a.H + h;
    const int states = a.S + 1;
    if (MATS > 1 && wave == 0) {
        // the token's own key and value: to the pages, and as a state of their own
        const int slot = a.slots[t];
        const bf16_t mine = reinterpret_cast<const bf16_t*>(sm.made[1])[lane], mine_v = reinterpret_cast<const bf16_t*>(sm.made[MATS - 1])[lane];
        const size_t at = static_cast<size_t>(slot) * a.kv_dim + h * QKV_DH + lane, own_state = pair * states + a.S;
        if (slot >= 0 && split == 0) a.k_pages[at] = mine;
        if (slot >= 0 && (MATS == 3 || split == 1)) a.v_pages[at] = mine_v;
        if (split == 0) {
            const float d = wave_sum(bf16_to_float(reinterpret_cast<const bf16_t*>(sm.made[0])[lane]) * bf16_to_float(mine)) * a.scale_log2e;
            if (lane == 0) {
                if (MATS == 3) { sm.m[QKV_WAVES] = d; sm.l[QKV_WAVES] = 1.f; }
                else *reinterpret_cast<float2*>(a.ws_ml + own_state * 2) = make_float2(d, 1.f);
            }
        }
        if (MATS == 3) sm.o[QKV_WAVES][lane] = bf16_to_float(mine_v);
        else if (split == 1) a.ws_o[own_state * QKV_DH + lane] = bf16_to_float(mine_v);
    }
    const uint4 qraw = sm.made[0][c];
    constexpr float NEG = -1.0e30f;
    float m = NEG, l = 0.f, o[8];
#pragma unroll
    for (int e = 0; e < 8; ++e) o[e] = 0.f;
    for (int j0 = kb + 8 * wave, first = kb;;) {
        float dot[UNR], mx = NEG;
#pragma unroll
        for (int u = 0; u < UNR; ++u) {
            const float d = group_sum<8>(dot16<bf16_t>(qraw, kraw[u])) * a.scale_log2e;
            dot[u] = j0 + 64 * u + g < ke ? d : NEG;
            mx = fmaxf(mx, dot[u]);
        }
        const float mn = fmaxf(m, mx), f = fast_exp2(m - mn);
        l *= f;
#pragma unroll
        for (int e = 0; e < 8; ++e) o[e] *= f;
#pragma unroll
        for (int u = 0; u < UNR; ++u) {
            const float pj = dot[u] > NEG ? fast_exp2(dot[u] - mn) : 0.f;
            float vf[8];
            Vec16<bf16_t>::widen(vraw[u], vf);
            l += pj;
#pragma unroll
            for (int e = 0; e < 8; ++e) o[e] = fmaf(pj, vf[e], o[e]);
        }
        m = mn;
        first += 64 * UNR;
        if (first >= ke) break;
        j0 += 64 * UNR;
        load_keys(j0);
    }
    if (ke <= kb) {              // no keys: whatever was loaded is dropped
        m = NEG; l = 0.f;
#pragma unroll
        for (int e = 0; e < 8; ++e) o[e] = 0.f;
    }
    wave_state<bf16_t, 8, 8>(m, l, o, &sm.m[wave], &sm.l[wave], sm.o[wave]);
    lds_barrier();
    if (wave != 0) return;
    constexpr int N = MATS == 3 ? QKV_WAVES + 1 : QKV_WAVES;
    float mx = sm.m[0];
#pragma unroll
    for (int i = 1; i < N; ++i) mx = fmaxf(mx, sm.m[i]);
    l = 0.f;
    float v = 0.f;
#pragma unroll
    for (int i = 0; i < N; ++i) {
        const float f = fast_exp2(sm.m[i] - mx);
        l = fmaf(f, sm.l[i], l);
        v = fmaf(f, sm.o[i][lane], v);
    }
    if (MATS == 3) {
        a.out[static_cast<size_t>(t) * a.out_stride + h * QKV_DH + lane] = float_to_bf16(v / l);
    } else {
        const size_t state = pair * states + split;
        a.ws_o[state * QKV_DH + lane] = v;
        if (lane == 0) *reinterpret_cast<float2*>(a.ws_ml + state * 2) = make_float2(mx, l);
    }
}

template <int CB, bool TWO, int UNR, bool ALL>
__global__ void __launch_bounds__(64 * QKV_WAVES)
qkv_attention_kernel(QkvAttention a) {
    __shared__ QkvShared sm;
    // workgroups of one head on one XCD, as far as the counts allow: they share the head's weights
    const unsigned per_xcd = gridDim.x / 8, i = (blockIdx.x % 8) * per_xcd + blockIdx.x / 8;
    if (i >= static_cast<unsigned>(a.T * a.H * a.S)) return;
    const int pair = a.S == 1 ? i : __umulhi(i, a.per_s), split = i - pair * a.S;
    const int h = a.T == 1 ? pair : __umulhi(static_cast<unsigned>(pair), a.per_t), t = pair - h * a.T;
    if constexpr (ALL) qkv_attention_body<CB, TWO, UNR, 3>(a, t, h, 0, sm);
    else if (split < 2) qkv_attention_body<CB, TWO, UNR, 2>(a, t, h, split, sm);
    else qkv_attention_body<CB, TWO, UNR, 1>(a, t, h, split, sm);
}

template <int CB, bool TWO, bool ALL>
static void launch_qkv_attention(const QkvAttention& a, int groups, int keys, hipStream_t stream) {
    if (keys <= 128) qkv_attention_kernel<CB, TWO, 2, ALL><<<groups, 64 * QKV_WAVES, 0, stream>>>(a);
    else if (keys <= 256) qkv_attention_kernel<CB, TWO, 4, ALL><<<groups, 64 * QKV_WAVES, 0, stream>>>(a);
    else if (keys <= 384) qkv_attention_kernel<CB, TWO, 6, ALL><<<groups, 64 * QKV_WAVES, 0, stream>>>(a);
    else qkv_attention_kernel<CB, TWO, 8, ALL><<<groups, 64 * QKV_WAVES, 0, stream>>>(a);
}

extern "C" {

// out[t, h * head_dim + e] from the states of `partial_out` (head_dim % 4 == 0).
int mllm_merge_attention_splits(const float* ws, int n_q, int n_heads, int head_dim, int nsplit, void* out,
                                int out_stride, int dtype, hipStream_t stream) {
    if (n_q <= 0) return 0;
    if (head_dim % 4 != 0 || head_dim < 4 || n_heads < 1 || nsplit < 1) return -1;
    const dim3 grid(n_q * n_heads, (head_dim / 4 + MERGE_THREADS - 1) / MERGE_THREADS);
    const float* ws_o = ws;
    const float* ws_ml = ws + static_cast<size_t>(n_q) * n_heads * nsplit * head_dim;
    if (dtype == MLLM_F32)
        merge_splits_kernel<float><<<grid, MERGE_THREADS, 0, stream>>>(ws_o, ws_ml, nsplit, head_dim, n_heads, static_cast<float*>(out), out_stride);
    else
        merge_splits_kernel<bf16_t><<<grid, MERGE_THREADS, 0, stream>>>(ws_o, ws_ml, nsplit, head_dim, n_heads, static_cast<bf16_t*>(out), out_stride);
    MLLM_LAUNCH_CHECK();
    return 0;
}

// Number of floats of workspace (partial outputs and their max/sum) for n_q tokens.
long mllm_decode_attention_ws_floats(int n_q, int n_heads, int head_dim, int nsplit) {
    return static_cast<long>(n_q) * n_heads * nsplit * (head_dim + 2);
}

// Returns 0, a HIP error code, or -1 for sizes the kernel refuses: head_dim * element size / 16
// must be a power of two in [2, 64], page_size a power of two, and max_blocks at most 4096. `counters` holds n_q*n_heads ints that are zero before the
// first launch (the kernel leaves them zero). With `slots` (n_q rows of the page pools, < 0: none) the
// tokens' own keys/values are taken from columns k_col/v_col of q and written to the pages by this
// kernel; without, they must be in the pages already.
// partial_out != 0: nothing is written to `out`; the workspace holds, for pair = token * n_heads + head
// and split s, the unnormalised output at ws[(pair * nsplit + s) * head_dim ..] and (maximum in base 2,
// sum) at ws[n_q * n_heads * nsplit * head_dim + (pair * nsplit + s) * 2 ..]; a split without keys has
// sum 0 and a large negative maximum.
int mllm_decode_attention(const void* q, int q_stride, int q_col, const void* k_pages, const void* v_pages,
                          int kv_dim, const int* block_tables, int max_blocks, const int* token_seq,
                          const int* positions, int n_q, int n_heads, int n_kv_heads, int head_dim,
                          int page_size, float scale, int window, int nsplit, int waves, void* out,
                          int out_stride, float* ws, int* counters, int k_col, int v_col, const int* slots,
                          int partial_out, int dtype, hipStream_t stream, const MllmScoreShape* shape, const float* gate, int ldg) {
    if (n_q <= 0) return 0;
    const int esz = dtype == MLLM_F32 ? 4 : 2;
    const int lpk = head_dim * esz / 16;
    if (head_dim * esz % 16 != 0 || n_heads % n_kv_heads != 0 || nsplit < 1 || nsplit > 65535 ||
        waves < 1 || waves > DEC_MAX_WAVES) return -1;
    if (page_size < 1 || (page_size & (page_size - 1)) != 0 || max_blocks > DEC_TABLE_LDS) return -1;
    dim3 grid(n_q * n_heads, nsplit);
    float* ws_o = ws;
    float* ws_ml = ws + static_cast<size_t>(n_q) * n_heads * nsplit * head_dim;
    // (shaped scores: the queries times the scale alone; the kernel goes to base 2 after the shaping)
    const float sl2 = shape ? scale : scale * 1.44269504088896340736f;
    if (shape && window > 0 && shape->chunk > 0) return -1;
    // (a gate goes with shaped scores, and with a result that this kernel finishes itself)
    if (gate != nullptr && (shape == nullptr || partial_out)) return -1;
    // (weights that are not normalised leave no sum for another kernel to divide by)
    if (shape && shape->sigmoid && partial_out) return -1;
    int rc;
    if (dtype == MLLM_F32)
        rc = launch_decode<float>(lpk, grid, waves, stream, (const float*)q, q_stride, q_col, (const float*)k_pages,
                                  (const float*)v_pages, kv_dim, block_tables, max_blocks, token_seq, positions,
                                  n_heads, n_kv_heads, page_size, sl2, window, nsplit, (float*)out, out_stride,
                                  ws_o, ws_ml, counters, (float*)k_pages, (float*)v_pages, k_col, v_col, slots, partial_out, shape, gate, ldg);
    else
        rc = launch_decode<bf16_t>(lpk, grid, waves, stream, (const bf16_t*)q, q_stride, q_col, (const bf16_t*)k_pages,
                                   (const bf16_t*)v_pages, kv_dim, block_tables, max_blocks, token_seq, positions,
                                   n_heads, n_kv_heads, page_size, sl2, window, nsplit, (bf16_t*)out, out_stride,
                                   ws_o, ws_ml, counters, (bf16_t*)k_pages, (bf16_t*)v_pages, k_col, v_col, slots, partial_out, shape, gate, ldg);
    if (rc != 0) return rc;
    MLLM_LAUNCH_CHECK();
    return 0;
}

// Layer norm of the fp32 rows x [n_q, K], QKV product and decode attention over the pages in one kernel: n_q sequences that bring one
// token each (row t of block_tables is token t's), heads of 64, as many key/value heads as query heads, w [3 n_heads 64, K] with
// queries, keys and values one behind the other. The new keys and values go to rows slots[t] (>= 0) of the pages. nsplit 1: the result
// goes to out (bfloat16). More: the states are left in ws as mllm_decode_attention's partial_out leaves them, nsplit + 1 of them a
// pair, the last the token's own. keys: the most keys any split has. Returns 0, a HIP error code, or -1 for sizes the kernel
// refuses: K must be a multiple of 64 up to 2,048 (nsplit 1: 768), ldw of 8, ldx of 4, page_size a power of two, max_blocks at most 4,096, all pairs' splits
// at most 16,384 (operands 16-byte aligned).
int mllm_ln_qkv_attention(const float* x, int ldx, const float* gamma, const float* beta, float eps, const void* w, int ldw, const float* bias,
                          int K, void* k_pages, void* v_pages, const int* block_tables, int max_blocks, const int* positions, const int* slots,
                          int n_q, int n_heads, int page_size, float scale, int nsplit, int keys, float* ws, void* out, int out_stride,
                          hipStream_t stream) {
    if (n_q <= 0) return 0;
    if (K < 64 || K % 64 != 0 || K > (nsplit == 1 ? 768 : QKV_MAX_K) || ldw % 8 != 0 || ldx % 4 != 0 || n_heads < 1 || nsplit < 1 || max_blocks < 1 || max_blocks > DEC_TABLE_LDS) return -1;
    if (page_size < 1 || (page_size & (page_size - 1)) != 0 || static_cast<long>(n_q) * n_heads * nsplit > 1 << 14) return -1;
    QkvAttention a;
    a.token_blocks = block_tables; a.max_blocks = max_blocks; a.positions = positions;
    a.T = n_q; a.H = n_heads; a.S = nsplit;
    // (exact below 2^16: the error of i ceil(2^32 / d) / 2^32 is less than i / 2^32, and i / d is 1 / d short of the next whole number)
    a.per_s = static_cast<unsigned>(((1ull << 32) + nsplit - 1) / nsplit);
    a.per_t = static_cast<unsigned>(((1ull << 32) + n_q - 1) / n_q);
    a.x = x; a.ldx = ldx; a.K = K; a.gamma = gamma; a.beta = beta; a.eps = eps;
    a.w = static_cast<const bf16_t*>(w); a.ldw = ldw; a.bias = bias;
    a.k_pages = static_cast<bf16_t*>(k_pages); a.v_pages = static_cast<bf16_t*>(v_pages);
    a.kv_dim = n_heads * QKV_DH; a.page_shift = __builtin_ctz(page_size); a.slots = slots;
    a.scale_log2e = scale * MLLM_LOG2E;
    a.ws_o = ws;
    a.ws_ml = ws + static_cast<size_t>(n_q) * n_heads * (nsplit + 1) * QKV_DH;
    a.out = static_cast<bf16_t*>(out); a.out_stride = out_stride;
    const int groups = (n_q * n_heads * nsplit + 7) / 8 * 8;
    if (nsplit == 1) {
        launch_qkv_attention<6, true, true>(a, groups, keys, stream);
    } else {
        if (K <= 768) launch_qkv_attention<6, true, false>(a, groups, keys, stream);
        else if (K <= 1024) launch_qkv_attention<8, true, false>(a, groups, keys, stream);
        else launch_qkv_attention<5, false, false>(a, groups, keys, stream);
    }
    MLLM_LAUNCH_CHECK();
    return 0;
}

}  // extern "C"
