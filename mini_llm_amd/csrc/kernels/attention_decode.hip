// Decode attention over the paged cache for gfx950: one query token per (token, head),
// its keys split over `nsplit` workgroups so that small batches still fill the chip.
//
// Inside a workgroup, LPK lanes share one key: each lane loads 16 bytes of the key row
// and of the value row (so a wavefront covers 64/LPK whole rows per load instruction),
// the LPK partial dot products are summed with DPP shuffles, and every lane keeps the
// running maximum, sum and its slice of the output for the keys of its lane group
// (recurrence of /root/reference/src/kernels/prefill/flashattention.cu:129-178, in base 2).
// Groups, wavefronts and splits are merged with the same (m, l, o) rule. The splits of a
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

#include <algorithm>
#include <type_traits>

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

// Two elements of a lane and of the lane OFF (16 or 32) away: the lower lane gets the first element of both, the upper one the second, `lo`
// from the lower lane and `hi` from the upper. The same element given twice: both get it.
template <int OFF>
__device__ __forceinline__ void lane_halves(float first, float second, float& lo, float& hi) {
    const unsigned u = __builtin_bit_cast(unsigned, first), v = __builtin_bit_cast(unsigned, second);
    if constexpr (OFF == 16) {
        const auto s = __builtin_amdgcn_permlane16_swap(u, v, false, false);
        lo = __builtin_bit_cast(float, static_cast<unsigned>(s[0])); hi = __builtin_bit_cast(float, static_cast<unsigned>(s[1]));
    } else {
        const auto s = __builtin_amdgcn_permlane32_swap(u, v, false, false);
        lo = __builtin_bit_cast(float, static_cast<unsigned>(s[0])); hi = __builtin_bit_cast(float, static_cast<unsigned>(s[1]));
    }
}

// Keys of a split, rounded up.
__device__ __forceinline__ int keys_per_split(int n_keys, int nsplit) { return nsplit == 1 ? n_keys : n_keys <= 0 ? 0 : 1 + uniform_quotient(n_keys - 1, nsplit); }

// SHAPED: the scores are shaped before the softmax and a chunked mask may stand in for the window (score_shape.h);
// the queries then come times the scale alone, and the shaped score goes to base 2 afterwards.
// MODE 0: plain softmax; 1: shaped scores; 2: shaped scores whose weights are sigmoid(score + bias of the head), every
// visible key on its own. The state keeps its form: the maximum stays 0 throughout, so every merge adds the outputs
// as they are, the sum is unused and nothing is divided at the end.
template <typename T, int LPK, int UNR, int MODE = 0>
__global__ void __launch_bounds__(UNR > 8 ? 512 : DEC_MAX_WAVES * MLLM_WAVE)
decode_attention_kernel(// the first 14 dwords arrive in registers with the wavefront: what the first loads need (an argument behind
                        // them is a load of its own from memory that no cache holds, 0.6 to 0.8 us)
                        const int* __restrict__ block_tables, const int* __restrict__ positions, const T* __restrict__ q,
                        const T* __restrict__ k_pages, const T* __restrict__ v_pages, int q_stride, unsigned heads, unsigned form, int nsplit,
                        // the rest is loaded by the kernel
                        const int* __restrict__ token_seq, int window, int kv_dim, float scale_log2e, T* __restrict__ out, int out_stride,
                        float* __restrict__ ws_o, float* __restrict__ ws_ml, int* __restrict__ counters,
                        int k_col, int v_col, const int* __restrict__ slots, int partial_out, MllmScoreShape shape,
                        const float* __restrict__ gate, int ldg) {
    constexpr bool SHAPED = MODE != 0, SIGMOID = MODE == 2;
    constexpr int EPL = Vec16<T>::N;        // elements per lane
    constexpr int DH = LPK * EPL;           // head size
    constexpr int KPW = MLLM_WAVE / LPK;    // keys per wavefront and load instruction
    __shared__ float2 sm_ml[DEC_MAX_WAVES];                                 // a wavefront's maximum and sum
    __shared__ __attribute__((aligned(16))) float sm_o[DEC_MAX_WAVES][DH];
    __shared__ int sm_last;
    __shared__ int sm_table[DEC_TABLE_LDS];
    // (the words as launch_decode packs them)
    const int n_heads = heads & 0xffff, n_kv_heads = heads >> 16;
    const int max_blocks = form & 0x1fff, shift = form >> 13 & 31, n_waves = form >> 18 & 31;
    const bool windowed = form >> 23 & 1, append = !SHAPED && (form >> 24 & 1), one_each = form >> 25 & 1;      // (shaped scores: the pages hold every key)

    // workgroups: (head, split, token)
    const int h = blockIdx.x, split = blockIdx.y, t = blockIdx.z;
    const int pair = t * n_heads + h;
    // (head / heads a key/value head in floating point: whole numbers below 2^16, a half away from the next quotient)
    const int hk = n_heads == n_kv_heads ? h : __builtin_amdgcn_readfirstlane(static_cast<int>((static_cast<float>(h) + 0.5f) * static_cast<float>(n_kv_heads) * __builtin_amdgcn_rcpf(static_cast<float>(n_heads))));
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / MLLM_WAVE), lane = threadIdx.x % MLLM_WAVE;
    const int c = lane % LPK, g = lane / LPK;
    // (every sequence brings one token, token t belongs to sequence t: the block table can be requested at once, beside the
    // position, instead of after a load of its own)
    int b = t;
    if (!one_each) {
        b = token_seq[t];
        asm volatile("" : "+s"(b));           // waited for in here, not where both ways meet
    }
    const int* gtable_row = block_tables + static_cast<size_t>(b) * max_blocks;
    // Without a window the keys start at block 0 whatever the position is, and rows of the table are
    // filled to their end (zeros behind a sequence's last block): the whole row goes to LDS without
    // waiting for the position. (A table without entries, where every token stands alone with its own key, is not read.)
    const bool whole_row = !windowed && static_cast<unsigned>(max_blocks - 1) < DEC_TABLE_LDS;
    const auto raw_q = load_raw16(q + static_cast<size_t>(t) * q_stride + h * DH + c * EPL);
    int entry = 0;
    if (whole_row) entry = gtable_row[min(static_cast<int>(threadIdx.x), max_blocks - 1)];
    const int p = positions[t];
    int lo = 0;
    if (windowed) lo = max(p - window + 1, 0);
    if (SHAPED && shape.chunk > 0) lo = p - p % shape.chunk;
    const float r1 = SHAPED ? mllm_bias_r1(shape, h) : 0.f, r2 = (SHAPED && shape.r1) ? shape.r2[h] : 0.f;
    const float sbias = (SIGMOID && shape.score_bias) ? shape.score_bias[h] : 0.f;
    // The visible keys are counted through: first the kept first positions that lie in front of the window (none
    // without them), then the window's. Key number v stands at position key_at(v); kb, ke and the loops below count
    // in these numbers, so the splits share kept and window keys alike.
    const int kf = (SHAPED && windowed && shape.keep_first > 0) ? min(shape.keep_first, lo) : 0;
    const int shift_pos = lo - kf;
    auto key_at = [&](int v) { return SHAPED && v < kf ? v : v + shift_pos; };
    const int n_keys = p - lo + 1 + kf;
    const int per = keys_per_split(n_keys, nsplit);
    const int kb = split * per;
    const int ke = min(n_keys, kb + per);
    // With `slots`, the token's own key and value are not in the pages yet: they are read from
    // its row of q (columns k_col, v_col), and written to the pages by the first query head of
    // each key/value head. That key is taken by one lane group after the loop over the pages.
    const bool own_here = append && ke == n_keys && kb <= n_keys - 1;     // this workgroup's range holds the token itself
    const int ke_pages = own_here ? n_keys - 1 : ke;                      // keys [kb, ke_pages) come from the pages
    const size_t col = static_cast<size_t>(hk) * DH + c * EPL;

    // The block table entries of this workgroup's keys go to LDS first, so that no key load waits
    // for a table load.
    // (with kept first positions the keys of a range need not be neighbours: the table from block 0 on)
    if (whole_row) {
        sm_table[threadIdx.x] = entry;        // (a table as large as a workgroup at least)
        for (int i = threadIdx.x + n_waves * MLLM_WAVE; i < max_blocks; i += n_waves * MLLM_WAVE) sm_table[i] = gtable_row[i];
    }
    const int first_blk = (whole_row || kf > 0) ? 0 : key_at(kb) >> shift;
    const int n_blk = ke_pages > kb ? (key_at(ke_pages - 1) >> shift) - first_blk + 1 : 0;
    if (!whole_row) {
        const int* gtable = gtable_row + first_blk;
        for (int i = threadIdx.x; i < n_blk; i += n_waves * MLLM_WAVE) sm_table[i] = gtable[i];
    }

    float qf[EPL];
    Vec16<T>::widen(raw_q, qf);
#pragma unroll
    for (int e = 0; e < EPL; ++e) qf[e] *= scale_log2e;
    // (The token's own row and the place of its key: behind what the first keys wait for, and left in flight over the barrier. The place
    // by a vector load: a scalar one in flight would be waited for at every LDS read.)
    uint4 k_own = make_uint4(0, 0, 0, 0), v_own = make_uint4(0, 0, 0, 0);
    int own_slot = -1;
    const bool own_lanes = own_here && wave == 0 && g == 0;
    if (own_here && wave == 0) {
        const T* src = q + static_cast<size_t>(t) * q_stride + col;
        k_own = load_raw16(src + k_col);
        v_own = load_raw16(src + v_col);
        int none = 0;
        asm volatile("" : "+v"(none));
        own_slot = slots[t + none];
    }
    lds_barrier();       // the table is in LDS

    // Running state (maximum in base 2, sum, output slice). The maximum starts at a large
    // negative finite number, so that no difference of two of them is NaN.
    constexpr float NEG = -1.0e30f;
    constexpr float M0 = SIGMOID ? 0.f : NEG;       // an empty state's maximum
    float m = M0, l = 0.f, o[EPL];
#pragma unroll
    for (int e = 0; e < EPL; ++e) o[e] = 0.f;
    // A sink is one more term of the denominator, exp(sink), without a value: one lane group of the first split
    // starts from it instead of from nothing.
    // (one at or below an empty state's maximum adds nothing)
    if (SHAPED && !SIGMOID && shape.sink != nullptr && split == 0 && wave == 0 && g == 0) {
        const float sink = shape.sink[h] * MLLM_LOG2E;
        if (!(sink <= NEG)) { m = sink; l = 1.f; }
    }

    // A wavefront takes UNR groups of 64/LPK keys at a time. All their loads are issued
    // first, unconditionally (a key beyond the range loads the last key of the range again and is
    // masked when used): a load under a condition, even one that is uniform over the wavefront,
    // makes every later use wait for all loads in flight (measured: 7.6 -> 8.4 us at 512 keys).
    const int mask = (1 << shift) - 1;
    const int group_keys = n_waves * KPW;                 // distance between a wavefront's groups
    const T *k_col_pages = k_pages + col, *v_col_pages = v_pages + col;
    for (int j0 = kb + wave * KPW; j0 < ke_pages; j0 += group_keys * UNR) {
        uint4 kraw[UNR], vraw[UNR];
        int j[UNR], block[UNR];
#pragma unroll
        for (int u = 0; u < UNR; ++u) {
            j[u] = key_at(min(j0 + u * group_keys + g, ke_pages - 1));
            block[u] = sm_table[(j[u] >> shift) - first_blk];
        }
        // (The table's entries together, then the loads together: left alone the compiler widens the first keys, and waits for them, between
        // the others' requests. Shaped scores, and heads that fill a wavefront with one key, have the work for that wait: 16 heads of 128 in 32
        // bits, one token of 4,096 keys 26.8 us so and 24.8 without, 8 heads of 256 2 % without.)
        constexpr bool ALL_AT_ONCE = !SHAPED && KPW > 1;
        if (ALL_AT_ONCE) __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int u = 0; u < UNR; ++u) {
            const uint64_t at = static_cast<uint64_t>((static_cast<uint32_t>(block[u]) << shift) + (j[u] & mask)) * static_cast<uint32_t>(kv_dim);
            kraw[u] = load_stream16(k_col_pages + at);
            vraw[u] = load_stream16(v_col_pages + at);
        }
        if (ALL_AT_ONCE) __builtin_amdgcn_sched_barrier(0);
        float dot[UNR];
        float mx = NEG;
#pragma unroll
        for (int u = 0; u < UNR; ++u) {
            float kf[EPL];
            Vec16<T>::widen(kraw[u], kf);
            float d = 0.f;
#pragma unroll
            for (int e = 0; e < EPL; ++e) d = fmaf(qf[e], kf[e], d);
            d = group_sum<LPK>(d);
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
        if (own_slot >= 0 && (n_heads == n_kv_heads || h % (n_heads / n_kv_heads) == 0)) {
            const size_t wrow = static_cast<size_t>(own_slot) * kv_dim + col;
            *reinterpret_cast<uint4*>(const_cast<T*>(k_pages) + wrow) = k_own;
            *reinterpret_cast<uint4*>(const_cast<T*>(v_pages) + wrow) = v_own;
        }
        float kf[EPL], vf[EPL];
        Vec16<T>::widen(k_own, kf);
        Vec16<T>::widen(v_own, vf);
        float d = 0.f;
#pragma unroll
        for (int e = 0; e < EPL; ++e) d = fmaf(qf[e], kf[e], d);
        d = group_sum<LPK>(d);
        if (SHAPED) d = mllm_shaped_score<sizeof(T) == 2>(d, shape, r1, r2, 0) * MLLM_LOG2E;
        const float mn = SIGMOID ? 0.f : fmaxf(m, d);
        const float a = SIGMOID ? 1.f : exp2_for<T>(m - mn);
        const float pj = SIGMOID ? 1.f / (1.f + exp2_for<T>(-(d + sbias * MLLM_LOG2E))) : exp2_for<T>(d - mn);
        l = l * a + pj;
#pragma unroll
        for (int e = 0; e < EPL; ++e) o[e] = fmaf(pj, vf[e], o[e] * a);       // (as the keys of the pages are added)
        m = mn;
    }
    // Merges the states of all lane groups and wavefronts, in a fixed order: lane groups whose numbers differ in one bit, from the
    // lowest bit on, then wavefronts (group G of KPW takes G, G + KPW, ..., then the groups as before). Where two groups meet
    // the lower one's output is the product that the fused multiply-add adds to in every lane, so that no result depends on who computes it.
    // Across the rows of 16 lanes each side keeps half of the elements: one swap then brings two elements' pairs together.
    // The wavefronts' states meet in wavefront 0, where lane i holds elements EW i .. EW i + EW - 1 of the output afterwards
    // (lanes beyond the head size those of lane i % DH). Bound by the instructions of one wavefront: with all of a lane's elements in every
    // lane and the wavefronts' states merged as the lane groups' it was 0.76 us of a launch's 5.0 (1 token, 12 heads, 768 keys), with the wavefronts merged an element a lane 0.56.
    constexpr int EW = DH > MLLM_WAVE ? DH / MLLM_WAVE : 1;
    float r[EW];
    auto block_merge = [&](bool again) {
        int first = 0;                  // of this lane's slice: the elements it still holds
        auto halve = [&](auto off_tag, auto n_tag) {
            constexpr int OFF = decltype(off_tag)::value, N = decltype(n_tag)::value, HALF = N > 1 ? N / 2 : 1;
            float m_lo, m_hi, l_lo, l_hi;
            if (OFF == 16) { lane_pair_16(m, m_lo, m_hi); lane_pair_16(l, l_lo, l_hi); }
            else { lane_pair_32(m, m_lo, m_hi); lane_pair_32(l, l_lo, l_hi); }
            const float mn = fmaxf(m_lo, m_hi), a = exp2_for<T>(m_lo - mn), b2 = exp2_for<T>(m_hi - mn);
            l = fmaf(l_lo, a, l_hi * b2);
            m = mn;
#pragma unroll
            for (int e = 0; e < HALF; ++e) {
                float lo, hi;
                lane_halves<OFF>(o[e], o[N > 1 ? e + HALF : e], lo, hi);
                o[e] = fmaf(hi, b2, lo * a);
            }
            if (N > 1) first += (lane & OFF) ? HALF : 0;
        };
        constexpr int N16 = EPL, N32 = LPK <= 16 && EPL > 1 ? EPL / 2 : EPL, N_LEFT = N32 > 1 && LPK <= 32 ? N32 / 2 : N32;
#pragma unroll
        for (int off = LPK; off < 16; off <<= 1) {
            const float m2 = lane_xor(m, off), l2 = lane_xor(l, off);
            float o2[EPL];
#pragma unroll
            for (int e = 0; e < EPL; ++e) o2[e] = lane_xor(o[e], off);
            merge_state<T, EPL>(m, l, o, m2, l2, o2);
        }
        if constexpr (LPK <= 16) halve(std::integral_constant<int, 16>{}, std::integral_constant<int, N16>{});
        if constexpr (LPK <= 32) halve(std::integral_constant<int, 32>{}, std::integral_constant<int, N32>{});
        if (again) lds_barrier();             // earlier readers of the LDS arrays are done
        if (lane == 0) sm_ml[wave] = make_float2(m, l);
        if ((lane & 15) / LPK == 0 || LPK >= 16) {        // (of lane groups inside a row of 16, the first)
            float* dst = &sm_o[wave][c * EPL + first];
#pragma unroll
            for (int e = 0; e < N_LEFT; ++e) dst[e] = o[e];
        }
        lds_barrier();      // (the store of the own key stays in flight)
        if (wave != 0) return;
        const float2 ml = sm_ml[min(lane, n_waves - 1)];
        const int at = (lane * EW) % DH;
        float wm[DEC_MAX_WAVES] = {}, wl[DEC_MAX_WAVES] = {}, wo[DEC_MAX_WAVES][EW] = {};
        auto join = [&](int x, int y) {        // state y into state x
            const float mn = fmaxf(wm[x], wm[y]), a = exp2_for<T>(wm[x] - mn), b2 = exp2_for<T>(wm[y] - mn);
            wl[x] = fmaf(wl[x], a, wl[y] * b2);
#pragma unroll
            for (int e = 0; e < EW; ++e) wo[x][e] = fmaf(wo[y][e], b2, wo[x][e] * a);
            wm[x] = mn;
        };
        // (four elements of 16 wavefronts and more: each four are joined before the next are read, which then needs a quarter of the
        // registers; 8 heads of 256 and 40 keys 6.3 > 6.1 us in 32 bits. The order is the same.)
        constexpr bool JOIN_AT_ONCE = EW >= 4;
#pragma unroll
        for (int w0 = 0; w0 < DEC_MAX_WAVES; w0 += 4) {
            if (w0 >= n_waves) continue;
#pragma unroll
            for (int w = w0; w < w0 + 4; ++w) {
#pragma unroll
                for (int e = 0; e < EW; ++e) wo[w][e] = sm_o[min(w, n_waves - 1)][at + e];
                wm[w] = row_lane(ml.x, w);
                wl[w] = row_lane(ml.y, w);
            }
            if (JOIN_AT_ONCE)
#pragma unroll
                for (int y = w0; y < w0 + 4; ++y)
                    if (y >= KPW && y < n_waves) join(y % KPW, y);
        }
        if (!JOIN_AT_ONCE)
#pragma unroll
            for (int y = KPW; y < DEC_MAX_WAVES; ++y)
                if (y < n_waves) join(y % KPW, y);
#pragma unroll
        for (int d = 1; d < KPW && d < DEC_MAX_WAVES; d <<= 1)
#pragma unroll
            for (int x = 0; x + d < KPW && x + d < DEC_MAX_WAVES; x += 2 * d)
                if (x + d < n_waves) join(x, x + d);
        m = wm[0];
        l = wl[0];
#pragma unroll
        for (int e = 0; e < EW; ++e) r[e] = wo[0][e];
    };
    const bool holds = wave == 0 && lane * EW < DH;      // lanes with elements of the result
    block_merge(false);
    T* op = out + static_cast<size_t>(t) * out_stride + h * DH + lane * EW;
    auto store_result = [&]() {
        if (!holds) return;
        const float inv = SIGMOID ? 1.f : 1.0f / l;
#pragma unroll
        for (int e = 0; e < EW; ++e) {
            float v = r[e] * inv;
            if (SHAPED && gate != nullptr) v *= 1.f / (1.f + __expf(-gate[static_cast<size_t>(t) * ldg + (shape.gate_per_head ? h : h * DH + lane * EW + e)]));
            op[e] = from_float<T>(v);
        }
    };
    if (nsplit == 1 && !partial_out) {
        store_result();
        return;
    }
    // the split's state as it is; with partial_out whoever reads the workspace merges
    const size_t slot = static_cast<size_t>(pair) * nsplit + split;
    if (holds) {
#pragma unroll
        for (int e = 0; e < EW; ++e) ws_o[slot * DH + lane * EW + e] = r[e];
        if (lane == 0) *reinterpret_cast<float2*>(ws_ml + slot * 2) = make_float2(m, l);
    }
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
    block_merge(true);
    store_result();
    if (threadIdx.x == 0) counters[pair] = 0;     // ready for the next launch
}

template <typename T>
static int launch_decode(int lpk, dim3 grid, int waves, hipStream_t stream, const T* q, int q_stride, int q_col,
                         const T* k_pages, const T* v_pages, int kv_dim, const int* block_tables,
                         int max_blocks, const int* token_seq, const int* positions, int n_heads,
                         int n_kv_heads, int page_size, float scale_log2e, int window, int nsplit, T* out,
                         int out_stride, float* ws_o, float* ws_ml, int* counters, int k_col, int v_col, const int* slots, int partial_out, const MllmScoreShape* shape,
                         const float* gate, int ldg) {
    const MllmScoreShape sh = shape ? *shape : MllmScoreShape{0.f, 0, nullptr, nullptr};
    const unsigned heads = n_heads | static_cast<unsigned>(n_kv_heads) << 16;
    const unsigned form = max_blocks | (__builtin_ffs(page_size) - 1) << 13 | waves << 18 | (window > 0 ? 1u << 23 : 0u) | (slots != nullptr ? 1u << 24 : 0u) |
                          (token_seq == nullptr ? 1u << 25 : 0u);
    // (the queries' first column belongs to their address, the other columns count from there)
#define DEC_ARGS block_tables, positions, q + q_col, k_pages, v_pages, q_stride, heads, form, nsplit, token_seq, window, kv_dim, scale_log2e, \
            out, out_stride, ws_o, ws_ml, counters, k_col - q_col, v_col - q_col, slots, partial_out, sh, gate, ldg
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
// kernel; without, they must be in the pages already, as they must for shaped scores (-1 otherwise).
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
    if (page_size < 1 || (page_size & (page_size - 1)) != 0 || max_blocks > DEC_TABLE_LDS || n_heads > 0xffff) return -1;
    float* ws_o = ws;
    float* ws_ml = ws + static_cast<size_t>(n_q) * n_heads * nsplit * head_dim;
    // (shaped scores: the queries times the scale alone; the kernel goes to base 2 after the shaping)
    const float sl2 = shape ? scale : scale * 1.44269504088896340736f;
    if (shape && window > 0 && shape->chunk > 0) return -1;
    // (a gate goes with shaped scores, and with a result that this kernel finishes itself)
    if (gate != nullptr && (shape == nullptr || partial_out)) return -1;
    // (weights that are not normalised leave no sum for another kernel to divide by)
    if (shape && shape->sigmoid && partial_out) return -1;
    // (the kernels of shaped scores read every key from the pages)
    if (shape && slots != nullptr) return -1;
    // (tokens are the grid's third dimension, which takes 65,535)
    for (int t0 = 0; t0 < n_q; t0 += 65535) {
        const dim3 grid(n_heads, nsplit, std::min(n_q - t0, 65535));
        const size_t first = t0, state = first * n_heads * nsplit;
        auto launch = [&](auto element) {
            using T = decltype(element);
            return launch_decode<T>(lpk, grid, waves, stream, static_cast<const T*>(q) + first * q_stride, q_stride, q_col, static_cast<const T*>(k_pages),
                                    static_cast<const T*>(v_pages), kv_dim, token_seq ? block_tables : block_tables + first * max_blocks, max_blocks,
                                    token_seq ? token_seq + first : nullptr, positions + first, n_heads, n_kv_heads, page_size, sl2, window, nsplit,
                                    static_cast<T*>(out) + first * out_stride, out_stride, ws_o + state * head_dim, ws_ml + state * 2,
                                    counters + first * n_heads, k_col, v_col, slots ? slots + first : nullptr, partial_out, shape,
                                    gate ? gate + first * ldg : nullptr, ldg);
        };
        const int rc = dtype == MLLM_F32 ? launch(float{}) : launch(bf16_t{});
        if (rc != 0) return rc;
    }
    MLLM_LAUNCH_CHECK();
    return 0;
}

}  // extern "C"
