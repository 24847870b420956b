// Causal attention over the paged cache, any dtype and head size: one wavefront
// per (query token, head). It serves prompt portions and decoded tokens alike: a
// query at position p of sequence b reads keys [lo, p] of b's pages, where
// lo = max(0, p - window + 1) for a windowed cache and 0 otherwise. The keys and
// values of the step's own tokens must already be in the pages.
//
// Scores, softmax and the value mix are fp32 with the running-maximum recurrence of
// /root/reference/src/kernels/prefill/flashattention.cu:129-178
// (m' = max(m, s); alpha = e^(m-m'); p = e^(s-m'); o = o*alpha + p*v; l = l*alpha + p; out = o/l),
// applied to 64 keys at a time. The reference's decode kernel adds 1e-6 to the
// denominator (/root/reference/src/kernels/decode/paged_attention.cu:97); this does not.
#include "common.h"
#include "lds_loads.h"
#include "query_tiles.h"

#define ATT_WAVES 4
#define ATT_MAX_ACC 4   // head_dim <= 64 * ATT_MAX_ACC

template <typename T>
__global__ void __launch_bounds__(ATT_WAVES * MLLM_WAVE)
paged_attention_generic(const T* __restrict__ q, int q_stride, int q_col,
                        const T* __restrict__ k_pages, const T* __restrict__ v_pages, int kv_dim,
                        const int* __restrict__ block_tables, int max_blocks,
                        const int* __restrict__ token_seq, const int* __restrict__ positions,
                        int n_tokens, int n_heads, int n_kv_heads, int head_dim, int page_size,
                        float scale, int window, T* __restrict__ out, int out_stride) {
    extern __shared__ float smem[];
    const int wave = threadIdx.x / MLLM_WAVE, lane = threadIdx.x % MLLM_WAVE;
    const int pair = blockIdx.x * ATT_WAVES + wave;
    if (pair >= n_tokens * n_heads) return;       // whole wave leaves; no block-wide sync below
    const int t = pair / n_heads, h = pair % n_heads;
    const int hk = h / (n_heads / n_kv_heads);
    const int b = token_seq[t];
    const int p = positions[t];
    const int lo = (window > 0 && p - window + 1 > 0) ? p - window + 1 : 0;
    const int* table = block_tables + static_cast<size_t>(b) * max_blocks;

    float* q_s = smem + wave * (head_dim + 2 * MLLM_WAVE);
    float* p_s = q_s + head_dim;
    int* row_s = reinterpret_cast<int*>(p_s + MLLM_WAVE);

    const T* qp = q + static_cast<size_t>(t) * q_stride + q_col + h * head_dim;
    for (int d = lane; d < head_dim; d += MLLM_WAVE) q_s[d] = to_float(qp[d]) * scale;
    wave_lds_sync();

    float m = -INFINITY, l = 0.f;
    float acc[ATT_MAX_ACC] = {0.f, 0.f, 0.f, 0.f};
    const int kv_off = hk * head_dim;

    for (int j0 = lo; j0 <= p; j0 += MLLM_WAVE) {
        // phase A: one key per lane
        const int j = j0 + lane;
        const bool valid = j <= p;
        float s = -INFINITY;
        int row = 0;
        if (valid) {
            row = table[j / page_size] * page_size + j % page_size;
            const T* kp = k_pages + static_cast<size_t>(row) * kv_dim + kv_off;
            float dot = 0.f;
            for (int d = 0; d < head_dim; d += 8) {
                float kv[8];
                load8(kp + d, kv);
#pragma unroll
                for (int i = 0; i < 8; ++i) dot = fmaf(q_s[d + i], kv[i], dot);
            }
            s = dot;
        }
        const float m_new = fmaxf(m, wave_max(s));
        const float alpha = (m == -INFINITY) ? 0.f : expf(m - m_new);
        const float pj = valid ? expf(s - m_new) : 0.f;
        l = l * alpha + wave_sum(pj);
        m = m_new;
        wave_lds_sync();          // the previous round's readers are done
        p_s[lane] = pj;
        row_s[lane] = row;
        wave_lds_sync();
        // phase B: one (or a few) output dimensions per lane; p_s/row_s are read wave-wide
        const int n_keys = min(MLLM_WAVE, p - j0 + 1);
#pragma unroll
        for (int a = 0; a < ATT_MAX_ACC; ++a) {
            const int d = lane + a * MLLM_WAVE;
            if (d < head_dim) {
                float o = acc[a] * alpha;
                for (int jj = 0; jj < n_keys; ++jj) {
                    const T* vp = v_pages + static_cast<size_t>(row_s[jj]) * kv_dim + kv_off;
                    o = fmaf(p_s[jj], to_float(vp[d]), o);
                }
                acc[a] = o;
            }
        }
    }
    T* op = out + static_cast<size_t>(t) * out_stride + h * head_dim;
    const float inv_l = 1.0f / l;
#pragma unroll
    for (int a = 0; a < ATT_MAX_ACC; ++a) {
        const int d = lane + a * MLLM_WAVE;
        if (d < head_dim) op[d] = from_float<T>(acc[a] * inv_l);
    }
}

// ---------------------------------------------------------------------------------------------
// Prompt portions at any head size (multiples of 16 up to 256), any page size, float32 or bfloat16
// storage: 64 queries of one sequence and one head per workgroup share tiles of 64 keys and values
// that are gathered through the block table into LDS as float32, and the two products run on the
// matrix cores in TRUE 32-bit (v_mfma_f32_16x16x4_f32: float32 operands, no reduced-precision mode).
// This is the 32-bit path's prefill attention, and the bfloat16 path's where the bfloat16 matrix-core
// kernel refuses the sizes. (The one-wavefront-per-query kernel above re-reads every key from memory
// for every query: 5.6 TFLOP/s at 8 x 512 tokens.)
//
// As in the bfloat16 kernel everything is computed transposed, so that a lane owns ONE query:
//   S^T = K Q^T    A = 16 keys x 4 dims from LDS, B = the lane's query fragment (registers)
//   O^T = V^T P^T  A = 16 dims x 4 keys from the transposed values in LDS, B = P^T straight from the S^T
//                  accumulators (the k index of a product may be permuted as long as both operands agree)
// Lane l of a wavefront has query l % 16; its k index l / 16 stands, in product j of a group of four, for
// dim 16c + 4 (l / 16) + j (keys: for key 4 (l / 16) + j), so that one 16-byte LDS read feeds four products.
// Recurrence: /root/reference/src/kernels/prefill/flashattention.cu:129-178, in base 2.
typedef float f32x4_t __attribute__((ext_vector_type(4)));
#define TL_BQ 64
#define TL_BK 64
#define TL_VSTRIDE (TL_BK + 4)      // floats per transposed value row: 17 x 16 bytes, odd, so 16-byte reads of 16 rows do not collide

template <typename T> __device__ __forceinline__ f32x4_t load4f(const T* p);
template <> __device__ __forceinline__ f32x4_t load4f<float>(const float* p) {
    const float4 v = *reinterpret_cast<const float4*>(p);
    return f32x4_t{v.x, v.y, v.z, v.w};
}
template <> __device__ __forceinline__ f32x4_t load4f<bf16_t>(const bf16_t* p) {
    const uint2 v = *reinterpret_cast<const uint2*>(p);
    return f32x4_t{__uint_as_float(v.x << 16), __uint_as_float(v.x & 0xffff0000u), __uint_as_float(v.y << 16),
                   __uint_as_float(v.y & 0xffff0000u)};
}
template <typename T> __device__ __forceinline__ void store4f(T* p, f32x4_t v);
template <> __device__ __forceinline__ void store4f<float>(float* p, f32x4_t v) {
    *reinterpret_cast<float4*>(p) = make_float4(v[0], v[1], v[2], v[3]);
}
template <> __device__ __forceinline__ void store4f<bf16_t>(bf16_t* p, f32x4_t v) {
    *reinterpret_cast<uint2*>(p) = make_uint2(pack_bf16x2(v[0], v[1]), pack_bf16x2(v[2], v[3]));
}

// The end of a tiled kernel: the sink, the division by the sum, the gate and the store. The lane holds O^T[dims 16c + 4G + i] of the query
// in row `row`, c < n_c.
template <typename T, int DC, bool SHAPED>
__device__ __forceinline__ void finish_tiled(f32x4_t (&o)[DC], int n_c, float m, float l, const MllmScoreShape& shape, const float* gate, int ldg,
                                             int h, int head_dim, int row, int G, T* out, int out_stride) {
    if (SHAPED && shape.sink != nullptr) {
        // the sink: one more term of the denominator, exp(sink), without a value (the maximum is in base 2)
        const float sk = shape.sink[h] * MLLM_LOG2E, m_new = fmaxf(m, sk);
        const float a = (m == -INFINITY) ? 0.f : exp2_for<T>(m - m_new);
        l = l * a + exp2_for<T>(sk - m_new);
#pragma unroll
        for (int c = 0; c < DC; ++c) o[c] *= a;
    }
    const float inv_l = 1.f / l;
    const bool head_gate = SHAPED && gate != nullptr && shape.gate_per_head;
    const float hg = head_gate ? 1.f / (1.f + expf(-gate[static_cast<size_t>(row) * ldg + h])) : 1.f;
    T* op = out + static_cast<size_t>(row) * out_stride + h * head_dim + 4 * G;
#pragma unroll
    for (int c = 0; c < DC; ++c) {
        if (c < n_c) {
            f32x4_t r = o[c] * inv_l;
            if (head_gate) {
                r *= hg;
            } else if (SHAPED && gate != nullptr) {
                const float* gp = gate + static_cast<size_t>(row) * ldg + h * head_dim + 4 * G + 16 * c;
#pragma unroll
                for (int i = 0; i < 4; ++i) r[i] *= 1.f / (1.f + expf(-gp[i]));
            }
            store4f<T>(op + 16 * c, r);
        }
    }
}

// DC: the most 16-dim chunks of a head (head_dim <= 16 DC); loops over chunks are unrolled to DC and
// predicated, so that the register arrays are indexed by constants.
// SHAPED: the scores are shaped before the softmax (score_shape.h), a chunked mask may stand in for the window, and
// the result may be multiplied by the sigmoid of a gate (fp32 rows). The queries then come times the scale alone.
template <typename T, int DC, bool SHAPED = false>
__global__ void __launch_bounds__(256)
paged_attention_tiled(const T* __restrict__ q, int q_stride, int q_col, const T* __restrict__ k_pages,
                      const T* __restrict__ v_pages, int kv_dim, const int* __restrict__ block_tables, int max_blocks,
                      const int* __restrict__ cu_q, const int* __restrict__ ctx_len, int n_seqs, int n_heads,
                      int n_kv_heads, int head_dim, int page_size, float scale_log2e, int window,
                      T* __restrict__ out, int out_stride, MllmScoreShape shape, const float* __restrict__ gate, int ldg) {
    extern __shared__ __attribute__((aligned(16))) float tl_smem[];
    const int n_c = head_dim / 16;                 // 16-dim chunks
    const int ldk = head_dim + 4;                  // floats per key row: (head_dim / 4 + 1) x 16 bytes, odd
    float* Ks = tl_smem;                           // [TL_BK][ldk]
    float* Vt = tl_smem + TL_BK * ldk;             // [head_dim][TL_VSTRIDE]

    const auto [b, tile, q_begin, q_len] = query_tile<TL_BQ>(cu_q, ctx_len, n_seqs, 1, blockIdx.y, gridDim.y);
    if (b < 0) return;                             // surplus workgroup; the whole workgroup leaves

    const int h = blockIdx.x, hk = h / (n_heads / n_kv_heads);
    const int tid = threadIdx.x, lane = tid % 64, wave = tid / 64;
    const int G = lane / 16, c16 = lane % 16;
    const int start = ctx_len[b] - q_len;          // position of the step's first query
    const int q0 = tile * TL_BQ;
    const int qi = q0 + wave * 16 + c16;           // this lane's query within the step's rows
    const bool q_ok = qi < q_len;
    const int p = start + min(qi, q_len - 1);      // its position (a lane beyond the last query repeats it; never stored)
    const int p_first = start + q0, p_last = start + min(q0 + TL_BQ, q_len) - 1;
    int k_lo = (window > 0 && p_first - window + 1 > 0) ? p_first - window + 1 : 0;
    int my_lo = (window > 0 && p - window + 1 > 0) ? p - window + 1 : 0;
    if (SHAPED && shape.chunk > 0) { k_lo = p_first - p_first % shape.chunk; my_lo = p - p % shape.chunk; }
    const float r1 = SHAPED ? mllm_bias_r1(shape, blockIdx.x) : 0.f, r2 = (SHAPED && shape.r1) ? shape.r2[blockIdx.x] : 0.f;
    // A window may keep the sequence's first kf positions visible: key tiles that lie wholly in front of the window's
    // first tile and hold kept keys run first (n_head of them); tile number vt is key tile tile_of(vt).
    const int kf = (SHAPED && window > 0) ? shape.keep_first : 0;
    const int kt_first = k_lo / TL_BK, kt_last = p_last / TL_BK;
    const int n_head = kf > 0 ? min((kf + TL_BK - 1) / TL_BK, kt_first) : 0;
    const int vt_last = n_head + kt_last - kt_first;
    // the last position any of this wavefront's queries may see (uniform over the wavefront)
    const int wave_last = start + min(q0 + wave * 16 + 15, q_len - 1);
    const int* table = block_tables + static_cast<size_t>(b) * max_blocks;
    const size_t kv_off = static_cast<size_t>(hk) * head_dim;

    // the lane's query fragment, scaled: qf[c][j] = q[16c + 4G + j] * scale * log2(e)
    f32x4_t qf[DC];
    f32x4_t o[DC];
    const T* qp = q + static_cast<size_t>(q_begin + min(qi, q_len - 1)) * q_stride + q_col + h * head_dim + 4 * G;
#pragma unroll
    for (int c = 0; c < DC; ++c) {
        o[c] = f32x4_t{0.f, 0.f, 0.f, 0.f};
        qf[c] = f32x4_t{0.f, 0.f, 0.f, 0.f};
        if (c < n_c) qf[c] = load4f<T>(qp + 16 * c) * scale_log2e;
    }
    float m = -INFINITY, l = 0.f;

    for (int vt = 0; vt <= vt_last; ++vt) {
        const int k0 = (vt < n_head ? vt : vt - n_head + kt_first) * TL_BK;
        __syncthreads();                           // the previous tile's readers are done
        // stage 64 keys and values: thread t has key t % 64 and a quarter of its dims. Keys outside
        // [k_lo, p_last] are not in the pages (not written yet, or given back by a window): zeros.
        {
            const int key = tid % TL_BK, part = tid / TL_BK, j = k0 + key;
            const bool live = (j >= k_lo || j < kf) && j <= p_last;
            size_t row = 0;
            if (live) row = static_cast<size_t>(table[j / page_size]) * page_size + j % page_size;
            const T* kp = k_pages + row * kv_dim + kv_off;
            const T* vp = v_pages + row * kv_dim + kv_off;
            const int d_per = head_dim / 4;        // a multiple of 4
            for (int d = part * d_per; d < (part + 1) * d_per; d += 4) {
                f32x4_t kv = f32x4_t{0.f, 0.f, 0.f, 0.f}, vv = kv;
                if (live) { kv = load4f<T>(kp + d); vv = load4f<T>(vp + d); }
                *reinterpret_cast<f32x4_t*>(Ks + key * ldk + d) = kv;
#pragma unroll
                for (int i = 0; i < 4; ++i) Vt[(d + i) * TL_VSTRIDE + key] = vv[i];
            }
        }
        __syncthreads();
        if (k0 > wave_last) continue;              // nothing here for this wavefront's queries (it still keeps the barriers)
        // S^T for the tile: 4 groups of 16 keys; lane holds keys k0 + 16 g + 4 G + i, i = 0..3, of its query
        f32x4_t s[4];
#pragma unroll
        for (int g = 0; g < 4; ++g) {
            s[g] = f32x4_t{0.f, 0.f, 0.f, 0.f};
            const float* kr = Ks + (g * 16 + c16) * ldk + 4 * G;
#pragma unroll
            for (int c = 0; c < DC; ++c) {
                if (c < n_c) {
                    const f32x4_t kf = *reinterpret_cast<const f32x4_t*>(kr + 16 * c);
#pragma unroll
                    for (int j = 0; j < 4; ++j) s[g] = __builtin_amdgcn_mfma_f32_16x16x4f32(kf[j], qf[c][j], s[g], 0, 0, 0);
                }
            }
        }
        // mask, running maximum and sum (scalars per lane, merged over the four lane groups of the query)
        float mx = -INFINITY;
#pragma unroll
        for (int g = 0; g < 4; ++g)
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const int j = k0 + 16 * g + 4 * G + i;
                if (SHAPED) s[g][i] = mllm_shaped_score<sizeof(T) == 2>(s[g][i], shape, r1, r2, max(p - j, 0)) * MLLM_LOG2E;
                s[g][i] = (j <= p && (j >= my_lo || j < kf)) ? s[g][i] : -INFINITY;
                mx = fmaxf(mx, s[g][i]);
            }
        const float m_new = fmaxf(m, rows_max(mx));
        // (a query none of whose keys has come yet keeps m = -inf: nothing to rescale, all weights zero)
        const float alpha = (m_new == -INFINITY) ? 1.f : exp2_for<T>(m - m_new);
        float sum = 0.f;
#pragma unroll
        for (int g = 0; g < 4; ++g)
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                s[g][i] = (m_new == -INFINITY) ? 0.f : exp2_for<T>(s[g][i] - m_new);
                sum += s[g][i];
            }
        l = l * alpha + rows_sum(sum);
        m = m_new;
        // O^T = O^T alpha + V^T P^T
#pragma unroll
        for (int c = 0; c < DC; ++c) {
            if (c < n_c) {
                o[c] *= alpha;
#pragma unroll
                for (int g = 0; g < 4; ++g) {
                    const f32x4_t vf = *reinterpret_cast<const f32x4_t*>(Vt + (16 * c + c16) * TL_VSTRIDE + 16 * g + 4 * G);
#pragma unroll
                    for (int i = 0; i < 4; ++i) o[c] = __builtin_amdgcn_mfma_f32_16x16x4f32(vf[i], s[g][i], o[c], 0, 0, 0);
                }
            }
        }
    }
    if (q_ok) finish_tiled<T, DC, SHAPED>(o, n_c, m, l, shape, gate, ldg, h, head_dim, q_begin + qi, G, out, out_stride);
}

// The same for 32-bit storage and heads of 64 or 128, which are most of what runs: key and value tiles go from the pages straight into LDS
// (lds_loads.h), a tile ahead, the block table's entries lie in LDS, and a workgroup has eight wavefronts: two share 16 queries, take
// half of every key tile each, and merge their states at the end, so that a tile's chain (wait, scores, softmax, values) is half as long
// and there are four wavefronts a SIMD to fill the gaps. Keys and values stand row-major, 16-byte piece p of row r in place p ^ (r % 16):
// the keys' 16-byte reads (16 rows, one piece) and the values' 4-byte reads (four rows, 16 columns) are free of bank conflicts.
// Bound by the chain of a workgroup's key tiles where workgroups are few (2.5 us a tile, of which the matrix instructions are 1.7), by the
// matrix cores for long prompts. 12 heads of 64, with the kernel above before: 8 x 256 tokens 30.7 > 22.7 us, 331 + 512 + 470 + 400
// 43.6 > 31, 2 x 1,024 91 > 60, 8,000 988 > 949 (104 TFLOP/s of 155); 8 heads of 128, 4 x 512 76 > 47.
// A place outside [k_lo, p_last] (not written yet, or given back by a window) loads the next key that is inside; its weight is 0, its values are taken as 0.
#define TD_TABLE 4096      // entries of a block table that fit LDS beside two stages of tiles, two workgroups a unit

template <int DH, bool SHAPED>
__global__ void __launch_bounds__(512)
paged_attention_tiled_f32(const float* __restrict__ q, int q_stride, int q_col, const float* __restrict__ k_pages,
                          const float* __restrict__ v_pages, int kv_dim, const int* __restrict__ block_tables, int max_blocks,
                          const int* __restrict__ cu_q, const int* __restrict__ ctx_len, int n_seqs, int n_heads,
                          int n_kv_heads, int page_size, float scale_log2e, int window,
                          float* __restrict__ out, int out_stride, MllmScoreShape shape, const float* __restrict__ gate, int ldg) {
    constexpr int DC = DH / 16, PIECES = DH / 4, KEYS_PER_LOAD = 64 / PIECES, LOADS = TL_BK / KEYS_PER_LOAD / 8;
    constexpr int TILE_BYTES = TL_BK * DH * 4, STAGE_BYTES = 2 * TILE_BYTES;       // keys, then values
    static_assert(LOADS * KEYS_PER_LOAD * 8 == TL_BK && PIECES % 16 == 0 && 4 * 64 * (DC * 4 + 2) * 4 <= 2 * STAGE_BYTES, "whole loads; the states fit");
    extern __shared__ __attribute__((aligned(16))) unsigned char td_smem[];
    int* table_s = reinterpret_cast<int*>(td_smem + 2 * STAGE_BYTES);

    const auto [b, tile, q_begin, q_len] = query_tile<TL_BQ>(cu_q, ctx_len, n_seqs, 1, blockIdx.y, gridDim.y);
    if (b < 0) return;                             // surplus workgroup; the whole workgroup leaves

    const int h = blockIdx.x, hk = h / (n_heads / n_kv_heads);
    const int tid = threadIdx.x, lane = tid % 64, wave = __builtin_amdgcn_readfirstlane(tid / 64), group = wave % 4, half = wave / 4;
    const int G = lane / 16, c16 = lane % 16;
    const int start = ctx_len[b] - q_len, q0 = tile * TL_BQ, qi = q0 + group * 16 + c16;
    const bool q_ok = qi < q_len;
    const int p = start + min(qi, q_len - 1);
    const int p_first = start + q0, p_last = start + min(q0 + TL_BQ, q_len) - 1;
    int k_lo = (window > 0 && p_first - window + 1 > 0) ? p_first - window + 1 : 0;
    int my_lo = (window > 0 && p - window + 1 > 0) ? p - window + 1 : 0;
    if (SHAPED && shape.chunk > 0) { k_lo = p_first - p_first % shape.chunk; my_lo = p - p % shape.chunk; }
    const float r1 = SHAPED ? mllm_bias_r1(shape, h) : 0.f, r2 = (SHAPED && shape.r1) ? shape.r2[h] : 0.f;
    const int kf = (SHAPED && window > 0) ? shape.keep_first : 0;
    const int kt_first = k_lo / TL_BK, kt_last = p_last / TL_BK;
    const int n_head = kf > 0 ? min((kf + TL_BK - 1) / TL_BK, kt_first) : 0;
    const int vt_last = n_head + kt_last - kt_first;
    const int wave_last = start + min(q0 + group * 16 + 15, q_len - 1);
    int wave_lo = (window > 0 && wave_last - window + 1 > 0) ? wave_last - window + 1 : 0;      // the first key that all its queries see
    if (SHAPED && shape.chunk > 0) wave_lo = wave_last - wave_last % shape.chunk;
    auto tile_start = [&](int vt) { return (vt < n_head ? vt : vt - n_head + kt_first) * TL_BK; };
    const int* table = block_tables + static_cast<size_t>(b) * max_blocks;
    for (int i = tid; i <= p_last / page_size; i += 512) table_s[i] = table[i];

    f32x4_t qf[DC], o[DC];
    const float* qp = q + static_cast<size_t>(q_begin + min(qi, q_len - 1)) * q_stride + q_col + h * DH + 4 * G;
#pragma unroll
    for (int c = 0; c < DC; ++c) {
        o[c] = f32x4_t{0.f, 0.f, 0.f, 0.f};
        qf[c] = load4f<float>(qp + 16 * c) * scale_log2e;
    }
    float m = -INFINITY, l = 0.f;
    __syncthreads();                               // the table is in LDS

    const unsigned lds0 = static_cast<unsigned>(reinterpret_cast<uintptr_t>((__attribute__((address_space(3))) unsigned char*)td_smem));
    const int page_shift = (page_size & (page_size - 1)) == 0 ? __ffs(page_size) - 1 : -1;
    auto fetch = [&](int vt) {
        const int k0 = tile_start(vt);
#pragma unroll
        for (int n = 0; n < LOADS; ++n) {
            const int first = (wave * LOADS + n) * KEYS_PER_LOAD, key = first + lane / PIECES;
            int j = min(k0 + key, p_last);
            if (j < k_lo && j >= kf) j = k_lo;
            const int block = page_shift >= 0 ? j >> page_shift : j / page_size;
            const size_t row = static_cast<size_t>(table_s[block]) * page_size + (j - block * page_size);
            const size_t at = (row * kv_dim + hk * DH) * 4 + (lane % PIECES ^ key % 16) * 16;
            const unsigned to = lds0 + (vt & 1) * STAGE_BYTES + first * DH * 4;
            load_to_lds(reinterpret_cast<const unsigned char*>(k_pages), at, to);
            load_to_lds(reinterpret_cast<const unsigned char*>(v_pages), at, to + TILE_BYTES);
        }
    };
    fetch(0);
    for (int vt = 0; vt <= vt_last; ++vt) {
        const int k0 = tile_start(vt);
        wait_loads_and_meet<0>();                  // this tile has come, the one before it has been read
        if (vt < vt_last) fetch(vt + 1);
        if (k0 + 32 * half > wave_last) continue;  // nothing here for this wavefront's queries (it still keeps the barriers)
        // S^T for 32 keys: lane holds keys k0 + 32 half + 16 g + 4 G + i, i = 0..3, of its query. All fragments are asked for in front
        // of what uses them, the values' in front of the softmax (the scheduling barriers keep them there).
        const unsigned char* keys = td_smem + (vt & 1) * STAGE_BYTES + 32 * half * DH * 4;
        const unsigned char* values = keys + TILE_BYTES;
        f32x4_t kr[DC][2], s[2] = {f32x4_t{0.f, 0.f, 0.f, 0.f}, f32x4_t{0.f, 0.f, 0.f, 0.f}};
        float vr[2][4][DC];
#pragma unroll
        for (int c = 0; c < DC; ++c)
#pragma unroll
            for (int g = 0; g < 2; ++g) kr[c][g] = *reinterpret_cast<const f32x4_t*>(keys + (16 * g + c16) * DH * 4 + ((4 * c + G) ^ c16) * 16);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int c = 0; c < DC; ++c)
#pragma unroll
            for (int j = 0; j < 4; ++j)
#pragma unroll
                for (int g = 0; g < 2; ++g) s[g] = __builtin_amdgcn_mfma_f32_16x16x4f32(kr[c][g][j], qf[c][j], s[g], 0, 0, 0);
#pragma unroll
        for (int i = 0; i < 4; ++i)
#pragma unroll
            for (int c = 0; c < DC; ++c)
#pragma unroll
                for (int g = 0; g < 2; ++g)
                    vr[g][i][c] = *reinterpret_cast<const float*>(values + (16 * g + 4 * G + i) * DH * 4 + ((4 * c + c16 / 4) ^ (4 * G + i)) * 16 + c16 % 4 * 4);
        __builtin_amdgcn_sched_barrier(0);
        if (SHAPED) {
#pragma unroll
            for (int g = 0; g < 2; ++g)
#pragma unroll
                for (int i = 0; i < 4; ++i)
                    s[g][i] = mllm_shaped_score<false>(s[g][i], shape, r1, r2, max(p - (k0 + 32 * half + 16 * g + 4 * G + i), 0)) * MLLM_LOG2E;
        }
        // (every query of the wavefront sees all 32 keys: nothing to mask)
        const int first = k0 + 32 * half;
        if (!(first + 31 <= start + q0 + group * 16 && first >= wave_lo)) {
#pragma unroll
            for (int g = 0; g < 2; ++g)
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    const int j = first + 16 * g + 4 * G + i;
                    s[g][i] = (j <= p && (j >= my_lo || j < kf)) ? s[g][i] : -INFINITY;
                }
            // (the places outside hold another key's values, which may be infinite: a weight of 0 does not take those away)
            if (first + 31 > p_last || first < k_lo) {
#pragma unroll
                for (int g = 0; g < 2; ++g)
#pragma unroll
                    for (int i = 0; i < 4; ++i) {
                        const int j = first + 16 * g + 4 * G + i;
                        const bool inside = j <= p_last && (j >= k_lo || j < kf);
#pragma unroll
                        for (int c = 0; c < DC; ++c) vr[g][i][c] = inside ? vr[g][i][c] : 0.f;
                    }
            }
        }
        float mx = fmaxf(fmaxf(fmaxf(s[0][0], s[0][1]), fmaxf(s[0][2], s[0][3])), fmaxf(fmaxf(s[1][0], s[1][1]), fmaxf(s[1][2], s[1][3])));
        const float m_new = fmaxf(m, rows_max(mx));
        // (A query none of whose scores so far is above -inf: all weights are zero against any finite number. Weights below the normal range
        // count as they do everywhere in 32 bits, 2^-130 of a value of 2^127 too; the bare instruction, which loses them, takes 4 to 5 % less:
        // 8 x 256 tokens 21.6 us for 22.7, 8,000 901 for 949.)
        const float against = m_new == -INFINITY ? 0.f : m_new, alpha = exp2_for<float>(m - against);
        float sum = 0.f;
#pragma unroll
        for (int g = 0; g < 2; ++g)
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                s[g][i] = exp2_for<float>(s[g][i] - against);
                sum += s[g][i];
            }
        l = l * alpha + rows_sum(sum);
        m = m_new;
#pragma unroll
        for (int c = 0; c < DC; ++c) o[c] *= alpha;
#pragma unroll
        for (int g = 0; g < 2; ++g)
#pragma unroll
            for (int i = 0; i < 4; ++i)
#pragma unroll
                for (int c = 0; c < DC; ++c) o[c] = __builtin_amdgcn_mfma_f32_16x16x4f32(vr[g][i][c], s[g][i], o[c], 0, 0, 0);
    }
    // the second half's states pass through LDS (no load is under way; the tiles have been read)
    lds_barrier();
    float* states = reinterpret_cast<float*>(td_smem) + (group * 64 + lane) * 4;
    constexpr int STATE_STEP = 4 * 64 * 4;
    if (half == 1) {
#pragma unroll
        for (int c = 0; c < DC; ++c) *reinterpret_cast<f32x4_t*>(states + c * STATE_STEP) = o[c];
        *reinterpret_cast<float2*>(states + DC * STATE_STEP - (group * 64 + lane) * 2) = make_float2(m, l);
    }
    lds_barrier();
    if (half == 1 || !q_ok) return;
    {
        const float2 other = *reinterpret_cast<const float2*>(states + DC * STATE_STEP - (group * 64 + lane) * 2);
        const float m_new = fmaxf(m, other.x), against = m_new == -INFINITY ? 0.f : m_new;     // (all its scores -inf: nothing but a sink counts)
        const float a = exp2_for<float>(m - against), a2 = exp2_for<float>(other.x - against);
        l = l * a + other.y * a2;
        m = m_new;
#pragma unroll
        for (int c = 0; c < DC; ++c) o[c] = o[c] * a + *reinterpret_cast<const f32x4_t*>(states + c * STATE_STEP) * a2;
    }
    finish_tiled<float, DC, SHAPED>(o, DC, m, l, shape, gate, ldg, h, DH, q_begin + qi, G, out, out_stride);
}

extern "C" {

// Returns 0, a HIP error code, or -1 for a head size the kernel refuses.
int mllm_paged_attention_generic(const void* q, int q_stride, int q_col, const void* k_pages,
                                 const void* v_pages, int kv_dim, const int* block_tables, int max_blocks,
                                 const int* token_seq, const int* positions, int n_tokens, int n_heads,
                                 int n_kv_heads, int head_dim, int page_size, float scale, int window,
                                 void* out, int out_stride, int dtype, hipStream_t stream) {
    if (n_tokens <= 0) return 0;
    if (head_dim % 8 != 0 || head_dim > 64 * ATT_MAX_ACC || n_heads % n_kv_heads != 0) return -1;
    const int pairs = n_tokens * n_heads;
    const int blocks = (pairs + ATT_WAVES - 1) / ATT_WAVES;
    const size_t smem = static_cast<size_t>(ATT_WAVES) * (head_dim + 2 * MLLM_WAVE) * sizeof(float);
    if (dtype == MLLM_F32)
        paged_attention_generic<float><<<blocks, ATT_WAVES * MLLM_WAVE, smem, stream>>>(
            (const float*)q, q_stride, q_col, (const float*)k_pages, (const float*)v_pages, kv_dim,
            block_tables, max_blocks, token_seq, positions, n_tokens, n_heads, n_kv_heads, head_dim,
            page_size, scale, window, (float*)out, out_stride);
    else
        paged_attention_generic<bf16_t><<<blocks, ATT_WAVES * MLLM_WAVE, smem, stream>>>(
            (const bf16_t*)q, q_stride, q_col, (const bf16_t*)k_pages, (const bf16_t*)v_pages, kv_dim,
            block_tables, max_blocks, token_seq, positions, n_tokens, n_heads, n_kv_heads, head_dim,
            page_size, scale, window, (bf16_t*)out, out_stride);
    MLLM_LAUNCH_CHECK();
    return 0;
}

// n_tiles_upper: an upper bound of the number of 64-query tiles, sum over sequences of ceil(q_len / 64)
// (e.g. n_tokens / 64 + n_seqs); surplus workgroups leave at once. The keys and values of the step's own
// tokens must already be in the pages. Returns 0, a HIP error code, or -1 for a head size that is no multiple
// of 16 or beyond 256, rows that are not 16-byte aligned, or more tiles than a grid holds.
int mllm_paged_attention_tiled(const void* q, int q_stride, int q_col, const void* k_pages, const void* v_pages,
                               int kv_dim, const int* block_tables, int max_blocks, const int* cu_q, const int* ctx_len,
                               int n_seqs, int n_tiles_upper, int n_heads, int n_kv_heads, int head_dim, int page_size,
                               float scale, int window, void* out, int out_stride, int dtype, hipStream_t stream,
                               const MllmScoreShape* shape, const float* gate, int ldg) {
    if (n_seqs <= 0 || n_tiles_upper <= 0) return 0;
    if ((shape == nullptr && gate != nullptr) || (shape && window > 0 && shape->chunk > 0)) return -1;
    const MllmScoreShape sh = shape ? *shape : MllmScoreShape{0.f, 0, nullptr, nullptr};
    if (head_dim % 16 != 0 || head_dim < 16 || head_dim > 256 || n_heads % n_kv_heads != 0 || n_tiles_upper > 65535 ||
        page_size < 1)
        return -1;
    const int esz = dtype == MLLM_F32 ? 4 : 2;
    if ((q_stride * esz) % 16 || (q_col * esz) % 16 || (kv_dim * esz) % 16 || (out_stride * esz) % 8) return -1;
    const dim3 grid(n_heads, n_tiles_upper);
    const size_t smem = (static_cast<size_t>(TL_BK) * (head_dim + 4) + static_cast<size_t>(head_dim) * TL_VSTRIDE) * sizeof(float);
    const float sl2 = shape ? scale : scale * 1.44269504088896340736f;
#define TL_CASE(TYPE, DC)                                                                                          \
    do {                                                                                                           \
        static bool lds_allowed = false;      /* more than 64 KB of LDS is asked for once */                       \
        if (!lds_allowed) {                                                                                        \
            hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(paged_attention_tiled<TYPE, DC, false>), \
                                               hipFuncAttributeMaxDynamicSharedMemorySize,                         \
                                               static_cast<int>((TL_BK * (16 * DC + 4) + 16 * DC * TL_VSTRIDE) * sizeof(float))); \
            if (e == hipSuccess) e = hipFuncSetAttribute(reinterpret_cast<const void*>(paged_attention_tiled<TYPE, DC, true>), \
                                               hipFuncAttributeMaxDynamicSharedMemorySize,                         \
                                               static_cast<int>((TL_BK * (16 * DC + 4) + 16 * DC * TL_VSTRIDE) * sizeof(float))); \
            if (e != hipSuccess) return static_cast<int>(e);                                                       \
            lds_allowed = true;                                                                                    \
        }                                                                                                          \
        if (shape) paged_attention_tiled<TYPE, DC, true><<<grid, 256, smem, stream>>>(                             \
            (const TYPE*)q, q_stride, q_col, (const TYPE*)k_pages, (const TYPE*)v_pages, kv_dim, block_tables,     \
            max_blocks, cu_q, ctx_len, n_seqs, n_heads, n_kv_heads, head_dim, page_size, sl2, window, (TYPE*)out,   \
            out_stride, sh, gate, ldg);                                                                            \
        else paged_attention_tiled<TYPE, DC, false><<<grid, 256, smem, stream>>>(                                  \
            (const TYPE*)q, q_stride, q_col, (const TYPE*)k_pages, (const TYPE*)v_pages, kv_dim, block_tables,     \
            max_blocks, cu_q, ctx_len, n_seqs, n_heads, n_kv_heads, head_dim, page_size, sl2, window, (TYPE*)out,   \
            out_stride, sh, nullptr, 0);                                                                           \
    } while (0)
#define TD_CASE(DH, SHAPED)                                                                                        \
    do {                                                                                                           \
        static bool lds_allowed = false;      /* more than 64 KB of LDS is asked for once */                       \
        constexpr int tiles_bytes = 2 * 2 * TL_BK * DH * 4;                                                        \
        if (!lds_allowed) {                                                                                        \
            const hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(paged_attention_tiled_f32<DH, SHAPED>), \
                                                     hipFuncAttributeMaxDynamicSharedMemorySize, tiles_bytes + 4 * TD_TABLE); \
            if (e != hipSuccess) return static_cast<int>(e);                                                       \
            lds_allowed = true;                                                                                    \
        }                                                                                                          \
        paged_attention_tiled_f32<DH, SHAPED><<<grid, 512, tiles_bytes + 4 * max_blocks, stream>>>(                \
            (const float*)q, q_stride, q_col, (const float*)k_pages, (const float*)v_pages, kv_dim, block_tables,  \
            max_blocks, cu_q, ctx_len, n_seqs, n_heads, n_kv_heads, page_size, sl2, window, (float*)out,           \
            out_stride, sh, shape ? gate : nullptr, ldg);                                                          \
    } while (0)
    if (dtype == MLLM_F32 && (head_dim == 64 || head_dim == 128) && max_blocks <= TD_TABLE) {
        if (head_dim == 64) {
            if (shape) TD_CASE(64, true); else TD_CASE(64, false);
        } else {
            if (shape) TD_CASE(128, true); else TD_CASE(128, false);
        }
        MLLM_LAUNCH_CHECK();
        return 0;
    }
#undef TD_CASE
    const int dc = head_dim <= 64 ? 4 : head_dim <= 128 ? 8 : 16;
    if (dtype == MLLM_F32) {
        if (dc == 4) TL_CASE(float, 4); else if (dc == 8) TL_CASE(float, 8); else TL_CASE(float, 16);
    } else {
        if (dc == 4) TL_CASE(bf16_t, 4); else if (dc == 8) TL_CASE(bf16_t, 8); else TL_CASE(bf16_t, 16);
    }
#undef TL_CASE
    MLLM_LAUNCH_CHECK();
    return 0;
}

}  // extern "C"
