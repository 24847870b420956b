// True fp32 matrix product for the 32-bit path: C[M,N] = A[M,K] * W[N,K]^T (+ bias, epilogue).
// fp32 products summed in fp32, on the vector units or the fp32 matrix cores; no reduced-precision matrix mode is
// involved. Every output is accumulated over k in an order that its kernel and tile shape fix, so which other
// rows share the launch matters only through their number, which chooses between these. Any M, N, K.
//
// Same contract as the reference's bounds-safe kernel
// (/root/reference/src/kernels/gemm.cu:238-392: alpha*acc + beta*old + bias, optional GELU),
// with the weight held as [N,K] (k contiguous) instead of [K,N].
#include <algorithm>
#include <type_traits>

#include "common.h"
#include "lds_loads.h"

#define F32_BM 64
#define F32_BN 64
#define F32_BK 16

__global__ void __launch_bounds__(256)
gemm_f32_kernel(const float* __restrict__ A, int lda, const float* __restrict__ W, int ldw,
                const float* __restrict__ bias, void* __restrict__ C, int ldc, int M, int N, int K, int mode) {
    __shared__ float As[F32_BK][F32_BM + 4];
    __shared__ float Ws[F32_BK][F32_BN + 4];
    const int tid = threadIdx.x;
    const int tx = tid % 16, ty = tid / 16;
    const int m0 = blockIdx.y * F32_BM, n0 = blockIdx.x * F32_BN;
    // loader mapping: 64 rows x 4 k-quads
    const int lrow = tid / 4, lk = (tid % 4) * 4;
    const bool vec_a = (lda % 4 == 0) && ((reinterpret_cast<uintptr_t>(A) & 15) == 0);
    const bool vec_w = (ldw % 4 == 0) && ((reinterpret_cast<uintptr_t>(W) & 15) == 0);

    float acc[4][4] = {};
    for (int k0 = 0; k0 < K; k0 += F32_BK) {
        float av[4] = {0.f, 0.f, 0.f, 0.f}, wv[4] = {0.f, 0.f, 0.f, 0.f};
        const int kk = k0 + lk;
        const int am = m0 + lrow, wn = n0 + lrow;
        if (am < M) {
            const float* p = A + static_cast<size_t>(am) * lda + kk;
            if (vec_a && kk + 3 < K) {
                float4 v = *reinterpret_cast<const float4*>(p);
                av[0] = v.x; av[1] = v.y; av[2] = v.z; av[3] = v.w;
            } else {
                for (int i = 0; i < 4; ++i) if (kk + i < K) av[i] = p[i];
            }
        }
        if (wn < N) {
            const float* p = W + static_cast<size_t>(wn) * ldw + kk;
            if (vec_w && kk + 3 < K) {
                float4 v = *reinterpret_cast<const float4*>(p);
                wv[0] = v.x; wv[1] = v.y; wv[2] = v.z; wv[3] = v.w;
            } else {
                for (int i = 0; i < 4; ++i) if (kk + i < K) wv[i] = p[i];
            }
        }
        __syncthreads();   // the previous tile's readers are done
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            As[lk + i][lrow] = av[i];
            Ws[lk + i][lrow] = wv[i];
        }
        __syncthreads();
#pragma unroll
        for (int k = 0; k < F32_BK; ++k) {
            float a[4], b[4];
#pragma unroll
            for (int i = 0; i < 4; ++i) a[i] = As[k][ty * 4 + i];
#pragma unroll
            for (int j = 0; j < 4; ++j) b[j] = Ws[k][tx * 4 + j];
#pragma unroll
            for (int i = 0; i < 4; ++i)
#pragma unroll
                for (int j = 0; j < 4; ++j) acc[i][j] = fmaf(a[i], b[j], acc[i][j]);
        }
    }
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const int m = m0 + ty * 4 + i;
        if (m >= M) continue;
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const int n = n0 + tx * 4 + j;
            if (n >= N) continue;
            epilogue<float>(mode, acc[i][j], bias ? bias[n] : 0.f, C, static_cast<size_t>(m) * ldc + n);
        }
    }
}

// Few rows (decode): the product is bound by reading W once, and tiles would
// start N/64 workgroups for it. Here a wavefront owns one output column (WAVES columns a workgroup):
// its lanes walk the column's weights in 16-byte steps (a wavefront's load is 1 KB of one row), the
// activations of up to ROWS rows wait in LDS in chunks of F32R_KC floats, and a lane's partial sums
// (k ascending) are added over the wavefront in a fixed order. M is at most ROWS.
// Needs K and the row strides in multiples of 4 floats and 16-byte aligned operands.
#define F32R_KC 512      // 128 16-byte steps: two per lane

template <int ROWS, int WAVES>
__global__ void __launch_bounds__(64 * WAVES)
gemm_f32_rows_kernel(// (the first 14 dwords arrive in registers with the wavefront, the rest comes from memory, 0.6 to 0.8 us later)
                     const float* __restrict__ A, const float* __restrict__ W, const float* __restrict__ bias, void* __restrict__ C,
                     int lda, int ldw, int ldc, int M, int N, int K, int mode) {
    __shared__ __attribute__((aligned(16))) float a_s[ROWS][F32R_KC];
    const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid / 64), lane = tid % 64;
    const int n = blockIdx.x * WAVES + wave;
    const float* wrow = W + static_cast<size_t>(min(n, N - 1)) * ldw;       // a surplus wavefront repeats the last column
    constexpr int STAGED = (ROWS * (F32R_KC / 4) + 64 * WAVES - 1) / (64 * WAVES);   // 16-byte steps of a chunk a thread stages
    static_assert(WAVES % 2 == 0 && F32R_KC == 512, "two wavefronts a staged row");
    float acc[ROWS];
#pragma unroll
    for (int r = 0; r < ROWS; ++r) acc[r] = 0.f;
    // With a handful of wavefronts on a compute unit nothing hides a load's latency but the kernel itself:
    // the weights and the activations of the next chunk are asked for before the chunk in LDS is used.
    // A chunk is at most two 16-byte steps per lane (the second from a clamped address; its product is
    // left out where it is past the chunk).
    const int q0 = lane, q1 = lane + 64;
    typedef float f4 __attribute__((ext_vector_type(4)));        // (float4s that are set under a condition would go through scratch memory)
    float4 w0, w1;
    f4 v[STAGED];
    // (a chunk's rows lie 128 steps apart, so that no step is found by a division; a row belongs to whole wavefronts, and rows beyond M
    // are neither read nor set: what stands in their place counts in no result that is stored)
    constexpr int PASS_ROWS = 64 * WAVES / 128;
    const int my_q = tid % 128, first_r = wave / 2;
    auto fetch = [&](int kc0) {
        const int quads = min(F32R_KC, K - kc0) / 4;
        w0 = *reinterpret_cast<const float4*>(wrow + kc0 + 4 * min(q0, quads - 1));
        w1 = *reinterpret_cast<const float4*>(wrow + kc0 + 4 * min(q1, quads - 1));
#pragma unroll
        for (int u = 0; u < STAGED; ++u) {
            const int r = first_r + u * PASS_ROWS;
            if (r < M) v[u] = *reinterpret_cast<const f4*>(A + static_cast<size_t>(r) * lda + kc0 + 4 * min(my_q, quads - 1));
        }
    };
    fetch(0);
    for (int kc0 = 0; kc0 < K; kc0 += F32R_KC) {
        const int quads = min(F32R_KC, K - kc0) / 4;
        const float4 c0 = w0, c1 = w1;
        __syncthreads();          // the chunk before has been read
#pragma unroll
        for (int u = 0; u < STAGED; ++u) {
            const int r = first_r + u * PASS_ROWS;
            if (r < M) *reinterpret_cast<f4*>(&a_s[r][4 * my_q]) = v[u];
        }
        if (kc0 + F32R_KC < K) fetch(kc0 + F32R_KC);
        __syncthreads();
        if (q0 < quads) {
#pragma unroll
            for (int r = 0; r < ROWS; ++r) {
                const float4 a4 = *reinterpret_cast<const float4*>(&a_s[r][4 * q0]);
                acc[r] = fmaf(a4.x, c0.x, acc[r]);
                acc[r] = fmaf(a4.y, c0.y, acc[r]);
                acc[r] = fmaf(a4.z, c0.z, acc[r]);
                acc[r] = fmaf(a4.w, c0.w, acc[r]);
            }
        }
        if (q1 < quads) {
#pragma unroll
            for (int r = 0; r < ROWS; ++r) {
                const float4 a4 = *reinterpret_cast<const float4*>(&a_s[r][4 * q1]);
                acc[r] = fmaf(a4.x, c1.x, acc[r]);
                acc[r] = fmaf(a4.y, c1.y, acc[r]);
                acc[r] = fmaf(a4.z, c1.z, acc[r]);
                acc[r] = fmaf(a4.w, c1.w, acc[r]);
            }
        }
    }
    float mine = 0.f;
#pragma unroll
    for (int r = 0; r < ROWS; ++r) {
        const float t = wave_sum(acc[r]);
        if (lane == r) mine = t;
    }
    if (n < N && lane < ROWS && lane < M)
        epilogue<float>(mode, mine, bias ? bias[n] : 0.f, C, static_cast<size_t>(lane) * ldc + n);
}

// The same for narrow results (the output projection, the feed-forward's second product), where one column a wavefront leaves few
// wavefronts and each waits for chunk after chunk of its column: two wavefronts share a column, 256 columns of K in turn, and
// ask for all their weights of a pass of KP = 512 STEPS columns at once, behind the pass's activations, which lie in LDS whole. One
// pass covers K up to 3,072; beyond, the next pass's weights are on their way while one is used. What the epilogue adds is asked for
// first. Bound by the chain launch, activations, weights, sums: 8 x 768 x 768 with two splits of attention merged in it and 8 x 768 x 3,072
// take 4.8 and 5.8 us in a decode step; unmerged and with a column a wavefront they took 17.1 together.
// RAGGED: K is no multiple of 256, and what lies beyond it has to be left out (8 x 1,600 x 1,600 7.4 us, 7.2 if it were not).
// MS > 0: A is the output of split decode attention, the states of MS splits of every (token, head) pair as attention_decode.hip leaves them
// (partial_out), merged while the rows are staged: weights over the full range of 32 bits, as the attention's own.
template <int ROWS, int STEPS, bool RAGGED, int MS>
__global__ void __launch_bounds__(512)
gemm_f32_narrow_kernel(// (the 14 dwords that arrive in registers)
                       const float* __restrict__ A, const float* __restrict__ W, const float* __restrict__ bias, void* __restrict__ C,
                       // columns and, in the upper half, columns summed; MS > 0: the splits' maxima and sums
                       const void* __restrict__ sizes_or_ml,
                       // MS > 0: head size and heads, 16 bits each, for the row stride
                       int lda, int ldw, int ldc,
                       unsigned form /* rows (4 bits), epilogue (4), MS > 0: columns */) {
    const int M = form & 15, mode = form >> 4 & 15;
    const int head_dim = lda & 0xffff, heads = static_cast<unsigned>(lda) >> 16;
    const int N = MS > 0 ? form >> 8 : static_cast<int>(reinterpret_cast<uintptr_t>(sizes_or_ml));
    const int K = MS > 0 ? heads * head_dim : static_cast<int>(reinterpret_cast<uintptr_t>(sizes_or_ml) >> 32);
    const float* split_ml = static_cast<const float*>(sizes_or_ml);
    constexpr int COLS = 4, KP = 512 * STEPS, STAGED = ROWS * KP / 4 / 512;
    static_assert(COLS * ROWS <= 64, "the first wavefront holds the outputs");
    __shared__ __attribute__((aligned(16))) float a_s[ROWS][KP];
    __shared__ float sums[2][COLS][ROWS];
    const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid / 64), lane = tid % 64;
    const int column = wave % COLS, half = wave / COLS;
    const float* wrow = W + static_cast<size_t>(min(blockIdx.x * COLS + column, static_cast<unsigned>(N - 1))) * ldw;   // (a surplus column repeats the last)
    const int out_r = tid % ROWS, out_n = blockIdx.x * COLS + tid / ROWS;
    const bool owns = tid < COLS * ROWS && out_r < M && out_n < N;
    const size_t out_at = static_cast<size_t>(min(out_r, M - 1)) * ldc + min(out_n, N - 1);
    float out_bias = 0.f, out_old = 0.f;
    if (owns && bias != nullptr) out_bias = bias[out_n];
    if (owns && mode == EPI_ADD_RESIDUAL) out_old = static_cast<const float*>(C)[out_at];
    float4 v[STAGED], w[STEPS], next[STEPS];
    auto fetch_rows = [&](int k0) {
#pragma unroll
        for (int u = 0; u < STAGED; ++u) {
            const int idx = tid + 512 * u, r = idx / (KP / 4), k = k0 + idx % (KP / 4) * 4;
            float4 a = make_float4(0.f, 0.f, 0.f, 0.f);
            if constexpr (MS == 0) {
                a = *reinterpret_cast<const float4*>(A + static_cast<size_t>(min(r, M - 1)) * lda + min(k, K - 4));
            } else if (r < M) {        // (uniform over a wavefront: a row is a quarter of a pass or more)
                // (k / head size in quarters, as small_quotient but lane by lane)
                const int kc = min(k, K - 4), h = static_cast<int>((static_cast<float>(kc / 4) + 0.5f) * __builtin_amdgcn_rcpf(static_cast<float>(head_dim / 4)));
                const size_t pair = static_cast<size_t>(r) * heads + h;
                float2 ml[MS];
                float4 o[MS];
#pragma unroll
                for (int s = 0; s < MS; ++s) {
                    ml[s] = *reinterpret_cast<const float2*>(split_ml + (pair * MS + s) * 2);
                    o[s] = *reinterpret_cast<const float4*>(A + (pair * MS + s) * head_dim + (kc - h * head_dim));
                }
                float mx = ml[0].x, l = 0.f;
#pragma unroll
                for (int s = 1; s < MS; ++s) mx = fmaxf(mx, ml[s].x);
#pragma unroll
                for (int s = 0; s < MS; ++s) {
                    const float weight = exp2f(ml[s].x - mx);
                    l = fmaf(weight, ml[s].y, l);
                    a.x = fmaf(weight, o[s].x, a.x); a.y = fmaf(weight, o[s].y, a.y); a.z = fmaf(weight, o[s].z, a.z); a.w = fmaf(weight, o[s].w, a.w);
                }
                const float inv = 1.0f / l;
                a = make_float4(a.x * inv, a.y * inv, a.z * inv, a.w * inv);
            }
            v[u] = r < M && k < K ? a : make_float4(0.f, 0.f, 0.f, 0.f);
        }
    };
    auto fetch_weights = [&](float4 (&to)[STEPS], int k0) {        // (beyond K: the row's last four)
#pragma unroll
        for (int s = 0; s < STEPS; ++s) to[s] = *reinterpret_cast<const float4*>(wrow + min(k0 + (2 * s + half) * 256 + 4 * lane, K - 4));
    };
    float acc[ROWS];
#pragma unroll
    for (int r = 0; r < ROWS; ++r) acc[r] = 0.f;
    fetch_rows(0);
    __builtin_amdgcn_sched_barrier(0);
    fetch_weights(w, 0);
    __builtin_amdgcn_sched_barrier(0);
    for (int k0 = 0; k0 < K; k0 += KP) {
        if (k0 > 0) lds_barrier();             // the pass before has been read
#pragma unroll
        for (int u = 0; u < STAGED; ++u) {
            const int idx = tid + 512 * u;
            *reinterpret_cast<float4*>(&a_s[idx / (KP / 4)][idx % (KP / 4) * 4]) = v[u];
        }
        lds_barrier();
        const bool more = k0 + KP < K;
        if (more) {
            fetch_rows(k0 + KP);
            fetch_weights(next, k0 + KP);
        } else if constexpr (RAGGED) {
            // What lies beyond K is zero in both factors (0 x infinity is none). Neither where it is loaded nor a branch a lane in
            // front of the products: the loads would wait for each other (8 x 1,600 x 1,600 18.2 us).
#pragma unroll
            for (int s = 0; s < STEPS; ++s)
                if (k0 + (2 * s + half) * 256 + 4 * lane >= K) w[s] = make_float4(0.f, 0.f, 0.f, 0.f);
        }
#pragma unroll
        for (int s = 0; s < STEPS; ++s) {
            const int q = (2 * s + half) * 256 + 4 * lane;
            if (k0 + (2 * s + half) * 256 >= K) continue;
#pragma unroll
            for (int r = 0; r < ROWS; ++r) {
                const float4 a4 = *reinterpret_cast<const float4*>(&a_s[r][q]);
                acc[r] = fmaf(a4.x, w[s].x, acc[r]);
                acc[r] = fmaf(a4.y, w[s].y, acc[r]);
                acc[r] = fmaf(a4.z, w[s].z, acc[r]);
                acc[r] = fmaf(a4.w, w[s].w, acc[r]);
            }
        }
        if (more) {
#pragma unroll
            for (int s = 0; s < STEPS; ++s) w[s] = next[s];
        }
    }
    float mine = 0.f;
#pragma unroll
    for (int r = 0; r < ROWS; ++r) {
        const float t = wave_sum(acc[r]);
        if (lane == r) mine = t;
    }
    if (lane < ROWS) sums[half][column][lane] = mine;
    lds_barrier();
    if (!owns) return;
    const float sum = sums[0][tid / ROWS][out_r] + sums[1][tid / ROWS][out_r];
    if (mode == EPI_ADD_RESIDUAL) static_cast<float*>(C)[out_at] = out_old + (sum + out_bias);
    else epilogue<float>(mode, sum, out_bias, C, out_at);
}

// The norm in front of a product of up to 8 rows, inside it: wavefront w normalises row w (K <= 2,048: a row lives in registers, NU float4
// a lane) into LDS while the weights of its CPW columns, all of them, are on their way; then every wavefront sums its columns as the few-row
// kernel does, in the same order, so that the result has the bits of norm and product apart. Every workgroup normalises the rows again,
// which costs it the rows and the norm's vectors from L2 (30 KB at K = 768) but no launch. RMS: the norm does not centre.
// Bound by its chain: launch, rows, norm, products, sums. At 8 rows of K = 768: 6.1 us for 2,304
// columns and 6.5 for 3,072 in a decode step, where the few-row kernel alone took 6.2 and 6.5 behind a norm of 2.2 and a launch's gap of 1.2.
template <int NU, int CPW, int ROWS>
__global__ void __launch_bounds__(512)
gemm_f32_normed_kernel(// (the 14 dwords that arrive in registers; K in the lower 12 bits of the last, rows (4), epilogue (4), the kind of norm)
                       const float* __restrict__ x, const float* __restrict__ W, const float* __restrict__ gamma, const float* __restrict__ beta,
                       const float* __restrict__ bias, int ldx, int ldw, int N, unsigned form,
                       void* __restrict__ C, int ldc, float eps) {
    static_assert(CPW * ROWS <= 64, "a lane an output");
    __shared__ float4 a_s[ROWS][NU * 64];
    const int K = form & 0xfff, M = form >> 12 & 15, mode = form >> 16 & 15;
    const bool rms = form >> 20 & 1;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / 64), lane = threadIdx.x % 64, nq = K / 4;
    const int n0 = (blockIdx.x * 8 + wave) * CPW;
    auto quad = [&](int u) { return u < NU - 1 ? lane + 64 * u : min(lane + 64 * u, nq - 1); };
    typedef float f4 __attribute__((ext_vector_type(4)));
    f4 v[NU], gg[NU], bb[NU], w[CPW][NU];
    const bool has_row = wave < M;
    if (has_row) {
        const f4* row = reinterpret_cast<const f4*>(x + static_cast<size_t>(wave) * ldx);
        const f4 *g4 = reinterpret_cast<const f4*>(gamma), *b4 = reinterpret_cast<const f4*>(beta != nullptr ? beta : gamma);
#pragma unroll
        for (int u = 0; u < NU; ++u) v[u] = row[quad(u)];
#pragma unroll
        for (int u = 0; u < NU; ++u) { gg[u] = g4[quad(u)]; bb[u] = b4[quad(u)]; }
    }
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int c = 0; c < CPW; ++c) {
        const f4* wrow = reinterpret_cast<const f4*>(W + static_cast<size_t>(min(n0 + c, N - 1)) * ldw);       // (a surplus column repeats the last)
#pragma unroll
        for (int u = 0; u < NU; ++u) w[c][u] = __builtin_nontemporal_load(wrow + quad(u));
    }
    const int out_r = lane % ROWS, out_n = n0 + lane / ROWS;
    const float out_bias = bias != nullptr ? bias[min(out_n, N - 1)] : 0.f;
    __builtin_amdgcn_sched_barrier(0);
    if (has_row) {
        float s = 0.f;
#pragma unroll
        for (int u = 0; u < NU; ++u)
            if (u < NU - 1 || lane + 64 * u < nq) s += (v[u].x + v[u].y) + (v[u].z + v[u].w);
        const float mean = rms ? 0.f : wave_sum(s) / static_cast<float>(K);
        float q = 0.f;
#pragma unroll
        for (int u = 0; u < NU; ++u) {
            if (u < NU - 1 || lane + 64 * u < nq) {
                q += squares_sum(v[u].x - mean, v[u].y - mean, v[u].z - mean, v[u].w - mean);
            }
        }
        const float inv = 1.0f / sqrtf(wave_sum(q) / static_cast<float>(K) + eps);
#pragma unroll
        for (int u = 0; u < NU; ++u) {
            const f4 g = gg[u], b = beta != nullptr ? bb[u] : f4{0.f, 0.f, 0.f, 0.f};
            a_s[wave][lane + 64 * u] = make_float4((v[u].x - mean) * inv * g.x + b.x, (v[u].y - mean) * inv * g.y + b.y,
                                                   (v[u].z - mean) * inv * g.z + b.z, (v[u].w - mean) * inv * g.w + b.w);
        }
    }
    lds_barrier();
    float acc[CPW][ROWS];
#pragma unroll
    for (int c = 0; c < CPW; ++c)
#pragma unroll
        for (int r = 0; r < ROWS; ++r) acc[c][r] = 0.f;
#pragma unroll
    for (int u = 0; u < NU; ++u) {
        if (u < NU - 1 || lane + 64 * u < nq) {
#pragma unroll
            for (int r = 0; r < ROWS; ++r) {        // (rows beyond M: what stands there counts in no result that is stored)
                const float4 a4 = a_s[r][lane + 64 * u];
#pragma unroll
                for (int c = 0; c < CPW; ++c) {
                    acc[c][r] = fmaf(a4.x, w[c][u].x, acc[c][r]);
                    acc[c][r] = fmaf(a4.y, w[c][u].y, acc[c][r]);
                    acc[c][r] = fmaf(a4.z, w[c][u].z, acc[c][r]);
                    acc[c][r] = fmaf(a4.w, w[c][u].w, acc[c][r]);
                }
            }
        }
    }
    float mine = 0.f;
#pragma unroll
    for (int c = 0; c < CPW; ++c)
#pragma unroll
        for (int r = 0; r < ROWS; ++r) {
            const float t = wave_sum(acc[c][r]);
            if (lane == c * ROWS + r) mine = t;
        }
    if (lane < CPW * ROWS && out_r < M && out_n < N) epilogue<float>(mode, mine, out_bias, C, static_cast<size_t>(out_r) * ldc + out_n);
}

template <int ROWS, int STEPS>
static void launch_f32_narrow(const float* A, int lda, const float* W, int ldw, const float* bias, void* C, int ldc, int M, int N, int K, int mode, hipStream_t stream) {
    const dim3 grid((N + 3) / 4);
    const void* sizes = reinterpret_cast<const void*>(static_cast<uintptr_t>(static_cast<unsigned>(N)) | static_cast<uintptr_t>(static_cast<unsigned>(K)) << 32);
    const unsigned form = M | (mode < 0 || mode > 15 ? 15 : mode) << 4;
    if (K % 256 != 0) gemm_f32_narrow_kernel<ROWS, STEPS, true, 0><<<grid, 512, 0, stream>>>(A, W, bias, C, sizes, lda, ldw, ldc, form);
    else gemm_f32_narrow_kernel<ROWS, STEPS, false, 0><<<grid, 512, 0, stream>>>(A, W, bias, C, sizes, lda, ldw, ldc, form);
}
template <int STEPS, int MS>
static void launch_f32_narrow_merged(const float* split_o, const float* split_ml, int heads, int head_dim, const float* W, int ldw, const float* bias, void* C,
                                     int ldc, int M, int N, int mode, hipStream_t stream) {
    const dim3 grid((N + 3) / 4);
    const unsigned form = M | mode << 4 | static_cast<unsigned>(N) << 8;
    if (heads * head_dim % 256 != 0) gemm_f32_narrow_kernel<8, STEPS, true, MS><<<grid, 512, 0, stream>>>(split_o, W, bias, C, split_ml, head_dim | heads << 16, ldw, ldc, form);
    else gemm_f32_narrow_kernel<8, STEPS, false, MS><<<grid, 512, 0, stream>>>(split_o, W, bias, C, split_ml, head_dim | heads << 16, ldw, ldc, form);
}

// More than a few rows, on the fp32 matrix cores (v_mfma_f32_16x16x4_f32, 256 operations a clock and compute unit). WM x WN
// wavefronts of TM x TN tiles of 16 x 16 each share k tiles of 32 columns (a row's piece is one 128-byte line) in STAGES stages of LDS,
// filled by loads that write LDS without passing through registers, one barrier a tile. KG such groups take the 32-column parts of
// a KG times as wide k tile and add their sums in LDS. A lane's 16-byte read holds the k columns of four matrix instructions (lane
// group l / 16 takes columns 4 (l / 16) to + 3 of 16, the same for both operands). The weights are the instruction's first operand, so
// that a lane ends up with four neighbouring columns of one row. While a step of 16 columns multiplies, the fragments of the next are
// read (the scheduling barriers keep the reads in front: left alone, the compiler puts them behind the products and waits for them) and the
// sums of the one before join the outputs'.
//
// How an output is summed decides its error: SUMS = 1 makes sums of 16 columns that join one after the other, 4 eight sums of four columns
// a k tile that are added pairwise first; the 32-column parts of K go to PARTS x KG sums in turn, which are added at the end (which
// of both the factors is does not change a bit). The error against 64 bits (2-norm over 2-norm, normal values, K = 768 and 3,072) is
// 1.5e-7 and 2.4e-7 with one sum, 1.2e-7 and 2.0e-7 with two, 9.1e-8 and 1.2e-7 with four of eight sums; one chain of FMAs had 5.0e-7 and
// 9.9e-7, the kernel for few rows has 9.3e-8 and 1.4e-7.
//
// Bound by the matrix cores (busy in 78 % of a unit's clocks at 2,048 x 3,072 x 768, where units idle for another 15 % of the
// launch, at its start and while the last tiles run out) or, where tiles are few, by a workgroup's chain of k tiles. Weights from memory,
// with loads that pass through registers before: 2,048 x 3,072 x 768 95 > 84 us (115 TFLOP/s of the 155 a loop of these instructions reaches),
// 2,048 x 768 x 3,072 102 > 88, 560 x 768 x 3,072 44 > 39, 64 x 768 x 3,072 25.2 > 20.1, 64 x 50,257 x 768 80 > 68. Larger tiles
// (128 x 128, 128 x 192) are no faster, so it is not the loads either. Needs K and the row strides in multiples of 4 floats,
// 16-byte aligned operands.
#define F32T_BK 32
typedef float f32x4v __attribute__((ext_vector_type(4)));

template <int WM, int WN, int TM, int TN, int KG, int PARTS, int STAGES, int SUMS, bool EDGE>
__global__ void __launch_bounds__(WM * WN * KG * 64)
gemm_f32_tiles_kernel(// (all that the first tiles' loads need is among the 14 dwords that arrive in registers)
                      const float* __restrict__ A, const float* __restrict__ W, const float* __restrict__ bias, void* __restrict__ C,
                      int lda, int ldw, int M, int N, int K, int ldc, int mode) {
    constexpr int NW = WM * WN, BM = WM * TM * 16, BN = WN * TN * 16, ROWS = BM + BN, BK = F32T_BK * KG, KS = F32T_BK / 16;
    constexpr int LOADS = (ROWS / 8 + NW - 1) / NW; // of a wavefront and k tile: 8 rows of its group's 32 columns each (the last again where there are fewer)
    constexpr int SLAB_BYTES = ROWS * F32T_BK * 4, STAGE_BYTES = SLAB_BYTES * KG;
    static_assert(ROWS % 8 == 0 && BM % 8 == 0 && KS == 2 && STAGES >= 2 && (KG == 1 || KG == 2 || KG == 4), "whole loads, two fragment sets");
    static_assert((KG - 1) * PARTS * NW * TM * TN * 64 * 16 <= STAGES * STAGE_BYTES, "the groups' sums fit the tiles' LDS");
    __shared__ __attribute__((aligned(16))) unsigned char smem[STAGES * STAGE_BYTES];
    const int tid = threadIdx.x, lane = tid % 64;
    const int kg = __builtin_amdgcn_readfirstlane(tid / (64 * NW)), wave = __builtin_amdgcn_readfirstlane(tid / 64 % NW);
    // an XCD (workgroup id % 8) takes an even share of the tiles, neighbours in one direction: with `down` it walks down the
    // rows of A for a few columns of tiles, else along the rows of W for a few rows of tiles
    const int tiles_m = (M + BM - 1) / BM, tiles_n = (N + BN - 1) / BN;
    const bool down = M <= N;
    const int tiles = tiles_m * tiles_n, per = (tiles + 7) / 8, at = (blockIdx.x % 8) * per + blockIdx.x / 8;
    if (static_cast<int>(blockIdx.x / 8) >= per || at >= tiles) return;
    const int side = down ? tiles_m : tiles_n, over = uniform_quotient(at, side), within = at - over * side;
    const int tm = down ? within : over, tn = down ? over : within;
    const int m0 = tm * BM, n0 = tn * BN;

    // A group's 32 columns of a k tile in LDS are its rows one behind the other (A's, then W's), as the loads leave them. 16-byte piece
    // p of row r stands in place p ^ swizzle(r): the 16 lanes that an LDS read serves at a time (16 rows, one piece) fall on 16
    // different groups of banks. A lane asks for the piece whose place is its own; rows beyond the matrices are the last one, never stored.
    auto swizzle = [](int row) { return (row >> 1) & 7; };
    const unsigned char* base[LOADS];
    size_t offset[LOADS];
    auto first_row = [&](int q) { return min((wave * LOADS + q) * 8, ROWS - 8); };
#pragma unroll
    for (int q = 0; q < LOADS; ++q) {
        const int first = first_row(q), row = first + lane / 8;
        const bool of_a = first < BM;
        base[q] = reinterpret_cast<const unsigned char*>(of_a ? A + static_cast<size_t>(m0) * lda : W + static_cast<size_t>(n0) * ldw);
        offset[q] = static_cast<size_t>(of_a ? min(row, M - 1 - m0) : min(row - BM, N - 1 - n0)) * (of_a ? lda : ldw) * 4 + kg * 128 + (lane % 8 ^ swizzle(row)) * 16;
    }
    const unsigned lds0 = static_cast<unsigned>(reinterpret_cast<uintptr_t>((__attribute__((address_space(3))) unsigned char*)smem)) + kg * SLAB_BYTES;
    const int nk = (K + BK - 1) / BK, rest = K - (nk - 1) * BK;      // k tiles; columns of the last
    auto fetch = [&](int q, int t, int stage) {
        size_t from = offset[q];
        if (EDGE && t == nk - 1) {         // (pieces beyond K: the row's last one, against zeros)
            const int column = kg * 128 + (lane % 8 ^ swizzle(first_row(q) + lane / 8)) * 16;
            from -= max(column - (rest * 4 - 16), 0);
        }
        load_to_lds(base[q] + static_cast<size_t>(t) * (BK * 4), from, lds0 + stage * STAGE_BYTES + first_row(q) * 128);
    };
    // lane l holds columns 4 (l / 16) to + 3 of row l % 16 of every 16 x 16 tile; what the epilogue adds there is asked for in front of the last tiles
    const int wm = wave / WN, wn = wave % WN, row16 = lane % 16, quad = lane / 16;
    const bool vec = ldc % 4 == 0 && (reinterpret_cast<uintptr_t>(C) & 15) == 0 && (bias == nullptr || (reinterpret_cast<uintptr_t>(bias) & 15) == 0);
#pragma unroll
    for (int s = 0; s < STAGES - 1; ++s) {
        if (s >= nk) break;
#pragma unroll
        for (int q = 0; q < LOADS; ++q) fetch(q, s, s);
    }

    const f32x4v zero = {0.f, 0.f, 0.f, 0.f};
    f32x4v acc[PARTS][TM][TN], sum[KS][SUMS][TM][TN], four[TM][TN], fa[KS][TM], fw[KS][TN];
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j) {
            four[i][j] = zero;
#pragma unroll
            for (int p = 0; p < PARTS; ++p) acc[p][i][j] = zero;
#pragma unroll
            for (int e = 0; e < SUMS; ++e) sum[1][e][i][j] = zero;
        }
    const int a_row = wm * TM * 16 + row16, w_row = BM + wn * TN * 16 + row16;       // (16 rows on the swizzle is the same)
    int a_at[KS], w_at[KS];
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) {
        a_at[ks] = kg * SLAB_BYTES + a_row * 128 + ((4 * ks + quad) ^ swizzle(a_row)) * 16;
        w_at[ks] = kg * SLAB_BYTES + w_row * 128 + ((4 * ks + quad) ^ swizzle(w_row)) * 16;
    }
    auto read_frags = [&](int stage_at, int ks) {
#pragma unroll
        for (int i = 0; i < TM; ++i) fa[ks][i] = *reinterpret_cast<const f32x4v*>(smem + stage_at + a_at[ks] + i * 16 * 128);
#pragma unroll
        for (int j = 0; j < TN; ++j) fw[ks][j] = *reinterpret_cast<const f32x4v*>(smem + stage_at + w_at[ks] + j * 16 * 128);
    };
    auto multiply = [&](int ks) {
#pragma unroll
        for (int e = 0; e < 4; ++e)
#pragma unroll
            for (int i = 0; i < TM; ++i)
#pragma unroll
                for (int j = 0; j < TN; ++j) {
                    f32x4v& to = sum[ks][e % SUMS][i][j];
                    to = __builtin_amdgcn_mfma_f32_16x16x4f32(fw[ks][j][e], fa[ks][i][e], e < SUMS ? zero : to, 0, 0, 0);
                }
    };
    // The sums of the step before join the outputs' while this step's are made. Eight sums of four columns (a k tile's, TM x TN of 1)
    // are added pairwise first.
    auto join = [&](int ks, f32x4v (&to)[TM][TN]) {
#pragma unroll
        for (int i = 0; i < TM; ++i)
#pragma unroll
            for (int j = 0; j < TN; ++j) {
                if constexpr (SUMS == 1) {
                    to[i][j] += sum[1 - ks][0][i][j];
                } else {
                    const f32x4v t = (sum[1 - ks][0][i][j] + sum[1 - ks][1][i][j]) + (sum[1 - ks][2][i][j] + sum[1 - ks][3][i][j]);
                    if (ks == 1) four[i][j] = t;
                    else to[i][j] += four[i][j] + t;
                }
            }
    };
    // Tile t is in stage t % STAGES, the tiles up to t + STAGES - 2 are on their way, and tile t + STAGES - 1 is asked for into the
    // stage that tile t - 1 left. The wavefronts wait for the next tile and meet in front of a tile's last products, and its first fragments
    // are read there: neither stands alone.
    wait_tiles_and_meet<STAGES - 2, LOADS>(nk - 1);
    read_frags(0, 0);
    int stage_at = 0, fetch_stage = STAGES - 1;
    auto step = [&](auto fetches, int t, int part) {
        constexpr bool FETCHES = decltype(fetches)::value;
        const int next_at = stage_at == (STAGES - 1) * STAGE_BYTES ? 0 : stage_at + STAGE_BYTES;
#pragma unroll
        for (int ks = 0; ks < KS; ++ks) {
            if (FETCHES && ks == 0) {
#pragma unroll
                for (int q = 0; q < LOADS; ++q) fetch(q, t + STAGES - 1, fetch_stage);
            }
            if (ks + 1 < KS) {
                read_frags(stage_at, ks + 1);
            } else if (FETCHES) {
                wait_loads_and_meet<(STAGES - 2) * LOADS>();
                read_frags(next_at, 0);
            } else if (t + 1 < nk) {
                wait_tiles_and_meet<(STAGES > 2 ? STAGES - 3 : 0), LOADS>(nk - 2 - t);
                read_frags(next_at, 0);
            }
            __builtin_amdgcn_sched_barrier(0);
            if (EDGE && !FETCHES && t == nk - 1 && kg * F32T_BK + 16 * ks + 4 * quad >= rest) {
#pragma unroll
                for (int i = 0; i < TM; ++i) fa[ks][i] = zero;
#pragma unroll
                for (int j = 0; j < TN; ++j) fw[ks][j] = zero;
            }
            multiply(ks);
            join(ks, acc[ks == 1 ? part : (part + PARTS - 1) % PARTS]);
            __builtin_amdgcn_sched_barrier(0);
        }
        stage_at = next_at;
        fetch_stage = fetch_stage == STAGES - 1 ? 0 : fetch_stage + 1;
    };
    const std::true_type asking;
    const std::false_type done;
    int t = 0;
    if constexpr (PARTS == 2) {
        for (; t + STAGES < nk; t += 2) {
            step(asking, t, 0);
            step(asking, t + 1, 1);
        }
    } else {
        for (; t + STAGES - 1 < nk; ++t) step(asking, t, 0);
    }
    float4 add[TN], old[TM][TN];
#pragma unroll
    for (int j = 0; j < TN; ++j) {
        const int n = n0 + (wn * TN + j) * 16 + 4 * quad;
        add[j] = make_float4(0.f, 0.f, 0.f, 0.f);
        if (vec && kg == 0 && bias != nullptr && n + 4 <= N) add[j] = *reinterpret_cast<const float4*>(bias + n);
#pragma unroll
        for (int i = 0; i < TM; ++i) {
            const int m = m0 + (wm * TM + i) * 16 + row16;
            old[i][j] = make_float4(0.f, 0.f, 0.f, 0.f);
            if (vec && kg == 0 && mode == EPI_ADD_RESIDUAL && m < M && n + 4 <= N) old[i][j] = *reinterpret_cast<const float4*>(static_cast<const float*>(C) + static_cast<size_t>(m) * ldc + n);
        }
    }
    if constexpr (PARTS == 2) {
        if (t + STAGES - 1 < nk) {
            step(asking, t, 0);
            step(done, t + 1, 1);
            t += 2;
        }
        for (; t < nk; t += 2) {
            step(done, t, 0);
            if (t + 1 < nk) step(done, t + 1, 1);
        }
    } else {
        for (; t < nk; ++t) step(done, t, 0);
    }
    if (PARTS == 2 && nk % 2 == 0) join(0, acc[PARTS - 1]);
    else join(0, acc[0]);
    // The other groups leave their sums in LDS and go; group 0 adds them: parts 0 of the groups in their order, then parts 1; of four groups,
    // two and two.
    if constexpr (KG > 1) {
        lds_barrier();               // (the tiles have been read; no load is under way)
        f32x4v* sums = reinterpret_cast<f32x4v*>(smem);
        auto place = [&](int g, int p, int i, int j) -> f32x4v& { return sums[((((g - 1) * PARTS + p) * NW + wave) * TM * TN + i * TN + j) * 64 + lane]; };
        if (kg > 0) {
#pragma unroll
            for (int p = 0; p < PARTS; ++p)
#pragma unroll
                for (int i = 0; i < TM; ++i)
#pragma unroll
                    for (int j = 0; j < TN; ++j) place(kg, p, i, j) = acc[p][i][j];
        }
        lds_barrier();
        if (kg > 0) return;
#pragma unroll
        for (int i = 0; i < TM; ++i)
#pragma unroll
            for (int j = 0; j < TN; ++j) {
                if constexpr (KG == 4) acc[0][i][j] = (acc[0][i][j] + place(1, 0, i, j)) + (place(2, 0, i, j) + place(3, 0, i, j));
                else if constexpr (PARTS == 2) acc[0][i][j] = (acc[0][i][j] + place(1, 0, i, j)) + (acc[1][i][j] + place(1, 1, i, j));
                else acc[0][i][j] += place(1, 0, i, j);
            }
    } else if constexpr (PARTS == 2) {
#pragma unroll
        for (int i = 0; i < TM; ++i)
#pragma unroll
            for (int j = 0; j < TN; ++j) acc[0][i][j] += acc[1][i][j];
    }
#pragma unroll
    for (int i = 0; i < TM; ++i) {
        const int m = m0 + (wm * TM + i) * 16 + row16;
        if (m >= M) continue;
#pragma unroll
        for (int j = 0; j < TN; ++j) {
            const int n = n0 + (wn * TN + j) * 16 + 4 * quad;
            float* out = static_cast<float*>(C) + static_cast<size_t>(m) * ldc + n;
            if (vec && n + 4 <= N) {
                const float v[4] = {acc[0][i][j][0] + add[j].x, acc[0][i][j][1] + add[j].y, acc[0][i][j][2] + add[j].z, acc[0][i][j][3] + add[j].w};
                float o[4] = {old[i][j].x, old[i][j].y, old[i][j].z, old[i][j].w};
#pragma unroll
                for (int e = 0; e < 4; ++e)
                    o[e] += mode == EPI_GELU_TANH ? gelu_tanh_precise(v[e]) : mode == EPI_GELU_ERF ? gelu_erf(v[e]) : mode == EPI_RELU2 ? relu2(v[e]) : v[e];
                *reinterpret_cast<float4*>(out) = make_float4(o[0], o[1], o[2], o[3]);
            } else {
                for (int e = 0; e < 4 && n + e < N; ++e)
                    epilogue<float>(mode, acc[0][i][j][e], bias ? bias[n + e] : 0.f, C, static_cast<size_t>(m) * ldc + n + e);
            }
        }
    }
}

template <int WM, int WN, int TM, int TN, int KG, int PARTS, int STAGES, int SUMS>
static void launch_f32_tiles(const float* A, int lda, const float* W, int ldw, const float* bias, void* C, int ldc, int M, int N, int K, int mode,
                             hipStream_t stream) {
    const int tiles_m = (M + 16 * WM * TM - 1) / (16 * WM * TM), tiles_n = (N + 16 * WN * TN - 1) / (16 * WN * TN);
    const dim3 grid((tiles_m * tiles_n + 7) / 8 * 8), block(64 * WM * WN * KG);
    if (K % (F32T_BK * KG) != 0)
        gemm_f32_tiles_kernel<WM, WN, TM, TN, KG, PARTS, STAGES, SUMS, true><<<grid, block, 0, stream>>>(A, W, bias, C, lda, ldw, M, N, K, ldc, mode);
    else
        gemm_f32_tiles_kernel<WM, WN, TM, TN, KG, PARTS, STAGES, SUMS, false><<<grid, block, 0, stream>>>(A, W, bias, C, lda, ldw, M, N, K, ldc, mode);
}

// Which tiles: 32 x 32 with four groups, two groups of two parts or one group of two parts; 64 x 32 in two parts; 128 x 64 in one.
enum TileShape { T32_FOUR, T32_TWO, T32_ONE, T64X32, T128X64 };

// Two questions. How exactly a result is summed is a rule on its sizes alone: in four sums of eight (tiles of 32 x 32) up to
// 64 rows, whose result is then as exact as that of the kernel for few rows, while there are at most 512 such tiles, and where
// they were the fastest choice when tiles were loaded through registers (the price of the fullest compute unit: its tiles
// times what they took there at K = 768, in tenths of a microsecond; with two groups a sixth of that is there at any K);
// otherwise in two sums, or in one where that was.
// Which tile then. Of 32 x 32: four groups where a unit has one tile and a long chain of k tiles (128 x 1,600 x 6,400: 40.8 us, two groups of
// two parts 43.5; 560 x 768 x 768, two tiles a unit: 12.3, four groups 15.4); one group where there are many tiles of at most four k tiles, whose
// eight wavefronts and three stages would be started for one round of loads (256 x 7,104 x 32 14.1 us with two groups, 7.9 with one, 512 x 3,328 x 100
// 16.8 and 12.2; the eight-sums error is the same up to there, and 0.1 to 9 % larger than in four sums behind it).
// Up to K = 48 64 x 32 and 128 x 64 make the same sums, and one of the latter costs what 3.3 of the former do
// (2,560 x 44,096 x 24 228 us with 64 x 32, 174 with 128 x 64; 320 x 22,272 x 4 16.9 and 18.1).
// Else of 64 x 32 in two sums, which is the fastest or within 3 % of it over 40 sizes from K = 256 on, and of 128 x 64 in one the cheaper, by prices
// fitted to those sizes (microseconds: 2,048 x 3,072 x 768 91 and 84 us, 1,812 x 768 x 2,048 60 and 79; up to K of about 470 they say 64 x 32
// for many tiles, which is the more exact and up to 12 % the slower: 4,096 x 4,096 x 256 90 and 80 us).
static TileShape tile_shape(int M, int N, int K) {
    const auto tiles = [&](int tm, int tn) { return static_cast<long>((M + 32 * tm - 1) / (32 * tm)) * ((N + 32 * tn - 1) / (32 * tn)); };
    const auto fullest = [&](int tm, int tn) { return ((tiles(tm, tn) + 7) / 8 + 31) / 32; };
    const long k = K <= 96 ? K : 768, two_groups = 5 * k + 768, one_group = 6 * k, never = 1L << 60;
    const long c11 = fullest(1, 1) * 44 * two_groups, c21 = tiles(2, 1) < 256 ? never : fullest(2, 1) * 80 * two_groups;
    const long c22 = std::min(tiles(2, 2) < 512 ? never : fullest(2, 2) * 144 * one_group, tiles(2, 3) < 512 ? never : fullest(2, 3) * 222 * one_group);
    if (M <= 64 || tiles(1, 1) <= 512) return tiles(1, 1) <= 256 && K >= 1536 ? T32_FOUR : T32_TWO;
    if (c11 < c21 && c11 < c22) return K <= 128 ? T32_ONE : T32_TWO;
    if (K <= 48) return 33 * fullest(4, 2) <= 10 * fullest(2, 1) ? T128X64 : T64X32;
    const float small = 4.96f + fullest(2, 1) * (K * 0.00973f - 0.43f), large = 3.49f + fullest(4, 2) * (K * 0.03264f + 1.26f);
    return c22 <= c21 && large < small ? T128X64 : T64X32;
}

// bfloat16 operands of any K, strides and alignment (what the matrix-core kernels of gemm_bf16.hip refuse:
// they read 16 bytes at a time): one wavefront per output column and 8 rows, the lanes over k, sums in fp32.
__global__ void __launch_bounds__(256)
gemm_bf16_plain_kernel(const bf16_t* __restrict__ A, int lda, const bf16_t* __restrict__ W, int ldw,
                       const float* __restrict__ bias, void* __restrict__ C, int ldc, int M, int N, int K, int mode) {
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / MLLM_WAVE), lane = threadIdx.x % MLLM_WAVE;
    const int n = blockIdx.x * 4 + wave;
    if (n >= N) return;
    const bf16_t* wr = W + static_cast<size_t>(n) * ldw;
    for (int m0 = blockIdx.y * 8; m0 < M; m0 += gridDim.y * 8) {
        float acc[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
        for (int k = lane; k < K; k += 64) {
            const float wv = to_float(wr[k]);
#pragma unroll
            for (int r = 0; r < 8; ++r) acc[r] += wv * to_float(A[static_cast<size_t>(min(m0 + r, M - 1)) * lda + k]);
        }
#pragma unroll
        for (int r = 0; r < 8; ++r) {
            const float v = wave_sum(acc[r]);
            if (lane == 0 && m0 + r < M) epilogue<bf16_t>(mode, v, bias ? bias[n] : 0.f, C, static_cast<size_t>(m0 + r) * ldc + n);
        }
    }
}

extern "C" {

int mllm_gemm_bf16_plain(const void* A, int lda, const void* W, int ldw, const float* bias, void* C, int ldc,
                         int M, int N, int K, int mode, hipStream_t stream) {
    if (M <= 0 || N <= 0) return 0;
    const dim3 grid((N + 3) / 4, std::min((M + 7) / 8, 256));
    gemm_bf16_plain_kernel<<<grid, 256, 0, stream>>>(static_cast<const bf16_t*>(A), lda, static_cast<const bf16_t*>(W), ldw, bias, C, ldc,
                                                     M, N, K, mode);
    MLLM_LAUNCH_CHECK();
    return 0;
}

// The product whose A is the output of split decode attention, merged from the splits' states while it is staged: see mllm_gemm_bf16_merged.
// Up to 8 rows, 2 to 4 splits, results of fewer than 2,048 columns, heads of a multiple of 4 columns, up to 3,072 in all. -1: misaligned
// operands, -2: sizes the kernel does not take.
int mllm_gemm_f32_merged(const float* split_o, const float* split_ml, int n_splits, int n_heads, int head_dim, const float* W, int ldw, const float* bias,
                         void* C, int ldc, int M, int N, int mode, hipStream_t stream) {
    const int K = n_heads * head_dim;
    if (M <= 0 || N <= 0) return 0;
    if (M > 8 || n_splits < 2 || n_splits > 4 || N >= 2048 || K > 3072 || head_dim % 4 != 0 || mode < 0 || mode > 15 || n_heads > 0xffff) return -2;
    if (ldw % 4 != 0 || ((reinterpret_cast<uintptr_t>(W) | reinterpret_cast<uintptr_t>(split_o)) & 15) || (reinterpret_cast<uintptr_t>(split_ml) & 7)) return -1;
#define MERGED(STEPS, MS) launch_f32_narrow_merged<STEPS, MS>(split_o, split_ml, n_heads, head_dim, W, ldw, bias, C, ldc, M, N, mode, stream)
#define MERGED_SPLITS(STEPS) do { if (n_splits == 2) MERGED(STEPS, 2); else if (n_splits == 3) MERGED(STEPS, 3); else MERGED(STEPS, 4); } while (0)
    if (K <= 1024) MERGED_SPLITS(2); else MERGED_SPLITS(3);
#undef MERGED_SPLITS
#undef MERGED
    MLLM_LAUNCH_CHECK();
    return 0;
}

// The norm of the fp32 rows x [M, K] (a LayerNorm, or with rms != 0 an RMS norm) inside the product of up to 8 of them: C = epilogue(norm(x) W^T + bias).
// -2: sizes the kernel does not take (more rows, K over 2,048 or no multiple of 4, operands that are not 16-byte aligned, or fewer columns than
// the few-row kernel has in this order of sums); norm and product apart are right for those. Inside / apart, back to back on cold weights, us, 1, 4 and 8
// rows: 2,304 x 768 3.6 / 6.8, 4.9 / 6.5, 5.6 / 7.5; 4,096 x 1,024 4.7 / 8.5, 6.1 / 8.2, 6.7 / 9.2; 5,120 x 1,280 7.1 / 9.9, 9.1 / 10.7, 10.4 / 12.1; 6,400 x 1,600
// 9.3 / 13.7, 12.7 / 14.7, 15.1 / 16.7; 8,192 x 2,048 13.4 / 16.7, 17.2 / 19.7, 19.1 / 20.3. Inside loses 2 to 6 % at 5 to 8 rows of 4,800 x 1,600 (14.6 / 14.0)
// and a row count or two of 2,304 and 6,144 x 2,048 (6 rows 17.4 / 16.4): no line drawn for those. (GPT-2 XL, 8 rows, a step: 3.64 > 3.49 ms.)
int mllm_norm_gemm_f32(const float* x, int ldx, const float* gamma, const float* beta, float eps, int rms, const float* W, int ldw, const float* bias,
                       void* C, int ldc, int M, int N, int K, int mode, hipStream_t stream) {
    if (M <= 0 || N <= 0) return 0;
    if (M > 8 || N < 2048 || K < 4 || K > 2048 || K % 4 != 0 || ldx % 4 != 0 || ldw % 4 != 0 || mode < 0 || mode > 15 || gamma == nullptr ||
        ((reinterpret_cast<uintptr_t>(x) | reinterpret_cast<uintptr_t>(W) | reinterpret_cast<uintptr_t>(gamma) | reinterpret_cast<uintptr_t>(beta)) & 15) != 0)
        return -2;
    const unsigned form = K | M << 12 | mode << 16 | (rms ? 1u << 20 : 0u);
    // (two columns a wavefront where one would take more than two rounds of workgroups)
    const bool two = N > 4096;
    const dim3 grid(two ? (N + 15) / 16 : (N + 7) / 8);
#define NORMED(NU, CPW, ROWS) gemm_f32_normed_kernel<NU, CPW, ROWS><<<grid, 512, 0, stream>>>(x, W, gamma, beta, bias, ldx, ldw, N, form, C, ldc, eps)
#define NORMED_CASE(NU)                                                                                   \
    case NU:                                                                                            \
        if (M <= 2) { if (two) NORMED(NU, 2, 2); else NORMED(NU, 1, 2); }                               \
        else if (two) NORMED(NU, 2, 8); else NORMED(NU, 1, 8);                                          \
        break;
    switch ((K + 255) / 256) {
        NORMED_CASE(1) NORMED_CASE(2) NORMED_CASE(3) NORMED_CASE(4) NORMED_CASE(5) NORMED_CASE(6) NORMED_CASE(7) NORMED_CASE(8)
    }
#undef NORMED_CASE
#undef NORMED
    MLLM_LAUNCH_CHECK();
    return 0;
}

// The tiles of a 32-bit product that runs on tiles (TileShape; for tests).
int mllm_gemm_f32_tile_shape(int M, int N, int K) { return tile_shape(M, N, K); }

int mllm_gemm_f32(const float* A, int lda, const float* W, int ldw, const float* bias, void* C, int ldc,
                  int M, int N, int K, int mode, hipStream_t stream) {
    if (M <= 0 || N <= 0) return 0;
    const bool quads = K % 4 == 0 && lda % 4 == 0 && ldw % 4 == 0 &&
                       ((reinterpret_cast<uintptr_t>(A) | reinterpret_cast<uintptr_t>(W)) & 15) == 0;
    if (quads && K > 0 && (M <= 8 || (M <= 16 && N < 16384))) {
        // (9 to 16 rows of a wide head: 73 us here, 55 on tiles at 50,257 columns.)
        // Workgroups start at a limited rate (a few hundred a microsecond over the chip): from 2,048 columns on
        // a workgroup takes eight instead of four, which also halves what is staged (sixteen lose again: at
        // 50,257 columns 54 us against 45).
        if (N >= 2048) {
            const dim3 rows_grid((N + 7) / 8);
            if (M <= 8) gemm_f32_rows_kernel<8, 8><<<rows_grid, 512, 0, stream>>>(A, W, bias, C, lda, ldw, ldc, M, N, K, mode);
            else gemm_f32_rows_kernel<16, 8><<<rows_grid, 512, 0, stream>>>(A, W, bias, C, lda, ldw, ldc, M, N, K, mode);
        } else {
            // (3,072 columns a pass take the LDS of a unit: while there is one workgroup a unit; 9 to 16 rows would take twice as much)
            const dim3 rows_grid((N + 3) / 4);
            if (M > 8) gemm_f32_rows_kernel<16, 4><<<rows_grid, 256, 0, stream>>>(A, W, bias, C, lda, ldw, ldc, M, N, K, mode);
            else if (K <= 1024) launch_f32_narrow<8, 2>(A, lda, W, ldw, bias, C, ldc, M, N, K, mode, stream);
            else if (N <= 1024) launch_f32_narrow<8, 6>(A, lda, W, ldw, bias, C, ldc, M, N, K, mode, stream);
            else launch_f32_narrow<8, 3>(A, lda, W, ldw, bias, C, ldc, M, N, K, mode, stream);
        }
        MLLM_LAUNCH_CHECK();
        return 0;
    }
    // Wide rows of an odd length leave the tiles an element at a time, which a short K does not hide: 130 x 50,257 x 64 35 us on tiles, 25 on
    // vector FMAs, 2,048 x 50,257 x 64 346 / 239; 192 x 32,000 x 128 31.4 / 29.9 (at 192 columns 35.6 / 40.4), 192 x 16,384 x 64 13.8 / 13.4.
    const bool odd_wide = M > 64 && ldc % 4 != 0 && N >= 16384 && K <= (N >= 32000 ? 128 : N >= 20000 ? 96 : 64);
    if (quads && K > 0 && !odd_wide) {
        switch (tile_shape(M, N, K)) {
            case T32_FOUR: launch_f32_tiles<2, 2, 1, 1, 4, 1, 3, 4>(A, lda, W, ldw, bias, C, ldc, M, N, K, mode, stream); break;
            case T32_TWO: launch_f32_tiles<2, 2, 1, 1, 2, 2, 3, 4>(A, lda, W, ldw, bias, C, ldc, M, N, K, mode, stream); break;
            case T32_ONE: launch_f32_tiles<2, 2, 1, 1, 1, 2, 3, 4>(A, lda, W, ldw, bias, C, ldc, M, N, K, mode, stream); break;
            case T64X32: launch_f32_tiles<2, 2, 2, 1, 1, 2, 3, 1>(A, lda, W, ldw, bias, C, ldc, M, N, K, mode, stream); break;
            case T128X64: launch_f32_tiles<4, 2, 2, 2, 1, 1, 3, 1>(A, lda, W, ldw, bias, C, ldc, M, N, K, mode, stream); break;
        }
        MLLM_LAUNCH_CHECK();
        return 0;
    }
    // any K, strides and alignment, and short K (see above)
    dim3 grid((N + F32_BN - 1) / F32_BN, (M + F32_BM - 1) / F32_BM);
    gemm_f32_kernel<<<grid, 256, 0, stream>>>(A, lda, W, ldw, bias, C, ldc, M, N, K, mode);
    MLLM_LAUNCH_CHECK();
    return 0;
}

}  // extern "C"
