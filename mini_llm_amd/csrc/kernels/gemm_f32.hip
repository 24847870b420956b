// True fp32 matrix product for the 32-bit path: C[M,N] = A[M,K] * W[N,K]^T (+ bias, epilogue).
// fp32 products summed in fp32, on the vector units or the fp32 matrix cores; no reduced-precision matrix mode is
// involved. Every output is accumulated over k in an order that its kernel and tile shape fix, so which other
// rows share the launch matters only through their number, which chooses between these. Any M, N, K.
//
// Same contract as the reference's bounds-safe kernel
// (/root/reference/src/kernels/gemm.cu:238-392: alpha*acc + beta*old + bias, optional GELU),
// with the weight held as [N,K] (k contiguous) instead of [K,N].
#include <algorithm>

#include "common.h"

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
gemm_f32_rows_kernel(const float* __restrict__ A, int lda, const float* __restrict__ W, int ldw,
                     const float* __restrict__ bias, void* __restrict__ C, int ldc, int M, int N, int K, int mode) {
    __shared__ __attribute__((aligned(16))) float a_s[ROWS][F32R_KC];
    const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid / 64), lane = tid % 64;
    const int n = blockIdx.x * WAVES + wave;
    const float* wrow = W + static_cast<size_t>(min(n, N - 1)) * ldw;       // a surplus wavefront repeats the last column
    constexpr int STAGED = (ROWS * (F32R_KC / 4) + 64 * WAVES - 1) / (64 * WAVES);   // 16-byte steps of a chunk a thread stages
    float acc[ROWS];
#pragma unroll
    for (int r = 0; r < ROWS; ++r) acc[r] = 0.f;
    // With a handful of wavefronts on a compute unit nothing hides a load's latency but the kernel itself:
    // the weights and the activations of the next chunk are asked for before the chunk in LDS is used.
    // A chunk is at most two 16-byte steps per lane (the second from a clamped address; its product is
    // left out where it is past the chunk).
    const int q0 = lane, q1 = lane + 64;
    float4 w0, w1, v[STAGED];
    auto fetch = [&](int kc0) {
        const int quads = min(F32R_KC, K - kc0) / 4;
        w0 = *reinterpret_cast<const float4*>(wrow + kc0 + 4 * min(q0, quads - 1));
        w1 = *reinterpret_cast<const float4*>(wrow + kc0 + 4 * min(q1, quads - 1));
#pragma unroll
        for (int u = 0; u < STAGED; ++u) {
            const int idx = tid + 64 * WAVES * u, r = idx / quads, q = idx % quads;
            v[u] = make_float4(0.f, 0.f, 0.f, 0.f);
            if (idx < ROWS * quads && r < M)
                v[u] = *reinterpret_cast<const float4*>(A + static_cast<size_t>(r) * lda + kc0 + 4 * q);
        }
    };
    fetch(0);
    for (int kc0 = 0; kc0 < K; kc0 += F32R_KC) {
        const int quads = min(F32R_KC, K - kc0) / 4;
        const float4 c0 = w0, c1 = w1;
        __syncthreads();          // the chunk before has been read
#pragma unroll
        for (int u = 0; u < STAGED; ++u) {
            const int idx = tid + 64 * WAVES * u, r = idx / quads, q = idx % quads;
            if (idx < ROWS * quads) *reinterpret_cast<float4*>(&a_s[r][4 * q]) = v[u];
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
// first. Bound by the chain launch, activations, weights, sums: 8 x 768 x 768 and 8 x 768 x 3,072 in a decode step 4.1 and 6.0
// us, together 17.1 with a column a wavefront.
// RAGGED: K is no multiple of 256, and what lies beyond it has to be left out (8 x 1,600 x 1,600 7.4 us, 7.2 if it were not).
template <int ROWS, int STEPS, bool RAGGED>
__global__ void __launch_bounds__(512)
gemm_f32_narrow_kernel(const float* __restrict__ A, int lda, const float* __restrict__ W, int ldw,
                       const float* __restrict__ bias, void* __restrict__ C, int ldc, int M, int N, int K, int mode) {
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
            const float4 a = *reinterpret_cast<const float4*>(A + static_cast<size_t>(min(r, M - 1)) * lda + min(k, K - 4));
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

template <int ROWS, int STEPS>
static void launch_f32_narrow(const float* A, int lda, const float* W, int ldw, const float* bias, void* C, int ldc, int M, int N, int K, int mode, hipStream_t stream) {
    const dim3 grid((N + 3) / 4);
    if (K % 256 != 0) gemm_f32_narrow_kernel<ROWS, STEPS, true><<<grid, 512, 0, stream>>>(A, lda, W, ldw, bias, C, ldc, M, N, K, mode);
    else gemm_f32_narrow_kernel<ROWS, STEPS, false><<<grid, 512, 0, stream>>>(A, lda, W, ldw, bias, C, ldc, M, N, K, mode);
}

// More than a few rows, on the fp32 matrix cores (v_mfma_f32_16x16x4_f32, 256 operations a clock and compute unit). Four
// wavefronts, two by two, of TM x TN tiles of 16 x 16 each share k tiles of 32 columns (a row's piece is one 128-byte line) in
// LDS, double buffered with one barrier a tile; the loads of the two tiles behind the next are in flight in registers. KG such
// groups take the 32-column parts of a KG times as wide k tile and add their sums in LDS: for few tiles, where the chain of
// k tiles (LDS write, barrier, read, products: 0.34 us) is what a workgroup waits for. A lane's 16-byte read holds the k
// columns of four matrix instructions (lane group l / 16 takes columns 4 (l / 16) to + 3 of 16, the same for both operands);
// rows are an odd number of 16-byte pieces apart (16 lanes on 16 different groups of banks). The weights are the
// instruction's first operand, so that a lane ends up with four neighbouring columns of one row. Sixteen columns are summed on
// their own before they join an output's sum, with tiles of 16 x 16 a wavefront 32 columns in eight sums: the error against 64 bits
// (2-norm over 2-norm, normal values) is 1.5e-7 at K = 768 and 2.0e-7 at 3,072, with eight sums and four groups 8.8e-8 and 1.2e-7,
// where one chain of FMAs had 5.0e-7 and 9.9e-7 and the kernel for few rows has 9.3e-8 and 1.4e-7. (Four sums of 16 columns, 9.6e-8
// and 1.5e-7, were a little less exact than that kernel, which took up to 64 rows before; up to K = 256 the two are alike.)
// Bound by the matrix cores where the tiles fill the chip evenly, else by the units that take one tile more or by that chain.
// 2,048 x 3,072 x 768: 91 us (106 TFLOP/s of the 155 a loop of these instructions reaches; a kernel of vector FMAs on 64 x 64
// tiles took 134); 2,048 x 768 x 3,072: 99 (209); 570 x 768 x 3,072: 40 (197); 64 x 768 x 3,072: 24 (the kernel for few
// rows: 59). Needs K and the row strides in multiples of 4 floats, 16-byte aligned operands.
#define F32T_BK 32
typedef float f32x4v __attribute__((ext_vector_type(4)));

template <int TM, int TN, int KG>
__global__ void __launch_bounds__(256 * KG)
gemm_f32_tiles_kernel(const float* __restrict__ A, int lda, const float* __restrict__ W, int ldw, const float* __restrict__ bias,
                      void* __restrict__ C, int ldc, int M, int N, int K, int mode, int tiles_m, int tiles_n, int down) {
    constexpr int BM = 32 * TM, BN = 32 * TN, ROWS = BM + BN, BK = F32T_BK * KG, STRIDE = BK + 4;
    constexpr int SUMS = TM * TN == 1 ? 4 : 1;      // an output's 16 columns in so many sums
    constexpr int THREADS = 256 * KG, PIECES = BK / 4, STEP = THREADS / PIECES, LOADS = ROWS / STEP;      // STEP: rows that all threads load at once
    static_assert(STEP == 32 && (KG == 1 || KG == 2 || KG == 4) && (KG - 1) * 4 * TM * TN * 64 * 4 <= 2 * ROWS * STRIDE, "the groups' sums fit the tiles' LDS");
    __shared__ __attribute__((aligned(16))) float tile_s[2][ROWS * STRIDE];      // rows of A, then rows of W
    const int tid = threadIdx.x, lane = tid % 64;
    const int kg = __builtin_amdgcn_readfirstlane(tid / 256), wave = __builtin_amdgcn_readfirstlane(tid / 64 % 4);
    // an XCD (workgroup id % 8) takes an even share of the tiles, neighbours in one direction: with `down` it walks down the
    // rows of A for a few columns of tiles, else along the rows of W for a few rows of tiles
    const int tiles = tiles_m * tiles_n, per = (tiles + 7) / 8, at = (blockIdx.x % 8) * per + blockIdx.x / 8;
    if (blockIdx.x / 8 >= per || at >= tiles) return;
    const int tm = down ? at % tiles_m : at / tiles_n, tn = down ? at / tiles_m : at % tiles_n;
    const int m0 = tm * BM, n0 = tn * BN;
    // a thread's 16-byte pieces of a tile: rows beyond the matrix read the last one and are never stored
    const float* src[LOADS];
    const int piece = 4 * (tid % PIECES), row0 = tid / PIECES;
#pragma unroll
    for (int i = 0; i < LOADS; ++i) {
        const int row = row0 + STEP * i;
        src[i] = (STEP * i < BM ? A + static_cast<size_t>(min(m0 + row, M - 1)) * lda : W + static_cast<size_t>(min(n0 + row - BM, N - 1)) * ldw) + piece;
    }
    float4 regs[2][LOADS];
    auto fetch = [&](int set, int k0) {          // (columns beyond K: the row's last ones, zeroed when they are staged)
        const int k = min(k0, K - 4 - piece);
#pragma unroll
        for (int i = 0; i < LOADS; ++i) regs[set][i] = *reinterpret_cast<const float4*>(src[i] + k);
    };
    auto stage = [&](int set, int buf, int k0) {
        const bool ok = k0 + piece < K;
#pragma unroll
        for (int i = 0; i < LOADS; ++i)
            *reinterpret_cast<float4*>(&tile_s[buf][(row0 + STEP * i) * STRIDE + piece]) = ok ? regs[set][i] : make_float4(0.f, 0.f, 0.f, 0.f);
    };
    f32x4v acc[TM][TN];
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j) acc[i][j] = f32x4v{0.f, 0.f, 0.f, 0.f};
    const int wm = wave / 2, wn = wave % 2, row16 = lane % 16, quad = lane / 16;
    const int a_off = (wm * TM * 16 + row16) * STRIDE + F32T_BK * kg + 4 * quad, w_off = (BM + wn * TN * 16 + row16) * STRIDE + F32T_BK * kg + 4 * quad;
    // TM x TN of 1: the 32 columns in eight sums of four that are added pairwise before they join; otherwise 16 columns in one sum each
    auto multiply = [&](int buf) {
        constexpr int KS = F32T_BK / 16;
        f32x4v sum[SUMS == 4 ? KS : 1][SUMS][TM][TN];
#pragma unroll
        for (int ks = 0; ks < KS; ++ks) {
            const int at = SUMS == 4 ? ks : 0;
            f32x4v fa[TM], fw[TN];
#pragma unroll
            for (int i = 0; i < TM; ++i) fa[i] = *reinterpret_cast<const f32x4v*>(&tile_s[buf][a_off + i * 16 * STRIDE + ks * 16]);
#pragma unroll
            for (int j = 0; j < TN; ++j) fw[j] = *reinterpret_cast<const f32x4v*>(&tile_s[buf][w_off + j * 16 * STRIDE + ks * 16]);
#pragma unroll
            for (int e = 0; e < 4; ++e)
#pragma unroll
                for (int i = 0; i < TM; ++i)
#pragma unroll
                    for (int j = 0; j < TN; ++j) {
                        f32x4v& to = sum[at][e % SUMS][i][j];
                        to = __builtin_amdgcn_mfma_f32_16x16x4f32(fw[j][e], fa[i][e], e < SUMS ? f32x4v{0.f, 0.f, 0.f, 0.f} : to, 0, 0, 0);
                    }
            if constexpr (SUMS == 1) {
#pragma unroll
                for (int i = 0; i < TM; ++i)
#pragma unroll
                    for (int j = 0; j < TN; ++j) acc[i][j] += sum[0][0][i][j];
            }
        }
        if constexpr (SUMS == 4) {
            static_assert(KS == 2, "two times four sums");
            auto four = [&](int ks) { return (sum[ks][0][0][0] + sum[ks][1][0][0]) + (sum[ks][2][0][0] + sum[ks][3][0][0]); };
            acc[0][0] += four(0) + four(1);
        }
    };
    const int nk = (K + BK - 1) / BK;
    // tile t multiplies from buffer t % 2 while tile t + 1 is staged into the other one, whose readers (tile t - 1) passed the
    // barrier before, and the loads of tile t + 3 go out into the registers that are free then (past the last tile: its own again)
    fetch(0, 0);
    fetch(1, min(1, nk - 1) * BK);
    stage(0, 0, 0);
    fetch(0, min(2, nk - 1) * BK);
    lds_barrier();
    for (int t = 0; t < nk; t += 2) {
        stage(1, 1, (t + 1) * BK);
        fetch(1, min(t + 3, nk - 1) * BK);
        multiply(0);
        lds_barrier();
        if (t + 1 >= nk) break;
        stage(0, 0, (t + 2) * BK);
        fetch(0, min(t + 4, nk - 1) * BK);
        multiply(1);
        lds_barrier();
    }
    if constexpr (KG > 1) {          // the other groups leave their sums in LDS and go; group 0 adds them in their order
        f32x4v* sums = reinterpret_cast<f32x4v*>(&tile_s[0][0]);
        if (kg > 0) {
#pragma unroll
            for (int i = 0; i < TM; ++i)
#pragma unroll
                for (int j = 0; j < TN; ++j) sums[(((kg - 1) * 4 + wave) * TM * TN + i * TN + j) * 64 + lane] = acc[i][j];
        }
        lds_barrier();
        if (kg > 0) return;
#pragma unroll
        for (int i = 0; i < TM; ++i)
#pragma unroll
            for (int j = 0; j < TN; ++j) {
                auto other = [&](int g) { return sums[((g * 4 + wave) * TM * TN + i * TN + j) * 64 + lane]; };
                if constexpr (KG == 4) acc[i][j] = (acc[i][j] + other(0)) + (other(1) + other(2));
                else acc[i][j] += other(0);
            }
    }
    // lane l holds columns 4 (l / 16) to + 3 of row l % 16 of every 16 x 16 tile
    const bool vec = ldc % 4 == 0 && (reinterpret_cast<uintptr_t>(C) & 15) == 0 && (bias == nullptr || (reinterpret_cast<uintptr_t>(bias) & 15) == 0);
#pragma unroll
    for (int i = 0; i < TM; ++i) {
        const int m = m0 + (wm * TM + i) * 16 + row16;
        if (m >= M) continue;
#pragma unroll
        for (int j = 0; j < TN; ++j) {
            const int n = n0 + (wn * TN + j) * 16 + 4 * quad;
            float* out = static_cast<float*>(C) + static_cast<size_t>(m) * ldc + n;
            if (vec && n + 4 <= N) {
                float v[4] = {acc[i][j][0], acc[i][j][1], acc[i][j][2], acc[i][j][3]}, o[4] = {0.f, 0.f, 0.f, 0.f};
                if (bias != nullptr) {
                    const float4 b = *reinterpret_cast<const float4*>(bias + n);
                    v[0] += b.x; v[1] += b.y; v[2] += b.z; v[3] += b.w;
                }
                if (mode == EPI_ADD_RESIDUAL) {
                    const float4 b = *reinterpret_cast<const float4*>(out);
                    o[0] = b.x; o[1] = b.y; o[2] = b.z; o[3] = b.w;
                }
#pragma unroll
                for (int e = 0; e < 4; ++e)
                    o[e] += mode == EPI_GELU_TANH ? gelu_tanh_precise(v[e]) : mode == EPI_GELU_ERF ? gelu_erf(v[e]) : mode == EPI_RELU2 ? relu2(v[e]) : v[e];
                *reinterpret_cast<float4*>(out) = make_float4(o[0], o[1], o[2], o[3]);
            } else {
                for (int e = 0; e < 4 && n + e < N; ++e)
                    epilogue<float>(mode, acc[i][j][e], bias ? bias[n + e] : 0.f, C, static_cast<size_t>(m) * ldc + n + e);
            }
        }
    }
}

template <int TM, int TN, int KG>
static void launch_f32_tiles(const float* A, int lda, const float* W, int ldw, const float* bias, void* C, int ldc, int M, int N, int K, int mode,
                             hipStream_t stream) {
    const int tiles_m = (M + 32 * TM - 1) / (32 * TM), tiles_n = (N + 32 * TN - 1) / (32 * TN);
    gemm_f32_tiles_kernel<TM, TN, KG><<<(tiles_m * tiles_n + 7) / 8 * 8, 256 * KG, 0, stream>>>(A, lda, W, ldw, bias, C, ldc, M, N, K, mode, tiles_m, tiles_n,
                                                                                             M > N ? 0 : 1);
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
            if (M <= 8) gemm_f32_rows_kernel<8, 8><<<rows_grid, 512, 0, stream>>>(A, lda, W, ldw, bias, C, ldc, M, N, K, mode);
            else gemm_f32_rows_kernel<16, 8><<<rows_grid, 512, 0, stream>>>(A, lda, W, ldw, bias, C, ldc, M, N, K, mode);
        } else {
            // (3,072 columns a pass take the LDS of a unit: while there is one workgroup a unit; 9 to 16 rows would take twice as much)
            const dim3 rows_grid((N + 3) / 4);
            if (M > 8) gemm_f32_rows_kernel<16, 4><<<rows_grid, 256, 0, stream>>>(A, lda, W, ldw, bias, C, ldc, M, N, K, mode);
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
        // Tiles of 32 x 32 shared by four groups up to 64 rows (whose sums are as exact as the kernel's for few rows) and while
        // there are at most two a compute unit (570 x 768 x 3,072: 40 us, with two groups 43, with tiles of 64 x 32 44).
        // Otherwise the shape whose fullest compute unit does least: its tiles times their size times what 32 x 32 outputs
        // take there at K = 768 (in tenths of a microsecond, measured at 2,048 rows). With two groups a sixth of that is there at
        // any K, which shows up to 96 columns (130 x 50,304 x 96: 40 us with 32 x 32, 29 with 64 x 64; 65 x 50,304 x 256: 40.1, 41.5). Large tiles need several workgroups a unit
        // to hide their barriers: 2,048 x 768 x 768 32 us with 64 x 32, 35 with 64 x 64 (384 tiles) and 64 x 96 (256).
        const auto tiles = [&](int tm, int tn) { return static_cast<long>((M + 32 * tm - 1) / (32 * tm)) * ((N + 32 * tn - 1) / (32 * tn)); };
        const auto cost = [&](int tm, int tn, int groups, long from, int each) {
            const long n = tiles(tm, tn), k = K <= 96 ? K : 768;
            return n < from ? (1L << 60) : ((n + 7) / 8 + 31) / 32 * tm * tn * each * (groups == 2 ? 5 * k + 768 : 6 * k);
        };
        if (M <= 64 || tiles(1, 1) <= 512) {
            launch_f32_tiles<1, 1, 4>(A, lda, W, ldw, bias, C, ldc, M, N, K, mode, stream);
        } else {
            const long c11 = cost(1, 1, 2, 0, 44), c21 = cost(2, 1, 2, 256, 40), c22 = cost(2, 2, 1, 512, 36), c23 = cost(2, 3, 1, 512, 37);
            const long least = std::min(std::min(c11, c21), std::min(c22, c23));
            if (least == c22) launch_f32_tiles<2, 2, 1>(A, lda, W, ldw, bias, C, ldc, M, N, K, mode, stream);
            else if (least == c23) launch_f32_tiles<2, 3, 1>(A, lda, W, ldw, bias, C, ldc, M, N, K, mode, stream);
            else if (least == c21) launch_f32_tiles<2, 1, 2>(A, lda, W, ldw, bias, C, ldc, M, N, K, mode, stream);
            else launch_f32_tiles<1, 1, 2>(A, lda, W, ldw, bias, C, ldc, M, N, K, mode, stream);
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
