// State-space mixer kernels for gfx950: the short causal convolution with its carried inputs, and the
// selective scan (Mamba-2 form: one decay per head and token) over a step's portions, the state carried
// in a per-request slot. Everything here is fp32.
//
// A request's slot holds [taps - 1][channels] convolution inputs (oldest first), then the scan's state
// laid out [head][n][p] (p contiguous).
#include <algorithm>

#include "common.h"

namespace {

__device__ __forceinline__ float silu_precise(float v) { return v / (1.f + expf(-v)); }
// log(1 + exp(v)) without overflow, no clamp
__device__ __forceinline__ float softplus_precise(float v) { return fmaxf(v, 0.f) + log1pf(expf(-fabsf(v))); }

// out[t, ch] = silu(bias[ch] + sum_j w[ch, j] * in(t - (taps - 1 - j), ch)): inputs before the portion come
// from the slot's carried rows (zeros for a fresh request: the slot was cleared). One thread per (t, ch).
__global__ void conv_silu_kernel(const float* __restrict__ proj, int ld, int col0, int C, const float* __restrict__ w,
                                 const float* __restrict__ bias, int taps, const int* __restrict__ token_seq,
                                 const int* __restrict__ cu_q, const int* __restrict__ state_slots,
                                 float* __restrict__ state, size_t slot_floats, float* __restrict__ out, int ldo,
                                 long long total, int carry) {
    const long long i = static_cast<long long>(blockIdx.x) * blockDim.x + threadIdx.x;
    if (i >= total) return;
    const int t = static_cast<int>(i / C), ch = static_cast<int>(i % C);
    const int b = token_seq[t], slot = state_slots[b];
    if (slot < 0) return;
    const int first = cu_q[b], k = t - first;
    float* carried = state + static_cast<size_t>(slot) * slot_floats;
    float acc = bias[ch];
    for (int j = 0; j < taps; ++j) {
        const int idx = k - (taps - 1 - j);
        const float v = idx >= 0 ? proj[static_cast<size_t>(first + idx) * ld + col0 + ch]
                                 : carried[static_cast<size_t>(taps - 1 + idx) * C + ch];
        acc += w[static_cast<size_t>(ch) * taps + j] * v;
        // `carry` (every portion of the step is a single token, so this thread is the channel's only reader): the
        // carried rows move up by one behind the read, and the token's input becomes the newest
        if (carry && j >= 1) carried[static_cast<size_t>(j - 1) * C + ch] = v;
    }
    out[static_cast<size_t>(t) * ldo + ch] = silu_precise(acc);
}

// The same four channels a thread, all loads of a token asked for together, as in conv_residual_vec_kernel below (which see):
// 2,048 tokens x 1,792 channels 14.3 us, one channel a thread 26.
template <int TAPS>
__global__ void conv_silu_vec_kernel(const float* __restrict__ in, int ld, int C, const float* __restrict__ w, const float* __restrict__ bias,
                                     const int* __restrict__ token_seq, const int* __restrict__ cu_q, const int* __restrict__ state_slots,
                                     const float* __restrict__ state, size_t slot_floats, float* __restrict__ out, int ldo, long long total4) {
    const long long i = static_cast<long long>(blockIdx.x) * blockDim.x + threadIdx.x;
    if (i >= total4) return;
    const int C4 = C / 4;
    const int t = static_cast<int>(i / C4), ch = static_cast<int>(i % C4) * 4;
    const int b = token_seq[t], slot = state_slots[b];
    if (slot < 0) return;
    const int first = cu_q[b], k = t - first;
    const float* carried = state + static_cast<size_t>(slot) * slot_floats;
    float4 wf[TAPS], v[TAPS];             // wf: the four channels' taps one behind the other (4 * TAPS floats)
    const float4 b4 = *reinterpret_cast<const float4*>(bias + ch);
#pragma unroll
    for (int j = 0; j < TAPS; ++j) wf[j] = *reinterpret_cast<const float4*>(w + static_cast<size_t>(ch) * TAPS + 4 * j);
    if (k >= TAPS - 1) {
#pragma unroll
        for (int j = 0; j < TAPS; ++j) v[j] = *reinterpret_cast<const float4*>(in + static_cast<size_t>(t - (TAPS - 1 - j)) * ld + ch);
    } else {
#pragma unroll
        for (int j = 0; j < TAPS; ++j) {
            const int idx = k - (TAPS - 1 - j);
            v[j] = idx >= 0 ? *reinterpret_cast<const float4*>(in + static_cast<size_t>(first + idx) * ld + ch)
                            : *reinterpret_cast<const float4*>(carried + static_cast<size_t>(TAPS - 1 + idx) * C + ch);
        }
    }
    float wv[4 * TAPS];
#pragma unroll
    for (int j = 0; j < TAPS; ++j) { wv[4 * j] = wf[j].x; wv[4 * j + 1] = wf[j].y; wv[4 * j + 2] = wf[j].z; wv[4 * j + 3] = wf[j].w; }
    float acc[4] = {b4.x, b4.y, b4.z, b4.w};
#pragma unroll
    for (int j = 0; j < TAPS; ++j) {
        acc[0] += wv[0 * TAPS + j] * v[j].x;
        acc[1] += wv[1 * TAPS + j] * v[j].y;
        acc[2] += wv[2 * TAPS + j] * v[j].z;
        acc[3] += wv[3 * TAPS + j] * v[j].w;
    }
    *reinterpret_cast<float4*>(out + static_cast<size_t>(t) * ldo + ch) =
        make_float4(silu_precise(acc[0]), silu_precise(acc[1]), silu_precise(acc[2]), silu_precise(acc[3]));
}

// A step of one token a sequence (token t is sequence t: no slot belongs to two tokens), a workgroup per token and 64 channel quads: the token's
// own row, the taps and the slot are asked for at once, from arguments that arrive with the wavefront and without a division; only the
// carried rows, which move up by one here, wait for the slot. A chain of latencies: 8 tokens x 1,792 channels 3.5 > 2.8 us.
template <int TAPS>
__global__ void __launch_bounds__(64)
conv_silu_single_kernel(const float* __restrict__ in, int ld, int C, const float* __restrict__ w, const float* __restrict__ bias,
                        const int* __restrict__ state_slots, float* __restrict__ state, size_t slot_floats, float* __restrict__ out, int ldo) {
    const int t = blockIdx.x, ch = (blockIdx.y * 64 + threadIdx.x) * 4;
    if (ch >= C) return;
    float4 wf[TAPS], v[TAPS];
    const float4 own = *reinterpret_cast<const float4*>(in + static_cast<size_t>(t) * ld + ch), b4 = *reinterpret_cast<const float4*>(bias + ch);
#pragma unroll
    for (int j = 0; j < TAPS; ++j) wf[j] = *reinterpret_cast<const float4*>(w + static_cast<size_t>(ch) * TAPS + 4 * j);
    const int slot = state_slots[t];
    if (slot < 0) return;
    float* carried = state + static_cast<size_t>(slot) * slot_floats;
#pragma unroll
    for (int j = 0; j < TAPS - 1; ++j) v[j] = *reinterpret_cast<const float4*>(carried + static_cast<size_t>(j) * C + ch);
    v[TAPS - 1] = own;
    float wv[4 * TAPS];
#pragma unroll
    for (int j = 0; j < TAPS; ++j) { wv[4 * j] = wf[j].x; wv[4 * j + 1] = wf[j].y; wv[4 * j + 2] = wf[j].z; wv[4 * j + 3] = wf[j].w; }
    float acc[4] = {b4.x, b4.y, b4.z, b4.w};
#pragma unroll
    for (int j = 0; j < TAPS; ++j) {
        acc[0] += wv[0 * TAPS + j] * v[j].x;
        acc[1] += wv[1 * TAPS + j] * v[j].y;
        acc[2] += wv[2 * TAPS + j] * v[j].z;
        acc[3] += wv[3 * TAPS + j] * v[j].w;
    }
#pragma unroll
    for (int j = 1; j < TAPS; ++j) *reinterpret_cast<float4*>(carried + static_cast<size_t>(j - 1) * C + ch) = v[j];
    *reinterpret_cast<float4*>(out + static_cast<size_t>(t) * ldo + ch) =
        make_float4(silu_precise(acc[0]), silu_precise(acc[1]), silu_precise(acc[2]), silu_precise(acc[3]));
}

// The same for many tokens, ROWS neighbours of them a thread: their inputs are asked for together, before the tokens' sequence is known (from
// rows of the step, whosever they are), and used if the tokens have one sequence and TAPS - 1 tokens of its portion in front of them; the
// taps are loaded once. Every token's own kernel above is bound by its chain of loads (sequence, slot, rows) and reads every row TAPS
// times. Same results. 2,048 tokens x 1,792 channels 13.3 > 10.1 us, 8,000 44 > 28.6 (eight rows a thread: 12.3 and 27.3).
template <int TAPS, int ROWS>
__global__ void __launch_bounds__(256)
conv_silu_rows_kernel(const float* __restrict__ in, int ld, int C, const float* __restrict__ w, const float* __restrict__ bias,
                      const int* __restrict__ token_seq, const int* __restrict__ cu_q, const int* __restrict__ state_slots,
                      const float* __restrict__ state, size_t slot_floats, float* __restrict__ out, int ldo, int T) {
    const int C4 = C / 4;
    const long long i = static_cast<long long>(blockIdx.x) * 256 + threadIdx.x;
    const int t0 = static_cast<int>(i / C4) * ROWS, ch = static_cast<int>(i % C4) * 4;
    if (t0 >= T) return;
    const int t1 = min(t0 + ROWS, T) - 1, b = token_seq[t0], b1 = token_seq[t1];
    float4 wf[TAPS], v[ROWS + TAPS - 1];
    const float4 b4 = *reinterpret_cast<const float4*>(bias + ch);
#pragma unroll
    for (int j = 0; j < TAPS; ++j) wf[j] = *reinterpret_cast<const float4*>(w + static_cast<size_t>(ch) * TAPS + 4 * j);
#pragma unroll
    for (int j = 0; j < ROWS + TAPS - 1; ++j) v[j] = *reinterpret_cast<const float4*>(in + static_cast<size_t>(min(max(t0 - (TAPS - 1) + j, 0), T - 1)) * ld + ch);
    float wv[4 * TAPS];
#pragma unroll
    for (int j = 0; j < TAPS; ++j) { wv[4 * j] = wf[j].x; wv[4 * j + 1] = wf[j].y; wv[4 * j + 2] = wf[j].z; wv[4 * j + 3] = wf[j].w; }
    auto put = [&](int t, const float4 (&x)[TAPS]) {
        float acc[4] = {b4.x, b4.y, b4.z, b4.w};
#pragma unroll
        for (int j = 0; j < TAPS; ++j) {
            acc[0] += wv[0 * TAPS + j] * x[j].x;
            acc[1] += wv[1 * TAPS + j] * x[j].y;
            acc[2] += wv[2 * TAPS + j] * x[j].z;
            acc[3] += wv[3 * TAPS + j] * x[j].w;
        }
        *reinterpret_cast<float4*>(out + static_cast<size_t>(t) * ldo + ch) =
            make_float4(silu_precise(acc[0]), silu_precise(acc[1]), silu_precise(acc[2]), silu_precise(acc[3]));
    };
    if (b == b1 && t0 - cu_q[b] >= TAPS - 1 && state_slots[b] >= 0) {
#pragma unroll
        for (int r = 0; r < ROWS; ++r) {
            if (t0 + r > t1) break;
            float4 x[TAPS];
#pragma unroll
            for (int j = 0; j < TAPS; ++j) x[j] = v[r + j];
            put(t0 + r, x);
        }
        return;
    }
    for (int t = t0; t <= t1; ++t) {         // the first tokens of a portion, or the end of one and the begin of another
        const int bt = token_seq[t], slot = state_slots[bt];
        if (slot < 0) continue;
        const int first = cu_q[bt], k = t - first;
        const float* carried = state + static_cast<size_t>(slot) * slot_floats;
        float4 x[TAPS];
#pragma unroll
        for (int j = 0; j < TAPS; ++j) {
            const int idx = k - (TAPS - 1 - j);
            x[j] = idx >= 0 ? *reinterpret_cast<const float4*>(in + static_cast<size_t>(first + idx) * ld + ch)
                            : *reinterpret_cast<const float4*>(carried + static_cast<size_t>(TAPS - 1 + idx) * C + ch);
        }
        put(t, x);
    }
}

// out[t, ch] = in[t, ch] + sum_j w[ch, j] * in(t - (taps - 1 - j), ch): the convolution added onto its own input,
// no bias and no activation, the result in the activation dtype. Carried rows as above. residual == 0: the
// convolution alone, its input not added.
template <typename OutT>
__global__ void conv_residual_kernel(const float* __restrict__ in, int ld, int C, const float* __restrict__ w, int taps,
                                     const int* __restrict__ token_seq, const int* __restrict__ cu_q,
                                     const int* __restrict__ state_slots, float* __restrict__ state, size_t slot_floats,
                                     OutT* __restrict__ out, int ldo, long long total, int carry, int residual) {
    const long long i = static_cast<long long>(blockIdx.x) * blockDim.x + threadIdx.x;
    if (i >= total) return;
    const int t = static_cast<int>(i / C), ch = static_cast<int>(i % C);
    const int b = token_seq[t], slot = state_slots[b];
    if (slot < 0) return;
    const int first = cu_q[b], k = t - first;
    float* carried = state + static_cast<size_t>(slot) * slot_floats;
    float acc = 0.f, own = 0.f;
    for (int j = 0; j < taps; ++j) {
        const int idx = k - (taps - 1 - j);
        const float v = idx >= 0 ? in[static_cast<size_t>(first + idx) * ld + ch]
                                 : carried[static_cast<size_t>(taps - 1 + idx) * C + ch];
        acc += w[static_cast<size_t>(ch) * taps + j] * v;
        own = v;
        if (carry && j >= 1) carried[static_cast<size_t>(j - 1) * C + ch] = v;
    }
    out[static_cast<size_t>(t) * ldo + ch] = from_float<OutT>(residual ? own + acc : acc);
}

// The same four channels a thread (16-byte loads; the rows' widths and the places are multiples of four floats). A
// token with taps - 1 tokens of its own portion in front of it reads them all from `in`, without conditions, so its
// loads are in flight together; the first tokens of a portion read the slot's carried rows where the portion has none.
// A wavefront holds one token's channels (or the border of two tokens), so the two ways seldom meet in one.
__device__ __forceinline__ void store4(float* p, const float (&v)[4]) { *reinterpret_cast<float4*>(p) = make_float4(v[0], v[1], v[2], v[3]); }
__device__ __forceinline__ void store4(bf16_t* p, const float (&v)[4]) {
    *reinterpret_cast<uint2*>(p) = make_uint2(pack_bf16x2(v[0], v[1]), pack_bf16x2(v[2], v[3]));
}
template <typename OutT, int TAPS>
__global__ void conv_residual_vec_kernel(const float* __restrict__ in, int ld, int C, const float* __restrict__ w,
                                         const int* __restrict__ token_seq, const int* __restrict__ cu_q,
                                         const int* __restrict__ state_slots, float* __restrict__ state, size_t slot_floats,
                                         OutT* __restrict__ out, int ldo, long long total4, int carry, int residual) {
    const long long i = static_cast<long long>(blockIdx.x) * blockDim.x + threadIdx.x;
    if (i >= total4) return;
    const int C4 = C / 4;
    const int t = static_cast<int>(i / C4), ch = static_cast<int>(i % C4) * 4;
    const int b = token_seq[t], slot = state_slots[b];
    if (slot < 0) return;
    const int first = cu_q[b], k = t - first;
    float* carried = state + static_cast<size_t>(slot) * slot_floats;
    float4 wf[TAPS], v[TAPS];             // wf: the four channels' taps one behind the other (4 * TAPS floats)
#pragma unroll
    for (int j = 0; j < TAPS; ++j) wf[j] = *reinterpret_cast<const float4*>(w + static_cast<size_t>(ch) * TAPS + 4 * j);
    if (k >= TAPS - 1) {
#pragma unroll
        for (int j = 0; j < TAPS; ++j) v[j] = *reinterpret_cast<const float4*>(in + static_cast<size_t>(t - (TAPS - 1 - j)) * ld + ch);
    } else {
#pragma unroll
        for (int j = 0; j < TAPS; ++j) {
            const int idx = k - (TAPS - 1 - j);
            v[j] = idx >= 0 ? *reinterpret_cast<const float4*>(in + static_cast<size_t>(first + idx) * ld + ch)
                            : *reinterpret_cast<const float4*>(carried + static_cast<size_t>(TAPS - 1 + idx) * C + ch);
        }
    }
    float wv[4 * TAPS];
#pragma unroll
    for (int j = 0; j < TAPS; ++j) { wv[4 * j] = wf[j].x; wv[4 * j + 1] = wf[j].y; wv[4 * j + 2] = wf[j].z; wv[4 * j + 3] = wf[j].w; }
    float r[4] = {v[TAPS - 1].x, v[TAPS - 1].y, v[TAPS - 1].z, v[TAPS - 1].w};
    if (!residual) r[0] = r[1] = r[2] = r[3] = 0.f;
    float acc[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int j = 0; j < TAPS; ++j) {
        acc[0] += wv[0 * TAPS + j] * v[j].x;
        acc[1] += wv[1 * TAPS + j] * v[j].y;
        acc[2] += wv[2 * TAPS + j] * v[j].z;
        acc[3] += wv[3 * TAPS + j] * v[j].w;
    }
    if (carry) {
#pragma unroll
        for (int j = 1; j < TAPS; ++j) *reinterpret_cast<float4*>(carried + static_cast<size_t>(j - 1) * C + ch) = v[j];
    }
#pragma unroll
    for (int q = 0; q < 4; ++q) r[q] += acc[q];
    store4(out + static_cast<size_t>(t) * ldo + ch, r);
}

// A step in which every sequence brings one token: h = x / sqrt(mean(x^2) + eps) * wn and out = h + conv(h) in one
// kernel, one workgroup per token. The earlier inputs of the convolution are the slot's carried rows, which move up
// by one behind the read; h becomes the newest.
// NB wavefronts, each with a block of 512 columns: its part of the row stays in registers between the statistics (the
// wavefronts' sums meet in LDS and are added in the order of the blocks) and the convolution. All loads of a block
// are issued together, without conditions, from clamped (always valid) places, and masked where they are used (a
// load under a condition, or in a loop of unknown length, is waited for before the next is asked for); TAPS is a
// constant for that reason.
// MODE 0: as above. MODE 1, a norm BEHIND a sub-layer and the next sub-layer's convolution: the stream's row becomes
// x + y / sqrt(mean(y^2) + eps) * wn (y: the sub-layer's result; x is written back), and h is that row. MODE 2: no norm,
// h = x.
template <typename OutT, int TAPS, int NB, int MODE>
__global__ void __launch_bounds__(64 * NB)
rmsnorm_conv_single_kernel(float* x, int ldx, const float* __restrict__ y, int ldy, const float* __restrict__ wn, float eps, int C,
                           const float* __restrict__ wc, const int* __restrict__ state_slots, float* __restrict__ state,
                           size_t slot_floats, OutT* __restrict__ out, int ldo, int write) {
    __shared__ float part[NB];
    const int b = __builtin_amdgcn_readfirstlane(threadIdx.x / MLLM_WAVE), lane = threadIdx.x % MLLM_WAVE;
    const int t = blockIdx.x;
    const int slot = state_slots[t];
    if (slot < 0) return;                      // (the whole workgroup: one token)
    float* xr = x + static_cast<size_t>(t) * ldx;
    int idx[8];
#pragma unroll
    for (int u = 0; u < 8; ++u) idx[u] = min(512 * b + lane + 64 * u, C - 1);
    float xv[8], yv[8], g[8], w[TAPS][8], v[TAPS > 1 ? TAPS - 1 : 1][8];
#pragma unroll
    for (int u = 0; u < 8; ++u) xv[u] = xr[idx[u]];
    if (MODE == 1) {
        const float* yr = y + static_cast<size_t>(t) * ldy;
#pragma unroll
        for (int u = 0; u < 8; ++u) yv[u] = yr[idx[u]];
    }
    const float* carried = state + static_cast<size_t>(slot) * slot_floats;
#pragma unroll
    for (int u = 0; u < 8; ++u) g[u] = MODE == 2 ? 1.f : wn[idx[u]];
#pragma unroll
    for (int j = 0; j < TAPS; ++j)
#pragma unroll
        for (int u = 0; u < 8; ++u) w[j][u] = wc[static_cast<size_t>(idx[u]) * TAPS + j];
#pragma unroll
    for (int j = 0; j + 1 < TAPS; ++j)
#pragma unroll
        for (int u = 0; u < 8; ++u) v[j][u] = carried[static_cast<size_t>(j) * C + idx[u]];
    float inv = 1.f;
    if (MODE != 2) {
        float ss = 0.f;
#pragma unroll
        for (int u = 0; u < 8; ++u) {
            const float z = MODE == 1 ? yv[u] : xv[u];
            ss += (512 * b + lane + 64 * u < C) ? z * z : 0.f;
        }
        ss = wave_sum(ss);
        if (NB > 1) {
            if (lane == 0) part[b] = ss;
            __syncthreads();
            ss = 0.f;
#pragma unroll
            for (int k = 0; k < NB; ++k) ss += part[k];
        }
        inv = 1.0f / sqrtf(ss / static_cast<float>(C) + eps);
    }
    float* carried_w = state + static_cast<size_t>(slot) * slot_floats;
#pragma unroll
    for (int u = 0; u < 8; ++u) {
        const float h = MODE == 0 ? xv[u] * inv * g[u] : MODE == 1 ? xv[u] + yv[u] * inv * g[u] : xv[u];
        float acc = w[TAPS - 1][u] * h;
#pragma unroll
        for (int j = 0; j + 1 < TAPS; ++j) acc += w[j][u] * v[j][u];
        if (512 * b + lane + 64 * u < C) {
            if (MODE == 1) xr[idx[u]] = h;
            if (write) {
#pragma unroll
                for (int j = 1; j + 1 < TAPS; ++j) carried_w[static_cast<size_t>(j - 1) * C + idx[u]] = v[j][u];
                if (TAPS > 1) carried_w[static_cast<size_t>(TAPS - 2) * C + idx[u]] = h;
            }
            out[static_cast<size_t>(t) * ldo + idx[u]] = from_float<OutT>(h + acc);
        }
    }
}

// The slot's carried rows after the portion: its last taps - 1 inputs, older ones shifted out; a portion
// shorter than that keeps the newest of the old rows. One thread per (sequence, channel); taps - 1 <= 15.
__global__ void conv_carry_kernel(const float* __restrict__ proj, int ld, int col0, int C, int taps,
                                  const int* __restrict__ cu_q, const int* __restrict__ state_slots,
                                  float* __restrict__ state, size_t slot_floats, int B) {
    const long long i = static_cast<long long>(blockIdx.x) * blockDim.x + threadIdx.x;
    if (i >= static_cast<long long>(B) * C) return;
    const int b = static_cast<int>(i / C), ch = static_cast<int>(i % C);
    const int slot = state_slots[b];
    if (slot < 0) return;
    const int first = cu_q[b], n = cu_q[b + 1] - first, keep = taps - 1;
    float* carried = state + static_cast<size_t>(slot) * slot_floats;
    float fresh[15];
#pragma unroll
    for (int r = 0; r < 15; ++r) {
        if (r < keep) {
            const int idx = n - keep + r;
            fresh[r] = idx >= 0 ? proj[static_cast<size_t>(first + idx) * ld + col0 + ch]
                                : carried[static_cast<size_t>(r + n) * C + ch];
        }
    }
#pragma unroll
    for (int r = 0; r < 15; ++r)
        if (r < keep) carried[static_cast<size_t>(r) * C + ch] = fresh[r];
}

// The scan. For head h (group g = h / (H / G)) and token t, in order:
//   dt = softplus(raw_dt[t, h] + dt_bias[h]);  a = exp(-exp(A_log[h]) dt)
//   S[n, p] = a S[n, p] + dt B[t, g, n] x[t, h, p];   y[t, h, p] = sum_n S[n, p] C[t, g, n] + D[h] x[t, h, p]
// One wavefront per (chunk of a sequence's portion, head, 64 values of p, slice of NS values of n): a lane owns
// one p and keeps its NS state values in registers, so B and C of the slice are the same for the whole wavefront
// (they arrive as scalars) and x is one coalesced load. The sum over n is split over the slices: slice s leaves its
// share in y + s * part_stride, and the reader (the gated norm) adds the shares in the order of s. The state in a
// slot is laid out [head][n][p] (p contiguous). xbc rows: [x: H*P | B: G*N | C: G*N].
//
// A portion longer than `chunk` tokens is cut into chunks that are scanned side by side: the first starts
// from the slot's state, the others from zero, and each leaves its last state in `chunk_state`
// ([chunk][H][N][P]) and, per token, the logarithm of the decay accumulated since its chunk began in `cumlog`
// ([T, H]). ssm_chunk_join_kernel then adds what the earlier chunks contribute. A portion of one chunk
// (decoding) is finished here and its state goes straight back to the slot.
struct ChunkOf {
    int b, k, n_chunks, first_chunk;      // sequence, chunk within it, chunks of the sequence, where its chunks' states start
                                          // (only portions of several chunks keep states: at most 2 T / chunk of them)
};
__device__ __forceinline__ ChunkOf chunk_of(int index, const int* cu_q, int n_seqs, int chunk, bool chunked) {
    // (no portion longer than a chunk: chunk i is sequence i, and no walk over the sequences, whose every step
    // would wait for a load)
    if (!chunked) return ChunkOf{index < n_seqs ? index : -1, 0, 1, 0};
    if (n_seqs <= 8) {
        ChunkOf c{0, index, 0, 0};
        for (; c.b < n_seqs; ++c.b) {
            c.n_chunks = max(1, (cu_q[c.b + 1] - cu_q[c.b] + chunk - 1) / chunk);
            if (c.k < c.n_chunks) return c;
            c.k -= c.n_chunks;
            if (c.n_chunks > 1) c.first_chunk += c.n_chunks;
        }
        c.b = -1;
        return c;
    }
    // Many sequences: 64 at a time, one a lane, their lengths arrive together and are summed over the lanes. One after the other, every
    // step waits for its load: 40 portions of 70 tokens, 24 heads of 128 x 64, scan and norm: 201 us > 158. (Up to eight the walk is
    // 1 us shorter.)
    const int lane = threadIdx.x % 64;
    int chunks_before = 0, states_before = 0;
    for (int b0 = 0; b0 < n_seqs; b0 += 64) {
        const int b = b0 + lane;
        const int n_tokens = cu_q[min(b + 1, n_seqs)] - cu_q[min(b, n_seqs)];
        const int n = b < n_seqs ? max(1, (n_tokens + chunk - 1) / chunk) : 0;
        int end = n;
#pragma unroll
        for (int off = 1; off < 64; off *= 2) {
            const int up = __shfl_up(end, off, 64);
            if (lane >= off) end += up;
        }
        const unsigned long long past = __ballot(chunks_before + end > index), single = __ballot(n == 1);
        if (past != 0) {
            const int at = __builtin_ctzll(past), n_chunks = __builtin_amdgcn_readlane(n, at);
            const int before = __builtin_amdgcn_readlane(end, at) - n_chunks;
            return ChunkOf{b0 + at, index - chunks_before - before, n_chunks,
                           states_before + before - static_cast<int>(__popcll(single & ((1ull << at) - 1)))};
        }
        const int all = __builtin_amdgcn_readlane(end, 63);
        chunks_before += all;
        states_before += all - static_cast<int>(__popcll(single));
    }
    return ChunkOf{-1, 0, 0, 0};
}

template <int NS>
__global__ void __launch_bounds__(64)
ssm_scan_kernel(const float* __restrict__ xbc, int ldx, const float* __restrict__ raw_dt, int ldd,
                const float* __restrict__ dt_bias, const float* __restrict__ A_log, const float* __restrict__ Dskip,
                const int* __restrict__ cu_q, const int* __restrict__ state_slots, int n_seqs, float* __restrict__ state,
                size_t slot_floats, size_t scan_offset, float* __restrict__ y, int ldy, size_t part_stride, int H, int P,
                int N, int G, int n_slices, int write, int chunk, float* __restrict__ chunk_state,
                float* __restrict__ cumlog) {
    const int lane = threadIdx.x;
    const int h = blockIdx.y, slice = blockIdx.x % n_slices, p = (blockIdx.x / n_slices) * 64 + lane;
    const ChunkOf co = chunk_of(blockIdx.z, cu_q, n_seqs, chunk, chunk_state != nullptr);
    if (co.b < 0) return;                                      // surplus workgroup
    const int slot = state_slots[co.b];
    if (slot < 0) return;
    const bool p_ok = p < P;
    const int pc = p_ok ? p : P - 1;
    const int g = h / (H / G), inner = H * P;
    const int n0 = slice * NS, nn = min(NS, N - n0);
    const int t0 = cu_q[co.b] + co.k * chunk, t1 = min(t0 + chunk, cu_q[co.b + 1]);
    float* sp = state + static_cast<size_t>(slot) * slot_floats + scan_offset + (static_cast<size_t>(h) * N + n0) * P + pc;
    // (every load below is issued without a condition, from a clamped index, and masked by a select afterwards: a
    // load under a condition waits for all loads in flight, which would make a token cost NS round trips)
    float S[NS];
#pragma unroll
    for (int j = 0; j < NS; ++j) S[j] = sp[static_cast<size_t>(min(j, nn - 1)) * P];
#pragma unroll
    for (int j = 0; j < NS; ++j) S[j] = (co.k == 0 && j < nn) ? S[j] : 0.f;
    const float bias = dt_bias[h], neg_rate = -expf(A_log[h]), skip = slice == 0 ? Dskip[h] : 0.f;
    const float* b_row = xbc + inner + g * N + n0;              // + t * ldx: B of the slice (the same for every lane)
    const float* c_row = b_row + G * N;
    float* yp = y + slice * part_stride + h * P + pc;
    // a token's operands are requested one token ahead; rows of the slice beyond N count as zeros
    float xv = 0.f, dtr = 0.f, Bv[NS], Cv[NS];
    auto load = [&](int t, float& x_, float& d_, float (&B_)[NS], float (&C_)[NS]) {
        x_ = xbc[static_cast<size_t>(t) * ldx + h * P + pc];
        d_ = raw_dt[static_cast<size_t>(t) * ldd + h];
        const float* Bt = b_row + static_cast<size_t>(t) * ldx;
        const float* Ct = c_row + static_cast<size_t>(t) * ldx;
#pragma unroll
        for (int j = 0; j < NS; ++j) {
            B_[j] = Bt[min(j, nn - 1)];
            C_[j] = Ct[min(j, nn - 1)];
        }
#pragma unroll
        for (int j = 0; j < NS; ++j) {
            B_[j] = j < nn ? B_[j] : 0.f;
            C_[j] = j < nn ? C_[j] : 0.f;
        }
    };
    load(min(t0, t1 - 1), xv, dtr, Bv, Cv);
    float cum = 0.f;
    for (int t = t0; t < t1; ++t) {
        float xn, dn, Bn[NS], Cn[NS];
        load(min(t + 1, t1 - 1), xn, dn, Bn, Cn);
        const float dt = softplus_precise(dtr + bias);
        const float a = expf(neg_rate * dt), dx = dt * xv;
        cum += neg_rate * dt;
        float acc = 0.f;
#pragma unroll
        for (int j = 0; j < NS; ++j) {
            S[j] = a * S[j] + dx * Bv[j];
            acc += S[j] * Cv[j];
        }
        if (p_ok) yp[static_cast<size_t>(t) * ldy] = acc + skip * xv;
        if (co.n_chunks > 1 && blockIdx.x == 0 && lane == 0) cumlog[static_cast<size_t>(t) * H + h] = cum;
        xv = xn; dtr = dn;
#pragma unroll
        for (int j = 0; j < NS; ++j) { Bv[j] = Bn[j]; Cv[j] = Cn[j]; }
    }
    if (!p_ok) return;
    if (co.n_chunks > 1) sp = chunk_state + ((static_cast<size_t>(co.first_chunk + co.k) * H + h) * N + n0) * P + p;
    if (write || co.n_chunks > 1) {
#pragma unroll
        for (int j = 0; j < NS; ++j)
            if (j < nn) sp[static_cast<size_t>(j) * P] = S[j];
    }
}

// The scan of sequences of at most CH tokens (decoding, short portions; longer ones leave at once and go through the chunk
// kernels below): one workgroup per (sequence, head, 64 values of p), a wavefront per slice of NS rows n (more
// slices than WAVES: in rounds). A wavefront's operands are staged in LDS first, x [CH][64], B and C of the slice [CH][NS] and the
// raw step sizes, all requested at once with 16-byte loads, so that the token loop waits for no memory (one token ahead is not enough
// to cover a load that another XCD's kernel wrote a moment ago). The slices' sums over n meet in LDS and are added in the order of
// the slices, so y leaves whole. WAVES of 1: a workgroup per slice, which stores its share in y + slice * part_stride for the reader to
// add. Needs 16-byte aligned rows and column offsets. Bound by the state that it reads and writes, at eight sequences
// (12.6 MB, 24 heads of 128 x 64) by the chain of one launch: 7.2 us a layer, and from a dozen tokens on by the chain of tokens,
// which sums that meet in LDS lengthen. LDS: floats a wavefront takes.
template <int NS, int CH> constexpr int ssm_short_floats() { return CH * 64 + 2 * CH * NS + 2 * CH; }
template <int NS, int CH, int WAVES>
__global__ void __launch_bounds__(64 * WAVES)
ssm_short_kernel(const float* __restrict__ xbc, int ldx, const float* __restrict__ raw_dt, int ldd,
                 const float* __restrict__ dt_bias, const float* __restrict__ A_log, const float* __restrict__ Dskip,
                 const int* __restrict__ cu_q, const int* __restrict__ state_slots, float* __restrict__ state,
                 size_t slot_floats, size_t scan_offset, float* __restrict__ y, int ldy, size_t part_stride, int H, int P, int N, int G, int write) {
    constexpr bool SHARES = WAVES == 1;
    extern __shared__ __attribute__((aligned(16))) float short_s[];
    const int lane = threadIdx.x % 64, wave = __builtin_amdgcn_readfirstlane(threadIdx.x / 64), waves = blockDim.x / 64;
    const int n_slices = (N + NS - 1) / NS;
    const int h = blockIdx.y, p0 = (SHARES ? blockIdx.x / n_slices : blockIdx.x) * 64, p = p0 + lane, b = blockIdx.z;
    const int t0 = cu_q[b], nt = cu_q[b + 1] - t0;
    const int slot = state_slots[b];
    if (slot < 0 || nt < 1 || nt > CH) return;                 // (the whole workgroup)
    const bool p_ok = p < P;
    const int pc = p_ok ? p : P - 1;
    const int g = h / (H / G), inner = H * P;
    float* xs = short_s + wave * ssm_short_floats<NS, CH>();
    float *Bs = xs + CH * 64, *Cs = Bs + CH * NS, *dts = Cs + CH * NS, *as = dts + CH;      // dts, as: the tokens' step sizes and decays
    for (int s0 = 0; s0 < (SHARES ? 1 : n_slices); s0 += waves) {
        const int slice = SHARES ? blockIdx.x % n_slices : s0 + wave;
        if (SHARES || slice < n_slices) {
            const int n0 = slice * NS, nn = min(NS, N - n0);
            float* sp = state + static_cast<size_t>(slot) * slot_floats + scan_offset + (static_cast<size_t>(h) * N + n0) * P + pc;
            float S[NS];
#pragma unroll
            for (int j = 0; j < NS; ++j) S[j] = sp[static_cast<size_t>(min(j, nn - 1)) * P];
            // Staging: quads of 4 floats, a fixed number per lane (CH * 16 quads of x, CH * NS / 4 of B and of C over 64
            // lanes), all requested before the first is written to LDS; tokens beyond the sequence's end repeat its last one,
            // a quad beyond the row's end (P or N no multiple of the tile) the row's last one.
            const int pq = min(64, P - p0) / 4, nq = nn / 4;           // whole quads of x and of B, C in this tile
            {
                constexpr int XQ = CH * 16 / 64, BQ = CH * (NS / 4) / 64;
                float4 xq[XQ], bq[BQ], cq[BQ];
#pragma unroll
                for (int u = 0; u < XQ; ++u) {
                    const int e = lane + 64 * u, tt = min(e / 16, nt - 1), q = min(e % 16, pq - 1);
                    xq[u] = *reinterpret_cast<const float4*>(xbc + static_cast<size_t>(t0 + tt) * ldx + h * P + p0 + 4 * q);
                }
#pragma unroll
                for (int u = 0; u < BQ; ++u) {
                    const int e = lane + 64 * u, tt = min(e / (NS / 4), nt - 1), q = min(e % (NS / 4), nq - 1);
                    const float* row = xbc + static_cast<size_t>(t0 + tt) * ldx + inner + g * N + n0 + 4 * q;
                    bq[u] = *reinterpret_cast<const float4*>(row);
                    cq[u] = *reinterpret_cast<const float4*>(row + G * N);
                }
#pragma unroll
                for (int u = 0; u < XQ; ++u) {
                    const int e = lane + 64 * u;
                    *reinterpret_cast<float4*>(&xs[e / 16 * 64 + 4 * (e % 16)]) = xq[u];
                }
#pragma unroll
                for (int u = 0; u < BQ; ++u) {
                    const int e = lane + 64 * u, qi = e % (NS / 4);
                    const bool real = qi < nq;                          // rows of the slice beyond N count as zeros
                    *reinterpret_cast<float4*>(&Bs[e / (NS / 4) * NS + 4 * qi]) = real ? bq[u] : make_float4(0.f, 0.f, 0.f, 0.f);
                    *reinterpret_cast<float4*>(&Cs[e / (NS / 4) * NS + 4 * qi]) = real ? cq[u] : make_float4(0.f, 0.f, 0.f, 0.f);
                }
            }
            // step sizes and decays are the same for every lane: lane t works them out for token t, once (softplus, two exponentials)
            const float neg_rate = -expf(A_log[h]), skip = slice == 0 ? Dskip[h] : 0.f;
            {
                static_assert(CH <= 64, "one lane per token");
                const float dt = softplus_precise(raw_dt[static_cast<size_t>(t0 + min(lane, nt - 1)) * ldd + h] + dt_bias[h]);
                if (lane < CH) {
                    dts[lane] = dt;
                    as[lane] = expf(neg_rate * dt);
                }
            }
#pragma unroll
            for (int j = 0; j < NS; ++j) S[j] = j < nn ? S[j] : 0.f;
            wave_lds_sync();
            for (int tt = 0; tt < nt; ++tt) {
                const float xv = xs[tt * 64 + lane];
                const float a = as[tt], dx = dts[tt] * xv;
                float acc[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
                for (int j = 0; j < NS; j += 4) {
                    const float4 b4 = *reinterpret_cast<const float4*>(&Bs[tt * NS + j]), c4 = *reinterpret_cast<const float4*>(&Cs[tt * NS + j]);
                    S[j] = a * S[j] + dx * b4.x;         acc[0] += S[j] * c4.x;
                    S[j + 1] = a * S[j + 1] + dx * b4.y; acc[1] += S[j + 1] * c4.y;
                    S[j + 2] = a * S[j + 2] + dx * b4.z; acc[2] += S[j + 2] * c4.z;
                    S[j + 3] = a * S[j + 3] + dx * b4.w; acc[3] += S[j + 3] * c4.w;
                }
                const float share = (acc[0] + acc[1]) + (acc[2] + acc[3]) + skip * xv;
                if constexpr (!SHARES) xs[tt * 64 + lane] = share;      // in x's place
                else if (p_ok) y[slice * part_stride + static_cast<size_t>(t0 + tt) * ldy + h * P + p] = share;
            }
            if (write && p_ok) {
#pragma unroll
                for (int j = 0; j < NS; ++j)
                    if (j < nn) sp[static_cast<size_t>(j) * P] = S[j];
            }
        }
        if constexpr (SHARES) return;
        __syncthreads();
        for (int i = threadIdx.x; i < nt * 64; i += blockDim.x) {
            if (p0 + i % 64 >= P) continue;
            float* out = y + static_cast<size_t>(t0 + i / 64) * ldy + h * P + p0 + i % 64;
            float v = s0 > 0 ? *out + short_s[i] : short_s[i];       // (an element's every round is the same thread's)
            for (int k = 1; k < min(waves, n_slices - s0); ++k) v += short_s[k * ssm_short_floats<NS, CH>() + i];
            *out = v;
        }
        if (s0 + waves < n_slices) __syncthreads();                  // the shares have been read
    }
}

// A portion of several chunks of SSM_TILE tokens in matrix form, on the fp32 matrix cores (v_mfma_f32_16x16x4_f32). With cum_t
// the logarithm of the decay accumulated from the chunk's start to token t:
//   state kernel:  L[n, p] = sum_s exp(cum_last - cum_s) dt_s B[s, n] x[s, p]          what the chunk adds to the state
//   join kernel:   S_0 = the slot's state, S_(k+1) = exp(cum_last of chunk k) S_k + L_k; S_k takes L_k's place, the last goes back
//   output kernel: y[t, p] = sum_(s <= t) (C_t . B_s) exp(cum_t - cum_s) dt_s x[s, p] + exp(cum_t) sum_n C[t, n] S_k[n, p] + D x[t, p]
// The same sums as token by token in another order; every exponent is at most 0. One workgroup of four wavefronts per (chunk,
// head, 64 values of p). n is walked in slices of SSM_NS rows that pass through LDS, the next slice's loads in flight during the
// products of one (45 KB of LDS: three workgroups a unit). Rows in LDS are an odd number of 16-byte pieces apart for operands read
// four k at a time, and 4 floats more than a multiple of 64 for those read one k at a time (16 neighbouring columns of four rows
// 4 apart): neither conflicts. A token after the other, as the short kernel does it, was bound by its chain of 64 tokens:
// 2,048 tokens of 24 heads of 128 x 64 took 85 us for the chunks and 45 to join them; the three kernels take 16.0, 11.7 and 28.0 us.
// A token's result must not depend on later ones: in the output kernel's second product their weights are 0, and 0 times an
// infinity is no 0, so the product takes zeros in place of x that are not finite, and a loop that a chunk without any skips
// adds these where they belong.
// Needs 16-byte aligned rows and column offsets.
#define SSM_TILE 64
#define SSM_NS 32
typedef float f32x4 __attribute__((ext_vector_type(4)));

// Step sizes and accumulated decays of a chunk's nt tokens, worked out by one wavefront (lane t: token t; past the end: dt 0).
// The logarithms are summed in double: their differences are small numbers between large ones (in 32 bits the logits of a small
// model were 5.8e-6 from the exact ones where the scan token by token is 1.5e-6 away, with this at most 1.5e-6).
__device__ __forceinline__ void chunk_decays(const float* raw_dt, int ldd, int t0, int nt, int h, const float* dt_bias, const float* A_log, int lane,
                                             float* dt_s, double* cum_s) {
    const float dt = softplus_precise(raw_dt[static_cast<size_t>(t0 + min(lane, nt - 1)) * ldd + h] + dt_bias[h]);
    // (a decay of exp(-1000) is 0 in fp32 like any smaller one; without the bound an infinite rate or step size leaves differences
    // of infinities, and a sum that holds a very large one has lost the small ones behind it. NaN stays.)
    double run = lane < nt ? -static_cast<double>(expf(A_log[h])) * dt : 0.0;
    if (run < -1000.0) run = -1000.0;
#pragma unroll
    for (int off = 1; off < 64; off *= 2) {
        const double up = __shfl_up(run, off, 64);
        if (lane >= off) run += up;
    }
    dt_s[lane] = lane < nt ? dt : 0.f;
    cum_s[lane] = run;
}

__global__ void __launch_bounds__(256)
ssm_chunk_state_kernel(const float* __restrict__ xbc, int ldx, const float* __restrict__ raw_dt, int ldd, const float* __restrict__ dt_bias,
                       const float* __restrict__ A_log, const int* __restrict__ cu_q, const int* __restrict__ state_slots, int n_seqs, int H, int P,
                       int N, int G, float* __restrict__ chunk_state, float* __restrict__ cumlog) {
    __shared__ __attribute__((aligned(16))) float Xs[SSM_TILE][68], Bs[SSM_TILE][SSM_NS + 4];
    __shared__ float dt_s[64];
    __shared__ double cum_s[64];
    const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid / 64), lane = tid % 64, col = lane % 16, quad = lane / 16;
    const int h = blockIdx.y, p0 = blockIdx.x * 64;
    const ChunkOf co = chunk_of(blockIdx.z, cu_q, n_seqs, SSM_TILE, true);
    if (co.b < 0 || co.n_chunks < 2 || state_slots[co.b] < 0) return;
    const int g = h / (H / G), inner = H * P;
    const int t0 = cu_q[co.b] + co.k * SSM_TILE, nt = min(t0 + SSM_TILE, cu_q[co.b + 1]) - t0;
    if (wave == 0) chunk_decays(raw_dt, ldd, t0, nt, h, dt_bias, A_log, lane, dt_s, cum_s);
    const int pq = min(64, P - p0) / 4;
    float4 xq[4], bq[2];
    const float* b_row = xbc + inner + g * N;
    auto fetch = [&](int n0) {
        const int nq = min(SSM_NS, N - n0) / 4;
#pragma unroll
        for (int u = 0; u < 2; ++u) {
            const int e = tid + 256 * u;
            bq[u] = *reinterpret_cast<const float4*>(b_row + static_cast<size_t>(t0 + min(e / 8, nt - 1)) * ldx + n0 + 4 * min(e % 8, nq - 1));
        }
    };
#pragma unroll
    for (int u = 0; u < 4; ++u) {
        const int e = tid + 256 * u;
        xq[u] = *reinterpret_cast<const float4*>(xbc + static_cast<size_t>(t0 + min(e / 16, nt - 1)) * ldx + h * P + p0 + 4 * min(e % 16, pq - 1));
    }
    fetch(0);
    __syncthreads();
    if (tid == 0) cumlog[static_cast<size_t>(t0 + nt - 1) * H + h] = static_cast<float>(cum_s[63]);
#pragma unroll
    for (int u = 0; u < 4; ++u) {          // (an infinity whose weight has underflowed stays one value that is not finite)
        const int e = tid + 256 * u, s = e / 16;
        const float w = expf(static_cast<float>(cum_s[63] - cum_s[s])) * dt_s[s];
        *reinterpret_cast<float4*>(&Xs[s][4 * (e % 16)]) = s < nt && e % 16 < pq ? make_float4(w * xq[u].x, w * xq[u].y, w * xq[u].z, w * xq[u].w) : make_float4(0.f, 0.f, 0.f, 0.f);
    }
    float* out = chunk_state + (static_cast<size_t>(co.first_chunk + co.k) * H + h) * N * P;
    for (int n0 = 0; n0 < N; n0 += SSM_NS) {
        const int nn = min(SSM_NS, N - n0);
        if (n0 > 0) __syncthreads();          // the slice before has been read
#pragma unroll
        for (int u = 0; u < 2; ++u) {
            const int e = tid + 256 * u;
            *reinterpret_cast<float4*>(&Bs[e / 8][4 * (e % 8)]) = e / 8 < nt && 4 * (e % 8) < nn ? bq[u] : make_float4(0.f, 0.f, 0.f, 0.f);
        }
        fetch(n0 + SSM_NS < N ? n0 + SSM_NS : n0);      // (past the last slice: it again, unused; under a condition it would be waited for here)
        __syncthreads();
        __builtin_amdgcn_sched_barrier(0);          // (the loads stay in front of the products)
        f32x4 acc[2] = {f32x4{0.f, 0.f, 0.f, 0.f}, f32x4{0.f, 0.f, 0.f, 0.f}};      // rows n of two tiles, columns p of the wavefront's
#pragma unroll
        for (int s = 0; s < SSM_TILE; s += 16)
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const int k = s + 4 * quad + e;
                const float xv = Xs[k][16 * wave + col];
#pragma unroll
                for (int i = 0; i < 2; ++i) acc[i] = __builtin_amdgcn_mfma_f32_16x16x4f32(Bs[k][16 * i + col], xv, acc[i], 0, 0, 0);
            }
#pragma unroll
        for (int i = 0; i < 2; ++i)
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const int n = 16 * i + 4 * quad + r, p = p0 + 16 * wave + col;
                if (n < nn && p < P) out[static_cast<size_t>(n0 + n) * P + p] = acc[i][r];
            }
    }
}

// One thread per element of a head's state; the chunks' sums are asked for four ahead.
__global__ void __launch_bounds__(256)
ssm_chunk_prefix_kernel(const int* __restrict__ cu_q, const int* __restrict__ state_slots, float* __restrict__ state, size_t slot_floats,
                        size_t scan_offset, int H, int NP, int write, float* __restrict__ chunk_state, const float* __restrict__ cumlog) {
    const int b = blockIdx.z, h = blockIdx.y, i = blockIdx.x * 256 + threadIdx.x;
    const int q0 = cu_q[b], q1 = cu_q[b + 1], n_chunks = (q1 - q0 + SSM_TILE - 1) / SSM_TILE;
    const int slot = state_slots[b];
    if (n_chunks < 2 || slot < 0) return;
    int first = 0;          // the states in front of the sequence's: 64 sequences at a time, as in chunk_of
    for (int k0 = 0; k0 < b; k0 += 64) {
        const int k = k0 + threadIdx.x % 64, n = (cu_q[min(k + 1, b)] - cu_q[min(k, b)] + SSM_TILE - 1) / SSM_TILE;      // (from b on: 0)
        int sum = n > 1 ? n : 0;
#pragma unroll
        for (int off = 32; off > 0; off /= 2) sum += __shfl_xor(sum, off, 64);
        first += sum;
    }
    first = __builtin_amdgcn_readfirstlane(first);
    if (i >= NP) return;
    float* sp = state + static_cast<size_t>(slot) * slot_floats + scan_offset + static_cast<size_t>(h) * NP + i;
    const size_t step = static_cast<size_t>(H) * NP;
    float* at = chunk_state + static_cast<size_t>(first) * step + static_cast<size_t>(h) * NP + i;
    float S = *sp;
    for (int k0 = 0; k0 < n_chunks; k0 += 4) {
        float L[4], a[4];
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            const int k = min(k0 + u, n_chunks - 1);
            L[u] = at[k * step];
            a[u] = cumlog[static_cast<size_t>(min(q0 + (k + 1) * SSM_TILE, q1) - 1) * H + h];
        }
#pragma unroll
        for (int u = 0; u < 4; ++u)
            if (k0 + u < n_chunks) {
                at[(k0 + u) * step] = S;
                S = expf(a[u]) * S + L[u];
            }
    }
    if (write) *sp = S;
}

__global__ void __launch_bounds__(256)
ssm_chunk_out_kernel(const float* __restrict__ xbc, int ldx, const float* __restrict__ raw_dt, int ldd, const float* __restrict__ dt_bias,
                     const float* __restrict__ A_log, const float* __restrict__ Dskip, const int* __restrict__ cu_q, const int* __restrict__ state_slots,
                     int n_seqs, float* __restrict__ y, int ldy, int H, int P, int N, int G, const float* __restrict__ chunk_state) {
    __shared__ __attribute__((aligned(16))) float Xs[SSM_TILE][68], Ps[SSM_NS][68];
    // the slices of B and C; once they are read, a wavefront's weights [16 tokens][64 tokens before] lie in their place
    __shared__ __attribute__((aligned(16))) float slices[2 * SSM_TILE * (SSM_NS + 4)];
    static_assert(4 * 16 * 68 <= 2 * SSM_TILE * (SSM_NS + 4), "the weights fit the slices");
    float (*Bs)[SSM_NS + 4] = reinterpret_cast<float (*)[SSM_NS + 4]>(slices), (*Cs)[SSM_NS + 4] = Bs + SSM_TILE;
    float (*Ms)[16][68] = reinterpret_cast<float (*)[16][68]>(slices);
    __shared__ float dt_s[64];
    __shared__ double cum_s[64];
    __shared__ int odd_s[4];          // whether a wavefront staged an x that is not finite
    const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid / 64), lane = tid % 64, col = lane % 16, quad = lane / 16;
    const int h = blockIdx.y, p0 = blockIdx.x * 64;
    const ChunkOf co = chunk_of(blockIdx.z, cu_q, n_seqs, SSM_TILE, true);
    if (co.b < 0 || co.n_chunks < 2 || state_slots[co.b] < 0) return;
    const int g = h / (H / G), inner = H * P;
    const int t0 = cu_q[co.b] + co.k * SSM_TILE, nt = min(t0 + SSM_TILE, cu_q[co.b + 1]) - t0;
    const int pq = min(64, P - p0) / 4;
    float4 xq[4], bq[2], cq[2], sq[2];
    const float* b_row = xbc + inner + g * N;
    const float* s_row = chunk_state + (static_cast<size_t>(co.first_chunk + co.k) * H + h) * N * P + p0;
    auto fetch = [&](int n0) {
        const int nn = min(SSM_NS, N - n0), nq = nn / 4;
#pragma unroll
        for (int u = 0; u < 2; ++u) {
            const int e = tid + 256 * u;
            const float* row = b_row + static_cast<size_t>(t0 + min(e / 8, nt - 1)) * ldx + n0 + 4 * min(e % 8, nq - 1);
            bq[u] = *reinterpret_cast<const float4*>(row);
            cq[u] = *reinterpret_cast<const float4*>(row + G * N);
            sq[u] = *reinterpret_cast<const float4*>(s_row + static_cast<size_t>(n0 + min(e / 16, nn - 1)) * P + 4 * min(e % 16, pq - 1));
        }
    };
    fetch(0);
#pragma unroll
    for (int u = 0; u < 4; ++u) {
        const int e = tid + 256 * u;
        xq[u] = *reinterpret_cast<const float4*>(xbc + static_cast<size_t>(t0 + min(e / 16, nt - 1)) * ldx + h * P + p0 + 4 * min(e % 16, pq - 1));
    }
    if (wave == 0) chunk_decays(raw_dt, ldd, t0, nt, h, dt_bias, A_log, lane, dt_s, cum_s);
    // the wavefront's tokens are rows 16 wave to + 15: gram, their products C_t . B_s with the tokens s of the tiles up to their own; acc, y
    f32x4 gram[4], acc[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) gram[j] = acc[j] = f32x4{0.f, 0.f, 0.f, 0.f};
    for (int n0 = 0; n0 < N; n0 += SSM_NS) {
        const int nn = min(SSM_NS, N - n0);
        if (n0 > 0) __syncthreads();
#pragma unroll
        for (int u = 0; u < 2; ++u) {
            const int e = tid + 256 * u;
            const bool real = e / 8 < nt && 4 * (e % 8) < nn;
            *reinterpret_cast<float4*>(&Bs[e / 8][4 * (e % 8)]) = real ? bq[u] : make_float4(0.f, 0.f, 0.f, 0.f);
            *reinterpret_cast<float4*>(&Cs[e / 8][4 * (e % 8)]) = real ? cq[u] : make_float4(0.f, 0.f, 0.f, 0.f);
            *reinterpret_cast<float4*>(&Ps[e / 16][4 * (e % 16)]) = e / 16 < nn && e % 16 < pq ? sq[u] : make_float4(0.f, 0.f, 0.f, 0.f);
        }
        if (n0 == 0) {
            bool odd = false;
#pragma unroll
            for (int u = 0; u < 4; ++u) {
                const int e = tid + 256 * u;
                const bool real = e / 16 < nt && e % 16 < pq;
                const float raw[4] = {xq[u].x, xq[u].y, xq[u].z, xq[u].w};
                float x[4];
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    const bool finite = __builtin_isfinite(raw[i]);
                    odd = odd || (real && !finite);
                    x[i] = real && finite ? raw[i] : 0.f;
                }
                *reinterpret_cast<float4*>(&Xs[e / 16][4 * (e % 16)]) = make_float4(x[0], x[1], x[2], x[3]);
            }
            const bool any_odd = __any(odd);
            if (lane == 0) odd_s[wave] = any_odd ? 1 : 0;
        }
        fetch(n0 + SSM_NS < N ? n0 + SSM_NS : n0);      // (past the last slice: it again, unused; under a condition it would be waited for here)
        __syncthreads();
        __builtin_amdgcn_sched_barrier(0);          // (the loads stay in front of the products)
#pragma unroll
        for (int q = 0; q < SSM_NS; q += 16) {
            // all operands first; products with tokens behind the wavefront's own, masked below, cost no more than the last
            // wavefront's, which needs all of them
            const f32x4 c4 = *reinterpret_cast<const f32x4*>(&Cs[16 * wave + col][q + 4 * quad]);
            f32x4 b4[4];
            float s4[4][4];
#pragma unroll
            for (int j = 0; j < 4; ++j) b4[j] = *reinterpret_cast<const f32x4*>(&Bs[16 * j + col][q + 4 * quad]);
#pragma unroll
            for (int e = 0; e < 4; ++e)
#pragma unroll
                for (int j = 0; j < 4; ++j) s4[e][j] = Ps[q + 4 * quad + e][16 * j + col];
#pragma unroll
            for (int e = 0; e < 4; ++e)
#pragma unroll
                for (int j = 0; j < 4; ++j) gram[j] = __builtin_amdgcn_mfma_f32_16x16x4f32(c4[e], b4[j][e], gram[j], 0, 0, 0);
#pragma unroll
            for (int e = 0; e < 4; ++e)
#pragma unroll
                for (int j = 0; j < 4; ++j) acc[j] = __builtin_amdgcn_mfma_f32_16x16x4f32(c4[e], s4[e][j], acc[j], 0, 0, 0);
        }
    }
    // (register r of a lane: row 4 quad + r, column col of a tile)
    double cum_t[4];
#pragma unroll
    for (int r = 0; r < 4; ++r) cum_t[r] = cum_s[16 * wave + 4 * quad + r];
#pragma unroll
    for (int r = 0; r < 4; ++r) {
        const float seen = expf(static_cast<float>(cum_t[r]));
#pragma unroll
        for (int j = 0; j < 4; ++j) acc[j][r] *= seen;
    }
    __syncthreads();          // the last slice has been read
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        const int s = 16 * j + col;
        const double cs = cum_s[s];
        const float ds = dt_s[s];
#pragma unroll
        for (int r = 0; r < 4; ++r)
            Ms[wave][4 * quad + r][s] = s <= 16 * wave + 4 * quad + r ? gram[j][r] * expf(static_cast<float>(cum_t[r] - cs)) * ds : 0.f;
    }
    wave_lds_sync();
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const f32x4 m4 = *reinterpret_cast<const f32x4*>(&Ms[wave][col][16 * i + 4 * quad]);
        float x4[4][4];
#pragma unroll
        for (int e = 0; e < 4; ++e)
#pragma unroll
            for (int j = 0; j < 4; ++j) x4[e][j] = Xs[16 * i + 4 * quad + e][16 * j + col];
#pragma unroll
        for (int e = 0; e < 4; ++e)
#pragma unroll
            for (int j = 0; j < 4; ++j) acc[j] = __builtin_amdgcn_mfma_f32_16x16x4f32(m4[e], x4[e][j], acc[j], 0, 0, 0);
    }
    const float skip = Dskip[h];
    if (odd_s[0] + odd_s[1] + odd_s[2] + odd_s[3] > 0) {          // infinities and NaN: to their own token and those behind it
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const float* x_col = xbc + static_cast<size_t>(t0) * ldx + h * P + min(p0 + 16 * j + col, P - 1);
            for (int s = 0; s < nt; ++s) {
                const float x = x_col[static_cast<size_t>(s) * ldx];
                if (__builtin_isfinite(x)) continue;
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    const int t = 16 * wave + 4 * quad + r;
                    if (s <= t) acc[j][r] += Ms[wave][4 * quad + r][s] * x + (s == t ? skip * x : 0.f);
                }
            }
        }
    }
#pragma unroll
    for (int j = 0; j < 4; ++j)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const int t = 16 * wave + 4 * quad + r, p = 16 * j + col;
            if (t < nt && p0 + p < P) y[static_cast<size_t>(t0 + t) * ldy + h * P + p0 + p] = acc[j][r] + skip * Xs[t][p];
        }
}

// What the chunks before chunk k of a portion contribute to it (see ssm_scan_kernel): with A_j the whole
// decay of chunk j and L_j its last local state, the state at the start of chunk k is
//   S = L_0 for k = 1;  S <- A_j S + L_j for j = 1 .. k - 1,
// every token t of chunk k gets  y[t] += exp(cumlog[t]) sum_n C[t, n] S[n, p] (slice by slice, as the scan), and
// the portion's last chunk writes A_k S + L_k back to the slot. Same grid and lane layout as the scan.
template <int NS>
__global__ void __launch_bounds__(64)
ssm_chunk_join_kernel(const float* __restrict__ xbc, int ldx, const int* __restrict__ cu_q, const int* __restrict__ state_slots,
                      int n_seqs, float* __restrict__ state, size_t slot_floats, size_t scan_offset, float* __restrict__ y,
                      int ldy, size_t part_stride, int H, int P, int N, int G, int n_slices, int write, int chunk,
                      const float* __restrict__ chunk_state, const float* __restrict__ cumlog) {
    const int lane = threadIdx.x;
    const int h = blockIdx.y, slice = blockIdx.x % n_slices, p = (blockIdx.x / n_slices) * 64 + lane;
    const ChunkOf co = chunk_of(blockIdx.z, cu_q, n_seqs, chunk, true);
    if (co.b < 0 || co.k == 0) return;                         // surplus, or a first chunk: nothing comes before it
    const int slot = state_slots[co.b];
    if (slot < 0) return;
    const bool p_ok = p < P;
    const int pc = p_ok ? p : P - 1;
    const int g = h / (H / G), inner = H * P;
    const int n0 = slice * NS, nn = min(NS, N - n0);
    const int q0 = cu_q[co.b], q1 = cu_q[co.b + 1];
    auto local_state = [&](int j) { return chunk_state + ((static_cast<size_t>(co.first_chunk + j) * H + h) * N + n0) * P + pc; };
    auto chunk_decay = [&](int j) { return expf(cumlog[static_cast<size_t>(min(q0 + (j + 1) * chunk, q1) - 1) * H + h]); };
    // (loads without conditions, from clamped indices, as in the scan; rows of the slice beyond N stay zero)
    float S[NS];
    {
        const float* l0 = local_state(0);
#pragma unroll
        for (int j = 0; j < NS; ++j) S[j] = l0[static_cast<size_t>(min(j, nn - 1)) * P];
#pragma unroll
        for (int j = 0; j < NS; ++j) S[j] = j < nn ? S[j] : 0.f;
    }
    for (int c = 1; c < co.k; ++c) {
        const float a = chunk_decay(c);
        const float* lc = local_state(c);
        float L[NS];
#pragma unroll
        for (int j = 0; j < NS; ++j) L[j] = lc[static_cast<size_t>(min(j, nn - 1)) * P];
#pragma unroll
        for (int j = 0; j < NS; ++j) S[j] = j < nn ? a * S[j] + L[j] : 0.f;
    }
    const int t0 = q0 + co.k * chunk, t1 = min(t0 + chunk, q1);
    const float* c_row = xbc + inner + G * N + g * N + n0;
    float* yp = y + slice * part_stride + h * P + pc;
    // the chunk's C rows of the slice and its tokens' decays go to LDS first, all requested at once (as the scan
    // stages its operands); y is then read, added to and written sixteen tokens at a time
    __shared__ float Cs[64][NS + 1];
    __shared__ float seen_s[64];
    const int nt = t1 - t0;
    {
        float cv[NS];
#pragma unroll
        for (int u = 0; u < NS; ++u) {
            const int e = lane + 64 * u, tt = min(e / NS, nt - 1), j = min(e % NS, nn - 1);
            cv[u] = c_row[static_cast<size_t>(t0 + tt) * ldx + j];
        }
        const float sv = cumlog[static_cast<size_t>(t0 + min(lane, nt - 1)) * H + h];
#pragma unroll
        for (int u = 0; u < NS; ++u) {
            const int e = lane + 64 * u;
            Cs[e / NS][e % NS] = cv[u];
        }
        seen_s[lane] = expf(sv);
    }
    wave_lds_sync();
    for (int t = 0; t < nt; t += 16) {
        float before[16];
#pragma unroll
        for (int u = 0; u < 16; ++u) before[u] = yp[static_cast<size_t>(t0 + min(t + u, nt - 1)) * ldy];     // (pc is a valid column for every lane)
#pragma unroll
        for (int u = 0; u < 16; ++u) {
            const int tt = min(t + u, nt - 1);
            float acc = 0.f;
#pragma unroll
            for (int j = 0; j < NS; ++j) acc += S[j] * Cs[tt][j];         // (S is zero beyond N)
            if (p_ok && t + u < nt) yp[static_cast<size_t>(t0 + t + u) * ldy] = before[u] + seen_s[tt] * acc;
        }
    }
    if (write && co.k == co.n_chunks - 1) {
        const float a = chunk_decay(co.k);
        const float* lk = local_state(co.k);
        float L[NS];
#pragma unroll
        for (int j = 0; j < NS; ++j) L[j] = lk[static_cast<size_t>(min(j, nn - 1)) * P];
        float* sp = state + static_cast<size_t>(slot) * slot_floats + scan_offset + (static_cast<size_t>(h) * N + n0) * P + pc;
#pragma unroll
        for (int j = 0; j < NS; ++j)
            if (j < nn && p_ok) sp[static_cast<size_t>(j) * P] = a * S[j] + L[j];
    }
}

}  // namespace

// The launch of rmsnorm_conv_single_kernel by taps, width and output type.
template <int MODE>
static int stream_conv_single_launch(float* x, int ldx, const float* y, int ldy, const float* wn, float eps, int C, const float* wc,
                                     int taps, const int* state_slots, float* state, size_t slot_floats, void* out, int ldo,
                                     int out_dtype, int T, int write, hipStream_t stream) {
#define RCS(TYPE, TAPS, NB)                                                                                            \
    rmsnorm_conv_single_kernel<TYPE, TAPS, NB, MODE><<<T, 64 * NB, 0, stream>>>(x, ldx, y, ldy, wn, eps, C, wc, state_slots, state, \
                                                                               slot_floats, static_cast<TYPE*>(out), ldo, write)
#define RCS_NB(TYPE, TAPS)                                                                                             \
    do {                                                                                                               \
        if (C <= 512) RCS(TYPE, TAPS, 1); else if (C <= 1024) RCS(TYPE, TAPS, 2); else if (C <= 1536) RCS(TYPE, TAPS, 3);   \
        else RCS(TYPE, TAPS, 4);                                                                                       \
    } while (0)
#define RCS_TAPS(TYPE)                                                                                                 \
    switch (taps) {                                                                                                    \
        case 1: RCS_NB(TYPE, 1); break; case 2: RCS_NB(TYPE, 2); break; case 3: RCS_NB(TYPE, 3); break;                \
        case 4: RCS_NB(TYPE, 4); break; case 5: RCS_NB(TYPE, 5); break; case 6: RCS_NB(TYPE, 6); break;                \
        case 7: RCS_NB(TYPE, 7); break; default: RCS_NB(TYPE, 8); break;                                               \
    }
    if (out_dtype == MLLM_F32) { RCS_TAPS(float) } else { RCS_TAPS(bf16_t) }
#undef RCS_TAPS
#undef RCS_NB
#undef RCS
    MLLM_LAUNCH_CHECK();
    return 0;
}

extern "C" {

// Convolution + silu of columns [col0, col0 + C) of proj's rows into out [T, C]; then, with `write`, the
// slots' carried rows are brought up to date (a second kernel: it overwrites what the first one reads).
// -1: taps outside 1..16.
int mllm_conv_silu(const float* proj, int ld, int col0, int C, const float* w, const float* bias, int taps,
                   const int* token_seq, const int* cu_q, const int* state_slots, float* state, size_t slot_floats,
                   float* out, int ldo, int T, int B, int write, hipStream_t stream) {
    if (T <= 0 || C <= 0) return 0;
    if (taps < 1 || taps > 16) return -1;
    const long long total = static_cast<long long>(T) * C;
    // (one token a sequence: the convolution's kernel brings the carried rows up to date itself)
    const bool single = T == B && write && taps > 1;
    const bool vec = taps <= 8 && C % 4 == 0 && col0 % 4 == 0 && ld % 4 == 0 && ldo % 4 == 0 && slot_floats % 4 == 0 &&
                     ((reinterpret_cast<uintptr_t>(proj) | reinterpret_cast<uintptr_t>(w) | reinterpret_cast<uintptr_t>(bias) |
                       reinterpret_cast<uintptr_t>(state) | reinterpret_cast<uintptr_t>(out)) & 15) == 0;
    if (vec) {
        const long long total4 = total / 4;
        const int blocks4 = static_cast<int>((total4 + 255) / 256);
        // (Fewer threads than that have nothing to hide their longer way behind, the more of them the fewer times a row is read. Four taps: 1,032 x 1,792
        // 8.3 us either way, 2,048 x 768 6.4, four rows a thread 7.1; three: 3,200 x 768 in portions of 65 10.7 and 11.1, 1,600 x 1,792 12.8 > 12.0; two:
        // 1,200 x 1,792 8.8 and 9.4, 2,400 14.1 > 12.6.)
        constexpr int ROWS = 4;
        if (!single && total4 * taps >= 1 << 21 && taps >= 2 && taps <= 4) {
            const int blocks = static_cast<int>(((T + ROWS - 1) / ROWS * static_cast<long long>(C / 4) + 255) / 256);
#define CSR(TAPS) case TAPS: conv_silu_rows_kernel<TAPS, ROWS><<<blocks, 256, 0, stream>>>(proj + col0, ld, C, w, bias, token_seq, cu_q, state_slots, state, \
                                                                                          slot_floats, out, ldo, T); break
            switch (taps) { CSR(2); CSR(3); default: CSR(4); }
#undef CSR
        } else
        if (single) {
#define CS1(TAPS) case TAPS: conv_silu_single_kernel<TAPS><<<dim3(T, (C / 4 + 63) / 64), 64, 0, stream>>>(proj + col0, ld, C, w, bias, state_slots, state, \
                                                                                                        slot_floats, out, ldo); break
            switch (taps) { CS1(2); CS1(3); CS1(4); CS1(5); CS1(6); CS1(7); CS1(8); }
#undef CS1
        } else
#define CSV(TAPS) case TAPS: conv_silu_vec_kernel<TAPS><<<blocks4, 256, 0, stream>>>(proj + col0, ld, C, w, bias, token_seq, cu_q, state_slots, state, \
                                                                                    slot_floats, out, ldo, total4); break
        switch (taps) { CSV(1); CSV(2); CSV(3); CSV(4); CSV(5); CSV(6); CSV(7); CSV(8); }
#undef CSV
    } else {
        conv_silu_kernel<<<static_cast<int>((total + 255) / 256), 256, 0, stream>>>(proj, ld, col0, C, w, bias, taps, token_seq, cu_q,
                                                                                    state_slots, state, slot_floats, out, ldo, total, single ? 1 : 0);
    }
    MLLM_LAUNCH_CHECK();
    if (write && taps > 1 && !single) {
        const long long pairs = static_cast<long long>(B) * C;
        conv_carry_kernel<<<static_cast<int>((pairs + 255) / 256), 256, 0, stream>>>(proj, ld, col0, C, taps, cu_q, state_slots, state,
                                                                                    slot_floats, B);
        MLLM_LAUNCH_CHECK();
    }
    return 0;
}

// out = in + conv(in) (residual == 0: conv(in) alone) over the C columns of in's rows (fp32), out in out_dtype; the
// slots' carried rows are brought up to date as by mllm_conv_silu. -1: taps outside 1..16.
int mllm_conv_residual(const float* in, int ld, int C, const float* w, int taps, const int* token_seq, const int* cu_q,
                       const int* state_slots, float* state, size_t slot_floats, void* out, int ldo, int out_dtype, int T,
                       int B, int write, hipStream_t stream, int residual) {
    if (T <= 0 || C <= 0) return 0;
    if (taps < 1 || taps > 16) return -1;
    const long long total = static_cast<long long>(T) * C;
    const bool single = T == B && write && taps > 1;
    const bool vec = taps <= 8 && C % 4 == 0 && ld % 4 == 0 && ldo % 4 == 0 && slot_floats % 4 == 0 &&
                     ((reinterpret_cast<uintptr_t>(in) | reinterpret_cast<uintptr_t>(w) | reinterpret_cast<uintptr_t>(state) |
                       reinterpret_cast<uintptr_t>(out)) & 15) == 0;
    if (vec) {
        const long long total4 = total / 4;
        const int blocks4 = static_cast<int>((total4 + 255) / 256);
#define CRV(TYPE, TAPS)                                                                                                \
    conv_residual_vec_kernel<TYPE, TAPS><<<blocks4, 256, 0, stream>>>(in, ld, C, w, token_seq, cu_q, state_slots, state, slot_floats, \
                                                                     static_cast<TYPE*>(out), ldo, total4, single ? 1 : 0, residual)
#define CRV_TAPS(TYPE)                                                                                                 \
    switch (taps) {                                                                                                    \
        case 1: CRV(TYPE, 1); break; case 2: CRV(TYPE, 2); break; case 3: CRV(TYPE, 3); break; case 4: CRV(TYPE, 4); break; \
        case 5: CRV(TYPE, 5); break; case 6: CRV(TYPE, 6); break; case 7: CRV(TYPE, 7); break; default: CRV(TYPE, 8); break; \
    }
        if (out_dtype == MLLM_F32) { CRV_TAPS(float) } else { CRV_TAPS(bf16_t) }
#undef CRV_TAPS
#undef CRV
    } else {
        const int blocks = static_cast<int>((total + 255) / 256);
        if (out_dtype == MLLM_F32)
            conv_residual_kernel<float><<<blocks, 256, 0, stream>>>(in, ld, C, w, taps, token_seq, cu_q, state_slots, state, slot_floats,
                                                                    static_cast<float*>(out), ldo, total, single ? 1 : 0, residual);
        else
            conv_residual_kernel<bf16_t><<<blocks, 256, 0, stream>>>(in, ld, C, w, taps, token_seq, cu_q, state_slots, state,
                                                                     slot_floats, static_cast<bf16_t*>(out), ldo, total, single ? 1 : 0, residual);
    }
    MLLM_LAUNCH_CHECK();
    if (write && taps > 1 && !single) {
        const long long pairs = static_cast<long long>(B) * C;
        conv_carry_kernel<<<static_cast<int>((pairs + 255) / 256), 256, 0, stream>>>(in, ld, 0, C, taps, cu_q, state_slots, state,
                                                                                    slot_floats, B);
        MLLM_LAUNCH_CHECK();
    }
    return 0;
}

// out = h + conv(h), h = rmsnorm(x) * wn, for a step of T sequences of one token each (token t is sequence t).
// -1: taps outside 1..16; -2: more than 8 taps or rows of more than 2,048 columns (nothing is launched).
int mllm_rmsnorm_conv_single(const float* x, int ldx, const float* wn, float eps, int C, const float* wc, int taps,
                             const int* state_slots, float* state, size_t slot_floats, void* out, int ldo, int out_dtype, int T,
                             int write, hipStream_t stream) {
    if (T <= 0 || C <= 0) return 0;
    if (taps < 1 || taps > 16) return -1;
    if (taps > 8 || C > 2048) return -2;           // sizes this kernel is not made for: norm and convolution apart
    // (this mode only reads x)
    return stream_conv_single_launch<0>(const_cast<float*>(x), ldx, nullptr, 0, wn, eps, C, wc, taps, state_slots, state, slot_floats, out,
                                        ldo, out_dtype, T, write, stream);
}

// For a step of T sequences of one token each, the stream's rows x [T, C] (fp32) and a block's input convolution:
// with y (a sub-layer's result, fp32 [T, C]) and wn: x += y / sqrt(mean(y^2) + eps) * wn first (x is written), then
// out = x + conv(x); with y null: out = x + conv(x) alone. Return codes as mllm_rmsnorm_conv_single's.
int mllm_stream_conv_single(float* x, int ldx, const float* y, int ldy, const float* wn, float eps, int C, const float* wc, int taps,
                            const int* state_slots, float* state, size_t slot_floats, void* out, int ldo, int out_dtype, int T,
                            int write, hipStream_t stream) {
    if (T <= 0 || C <= 0) return 0;
    if (taps < 1 || taps > 16 || (y != nullptr && wn == nullptr)) return -1;
    if (taps > 8 || C > 2048) return -2;
    if (y != nullptr)
        return stream_conv_single_launch<1>(x, ldx, y, ldy, wn, eps, C, wc, taps, state_slots, state, slot_floats, out, ldo, out_dtype, T,
                                            write, stream);
    return stream_conv_single_launch<2>(x, ldx, nullptr, 0, nullptr, eps, C, wc, taps, state_slots, state, slot_floats, out, ldo,
                                        out_dtype, T, write, stream);
}

// Tokens of a chunk, rows of n a wavefront keeps, and what the chunks' workspace must hold for a step of T tokens.
#define SSM_CHUNK 64
#define SSM_SLICE 32
static size_t chunk_states(int T) { return 2 * static_cast<size_t>(T) / SSM_CHUNK + 1; }
size_t mllm_ssm_scan_workspace_floats(int T, int B, int H, int P, int N) {
    (void)B;
    return chunk_states(T) * H * P * N + static_cast<size_t>(T) * H + 3;      // (3: the states start at a 16-byte border inside)
}
// Whether the kernels that read 16 bytes at a time take these rows: the short one and the ones in matrix form.
static bool ssm_by_quads(const float* xbc, int ldx, int P, int N) {
    return ldx % 4 == 0 && P % 4 == 0 && N % 4 == 0 && (reinterpret_cast<uintptr_t>(xbc) & 15) == 0;
}
// Whether the short kernel leaves a share per slice. One share costs every token's chain a store to LDS and the end a barrier, several are
// written and read again: scan and norm, us, one share / one a slice: 24 heads of 128 x 64: 1 x 32 tokens 23.0 / 21.0, 1 x 64 34.8 / 31.2,
// 8 x 32 24.5 / 25.4, 8 x 64 37.9 / 37.5; 24 heads of 64 x 64, 8 x 64: 36.6 / 33.6; 8 heads of 16 x 64 (a share either way), 8 x 64: 35.6 / 29.0;
// 4 heads of 256 x 128 (one share in two rounds), 1 x 64: 61.5 / 44.6. Up to 8 tokens one share is even for one sequence (8 tokens: 13.1 / 12.9)
// and ahead for several (8 x 8: 13.8 / 15.1; 64 x 1: 25.4 / 39.9).
static bool ssm_shares(int T, int max_q_len, int H, int P, int n_slices) {
    return max_q_len > 8 && max_q_len <= SSM_CHUNK && (n_slices > 4 || static_cast<double>(T) * H * P * (n_slices - 1) <= 1 << 20);
}
// The scan leaves y as this many shares, part_stride floats apart: one, or one per slice of the state's rows.
int mllm_ssm_scan_parts(const float* xbc, int ldx, int T, int max_q_len, int H, int P, int N) {
    const int n_slices = (N + SSM_SLICE - 1) / SSM_SLICE;
    return ssm_by_quads(xbc, ldx, P, N) && !ssm_shares(T, max_q_len, H, P, n_slices) ? 1 : n_slices;
}

// The scan over every sequence's portion (see the kernels). `workspace` (mllm_ssm_scan_workspace_floats floats)
// is needed when a portion is longer than one chunk (max_q_len > 64). -1: H is no multiple of G, or the
// workspace is missing.
int mllm_ssm_scan(const float* xbc, int ldx, const float* raw_dt, int ldd, const float* dt_bias, const float* A_log,
                  const float* Dskip, const int* cu_q, const int* state_slots, float* state, size_t slot_floats,
                  size_t scan_offset, float* y, int ldy, size_t part_stride, int T, int B, int max_q_len, int H, int P, int N,
                  int G, int write, float* workspace, hipStream_t stream) {
    if (B <= 0 || T <= 0) return 0;
    if (H < 1 || G < 1 || H % G != 0 || N < 1 || P < 1) return -1;
    const bool chunked = max_q_len > SSM_CHUNK;
    if (chunked && workspace == nullptr) return -1;
    const int n_chunks = chunked ? T / SSM_CHUNK + B : B;
    float* chunk_state = reinterpret_cast<float*>((reinterpret_cast<uintptr_t>(workspace) + 15) & ~static_cast<uintptr_t>(15));
    float* cumlog = workspace ? chunk_state + chunk_states(T) * H * P * N : nullptr;
    const int n_slices = (N + SSM_SLICE - 1) / SSM_SLICE;
    if (ssm_by_quads(xbc, ldx, P, N)) {
        const int p_tiles = (P + 63) / 64;
#define SSM_SHORT(CH, WAVES)                                                                                           \
    do {                                                                                                               \
        constexpr int floats = ssm_short_floats<SSM_SLICE, CH>();                                                      \
        auto kernel = ssm_short_kernel<SSM_SLICE, CH, WAVES>;                                                          \
        static bool lds_allowed = WAVES * floats * 4 <= 64 * 1024;      /* more has to be asked for once */            \
        if (!lds_allowed) {                                                                                            \
            const hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(kernel), hipFuncAttributeMaxDynamicSharedMemorySize, WAVES * floats * 4); \
            if (e != hipSuccess) return static_cast<int>(e);                                                           \
            lds_allowed = true;                                                                                        \
        }                                                                                                              \
        const int waves = std::min(n_slices, WAVES);                                                                   \
        kernel<<<dim3(WAVES == 1 ? p_tiles * n_slices : p_tiles, H, B), 64 * waves, waves * floats * 4, stream>>>(xbc, ldx, raw_dt, ldd, dt_bias, A_log, \
            Dskip, cu_q, state_slots, state, slot_floats, scan_offset, y, ldy, part_stride, H, P, N, G, write);        \
    } while (0)
        if (max_q_len <= 8) {
            if (n_slices > 4) SSM_SHORT(8, 8); else SSM_SHORT(8, 4);
        } else if (ssm_shares(T, max_q_len, H, P, n_slices)) {
            SSM_SHORT(SSM_CHUNK, 1);
        } else if (!chunked || T < static_cast<long>(B) * max_q_len) {      // (equally long portions of several chunks: none)
            SSM_SHORT(SSM_CHUNK, 4);
        }
#undef SSM_SHORT
        if (chunked) {
            const dim3 tiles(p_tiles, H, n_chunks);
            ssm_chunk_state_kernel<<<tiles, 256, 0, stream>>>(xbc, ldx, raw_dt, ldd, dt_bias, A_log, cu_q, state_slots, B, H, P, N, G, chunk_state, cumlog);
            ssm_chunk_prefix_kernel<<<dim3((N * P + 255) / 256, H, B), 256, 0, stream>>>(cu_q, state_slots, state, slot_floats, scan_offset, H, N * P,
                                                                                        write, chunk_state, cumlog);
            ssm_chunk_out_kernel<<<tiles, 256, 0, stream>>>(xbc, ldx, raw_dt, ldd, dt_bias, A_log, Dskip, cu_q, state_slots, B, y, ldy, H, P, N, G, chunk_state);
        }
        MLLM_LAUNCH_CHECK();
        return 0;
    }
    const dim3 grid(((P + 63) / 64) * n_slices, H, n_chunks);
    ssm_scan_kernel<SSM_SLICE><<<grid, 64, 0, stream>>>(xbc, ldx, raw_dt, ldd, dt_bias, A_log, Dskip, cu_q, state_slots, B, state,
                                                       slot_floats, scan_offset, y, ldy, part_stride, H, P, N, G, n_slices, write,
                                                       SSM_CHUNK, chunked ? chunk_state : nullptr, cumlog);
    if (chunked)
        ssm_chunk_join_kernel<SSM_SLICE><<<grid, 64, 0, stream>>>(xbc, ldx, cu_q, state_slots, B, state, slot_floats, scan_offset, y,
                                                                 ldy, part_stride, H, P, N, G, n_slices, write, SSM_CHUNK,
                                                                 chunk_state, cumlog);
    MLLM_LAUNCH_CHECK();
    return 0;
}

}  // extern "C"
