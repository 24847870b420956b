// Test-only kernels: what the lane exchanges of the kernels' common.h and the orders of query_tiles.h give, for tests of them
// (tests/test_kernels_gpu.py). Not part of the engine.
#include "common.h"
#include "query_tiles.h"

// out[lane] = maximum, out[64 + lane] = sum over lanes l, l ^ 16, l ^ 32, l ^ 48 of in[lane] (one wavefront),
// then in[lane ^ 8], in[lane ^ 16], in[lane ^ 32], in[lane ^ 4]: what rows_max, rows_sum and lane_xor give.
// out: 384 floats.
__global__ void rows_check_kernel(const float* __restrict__ in, float* __restrict__ out) {
    const float v = in[threadIdx.x];
    out[threadIdx.x] = rows_max(v);
    out[64 + threadIdx.x] = rows_sum(v);
    out[128 + threadIdx.x] = lane_xor(v, 8);
    out[192 + threadIdx.x] = lane_xor(v, 16);
    out[256 + threadIdx.x] = lane_xor(v, 32);
    out[320 + threadIdx.x] = lane_xor(v, 4);
}

extern "C" int mllm_rows_check(const float* in, float* out, hipStream_t stream) {
    rows_check_kernel<<<1, 64, 0, stream>>>(in, out);
    MLLM_LAUNCH_CHECK();
    return 0;
}

// out[place] = (sequence, tile, first query, queries) of workgroup `place`. order 0: query_tile, 1: next_tile, 2: longest_tile (at most 64 sequences).
__global__ void query_tiles_kernel(const int* __restrict__ cu_q, const int* __restrict__ ctx_len, int n_seqs, int rows, int order, int4* __restrict__ out) {
    const int place = blockIdx.x, places = gridDim.x;
    const QueryTile t = order == 0 ? query_tile<64>(cu_q, ctx_len, n_seqs, rows, place, places)
                        : order == 1 ? next_tile<64>(cu_q, n_seqs, rows, place, places) : longest_tile<64>(cu_q, ctx_len, n_seqs, rows, place);
    if (threadIdx.x == 0) out[place] = make_int4(t.b, t.tile, t.q_begin, t.q_len);
}

extern "C" int mllm_query_tiles(const int* cu_q, const int* ctx_len, int n_seqs, int rows, int order, int places, void* out, hipStream_t stream) {
    if (n_seqs < 1 || rows < 1 || places < 1 || order < 0 || order > 2 || (order == 2 && n_seqs > 64)) return -1;
    query_tiles_kernel<<<places, 256, 0, stream>>>(cu_q, ctx_len, n_seqs, rows, order, static_cast<int4*>(out));
    MLLM_LAUNCH_CHECK();
    return 0;
}
