"""Each HIP kernel alone against its plain reference (tests/plain_ops.py), at sizes other
than the engine's tiny models: widths and vocabularies that are no power of two,
ragged row counts, several head sizes and group counts."""
import math

import pytest
import torch

import plain_ops
import ref_ops

pytestmark = pytest.mark.gpu

DEV = "cuda:0"
DTYPES = [torch.float32, torch.bfloat16]


@pytest.fixture(scope="module")
def ops():
    from mini_llm_amd.kernels import ops as o
    return o


def _tol(dtype, scale=1.0):
    return (2e-5 if dtype == torch.float32 else 1.6e-2) * scale


def _rand(shape, dtype, gen, std=1.0):
    return (torch.randn(shape, generator=gen, dtype=torch.float32) * std).to(dtype)


def test_loaded_libraries_are_in_tree(ops):
    """After an op has run, the native code mapped into this process is the in-tree build: the engine
    library and the kernel libraries it links, all from the package's own folder and nowhere else."""
    import os
    from mini_llm_amd import build
    out = torch.empty(2, dtype=torch.int32, device=DEV)
    ops.argmax(torch.tensor([[0.0, 2.0, 1.0], [3.0, 2.0, 1.0]], device=DEV), out)
    assert out.tolist() == [1, 0]
    with open("/proc/self/maps") as f:
        mapped = {line.split()[-1] for line in f if "libmllm_" in line}
    names = {os.path.basename(m) for m in mapped}
    for lib in ("engine", "elementwise", "gemm_bf16", "gemm_f32", "attention_decode", "attention_prefill", "sampling"):
        assert os.path.basename(build.lib_path(lib)) in names, (lib, names)
    here = os.path.realpath(os.path.join(os.path.dirname(os.path.abspath(__file__)), "native", "_lib"))     # the tests' own
    assert all(os.path.dirname(os.path.realpath(m)) in (os.path.realpath(build.LIB_DIR), here) for m in mapped), mapped


def test_lane_exchange_between_rows(ops):
    """The reductions over one lane of each 16-lane row (built on gfx950's row swaps) against their meaning."""
    import ctypes
    import toy  # noqa: F401  (registers the test-only library)
    from mini_llm_amd import build
    lib = build.load_library("lane_check")
    g = torch.Generator().manual_seed(3)
    v = torch.randn(64, generator=g)
    out = torch.zeros(384, device=DEV)
    rc = lib.mllm_rows_check(ctypes.c_void_p(v.to(DEV).data_ptr()), ctypes.c_void_p(out.data_ptr()),
                             ctypes.c_void_p(torch.cuda.current_stream().cuda_stream))
    assert rc == 0
    groups = v.view(4, 16)
    assert torch.equal(out[:64].cpu().view(4, 16), groups.max(0).values.expand(4, 16))
    want = (groups[0] + groups[1]) + (groups[2] + groups[3])
    assert torch.equal(out[64:128].cpu().view(4, 16), want.expand(4, 16))
    lanes = torch.arange(64)
    for i, off in enumerate((8, 16, 32, 4)):
        assert torch.equal(out[128 + 64 * i:192 + 64 * i].cpu(), v[lanes ^ off]), off


def test_ops_refuse_cpu_tensors(ops):
    x = torch.zeros(2, 8)
    with pytest.raises(ops.KernelError, match="not on the GPU"):
        ops.layernorm(x, torch.ones(8), None, 1e-5, torch.empty(2, 8))


@pytest.mark.parametrize("dtype", DTYPES)
def test_embed_reference_vector(ops, dtype):
    # /root/reference/tests/kernels/embedding/gen.py:13-27
    V, P, D = 64, 32, 768
    wte = (torch.arange(V)[:, None] * 0.01 + torch.arange(D)[None, :] * 0.0001).to(dtype)
    wpe = (torch.arange(P)[:, None] * 0.001 + torch.arange(D)[None, :] * 0.00001).to(dtype)
    ids = torch.tensor([3, 5, 7, 5, 11, 13, 17], dtype=torch.int32)
    pos = torch.arange(7, dtype=torch.int32)
    out = torch.empty(7, D, dtype=torch.float32, device=DEV)
    ops.embed(ids.to(DEV), pos.to(DEV), wte.to(DEV), wpe.to(DEV), out)
    ref = wte[ids.long()].float() + wpe[pos.long()].float()
    assert (out.cpu() - ref).abs().max() <= 1e-6
    # without a position table
    ops.embed(ids.to(DEV), None, wte.to(DEV), None, out)
    assert torch.equal(out.cpu(), wte[ids.long()].float())
    # tokens taken on the device from what an earlier step sampled: rows 1, 4 and 6 (a source beyond the
    # sampled tokens is ignored, as by select_tokens)
    src = torch.tensor([-1, 2, -1, -1, 0, 9, 1], dtype=torch.int32)
    prev = torch.tensor([60, 61, 62], dtype=torch.int32)
    ops.embed(ids.to(DEV), pos.to(DEV), wte.to(DEV), wpe.to(DEV), out, src=src.to(DEV), prev=prev.to(DEV))
    fed = torch.tensor([3, 62, 7, 5, 60, 13, 61])
    assert (out.cpu() - (wte[fed].float() + wpe[pos.long()].float())).abs().max() <= 1e-6
    want = plain_ops.embed(ids, pos, wte, wpe, torch.empty(7, D, dtype=torch.float64), src=src, prev=prev)
    assert (out.cpu().double() - want).abs().max() <= 1e-6


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("rows,D,eps", [(17, 768, 1e-5), (5, 100, 1e-6), (3, 1600, 1e-5), (1, 16, 1e-3),
                                        (2050, 768, 1e-5), (6, 2048, 1e-5), (5, 2052, 1e-5), (4, 98, 1e-6)])
def test_layernorm(ops, dtype, rows, D, eps):
    g = torch.Generator().manual_seed(0)
    x = _rand((rows, D), torch.float32, g) + 0.5
    gamma = 1 + 0.1 * _rand((D,), torch.float32, g)
    beta = 0.1 * _rand((D,), torch.float32, g)
    out = torch.empty(rows, D, dtype=dtype, device=DEV)
    ops.layernorm(x.to(DEV), gamma.to(DEV), beta.to(DEV), eps, out)
    ref = plain_ops.layernorm(x, gamma, beta, eps, torch.empty(rows, D, dtype=torch.float64))
    assert (out.cpu().double() - ref).abs().max() <= _tol(dtype, 4)
    # selected rows, no bias
    sel = torch.tensor([rows - 1, 0], dtype=torch.int32)
    out2 = torch.empty(2, D, dtype=dtype, device=DEV)
    ops.layernorm(x.to(DEV), gamma.to(DEV), None, eps, out2, rows=sel.to(DEV))
    ref2 = plain_ops.layernorm(x, gamma, None, eps, torch.empty(2, D, dtype=torch.float64), rows=sel)
    assert (out2.cpu().double() - ref2).abs().max() <= _tol(dtype, 4)


def test_layernorm_constant_row_gives_beta(ops):
    D = 96
    x = torch.full((2, D), 3.25)
    beta = torch.linspace(-1, 1, D)
    out = torch.empty(2, D, dtype=torch.float32, device=DEV)
    ops.layernorm(x.to(DEV), torch.ones(D, device=DEV), beta.to(DEV), 1e-6, out)
    assert (out.cpu() - beta).abs().max() <= 1e-6


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("M,N,K", [(67, 79, 40), (5, 2304, 768), (1, 1000, 96), (130, 320, 96),
                                   (9, 73, 320), (200, 50257, 64), (33, 96, 3072), (257, 257, 264),
                                   (300, 4800, 1600), (100, 1600, 6400)])
@pytest.mark.parametrize("epi", ["store", "gelu_tanh", "gelu_erf", "add_residual", "store_f32"])
def test_linear(ops, dtype, M, N, K, epi):
    if N == 50257 and epi not in ("store_f32", "store"):
        pytest.skip("the wide case is the logits head")
    g = torch.Generator().manual_seed(M * 1000 + N + K)
    a = _rand((M, K), dtype, g)
    w = _rand((N, K), dtype, g, std=1.0 / math.sqrt(K))
    bias = 0.5 * _rand((N,), torch.float32, g)
    f32_out = epi in ("add_residual", "store_f32")
    out0 = _rand((M, N), torch.float32 if f32_out else dtype, g)
    out = out0.clone().to(DEV)
    ops.linear(a.to(DEV), w.to(DEV), bias.to(DEV), out, epi)
    ref = plain_ops.linear(a, w, bias, out0.double().clone(), epi)
    err = (out.cpu().double() - ref).abs().max().item()
    tol = 3e-5 if dtype == torch.float32 else (2e-5 + 2e-5 * math.sqrt(K) if f32_out else 4e-2)
    assert err <= tol, (err, tol)
    # no bias, strided input rows
    a2 = _rand((M, K + 8), dtype, g).to(DEV)[:, :K]
    out = out0.clone().to(DEV)
    ops.linear(a2, w.to(DEV), None, out, epi)
    ref = plain_ops.linear(a2.cpu(), w, None, out0.double().clone(), epi)
    assert (out.cpu().double() - ref).abs().max().item() <= tol


@pytest.mark.parametrize("M,N,K", [(2000, 2300, 776),      # 128x192 tiles, one round, ragged in M, N and K
                                   (2048, 3072, 768),      # 128x192 tiles, no edge
                                   (2900, 3000, 72),       # 128x192 tiles, two rounds, ragged
                                   (2040, 4090, 136),      # 128x256 tiles, ragged
                                   (2040, 1800, 200),      # 128x128 tiles, one round, ragged
                                   (2040, 1000, 200),      # 64x128 tiles, ragged
                                   (2040, 760, 136),       # 64x96 tiles, one round, ragged
                                   (2048, 768, 3072),      # 64x96 tiles, long K: two wavefront groups per workgroup
                                   (2040, 1800, 2056),     # 128x128 tiles, two groups, K not a multiple of their k tile
                                   (1000, 1000, 2056),     # 64x64 tiles, two groups, ragged
                                   (300, 500, 4104),       # 64x32 tiles (few workgroups), long ragged K
                                   (1000, 1000, 40),       # 64x64 tiles, K below one k tile
                                   (257, 257, 264)])       # 64x32 tiles, few workgroups
@pytest.mark.parametrize("epi", ["store", "add_residual"])
def test_linear_bf16_tile_choices(ops, M, N, K, epi):
    """Every tile shape of the many-row product, with edges in all three dimensions."""
    g = torch.Generator().manual_seed(M + 3 * N + 7 * K)
    a = _rand((M, K), torch.bfloat16, g)
    w = _rand((N, K), torch.bfloat16, g, std=1.0 / math.sqrt(K))
    bias = 0.5 * _rand((N,), torch.float32, g)
    f32_out = epi == "add_residual"
    out0 = _rand((M, N), torch.float32 if f32_out else torch.bfloat16, g)
    out = out0.clone().to(DEV)
    ops.linear(a.to(DEV), w.to(DEV), bias.to(DEV), out, epi)
    ref = plain_ops.linear(a, w, bias, out0.double().clone(), epi)
    err = (out.cpu().double() - ref).abs().max().item()
    assert err <= (2e-5 + 2e-5 * math.sqrt(K) if f32_out else 4e-2), err


@pytest.mark.parametrize("M,N", [(33, 40), (100, 768), (260, 1000), (520, 772), (1000, 1024), (1030, 3072), (2100, 2300), (2048, 6400)])
@pytest.mark.parametrize("K", [8, 56, 64, 72, 136, 200, 328, 2048, 2056, 2120, 2184])
def test_linear_bf16_stages_and_remainders(ops, M, N, K):
    """Products on every tile, with fewer k tiles than stages and with 8 to 64 columns in the last: every element against the
    sum in fp32 of the same bfloat16 values. Rounding to bfloat16 is 2^-9 of the result (2^-8 allowed), the sums' own order K^0.5 2^-24 of the terms."""
    g = torch.Generator().manual_seed(M + N + K)
    a, w = _rand((M, K), torch.bfloat16, g), _rand((N, K), torch.bfloat16, g, K ** -0.5)
    bias = _rand((N,), torch.float32, g)
    want = a.to(DEV).float() @ w.to(DEV).float().T + bias.to(DEV)
    out = torch.full((M, N), float("nan"), dtype=torch.bfloat16, device=DEV)
    ops.linear(a.to(DEV), w.to(DEV), bias.to(DEV), out)
    assert bool(((out.float() - want).abs() <= 2.0 ** -8 * want.abs() + 1e-4).all())
    x = _rand((M, N), torch.float32, g).to(DEV)
    got = x.clone()
    ops.linear(a.to(DEV), w.to(DEV), bias.to(DEV), got, "add_residual")
    assert bool(((got - (x + want)).abs() <= 1e-4).all())


@pytest.mark.parametrize("M,N,K", [(33, 1001, 72), (100, 37, 200), (260, 1003, 776), (300, 70, 2048), (520, 771, 2056), (1030, 3001, 72), (2100, 2305, 200)])
@pytest.mark.parametrize("start", [0, 1, 3])
def test_linear_bf16_rows_that_start_anywhere(ops, M, N, K, start):
    """16-bit results whose rows are no multiple of 8 bytes apart, or whose first element is not aligned, to the bit as in aligned rows (every
    tile, every epilogue that stores 16 bits), and nothing beside them is written."""
    import ctypes
    g = torch.Generator().manual_seed(M + N + K)
    a, w, up = (_rand((n, K), torch.bfloat16, g, s).to(DEV) for n, s in ((M, 1), (N, K ** -0.5), (N, K ** -0.5)))
    bias = _rand((N,), torch.float32, g).to(DEV)
    stride, even = N + 2 + (N % 2 == 0), (N + 15) // 8 * 8
    assert stride % 2 == 1

    def rooms():
        odd = torch.full((start + (M + 1) * stride,), 7.0, dtype=torch.bfloat16, device=DEV)[start:].view(M + 1, stride)
        return torch.full((M, even), 7.0, dtype=torch.bfloat16, device=DEV), odd

    def check(near, odd, what):
        assert torch.equal(near[:, :N], odd[:M, :N]), what
        assert bool((odd[:M, N:] == 7).all()) and bool((odd[M] == 7).all()), what

    for epilogue in ("store", "gelu_tanh", "gelu_erf"):
        near, odd = rooms()
        ops.linear(a, w, bias, near[:, :N], epilogue)
        ops.linear(a, w, bias, odd[:M, :N], epilogue)
        check(near, odd, epilogue)
    vp, i, f = ctypes.c_void_p, ctypes.c_int, ctypes.c_float
    fn = ops.engine_library().mllm_gated_gemm_bf16
    fn.argtypes = [vp, i, vp, vp, i, f, f, vp, i, i, i, i, vp]
    near, odd = rooms()
    for out, ld in ((near, even), (odd, stride)):
        assert fn(a.data_ptr(), K, w.data_ptr(), up.data_ptr(), K, 7.0, 1.702, out.data_ptr(), ld, M, N, K, None) == 0
    torch.cuda.synchronize()
    check(near, odd, "gated")


@pytest.mark.parametrize("M,N", [(2048, 16384), (1024, 16384), (8192, 2048)])
def test_linear_bf16_short_sums_are_not_slower(ops, M, N):
    """The tile chosen for few columns of K suits them: products of 64 take no longer than those of 512 (half as long is usual; 1.4
    times as long were those on tiles priced far outside what the prices know)."""
    took = {}
    for K in (64, 512):
        a, w = (torch.randn(n, K, device=DEV).bfloat16() for n in (M, N))
        out = torch.empty(M, N, dtype=torch.bfloat16, device=DEV)
        marks = [torch.cuda.Event(enable_timing=True) for _ in range(12)]
        for m in marks:
            ops.linear(a, w, None, out)
            m.record()
        torch.cuda.synchronize()
        took[K] = sorted(x.elapsed_time(y) for x, y in zip(marks[2:], marks[3:]))[4]
    assert took[64] <= took[512], took


@pytest.mark.parametrize("M,N", [(300, 40), (520, 772), (1030, 3072), (2100, 2300)])
def test_linear_bf16_of_no_columns(ops, M, N):
    """A product on tiles that has no k tile asks for none: the bias alone, on every tile, and the old values stay."""
    import ctypes
    vp, i = ctypes.c_void_p, ctypes.c_int
    fn = ops.engine_library().mllm_gemm_bf16
    fn.argtypes = [vp, i, vp, i, vp, vp, i, i, i, i, i, vp, ctypes.c_size_t, vp]
    g = torch.Generator().manual_seed(M + N)
    bias, x = _rand((N,), torch.float32, g).to(DEV), _rand((M, N), torch.float32, g).to(DEV)
    row = torch.zeros(64, dtype=torch.bfloat16, device=DEV)
    for mode, out, want in ((0, torch.empty(M, N, dtype=torch.bfloat16, device=DEV), bias.bfloat16().expand(M, N)), (3, x.clone(), x + bias)):
        assert fn(row.data_ptr(), 0, row.data_ptr(), 0, bias.data_ptr(), out.data_ptr(), N, M, N, 0, mode, None, 0, None) == 0
        torch.cuda.synchronize()
        assert torch.equal(out, want), mode


@pytest.mark.parametrize("N,K,rows", [(1000, 2120, (260, 520, 1030, 1300, 2100)),      # sums in halves: 64x32, 64x64, 64x96, 64x128, 128x128
                                      (1600, 2056, (260, 520, 1300, 2100)),            # and 128x192
                                      (2304, 776, (260, 400, 800, 1700, 2600))])       # in one: 64x64 to 128x256
@pytest.mark.parametrize("epi", ["store", "add_residual"])
def test_linear_bf16_tiles_add_in_one_order(ops, N, K, rows, epi):
    """Row counts that take different tiles, with sums of one kind: the rows they share have the same bits."""
    g = torch.Generator().manual_seed(N + K)
    a, w = _rand((max(rows), K), torch.bfloat16, g).to(DEV), _rand((N, K), torch.bfloat16, g, K ** -0.5).to(DEV)
    bias, x = _rand((N,), torch.float32, g).to(DEV), _rand((max(rows), N), torch.float32, g).to(DEV)
    first = None
    for M in rows:
        out = x[:M].clone() if epi == "add_residual" else torch.empty(M, N, dtype=torch.bfloat16, device=DEV)
        ops.linear(a[:M], w, bias, out, epi)
        first = out if first is None else first
        assert torch.equal(out[:rows[0]], first), M


@pytest.mark.parametrize("M,N,K,far", [(17, 48, 200, "aw"),             # few rows
                                       (2, 16404, 4096, "a"),           # of a width that the few-row kernel refuses
                                       (300, 48, 200, "aw"), (300, 48, 2056, "aw"), (300, 48, 2048, "w"),     # sums in halves
                                       (200, 4104, 200, "a"), (200, 4104, 2056, "a")])                        # and in one
def test_linear_bf16_rows_far_apart(ops, M, N, K, far):
    """Rows more than 2^23 elements apart, where a tile's 32-bit offsets end: every form of the product gives the bits it gives for
    the same rows side by side."""
    import ctypes
    stride = (1 << 23) + 8
    g = torch.Generator().manual_seed(M + N + K)

    def apart(t):
        out = torch.empty((t.shape[0] - 1) * stride + K, dtype=t.dtype, device=DEV).as_strided(t.shape, (stride, 1))
        return out.copy_(t)

    a, w, up = (_rand((n, K), torch.bfloat16, g, s).to(DEV) for n, s in ((M, 1), (N, K ** -0.5), (N, K ** -0.5)))
    bias, x = _rand((N,), torch.float32, g).to(DEV), _rand((M, N), torch.float32, g).to(DEV)
    a2, w2, up2 = apart(a) if "a" in far else a, apart(w) if "w" in far else w, apart(up) if "w" in far else up
    for epilogue in ("store", "gelu_tanh", "gelu_erf", "add_residual", "store_f32"):
        got = [x.clone() if epilogue in ("add_residual", "store_f32") else x.bfloat16() for _ in range(2)]
        ops.linear(a, w, bias, got[0], epilogue)
        ops.linear(a2, w2, bias, got[1], epilogue)
        assert torch.equal(*got), epilogue
    kv = N // 3 // 4 * 4
    pages, got = [[torch.zeros(M, kv, dtype=torch.bfloat16, device=DEV) for _ in range(2)] for _ in range(2)], [x.bfloat16() for _ in range(2)]
    slots = torch.randperm(M, generator=g).to(torch.int32).to(DEV)
    ops.linear(a, w, bias, got[0], "store", kv_scatter=(slots, *pages[0], N - 2 * kv))
    ops.linear(a2, w2, bias, got[1], "store", kv_scatter=(slots, *pages[1], N - 2 * kv))
    assert torch.equal(*got) and all(torch.equal(*p) for p in zip(*pages))
    streams, copies, rooms = [x.clone() for _ in range(2)], [x.bfloat16() for _ in range(2)], [torch.empty_like(x) for _ in range(2)]
    ops.linear_stream_add(a, w, streams[0], bias, rooms[0], copy=copies[0])
    ops.linear_stream_add(a2, w2, streams[1], bias, rooms[1], copy=copies[1])
    assert torch.equal(*streams) and torch.equal(*copies)
    vp, i, f = ctypes.c_void_p, ctypes.c_int, ctypes.c_float
    fn = ops.engine_library().mllm_gated_gemm_bf16
    fn.argtypes = [vp, i, vp, vp, i, f, f, vp, i, i, i, i, vp]
    got = [torch.full((M, N), float("nan"), dtype=torch.bfloat16, device=DEV) for _ in range(2)]
    for out, (p, q, r) in zip(got, ((a, w, up), (a2, w2, up2))):
        assert fn(p.data_ptr(), p.stride(0), q.data_ptr(), r.data_ptr(), q.stride(0), 7.0, 1.702, out.data_ptr(), N, M, N, K, None) == 0
    torch.cuda.synchronize()
    assert torch.equal(*got)


@pytest.mark.parametrize("M,H,Hkv,dh,K", [(2048, 12, 12, 64, 768),      # 128x192 tiles
                                          (300, 6, 2, 16, 96),         # 64x64 tiles, ragged, grouped heads
                                          (70, 3, 3, 48, 144),         # just above the few-row kernel
                                          (1000, 16, 4, 32, 520)])
def test_linear_bf16_scatters_keys_and_values(ops, M, H, Hkv, dh, K):
    """The fused QKV product with the page write in its epilogue: output as without, and the key
    and value columns of every row with a slot arrive in that row of the pages, nothing else."""
    g = torch.Generator().manual_seed(M + K)
    q_cols, kv_dim = H * dh, Hkv * dh
    N = q_cols + 2 * kv_dim
    a = _rand((M, K), torch.bfloat16, g)
    w = _rand((N, K), torch.bfloat16, g, std=1.0 / math.sqrt(K))
    bias = 0.5 * _rand((N,), torch.float32, g)
    rows = M + 37
    perm = torch.randperm(rows, generator=g)[:M].to(torch.int32)
    perm[::7] = -1                                   # rows that write nothing
    k0 = _rand((rows, kv_dim), torch.bfloat16, g)
    v0 = _rand((rows, kv_dim), torch.bfloat16, g)
    kp, vp = k0.clone().to(DEV), v0.clone().to(DEV)
    out = torch.empty((M, N), dtype=torch.bfloat16, device=DEV)
    ops.linear(a.to(DEV), w.to(DEV), bias.to(DEV), out, "store", kv_scatter=(perm.to(DEV), kp, vp, q_cols))
    plain = torch.empty((M, N), dtype=torch.bfloat16, device=DEV)
    ops.linear(a.to(DEV), w.to(DEV), bias.to(DEV), plain, "store")
    if M > 256:
        assert torch.equal(out, plain)               # the same kernel with and without the page write
    else:                                            # without, fewer rows may take the weight-streaming kernel
        assert (out.float() - plain.float()).abs().max().item() <= 4e-2
    ref = plain_ops.linear(a, w, bias, torch.empty((M, N), dtype=torch.float64))
    assert (out.cpu().double() - ref).abs().max().item() <= 4e-2
    kr, vr = k0.clone(), v0.clone()
    plain_ops.kv_append(out.cpu(), q_cols, q_cols + kv_dim, kv_dim, kr, vr, perm)
    assert torch.equal(kp.cpu(), kr) and torch.equal(vp.cpu(), vr)
    # few rows: the product's kernel has no such epilogue and a copy kernel follows it; same contract
    kp8, vp8 = k0.clone().to(DEV), v0.clone().to(DEV)
    ops.linear(a[:8].to(DEV), w.to(DEV), bias.to(DEV), out[:8], "store", kv_scatter=(perm[:8].to(DEV), kp8, vp8, q_cols))
    kr, vr = k0.clone(), v0.clone()
    plain_ops.kv_append(out[:8].cpu(), q_cols, q_cols + kv_dim, kv_dim, kr, vr, perm[:8])
    assert torch.equal(kp8.cpu(), kr) and torch.equal(vp8.cpu(), vr)
    with pytest.raises(ops.KernelError, match="scatter"):
        ops.linear(a.to(DEV), w.to(DEV), None, torch.empty((M, N), dtype=torch.float32, device=DEV), "store_f32",
                   kv_scatter=(perm.to(DEV), kp, vp, q_cols))


@pytest.mark.parametrize("M,H,Hkv,dh,K", [(65, 12, 12, 64, 768), (256, 25, 25, 64, 1600), (100, 6, 2, 32, 200), (8, 4, 4, 16, 64),
                                          (64, 12, 12, 64, 768), (300, 3, 3, 32, 96)])
def test_ln_linear_scatters_keys_and_values(ops, M, H, Hkv, dh, K):
    """The norm, the QKV product and the page write in one call: the output of the norm followed by the
    product, and the key and value columns in their slots."""
    g = torch.Generator().manual_seed(M + K)
    q_cols, kv_dim = H * dh, Hkv * dh
    N = q_cols + 2 * kv_dim
    x = _rand((M, K), torch.float32, g, std=2.0) + 0.3
    gamma, beta = 1 + 0.1 * _rand((K,), torch.float32, g), 0.1 * _rand((K,), torch.float32, g)
    w = _rand((N, K), torch.bfloat16, g, std=1.0 / math.sqrt(K))
    bias = 0.5 * _rand((N,), torch.float32, g)
    rows = M + 37
    slots = torch.randperm(rows, generator=g)[:M].to(torch.int32)
    slots[::7] = -1
    k0, v0 = _rand((rows, kv_dim), torch.bfloat16, g), _rand((rows, kv_dim), torch.bfloat16, g)
    kp, vp = k0.clone().to(DEV), v0.clone().to(DEV)
    out = torch.empty((M, N), dtype=torch.bfloat16, device=DEV)
    ops.ln_linear(x.to(DEV), gamma.to(DEV), beta.to(DEV), 1e-5, w.to(DEV), bias.to(DEV), out, "store",
                  kv_scatter=(slots.to(DEV), kp, vp, q_cols))
    h = plain_ops.layernorm(x, gamma, beta, 1e-5, torch.empty(M, K, dtype=torch.bfloat16))
    ref = plain_ops.linear(h, w, bias, torch.empty((M, N), dtype=torch.float64))
    assert (out.cpu().double() - ref).abs().max().item() <= 4e-2
    kr, vr = k0.clone(), v0.clone()
    plain_ops.kv_append(out.cpu(), q_cols, q_cols + kv_dim, kv_dim, kr, vr, slots)
    assert torch.equal(kp.cpu(), kr) and torch.equal(vp.cpu(), vr)


@pytest.mark.parametrize("M,H,Hkv,dh,K", [(1, 12, 12, 64, 768), (7, 12, 3, 64, 768), (16, 25, 25, 64, 1600),     # (two column tiles a workgroup)
                                          (17, 12, 12, 64, 768), (32, 5, 1, 40, 96), (33, 6, 2, 32, 200),
                                          (17, 25, 25, 64, 1600), (32, 22, 21, 64, 256), (32, 22, 22, 64, 256),      # (both sides of 4,096 columns)
                                          (9, 3, 3, 10, 64), (40, 3, 3, 10, 64),                     # widths that are no multiple of 4
                                          (3, 2, 2, 16, 100)])                                       # K that is no multiple of 8
def test_ln_linear_scatters_few_rows(ops, M, H, Hkv, dh, K):
    """The same from the few-row product's epilogue (with the norm inside up to 32 rows), and where it does not take the sizes."""
    test_ln_linear_scatters_keys_and_values(ops, M, H, Hkv, dh, K)


@pytest.mark.parametrize("M", [1, 8, 16, 17, 48, 64])
@pytest.mark.parametrize("N,K", [(2304, 768), (768, 3072), (1000, 96), (50257, 768), (72, 1600), (4800, 1600),
                                 (1600, 6400), (1024, 4096),
                                 # more than 256 tiles of 16 columns: two tiles per workgroup, the second narrower
                                 (4104, 72), (6400, 1600), (8190, 200)])
def test_linear_bf16_few_rows(ops, M, N, K):
    """The weight-streaming kernel of decode steps (M <= 64), every wavefront count and m-tile count."""
    g = torch.Generator().manual_seed(M + N + K)
    a = _rand((M, K), torch.bfloat16, g)
    w = _rand((N, K), torch.bfloat16, g, std=1.0 / math.sqrt(K))
    bias = 0.5 * _rand((N,), torch.float32, g)
    for epi in ("store_f32", "add_residual", "gelu_tanh"):
        f32_out = epi != "gelu_tanh"
        out0 = _rand((M, N), torch.float32 if f32_out else torch.bfloat16, g)
        out = out0.clone().to(DEV)
        ops.linear(a.to(DEV), w.to(DEV), bias.to(DEV), out, epi)
        ref = plain_ops.linear(a, w, bias, out0.double().clone(), epi)
        err = (out.cpu().double() - ref).abs().max().item()
        assert err <= (2e-5 + 2e-5 * math.sqrt(K) if f32_out else 4e-2), (epi, err)


@pytest.mark.parametrize("M", [1, 8, 9, 16])
@pytest.mark.parametrize("N,K", [(96, 2304), (96, 2312), (96, 3072), (96, 3080), (96, 3136), (40, 64), (40, 5056), (4104, 768), (4104, 776), (4104, 832)])
def test_linear_bf16_few_rows_at_the_chunks_borders(ops, M, N, K):
    """A wavefront's blocks of K that fill one chunk, the next block, and part of one: kernels of one chunk and of several."""
    test_linear_bf16_few_rows(ops, M, N, K)


@pytest.mark.parametrize("M,N,K", [(65, 768, 768), (96, 2304, 768), (100, 1000, 96), (128, 768, 3072), (200, 72, 1600),
                                   (256, 768, 768), (256, 1024, 4096), (250, 40, 6400), (129, 2304, 768), (64, 6400, 1600)])
def test_linear_bf16_up_to_256_rows(ops, M, N, K):
    """Between 65 and 256 rows the weight-streaming kernel (many 16-row blocks) or the tiled kernel
    runs, by the number of workgroups the former would need."""
    g = torch.Generator().manual_seed(M + N + K)
    a = _rand((M, K), torch.bfloat16, g)
    w = _rand((N, K), torch.bfloat16, g, std=1.0 / math.sqrt(K))
    bias = 0.5 * _rand((N,), torch.float32, g)
    for epi in ("store", "add_residual", "gelu_erf"):
        f32_out = epi == "add_residual"
        out0 = _rand((M, N), torch.float32 if f32_out else torch.bfloat16, g)
        out = out0.clone().to(DEV)
        ops.linear(a.to(DEV), w.to(DEV), bias.to(DEV), out, epi)
        ref = plain_ops.linear(a, w, bias, out0.double().clone(), epi)
        err = (out.cpu().double() - ref).abs().max().item()
        assert err <= (2e-5 + 2e-5 * math.sqrt(K) if f32_out else 4e-2), (epi, err)


@pytest.mark.parametrize("M,N,K", [(8, 1600, 6400), (1, 1280, 5120), (16, 72, 8192), (5, 200, 5192), (32, 40, 6400),
                                   (64, 24, 5128)])
def test_linear_bf16_few_rows_long_k_shares_tiles(ops, M, N, K):
    """Narrow products with a long K: several workgroups share a tile and the last to arrive adds their
    parts. Every call gives the same bits (the parts are added in a fixed order, the counters are
    left at zero), on any stream."""
    g = torch.Generator().manual_seed(M + N + K)
    a = _rand((M, K), torch.bfloat16, g).to(DEV)
    w = _rand((N, K), torch.bfloat16, g, std=1.0 / math.sqrt(K)).to(DEV)
    bias = (0.5 * _rand((N,), torch.float32, g)).to(DEV)
    x0 = _rand((M, N), torch.float32, g)
    ref = plain_ops.linear(a.cpu(), w.cpu(), bias.cpu(), x0.double().clone(), "add_residual")
    outs = []
    for _ in range(3):
        x = x0.clone().to(DEV)
        ops.linear(a, w, bias, x, "add_residual")
        outs.append(x.cpu())
    assert (outs[0].double() - ref).abs().max().item() <= 2e-5 + 2e-5 * math.sqrt(K)
    assert torch.equal(outs[0], outs[1]) and torch.equal(outs[0], outs[2])
    # another epilogue between two runs, and a second stream with scratch of its own: the same bits again
    y = torch.empty(M, N, dtype=torch.bfloat16, device=DEV)
    ops.linear(a, w, bias, y, "gelu_tanh")
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        x = x0.clone().to(DEV)
        ops.linear(a, w, bias, x, "add_residual")
        assert ops.scratch_address("gemm_workspace") != 0
    side.synchronize()
    assert torch.equal(x.cpu(), outs[0])


@pytest.mark.parametrize("M", [1, 3, 8])
@pytest.mark.parametrize("N", [12, 767, 1030, 1500, 2040, 2050])          # 4, 4, 5, 6, 8 and 9 columns a workgroup
@pytest.mark.parametrize("K", [3016, 3072, 3080, 4104, 5000])             # 48 to 79 k blocks: one chunk a wavefront, a second one with 1 to 3 left
def test_linear_bf16_few_rows_of_narrow_tiles(ops, M, N, K):
    """Products with a long K whose columns are dealt out in fewer than 16 a workgroup: each result next to the plain one, and a row has the
    same bits alone, among others, and among so many that another kernel of the same sums takes them."""
    g = torch.Generator().manual_seed(M + N + K)
    a = _rand((9, K), torch.bfloat16, g)
    w = _rand((N, K), torch.bfloat16, g, std=1.0 / math.sqrt(K))
    bias = 0.5 * _rand((N,), torch.float32, g)
    x0 = _rand((9, N), torch.float32, g)
    outs = []
    for rows in (M, 9):
        x = x0[:rows].clone().to(DEV)
        ops.linear(a[:rows].to(DEV), w.to(DEV), bias.to(DEV), x, "add_residual")
        outs.append(x.cpu())
    assert torch.equal(outs[0], outs[1][:M])
    want = x0[:M].double() + a[:M].double() @ w.double().T + bias.double()
    # fp32 sums: at most one rounding of 2^-24 for every eighth of the terms and of their magnitude, and a few for bias and residual
    bound = 2.0 ** -24 * (K / 8 + 8) * (a[:M].double().abs() @ w.double().abs().T + x0[:M].double().abs() + bias.double().abs())
    assert ((outs[0].double() - want).abs() <= bound).all()


@pytest.mark.parametrize("M", [1, 3, 8])
@pytest.mark.parametrize("N,K", [(1361, 5128), (1600, 6400), (2048, 5120), (2040, 7000), (1500, 9216), (1500, 9224)])
def test_linear_bf16_few_rows_with_both_parts_of_k_inside(ops, M, N, K):
    """Long sums in two parts: up to 8 rows one workgroup has both (a chunk of 4 to 6 blocks of K each), from 9 on two share a tile. The same bits."""
    test_linear_bf16_few_rows_of_narrow_tiles(ops, M, N, K)


@pytest.mark.parametrize("M", [17, 25, 32])
@pytest.mark.parametrize("N,K", [(2048, 768), (2049, 768), (2304, 768), (2500, 1024), (4096, 768), (4097, 768), (4097, 1032), (6400, 1600)])
@pytest.mark.parametrize("epi", ["store", "gelu_tanh"])
def test_ln_linear_two_tiles_a_workgroup(ops, M, N, K, epi):
    """17 to 32 rows behind the fused norm, where a workgroup has one tile of columns and where it has two, the second narrower: which rows
    share a launch does not change a bit."""
    g = torch.Generator().manual_seed(M + N + K)
    x = (_rand((M, K), torch.float32, g, std=2.0) + 0.3).to(DEV)
    gamma, beta = (1 + 0.1 * _rand((K,), torch.float32, g)).to(DEV), (0.1 * _rand((K,), torch.float32, g)).to(DEV)
    w, bias = _rand((N, K), torch.bfloat16, g, std=1.0 / math.sqrt(K)).to(DEV), (0.5 * _rand((N,), torch.float32, g)).to(DEV)
    out, parts = (torch.full((M, N), 7.0, dtype=torch.bfloat16, device=DEV) for _ in range(2))
    ops.ln_linear(x, gamma, beta, 1e-5, w, bias, out, epi)
    for m in range(0, M, 16):
        ops.ln_linear(x[m:m + 16], gamma, beta, 1e-5, w, bias, parts[m:m + 16], epi)
    assert torch.equal(out, parts)
    ref = plain_ops.ln_linear(x.cpu(), gamma.cpu(), beta.cpu(), 1e-5, w.cpu(), bias.cpu(), torch.empty(M, N, dtype=torch.float64), epi)
    assert (out.cpu().double() - ref).abs().max().item() <= 4e-2


@pytest.mark.parametrize("M", [1, 16, 17, 32])
@pytest.mark.parametrize("N", [2304, 4096, 4112, 8192])
@pytest.mark.parametrize("K", [2008, 2016, 2024, 2048])
@pytest.mark.parametrize("rms", [False, True])
def test_norm_and_product_in_one_kernel_up_to_2048_columns(ops, M, N, K, rms):
    """The kernel itself, without room for normalised rows: from K = 2,024 on two tiles of columns do not fit a workgroup's LDS, and it takes the
    same sizes with one. Which rows share a launch does not change a bit. The op is as close to the reference on either way."""
    import ctypes
    from mini_llm_amd import build
    lib = build.load_library("gemm_bf16")
    g = torch.Generator().manual_seed(M + N + K)
    x = (_rand((M, K), torch.float32, g, std=2.0) + 0.3).to(DEV)
    gamma, beta = (1 + 0.1 * _rand((K,), torch.float32, g)).to(DEV), (0.1 * _rand((K,), torch.float32, g)).to(DEV)
    w, bias = _rand((N, K), torch.bfloat16, g, std=1.0 / math.sqrt(K)).to(DEV), (0.5 * _rand((N,), torch.float32, g)).to(DEV)

    def run(m0, m1, out):
        p, i = (lambda t: ctypes.c_void_p(t.data_ptr())), ctypes.c_int
        f, norm = (lib.mllm_rms_gemm_bf16, [p(gamma)]) if rms else (lib.mllm_ln_gemm_bf16, [p(gamma), p(beta)])
        assert f(p(x[m0:]), i(K), ctypes.c_void_p(0), *norm, ctypes.c_float(1e-5), p(w), i(K), p(bias), p(out[m0:]), i(N), i(m1 - m0), i(N), i(K), i(0),
                 ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)) == 0

    out, parts = (torch.full((M, N), 7.0, dtype=torch.bfloat16, device=DEV) for _ in range(2))
    run(0, M, out)
    for m in range(M):
        run(m, m + 1, parts)
    assert torch.equal(out, parts)
    x64 = x.double() - (0.0 if rms else x.double().mean(1, keepdim=True))
    h = x64 / torch.sqrt((x64 * x64).mean(1, keepdim=True) + 1e-5) * gamma.double() + (0.0 if rms else beta.double())
    want = h @ w.double().T + bias.double()
    assert (out.double() - want).abs().max().item() <= 4e-2
    if not rms:
        ops.ln_linear(x, gamma, beta, 1e-5, w, bias, out, "store")
        assert (out.double() - want).abs().max().item() <= 4e-2


@pytest.mark.parametrize("M", [17, 32])
@pytest.mark.parametrize("N,K", [(2064, 2024), (2304, 2048), (4096, 2048), (8208, 2024)])
def test_ln_linear_of_17_to_32_wide_rows_has_the_bits_of_16(ops, M, N, K):
    """From K = 2,024 on the norm stays inside the product for 17 to 32 rows: a row has the bits that it has among up to 16."""
    g = torch.Generator().manual_seed(M + N + K)
    x = (_rand((M, K), torch.float32, g, std=2.0) + 0.3).to(DEV)
    gamma, beta = (1 + 0.1 * _rand((K,), torch.float32, g)).to(DEV), (0.1 * _rand((K,), torch.float32, g)).to(DEV)
    w, bias = _rand((N, K), torch.bfloat16, g, std=1.0 / math.sqrt(K)).to(DEV), (0.5 * _rand((N,), torch.float32, g)).to(DEV)
    out, parts = (torch.full((M, N), 7.0, dtype=torch.bfloat16, device=DEV) for _ in range(2))
    ops.ln_linear(x, gamma, beta, 1e-5, w, bias, out, "store")
    for m in range(0, M, 16):
        ops.ln_linear(x[m:m + 16], gamma, beta, 1e-5, w, bias, parts[m:m + 16], "store")
    assert torch.equal(out, parts)


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("M,N,K", [(1, 2304, 768), (8, 3072, 768), (16, 320, 96), (5, 200, 1600), (17, 96, 64),
                                   (3, 64, 4096), (16, 6400, 1600), (9, 50257, 1024), (16, 3072, 1024), (33, 2304, 768),
                                   (64, 50257, 768), (64, 104, 1600), (65, 96, 64),
                                   # more than 256 tiles: two per workgroup
                                   (8, 4800, 1600), (3, 4104, 72), (16, 8190, 200),
                                   # more than 32 rows: the norm runs as a kernel of its own
                                   (64, 3072, 768), (48, 4096, 1024), (50, 136, 200), (100, 320, 96), (200, 4800, 1600),
                                   (256, 3072, 776), (17, 40, 72), (31, 1000, 2048), (300, 320, 96)])
@pytest.mark.parametrize("epi", ["store", "gelu_tanh", "gelu_erf", "store_f32"])
def test_ln_linear(ops, dtype, M, N, K, epi):
    """LayerNorm fused into the product (bf16, few rows) and its unfused form give the plain result."""
    g = torch.Generator().manual_seed(M * 7 + N + K)
    x = _rand((M, K), torch.float32, g, std=2.0) + 0.3
    gamma = 1 + 0.1 * _rand((K,), torch.float32, g)
    beta = 0.1 * _rand((K,), torch.float32, g)
    w = _rand((N, K), dtype, g, std=1.0 / math.sqrt(K))
    bias = 0.5 * _rand((N,), torch.float32, g)
    odt = torch.float32 if epi == "store_f32" else dtype
    out = torch.zeros(M, N, dtype=odt, device=DEV)
    ops.ln_linear(x.to(DEV), gamma.to(DEV), beta.to(DEV), 1e-5, w.to(DEV), bias.to(DEV), out, epi)
    h = plain_ops.layernorm(x, gamma, beta, 1e-5, torch.empty(M, K, dtype=dtype))     # rounded as the kernel rounds
    ref = plain_ops.linear(h, w, bias, torch.zeros(M, N, dtype=torch.float64), epi)
    tol = 3e-5 if dtype == torch.float32 else (2e-2 if epi == "store_f32" else 4e-2)
    assert (out.cpu().double() - ref).abs().max().item() <= tol
    # no bias, rows gathered in another order
    sel = torch.tensor(list(range(M - 1, -1, -1)), dtype=torch.int32)
    out2 = torch.zeros(M, N, dtype=odt, device=DEV)
    ops.ln_linear(x.to(DEV), gamma.to(DEV), None, 1e-5, w.to(DEV), None, out2, epi, rows=sel.to(DEV))
    h = plain_ops.layernorm(x, gamma, None, 1e-5, torch.empty(M, K, dtype=dtype), rows=sel)
    ref = plain_ops.linear(h, w, None, torch.zeros(M, N, dtype=torch.float64), epi)
    assert (out2.cpu().double() - ref).abs().max().item() <= tol


@pytest.mark.parametrize("K", [k for n in range(1, 9) for k in (256 * n - 8, 256 * n, 256 * n + 8)][:-1])
@pytest.mark.parametrize("M,N", [(1, 48), (9, 4104)])
def test_ln_linear_at_every_number_of_columns_a_lane(ops, M, N, K):
    """The product behind the norm has an instance for every 256 columns of K: around each, with one tile a workgroup and with two."""
    test_ln_linear(ops, torch.bfloat16, M, N, K, "store")


@pytest.mark.parametrize("M", [1, 2, 3, 8])
@pytest.mark.parametrize("N,K", [(2048, 4), (2050, 252), (2304, 256), (2048, 260), (2304, 768), (3072, 768), (4096, 1024), (4097, 772), (4800, 1600),
                                 (6400, 1600), (2056, 2044), (4104, 2048)])
@pytest.mark.parametrize("epi", ["store", "gelu_tanh"])
def test_ln_linear_fp32_inside_has_the_bits_of_norm_and_product(ops, monkeypatch, M, N, K, epi):
    """The 32-bit norm inside the few-row product, around every 256 columns a lane's share grows by: the bits of norm and product apart."""
    g = torch.Generator().manual_seed(M + N + K)
    x = (_rand((M, K), torch.float32, g, std=2.0) + 0.3).to(DEV)
    gamma, beta = (1 + 0.1 * _rand((K,), torch.float32, g)).to(DEV), (0.1 * _rand((K,), torch.float32, g)).to(DEV)
    w, bias = _rand((N, K), torch.float32, g, std=1.0 / math.sqrt(K)).to(DEV), (0.5 * _rand((N,), torch.float32, g)).to(DEV)
    inside, apart = (torch.full((M, N), 7.0, device=DEV) for _ in range(2))
    for b, c in ((beta, bias), (None, None)):
        ops.ln_linear(x, gamma, b, 1e-5, w, c, inside, epi)
        with monkeypatch.context() as m:
            m.setattr(ops, "LN_FUSE_MAX_ROWS", 0)
            ops.ln_linear(x, gamma, b, 1e-5, w, c, apart, epi)
        assert torch.equal(inside, apart)
    h = plain_ops.layernorm(x.cpu(), gamma.cpu(), None, 1e-5, torch.empty(M, K, dtype=torch.float64))
    ref = plain_ops.linear(h, w.cpu().double(), None, torch.zeros(M, N, dtype=torch.float64), epi)
    assert (inside.cpu().double() - ref).abs().max().item() <= 3e-5


@pytest.mark.parametrize("dtype,M,K", [(torch.float32, 1, 2048), (torch.float32, 8, 2048), (torch.bfloat16, 1, 768), (torch.bfloat16, 16, 768),
                                       (torch.bfloat16, 32, 1600)])
def test_ln_linear_over_its_own_rows(ops, dtype, M, K):
    """x += norm(x) W^T in place: a norm inside the product would read rows that other workgroups have added their results to."""
    g = torch.Generator().manual_seed(M + K)
    x = _rand((M, K), torch.float32, g, std=2.0)
    gamma, bias = (1 + 0.1 * _rand((K,), torch.float32, g)).to(DEV), (0.5 * _rand((K,), torch.float32, g)).to(DEV)
    w = _rand((K, K), dtype, g, std=1.0 / math.sqrt(K)).to(DEV)
    here, there = x.to(DEV), x.to(DEV)
    ops.ln_linear(here, gamma, None, 1e-5, w, bias, here, "add_residual")
    h = ops.layernorm(x.to(DEV), gamma, None, 1e-5, torch.empty(M, K, dtype=dtype, device=DEV))
    ops.linear(h, w, bias, there, "add_residual")
    assert torch.equal(here, there)


def test_linear_fp32_is_true_fp32(ops):
    """Values that bf16 or tf32 inputs would destroy: 1 + 2^-20 differs from 1 only in true fp32."""
    K = 64
    a = torch.ones(4, K)
    a[:, 0] = 1 + 2.0 ** -20
    w = torch.zeros(3, K)
    w[0, 0], w[0, 1] = 1.0, -1.0
    out = torch.empty(4, 3, device=DEV)
    ops.linear(a.to(DEV), w.to(DEV), None, out, "store")
    assert out[0, 0].item() == 2.0 ** -20


@pytest.mark.parametrize("M,N,K,pad", [(5, 70, 42, 0),        # K no multiple of 4: the tiled kernel
                                         (7, 33, 1028, 3),      # row strides no multiple of 4 floats
                                         (8, 50257, 64, 0),     # the few-row kernel, one pass, wide
                                         (64, 130, 1600, 0),    # four passes of 16 rows, k chunks with a rest
                                         (17, 5, 8, 4)])        # fewer columns than a workgroup has wavefronts
def test_linear_fp32_few_rows(ops, M, N, K, pad):
    """The 32-bit product of few rows streams the weights, one column per wavefront, where the operands
    are 16-byte aligned, and falls back to the tiled kernel where they are not."""
    g = torch.Generator().manual_seed(M + N + K)
    a = _rand((M, K + pad), torch.float32, g).to(DEV)[:, :K]
    w = _rand((N, K + pad), torch.float32, g, std=1.0 / math.sqrt(K)).to(DEV)[:, :K]
    bias = 0.5 * _rand((N,), torch.float32, g)
    for epi in ("store", "add_residual", "gelu_tanh"):
        out0 = _rand((M, N), torch.float32, g)
        out = out0.clone().to(DEV)
        ops.linear(a, w, bias.to(DEV), out, epi)
        ref = plain_ops.linear(a.cpu(), w.cpu(), bias, out0.double().clone(), epi)
        assert (out.cpu().double() - ref).abs().max().item() <= 3e-5


@pytest.mark.parametrize("M,N,K,pad,tiles", [(17, 40, 4, 0, "32 x 32, two groups"), (33, 97, 100, 4, "32 x 32, two groups"), (64, 193, 772, 0, "32 x 32, two groups"),
                                             (64, 193, 1540, 4, "32 x 32, four groups"),
                                             (9, 16400, 36, 0, "32 x 32, two groups"),            # few rows of a wide head
                                             (800, 700, 132, 8, "32 x 32, two groups"), (800, 700, 100, 8, "32 x 32, one group"),
                                             (1025, 800, 260, 0, "64 x 32"), (1900, 1500, 292, 0, "64 x 32"),
                                             (2049, 2308, 20, 4, "128 x 64"), (1812, 2050, 772, 4, "128 x 64"), (1813, 2050, 780, 0, "128 x 64"),
                                             (1801, 3073, 804, 0, "128 x 64"), (2048, 3072, 768, 0, "128 x 64")])
@pytest.mark.parametrize("epi", ["store", "gelu_tanh", "add_residual"])
def test_linear_fp32_tiles(ops, M, N, K, pad, tiles, epi):
    """Every tile shape of the 32-bit product at its edges (rows, columns and K that fill no tile, strides wider than the rows):
    an output's products pass through at most 16 roundings, one for each further 16 columns, and a few to join groups, bias and
    residual, so its error is at most that many units of 2^-24 of the sum of their magnitudes (GELU: at most 1.13 times as
    steep, and 8 units of its own result). A row of infinities leaves the others as they are."""
    assert _tiles32(M, N, K) == tiles
    g = torch.Generator().manual_seed(M + K)
    a, w, b = _rand((M, K + pad), torch.float32, g), _rand((N, K + pad), torch.float32, g, 0.1), _rand((N,), torch.float32, g)
    a[M // 2] = float("inf")
    old = _rand((M, N + pad), torch.float32, g)
    out = old.to(DEV)
    ops.linear(a.to(DEV)[:, :K], w.to(DEV)[:, :K], b.to(DEV), out[:, :N], epi)
    assert torch.equal(out[:, N:].cpu(), old[:, N:])
    keep = torch.arange(M) != M // 2
    a64, w64 = a[keep, :K].double(), w[:, :K].double()
    want = a64 @ w64.T + b.double()
    size = a64.abs() @ w64.abs().T + b.double().abs()
    if epi == "gelu_tanh":
        want = 0.5 * want * (1.0 + torch.tanh(0.7978845608 * (want + 0.044715 * want ** 3)))
    elif epi == "add_residual":
        want, size = want + old[keep, :N].double(), size + old[keep, :N].double().abs()
    limit = 2.0 ** -24 * (1.13 * (16 + -(-K // 16) + 8) * size + 8 * want.abs())
    assert ((out[:, :N].cpu()[keep].double() - want).abs() <= limit).all()
    assert not torch.isfinite(out[M // 2, :N]).any() or epi == "gelu_tanh"


@pytest.mark.parametrize("M,N,K0", [(33, 70, 0), (130, 96, 1536), (600, 1100, 0), (1812, 772, 0), (2049, 1540, 0)])
@pytest.mark.parametrize("K", [4, 32, 36, 64, 100, 128, 132, 160, 192, 228])
def test_linear_fp32_tiles_of_few_k_tiles(ops, M, N, K0, K):
    """Every tile shape with few k tiles, odd and even in number, with a last one that is full or not; all but 32 x 32 with four groups (which has
    at least twelve) also with fewer of them than stages of LDS. The error is at most one rounding of 2^-24 a term of the terms'
    absolute sum, and rows that lie apart are met."""
    K += K0
    g = torch.Generator().manual_seed(M + N + K)
    a, w = _rand((M, K + 8), torch.float32, g).to(DEV), _rand((N, K + 4), torch.float32, g).to(DEV)
    a[:, K:], w[:, K:] = math.inf, math.nan
    bias, out = _rand((N,), torch.float32, g).to(DEV), torch.full((M, N + 4), 7.0, device=DEV)
    ops.linear(a[:, :K], w[:, :K], bias, out[:, :N], "store")
    a, w = a[:, :K].double(), w[:, :K].double()
    assert ((out[:, :N].double() - (a @ w.T + bias.double())).abs() <= 2.0 ** -24 * (K + 2) * (a.abs() @ w.abs().T + bias.abs().double())).all()
    assert (out[:, N:] == 7).all()


TILES32 = ("32 x 32, four groups", "32 x 32, two groups", "32 x 32, one group", "64 x 32", "128 x 64")      # TileShape of gemm_f32.hip


def _tiles32(M, N, K):
    from mini_llm_amd import build
    return TILES32[build.load_library("gemm_f32").mllm_gemm_f32_tile_shape(M, N, K)]


@pytest.mark.parametrize("M,N,K,tiles,few,few_tiles", [
    *[(600, 1100, k, "32 x 32, one group", 64, "32 x 32, two groups") for k in (4, 32, 36, 60, 64)],
    *[(600, 1100, k, "32 x 32, one group", 0, "") for k in (68, 96, 100, 128)], (600, 1100, 132, "32 x 32, two groups", 0, ""),
    *[(2049, 1540, k, "128 x 64", 1500, "64 x 32") for k in (4, 28, 32, 36, 48)], (2049, 1540, 52, "64 x 32", 1500, "64 x 32")])
def test_linear_fp32_tiles_of_short_sums(ops, M, N, K, tiles, few, few_tiles):
    """Short sums on the tiles that are the shorter way there: the same bits as on the others where the sums are the same (`few` of the rows
    run on other tiles), and at most one rounding of 2^-24 a term of the terms' absolute sum everywhere."""
    assert _tiles32(M, N, K) == tiles
    g = torch.Generator().manual_seed(M + N + K)
    a, w, bias = _rand((M, K), torch.float32, g).to(DEV), _rand((N, K), torch.float32, g).to(DEV), _rand((N,), torch.float32, g).to(DEV)
    out = torch.full((M, N + 4), 7.0, device=DEV)
    ops.linear(a, w, bias, out[:, :N], "store")
    assert (out[:, N:] == 7).all()
    want, size = a.double() @ w.double().T + bias.double(), a.double().abs() @ w.double().abs().T + bias.double().abs()
    assert ((out[:, :N].double() - want).abs() <= 2.0 ** -24 * (K + 2) * size).all()
    if few:
        assert _tiles32(few, N, K) == few_tiles
        part = torch.empty(few, N, device=DEV)
        ops.linear(a[:few], w, bias, part, "store")
        assert torch.equal(part, out[:few, :N])


@pytest.mark.parametrize("K", [768, 1600, 3072])
def test_linear_fp32_is_as_exact_on_tiles_as_for_few_rows(ops, K):
    """64 rows run on tiles, 16 at a time on the kernel for few rows: the former's error against 64 bits is no larger."""
    g = torch.Generator().manual_seed(K)
    a, w = _rand((64, K), torch.float32, g).to(DEV), _rand((768, K), torch.float32, g).to(DEV)
    want, tiles, rows = a.double() @ w.double().T, torch.empty(64, 768, device=DEV), torch.empty(64, 768, device=DEV)
    ops.linear(a, w, None, tiles, "store")
    for m in range(0, 64, 16):
        ops.linear(a[m:m + 16], w, None, rows[m:m + 16], "store")
    assert not torch.equal(tiles, rows)
    assert (tiles.double() - want).norm() <= (rows.double() - want).norm()


@pytest.mark.parametrize("M", [1, 5, 8])
@pytest.mark.parametrize("N,K", [(3, 4), (70, 252), (70, 260), (768, 1020), (768, 1024), (1024, 1028), (1024, 3072), (1024, 3076), (1025, 1536), (1600, 1540), (1600, 6400)])
@pytest.mark.parametrize("epi", ["store", "add_residual"])
def test_linear_fp32_narrow_results(ops, M, N, K, epi):
    """Up to 8 rows of narrow results: passes of 1,024, 1,536 and 3,072 columns of K, filled, missed and begun by four. A lane sums at
    most 2 K / 128 + 48 terms in a chain, so the error is below that many halves of 2^-23 of the terms' absolute sum."""
    g = torch.Generator().manual_seed(M + N + K)
    a, w, bias, x = _rand((M, K), torch.float32, g), _rand((N, K), torch.float32, g), _rand((N,), torch.float32, g), _rand((M, N), torch.float32, g)
    want = a.double() @ w.double().T + bias.double() + (x.double() if epi == "add_residual" else 0)
    bound = (K / 64 + 48) * 2.0 ** -24 * (a.double().abs() @ w.double().abs().T + 2.0)
    out = x.to(DEV)
    ops.linear(a.to(DEV), w.to(DEV), bias.to(DEV), out, epi)
    assert bool(((out.cpu().double() - want).abs() <= bound).all())


@pytest.mark.parametrize("M", [1, 8])
@pytest.mark.parametrize("N,K", [(70, 252), (70, 1000), (1024, 1028), (1024, 3076), (1025, 1540), (1600, 3076)])
def test_linear_fp32_narrow_results_keep_infinite_weights(ops, M, N, K):
    """K that ends within a piece of 256: lanes beyond it must not multiply the row's last weights by anything. An infinity there
    meets an activation of 1 and gives an infinity of its sign, an infinite activation meets a weight of 1; other columns stay as they are."""
    g = torch.Generator().manual_seed(M + N + K)
    a, w = _rand((M, K), torch.float32, g), _rand((N, K), torch.float32, g)
    a[:, -4:] = 1.0
    clean = torch.empty(M, N, device=DEV)
    ops.linear(a.to(DEV), w.to(DEV), None, clean)
    w[1, -1], w[2, -4] = math.inf, -math.inf
    out = torch.empty(M, N, device=DEV)
    ops.linear(a.to(DEV), w.to(DEV), None, out)
    assert bool((out[:, 1] == math.inf).all()) and bool((out[:, 2] == -math.inf).all())
    assert torch.equal(out[:, 3:], clean[:, 3:]) and torch.equal(out[:, 0], clean[:, 0])
    w[:, -4:] = 1.0
    a[M - 1, -2] = math.inf
    ops.linear(a.to(DEV), w.to(DEV), None, out)
    assert bool((out[M - 1] == math.inf).all()) and bool(out[:M - 1].isfinite().all())


@pytest.mark.parametrize("N,K", [(16381, 64), (16385, 64), (16385, 68), (20001, 96), (32001, 128), (32001, 132), (16384, 96), (16384, 100), (20000, 16)])
@pytest.mark.parametrize("M", [64, 65, 130])
def test_linear_fp32_wide_rows_of_short_sums(ops, M, N, K):
    """Both sides of the rules for wide results of short sums (odd rows off the tiles; the tiles' shapes): the error is at most one
    rounding a term of the magnitudes' sum, and what stands beside the columns stays."""
    g = torch.Generator().manual_seed(M + N + K)
    a, w = _rand((M, K), torch.float32, g).to(DEV), _rand((N, K), torch.float32, g).to(DEV)
    bias = _rand((N,), torch.float32, g).to(DEV)
    out = torch.full((M, N + 4), 7.0, device=DEV)          # (a row stride as odd as N)
    ops.linear(a, w, bias, out[:, :N], "store")
    want, size = a.double() @ w.double().T + bias.double(), a.double().abs() @ w.double().abs().T + bias.double().abs()
    assert ((out[:, :N].double() - want).abs() <= 2.0 ** -24 * (K + 2) * size).all()
    assert (out[:, N:] == 7).all()


@pytest.mark.parametrize("M, N, K", [(4, 8, 36), (70, 33, 44), (9, 5, 7)])
def test_linear_bf16_takes_any_k_through_the_plain_kernel(ops, M, N, K):
    """A K that is no multiple of 8 (the matrix-core kernels read 16 bytes at a time) runs on the plain kernel."""
    g = torch.Generator().manual_seed(M + N + K)
    a = _rand((M, K), torch.float32, g).to(torch.bfloat16)
    w = _rand((N, K), torch.float32, g, std=1.0 / math.sqrt(K)).to(torch.bfloat16)
    bias = 0.5 * _rand((N,), torch.float32, g)
    out = torch.empty(M, N, dtype=torch.bfloat16, device=DEV)
    ops.linear(a.to(DEV), w.to(DEV), bias.to(DEV), out)
    ref = a.double() @ w.double().T + bias.double()
    assert (out.cpu().double() - ref).abs().max().item() <= 2e-2
    res = _rand((M, N), torch.float32, g)
    acc = res.clone().to(DEV)
    ops.linear(a.to(DEV), w.to(DEV), None, acc, "add_residual")
    assert (acc.cpu().double() - (res.double() + a.double() @ w.double().T)).abs().max().item() <= 1e-4


@pytest.mark.parametrize("dtype", DTYPES)
def test_kv_append_reference_vector(ops, dtype):
    # /root/reference/tests/kernels/append_kv/gen.py:12-24: blocks [3,3,7,7,7,9], offsets [0,1,0,1,2,4]
    D, BS, NB = 768, 16, 12
    blocks = torch.tensor([3, 3, 7, 7, 7, 9])
    offs = torch.tensor([0, 1, 0, 1, 2, 4])
    qkv = torch.zeros(6, 3 * D)
    for t in range(6):
        for part, base in enumerate((10000, 20000, 30000)):
            qkv[t, part * D:(part + 1) * D] = (base + t * 100 + torch.arange(D)) / 64.0
    qkv = qkv.to(dtype)
    kp = torch.full((NB * BS, D), -1.0, dtype=dtype, device=DEV)
    vp = torch.full((NB * BS, D), -1.0, dtype=dtype, device=DEV)
    slots = (blocks * BS + offs).to(torch.int32)
    slots_skip = torch.cat([slots, torch.tensor([-1], dtype=torch.int32)])
    src = torch.cat([qkv, torch.ones(1, 3 * D, dtype=dtype)])
    ops.kv_append(src.to(DEV), D, 2 * D, D, kp, vp, slots_skip.to(DEV))
    assert torch.equal(kp.cpu()[slots.long()], qkv[:, D:2 * D])
    assert torch.equal(vp.cpu()[slots.long()], qkv[:, 2 * D:])
    untouched = torch.ones(NB * BS, dtype=torch.bool)
    untouched[slots.long()] = False
    assert (kp.cpu()[untouched] == -1).all() and (vp.cpu()[untouched] == -1).all()


def _attention_case(ops, dtype, H, Hkv, dh, page, seqs, window, gen, boost=None, n_single=0, q_col=8, shape=None, gated=False, edit=None):
    """seqs: list of (start, q_len). Builds pages in scrambled order, garbage elsewhere. `edit(b, q, k, v)` may change a sequence's rows."""
    B = len(seqs)
    ctx = [s + n for s, n in seqs]
    nblk = [-(-c // page) for c in ctx]
    n_pages = sum(nblk) + 3
    perm = torch.randperm(n_pages, generator=gen).tolist()
    kv_dim = Hkv * dh
    kp = torch.full((n_pages * page, kv_dim), float("nan"), dtype=dtype)
    vp = torch.full((n_pages * page, kv_dim), float("nan"), dtype=dtype)
    tables = torch.zeros(B, max(nblk), dtype=torch.int32)
    T = sum(n for _, n in seqs)
    q = _rand((T, H * dh + 16), dtype, gen)
    token_seq, positions = [], []
    used = 0
    for b, (s, n) in enumerate(seqs):
        for j in range(nblk[b]):
            tables[b, j] = perm[used]
            used += 1
        k = _rand((ctx[b], kv_dim), dtype, gen)
        v = _rand((ctx[b], kv_dim), dtype, gen)
        if boost is not None and ctx[b] > boost[0]:
            # one far key stands out: its score dominates for the last query
            far = boost[0]
            k[far] = k[far] * 0 + (q[len(token_seq) + n - 1, q_col:q_col + H * dh].float().view(H, dh)[::H // Hkv]
                                   .reshape(-1) * boost[1]).to(dtype)
        if edit is not None:
            edit(b, q[len(token_seq):len(token_seq) + n, q_col:q_col + H * dh].view(n, H, dh), k.view(-1, Hkv, dh), v.view(-1, Hkv, dh))
        js = torch.arange(ctx[b])
        rows = tables[b].long()[js // page] * page + js % page
        kp[rows] = k
        vp[rows] = v
        token_seq += [b] * n
        positions += list(range(s, s + n))
    token_seq = torch.tensor(token_seq, dtype=torch.int32)
    positions = torch.tensor(positions, dtype=torch.int32)
    scale = dh ** -0.5
    out = torch.zeros(T, H * dh, dtype=dtype, device=DEV)
    cu = torch.tensor([0] + list(torch.tensor([n for _, n in seqs]).cumsum(0)), dtype=torch.int32)
    gate = torch.randn(T, H * dh + 4, generator=gen) * 2 if gated else None
    on_dev = None
    if shape is not None:
        on_dev = {k: (v.to(DEV) if torch.is_tensor(v) else v) for k, v in shape.items()}
    ops.paged_attention(q.to(DEV), q_col, H, Hkv, dh, kp.to(DEV), vp.to(DEV), page, tables.to(DEV),
                        token_seq.to(DEV), positions.to(DEV), scale, window, out,
                        cu_q=cu.to(DEV), ctx_len=torch.tensor(ctx, dtype=torch.int32).to(DEV),
                        max_q_len=max(n for _, n in seqs), max_ctx_len=max(ctx), n_single=n_single,
                        shape=on_dev, gate=gate.to(DEV) if gated else None)
    ref = torch.zeros(T, H * dh, dtype=torch.float64)
    plain_ops.paged_attention(q, q_col, H, Hkv, dh, kp, vp, page, tables, token_seq, positions, scale, window, ref,
                              shape=shape, gate=gate)
    if shape is None and edit is None and sum(c * n for c, (_, n) in zip(ctx, seqs)) * H * dh <= 2e8:
        # the second oracle, the plain C++ twin, says the same
        twin = ref_ops.paged_attention(q, 8, H, Hkv, dh, kp, vp, page, tables, token_seq, positions, scale, window)
        assert (twin.double() - ref).abs().max() <= 2e-6
    return out.cpu().double(), ref


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("H,Hkv,dh,page", [(12, 12, 64, 16), (4, 4, 16, 4), (3, 3, 32, 8), (6, 2, 48, 16),
                                           (5, 1, 128, 32), (2, 2, 256, 64)])
def test_paged_attention_mixed_batch(ops, dtype, H, Hkv, dh, page):
    g = torch.Generator().manual_seed(H * 100 + dh)
    seqs = [(0, 37), (130, 1), (64, 2), (5, 70), (0, 1), (199, 1)]
    out, ref = _attention_case(ops, dtype, H, Hkv, dh, page, seqs, 0, g)
    assert torch.isfinite(out).all()
    assert (out - ref).abs().max() <= _tol(dtype, 2)


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("H,Hkv,dh,page", [(12, 12, 64, 16), (4, 4, 16, 4), (3, 3, 32, 8), (6, 2, 128, 16),
                                           (2, 1, 256, 64), (5, 5, 48, 16)])
@pytest.mark.parametrize("window", [0, 33])
@pytest.mark.parametrize("shape", [None, (3, 4), (8, 2), (1, 6), (1, 16)])
def test_paged_attention_decode_only(ops, dtype, H, Hkv, dh, page, window, shape):
    """Every query a single token: the decode kernel (power-of-two head sizes; others fall back),
    in its default launch shape and with the keys of a query split over 3 and 8 workgroups whose
    partial results the last one merges; contexts from 1 token to a thousand so that splits are
    empty, partial and full."""
    g = torch.Generator().manual_seed(H * 10 + dh + window)
    ops.DECODE_SHAPE_OVERRIDE = shape
    try:
        for seqs in ([(0, 1)], [(1023, 1), (0, 1), (63, 1), (64, 1), (500, 1), (17, 1), (129, 1), (255, 1)],
                     [(s, 1) for s in range(3, 300, 7)]):
            out, ref = _attention_case(ops, dtype, H, Hkv, dh, page, seqs, window, g)
            assert torch.isfinite(out).all()
            assert (out - ref).abs().max() <= _tol(dtype, 2)
        # run twice in a row: the split counters must be back at zero
        out, ref = _attention_case(ops, dtype, H, Hkv, dh, page, [(700, 1), (2, 1)], window, g)
        assert (out - ref).abs().max() <= _tol(dtype, 2)
    finally:
        ops.DECODE_SHAPE_OVERRIDE = None


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("T,H,Hkv,dh", [(9, 16, 16, 64), (9, 17, 17, 64), (17, 12, 4, 64), (12, 25, 5, 64), (10, 16, 4, 128)])
@pytest.mark.parametrize("blocks", [1, 4, 5, 8, 9, 10, 12, 13])
def test_paged_attention_decode_wavefronts(ops, dtype, T, H, Hkv, dh, blocks):
    """As many wavefronts as the longest context's keys occupy, within 4 to 12 and the limits by pairs: contexts on both sides of
    every step of that rule, in one launch with short ones."""
    per = 512 // (dh * (2 if dtype == torch.bfloat16 else 4) // 16)
    g = torch.Generator().manual_seed(T * H + blocks)
    for longest in (per * blocks, per * blocks + 1):
        out, ref = _attention_case(ops, dtype, H, Hkv, dh, 16, [((longest - 1) // (1 + k % 3), 1) for k in range(T)], 0, g)
        assert torch.isfinite(out).all()
        assert (out - ref).abs().max() <= _tol(dtype, 2)


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("H,Hkv,dh,page", [(4, 2, 64, 16), (6, 2, 128, 16), (3, 3, 32, 8), (5, 5, 48, 16), (2, 1, 40, 4)])
@pytest.mark.parametrize("kind", ["window_bias", "chunk_gate", "sigmoid", "slope_sink", "window_keep"])
def test_paged_attention_with_shaped_scores(ops, dtype, H, Hkv, dh, page, kind):
    """Scores capped and biased by the distance under a sliding window, or a chunked mask with a gate on the result,
    on every kernel of the dispatch: prompt portions (matrix-core tiles in bfloat16 and in 32-bit; the row kernel for
    a head of 40), single tokens (split keys), and a mixed step whose single tokens stand in front. One far key is
    boosted so that a lost key, a chunk's or a window's edge one off shows."""
    g = torch.Generator().manual_seed(H * 7 + dh + len(kind))
    if kind == "window_bias":
        window = 150
        shape = {"softcap": 6.0, "r1": torch.rand(H, generator=g) + 0.2, "r2": torch.rand(H, generator=g) + 0.1}
    elif kind == "sigmoid":
        # weights that are sigmoids of the scores plus a bias per head, a gate per head: the matrix-core tiles and the
        # split keys take them in bfloat16 at head sizes 32, 64 and 128 (the caller keeps other cases off them)
        if dtype != torch.bfloat16 or dh not in (32, 64, 128):
            pytest.skip("sigmoid weights run on these kernels in bfloat16 at head sizes 32, 64, 128")
        window = 150
        shape = {"sigmoid": 1, "score_bias": torch.randn(H, generator=g) - 4.0, "gate_per_head": 1}
    elif kind == "slope_sink":
        # a penalty that grows linearly with the distance, a sink per head in the denominator (some as large as the
        # boosted key's score), a gate per head: every kernel of the dispatch takes them, in both precisions
        window = 0
        shape = {"slope": torch.rand(H, generator=g) * 0.02, "sink": torch.randn(H, generator=g) * 3.0 + 2.0, "gate_per_head": 1}
    elif kind == "window_keep":
        # a window of 150 that also sees the first 70 positions (more than a key tile of the 32-bit kernel, less than one
        # of the matrix-core kernel), with a sink
        window = 150
        shape = {"keep_first": 70, "sink": torch.randn(H, generator=g)}
    else:
        window = 0
        shape = {"chunk": 70}
    gated = kind in ("chunk_gate", "sigmoid", "slope_sink")
    cases = [([(0, 37), (130, 70), (64, 2), (5, 300)], 0), ([(1023, 1), (0, 1), (63, 1), (149, 1), (150, 1), (69, 1), (70, 1), (500, 1)], 8),
             ([(300, 1), (12, 1), (0, 100), (200, 64), (139, 1)], 2)]
    for seqs, n_single in cases:
        # (kept first positions: the boosted key is one of them, far in front of the last sequence's window)
        far = 5 if kind == "window_keep" else max(0, seqs[0][0] + seqs[0][1] - 3)
        out, ref = _attention_case(ops, dtype, H, Hkv, dh, page, seqs, window, g, boost=(far, 0.5),
                                   n_single=n_single, q_col=0, shape=shape, gated=gated)
        assert torch.isfinite(out).all()
        # (sums of weights that are not normalised grow with the keys: relative to the largest value)
        assert (out - ref).abs().max() <= _tol(dtype, 2) * max(1.0, ref.abs().max().item() if kind == "sigmoid" else 1.0)


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("H,Hkv,dh,page,qlens", [(12, 12, 64, 16, (1, 1, 1)), (6, 2, 32, 8, (1, 1, 1)),
                                                   (5, 5, 48, 16, (1, 1, 1)), (4, 2, 64, 4, (3, 1, 9))])
def test_paged_attention_appends_own_keys(ops, dtype, H, Hkv, dh, page, qlens):
    """With append=..., the step's keys/values come from the q rows and land in the pages:
    fused into the decode kernel (single-token queries, power-of-two heads) or copied first."""
    g = torch.Generator().manual_seed(H + dh + sum(qlens))
    starts = (200, 0, 31)
    kv_dim, qd = Hkv * dh, H * dh
    n_pages = sum(-(-(s + n) // page) for s, n in zip(starts, qlens)) + 2
    kp = torch.full((n_pages * page, kv_dim), float("nan"), dtype=dtype)
    vp = torch.full((n_pages * page, kv_dim), float("nan"), dtype=dtype)
    ref_kp, ref_vp = kp.clone(), vp.clone()
    maxb = max(-(-(s + n) // page) for s, n in zip(starts, qlens))
    tables = torch.zeros(3, maxb, dtype=torch.int32)
    T = sum(qlens)
    qkv = _rand((T, qd + 2 * kv_dim), dtype, g)
    token_seq, positions, slots = [], [], []
    used = t = 0
    for b, (s, n) in enumerate(zip(starts, qlens)):
        nb = -(-(s + n) // page)
        tables[b, :nb] = torch.arange(used, used + nb, dtype=torch.int32)
        used += nb
        js = torch.arange(s + n)
        rows = tables[b].long()[js // page] * page + js % page
        k, v = _rand((s + n, kv_dim), dtype, g), _rand((s + n, kv_dim), dtype, g)
        k[s:], v[s:] = qkv[t:t + n, qd:qd + kv_dim], qkv[t:t + n, qd + kv_dim:]
        ref_kp[rows], ref_vp[rows] = k, v
        kp[rows[:s]], vp[rows[:s]] = k[:s], v[:s]             # the step's own rows are still empty
        token_seq += [b] * n
        positions += list(range(s, s + n))
        slots += rows[s:].tolist()
        t += n
    token_seq, positions, slots = (torch.tensor(a, dtype=torch.int32) for a in (token_seq, positions, slots))
    kp_d, vp_d = kp.to(DEV), vp.to(DEV)
    out = torch.zeros(T, qd, dtype=dtype, device=DEV)
    ops.paged_attention(qkv.to(DEV), 0, H, Hkv, dh, kp_d, vp_d, page, tables.to(DEV), token_seq.to(DEV),
                        positions.to(DEV), dh ** -0.5, 0, out, max_q_len=max(qlens), max_ctx_len=210,
                        append=(qd, qd + kv_dim, slots.to(DEV)))
    ref = torch.zeros(T, qd, dtype=torch.float64)
    plain_ops.paged_attention(qkv, 0, H, Hkv, dh, ref_kp, ref_vp, page, tables, token_seq, positions, dh ** -0.5, 0, ref)
    assert (out.cpu().double() - ref).abs().max() <= _tol(dtype, 2)
    written = slots.long()
    assert torch.equal(kp_d.cpu()[written], ref_kp[written]) and torch.equal(vp_d.cpu()[written], ref_vp[written])


@pytest.mark.parametrize("H,Hkv,dh,page", [(12, 12, 64, 16), (3, 3, 32, 8), (4, 1, 128, 16), (6, 2, 64, 4)])
@pytest.mark.parametrize("window", [0, 1, 50, 64, 200])
def test_paged_attention_prefill_tiles(ops, H, Hkv, dh, page, window):
    """The MFMA prefill kernel (bf16, head sizes 32/64/128): query tiles that are full, partial and
    a single row; portions that start mid-sequence and mid-page; windows that cut inside a key tile."""
    g = torch.Generator().manual_seed(H + dh + window)
    seqs = [(0, 64), (0, 150), (37, 2), (100, 129), (511, 1), (64, 64), (5, 63)]
    out, ref = _attention_case(ops, torch.bfloat16, H, Hkv, dh, page, seqs, window, g)
    assert torch.isfinite(out).all()
    assert (out - ref).abs().max() <= _tol(torch.bfloat16, 2)


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("H,Hkv,dh,page", [(12, 12, 64, 16), (4, 4, 16, 4), (6, 2, 48, 12), (5, 1, 80, 8), (3, 3, 128, 20),
                                           (2, 1, 256, 64), (7, 7, 32, 1)])
@pytest.mark.parametrize("window", [0, 1, 50, 64, 200])
def test_paged_attention_tiles_in_true_32_bit(ops, dtype, H, Hkv, dh, page, window):
    """The prompt-portion kernel that shares key tiles among 64 queries at any head size (steps of 16 up to 256),
    any page size (12 and 20 are no powers of two; 1), grouped heads, float32 and bfloat16 storage: query tiles that
    are full, partial and a single row; portions that start mid-sequence and mid-page; windows that cut inside a key
    tile. Read back from the ops: this kernel ran wherever the bfloat16 matrix-core kernel does not take the sizes."""
    g = torch.Generator().manual_seed(H + dh + window + page)
    seqs = [(0, 64), (0, 150), (37, 2), (100, 129), (511, 1), (64, 64), (5, 63)]
    ops.reset_seen()
    out, ref = _attention_case(ops, dtype, H, Hkv, dh, page, seqs, window, g)
    mfma_bf16 = dtype == torch.bfloat16 and dh in (32, 64, 128) and page & (page - 1) == 0 and page >= dh // 16
    assert ops.seen("tiled_f32_launches") == (0 if mfma_bf16 else 1) and ops.seen("generic_attention_launches") == 0
    assert torch.isfinite(out).all()
    assert (out - ref).abs().max() <= _tol(dtype, 2)
    # single tokens in front of the portions (a mixed step): at page sizes the decode kernel refuses they go to the
    # one-wavefront-per-query kernel, the portions to the tiles
    seqs = [(300, 1), (0, 1), (77, 1), (0, 70), (130, 3), (64, 129)]
    ops.reset_seen()
    out, ref = _attention_case(ops, dtype, H, Hkv, dh, page, seqs, window, g, n_single=3)
    assert ops.seen("tiled_f32_launches") == (0 if mfma_bf16 else 1)
    assert torch.isfinite(out).all()
    assert (out - ref).abs().max() <= _tol(dtype, 2)


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("seqs", [[(5000, 70), (0, 300)],                               # one far in front of the other: their tiles' places are halved
                                  [(4200, 130), (0, 1), (64, 64), (63, 65), (10, 129)],
                                  [(i % 3 * 64, 1 + 37 * i % 140) for i in range(64)],   # a sequence a lane
                                  [(0, 1 + i % 67) for i in range(65)]])                 # more of them
@pytest.mark.parametrize("H,Hkv,dh", [(3, 1, 64), (2, 2, 128)])
def test_paged_attention_gives_every_tile_away(ops, dtype, seqs, H, Hkv, dh):
    """The order in which workgroups take the query tiles of several sequences, by how many keys they see: every row is written."""
    g = torch.Generator().manual_seed(len(seqs) + dh)
    out, ref = _attention_case(ops, dtype, H, Hkv, dh, 16, seqs, 0, g)
    assert torch.isfinite(out).all()
    assert (out - ref).abs().max() <= _tol(dtype, 2)


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("dh", [16, 32, 64, 128, 256])
@pytest.mark.parametrize("waves", [1, 2, 3, 4, 5, 8, 9, 12, 13, 16])
@pytest.mark.parametrize("nsplit", [1, 3])
def test_decode_attention_merges_every_number_of_wavefronts(ops, monkeypatch, dtype, dh, waves, nsplit):
    """The states of lane groups, wavefronts and splits, with wavefronts that have keys and some that have none."""
    g = torch.Generator().manual_seed(waves * 3 + dh)
    monkeypatch.setattr(ops, "DECODE_SHAPE_OVERRIDE", (nsplit, waves))
    out, ref = _attention_case(ops, dtype, 6, 2, dh, 16, [(0, 1), (40, 1), (700, 1), (1500, 1)], 0, g)
    assert (out - ref).abs().max() <= _tol(dtype, 2)


@pytest.mark.parametrize("seqs", [[(0, 1)], [(5000, 70), (0, 300)], [(0, 300), (5000, 70)], [(4200, 130), (0, 1), (64, 64), (63, 65), (10, 129)],
                                  [(0, 512)] * 4, [(i % 3 * 64, 1 + 37 * i % 140) for i in range(64)], [(i * 977 % 90000, i % 5 * 33) for i in range(64)],
                                  [(0, 1 + i % 67) for i in range(65)]])
@pytest.mark.parametrize("rows", [1, 5, 12])
def test_every_query_tile_is_given_to_one_workgroup(seqs, rows):
    """Each order gives every tile of 64 rows (a query has `rows`) to exactly one of the workgroups, the rest get none, and the order by length
    begins with the pairs of tiles that see most."""
    import ctypes
    import toy  # noqa: F401  (registers the test-only library)
    from mini_llm_amd import build
    lib = build.load_library("lane_check")
    cu = [sum(n for _, n in seqs[:b]) for b in range(len(seqs) + 1)]
    want = {(b, t, cu[b], n) for b, (_, n) in enumerate(seqs) for t in range(-(-n * rows // 64))}
    places = cu[-1] * rows // 64 + len(seqs)
    on_dev = [torch.tensor(a, dtype=torch.int32, device=DEV) for a in (cu, [s + n for s, n in seqs])]
    for order in (0, 1, 2) if len(seqs) <= 64 else (0, 1):
        out = torch.full((places, 4), 77, dtype=torch.int32, device=DEV)
        assert lib.mllm_query_tiles(*(ctypes.c_void_p(a.data_ptr()) for a in on_dev), len(seqs), rows, order, places, ctypes.c_void_p(out.data_ptr()),
                                    ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)) == 0
        got = [tuple(t) for t in out.cpu().tolist()]
        given = [t for t in got if t[0] >= 0]
        assert len(given) == len(want) and set(given) == want and all(t[0] == -1 for t in got if t not in want)
        if order == 2:
            sees = [(seqs[b][0] * rows // 64 + t) // 2 for b, t, _, _ in given]
            assert sees == sorted(sees, reverse=True) and got[:len(given)] == given


@pytest.mark.parametrize("n_seqs,places,order", [(1, 300, 1), (2, 256, 1), (2, 257, 2), (7, 256, 1), (7, 257, 2), (8, 40, 2), (64, 300, 2), (65, 300, 1)])
def test_query_tiles_are_ordered_where_it_pays(n_seqs, places, order):
    """The longest tiles come first (order 2) from eight sequences on, and with two to seven where there are more workgroups than compute units; otherwise,
    and with more than 64 sequences, a sequence's tiles come one after the other (order 1)."""
    import ctypes
    import toy  # noqa: F401  (registers the test-only library)
    from mini_llm_amd import build
    lib = build.load_library("lane_check")
    lens = [70 + 10 * (b % 7) for b in range(n_seqs)]
    cu, ctx = [sum(lens[:b]) for b in range(n_seqs + 1)], [n + 64 * (b % 3) for b, n in enumerate(lens)]
    on_dev = [torch.tensor(a, dtype=torch.int32, device=DEV) for a in (cu, ctx)]
    got = []
    for o in (0, order):
        out = torch.full((places, 4), 77, dtype=torch.int32, device=DEV)
        assert lib.mllm_query_tiles(*(ctypes.c_void_p(a.data_ptr()) for a in on_dev), n_seqs, 1, o, places, ctypes.c_void_p(out.data_ptr()),
                                    ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)) == 0
        got.append(out.cpu())
    assert torch.equal(*got)


@pytest.mark.parametrize("H,Hkv,dh", [(2, 1, 64), (1, 1, 128)])
@pytest.mark.parametrize("ctx", [4095, 4096, 4097])
@pytest.mark.parametrize("shaped", [False, True])
def test_paged_attention_of_the_longest_block_tables(ops, H, Hkv, dh, ctx, shaped):
    """32-bit portions with pages of one token: a table of 4,096 entries is the longest that lies in LDS beside the tiles, one more runs on the
    kernel that reads it from memory."""
    g = torch.Generator().manual_seed(ctx + dh)
    shape = {"sink": torch.randn(H, generator=g)} if shaped else None
    ops.reset_seen()
    out, ref = _attention_case(ops, torch.float32, H, Hkv, dh, 1, [(ctx - 70, 70), (0, 3), (ctx - 64, 64)], 0, g, q_col=0 if shaped else 8, shape=shape)
    assert ops.seen("tiled_f32_launches") == 1
    assert torch.isfinite(out).all() and (out - ref).abs().max() <= _tol(torch.float32, 2)


@pytest.mark.parametrize("H,Hkv,dh", [(3, 3, 32), (3, 1, 64), (2, 2, 128)])
@pytest.mark.parametrize("window", [0, 1])
def test_paged_attention_of_scores_at_the_lowest_end(ops, H, Hkv, dh, window):
    """32-bit portions. Scores of -inf beside a sink: a query that sees no other key has the sink's weight alone, in either half of a
    key tile, and gives 0. A score just above the lowest float, in base 2 too, is a score like any other."""
    g = torch.Generator().manual_seed(dh + window)
    seqs, at = [(0, 130), (0, 70), (60, 9)], [0, 5, 40, 64, 100]

    def lowest(b, q, k, v):
        if window == 0 and b == 1:                            # all that the sequence's queries see
            k[..., 0], q[..., 0] = math.inf, -q[..., 0].abs() - 0.1
        elif window == 1 and b == 0:                          # a query's own key
            k[at, :, 0], q[at, :, 0] = math.inf, -q[at, :, 0].abs() - 0.1

    out, ref = _attention_case(ops, torch.float32, H, Hkv, dh, 16, seqs, window, g, q_col=0, shape={"sink": torch.randn(H, generator=g)}, edit=lowest)
    rows = [130 + i for i in range(70)] if window == 0 else at
    assert (out[rows] == 0).all() and (ref[rows] == 0).all()
    assert (out - ref).abs().max() <= _tol(torch.float32, 2)

    def low(b, q, k, v):
        if b == 0:
            q[at, :], k[at, :] = 0.0, 0.0
            q[at, :, 0], k[at, :, 0] = -16.0, 2.2e38 * math.sqrt(dh) / 16

    if window == 1:
        out, ref = _attention_case(ops, torch.float32, H, Hkv, dh, 16, seqs, window, g, edit=low)
        assert (out - ref).abs().max() <= _tol(torch.float32, 2)


@pytest.mark.parametrize("H,Hkv,dh", [(3, 3, 32), (3, 1, 64), (2, 2, 128)])
def test_paged_attention_keeps_weights_below_the_normal_range(ops, H, Hkv, dh):
    """32-bit portions: a weight of 2^-130 against a value of 2^127, in either half of a key tile and in an earlier one than the highest score's.
    The score of 130 has a rounding of some units of 2^-24 of itself, which the weight shows ln 2 times."""
    g = torch.Generator().manual_seed(dh)
    seqs, high = [(0, 130)] * 3, [1, 40, 70]

    def far(b, q, k, v):
        q[:], k[:], v[:] = 0.0, 0.0, 0.0
        q[..., 0], k[high[b], :, 0], v[0] = 1.0, 130 * math.log(2) * math.sqrt(dh), 2.0 ** 127

    out, ref = _attention_case(ops, torch.float32, H, Hkv, dh, 16, seqs, 0, g, q_col=0, edit=far)
    for b, first in enumerate(high):
        assert (ref[130 * b + first:130 * (b + 1)] - 0.125).abs().max() <= 1e-3
    assert ((out - ref).abs() <= 130 * 8 * 2.0 ** -24 * ref.abs()).all()


@pytest.mark.parametrize("H,Hkv,dh", [(3, 3, 32), (3, 1, 64), (2, 2, 128)])
@pytest.mark.parametrize("window,keep", [(0, 0), (8, 0), (8, 3), (40, 70)])
def test_paged_attention_of_infinite_values_beside_empty_places(ops, H, Hkv, dh, window, keep):
    """32-bit portions of one query (in a step with a longer one): an infinite value at the first and at the last key that it sees gives
    an infinity. The places of a key tile in front of the first and behind the last have no values at all."""
    g = torch.Generator().manual_seed(dh + window + keep)
    seqs = [(0, 66), (0, 1), (31, 1), (70, 1), (127, 1), (300, 1)]
    shape = {"keep_first": keep, "sink": torch.randn(H, generator=g)} if keep else None
    for last in (True, False):
        def infinite(b, q, k, v):
            p = seqs[b][0]
            if b > 0:
                v[p if last or not window else max(0, p - window + 1)] = math.inf

        out, ref = _attention_case(ops, torch.float32, H, Hkv, dh, 16, seqs, window, g, q_col=0, shape=shape, edit=infinite)
        assert (out[66:] == math.inf).all() and (ref[66:] == math.inf).all()
        assert (out[:66] - ref[:66]).abs().max() <= _tol(torch.float32, 2)


@pytest.mark.parametrize("T", [1, 8, 16])
@pytest.mark.parametrize("H,Hkv,dh,page,N", [(12, 12, 64, 16, 768), (25, 25, 64, 16, 1600), (3, 3, 32, 8, 96),
                                             (4, 2, 128, 16, 200), (16, 16, 64, 16, 1024)])
@pytest.mark.parametrize("shape", [(2, 4), (3, 2), (4, 12), None])
def test_decode_attention_splits_merged_by_the_next_product(ops, T, H, Hkv, dh, page, N, shape):
    """Single tokens whose keys are split over several workgroups per (token, head): the attention op
    hands back the splits unmerged and the product that follows merges them while it loads. Equal to
    attention followed by the product on merged rows; contexts from one key (most splits empty) to
    several hundred; the tokens' own keys come from their qkv rows and reach the pages."""
    g = torch.Generator().manual_seed(T * 31 + H + dh)
    ctx = [1, 700, 130, 2, 64, 65, 300, 17, 1000, 5, 129, 511, 33, 256, 90, 3][:T]
    nblk = [-(-c // page) for c in ctx]
    n_pages = sum(nblk) + 2
    perm = torch.randperm(n_pages, generator=g).tolist()
    kv_dim, D = Hkv * dh, H * dh
    kp = torch.full((n_pages * page, kv_dim), float("nan"), dtype=torch.bfloat16)
    vp = torch.full((n_pages * page, kv_dim), float("nan"), dtype=torch.bfloat16)
    tables = torch.zeros(T, max(nblk), dtype=torch.int32)
    qkv = _rand((T, D + 2 * kv_dim), torch.bfloat16, g)
    slots = torch.zeros(T, dtype=torch.int32)
    used = 0
    for b in range(T):
        for j in range(nblk[b]):
            tables[b, j] = perm[used]
            used += 1
        js = torch.arange(ctx[b] - 1)                   # the last key is the token's own, not in the pages yet
        rows = tables[b].long()[js // page] * page + js % page
        kp[rows] = _rand((ctx[b] - 1, kv_dim), torch.bfloat16, g)
        vp[rows] = _rand((ctx[b] - 1, kv_dim), torch.bfloat16, g)
        slots[b] = int(tables[b, (ctx[b] - 1) // page]) * page + (ctx[b] - 1) % page
    token_seq = torch.arange(T, dtype=torch.int32)
    positions = torch.tensor([c - 1 for c in ctx], dtype=torch.int32)
    w = _rand((N, D), torch.bfloat16, g, std=1.0 / math.sqrt(D))
    bias = 0.5 * _rand((N,), torch.float32, g)
    x0 = _rand((T, N), torch.float32, g)
    # reference: append, attention, product, all plain
    rk, rv = kp.clone(), vp.clone()
    att = torch.zeros(T, D, dtype=torch.float64)
    plain_ops.paged_attention(qkv, 0, H, Hkv, dh, rk, rv, page, tables, token_seq, positions, dh ** -0.5, 0, att,
                              append=(D, D + kv_dim, slots))
    ref = plain_ops.linear(att, w.double(), bias, x0.double().clone(), "add_residual")
    kd, vd = kp.to(DEV), vp.to(DEV)
    out = torch.empty(T, D, dtype=torch.bfloat16, device=DEV)
    ops.DECODE_UNMERGED_SHAPE = shape
    try:
        a = ops.paged_attention(qkv.to(DEV), 0, H, Hkv, dh, kd, vd, page, tables.to(DEV), token_seq.to(DEV),
                                positions.to(DEV), dh ** -0.5, 0, out, max_q_len=1, max_ctx_len=max(ctx),
                                append=(D, D + kv_dim, slots.to(DEV)), may_split=True)
    finally:
        ops.DECODE_UNMERGED_SHAPE = None
    if shape is not None or (max(ctx) >= 256 and T * H <= 128):
        assert isinstance(a, ops.AttentionSplits) and a.nsplit == (shape[0] if shape else a.nsplit) and a.nsplit > 1
    x = x0.clone().to(DEV)
    ops.linear(a, w.to(DEV), bias.to(DEV), x, "add_residual")
    assert torch.isfinite(x).all()
    assert (x.cpu().double() - ref).abs().max() <= 3e-2
    written = slots.long()
    assert torch.equal(kd.cpu()[written], rk[written]) and torch.equal(vd.cpu()[written], rv[written])
    if isinstance(a, ops.AttentionSplits):
        # merged into an ordinary activation by the kernel of its own: the same rows
        merged = a.tensor()
        assert (merged.cpu().double() - att).abs().max() <= 2e-2
        y = torch.empty(T, N, dtype=torch.bfloat16, device=DEV)
        ops.linear(a, w.to(DEV), bias.to(DEV), y, "gelu_tanh")
        ref_y = plain_ops.linear(att, w.double(), bias, torch.empty(T, N, dtype=torch.float64), "gelu_tanh")
        assert (y.cpu().double() - ref_y).abs().max() <= 3e-2


@pytest.mark.parametrize("T", [1, 3, 8])
@pytest.mark.parametrize("H,dh,N", [(12, 64, 768), (25, 64, 1600), (6, 16, 96), (5, 128, 200), (24, 128, 2047), (12, 64, 2048)])
@pytest.mark.parametrize("shape", [(2, 4), (3, 2), (4, 12), None])
def test_decode_attention_splits_merged_by_the_32_bit_product(ops, T, H, dh, N, shape):
    """The same in 32 bits: the product merges while it stages its rows, and a merge of its own stands in front of products that do not."""
    g = torch.Generator().manual_seed(T * 31 + H + dh)
    page, D = 16, H * dh
    ctx = [1, 700, 130, 2, 64, 65, 300, 17][:T] if T > 1 else [700]
    nblk = [-(-c // page) for c in ctx]
    perm = torch.randperm(sum(nblk) + 2, generator=g).tolist()
    kp, vp = (torch.full((len(perm) * page, D), float("nan")) for _ in range(2))
    tables, slots = torch.zeros(T, max(nblk), dtype=torch.int32), torch.zeros(T, dtype=torch.int32)
    qkv = _rand((T, 3 * D), torch.float32, g)
    for b in range(T):
        tables[b, :nblk[b]] = torch.tensor([perm.pop() for _ in range(nblk[b])])
        js = torch.arange(ctx[b] - 1)
        rows = tables[b].long()[js // page] * page + js % page
        kp[rows], vp[rows] = _rand((ctx[b] - 1, D), torch.float32, g), _rand((ctx[b] - 1, D), torch.float32, g)
        slots[b] = int(tables[b, (ctx[b] - 1) // page]) * page + (ctx[b] - 1) % page
    token_seq, positions = torch.arange(T, dtype=torch.int32), torch.tensor([c - 1 for c in ctx], dtype=torch.int32)
    w, bias, x0 = _rand((N, D), torch.float32, g, std=1.0 / math.sqrt(D)), 0.5 * _rand((N,), torch.float32, g), _rand((T, N), torch.float32, g)
    att = torch.zeros(T, D, dtype=torch.float64)
    plain_ops.paged_attention(qkv, 0, H, H, dh, kp.clone(), vp.clone(), page, tables, token_seq, positions, dh ** -0.5, 0, att, append=(D, 2 * D, slots))
    ref = plain_ops.linear(att, w.double(), bias, x0.double().clone(), "add_residual")
    ops.DECODE_UNMERGED_SHAPE = shape
    try:
        a = ops.paged_attention(qkv.to(DEV), 0, H, H, dh, kp.to(DEV), vp.to(DEV), page, tables.to(DEV), token_seq.to(DEV), positions.to(DEV), dh ** -0.5, 0,
                                torch.empty(T, D, device=DEV), max_q_len=1, max_ctx_len=max(ctx), append=(D, 2 * D, slots.to(DEV)), may_split=True)
    finally:
        ops.DECODE_UNMERGED_SHAPE = None
    assert isinstance(a, ops.AttentionSplits) == (shape is not None or T * H <= 128) and (shape is None or a.nsplit == shape[0])
    x = x0.clone().to(DEV)
    ops.linear(a, w.to(DEV), bias.to(DEV), x, "add_residual")
    # (a score's rounding, 2^-24 of its terms' sum, moves its weight by as much; then fp32 sums)
    assert (x.cpu().double() - ref).abs().max() <= 3e-5


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("H,Hkv,dh,page,window", [(12, 12, 64, 16, 0), (3, 3, 32, 8, 0), (4, 1, 128, 16, 40), (4, 4, 16, 4, 0)])
def test_paged_attention_single_tokens_before_portions(ops, dtype, H, Hkv, dh, page, window):
    """A scheduler's mixed step: decoded tokens first, then prompt portions. The leading single tokens
    (`n_single` of them) go to the single-query kernel and the rest to the query tiles; a single token
    that stands among the portions stays with them. Same result as without the hint."""
    g = torch.Generator().manual_seed(H + dh)
    seqs = [(130, 1), (0, 1), (299, 1), (64, 1), (0, 37), (17, 1), (5, 70), (100, 130)]
    out, ref = _attention_case(ops, dtype, H, Hkv, dh, page, seqs, window, g, n_single=4)
    assert torch.isfinite(out).all()
    assert (out - ref).abs().max() <= _tol(dtype, 2)
    g = torch.Generator().manual_seed(H + dh)
    plain, _ = _attention_case(ops, dtype, H, Hkv, dh, page, seqs, window, g)
    assert (out - plain).abs().max() <= _tol(dtype, 2)


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("H,Hkv,dh,page", [(4, 4, 64, 4), (2, 1, 128, 16)])
def test_paged_attention_long_contexts(ops, dtype, H, Hkv, dh, page):
    """Contexts far beyond the tiny models': block tables longer than the prefill kernel stages in
    LDS (2048 blocks), decode over 20,000 keys, a portion that ends a long prompt, with and without
    a window."""
    g = torch.Generator().manual_seed(dh + page)
    for seqs, window in (([(9000, 1), (5, 1)], 0), ([(8300, 200)], 0), ([(0, 2300)], 777), ([(20000, 1)], 0),
                         ([(8190, 3), (100, 40)], 777), ([(8000, 192)], 0)):        # (the last: 2048 blocks of 4 exactly)
        out, ref = _attention_case(ops, dtype, H, Hkv, dh, page, seqs, window, g)
        assert torch.isfinite(out).all()
        assert (out - ref).abs().max() <= _tol(dtype, 2), (seqs, window)


@pytest.mark.parametrize("dtype", DTYPES)
def test_decode_attention_splits_long_contexts_over_the_chip(ops, dtype):
    """Few pairs with thousands of keys: the keys of a pair are split over up to 256 workgroups and a small
    kernel merges their states. Same result as one workgroup a pair, with a short sequence beside the long
    ones (splits that hold no key) and with a window."""
    g = torch.Generator().manual_seed(5)
    for seqs, window in (([(6000, 1), (3, 1), (4500, 1)], 0), ([(9000, 1)], 0), ([(7000, 1), (5000, 1)], 1300)):
        results = []
        for on in (True, False):
            ops.LONG_CONTEXT_SPLITS = on
            try:
                gg = torch.Generator().manual_seed(int(g.initial_seed()) + len(seqs))
                out, ref = _attention_case(ops, dtype, 6, 2, 64, 16, seqs, window, gg)
            finally:
                ops.LONG_CONTEXT_SPLITS = True
            assert (out - ref).abs().max() <= _tol(dtype, 2), (seqs, window, on)
            results.append(out)
        assert (results[0] - results[1]).abs().max() <= _tol(dtype, 2)


@pytest.mark.parametrize("dtype", DTYPES)
def test_paged_attention_far_key_stands_out(ops, dtype):
    """One key hundreds of positions back carries almost all the weight of the last query."""
    g = torch.Generator().manual_seed(7)
    out, ref = _attention_case(ops, dtype, 4, 2, 64, 16, [(600, 3), (0, 300)], 0, g, boost=(3, 4.0))
    assert (out - ref).abs().max() <= _tol(dtype, 2)


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("window", [1, 7, 64, 65])
def test_paged_attention_window_edge(ops, dtype, window):
    g = torch.Generator().manual_seed(window)
    out, ref = _attention_case(ops, dtype, 4, 2, 32, 8, [(0, 80), (130, 1), (63, 3)], window, g)
    assert (out - ref).abs().max() <= _tol(dtype, 2)


@pytest.mark.parametrize("dtype", DTYPES)
def test_kernels_against_their_cpp_twins(ops, dtype):
    """Every kernel against the plain C++ statement of its operation (csrc/ref/ref_ops.cc)."""
    g = torch.Generator().manual_seed(11)
    V, P, D, T = 301, 40, 200, 37
    wte, wpe = _rand((V, D), dtype, g), _rand((P, D), dtype, g)
    ids = torch.randint(0, V, (T,), generator=g, dtype=torch.int32)
    pos = torch.randint(0, P, (T,), generator=g, dtype=torch.int32)
    x = torch.empty(T, D, dtype=torch.float32, device=DEV)
    ops.embed(ids.to(DEV), pos.to(DEV), wte.to(DEV), wpe.to(DEV), x)
    assert (x.cpu() - ref_ops.embed(ids, pos, wte, wpe)).abs().max() <= 1e-6
    gamma, beta = 1 + 0.1 * _rand((D,), torch.float32, g), 0.1 * _rand((D,), torch.float32, g)
    h = torch.empty(T, D, dtype=dtype, device=DEV)
    ops.layernorm(x, gamma.to(DEV), beta.to(DEV), 1e-5, h)
    assert (h.cpu().float() - ref_ops.layernorm(x.cpu(), gamma, beta, 1e-5)).abs().max() <= _tol(dtype, 4)
    for M, N, K, epi in [(T, 3 * D, D, "store"), (5, 72, D, "gelu_tanh"), (T, D, D, "add_residual"), (70, V, D, "store_f32"),
                         (3, 90, D, "gelu_erf")]:
        a, w, bias = _rand((M, K), dtype, g), _rand((N, K), dtype, g, std=K ** -0.5), 0.5 * _rand((N,), torch.float32, g)
        f32_out = epi in ("add_residual", "store_f32")
        out0 = _rand((M, N), torch.float32 if f32_out else dtype, g)
        out = out0.clone().to(DEV)
        ops.linear(a.to(DEV), w.to(DEV), bias.to(DEV), out, epi)
        tol = 3e-5 if dtype == torch.float32 else (2e-5 + 2e-5 * math.sqrt(K) if f32_out else 4e-2)
        assert (out.cpu().float() - ref_ops.linear(a, w, bias, out0, epi)).abs().max() <= tol, (M, N, K, epi)
        if epi != "add_residual":
            xs = _rand((M, K), torch.float32, g) + 0.3
            out = out0.clone().to(DEV)
            ops.ln_linear(xs.to(DEV), gamma.to(DEV), beta.to(DEV), 1e-5, w.to(DEV), bias.to(DEV), out, epi)
            hn = ref_ops.layernorm(xs, gamma, beta, 1e-5).to(dtype)
            # (a normalised value next to a bf16 rounding boundary may round the other way in the kernel)
            tol_ln = 3e-5 if dtype == torch.float32 else (2e-2 if epi == "store_f32" else 4e-2)
            assert (out.cpu().float() - ref_ops.linear(hn, w, bias, out0, epi)).abs().max() <= tol_ln, (M, N, K, epi)
    H, Hkv, dh, page = 6, 2, 32, 8
    src = _rand((9, 3 * Hkv * dh), dtype, g)
    slots = torch.tensor([5, -1, 0, 9, 70, 71, 72, 3, 11], dtype=torch.int32)
    kp, vp = torch.zeros(80, Hkv * dh, dtype=dtype, device=DEV), torch.zeros(80, Hkv * dh, dtype=dtype, device=DEV)
    ops.kv_append(src.to(DEV), Hkv * dh, 2 * Hkv * dh, Hkv * dh, kp, vp, slots.to(DEV))
    k2, v2 = torch.zeros(80, Hkv * dh), torch.zeros(80, Hkv * dh)
    ref_ops.kv_append(src, Hkv * dh, 2 * Hkv * dh, Hkv * dh, k2, v2, slots)
    assert torch.equal(kp.cpu().float(), k2) and torch.equal(vp.cpu().float(), v2)
    _attention_case(ops, dtype, H, Hkv, dh, page, [(40, 1), (0, 70), (9, 5), (130, 1)], 0, g)   # (compares both oracles)
    logits = _rand((6, 1000), torch.float32, g, std=2.0)
    out = torch.empty(6, dtype=torch.int32, device=DEV)
    ops.argmax(logits.to(DEV), out)
    assert torch.equal(out.cpu(), ref_ops.argmax(logits))
    temp, u = torch.tensor([0.0, 0.7, 1.0, 1.3, 0.2, 5.0]), torch.tensor([0.3, 0.0, 0.999, 0.5, 0.25, 0.75])
    ops.sample(logits.to(DEV), temp.to(DEV), u.to(DEV), out)
    got, want = out.cpu(), ref_ops.sample(logits, temp, u)
    for r in range(6):                  # next to a boundary of the cumulative mass either neighbour is right
        assert abs(int(got[r]) - int(want[r])) <= 1, (r, got, want)


def test_argmax_ties_take_lowest_index(ops):
    V = 50257
    g = torch.Generator().manual_seed(3)
    logits = _rand((5, V), torch.float32, g)
    logits[0, 40000] = logits[0, 123] = 9.0
    logits[1, V - 1] = 10.0
    logits[2, 0] = 10.0
    logits[3, :] = 0.5
    out = torch.empty(5, dtype=torch.int32, device=DEV)
    ops.argmax(logits.to(DEV), out)
    ref = plain_ops.argmax(logits, torch.empty(5, dtype=torch.int32))
    assert out.cpu().tolist() == ref.tolist()
    assert out.cpu().tolist()[:4] == [123, V - 1, 0, 0]


@pytest.mark.parametrize("V", [4, 1000, 50257])
def test_sample_inverse_cdf(ops, V):
    g = torch.Generator().manual_seed(V)
    n = 64
    logits = _rand((n, V), torch.float32, g, std=2.0)
    temps = torch.rand(n, generator=g) * 1.5 + 0.2
    temps[::7] = 0.0
    u = torch.rand(n, generator=g)
    out = torch.empty(n, dtype=torch.int32, device=DEV)
    ops.sample(logits.to(DEV), temps.to(DEV), u.to(DEV), out)
    got = out.cpu().tolist()
    for i in range(n):
        row = logits[i].double()
        if temps[i] <= 0:
            assert got[i] == int(row.argmax())
            continue
        p = torch.softmax(row / temps[i].double(), 0)
        c = torch.cumsum(p, 0)
        lo = float(c[got[i] - 1]) if got[i] > 0 else 0.0
        hi = float(c[got[i]])
        assert lo - 1e-5 <= float(u[i]) <= hi + 1e-5, (i, got[i], lo, float(u[i]), hi)


def _merge_splits(ops, ws, tokens, heads, head_dim, nsplit, out):
    import ctypes
    vp, i = ctypes.c_void_p, ctypes.c_int
    fn = ops.engine_library().mllm_merge_attention_splits
    fn.argtypes = [vp, i, i, i, i, vp, i, i, vp]
    return fn(ws.data_ptr(), tokens, heads, head_dim, nsplit, out.data_ptr(), out.stride(0), 0 if out.dtype == torch.float32 else 1,
              ctypes.c_void_p(torch.cuda.current_stream().cuda_stream))


# (256 threads are 1,024 / head_dim groups, each for every so-manieth split: one split, fewer than groups, as many, one more, several
# rounds; head sizes that leave threads over, one group, and more elements than threads)
@pytest.mark.parametrize("head_dim,nsplit", [(64, 1), (64, 15), (64, 16), (64, 17), (64, 64), (40, 25), (40, 26), (40, 60), (128, 9), (512, 2), (512, 9),
                                             (516, 5), (1024, 3), (4, 64), (1100, 3), (2048, 2)])
@pytest.mark.parametrize("dtype", DTYPES)
def test_merge_of_splits(ops, head_dim, nsplit, dtype):
    """The states of splits (maximum base 2, sum, unnormalised output) joined, empty ones (maximum -1e30, sum 0) among them. A state
    passes at most two exponentials and two products a merge, in 32 bits (with arguments of at most 40 in all: as many roundings)."""
    tokens, heads, pad = 3, 2, 8
    g = torch.Generator().manual_seed(head_dim + nsplit)
    o = torch.randn(tokens, heads, nsplit, head_dim, generator=g)
    m, l = 8 * torch.rand(tokens, heads, nsplit, generator=g), 1 + 30 * torch.rand(tokens, heads, nsplit, generator=g)
    if nsplit > 1:
        for t in range(tokens):
            empty = [t % nsplit] if nsplit == 2 else [t % nsplit, nsplit - 1]
            m[t, 1, empty], l[t, 1, empty], o[t, 1, empty] = -1.0e30, 0.0, 0.0
    ws = torch.cat([o.reshape(-1), torch.stack([m, l], -1).reshape(-1)]).to(DEV)
    out = torch.full((tokens, heads * head_dim + pad), 7.0, dtype=dtype, device=DEV)
    assert _merge_splits(ops, ws, tokens, heads, head_dim, nsplit, out) == 0
    w = torch.exp2(m.double() - m.double().amax(-1, keepdim=True))
    total = (w * l.double()).sum(-1, keepdim=True)
    want = ((w[..., None] * o.double()).sum(2) / total).reshape(tokens, -1)
    size = ((w[..., None] * o.double().abs()).sum(2) / total).reshape(tokens, -1)
    got = out.cpu().double()
    limit = 2 * 2.0 ** -24 * (40 + 8 * nsplit) * size + (2.0 ** -8 * want.abs() if dtype == torch.bfloat16 else 0)
    assert ((got[:, :heads * head_dim] - want).abs() <= limit).all()
    assert (got[:, heads * head_dim:] == 7).all()


@pytest.mark.parametrize("nsplit", [9, 15, 17, 21, 33, 64])
def test_merge_of_splits_rounds_no_more_than_one_weight_a_split(ops, nsplit):
    """In 32 bits the error against float64 is no larger than that of one weight for every split, sums in their order
    and the sum's reciprocal (the kernel's own last step, two roundings)."""
    tokens, heads, head_dim = 64, 12, 64
    g = torch.Generator().manual_seed(nsplit)
    o = torch.randn(tokens, heads, nsplit, head_dim, generator=g)
    m, l = torch.randn(tokens, heads, nsplit, generator=g), 1 + 30 * torch.rand(tokens, heads, nsplit, generator=g)
    out = torch.empty(tokens, heads * head_dim, device=DEV)
    assert _merge_splits(ops, torch.cat([o.reshape(-1), torch.stack([m, l], -1).reshape(-1)]).to(DEV), tokens, heads, head_dim, nsplit, out) == 0

    def plain(dtype):
        w = torch.exp2(m.to(dtype) - m.amax(-1, keepdim=True).to(dtype))
        total, sums = torch.zeros(tokens, heads, 1, dtype=dtype), torch.zeros(tokens, heads, head_dim, dtype=dtype)
        for s in range(nsplit):
            total += (w * l.to(dtype))[..., s:s + 1]
            sums += w[..., s:s + 1] * o[:, :, s].to(dtype)
        return (sums * (1 / total)).reshape(tokens, -1)

    want = plain(torch.float64)
    assert (out.cpu().double() - want).norm() <= (plain(torch.float32).double() - want).norm()


def test_merge_of_splits_refuses(ops):
    ws, out = torch.zeros(64, device=DEV), torch.zeros(1, 64, device=DEV)
    for tokens, heads, head_dim, nsplit in ((1, 1, 0, 1), (1, 1, -4, 1), (1, 1, 6, 1), (1, 0, 8, 1), (1, -1, 8, 1), (1, 1, 8, 0)):
        assert _merge_splits(ops, ws, tokens, heads, head_dim, nsplit, out) == -1
    assert _merge_splits(ops, ws, 0, 1, 8, 1, out) == 0


def test_sample_edge_rows(ops):
    """All mass on one entry, a flat row, u at both ends, masses that underflow to zero."""
    V = 5000
    logits = torch.full((6, V), -50.0)
    logits[0, 4321] = 30.0
    logits[1] = 0.0
    logits[2] = 0.0
    logits[3, V - 1] = 30.0
    logits[4, 0] = 30.0
    logits[5, 2047:2050] = 5.0                      # the mass straddles a tile edge
    u = torch.tensor([0.5, 0.0, 0.99999994, 0.99999994, 0.0, 0.5])
    temps = torch.full((6,), 1.0)
    out = torch.empty(6, dtype=torch.int32, device=DEV)
    ops.sample(logits.to(DEV), temps.to(DEV), u.to(DEV), out)
    got = out.cpu().tolist()
    assert got[0] == 4321 and got[1] == 0 and got[2] == V - 1 and got[3] == V - 1 and got[4] == 0
    assert got[5] == 2048


def test_sample_frequencies_follow_softmax(ops):
    logits = torch.tensor([[0.0, 1.0, 2.0, -1.0]]).repeat(4096, 1)
    g = torch.Generator().manual_seed(11)
    u = torch.rand(4096, generator=g)
    temps = torch.full((4096,), 0.8)
    out = torch.empty(4096, dtype=torch.int32, device=DEV)
    ops.sample(logits.to(DEV), temps.to(DEV), u.to(DEV), out)
    freq = torch.bincount(out.cpu().long(), minlength=4).double() / 4096
    p = torch.softmax(logits[0].double() / 0.8, 0)
    assert (freq - p).abs().max() < 4 * math.sqrt(0.25 / 4096)


def _entry(library, name, *args):
    """A kernel library's C entry point on the null stream; tensors go in as their addresses, doubles and floats by their ctypes."""
    import ctypes
    from mini_llm_amd import build
    f = getattr(build.load_library(library), name)
    conv = [ctypes.c_void_p(a.data_ptr()) if isinstance(a, torch.Tensor) else ctypes.c_void_p(None) if a is None else
            ctypes.c_int(a) if isinstance(a, int) else a for a in args]
    torch.cuda.synchronize()
    rc = f(*conv)
    torch.cuda.synchronize()
    return rc


@pytest.mark.parametrize("D", [4, 64, 252, 256, 260, 512, 516, 768, 1024, 1600, 2048])
def test_a_rows_norm_has_the_same_bits_among_few_and_many(D):
    """The RMS norms and those that go into the stream, 8 rows and 600 (other instances), around the 256 columns that an instance has: the same
    bits."""
    import ctypes
    g = torch.Generator().manual_seed(D)
    x, res, w, gate, nx = (_rand(s, torch.float32, g, std=2.0).to(DEV) for s in ((600, D), (600, D), (D,), (600, D), (D,)))
    eps, mult = ctypes.c_float(1e-5), ctypes.c_float(0.7)
    for use_gate in (False, True):
        outs = []
        for n in (8, 600):
            y = torch.zeros(n, D, device=DEV)
            assert _entry("norm_gate", "mllm_rmsnorm", x, D, None, w, gate if use_gate else None, D, y, D, n, D, 1, eps, 0, 1, ctypes.c_size_t(0), None) == 0
            outs.append(y)
        assert torch.equal(outs[0], outs[1][:8])
    for center in (0, 1):
        outs = []
        for n in (8, 600):
            y, s = x[:n].clone(), res[:n].clone()
            assert _entry("norm_gate", "mllm_norm_add", y, w, None, None, mult, eps, s, n, D, 0, center, None, None) == 0
            outs.append(s)
        assert torch.equal(outs[0], outs[1][:8])
    outs = []
    for n in (8, 600):
        y, s, c = x[:n].clone(), res[:n].clone(), torch.zeros(n, D, dtype=torch.bfloat16, device=DEV)
        assert _entry("norm_gate", "mllm_rmsnorm_add_norm", y, w, None, mult, eps, s, n, D, 0, nx, eps, c, None) == 0
        outs.append((s, c))
    assert torch.equal(outs[0][0], outs[1][0][:8]) and torch.equal(outs[0][1], outs[1][1][:8])


@pytest.mark.parametrize("M", [1, 2, 3, 8])
@pytest.mark.parametrize("N,K", [(2048, 4), (2050, 252), (2304, 256), (2048, 260), (2304, 768), (4096, 1024), (4097, 772), (4800, 1600), (2056, 2044),
                                 (6400, 2048)])
@pytest.mark.parametrize("epi", ["store", "gelu_tanh"])
def test_rms_norm_fp32_inside_has_the_bits_of_norm_and_product(ops, M, N, K, epi):
    """The RMS form of the 32-bit norm inside the few-row product, around every 256 columns of K, with one column a wavefront and with two."""
    import ctypes
    g = torch.Generator().manual_seed(M + N + K)
    x = _rand((M, K), torch.float32, g, std=2.0) + 0.3
    w, weight, bias = _rand((N, K), torch.float32, g, std=1.0 / math.sqrt(K)), 1 + 0.1 * _rand((K,), torch.float32, g), 0.5 * _rand((N,), torch.float32, g)
    mode, eps = ops.EPILOGUES[epi], ctypes.c_float(1e-5)
    for b in (bias.to(DEV), None):
        inside, apart = (torch.full((M, N), 7.0, device=DEV) for _ in range(2))
        h = torch.full((M, K), 7.0, device=DEV)
        assert _entry("gemm_f32", "mllm_norm_gemm_f32", x.to(DEV), K, weight.to(DEV), None, eps, 1, w.to(DEV), K, b, inside, N, M, N, K, mode, None) == 0
        assert _entry("norm_gate", "mllm_rmsnorm", x.to(DEV), K, None, weight.to(DEV), None, 0, h, K, M, K, 1, eps, 0, 1, ctypes.c_size_t(0), None) == 0
        assert _entry("gemm_f32", "mllm_gemm_f32", h, K, w.to(DEV), K, b, apart, N, M, N, K, mode, None) == 0
        assert torch.equal(inside, apart)
    norm = x.double() / (x.double().square().mean(1, keepdim=True) + 1e-5).sqrt() * weight.double()
    ref = plain_ops.linear(norm, w.double(), None, torch.zeros(M, N, dtype=torch.float64), epi)
    assert (inside.cpu().double() - ref).abs().max().item() <= 3e-5          # (as for the LayerNorm)


@pytest.mark.parametrize("dtype", DTYPES)
def test_decode_attention_of_first_tokens_without_a_table(dtype):
    """Tokens at position 0 whose keys stand in their own rows alone: a table of no entries is not read, and the result is the value."""
    import ctypes
    T, H, dh = 3, 4, 64
    D, g = H * dh, torch.Generator().manual_seed(5)
    q = _rand((T, 3 * D), dtype, g)
    qd, out, pages = q.to(DEV), torch.zeros(T, D, dtype=dtype, device=DEV), [torch.zeros(32, D, dtype=dtype, device=DEV) for _ in range(2)]
    ws, counters = torch.zeros(T * H * (dh + 2), device=DEV), torch.zeros(T * H, dtype=torch.int32, device=DEV)
    positions, slots = torch.zeros(T, dtype=torch.int32, device=DEV), torch.tensor([17, 3, -1], dtype=torch.int32, device=DEV)
    assert _entry("attention_decode", "mllm_decode_attention", qd, 3 * D, 0, *pages, D, None, 0, None, positions, T, H, H, dh, 16, ctypes.c_float(dh ** -0.5), 0, 1, 4,
                  out, D, ws, counters, D, 2 * D, slots, 0, 0 if dtype == torch.float32 else 1, None, None, None, 0) == 0
    assert torch.equal(out.cpu(), q[:, 2 * D:])
    assert torch.equal(pages[0][[17, 3]].cpu(), q[:2, D:2 * D]) and torch.equal(pages[1][[17, 3]].cpu(), q[:2, 2 * D:])


@pytest.mark.parametrize("T", [1, 15, 16, 17, 63, 64, 65, 130])
@pytest.mark.parametrize("H,Dn,Dr,R,Dv,rot,half", [(12, 64, 32, 256, 64, 32, 0), (5, 32, 16, 128, 96, 8, 1), (1, 96, 32, 512, 40, 32, 0), (7, 128, 64, 96, 128, 64, 1),
                                                   (6, 64, 0, 100, 72, 0, 0)])
@pytest.mark.parametrize("wide", [False, True])          # queries in 32 bits, results behind a gate
def test_latent_products_per_head(T, H, Dn, Dr, R, Dv, rot, half, wide):
    """Queries into the latent space and results out of it: up to 16 tokens (a kernel of their own) and more, heads that are no multiple of 4,
    output columns that are no multiple of 64, and the turned columns next to their angles in double."""
    import ctypes
    g = torch.Generator().manual_seed(T + R + H)
    E, q_dtype = R + Dr, torch.float32 if wide else torch.bfloat16
    q, w = _rand((T, H * (Dn + Dr)), q_dtype, g), _rand((R, H * Dn), torch.bfloat16, g, std=Dn ** -0.5)
    pos = torch.randint(0, 8000, (T,), generator=g, dtype=torch.int32)
    qa = torch.full((T, H * E), float("nan"), dtype=torch.bfloat16, device=DEV)
    assert _entry("latent_attention", "mllm_latent_absorb", q.to(DEV), H * (Dn + Dr), w.to(DEV), H * Dn, qa, H * E, pos.to(DEV), T, H, Dn, Dr, R,
                  ctypes.c_double(1e4), rot, 1, None, 0 if wide else 1, half) == 0
    rows = q.view(T, H, Dn + Dr).double()
    plain = rows[..., :Dn].bfloat16().double()
    want = torch.einsum("thd,rhd->thr", plain, w.view(R, H, Dn).double())
    size = torch.einsum("thd,rhd->thr", plain.abs(), w.view(R, H, Dn).double().abs())
    tail = rows[..., Dn:].clone()
    i = torch.arange(rot // 2)
    a, b = (i, i + rot // 2) if half else (2 * i, 2 * i + 1)
    if rot:
        angle = pos.double()[:, None, None] * 1e4 ** (-2.0 * i.double() / rot)
        tail[..., a], tail[..., b] = (rows[..., Dn + a] * angle.cos() - rows[..., Dn + b] * angle.sin(), rows[..., Dn + b] * angle.cos() + rows[..., Dn + a] * angle.sin())
    got = qa.cpu().view(T, H, E).double()
    # one rounding to 8 bits of mantissa, 32-bit sums before it
    assert ((got[..., :R] - want).abs() <= 2.0 ** -8 * want.abs() + 2.0 ** -22 * size).all()
    assert ((got[..., R:] - tail).abs() <= 2.0 ** -8 * tail.abs() + 2.0 ** -20).all()
    if R % 32:
        return
    o, wv = _rand((T, H * R), torch.bfloat16, g), _rand((H * Dv, R), torch.bfloat16, g, std=R ** -0.5)
    gate = _rand((T, H), torch.float32, g) if wide else None
    out = torch.full((T, H * Dv), float("nan"), dtype=torch.bfloat16, device=DEV)
    assert _entry("latent_attention", "mllm_latent_expand", o.to(DEV), H * R, wv.to(DEV), R, out, H * Dv, T, H, Dv, R, 1, None,
                  gate.to(DEV) if wide else None, H if wide else 0) == 0
    want = torch.einsum("thr,hvr->thv", o.view(T, H, R).double(), wv.view(H, Dv, R).double())
    size = torch.einsum("thr,hvr->thv", o.view(T, H, R).double().abs(), wv.view(H, Dv, R).double().abs())
    if wide:
        want, size = want * torch.sigmoid(gate.double())[..., None], size * torch.sigmoid(gate.double())[..., None]
    assert ((out.cpu().view(T, H, Dv).double() - want).abs() <= 2.0 ** -8 * want.abs() + 2.0 ** -21 * size).all()


@pytest.mark.parametrize("C,taps", [(4, 2), (252, 4), (256, 3), (260, 8), (1792, 4), (1028, 5)])
@pytest.mark.parametrize("T", [1, 8])
def test_conv_of_one_token_a_sequence(T, C, taps):
    """Around a workgroup's 256 channels: results, the carried rows moved up by one, and a sequence without a slot left alone."""
    import ctypes
    g = torch.Generator().manual_seed(C + taps + T)
    ld, slot_floats = C + 8, (taps - 1) * C + 12
    x, w, bias = _rand((T, ld), torch.float32, g), _rand((C, taps), torch.float32, g), _rand((C,), torch.float32, g)
    state = _rand((T + 1, slot_floats), torch.float32, g)
    slots = torch.randperm(T + 1, generator=g)[:T].int()
    if T > 1:
        slots[2] = -1
    seq, cu = torch.arange(T, dtype=torch.int32), torch.arange(T + 1, dtype=torch.int32)
    out, dev_state = torch.full((T, C), 7.0, device=DEV), state.clone().to(DEV)
    assert _entry("ssm", "mllm_conv_silu", x.to(DEV), ld, 4, C, w.to(DEV), bias.to(DEV), taps, seq.to(DEV), cu.to(DEV), slots.to(DEV), dev_state,
                  ctypes.c_size_t(slot_floats), out, C, T, T, 1, None) == 0
    want, after = torch.full((T, C), 7.0, dtype=torch.float64), state.clone()
    for t in range(T):
        if slots[t] < 0:
            continue
        rows = torch.cat([state[slots[t], :(taps - 1) * C].view(taps - 1, C), x[t:t + 1, 4:4 + C]])
        v = bias.double() + (w.double().T * rows.double()).sum(0)
        want[t] = v * torch.sigmoid(v)
        after[slots[t], :(taps - 1) * C] = rows[1:].reshape(-1)
    assert torch.equal(dev_state.cpu(), after)
    # a rounding of 2^-24 for each of up to nine terms of up to about 16, and the exponential's
    assert (out.cpu().double() - want).abs().max() <= 9 * 16 * 2.0 ** -23


@pytest.mark.parametrize("R,Dr", [(64, 32), (256, 32), (512, 32)])
@pytest.mark.parametrize("nsplit", [2, 4, 5, 8, 9, 12, 13, 16, 17, 20])
def test_latent_attention_merges_every_number_of_splits(R, Dr, nsplit):
    """The splits' states merged, around every four splits whose columns are asked for together, next to the same kernel without splits."""
    import ctypes
    g = torch.Generator().manual_seed(R + nsplit)
    H, page, ctx, B = 5, 16, 64 * 20 + 7, 2
    E, n_pages = R + Dr, -(-ctx // page)
    qa = (_rand((B * H, E), torch.bfloat16, g)).to(DEV)
    pages = _rand((B * n_pages, page, E), torch.bfloat16, g)
    vt = pages[..., :R].transpose(1, 2).contiguous().to(DEV)
    tables = torch.randperm(B * n_pages, generator=g).int().view(B, n_pages).to(DEV)
    cu, lens = torch.arange(B + 1, dtype=torch.int32, device=DEV), torch.tensor([ctx, 3 * 64], dtype=torch.int32, device=DEV)
    outs = []
    for n in (1, nsplit):
        out = torch.full((B * H, R), float("nan"), dtype=torch.bfloat16, device=DEV)
        part = torch.full((B * H * n * (R + 2),), float("nan"), device=DEV)
        assert _entry("latent_attention", "mllm_latent_attention_tiles", qa, pages.to(DEV), vt, tables, n_pages, cu, lens, B, B, H, R, Dr, page,
                      ctypes.c_float(E ** -0.5), 0, out, B * H, n, part, 1, None) == 0
        outs.append(out.cpu().double())
    # weights are 16-bit operands of the second product: each split's maximum moves their rounding (2^-9 of each, at most 2^-8 of values of up to about 4)
    assert (outs[0] - outs[1]).abs().max() <= 2.0 ** -6
