"""Kugulorn through the engine on the GPU against the plain implementation (tests/plain_kugulorn.py), in
32-bit and in bfloat16: each mechanism alone, whole prompts against token-by-token decoding, portions down
to two tokens, mixed batches against each request alone, pages and state slots that are used again, keys at
window and page borders, the first tokens, long decoding, and greedy generation through the engine's own
entry point and scheduler."""
import numpy as np
import pytest

import kugulorn_cases as kc
import plain_kugulorn as pk
import replay_util as ru

pytestmark = pytest.mark.gpu
DTYPES = ["float32", "bfloat16"]


@pytest.fixture(scope="module")
def dirs(tmp_path_factory):
    from mini_llm_amd import write_random_model
    made = {}

    def get(name, seed=3):
        if name not in made:
            d = tmp_path_factory.mktemp("kugulorn_" + name)
            write_random_model(dict(getattr(kc, name)), str(d), seed)
            made[name] = str(d)
        return made[name]
    return get


def _runner(model_dir, dtype, n_pages, page=4, max_num_seqs=4):
    from mini_llm_amd import Runner
    r = Runner(model_dir=model_dir, dtype=dtype, page_size=page, n_pages=n_pages, max_num_seqs=max_num_seqs)
    r.poison_cache()               # a stale or unwritten page or slot that is read shows up as NaN
    return r


def _families(reqs, seed):
    mixed, _ = ru.trace_mixed(reqs, seed=seed, max_live=4, tail=6)
    return {"whole": ru.trace_whole(reqs), "decode": ru.trace_decode_tail(reqs, tail=11),
            "chunks": ru.trace_chunks(reqs, seed=seed), "mixed": mixed}


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("name", ["ONLY_MAMBA", "ONLY_MAMBA_WIDE_STATE", "ONLY_LATENT", "ONLY_LATENT_MLP"])
def test_each_mechanism_alone(dirs, name, dtype):
    cfg, d = getattr(kc, name), dirs(name)
    # (portions of more than 64 tokens: the scan cuts them into chunks that run side by side)
    reqs = kc.requests(cfg["vocab"], [1, 2, 3, 9, 37, 64, 65, 200], seed=5)
    for label, steps in (("whole", ru.trace_whole(reqs)), ("chunks", ru.trace_chunks(reqs, seed=1)),
                         ("long chunks", ru.trace_chunks(reqs, seed=1, sizes=(70, 3, 129)))):
        runner = _runner(d, dtype, n_pages=ru.peak_tokens(steps) // 4)
        kc.check_against_plain(d, reqs, steps, ru.run_in_process(runner, steps), dtype, cfg["vocab"], f"{name} {label}")
        assert runner.check() == "" and runner.info()["n_requests"] == 0


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("name", ["MIXED_A", "MIXED_B", "ODD"])
@pytest.mark.parametrize("family", ["whole", "decode", "chunks", "mixed"])
def test_schedule_families_match_plain(dirs, name, family, dtype):
    """Each request whole; most of it at once and the rest token by token; portions down to two tokens; up to
    four live requests in mixed batches. The pool holds just the peak of live tokens and there are four state
    slots for seven requests, so pages and slots are used again (and were filled with NaN before)."""
    cfg, d = getattr(kc, name), dirs(name)
    reqs = kc.requests(cfg["vocab"], [1, 2, 3, 4, 5, 29, 64, 71] + ([150] if name == "ODD" else []), seed=11)
    steps = _families(reqs, seed=2)[family]
    n_pages = ru.peak_tokens(steps) // 4
    runner = _runner(d, dtype, n_pages)
    kc.check_against_plain(d, reqs, steps, ru.run_in_process(runner, steps), dtype, cfg["vocab"], f"{name} {family}")
    info = runner.info()
    assert runner.check() == "" and info["free_pages"] == n_pages and info["n_requests"] == 0


@pytest.mark.parametrize("page", [8, 16, 64])
@pytest.mark.parametrize("family", ["whole", "decode", "chunks", "mixed"])
def test_prompt_portions_on_the_matrix_cores(dirs, family, page):
    """bfloat16 at sizes and page sizes that the matrix-core kernel takes: prompts of up to 300 tokens (several
    key tiles, windows that end inside a tile), portions, and mixed batches whose single tokens ride along."""
    from mini_llm_amd.kernels import ops
    cfg, d = kc.TILED, dirs("TILED")
    reqs = kc.requests(cfg["vocab"], [1, 2, 17, 63, 64, 65, 130, 300], seed=71)
    steps = _families(reqs, seed=6)[family]
    ops.reset_seen()
    runner = _runner(d, "bfloat16", n_pages=-(-ru.peak_tokens(steps) // page), page=page)
    kc.check_against_plain(d, reqs, steps, ru.run_in_process(runner, steps), "bfloat16", cfg["vocab"], f"tiled page {page} {family}")
    assert ops.seen("latent_tile_launches") > 0
    assert runner.check() == "" and runner.info()["n_requests"] == 0


@pytest.mark.parametrize("name,page", [("TILED", 16), ("ODD", 4)])
def test_norms_of_neighbouring_layers_join_from_33_rows(dirs, name, page):
    """Up to 32 rows a layer's first products take their norm inside; from 33 on the norm behind the layer in front leaves it. Portions on
    both sides of the line, and one that ends a request which began on the other side."""
    cfg, d = getattr(kc, name), dirs(name)
    reqs = kc.requests(cfg["vocab"], [31, 32, 33, 34, 65], seed=75)
    for label, steps in (("whole", ru.trace_whole(reqs)), ("chunks", ru.trace_chunks(reqs, seed=3, sizes=(33, 32)))):
        runner = _runner(d, "bfloat16", n_pages=ru.peak_tokens(steps) // page, page=page)
        kc.check_against_plain(d, reqs, steps, ru.run_in_process(runner, steps), "bfloat16", cfg["vocab"], f"{name} {label}")
        assert runner.check() == "" and runner.info()["n_requests"] == 0


@pytest.mark.parametrize("name,page", [("TILED", 16), ("ODD", 4)])
def test_norms_of_neighbouring_layers_join_with_the_same_bits(dirs, name, page):
    """The norm is left by the layer in front in steps of 33 and more rows and in no others, for every layer but the first, and the logits are those
    of the two norms on their own."""
    from mini_llm_amd.kernels import ops
    cfg, d = getattr(kc, name), dirs(name)
    got = []
    try:
        for on in (True, False):
            ops.set_joined_norms(on)
            runner = _runner(d, "bfloat16", n_pages=-(-65 // page), page=page)
            got.append([])
            for n in (31, 32, 33, 65):
                ops.reset_seen()
                steps = ru.trace_whole(kc.requests(cfg["vocab"], [n], seed=n))
                got[-1].append(ru.run_in_process(runner, steps)[0])
                assert ops.seen("joined_norms") == (len(cfg["layers"]) - 1 if on and n > 32 else 0)
    finally:
        ops.set_joined_norms(True)
    assert all(np.isfinite(a).all() and np.array_equal(a, b) for a, b in zip(*got))


@pytest.mark.parametrize("family", ["whole", "mixed"])
def test_widest_rows_on_the_matrix_cores(dirs, family):
    from mini_llm_amd.kernels import ops
    cfg, d = kc.WIDE, dirs("WIDE")
    reqs = kc.requests(cfg["vocab"], [3, 70, 129, 260], seed=73)
    steps = _families(reqs, seed=7)[family]
    ops.reset_seen()
    runner = _runner(d, "bfloat16", n_pages=ru.peak_tokens(steps) // 16, page=16)
    kc.check_against_plain(d, reqs, steps, ru.run_in_process(runner, steps), "bfloat16", cfg["vocab"], f"wide {family}")
    assert ops.seen("latent_tile_launches") > 0 and ops.seen("latent_token_launches") == 0


def test_matrix_core_kernel_against_the_per_token_kernel(dirs):
    """The same whole prompts with the matrix-core kernel switched off: both kernels round differently, no more."""
    from mini_llm_amd.kernels import ops
    cfg, d = kc.TILED, dirs("TILED")
    reqs = kc.requests(cfg["vocab"], [5, 100, 257], seed=72)
    steps = ru.trace_whole(reqs)
    got = []
    try:
        for on in (True, False):
            ops.set_latent_tiles(on)
            ops.reset_seen()
            runner = _runner(d, "bfloat16", n_pages=ru.peak_tokens(steps) // 16, page=16)
            got.append(ru.collect(steps, ru.run_in_process(runner, steps), cfg["vocab"]))
            assert (ops.seen("latent_tile_launches") > 0) == on
    finally:
        ops.set_latent_tiles(True)
    worst = max(kc.row_error(got[0][r][p], got[1][r][p].astype(np.float64)) for r in reqs for p in range(len(reqs[r])))
    print(f"matrix-core kernel against the per-token kernel: {worst:.3e}")
    assert worst <= 2e-2


@pytest.mark.parametrize("page", [2, 4, 16])
def test_window_and_page_borders_with_peaked_scores(dirs, page):
    """Scores scaled so that single keys dominate, windows of 5, 6 and 16 over pages of 2, 4 and 16 tokens: a
    window that is one key off or a key lost at a page's border changes whole rows. Prompts and decoding."""
    cfg, d = kc.PEAKED, dirs("PEAKED")
    reqs = kc.requests(cfg["vocab"], [40, 23, 17], seed=21)
    for label, steps in (("whole", ru.trace_whole(reqs)), ("decode", ru.trace_decode_tail(reqs, tail=19)),
                         ("chunks", ru.trace_chunks(reqs, seed=3, sizes=(2, 5, 3, 16, 7, 2, 4)))):
        runner = _runner(d, "float32", n_pages=-(-ru.peak_tokens(steps) // page), page=page)
        kc.check_against_plain(d, reqs, steps, ru.run_in_process(runner, steps), "float32", cfg["vocab"], f"peaked page {page} {label}",
                               tol=kc.TOL_PEAKED)


@pytest.mark.parametrize("page", [4, 16])
def test_far_keys_among_hundreds_with_peaked_scores(dirs, page):
    """Windows of 300 and 190 keys and scores that single keys dominate: a key far back that is lost (a page of the
    table, a tile's edge, a window that ends early) changes whole rows. Prompts, portions and decoding, 32-bit."""
    cfg, d = kc.PEAKED_FAR, dirs("PEAKED_FAR")
    reqs = kc.requests(cfg["vocab"], [330, 200], seed=23)
    for label, steps in (("whole", ru.trace_whole(reqs)), ("decode", ru.trace_decode_tail(reqs, tail=40)),
                         ("chunks", ru.trace_chunks(reqs, seed=4, sizes=(2, 70, 3, 129, 16)))):
        runner = _runner(d, "float32", n_pages=-(-ru.peak_tokens(steps) // page), page=page)
        kc.check_against_plain(d, reqs, steps, ru.run_in_process(runner, steps), "float32", cfg["vocab"], f"far keys page {page} {label}",
                               tol=kc.TOL_PEAKED)


def test_peaked_scores_would_show_a_window_one_key_off(dirs):
    """The test above has teeth: the plain model with every window one key wider differs from the plain model
    by far more than the tolerance, in most rows."""
    import copy
    d = dirs("PEAKED")
    cfg, w = pk.read_model(d)
    off = copy.deepcopy(cfg)
    for l in off["layers"]:
        l["mixer"]["mask"]["size"] += 1
    toks = kc.requests(cfg["vocab"], [40], seed=21)["r0"]
    a, b = pk.forward(cfg, w, toks).numpy(), pk.forward(off, w, toks).numpy()
    errs = np.array([kc.row_error(b[p], a[p]) for p in range(8, 40)])
    assert (errs > 20 * kc.TOL_PEAKED).mean() > 0.8


@pytest.mark.parametrize("dtype", DTYPES)
def test_long_decoding_and_slots_used_again(dirs, dtype):
    """One state slot and a small pool: three requests one after the other, each a short prompt and then 150
    tokens one by one, every one of them compared; the slot and the pages are the same ones each time."""
    cfg, d = kc.MIXED_A, dirs("MIXED_A")
    reqs = kc.requests(cfg["vocab"], [153, 151, 152], seed=31)
    steps = ru.trace_decode_tail(reqs, tail=150)
    runner = _runner(d, dtype, n_pages=40, max_num_seqs=1)
    kc.check_against_plain(d, reqs, steps, ru.run_in_process(runner, steps), dtype, cfg["vocab"], "long decoding")
    assert runner.check() == "" and runner.info()["free_pages"] == 40


def test_batches_of_unequal_requests_equal_each_alone(dirs):
    """The logits of a position do not depend on what else is in the batch, beyond rounding: the mixed family's
    rows against the same requests run whole and alone, engine against engine, in bfloat16."""
    cfg, d = kc.MIXED_B, dirs("MIXED_B")
    reqs = kc.requests(cfg["vocab"], [3, 50, 18, 64, 7], seed=41)
    fam = _families(reqs, seed=4)
    got = {}
    for family in ("whole", "mixed"):
        runner = _runner(d, "bfloat16", n_pages=ru.peak_tokens(fam[family]) // 4)
        got[family] = ru.collect(fam[family], ru.run_in_process(runner, fam[family]), cfg["vocab"])
    worst = max(kc.row_error(got["mixed"][r][p], got["whole"][r][p].astype(np.float64)) for r in reqs for p in range(len(reqs[r])))
    print(f"mixed against alone, bfloat16: {worst:.3e}")
    assert worst <= 2e-2


@pytest.mark.parametrize("dtype", DTYPES)
def test_trace_run_program(dirs, tmp_path, dtype):
    """The mixed family through bin/trace_run as a user drives it (its default page size and four state slots)."""
    cfg, d = kc.MIXED_A, dirs("MIXED_A")
    reqs = kc.requests(cfg["vocab"], [2, 33, 64, 5, 70, 21], seed=51)
    steps, _ = ru.trace_mixed(reqs, seed=5, max_live=4, tail=5)
    out = ru.run_trace_run(d, dtype, steps, str(tmp_path / "out"), ru.peak_tokens(steps))
    kc.check_against_plain(d, reqs, steps, out, dtype, cfg["vocab"], "program mixed")


@pytest.mark.parametrize("dtype", DTYPES)
def test_greedy_generation_through_the_engine(dirs, dtype):
    """Engine.generate (scheduler, continuous batching, prompt portions of 7 tokens, two requests at a time for
    five prompts, pages of 4) against the plain model's greedy tokens."""
    import torch
    from mini_llm_amd import Engine, EngineOptions, SamplingParams
    cfg_d, d = kc.MIXED_A, dirs("MIXED_A")
    cfg, w = pk.read_model(d)
    prompts = list(kc.requests(cfg_d["vocab"], [1, 6, 19, 30, 11], seed=61).values())
    engine = Engine.from_pretrained(d, dtype=dtype, options=EngineOptions(kv_block_size=4, total_kv_blocks=64, max_batch_num=2,
                                                                          max_tokens_per_step=16, prefill_chunk=7))
    outs = engine.generate(prompts, SamplingParams(max_new_tokens=9, ignore_eos=True))
    for p, o in zip(prompts, outs):
        assert len(o) == 9
        if dtype == "float32":
            assert o == pk.greedy_generate(cfg, w, p, 9)
        else:
            # bfloat16 may turn a near-tie: every token must be one the plain model chose or nearly chose
            ids = list(p)
            for t in o:
                row = pk.forward(cfg, w, ids)[-1]
                assert float(row[t]) >= float(row.max()) - 0.08 * float(row.std()), (o, t)
                ids.append(t)


@pytest.mark.parametrize("heads,vdim,state,groups,conv", [(2, 64, 128, 1, 4), (3, 68, 36, 1, 4),      # a second tile of 4 columns; a slice of 4 rows
                                                          (4, 8, 20, 2, 2), (2, 16, 160, 1, 9),      # five slices: two rounds; more taps than vector loads
                                                          (2, 6, 10, 1, 3)])                         # sizes that are no whole 16 bytes
@pytest.mark.parametrize("sizes", [(8, 9, 64), (65, 1, 200, 7), (63, 128, 129, 2)])
def test_scan_portions_of_every_length(tmp_path, heads, vdim, state, groups, conv, sizes):
    """The scan's kernels at their borders, in 32 bits: portions of at most 8 and 64 tokens, of several chunks and of one more
    than that, side by side in one step and carried from step to step, with decoded tokens among them."""
    from mini_llm_amd import write_random_model
    cfg = kc.model([kc.mamba(heads=heads, vdim=vdim, state=state, groups=groups, conv=conv, norm_groups=1)], vocab=200, width=48)
    write_random_model(dict(cfg), str(tmp_path), 5)
    reqs = kc.requests(cfg["vocab"], [1, 8, 9, 64, 65, 129, 193, 280], seed=heads + state)
    steps, _ = ru.trace_mixed(reqs, seed=state, max_live=4, tail=3, sizes=sizes)
    runner = _runner(str(tmp_path), "float32", n_pages=ru.peak_tokens(steps) // 4)
    kc.check_against_plain(str(tmp_path), reqs, steps, ru.run_in_process(runner, steps), "float32", cfg["vocab"], f"scan {sizes}")
    assert runner.check() == ""


# (rows: one or two row tiles behind the norm, then the smallest and the larger tiles; columns: less than a tile, no whole tile,
# whole ones; K with and without a remainder of the k tile)
@pytest.mark.parametrize("rows", [1, 8, 9, 16, 17, 32, 33, 64, 65, 130, 513])
@pytest.mark.parametrize("ff,k", [(16, 64), (40, 72), (200, 768), (2048, 768), (1000, 1608), (200, 2112)])
def test_gate_and_up_in_one_product(rows, ff, k):
    """Gate, up map and clamped activation in one kernel, with the RMS norm inside (few rows) and without."""
    import ctypes
    import torch
    from mini_llm_amd.kernels import ops
    lib = ops.engine_library()
    vp, i, f = ctypes.c_void_p, ctypes.c_int, ctypes.c_float
    g = torch.Generator().manual_seed(rows * 7 + ff + k)
    x = torch.randn(rows, k, generator=g)
    gamma = 1 + 0.1 * torch.randn(k, generator=g)
    gate, up = (torch.randn(ff, k, generator=g) * (2.0 / k ** 0.5) for _ in range(2))
    gate, up = gate.bfloat16(), up.bfloat16()
    limit, alpha, eps = 3.0, 1.702, 1e-5
    fused = rows <= 32 and k <= 2048           # (wider norms stay outside)
    a = (pk.rms_norm(x.double(), gamma.double(), eps) if fused else x).bfloat16()
    gv, uv = (torch.clamp(a.double() @ gate.double().T, max=limit), torch.clamp(a.double() @ up.double().T, min=-limit, max=limit))
    want = gv * torch.sigmoid(alpha * gv) * (uv + 1)
    dev = [t.cuda() for t in (x, gamma, gate, up, a)]
    out = torch.full((rows + 1, ff + 8), 7.0, dtype=torch.bfloat16, device="cuda")      # (what lies beside the result stays)
    if fused:
        fn = lib.mllm_rms_gated_gemm_bf16
        fn.argtypes = [vp, i, vp, f, vp, vp, i, f, f, vp, i, i, i, i, vp]
        rc = fn(dev[0].data_ptr(), k, dev[1].data_ptr(), eps, dev[2].data_ptr(), dev[3].data_ptr(), k, limit, alpha, out.data_ptr(), ff + 8, rows, ff, k, None)
    else:
        fn = lib.mllm_gated_gemm_bf16
        fn.argtypes = [vp, i, vp, vp, i, f, f, vp, i, i, i, i, vp]
        rc = fn(dev[4].data_ptr(), k, dev[2].data_ptr(), dev[3].data_ptr(), k, limit, alpha, out.data_ptr(), ff + 8, rows, ff, k, None)
    assert rc == 0
    torch.cuda.synchronize()
    got = out.cpu().double()
    assert (got[:, ff:] == 7).all() and (got[rows:] == 7).all()
    # one rounding to bfloat16, fp32 sums; behind the norm a normalised value may round the other way: 2^-8 |h| |w| of a few of
    # the K terms, times the slope of the activation (under 1.1 (limit + 1) in g, limit in u)
    slack = 1e-4 if not fused else 4 * 2.0 ** -8 * 3 * float(gate.abs().max()) * 1.1 * (limit + 1)
    err = (got[:rows, :ff] - want).abs() - 2.0 ** -8 * want.abs()
    assert float(err.max()) <= slack, (float(err.max()), slack)


@pytest.mark.parametrize("rows", [1, 9, 17, 32, 33, 130, 300])
@pytest.mark.parametrize("ff,k", [(1, 64), (5, 200), (18, 768), (1001, 72), (2050, 1608)])
def test_gate_and_up_at_odd_sizes_to_the_last_rounding(rows, ff, k):
    """The same for widths and row strides that fill no vector store, on rows so faint that eps counts in the norm, against a bound
    that a rounding of gate or up before the activation exceeds: half a unit of the result in bfloat16, the fp32 sums' error and,
    behind the norm, those of its values that lie so close to a border of bfloat16 that they may round either way."""
    import ctypes
    import torch
    from mini_llm_amd.kernels import ops
    lib = ops.engine_library()
    vp, i, f = ctypes.c_void_p, ctypes.c_int, ctypes.c_float
    g = torch.Generator().manual_seed(rows * 7 + ff + k)
    x = 0.01 * torch.randn(rows, k, generator=g)
    gamma = 1 + 0.1 * torch.randn(k, generator=g)
    gate, up = ((torch.randn(ff, k, generator=g) * (2.0 / k ** 0.5)).bfloat16() for _ in range(2))
    limit, alpha, eps = 3.0, 1.702, 1e-4            # (the rows' mean square is 1e-4 as well)
    fused = rows <= 32
    normed = pk.rms_norm(x.double(), gamma.double(), eps)
    a = (normed if fused else 100 * x).bfloat16()
    unsure = torch.zeros(rows, k, dtype=torch.float64)
    if fused:          # the norm's relative error: a few roundings and half of those of a sum of k squares over 64 lanes
        delta = (4 + (k / 64 + 8) / 2) * 2.0 ** -24
        unsure = ((normed * (1 + delta)).bfloat16().double() - (normed * (1 - delta)).bfloat16().double()).abs()
    gv, uv = a.double() @ gate.double().T, a.double() @ up.double().T
    sums = [2.0 ** -24 * (k / 16 + 16) * (a.double().abs() @ w.double().abs().T) + unsure @ w.double().abs().T for w in (gate, up)]
    gv, uv = torch.clamp(gv, max=limit), torch.clamp(uv, min=-limit, max=limit)
    want = gv * torch.sigmoid(alpha * gv) * (uv + 1)
    dev = [t.cuda() for t in (x, gamma, gate, up, a)]
    stride = ff + 7 + ff % 2                         # (odd)
    out = torch.full((rows + 1, stride), 7.0, dtype=torch.bfloat16, device="cuda")
    if fused:
        fn = lib.mllm_rms_gated_gemm_bf16
        fn.argtypes = [vp, i, vp, f, vp, vp, i, f, f, vp, i, i, i, i, vp]
        rc = fn(dev[0].data_ptr(), k, dev[1].data_ptr(), eps, dev[2].data_ptr(), dev[3].data_ptr(), k, limit, alpha, out.data_ptr(), stride, rows, ff, k, None)
    else:
        fn = lib.mllm_gated_gemm_bf16
        fn.argtypes = [vp, i, vp, vp, i, f, f, vp, i, i, i, i, vp]
        rc = fn(dev[4].data_ptr(), k, dev[2].data_ptr(), dev[3].data_ptr(), k, limit, alpha, out.data_ptr(), stride, rows, ff, k, None)
    assert rc == 0
    torch.cuda.synchronize()
    got = out.cpu().double()
    assert (got[:, ff:] == 7).all() and (got[rows:] == 7).all()
    # (the activation's slope: under 1.1 (limit + 1) in g, at most limit in u; exponential and reciprocal to 2^-20)
    half_unit = torch.ldexp(torch.ones_like(want), torch.frexp(want.abs() * (1 + 2.0 ** -9))[1] - 9)       # (8 bits)
    bound = half_unit + 2.0 ** -18 * want.abs() + 1.1 * (limit + 1) * sums[0] + limit * sums[1]
    assert ((got[:rows, :ff] - want).abs() <= bound).all()


@pytest.mark.parametrize("rows,width", [(1, 4), (5, 68), (33, 256), (3, 260), (511, 768), (513, 768), (9, 2048)])
def test_norm_behind_a_sub_layer_and_the_next_in_front(rows, width):
    """x += mult scale rmsnorm(y) and the bfloat16 RMS norm of the new x, in one kernel."""
    import ctypes
    import torch
    from mini_llm_amd.kernels import ops
    vp, i, f = ctypes.c_void_p, ctypes.c_int, ctypes.c_float
    fn = ops.engine_library().mllm_rmsnorm_add_norm
    fn.argtypes = [vp, vp, vp, f, f, vp, i, i, i, vp, f, vp, vp]
    g = torch.Generator().manual_seed(rows + width)
    x, y = torch.randn(rows, width, generator=g), torch.randn(rows, width, generator=g)
    w, scale, w2 = (1 + 0.2 * torch.randn(width, generator=g) for _ in range(3))
    mult, eps, eps2 = 0.7, 1e-5, 1e-6
    for clear in (0, 1):
        xd, yd, out = x.cuda(), y.cuda(), torch.full((rows + 1, width), 7.0, dtype=torch.bfloat16, device="cuda")
        dev = [t.cuda() for t in (w, scale, w2)]
        assert fn(yd.data_ptr(), dev[0].data_ptr(), dev[1].data_ptr(), mult, eps, xd.data_ptr(), rows, width, clear, dev[2].data_ptr(), eps2, out.data_ptr(), None) == 0
        torch.cuda.synchronize()
        new = x.double() + mult * scale.double() * pk.rms_norm(y.double(), w.double(), eps)
        want = pk.rms_norm(new, w2.double(), eps2)
        # a row's fp32 sums of `width` squares (relative error under width / 2 * 2^-24 a sum), then one rounding to bfloat16
        tol = (width / 2 + 16) * 2.0 ** -24
        assert float((xd.cpu().double() - new).abs().max()) <= tol * (1 + float(new.abs().max()))
        got = out.cpu().double()
        assert (got[rows:] == 7).all()
        assert float(((got[:rows] - want).abs() - 2.0 ** -8 * want.abs()).max()) <= 4 * tol * (1 + float(want.abs().max()))
        assert torch.equal(yd.cpu(), torch.zeros_like(y) if clear else y)


def _scan_inputs(sizes, heads=2, vdim=68, state=36, seed=0):
    """Inputs of the scan alone: x [T, H, P], B and C [T, 1, N], raw step sizes [T, H], and the heads' dt_bias, A_log and D."""
    import torch
    g = torch.Generator().manual_seed(seed)
    T = sum(sizes)
    made = [torch.randn(T, heads, vdim, generator=g), torch.randn(T, 1, state, generator=g), torch.randn(T, 1, state, generator=g),
            torch.randn(T, heads, generator=g) - 2, 0.1 * torch.randn(heads, generator=g), 0.3 * torch.randn(heads, generator=g), torch.randn(heads, generator=g)]
    return dict(zip(("x", "B", "C", "raw_dt", "dt_bias", "A_log", "D"), made))


def _scan(sizes, given, workspace_floats_off=0):
    """The scan's kernels alone over portions of these sizes, states that start at 0: (y [T, H, P], states [sequences, H, N, P])."""
    import ctypes
    import torch
    from mini_llm_amd.kernels import ops
    lib = ops.engine_library()
    vp, i, sz = ctypes.c_void_p, ctypes.c_int, ctypes.c_size_t
    fn, need = lib.mllm_ssm_scan, lib.mllm_ssm_scan_workspace_floats
    need.argtypes, need.restype = [i] * 5, sz
    fn.argtypes = [vp, i, vp, i, vp, vp, vp, vp, vp, vp, sz, sz, vp, i, sz, i, i, i, i, i, i, i, i, vp, vp]
    T, H, P = given["x"].shape
    N, b = given["B"].shape[-1], len(sizes)
    xbc = torch.cat([given["x"].reshape(T, -1), given["B"][:, 0], given["C"][:, 0]], 1).cuda()
    dev = [given[k].cuda() for k in ("raw_dt", "dt_bias", "A_log", "D")]
    cu_q = torch.tensor(np.cumsum([0] + list(sizes)), dtype=torch.int32, device="cuda")
    slots = torch.arange(b, dtype=torch.int32, device="cuda")
    state = torch.zeros(b, H, N, P, device="cuda")
    shares = lib.mllm_ssm_scan_parts
    shares.argtypes = [vp, i, i, i, i, i, i]
    parts = shares(xbc.data_ptr(), xbc.stride(0), T, max(sizes), H, P, N)
    y = torch.full((parts, T, H, P), 7.0, device="cuda")
    ws = torch.full((need(T, b, H, P, N) + workspace_floats_off,), float("nan"), device="cuda")
    rc = fn(xbc.data_ptr(), xbc.stride(0), dev[0].data_ptr(), H, *(d.data_ptr() for d in dev[1:]), cu_q.data_ptr(), slots.data_ptr(), state.data_ptr(),
            H * N * P, 0, y.data_ptr(), H * P, T * H * P, T, b, max(sizes), H, P, N, 1, 1, ws.data_ptr() + 4 * workspace_floats_off, None)
    assert rc == 0
    torch.cuda.synchronize()
    return y.sum(0).cpu(), state.cpu()


def _scan_plain(sizes, given, magnitudes=False):
    """The same token by token in float64; `magnitudes`: of the terms' absolute values."""
    import torch
    d = {k: v.double() for k, v in given.items()}
    dt = pk.softplus(d["raw_dt"] + d["dt_bias"])
    ys, states, at = [], [], 0
    for n in sizes:
        part = [d[k][at:at + n].abs() if magnitudes else d[k][at:at + n] for k in ("x", "B", "C")]
        y, s = pk.ssm_scan(*part, dt[at:at + n], d["A_log"], d["D"].abs() if magnitudes else d["D"], 1)
        ys.append(y)
        states.append(s)
        at += n
    return torch.cat(ys), torch.stack(states)


@pytest.mark.parametrize("value", [float("inf"), float("-inf"), float("nan")])
@pytest.mark.parametrize("at", [0, 37, 63, 100, 199])
def test_scan_keeps_tokens_before_a_non_finite_value(value, at):
    """An infinite or NaN x (first, last and other tokens of a chunk) reaches its own token and those behind it in its column, as
    token by token; every other value keeps its bits."""
    import torch
    sizes = (200, 70, 5)
    given = _scan_inputs(sizes, seed=at)
    before, _ = _scan(sizes, given)
    given["x"][at, 1, 66] = value
    got, _ = _scan(sizes, given)
    want, _ = _scan_plain(sizes, given)
    assert torch.equal(torch.isfinite(got), torch.isfinite(want)) and not torch.isfinite(got[at:200, 1, 66]).any()
    kept = torch.isfinite(want)
    assert torch.equal(got[kept], before[kept])


@pytest.mark.parametrize("value", [float("inf"), float("nan")])
def test_scan_keeps_a_non_finite_value_in_the_state(value):
    """Decays of about 1e-6 a token: at its chunk's end the token's weight has underflowed, but an infinite or NaN state stays one."""
    import torch
    sizes = (200, 70)
    given = _scan_inputs(sizes, seed=8)
    given["A_log"][:], given["raw_dt"][:] = 1.0, 5.0
    given["x"][70, 1, 3] = value
    y, state = _scan(sizes, given)
    for got, want in zip((y, state), _scan_plain(sizes, given)):
        assert torch.equal(torch.isfinite(got), torch.isfinite(want))
    assert not torch.isfinite(y[70:200, 1, 3]).any() and not torch.isfinite(state[0, 1, :, 3]).any()


@pytest.mark.parametrize("log_rate,raw", [(0.3, 0.0), (100.0, 0.0), (20.0, 3.0), (1.0, 1e30), (3.0, 40.0), (-30.0, -2.0)])
def test_scan_with_decays_of_any_size(log_rate, raw):
    """Rates and step sizes whose decays underflow (infinite in 32 bits for the first head's log rate of 100), and faint ones, beside
    a head of ordinary ones: every token forgets what it has to and nothing else. A sum's error is at most a rounding per term of its
    magnitudes' sum (the state's rows, the tokens of a chunk) and one per unit of the decays' logarithms that still count."""
    import torch
    sizes = (200, 64, 130, 3)
    given = _scan_inputs(sizes, seed=3)
    given["A_log"][0] = log_rate
    given["raw_dt"][20:180:7, 0] = raw
    y, state = _scan(sizes, given)
    for got, want, size in zip((y, state), _scan_plain(sizes, given), _scan_plain(sizes, given, magnitudes=True)):
        assert torch.isfinite(got).all()
        assert ((got.double() - want).abs() <= 2.0 ** -24 * (given["B"].shape[-1] + 64 + 200) * size).all()


def test_scan_takes_a_workspace_at_any_float():
    """A workspace that starts off a 16-byte border (and is of the size asked for) is as good as any other."""
    import torch
    sizes = (200, 70)
    given = _scan_inputs(sizes, seed=5)
    first = _scan(sizes, given)
    for off in (1, 2, 3):
        assert all(torch.equal(a, b) for a, b in zip(first, _scan(sizes, given, off)))


@pytest.mark.parametrize("sizes", [(64,), (9, 64, 1, 33), (64,) * 40, (8, 1, 5), (3,), (64, 65, 8)])
@pytest.mark.parametrize("heads,vdim,state", [(2, 68, 36), (3, 64, 16), (24, 64, 64), (2, 64, 132), (1, 32, 260), (2, 36, 300)])
def test_short_portions_leave_one_share_or_one_a_slice(sizes, heads, vdim, state):
    """Portions of at most 64 tokens on both sides of the rule for shares, states of one slice of 32 rows to ten. A sum's error is at
    most a rounding per term of its magnitudes' sum (the state's rows, the tokens) and one per unit of the decays' logarithms."""
    import torch
    given = _scan_inputs(sizes, heads, vdim, state, seed=state + len(sizes))
    for got, want, size in zip(_scan(sizes, given), _scan_plain(sizes, given), _scan_plain(sizes, given, magnitudes=True)):
        assert ((got.double() - want).abs() <= 2.0 ** -24 * (state + 64 + 200) * size).all()


@pytest.mark.parametrize("sizes", [(70,) * 9, (1, 65, 64, 200, 3, 3, 128, 129, 1) * 8, (1,) * 64 + (130,), (1,) * 63 + (66, 66), (5,) * 130 + (70, 65)])
@pytest.mark.parametrize("vdim,state", [(4, 4), (3, 5)])
def test_scan_finds_chunks_among_many_portions(sizes, vdim, state):
    """More than 8 sequences: their chunks are counted 64 at a time, on both sides of that and of portions of one chunk (in matrix form,
    and at widths that only the scan token by token takes)."""
    import torch
    given = _scan_inputs(sizes, 1, vdim, state, seed=len(sizes))
    for got, want, size in zip(_scan(sizes, given), _scan_plain(sizes, given), _scan_plain(sizes, given, magnitudes=True)):
        assert ((got.double() - want).abs() <= 2.0 ** -24 * (state + 64 + 200) * size).all()


@pytest.mark.parametrize("taps", [2, 3, 4])
@pytest.mark.parametrize("lens", [[1300], [1, 700, 2, 3, 597, 1], [1029, 250], [2400], [1, 1400, 2, 3, 1033, 1]])
def test_convolution_of_many_tokens(taps, lens):
    """From 2^23 inputs times taps on a thread has four tokens: portions that begin and end within the four, and are shorter than they, have the bits that
    every portion has alone, the carried rows in front of it and behind it too."""
    import ctypes
    import torch
    from mini_llm_amd import build
    f = build.load_library("ssm").mllm_conv_silu
    C, T, B, dev, g = 1792, sum(lens), len(lens), "cuda:0", torch.Generator().manual_seed(taps)
    x, w, bias = torch.randn(T, C + 8, generator=g).to(dev), torch.randn(C, taps, generator=g).to(dev), torch.randn(C, generator=g).to(dev)
    state = torch.randn(B + 1, (taps - 1) * C + 4, generator=g).to(dev)
    cu = [sum(lens[:i]) for i in range(B + 1)]

    def run(rows, slots, seqs, state, out):
        arrays = [torch.tensor(a, dtype=torch.int32, device=dev) for a in (seqs, [0] + [sum(1 for s in seqs if s <= b) for b in range(max(seqs) + 1)], slots)]
        rc = f(*(ctypes.c_void_p(a.data_ptr()) if torch.is_tensor(a) else ctypes.c_int(a) for a in (rows, rows.stride(0), 8, C, w, bias, taps, *arrays, state)),
               ctypes.c_size_t(state.stride(0)), ctypes.c_void_p(out.data_ptr()), *(ctypes.c_int(a) for a in (C, len(seqs), len(slots), 1)),
               ctypes.c_void_p(torch.cuda.current_stream().cuda_stream))
        assert rc == 0
        torch.cuda.synchronize()

    together, alone, s1, s2 = torch.zeros(T, C, device=dev), torch.zeros(T, C, device=dev), state.clone(), state.clone()
    run(x, list(range(1, B + 1)), [b for b, n in enumerate(lens) for _ in range(n)], s1, together)
    for b in range(B):
        for t in range(cu[b], cu[b + 1], 1024):          # (cut, so that each call is below the line)
            n = min(1024, cu[b + 1] - t)
            run(x[t:t + n], [b + 1], [0] * n, s2, alone[t:t + n])
    assert torch.equal(together, alone) and torch.equal(s1, s2)
    first = torch.cat([s.reshape(taps - 1, C) for s in state[1:2, :(taps - 1) * C]] + [x[:lens[0], 8:]]).double()
    y = sum(first[j:j + lens[0]] * w[:, j].double() for j in range(taps)) + bias.double()
    assert (together[:lens[0]].double() - y * torch.sigmoid(y)).abs().max() <= 1e-5
