"""GPU parity: router GEMM, softmax top-k, grouping and gather against the CPU oracle.

Integer stages (ids, histogram, PfPlan bytes, tile list, src/dst, gathered rows) and the
route weights must be bit-exact; the F32 router logits are checked against FP64 within
a magnitude-scaled bound, and top-k is then checked bit-exact on the GPU's own logits.
"""
import numpy as np
import pytest

import gpu_util as gu
import ref_patterns as rp

pytestmark = pytest.mark.gpu


def _route_case(moe, orc, ctx, stream, logits, K, divide):
    import torch
    T, E = logits.shape
    shape = moe.Shape(T, 256, E, K, 64, 0)
    L = ctx.register(gu.dev(logits))
    ids = ctx.register(torch.full((T * K,), -7, dtype=torch.int32, device="cuda"))
    w = ctx.register(torch.zeros(T * K, dtype=torch.float32, device="cuda"))
    b = moe.RouteBuffers(L.view(), ids.view(), w.view())
    gu.run(ctx, stream, lambda s: s.encode_moe_route(shape, divide, b))
    return gu.host(ids, np.int32).reshape(T, K), gu.host(w, np.float32).reshape(T, K)


# Two layouts, one token per wave (ranks counted among the candidates, or rounds past K = 20) and
# two tokens per wave (rounds); many tokens take the second where K times the slots is small, or
# K is past 20. Both meet every slot count (E up to 64 / 128 / 256 / 512 per wave, 32 / 64 / 128 /
# 256 / 512 per half-wave) and the reference's golden rows.
@pytest.mark.parametrize("T,E,K", [(64, 16, 4), (4096, 512, 10), (1000, 256, 8), (37, 40, 5), (9, 512, 32),
                                   (8, 512, 10), (300, 100, 6), (1025, 100, 6), (2000, 40, 10), (1500, 200, 10),
                                   (1025, 16, 4), (4096, 256, 10), (5000, 512, 8), (1100, 512, 21), (3072, 64, 16),
                                   (3073, 64, 16)])
@pytest.mark.parametrize("divide", [True, False])
def test_route_topk_bit_exact(moe, orc, gpu_ctx, stream, T, E, K, divide):
    print(f"case route T={T} E={E} K={K} divide={divide}", flush=True)
    rng = np.random.default_rng(1000 * T + E + K)
    logits = (rng.standard_normal((T, E)) * 1.5).astype(np.float32)
    if E >= 20 and T >= 8:
        logits[:4] = rp.special_logits(E)
        logits[4:8] = rp.shuffled_rank_logits(4, E, T)
    if T > 12:  # NaN / inf rows exercise the -FLT_MAX replacement
        logits[9, 3] = np.nan
        logits[10, 1] = np.inf
        logits[11, :] = -np.inf
        logits[12, :] = 0.0
    ids, w = _route_case(moe, orc, gpu_ctx, stream, logits, K, divide)
    ids_ref, w_ref = orc.route(logits, K, divide)
    assert np.array_equal(ids, ids_ref)
    assert np.array_equal(w.view(np.uint32), w_ref.view(np.uint32))
    if E in (256, 512) and K == 10 and T >= 8:  # the expert counts the golden rows hold for
        assert np.array_equal(ids[:4], rp.special_ids(E))
        gold = rp.NONUNIFORM_DIVIDE_BITS if divide else rp.NONUNIFORM_MULTIPLY_BITS
        assert list(w[2].view(np.uint32)) == gold
        assert list(w[0].view(np.uint32)) == rp.EQUAL_WEIGHT_BITS


def _edge_rows(rng, E, K):
    """Rows that put a chosen number of equal values at the top (63, 64 and 65 around the 64
    candidates that are ranked by counting, all of them equal, and ties on both sides of rank K),
    and rows where K - 1 larger values leave one rank to equal ones of the same and of other lanes."""
    rows = []
    for n in sorted({K, K + 1, 63, 64, 65, E - 1, E}):
        if n <= E:
            row = rng.permutation(E).astype(np.float32) * np.float32(-0.01) - np.float32(1.0)
            row[rng.permutation(E)[:n]] = 2.0
            rows.append(row)
    for step in (1, 31, 32, 33):
        row = rng.permutation(E).astype(np.float32) * np.float32(-0.01) - np.float32(1.0)
        tied = (int(rng.integers(E)) + step * np.arange(3)) % E
        top = [e for e in rng.permutation(E) if e not in tied][:K - 1]
        row[top] = 3.0 + np.arange(len(top), dtype=np.float32) * np.float32(0.125)
        row[tied] = 2.0
        rows.append(row)
    return np.stack(rows)


# 1100 rows: two tokens per wave for K = 1 and 4 at every E, 10 at up to 128 experts, 21 and 32 at
# more than 64; one per wave otherwise.
@pytest.mark.parametrize("T", [11, 1100])
@pytest.mark.parametrize("E,K", [(65, 1), (65, 10), (65, 32), (128, 10), (128, 20), (128, 21), (512, 4), (512, 10),
                                 (512, 20), (512, 21), (512, 32), (33, 32), (64, 32)])
def test_route_topk_ties_and_candidate_count(moe, orc, gpu_ctx, stream, T, E, K):
    print(f"case route ties T={T} E={E} K={K}", flush=True)
    rows = _edge_rows(np.random.default_rng(E * 64 + K), E, K)
    logits = rows[np.arange(T) % len(rows)]
    ids, w = _route_case(moe, orc, gpu_ctx, stream, logits, K, True)
    ids_ref, w_ref = orc.route(logits, K, True)
    assert np.array_equal(ids, ids_ref)
    assert np.array_equal(w.view(np.uint32), w_ref.view(np.uint32))


@pytest.mark.parametrize("E", [256, 512])
@pytest.mark.parametrize("T", [1, 7, 25, 26, 64, 300, 4096])
@pytest.mark.parametrize("pattern", rp.PATTERNS)
def test_grouping_gather_bit_exact(moe, orc, gpu_ctx, stream, pattern, T, E):
    _check_grouping_gather(moe, orc, gpu_ctx, stream, pattern, T, E)


# One workgroup groups up to 80 tiles (8 or 40 counts held per thread): 409 tokens x 10 is 16
# tiles, 410 is 17, 2048 is 80 and 2049 is 81.
@pytest.mark.parametrize("E", [40, 512])
@pytest.mark.parametrize("T", [409, 410, 2048, 2049])
@pytest.mark.parametrize("pattern", ["mixed", "invalid_ids"])
def test_grouping_one_workgroup_limits(moe, orc, gpu_ctx, stream, pattern, T, E):
    _check_grouping_gather(moe, orc, gpu_ctx, stream, pattern, T, E)


# With a residency table (experts at or above 0 are resident): the plan's per-group flags, its miss
# count and skip flag, on both sides of 80 tiles.
@pytest.mark.parametrize("T,E", [(26, 64), (410, 512), (2048, 512), (2049, 512), (2049, 40), (4096, 300)])
@pytest.mark.parametrize("cold", ["some", "none", "unused"])
def test_grouping_residency(moe, orc, gpu_ctx, stream, T, E, cold):
    print(f"case grouping residency T={T} E={E} cold={cold}", flush=True)
    K, d = 10, 256
    rng = np.random.default_rng(T + E)
    ids = np.stack([rng.permutation(E - 1)[:K] for _ in range(T)]).astype(np.int32)  # the last expert is never used
    resident = rng.integers(0, 1000, (2, E)).astype(np.int32)
    resident[1, E - 1] = -1 if cold != "none" else 0
    if cold == "some":
        resident[1, ::3] = -1
    resident[0] = -1  # the other layer's table must not be read
    reg, N, shape = gpu_ctx.register, T * K, moe.Shape(T, d, E, K, 64, 0)
    b_ids, b_x, b_res = reg(gu.dev(ids)), reg(gu.dev(np.zeros((T, d), np.uint16))), reg(gu.dev(resident))
    hist, plan = reg(gu.poison(moe.histogram_bytes(shape))), reg(gu.poison(moe.PLAN_SLOT_BYTES))
    tiles, xs = reg(gu.poison(moe.tiles_bytes(shape))), reg(gu.poison(N * d * 2))
    src, dst = reg(gu.poison(N * 4)), reg(gu.poison(N * 4))
    b = moe.GroupingBuffers(b_ids.view(), b_x.view(), hist.view(), plan.view(), tiles.view(), src.view(), dst.view(),
                            xs.view(), b_res.view(), 1)
    gu.run(gpu_ctx, stream, lambda s: s.encode_prefill_moe_grouping(shape, b))
    ref = orc.grouping(ids, E)
    want = ref["plan"].copy()
    w = want[:6180].view(np.int32)
    groups = int(w[0])
    flags = (resident[1][w[8:8 + groups]] >= 0).astype(np.int32)
    w[520:520 + groups] = flags
    w[2] = groups - int(flags.sum())
    w[3] = int(w[2] == 0)
    assert (w[2] > 0) == (cold == "some")
    assert np.array_equal(gu.host(plan, np.uint8), want)
    assert np.array_equal(gu.host(dst, np.int32), ref["dst"]) and np.array_equal(gu.host(src, np.int32), ref["src"])


# The scan keeps up to 16 of its 256-entry tiles per thread in registers (512 tiles: N = 131072
# entries); longer columns take its re-reading loop. 13107 tokens x 10 is 512 tiles, 16384 x 10
# is 640.
@pytest.mark.parametrize("T", [13107, 16384])
@pytest.mark.parametrize("pattern", ["mixed", "invalid_ids"])
def test_grouping_gather_long_columns(moe, orc, gpu_ctx, stream, pattern, T):
    _check_grouping_gather(moe, orc, gpu_ctx, stream, pattern, T, 512)


def _check_grouping_gather(moe, orc, gpu_ctx, stream, pattern, T, E):
    import torch
    print(f"case grouping pattern={pattern} T={T} E={E}", flush=True)
    K, d = 10, 256
    shape = moe.Shape(T, d, E, K, 64, 0)
    N = T * K
    ids = rp.grouping_ids(T, E, pattern, K)
    x = moe.synth_normal_f16(7, T, 1.0, T * d).reshape(T, d)
    ctx = gpu_ctx
    reg = ctx.register
    b_ids, b_x = reg(gu.dev(ids)), reg(gu.dev(x))
    hist = reg(gu.poison(moe.histogram_bytes(shape)))
    plan = reg(gu.poison(moe.PLAN_SLOT_BYTES))
    tiles = reg(gu.poison(moe.tiles_bytes(shape)))
    src, dst = reg(gu.poison(N * 4)), reg(gu.poison(N * 4))
    xs = reg(gu.poison(N * d * 2))
    b = moe.GroupingBuffers(b_ids.view(), b_x.view(), hist.view(), plan.view(), tiles.view(), src.view(),
                            dst.view(), xs.view())
    gu.run(ctx, stream, lambda s: s.encode_prefill_moe_grouping(shape, b))
    ref = orc.grouping(ids, E)
    pf = orc.plan_fields(ref["plan"])
    n_valid = N - pf["bad"]
    n_count = (N + 255) // 256
    assert np.array_equal(gu.host(plan, np.uint8), ref["plan"]), "PfPlan slot bytes"
    assert np.array_equal(gu.host(hist, np.uint32).reshape(-1, E)[:n_count], ref["hist"]), "histogram"
    tl = gu.host(tiles, np.uint32).reshape(-1, 2)
    assert np.array_equal(tl[: ref["n_tiles"]], ref["tiles"]), "tile list"
    g_src, g_dst = gu.host(src, np.int32), gu.host(dst, np.int32)
    assert np.array_equal(g_src[:n_valid], ref["src"][:n_valid]), "source rows"
    assert np.array_equal(g_dst[:n_valid], ref["dst"][:n_valid]), "destination rows"
    poison32 = np.frombuffer(b"\xa5" * 4, np.int32)[0]
    assert (g_src[n_valid:] == poison32).all() and (g_dst[n_valid:] == poison32).all(), "tails written"
    g_xs = gu.host(xs, np.uint16).reshape(N, d)
    assert np.array_equal(g_xs[:n_valid], orc.gather(x, ref["src"], n_valid)), "gathered rows"
    assert (g_xs[n_valid:] == 0xA5A5).all(), "gather tail written"
    torch.cuda.synchronize()


@pytest.mark.parametrize("cfg_index", [0, 1])
def test_route_gather_composition(moe, layer, orc, gpu_ctx, stream, cfg_index):
    """Steps 1-6 as one segment at configuration 0 and 1 (T=4096, E=512, k=10)."""
    print(f"case route_gather config={cfg_index}", flush=True)
    cfg = layer.CONFIGS[cfg_index]
    inp = layer.make_inputs(cfg, with_experts=False)
    ws = layer.LayerWorkspace(gpu_ctx, cfg, inp)
    rg = ws.route_gather_buffers()
    gu.run(gpu_ctx, stream, lambda s: s.encode_prefill_moe_full_mode_route_gather(cfg.shape(), rg))
    T, E, K, d = cfg.rows, cfg.n_experts, cfg.top_k, cfg.hidden
    logits = gu.host(ws.logits, np.float32).reshape(T, E)
    ref64 = orc.router_ref(inp.x[:T], inp.w_router)
    # F32-class bound on the logits: |err| <= 2^-20 * sum_k |x_k w_k| (plus a floor).
    mag = np.abs(inp.x[:T].view(np.float16).astype(np.float64)) @ np.abs(inp.w_router.astype(np.float64)).T
    assert (np.abs(logits - ref64) <= 2.0 ** -20 * mag + 1e-7).all(), "router logits"
    ids = gu.host(ws.ids, np.int32).reshape(T, K)
    w = gu.host(ws.route_w, np.float32).reshape(T, K)
    ids_ref, w_ref = orc.route(logits, K, True)
    assert np.array_equal(ids, ids_ref) and np.array_equal(w.view(np.uint32), w_ref.view(np.uint32))
    # How many tokens would flip between the GPU logits and FP64 logits (reported, not failed).
    ids64, _ = orc.route(ref64.astype(np.float32), K, True)
    flips = int((ids64 != ids).any(axis=1).sum())
    print(f"route_gather config={cfg_index}: tokens whose top-{K} differs under FP64 logits: {flips}/{T}")
    g = orc.grouping(ids_ref, E)
    n_valid = T * K - orc.plan_fields(g["plan"])["bad"]
    # In this composition top-k counts the entries into the histogram (the router clears it)
    # and the count kernel does not run: the per-tile counts must still be the count kernel's.
    n_count = (T * K + 255) // 256
    assert np.array_equal(gu.host(ws.hist, np.uint32).reshape(-1, E)[:n_count], g["hist"]), "histogram"
    assert np.array_equal(gu.host(ws.plan, np.uint8), g["plan"])
    assert np.array_equal(gu.host(ws.src, np.int32)[:n_valid], g["src"][:n_valid])
    assert np.array_equal(gu.host(ws.dst, np.int32)[:n_valid], g["dst"][:n_valid])
    xs = gu.host(ws.xs, np.uint16).reshape(T * K, d)
    assert np.array_equal(xs[:n_valid], orc.gather(inp.x[:T], g["src"], n_valid))


@pytest.mark.parametrize("T,E,d", [(1, 16, 256), (33, 65, 512), (100, 512, 768), (800, 256, 1280), (801, 256, 1280)])
def test_router_few_tiles(moe, layer, orc, gpu_ctx, stream, T, E, d):
    """Router logits with 2 to 10 stage pairs, ragged token and expert tiles, and on both sides of
    the token count up to which stages run in pairs (800)."""
    print(f"case router T={T} E={E} d={d}", flush=True)
    cfg = layer.LayerConfig("router_few", T, d, E, 4, 128, 0, moe.Q8_0, moe.Q8_0, moe.F16, seed=95)
    inp = layer.make_inputs(cfg, with_experts=False)
    ws = layer.LayerWorkspace(gpu_ctx, cfg, inp)
    rg = ws.route_gather_buffers()
    gu.run(gpu_ctx, stream, lambda s: s.encode_prefill_moe_full_mode_route_gather(cfg.shape(), rg))
    logits = gu.host(ws.logits, np.float32).reshape(T, E)
    mag = np.abs(inp.x[:T].view(np.float16).astype(np.float64)) @ np.abs(inp.w_router.astype(np.float64)).T
    assert (np.abs(logits - orc.router_ref(inp.x[:T], inp.w_router)) <= 2.0 ** -20 * mag + 1e-7).all(), "router logits"
