"""GPU parity of the multi-token grouped-expert step through the C ABI.

Config 2: T in {4, 16, 64} tokens (bf16 N(0,1) hidden, normed), routing
biased by the seeded Zipf(1.1) prior; outputs within bf16 tolerance
(rel 1e-2) of the oracle's moe_grouped (moe_infer data movement, per-token
combine of reference_decode.moe), and grouped(T) equal to T batch-1 outputs.
The multi-token semantics have no reference test with T > 1, so they are
pinned by that invariant (see tests/test_oracle.py)."""
from __future__ import annotations

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")

from fleet_moe import ops, synth  # noqa: E402
from fleet_moe.layout import DSV2_LITE  # noqa: E402
from oracle import moe_oracle as orc  # noqa: E402


def say(msg: str) -> None:
    print(f"[gpu] {msg}", flush=True)


def rel_err(got, want) -> float:
    got, want = np.asarray(got, np.float64), np.asarray(want, np.float64)
    return float(np.max(np.abs(got - want)) / max(np.max(np.abs(want)), 1e-30))


@pytest.fixture(scope="module")
def dev(full_layer):
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    blob, lay, pl = full_layer
    say("upload layer")
    layer = ops.DeviceLayer.from_host(blob, lay, 1, DSV2_LITE, device="cuda")
    pl.widen()
    return layer, pl


@pytest.mark.parametrize("T", [1, 4, 16, 64])
def test_grouped_matches_oracle(dev, T):
    layer, pl = dev
    runner = ops.GroupedRunner(64, DSV2_LITE)
    bias = synth.zipf_logit_bias(0)
    xn = orc.rms_norm(synth.hidden_inputs(10 + T, T))
    _, ids, ws = orc.route(pl.router_f32(), xn, logit_bias=bias)
    say(f"grouped T={T} distinct={len(np.unique(ids))}")
    out = runner.run(layer, torch.from_numpy(orc.bf16_bits(xn).view(np.int16)).cuda(),
                     torch.from_numpy(ids).cuda(), torch.from_numpy(ws).cuda())
    torch.cuda.synchronize()
    got = ops.bf16_bits_to_f32(out).cpu().numpy()
    want = orc.moe_grouped(pl, xn, ids, ws)["out"]
    assert rel_err(got, want) <= 1e-2
    # MFMA and NumPy sum in different orders; most elements still agree exactly
    assert np.mean(got == want) > 0.95
    assert runner.status() == 0


@pytest.mark.parametrize("T", [8, 9, 256])
def test_grouped_edges_uniform_routing(dev, T):
    """Unbiased routing at the edges of the launch plans: T = 8 (the largest
    single-launch step), T = 9 (the smallest two-launch step, the first with
    MFMA-eligible units) and T = 256 (the largest step: every expert an MFMA
    unit, the shared expert four 64-token passes)."""
    layer, pl = dev
    runner = ops.GroupedRunner(T, DSV2_LITE)
    xn = orc.rms_norm(synth.hidden_inputs(50 + T, T))
    _, ids, ws = orc.route(pl.router_f32(), xn)
    say(f"grouped edge T={T} distinct={len(np.unique(ids))}")
    out = runner.run(layer, torch.from_numpy(orc.bf16_bits(xn).view(np.int16)).cuda(),
                     torch.from_numpy(ids).cuda(), torch.from_numpy(ws).cuda())
    torch.cuda.synchronize()
    got = ops.bf16_bits_to_f32(out).cpu().numpy()
    want = orc.moe_grouped(pl, xn, ids, ws)["out"]
    assert rel_err(got, want) <= 1e-2
    assert np.mean(got == want) > 0.95
    assert runner.status() == 0


def test_grouped_equals_batch1_decode(dev):
    """grouped(T) == T batch-1 MoE outputs (decode kernel's moe_out)."""
    layer, pl = dev
    T = 8
    x = synth.hidden_inputs(21, T)
    xn = orc.rms_norm(x)
    dec = ops.LayerDecoder(DSV2_LITE)
    runner = ops.GroupedRunner(T, DSV2_LITE)
    outs, idl, wl = [], [], []
    say("batch-1 decode x8")
    for t in range(T):
        r = dec.decode(layer, torch.from_numpy(x[t]).cuda())
        outs.append(ops.bf16_bits_to_f32(r["moe_out"]))
        idl.append(r["ids"])
        wl.append(r["weights"])
    ids = torch.stack(idl)
    ws = torch.stack(wl)
    say("grouped T=8 with the decode routing")
    g = runner.run(layer, torch.from_numpy(orc.bf16_bits(xn).view(np.int16)).cuda(), ids, ws)
    torch.cuda.synchronize()
    got = ops.bf16_bits_to_f32(g).cpu().numpy()
    want = torch.stack(outs).cpu().numpy()
    assert rel_err(got, want) <= 1e-2
    assert np.mean(got == want) > 0.95


def test_grouped_hot_expert_over_64_tokens(dev):
    """Every token routed to the same 6 experts, T = 96 > one 64-token group."""
    layer, pl = dev
    T = 96
    runner = ops.GroupedRunner(T, DSV2_LITE)
    xn = orc.rms_norm(synth.hidden_inputs(30, T))
    ids = np.tile(np.array([5, 17, 3, 60, 0, 41], np.int32), (T, 1))
    ws = np.full((T, 6), 0.125, np.float32)
    say("grouped T=96 hot experts")
    out = runner.run(layer, torch.from_numpy(orc.bf16_bits(xn).view(np.int16)).cuda(),
                     torch.from_numpy(ids).cuda(), torch.from_numpy(ws).cuda())
    torch.cuda.synchronize()
    got = ops.bf16_bits_to_f32(out).cpu().numpy()
    want = orc.moe_grouped(pl, xn, ids, ws)["out"]
    assert rel_err(got, want) <= 1e-2


def test_grouped_workspace_reuse_across_token_counts(dev):
    """One workspace, calls of T = 64, 4, 16, 1, 64 in a row: words left by a
    larger earlier call are never taken for the current call's (each call's
    words carry its own call count), so every result matches the oracle."""
    layer, pl = dev
    runner = ops.GroupedRunner(64, DSV2_LITE)
    bias = synth.zipf_logit_bias(1)
    for n, T in enumerate((64, 4, 16, 1, 64)):
        xn = orc.rms_norm(synth.hidden_inputs(70 + n, T))
        _, ids, ws = orc.route(pl.router_f32(), xn, logit_bias=bias)
        say(f"grouped reuse call {n} T={T}")
        out = runner.run(layer, torch.from_numpy(orc.bf16_bits(xn).view(np.int16)).cuda(),
                         torch.from_numpy(ids).cuda(), torch.from_numpy(ws).cuda())
        torch.cuda.synchronize()
        got = ops.bf16_bits_to_f32(out).cpu().numpy()
        want = orc.moe_grouped(pl, xn, ids, ws)["out"]
        assert rel_err(got, want) <= 1e-2, f"call {n} T={T}"
    assert runner.status() == 0


def test_grouped_out_of_range_ids_raise_the_status_bit(dev):
    """An id outside [0, 64) is clamped (the addresses stay in bounds) and
    reported through FLEET_MOE_ABORT_BAD_ID; a valid call reports nothing."""
    layer, pl = dev
    from fleet_moe import _lib
    T = 4
    xn = orc.rms_norm(synth.hidden_inputs(90, T))
    _, ids, ws = orc.route(pl.router_f32(), xn)
    x = torch.from_numpy(orc.bf16_bits(xn).view(np.int16)).cuda()
    runner = ops.GroupedRunner(T, DSV2_LITE)
    say("grouped valid ids")
    runner.run(layer, x, torch.from_numpy(ids).cuda(), torch.from_numpy(ws).cuda())
    torch.cuda.synchronize()
    assert runner.status() == 0
    bad = ids.copy()
    bad[2, 3] = 64
    bad[0, 0] = -1
    say("grouped ids out of range")
    runner.run(layer, x, torch.from_numpy(bad).cuda(), torch.from_numpy(ws).cuda())
    torch.cuda.synchronize()
    assert runner.status() == _lib.ABORT_BAD_ID


def test_grouped_call_count_wrap_restarts_a_clean_workspace(dev):
    """Workspace words carry a 32-bit call count. The header is seeded from the
    host as if 2^32 - 3 calls had run; the call numbered 2^32 - 1 clears the
    tagged words and restarts the count at 0, so the calls on either side of
    the wrap give the same outputs as a fresh workspace, bit for bit."""
    layer, pl = dev
    T_max = 64
    runner = ops.GroupedRunner(T_max, DSV2_LITE)
    fresh = ops.GroupedRunner(T_max, DSV2_LITE)
    start = 0xFFFFFFFD          # header words: call count, exit count (256 per call)
    head0 = np.array([start, (start * 256) & 0xFFFFFFFF], np.uint32)
    runner.workspace[:8].copy_(torch.from_numpy(head0.view(np.uint8)).cuda())
    bias = synth.zipf_logit_bias(3)
    for n, T in enumerate((16, 4, 64, 9, 4)):
        xn = orc.rms_norm(synth.hidden_inputs(110 + n, T))
        _, ids, ws = orc.route(pl.router_f32(), xn, logit_bias=bias)
        x = torch.from_numpy(orc.bf16_bits(xn).view(np.int16)).cuda()
        idt, wst = torch.from_numpy(ids).cuda(), torch.from_numpy(ws).cuda()
        say(f"grouped wrap call {n} (count {(start + 1 + n) & 0xFFFFFFFF:#x}) T={T}")
        got = runner.run(layer, x, idt, wst)
        want = fresh.run(layer, x, idt, wst)
        torch.cuda.synchronize()
        assert torch.equal(got, want), f"call {n} T={T}"
        head = runner.workspace[:8].cpu().numpy().view(np.uint32).tolist()
        if n == 0:
            assert head == [start + 1, ((start + 1) * 256) & 0xFFFFFFFF]
        else:           # the call numbered 2^32 - 1 (n = 1) restarted the count at 0
            assert head == [n - 1, 256 * (n - 1)]
    assert runner.status() == 0


def test_grouped_call_count_wrap_beside_tiles(dev):
    """The same on a workspace for 256 tokens, tile steps (which take no number)
    between the calls: the tagged words alone are cleared, and all of them."""
    layer, pl = dev
    runner = ops.GroupedRunner(256, DSV2_LITE)
    start = 0xFFFFFFFD
    head0 = np.array([start, (start * 256) & 0xFFFFFFFF], np.uint32)
    runner.workspace[:8].copy_(torch.from_numpy(head0.view(np.uint8)).cuda())
    for n, T in enumerate((64, 256, 64, 8, 65, 64)):
        xn = orc.rms_norm(synth.hidden_inputs(130 + n, T))
        _, ids, ws = orc.route(pl.router_f32(), xn)
        a = (torch.from_numpy(orc.bf16_bits(xn).view(np.int16)).cuda(),
             torch.from_numpy(ids).cuda(), torch.from_numpy(ws).cuda())
        say(f"grouped wrap beside tiles, call {n} T={T}")
        got = runner.run(layer, *a)
        assert torch.equal(got, ops.GroupedRunner(T, DSV2_LITE).run(layer, *a)), f"call {n} T={T}"
    assert runner.workspace[:8].cpu().numpy().view(np.uint32).tolist() == [2, 512]
    assert runner.status() == 0


@pytest.mark.parametrize("T, routing", [(64, "zipf"), (65, "uniform"), (65, "hot"),
                                        (83, "uniform"), (84, "uniform"), (84, "zipf"),
                                        (97, "hot"), (129, "zipf"), (193, "uniform"),
                                        (255, "hot"), (256, "zipf"), (256, "one")])
def test_grouped_tiles(dev, T, routing):
    """The tiled plan from its first token count (65) to the largest, at block
    edges (m = 1 mod 16, 64 + 1, 256): uniform and Zipf routing, the same six
    experts for all (blocks of 64 of one expert), and one expert six times
    per token (24 blocks). bf16 tolerance, as for the other plans. (The oracle
    counts a token once per expert, so it has no value for "one": that is
    compared with the same tokens in steps of 64, the other plan.)"""
    layer, pl = dev
    runner = ops.GroupedRunner(T, DSV2_LITE)
    xn = orc.rms_norm(synth.hidden_inputs(150 + T, T))
    bias = synth.zipf_logit_bias(2) if routing == "zipf" else None
    _, ids, ws = orc.route(pl.router_f32(), xn, logit_bias=bias)
    if routing in ("hot", "one"):
        ids = np.tile(np.array([5, 17, 3, 63, 0, 41] if routing == "hot" else [9] * 6, np.int32),
                      (T, 1))
    say(f"grouped tiles T={T} {routing}")
    a = (torch.from_numpy(orc.bf16_bits(xn).view(np.int16)).cuda(),
         torch.from_numpy(ids).cuda(), torch.from_numpy(ws).cuda())
    out = runner.run(layer, *a)
    torch.cuda.synchronize()
    got = ops.bf16_bits_to_f32(out).cpu().numpy()
    if routing == "one":
        parts = [runner.run(layer, *(v[k: k + 64].contiguous() for v in a)) for k in range(0, T, 64)]
        want = ops.bf16_bits_to_f32(torch.cat(parts)).cpu().numpy()
    else:
        want = orc.moe_grouped(pl, xn, ids, ws)["out"]
    assert rel_err(got, want) <= 1e-2
    assert np.mean(got == want) > 0.95
    assert runner.status() == 0


def routing_of(T: int, kind: str) -> np.ndarray:
    """ids [T][6]: "windows": every expert's tokens lie in one window of 64, from
    one token to the whole window per expert; "hot": six experts for all; "one":
    one expert, six times; "skewed": experts of 1 to T tokens anywhere."""
    g = np.random.default_rng(T)
    if kind == "hot":
        return np.tile(np.array([5, 17, 3, 63, 0, 41], np.int32), (T, 1))
    if kind == "one":
        return np.full((T, 6), 9, np.int32)
    if kind == "skewed":
        p = np.arange(1, 65) ** -1.5
        return np.stack([g.choice(64, 6, replace=False, p=p / p.sum()) for _ in range(T)]
                        ).astype(np.int32)
    ids = np.empty((T, 6), np.int32)
    for n, w in enumerate(range(0, T, 64)):
        p = np.arange(1, 17) ** -1.5
        for t in range(w, min(w + 64, T)):
            ids[t] = 4 * g.choice(16, 6, replace=False, p=p / p.sum()) + n
    return ids


def device_step(T: int, ids: np.ndarray):
    x = torch.from_numpy(orc.bf16_bits(orc.rms_norm(synth.hidden_inputs(400 + T, T))).view(np.int16))
    ws = torch.rand((T, 6), generator=torch.Generator().manual_seed(T))
    return x.cuda(), torch.from_numpy(ids).cuda(), ws.cuda()


@pytest.mark.parametrize("T, kind", [(73, "windows"), (128, "windows"), (201, "windows"),
                                     (256, "windows"), (137, "hot"), (256, "hot"), (256, "one")])
def test_grouped_tiles_are_the_other_plans_bits(dev, T, kind):
    """Where every unit holds at most 8 tokens in steps of 64 exactly when it does
    in the whole step, the tiles give the bits of those steps (the other plan):
    the same sums in the same order, in units of 1 to 256 tokens."""
    layer, pl = dev
    runner = ops.GroupedRunner(T, DSV2_LITE)
    ids = routing_of(T, kind)
    counts = np.bincount(ids.ravel(), minlength=64)
    say(f"tiles against steps T={T} {kind} counts {sorted(set(counts.tolist()))}")
    a = device_step(T, ids)
    got = runner.run(layer, *a)
    parts = [runner.run(layer, *(v[k: k + 64].contiguous() for v in a)) for k in range(0, T, 64)]
    torch.cuda.synchronize()
    assert torch.equal(got, torch.cat(parts))
    assert runner.status() == 0


@pytest.mark.parametrize("T, kind", [(66, "skewed"), (97, "hot"), (150, "hot"), (192, "skewed"),
                                     (200, "hot"), (256, "skewed"), (256, "one")])
def test_grouped_tiles_do_not_depend_on_the_order(dev, T, kind):
    """The same call gives the same bits every time, and a token's result does not
    depend on its place in the batch: experts that fill several token blocks,
    whose tokens fall into them in no fixed order."""
    layer, pl = dev
    runner = ops.GroupedRunner(T, DSV2_LITE)
    x, ids, ws = device_step(T, routing_of(T, kind))
    want = runner.run(layer, x, ids, ws)
    g = torch.Generator().manual_seed(T)
    for n in range(4):
        say(f"order T={T} {kind} {n}")
        assert torch.equal(runner.run(layer, x, ids, ws), want), n
        p = torch.randperm(T, generator=g).cuda()
        got = runner.run(layer, x[p].contiguous(), ids[p].contiguous(), ws[p].contiguous())
        assert torch.equal(got, want[p]), n
    assert runner.status() == 0


def test_grouped_plans_share_a_workspace(dev):
    """Tiled and tagged-word steps in turn on one workspace, a tile step with
    ids out of range, and both under graph capture: every result equals that
    of a workspace of its own."""
    layer, pl = dev
    from fleet_moe import _lib
    runner = ops.GroupedRunner(256, DSV2_LITE)
    calls = []
    for n, T in enumerate((256, 4, 84, 64, 8, 100, 16)):
        xn = orc.rms_norm(synth.hidden_inputs(210 + n, T))
        _, ids, ws = orc.route(pl.router_f32(), xn)
        a = (torch.from_numpy(orc.bf16_bits(xn).view(np.int16)).cuda(),
             torch.from_numpy(ids).cuda(), torch.from_numpy(ws).cuda())
        calls.append((a, ops.GroupedRunner(256, DSV2_LITE).run(layer, *a)))
    for n, (a, want) in enumerate(calls):
        say(f"shared workspace call {n}")
        assert torch.equal(runner.run(layer, *a), want), n
    outs = [torch.empty_like(w) for _, w in calls]
    s = torch.cuda.Stream()
    s.wait_stream(torch.cuda.current_stream())
    graph = torch.cuda.CUDAGraph()
    say("capture")
    with torch.cuda.stream(s), torch.cuda.graph(graph, stream=s):
        for (a, _), o in zip(calls, outs):
            runner.run_into(layer, *a, o)
    torch.cuda.current_stream().wait_stream(s)
    for _ in range(3):
        for o in outs:
            o.zero_()
        graph.replay()
        runner.run(layer, *calls[1][0])
        torch.cuda.synchronize()
        for (_, want), o in zip(calls, outs):
            assert torch.equal(o, want)
    assert runner.status() == 0
    (x, ids, ws), _ = calls[2]
    bad = ids.clone()
    bad[70, 2], bad[3, 0] = 64, -5
    say("tile step with ids out of range")
    runner.run(layer, x, bad, ws)
    torch.cuda.synchronize()
    assert runner.status() == _lib.ABORT_BAD_ID


@pytest.mark.parametrize("T", [1, 5, 84])
def test_moe_equals_its_parts(dev, T):
    """ops.moe (router, bf16 rounding in the router's launch, grouped step)
    equals route + f32_to_bf16_bits + run bit for bit; the rounding also on
    ties, signs, subnormals and non-finite values."""
    layer, pl = dev
    runner = ops.GroupedRunner(T, DSV2_LITE)
    x = torch.from_numpy(orc.rms_norm(synth.hidden_inputs(300 + T, T))).cuda()
    logits, ids, ws = ops.route(layer, x)
    want = runner.run(layer, ops.f32_to_bf16_bits(x), ids, ws)
    r = ops.moe(layer, x, runner)
    torch.cuda.synchronize()
    for a, b in ((r["logits"], logits), (r["ids"], ids), (r["weights"], ws), (r["out"], want)):
        assert torch.equal(a, b)
    g = torch.Generator(device="cuda").manual_seed(T)
    odd = torch.randint(-2**31, 2**31 - 1, (T, 2048), generator=g, device="cuda",
                        dtype=torch.int64).to(torch.int32).view(torch.float32)
    bits = torch.empty((T, 2048), dtype=torch.int16, device="cuda")
    say("bf16 bits of arbitrary fp32 patterns")
    ops._route(layer, odd, None, bits, None)
    torch.cuda.synchronize()
    assert torch.equal(bits, ops.f32_to_bf16_bits(odd))


@pytest.mark.parametrize("T", [1023, 1024, 2501])
def test_route_of_many_tokens(dev, T):
    """Both router kernels (four waves to a token from 1,024 tokens on) give the
    same logits, picks, weights and bf16 rows, and the oracle's."""
    layer, pl = dev
    xn = orc.rms_norm(synth.hidden_inputs(500 + T, T))
    x = torch.from_numpy(xn).cuda()
    bias = torch.from_numpy(synth.zipf_logit_bias(5)).cuda()
    bits = torch.empty((T, 2048), dtype=torch.int16, device="cuda")
    say(f"route T={T}")
    got = ops._route(layer, x, bias, bits, None)
    parts = [ops.route(layer, x[k: k + 500].contiguous(), bias) for k in range(0, T, 500)]
    torch.cuda.synchronize()
    for a, b in zip(got, (torch.cat(v) for v in zip(*parts))):
        assert torch.equal(a, b)
    assert torch.equal(bits, ops.f32_to_bf16_bits(x))
    logits, ids, ws = orc.route(pl.router_f32(), xn[-40:], logit_bias=synth.zipf_logit_bias(5))
    assert np.array_equal(got[0][-40:].cpu().numpy(), logits)
    assert np.array_equal(got[1][-40:].cpu().numpy(), ids)
    assert np.array_equal(got[2][-40:].cpu().numpy(), ws)


def test_moe_on_another_stream_keeps_its_rows(dev):
    """ops.moe with a stream: the bf16 rows it makes are its own until that
    stream has read them, whatever the current stream allocates meanwhile."""
    layer, pl = dev
    runner = ops.GroupedRunner(4, DSV2_LITE)
    x = torch.from_numpy(orc.rms_norm(synth.hidden_inputs(330, 4))).cuda()
    want = ops.moe(layer, x, runner)["out"].clone()
    s = torch.cuda.Stream()
    torch.cuda.synchronize()
    with torch.cuda.stream(s):
        torch.cuda._sleep(200_000_000)            # about 0.1 s
    say("moe behind a sleeping stream")
    r = ops.moe(layer, x, runner, stream=s)
    mine = [torch.full((4, 2048), 77, dtype=torch.int16, device="cuda") for _ in range(8)]
    torch.cuda.synchronize()
    assert torch.equal(r["out"], want)
    assert all(bool((m == 77).all()) for m in mine)
