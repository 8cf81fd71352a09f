"""GPU: a prompt taken through the layers together (fleet_prefill) leaves what
teacher-forced decode steps leave: every cache row, the last token's residual,
the pick and the position, compared bit for bit. The steps themselves are
checked against the oracle in test_gpu_decode_model.py and test_gpu_step.py. (The
attention's fp64 sums alone are taken in another order than the steps', a
difference of some 1e-8 of the fp32 unit they are rounded to; with the fixed
tokens and weights here it reaches no bit.) Lengths around the 16-token tiles, the
changes of shape (65, 137, 257) and the 528-token chunk."""
from __future__ import annotations

import pytest

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")

from fleet_moe import layout as lay_mod, ops, synth_gpu  # noqa: E402
from fleet_moe.layout import DSV2_LITE  # noqa: E402

MAX_POS = 600


def say(msg: str) -> None:
    print(f"[gpu] {msg}", flush=True)


@pytest.fixture(scope="module")
def pair():
    """(batched, stepping) decoders on one 3-layer model (dense, MoE, MoE)
    with norms that are not 1."""
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    lay = lay_mod.model_layout(DSV2_LITE, n_layers=3)
    blob = torch.empty(lay.nbytes, dtype=torch.uint8, device="cuda")
    say("fill model")
    synth_gpu.fill_model(blob, lay, seed=3)
    g = torch.Generator(device="cuda").manual_seed(4)
    for name, t in lay.tensors.items():
        if "norm" in name:
            v = blob.view(torch.bfloat16)[t.offset // 2: (t.offset + t.nbytes) // 2]
            v.copy_(1.0 + 0.1 * torch.randn(v.shape, generator=g, device="cuda"))
    return (ops.Decoder(blob, lay, DSV2_LITE, max_pos=MAX_POS),
            ops.Decoder(blob, lay, DSV2_LITE, max_pos=MAX_POS, fused=False))


def state(dec):
    return {"x": dec.x.clone(), "token": dec.token.clone(), "token_out": dec.token_out.clone(),
            "pos": dec.pos.clone(), "cache": dec.cache.clone()}


def check(pair, tokens):
    got, want = pair
    for d in pair:
        d.cache.zero_()
    say(f"n={tokens.numel()} batched")
    got.prefill(tokens)
    torch.cuda.synchronize()
    say("steps")
    want.prefill(tokens)
    torch.cuda.synchronize()
    a, b = state(got), state(want)
    for k in b:
        d = (a[k] != b[k]).double().mean().item()
        assert d == 0.0, f"{k}: {d:.2e} of the values differ"


@pytest.mark.parametrize("n", [1, 3, 4, 5, 16, 17, 33, 64, 65, 128, 129, 136, 137, 176, 177, 257,
                               401, 528, 530])
def test_prefill_equals_steps(pair, n):
    g = torch.Generator(device="cuda").manual_seed(n)
    tokens = torch.randint(0, lay_mod.VOCAB, (n,), generator=g, device="cuda", dtype=torch.int32)
    check(pair, tokens)
    assert pair[0].status() == 0 and pair[1].status() == 0


def test_long_prompt(pair):
    """Three chunks, and attention over more than a thousand cache rows."""
    got, want = (ops.Decoder(d.blob, d.layout, DSV2_LITE, max_pos=1120, fused=d.fused) for d in pair)
    g = torch.Generator(device="cuda").manual_seed(11)
    tokens = torch.randint(0, lay_mod.VOCAB, (1100,), generator=g, device="cuda", dtype=torch.int32)
    check((got, want), tokens)
    assert got.status() == 0 and want.status() == 0


@pytest.mark.parametrize("parts", [(37, 60), (1, 2, 130), (530, 5, 40)])
def test_prompt_in_parts(pair, parts):
    """fleet_prefill from a position other than 0 continues the rows that are
    there: a prompt given in parts leaves what it leaves in one piece."""
    import ctypes

    from fleet_moe import _lib
    got, want = pair
    g = torch.Generator(device="cuda").manual_seed(sum(parts))
    tokens = torch.randint(0, lay_mod.VOCAB, (sum(parts),), generator=g, device="cuda",
                           dtype=torch.int32)
    for d in pair:
        d.cache.zero_()
    status = torch.zeros(1, dtype=torch.int32, device="cuda")
    lib, at = _lib.load(), 0
    for n in parts:
        say(f"part {n} at {at}")
        rc = lib.fleet_prefill(ctypes.byref(got.step_model), got.step_rows,
                               tokens[at:].data_ptr(), n, at, got.x.data_ptr(), status.data_ptr(),
                               got.prefill_ws.data_ptr(), got.prefill_ws.numel(),
                               ctypes.byref(got.attn._dims),
                               torch.cuda.current_stream().cuda_stream)
        _lib.check(rc, "fleet_prefill")
        at += n
    torch.cuda.synchronize()
    say("steps")
    want.prefill(tokens)
    torch.cuda.synchronize()
    assert torch.equal(got.cache, want.cache) and torch.equal(got.x, want.x)
    assert int(status.item()) == 0


def test_wide_exponents_and_zero_rows(pair):
    """Weights whose magnitudes span 2^40 within a row, zero rows, rows far
    below 2^-87 and norms of 0: where a dot product cannot be certified from
    its leading digits, the fp64 path decides, and the bits stay the steps'."""
    got, want = pair
    blob, lay = got.blob, got.layout
    kept = blob.clone()
    g = torch.Generator(device="cuda").manual_seed(9)
    words = blob.view(torch.bfloat16)
    for name, t in lay.tensors.items():
        v = words[t.offset // 2: (t.offset + t.nbytes) // 2]
        if name.endswith(("qkv", "o_proj", "dense", "shared", "experts")):
            for part in v.split(1 << 26):
                e = torch.randint(-34, 7, part.shape, generator=g, device="cuda")
                part.mul_(torch.exp2(e.float()).bfloat16())
            rows = v[: v.numel() // 2048 * 2048].view(-1, 2048)
            rows[3::40] = 0
            rows[5::40] *= 1e-35
        elif name.endswith("norm_post"):
            v[::7] = 0
    try:
        n = 40
        tokens = torch.randint(0, lay_mod.VOCAB, (n,), generator=g, device="cuda",
                               dtype=torch.int32)
        check(pair, tokens)
        assert bool(torch.isfinite(got.x).all())
    finally:
        blob.copy_(kept)


def test_one_token_repeated(pair):
    """Every token the same: one token block per expert, all rows alike."""
    check(pair, torch.full((70,), 17, dtype=torch.int32, device="cuda"))


def test_then_generate_and_capture(pair):
    """The state left behind drives the decode steps; a captured prompt
    replays (no allocation, no fill outside the stream)."""
    got, want = pair
    tokens = torch.arange(100, 140, dtype=torch.int32, device="cuda")
    check(pair, tokens)
    assert torch.equal(got.generate(3), want.generate(3))
    s = torch.cuda.Stream()
    s.wait_stream(torch.cuda.current_stream())
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.stream(s), torch.cuda.graph(graph, stream=s):
        got.prefill(tokens)
    torch.cuda.current_stream().wait_stream(s)
    want.cache.zero_()
    want.prefill(tokens)
    for _ in range(3):
        got.cache.zero_()
        graph.replay()
        torch.cuda.synchronize()
        for k, v in state(want).items():
            assert torch.equal(state(got)[k], v), k


def test_tokens_of_other_kinds(pair):
    """Host tensors, other integer types and strided views are accepted, a
    token outside the vocabulary raises the status bit, and a prompt longer
    than the cache fills it and raises the position bit, as steps do."""
    got, want = pair
    tokens = torch.arange(7, 47, dtype=torch.int32, device="cuda")
    check(pair, tokens.cpu().long())
    check(pair, tokens[::3])
    fresh = ops.Decoder(got.blob, got.layout, DSV2_LITE, max_pos=MAX_POS)
    bad = tokens.clone()
    bad[5] = lay_mod.VOCAB
    fresh.prefill(bad)
    torch.cuda.synchronize()
    assert fresh.status() == 0x10
    long = ops.Decoder(got.blob, got.layout, DSV2_LITE, max_pos=32)
    long.prefill(tokens)
    torch.cuda.synchronize()
    assert long.status() == 0x8 and int(long.pos.item()) == 32
    want.cache.zero_()
    want.prefill(tokens[:32])
    assert torch.equal(long.cache, want.cache[:, :32])
