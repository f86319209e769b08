"""Weights are read past the last-level cache where a model's exceed it, and only
there: the model says so to every projection."""

import pytest
import torch

from quickstart_streaming_agents_amd.models import build_model
from quickstart_streaming_agents_amd.models.layers import Linear, projections
from quickstart_streaming_agents_amd.ops import dispatch as D

PRESETS = ["tiny", "tiny-qwen", "tiny-moe", "tiny-lunulix", "tiny-luzalorn"]


@pytest.mark.parametrize("preset", ["tiny-lunulix", "tiny-luzalorn"])
@pytest.mark.parametrize("line,far", [(192 << 20, False), (0, True)])
def test_every_projection_of_a_mixer_decoder(preset, line, far, monkeypatch):
    made = []
    monkeypatch.setattr(D, "FAR_WEIGHTS", line)
    init = Linear.__init__
    monkeypatch.setattr(Linear, "__init__",
                        lambda self, w: made.append(self) or init(self, w))
    model = build_model(preset, device="cpu", dtype=torch.float32)
    assert made and {id(p) for p in made} == {id(p) for p in projections(model)}
    assert all(p.far is far for p in made)


@pytest.mark.parametrize("preset", ["tiny", "tiny-qwen", "tiny-moe"])
@pytest.mark.parametrize("line,far", [(192 << 20, False), (0, True)])
def test_llama_family(preset, line, far, monkeypatch):
    monkeypatch.setattr(D, "FAR_WEIGHTS", line)
    model = build_model(preset, device="cpu", dtype=torch.float32)
    assert model.weights_far is far and model.stored_far is far
    total = sum(model._weight_bytes(False))
    want = model.lm_head.nbytes
    for L in model.layers:
        want += sum(L[k].nbytes for k in ("wqkv", "wo", "wgu", "wdown") if k in L)
        want += sum(a.nbytes + b.nbytes for a, b in L.get("experts", {}).values())
    assert total == want


@pytest.mark.gpu
@pytest.mark.parametrize("rows", [1, 4, 24, 40, 100])
@pytest.mark.parametrize("preset", PRESETS)
@pytest.mark.parametrize("line", [192 << 20, 0])
def test_what_the_kernels_are_told(preset, rows, line, monkeypatch):
    """Every product of a decoding step is given the model's answer."""
    from quickstart_streaming_agents_amd.ops import ext, lm_ext
    monkeypatch.setattr(D, "FAR_WEIGHTS", line)
    model = build_model(preset, device="cuda:0")
    told = []

    class Told:
        def __init__(self, module):
            self.module = module

        def __getattr__(self, name):
            fn = getattr(self.module, name)
            if name not in ("gemm", "gemm_parts", "glu_gemm", "skinny_gemm",
                            "skinny_gemm_fp8", "skinny_gemm_fp8_norm",
                            "skinny_gemm_fp8_residual"):
                return fn

            def call(*a, **kw):
                told.append(kw.get("far", a[-1]))
                return fn(*a, **kw)
            return call

    a, b = Told(ext()), Told(lm_ext())
    monkeypatch.setattr(D, "ext", lambda: a)
    monkeypatch.setattr(D, "lm_ext", lambda: b)
    kv = model.new_kv_cache(rows, rows)
    for i in range(rows):
        kv.allocate(i, 3)
    ids = list(range(rows))
    more = [kv.slots_tensor(ids)] if kv.has_state else []
    sl = kv.seq_lens_tensor(ids)
    model.forward_decode(torch.arange(rows, device="cuda:0"), kv,
                         kv.block_table(ids), sl, sl - 1, *more)
    assert told and all(t is (line == 0) for t in told), told


@pytest.mark.gpu
@pytest.mark.parametrize("M", [1, 17, 33, 100, 192, 193])
def test_the_same_bits(M):
    from quickstart_streaming_agents_amd.ops import lm_ext
    g = torch.Generator().manual_seed(M)
    x = torch.randn(M, 1088, generator=g).bfloat16().to("cuda:0")
    w = torch.randn(4128, 1088, generator=g).bfloat16().to("cuda:0")
    for run in (D.linear, D.linear_parts, D.glu_linear, lm_ext().rows_gemm):
        assert torch.equal(run(x, w, far=True), run(x, w, far=False))
        assert torch.equal(run(x, w), run(x, w, far=False))
    if M <= 32:
        w = w[:4096, :1024].contiguous()
        x, f = x[:, :1024].contiguous(), D.pack_weight_frag(w)
        q, s = D.pack_weight_fp8(w)
        for far in (False, True):
            assert torch.equal(D.skinny_linear(x, f, 4096, 1024),
                               D.skinny_linear(x, f, 4096, 1024, far))
            assert torch.equal(D.skinny_linear_fp8(x, q, s, 4096, 1024),
                               D.skinny_linear_fp8(x, q, s, 4096, 1024, far))
