"""A long chunk whose tiles are dequantized once into the workspace gives bit for
bit what the same launch gives when its workgroups dequantize them (the path
the oracle's tests pin), and takes that path when the memory is refused."""

import pytest
import torch

import rec_amd
from rec_amd import _lib, attention

pytestmark = pytest.mark.gpu

FORMATS = {"int8": (32, 8, 8), "uint4": (32, 4, 4), "k8v4": (32, 8, 4), "k4v8": (32, 4, 8), "affine": (64, 8, 4)}


class WithoutImages:
    """The library, asking for the partials' workspace only."""

    def __init__(self, lib):
        self.lib = lib

    def __getattr__(self, name):
        return getattr(self.lib, name)

    def rec_prefill_quantized_workspace_bytes(self, B, Hq, Hkv, L, T, splits):
        return self.lib.rec_prefill_workspace_bytes(B, Hq, Hkv, L, splits)


CASES = [
    # fmt, dtype, B, Hq, Hkv, held, new, mask
    ("int8", "bf16", 1, 8, 1, 3712, 384, "causal"),      # the fewest rows and keys of the rule, whole tiles
    ("int8", "fp16", 1, 8, 1, 0, 4097, "causal"),        # no prefix, a last tile of one token
    ("uint4", "bf16", 2, 16, 2, 4000, 600, "causal"),
    ("uint4", "fp16", 1, 8, 1, 9000, 520, "causal"),     # one fp16 part of P'
    ("k8v4", "bf16", 1, 16, 2, 8300, 531, "causal"),
    ("k4v8", "fp16", 1, 8, 1, 3500, 700, None),
    ("affine", "bf16", 1, 32, 4, 4097, 1000, "causal"),  # key splits and partials
    ("affine", "fp16", 1, 8, 2, 5000, 1100, "causal"),   # groups of 4 heads
    ("affine", "bf16", 1, 32, 4, 9000, 2048, "causal"),  # a full grid: blocks placed by XCD
]


@pytest.mark.parametrize("case", CASES, ids=lambda c: f"{c[0]}_{c[1]}_{c[5]}_{c[6]}")
def test_image_equals_in_kernel_dequantization(gpu, monkeypatch, case):
    fmt, dtype, B, Hq, Hkv, held, new, mask = case
    dt = torch.bfloat16 if dtype == "bf16" else torch.float16
    g = torch.Generator(device="cuda").manual_seed(held + new)
    cache = rec_amd.QuantizedKVCache(*FORMATS[fmt], max_tokens=held + new)
    k, v = (torch.randn((B, Hkv, held + new, 128), generator=g, device="cuda").to(dt) for _ in range(2))
    keys, values = cache.update_and_fetch(k, v)
    q = torch.randn((B, Hq, new, 128), generator=g, device="cuda").to(dt)
    sinks = torch.randn((Hq,), generator=g, device="cuda")
    lib = _lib.load()
    assert lib.rec_prefill_quantized_workspace_bytes(B, Hq, Hkv, new, held + new, 0) > \
        lib.rec_prefill_workspace_bytes(B, Hq, Hkv, new, 0)

    def run():
        return rec_amd.quantized_attention_with_sinks(q, keys, values, 0.09, mask, sinks, *FORMATS[fmt])

    def refused(*a, **kw):
        raise torch.OutOfMemoryError

    got = run()
    with monkeypatch.context() as m:
        m.setattr(attention._lib, "load", lambda: WithoutImages(lib))
        want = run()
    assert torch.isfinite(want).all() and torch.equal(got.view(torch.int16), want.view(torch.int16))
    attention.prefill_workspace(q.device, B, Hq, Hkv, new, 0, torch.cuda.current_stream().cuda_stream)
    out = torch.empty_like(got)
    with monkeypatch.context() as m:
        m.setattr(attention, "_new_out", lambda *a: (out, dt))
        m.setattr(torch, "empty", refused)
        fallback = run()
    assert torch.equal(fallback.view(torch.int16), want.view(torch.int16))
