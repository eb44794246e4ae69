"""The native host path of a decode step and of the projections gives what the
general Python path gives, over the forms it accepts and those it leaves to the
general path (which out_dtype selects), and refuses what that refuses."""

import pytest
import torch

import rec_amd
from rec_amd import Q4Matrix, q4_gemv
from rec_amd.kvstorage import FixedSlidingKVCache

pytestmark = pytest.mark.gpu

B, H, G, T = 2, 2, 4, 70


def view(t, form):
    """The same values behind other strides or alignments."""
    if form == "plain":
        return t
    if form == "wide":  # rows 16-byte aligned, longer strides
        big = torch.zeros((*t.shape[:-1], 160), dtype=t.dtype, device=t.device)
        big[..., :128] = t
        return big[..., :128]
    if form == "token_major":  # (B, L, heads, 128) transposed
        return t.transpose(1, 2).contiguous().transpose(1, 2)
    big = torch.zeros((*t.shape[:-1], 131), dtype=t.dtype, device=t.device)  # "odd": no vector loads
    big[..., 3:] = t
    return big[..., 3:]


def make(kind, kv):
    if kind == "ring":
        c = FixedSlidingKVCache(max_sequence_tokens=1 << 12, num_kv_heads=H, head_dim=128, window_size=33, batch=B)
        kv = torch.bfloat16
    else:
        c = rec_amd.QuantizedKVCache(*{"int8": (32, 8, 8), "uint4": (32, 4, 4), "affine": (64, 8, 4)}[kind], max_tokens=T + 2)
    g = torch.Generator(device="cuda").manual_seed(7)
    k, v = (torch.randn((B, H, T, 128), generator=g, device="cuda").to(kv) for _ in range(2))
    c.update_and_fetch(k, v)
    return c


def state(c):
    ts = c.state if isinstance(c, FixedSlidingKVCache) else (*c.keys, *c.values)
    return [t.contiguous().view(torch.uint8) for t in ts if t is not None]


@pytest.mark.parametrize("kind", ["ring", "int8", "uint4", "affine"])
@pytest.mark.parametrize("q_dtype,kv_dtype", [(torch.bfloat16, torch.bfloat16), (torch.float16, torch.float16),
                                              (torch.float32, torch.float32), (torch.bfloat16, torch.float16)])
@pytest.mark.parametrize("form", ["plain", "wide", "token_major", "odd"])
@pytest.mark.parametrize("sinks", [None, "fp32", "bf16", "strided"])
def test_decode_step(gpu, kind, q_dtype, kv_dtype, form, sinks):
    g = torch.Generator(device="cuda").manual_seed(3)
    q = torch.randn((B, H * G, 1, 128), generator=g, device="cuda").to(q_dtype)
    k, v = (torch.randn((B, H, 1, 128), generator=g, device="cuda").to(kv_dtype) for _ in range(2))
    s = torch.randn((H * G, 2), generator=g, device="cuda")
    s = {None: None, "fp32": s[:, 0].contiguous(), "bf16": s[:, 0].bfloat16(), "strided": s[:, 0]}[sinks]
    q, k, v = (view(t, form) for t in (q, k, v))
    a, b = make(kind, kv_dtype), make(kind, kv_dtype)
    for _ in range(2):  # (the second step has a workspace in any case)
        want = rec_amd.attend(q, k, v, b, 0.09, None, s, out_dtype=q_dtype)
        got = rec_amd.attend(q, k, v, a, 0.09, None, s)
        assert got.shape == want.shape and got.dtype == want.dtype
        assert torch.equal(got.view(torch.uint8), want.view(torch.uint8))
        assert a.offset == b.offset and all(torch.equal(x, y) for x, y in zip(state(a), state(b)))


@pytest.mark.parametrize("kind", ["ring", "int8"])
def test_refusals(gpu, kind):
    """A full cache, other shapes and types raise as before and leave the cache as it was."""
    dt = torch.bfloat16
    q = torch.randn((B, H * G, 1, 128), device="cuda").to(dt)
    k = torch.randn((B, H, 1, 128), device="cuda").to(dt)
    c = make(kind, dt)
    rec_amd.attend(q, k, k, c, 0.09)
    before, off = [t.clone() for t in state(c)], c.offset
    for args in ((q[:1], k, k), (q, k[:1], k[:1]), (q, k, k[:, :1]), (q, k[:, :1], k[:, :1]), (q, k, k.float()),
                 (q.double(), k, k), (q[:, :3], k, k), (q.cpu(), k, k)):
        with pytest.raises((ValueError, NotImplementedError)):
            rec_amd.attend(*args, c, 0.09)
    with pytest.raises(ValueError):
        rec_amd.attend(q, k, k, c, 0.09, None, torch.zeros(H * G - 1, device="cuda"))
    assert c.offset == off and all(torch.equal(x, y) for x, y in zip(state(c), before))
    if kind == "int8":
        rec_amd.attend(q, k, k, c, 0.09)
        with pytest.raises(ValueError, match="context limit"):
            rec_amd.attend(q, k, k, c, 0.09)


@pytest.mark.parametrize("rows", [1, 8, 9])
@pytest.mark.parametrize("out", [torch.bfloat16, torch.float32])
def test_projection_forms(gpu, rows, out):
    g = torch.Generator(device="cuda").manual_seed(rows)
    N, K = 48, 256
    w = torch.randint(-(2**31), 2**31, (N, K // 8), generator=g, device="cuda", dtype=torch.int64).to(torch.int32)
    s, b = (torch.rand((N, K // 64), generator=g, device="cuda").to(torch.bfloat16) for _ in range(2))
    m = Q4Matrix(w, s, b)
    x = torch.randn((rows, K), generator=g, device="cuda").to(torch.bfloat16)
    want = q4_gemv(x, m, out)
    wide, odd = torch.zeros((rows, K + 8), device="cuda").bfloat16(), torch.zeros((rows, K + 3), device="cuda").bfloat16()
    wide[:, :K] = x
    odd[:, 3:] = x
    forms = {"wide": wide[:, :K], "odd": odd[:, 3:], "column": x.t().contiguous().t(), "3d": x.reshape(rows, 1, K),
             "3d strided": wide[:, None, :K], "4d": x.reshape(1, rows, 1, K), "grad": x.clone().requires_grad_()}
    if rows == 1:  # one misaligned row counts as contiguous and is refused
        with pytest.raises(ValueError):
            q4_gemv(forms.pop("odd"), m, out)
    for name, f in forms.items():
        y = q4_gemv(f, m, out)
        assert y.shape == (*f.shape[:-1], N) and not y.requires_grad, name
        assert torch.equal(y.reshape(rows, N), want), name
    assert torch.equal(q4_gemv(x[0], m, out), q4_gemv(x[:1], m, out)[0])
    assert q4_gemv(x[:0], m, out).shape == (0, N)
    with pytest.raises(ValueError):
        q4_gemv(x[:, :128], m, out)
    with pytest.raises(ValueError):
        q4_gemv(x.float(), m, out)
