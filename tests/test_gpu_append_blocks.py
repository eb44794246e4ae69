"""A long append (one wavefront per whole 32-token block) leaves the same cache
bytes as the same rows appended a few at a time (one wavefront per row, the
path the oracle's tests pin), for every format and input type."""

import pytest
import torch

import rec_amd

pytestmark = pytest.mark.gpu

FORMATS = {"int8": (32, 8, 8), "uint4": (32, 4, 4), "k8v4": (32, 8, 4), "k4v8": (32, 4, 8), "affine": (64, 8, 4)}
DTYPES = {"bf16": torch.bfloat16, "fp16": torch.float16, "fp32": torch.float32}
B, H, T = 2, 8, 640


def rows(dtype, seed):
    """Normal rows among ones that reach every branch: exact ties, constant,
    zero, tiny, huge, infinite and NaN values."""
    g = torch.Generator().manual_seed(seed)
    x = torch.randn((B, H, T, 128), generator=g) * torch.exp(torch.randn((B, H, T, 1), generator=g) * 3)
    x[:, :, 3::17] = torch.randint(-254, 255, x[:, :, 3::17].shape, generator=g) * 0.5  # halves of the step when 127 is hit
    x[:, :, 3::34, ::32] = 127.0
    x[:, :, 5::41] = 0.0
    x[:, :, 6::43] = 2.5
    x[:, :, 7::47] *= 1e-9
    x[:, :, 8::53, :64] = torch.randint(0, 16, (64,), generator=g).float()
    x[0, :, 9::59, 5] = float("inf")
    x[1, :, 9::59, 70] = float("-inf")
    x[:, :, 10::61, 33] = float("nan")
    x[0, 0, 11::67] = float("nan")
    if dtype != torch.float16:
        x[:, 1, 12::71] *= 1e30
    return x.to(dtype).cuda()


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("fmt", FORMATS)
@pytest.mark.parametrize("offset", [0, 37])
def test_blocks_equal_rows(gpu, fmt, dtype, offset):
    k, v = rows(DTYPES[dtype], 1), rows(DTYPES[dtype], 2)
    long, short = (rec_amd.QuantizedKVCache(*FORMATS[fmt], max_tokens=704) for _ in range(2))
    if offset:
        for c in (long, short):
            c.update_and_fetch(k[:, :, :offset], v[:, :, :offset])
    n = T - offset - 9  # 18 or 19 whole blocks of 16 heads, and rows at the ends
    end = offset + n
    long.update_and_fetch(k[:, :, offset:end], v[:, :, offset:end])
    for t in range(offset, end, 50):
        short.update_and_fetch(k[:, :, t:min(t + 50, end)], v[:, :, t:min(t + 50, end)])
    torch.cuda.synchronize()
    for a, b in zip((*long.keys, *long.values), (*short.keys, *short.values)):
        if a is not None:
            assert torch.equal(a.view(torch.uint8), b.view(torch.uint8))
