"""The native host module as built (no GPU): it loads, leaves what it does not
take to the general path, and brings no thread-local storage (which would slow
down every other library's, see rec_amd/build.py)."""

import struct

from rec_amd import _lib, build


def test_no_thread_local_storage():
    with open(build.HOST, "rb") as f:
        elf = f.read()
    assert elf[:4] == b"\x7fELF" and elf[4] == 2  # 64-bit
    off, = struct.unpack_from("<Q", elf, 32)
    size, count = struct.unpack_from("<HH", elf, 54)
    kinds = [struct.unpack_from("<I", elf, off + i * size)[0] for i in range(count)]
    assert 1 in kinds and 7 not in kinds  # PT_LOAD, no PT_TLS


def test_general_path_left_alone():
    import torch

    h = _lib.host()
    x = torch.zeros((2, 128), dtype=torch.bfloat16)  # host tensors, other arguments, too few of them
    assert h.q4_matmul(x, x, 16, 128, False, 9, 0) is None
    assert h.q4_matmul(None, x, 16, 128, False, 9, 0) is None
    assert h.q4_matmul(x) is None and h.decode_ring(x) is None and h.decode_quantized(x) is None
