"""Workspaces handed to kernels: a captured graph keeps the address it was
recorded with, so a buffer that a larger call outgrows stays allocated; and the
K parts of the tiles matmul, which its workspace holds."""

import weakref

import pytest
import torch

from mtplx_amd import _lib


def test_an_outgrown_buffer_stays_allocated(monkeypatch):
    zeros = torch.zeros
    monkeypatch.setattr(_lib, "stream_handle", lambda dev=None: 0)
    monkeypatch.setattr(torch, "zeros", lambda n, dtype, device: zeros(n, dtype=dtype))   # host memory in its place
    pool = _lib._Workspaces()
    small = pool.get(1000, "tag", "cuda:0")
    address = small.data_ptr()
    alive = weakref.ref(small)
    del small
    assert pool.get(900, "tag", "cuda:0").data_ptr() == address
    large = pool.get(5000, "tag", "cuda:0")
    assert large.numel() >= 5000 and large.data_ptr() != address
    assert alive() is not None and alive().data_ptr() == address
    # sizes at least double: what is kept is no larger than the buffer in use
    for n in range(5000, 60000, 999):
        last = pool.get(n, "tag", "cuda:0")
    assert sum(b.numel() for b in pool._outgrown) <= last.numel()


@pytest.mark.parametrize("m,n,k,parts", [
    (512, 5120, 17408, 3), (512, 5120, 4096, 1),     # 40 workgroups on each XCD's 32 CUs: long and short parts
    (768, 4096, 12288, 2), (1536, 1536, 17408, 2),   # 48 (of 12 column groups: on half of the XCDs)
    (768, 5120, 17408, 1), (512, 7168, 17408, 1),    # 60, 56: parts would not shorten the fullest CU's work
    (512, 4096, 12288, 1),                           # one on every CU
    (512, 17408, 5120, 1), (128, 5120, 17408, 3), (65, 1024, 5120, 8),
])
def test_tiles_parts(m, n, k, parts):
    if torch.cuda.is_available() and torch.cuda.get_device_properties(0).multi_processor_count != 256:
        pytest.skip("planned for 256 CUs")
    sums = (m * (k // 256) * 32 + 255) // 256 * 256
    held = _lib.query("mtp_qmm_tiles_workspace_bytes", m, n, k) - sums
    assert held == (4 * parts * m * n if parts > 1 else 0)
