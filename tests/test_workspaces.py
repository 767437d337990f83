"""Workspaces handed to kernels: a captured graph keeps the address it was
recorded with, so a buffer that a larger call outgrows stays allocated."""

import weakref

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
