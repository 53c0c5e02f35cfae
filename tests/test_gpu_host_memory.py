"""Transforms on host memory equal those on device memory bit for bit: pageable memory goes through
a ring of two 1 MiB chunks, pinned memory directly."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("N,P,single", [
    (2 ** 13, 4, False),                # below one chunk, copied by one thread
    (2 ** 16, 8, False),                # one chunk exactly
    (3 * 2 ** 15, 8, False),            # 1.5 chunks
    (2 ** 17, 8, False),                # the ring once
    (5 * 2 ** 16, 8, True),             # 2.5 chunks
    (9 * 2 ** 15, 8, False),            # 4.5: the slots again, a partial chunk last
    (2 ** 16, 16, True),
])
def test_host_matches_device(soi, torch_cuda, N, P, single):
    torch = torch_cuda
    prec = soi.SOI_PREC_FP32 if single else soi.SOI_PREC_FP64
    d = soi.make_descriptor(N, P, precision=prec)
    rng = np.random.default_rng(N)
    x = (rng.uniform(-1, 1, N) + 1j * rng.uniform(-1, 1, N)).astype(np.complex64 if single else np.complex128)
    t = torch.from_numpy(x).cuda()
    torch.cuda.synchronize()
    print(f"case host N={N} P={P} single={single}", flush=True)
    try:
        soi.compute_soi(d, t.data_ptr())
        ref = t.cpu().numpy()
        pageable = np.full(N + 16, 7, x.dtype)
        for _ in range(2):
            pageable[8:N + 8] = x
            soi.compute_soi(d, pageable[8:].ctypes.data)
            assert np.array_equal(pageable[8:N + 8].view(np.uint8), ref.view(np.uint8))
            assert np.all(pageable[:8] == 7) and np.all(pageable[N + 8:] == 7)
        pinned = torch.empty(N, dtype=t.dtype, pin_memory=True)
        pinned.copy_(torch.from_numpy(x))
        soi.compute_soi(d, pinned.data_ptr())
        assert np.array_equal(pinned.numpy().view(np.uint8), ref.view(np.uint8))
    finally:
        soi.free_soi_descriptor(d)


@pytest.mark.parametrize("N", [2 ** 14, 2 ** 18])
def test_pageable_memory_is_read_in_stream_order(soi, torch_cuda, N):
    """A host function on the caller's stream fills the pageable buffer; the transform that follows in the stream
    reads what it wrote, on a plan's first call and later ones (one chunk and a ring)."""
    import ctypes
    import time

    from gpu_util import hip
    torch = torch_cuda
    rng = np.random.default_rng(N)
    x = rng.uniform(-1, 1, N) + 1j * rng.uniform(-1, 1, N)
    d = soi.make_descriptor(N, 4)
    t = torch.from_numpy(x).cuda()
    torch.cuda.synchronize()
    buf = np.zeros_like(x)

    @ctypes.CFUNCTYPE(None, ctypes.c_void_p)
    def fill(_):
        time.sleep(0.05)
        buf[:] = x

    s = torch.cuda.Stream()
    print(f"case host function N={N}", flush=True)
    try:
        soi.compute_soi(d, t.data_ptr())
        ref = t.cpu().numpy()
        for _ in range(3):
            buf[:] = 0
            assert hip().hipLaunchHostFunc(ctypes.c_void_p(s.cuda_stream), fill, None) == 0
            soi.compute_soi_async(d, buf.ctypes.data, s.cuda_stream)
            s.synchronize()
            assert np.array_equal(buf.view(np.uint8), ref.view(np.uint8))
    finally:
        soi.free_soi_descriptor(d)
