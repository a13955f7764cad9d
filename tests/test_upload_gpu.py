"""rr_upload: blocks of host memory to device memory through one pinned buffer, byte
for byte (the parameters of a served batch)."""
import numpy as np
import pytest
import torch

from pytransit_amd import _lib


@pytest.mark.gpu
@pytest.mark.parametrize('sizes', [(1,), (16,), (15, 17, 0, 4096), (256,) * 16, (0, 0), (3_000_001, 8, 1_048_576)])
def test_blocks_arrive_unchanged(sizes):
    lib = _lib.load()
    rng = np.random.default_rng(len(sizes))
    src = [rng.integers(0, 256, n, dtype=np.uint8) for n in sizes]
    room = [(n + 15) // 16 * 16 for n in sizes]
    staging = torch.empty(max(sum(room), 16), dtype=torch.uint8, pin_memory=True)
    dst = [torch.full((r + 16,), 7, dtype=torch.uint8, device='cuda') for r in room]
    pieces = (_lib.RRPiece * len(sizes))(*[_lib.RRPiece(s.ctypes.data, d.data_ptr(), n)
                                           for s, d, n in zip(src, dst, sizes)])
    _lib.check(lib.rr_upload(len(sizes), pieces, staging.data_ptr(), staging.numel(),
                             _lib.stream_handle(dst[0].device)))
    torch.cuda.synchronize()
    for s, d, n, r in zip(src, dst, sizes, room):
        assert np.array_equal(d.cpu().numpy()[:n], s)
        assert (d.cpu().numpy()[r:] == 7).all()


@pytest.mark.parametrize('n, nbytes, room, shift', [(17, 16, 4096, 0), (1, 17, 16, 0), (1, 16, 4096, 8), (-1, 0, 0, 0)])
def test_bad_blocks_are_refused(n, nbytes, room, shift):
    lib = _lib.load(require_gpu=False)
    host = np.zeros(8192, np.uint8)
    base = (host.ctypes.data + 63) // 64 * 64
    pieces = (_lib.RRPiece * 17)(*[_lib.RRPiece(base, base + shift, nbytes)] * 17)
    assert lib.rr_upload(n, pieces, base, room, None) != 0
