"""The tiled Hadamard passes against the float32 butterflies of fwht_numpy
(src/rht/transform.py:26-42) in torch.  The additions and their order are the same and the
scales used are exact, so results are equal bit for bit (up to the sign of a zero)."""
import ctypes

import pytest
import torch

pytestmark = pytest.mark.gpu


def _fwht(x, dim):
    x = x.transpose(dim, -1).contiguous()
    shape, h = x.shape, 1
    while h < shape[-1]:
        y = x.view(-1, shape[-1] // (2 * h), 2, h)
        x = torch.stack([y[:, :, 0] + y[:, :, 1], y[:, :, 0] - y[:, :, 1]], 2).view(shape)
        h *= 2
    return x.transpose(dim, -1).contiguous()


def _signs(*shape, seed):
    return torch.randint(0, 2, shape, device="cuda", generator=torch.Generator("cuda").manual_seed(seed)).float() * 2 - 1


# One pass: tiles below a wave's block, of 2^11, and with 1, 2 and 3 exchanged bits.  Two
# passes: every number of row bits of the second (1-5 in registers, 6-10 with an exchange).
# (2048, 16384): 10 row bits and one more pass.
SHAPES = [(1, 64), (8, 64), (32, 64), (64, 64), (2, 4096), (1, 8192), (1, 16384), (256, 64), (2, 16384), (4, 16384),
          (8, 16384), (512, 64), (1024, 64), (64, 1024), (2048, 64), (256, 2048), (512, 2048), (16384, 128),
          (2048, 2048), (4096, 2048), (8192, 2048), (2048, 16384)]


@pytest.mark.parametrize("batch", [1, 3])
@pytest.mark.parametrize("m,n", SHAPES)
def test_rht_passes(bcjr_mod, m, n, batch):
    if batch > 1 and m * n > 1 << 22:
        pytest.skip("one matrix of this size fills the device")
    print(f"rht passes {batch} x {m} x {n}", flush=True)
    W = torch.randn(batch, m, n, device="cuda", generator=torch.Generator("cuda").manual_seed(m + n))
    sl, sr = _signs(batch, m, seed=1), _signs(batch, n, seed=2)
    # float32(1 / sqrt(m n)) multiplies once at the end
    s = torch.tensor(1.0 / (m * n) ** 0.5, dtype=torch.float32, device="cuda")
    got = bcjr_mod.apply_rht_batched(W, sl, sr)
    assert torch.equal(got, _fwht(_fwht(W * sr[:, None], 2) * sl[:, :, None], 1) * s)
    got = bcjr_mod.apply_inverse_rht_batched(W, sl, sr)
    assert torch.equal(got, sl[:, :, None] * _fwht(_fwht(W, 2) * sr[:, None], 1) * s)


@pytest.mark.parametrize("rows,n", [(1, 64), (33, 64), (96, 64), (3, 1024), (16, 1024), (5, 4096), (8, 4096),
                                    (3, 8192), (2, 16384)])
@pytest.mark.parametrize("offset", [0, 1])
def test_hadamard_rows_and_unaligned_output(bcjr_mod, rows, n, offset):
    """Rows only, and an output that is not 16-byte aligned, through the C ABI."""
    from bcjr import _lib
    print(f"hadamard {rows} x {n}, output offset {offset}", flush=True)
    x = torch.randn(rows, n, device="cuda", generator=torch.Generator("cuda").manual_seed(n))
    buf = torch.full((rows * n + 8,), 7.0, device="cuda")
    rc = _lib.load().bcjr_hadamard(x.data_ptr(), buf.data_ptr() + 4 * offset, rows, n, 0.25,
                                   ctypes.c_void_p(torch.cuda.current_stream().cuda_stream))
    assert rc == 0
    assert torch.equal(buf[offset:offset + rows * n].view(rows, n), _fwht(x, 1) * 0.25)
    assert bool((buf[:offset] == 7.0).all()) and bool((buf[offset + rows * n:] == 7.0).all())
