"""One row of layers that fill the chip: waves of half a Hadamard block in workgroups of eight and of four."""
import ctypes

import pytest
import torch

from conftest import rel_l2

pytestmark = pytest.mark.gpu
# at activations of 1 and of 1e-5 (whose sums a coarse grid would lose): fp16 rounding of the output, fp16 rotated activations, the exact sum of a weight's halves (4.8e-4 at most)
TOL = 1e-3


def _plan(k, n_in, n_out):
    from ponyexl3_amd import _lib

    out = [ctypes.c_int() for _ in range(4)]
    _lib.check(_lib.load().exl3_linear_plan(1, n_in // 16, n_out // 16, k, *[ctypes.byref(v) for v in out]), "plan")
    return tuple(v.value for v in out)  # splits, tile rows, waves, accumulators


# (tile rows of a wave, waves of a workgroup, accumulators or partial rows) that the layer is to take: a last workgroup with
# waves to spare (33 blocks), 15 contributors in half blocks and the first count beyond them, whose words would be coarser than those
# of whole blocks, 31 where whole blocks have 16, two blocks, one block in partial rows, four waves up to 15 contributors and eight beyond
@pytest.mark.parametrize("k,cb,n_in,n_out,tile_rows,waves,atomics", [
    (4, 0, 4224, 24576, 4, 8, 1), (6, 1, 7680, 9216, 4, 8, 1), (6, 1, 8320, 8192, 16, 4, 1), (8, 2, 15872, 4352, 4, 8, 1),
    (5, 0, 17408, 5120, 16, 4, 1), (4, 0, 17408, 10240, 8, 8, 1), (3, 1, 3072, 24576, 4, 4, 1), (7, 0, 256, 262144, 4, 8, 1),
    (7, 0, 128, 524288, 8, 4, 0), (2, 0, 1024, 65536, 4, 4, 1), (4, 1, 3840, 17536, 4, 4, 1), (4, 1, 4096, 16896, 4, 8, 1)])
def test_half_block_waves_of_a_full_chip(cuda, k, cb, n_in, n_out, tile_rows, waves, atomics):
    splits, rows_of_wave, wg_waves, atomic = _plan(k, n_in, n_out)
    assert (rows_of_wave, wg_waves, atomic) == (tile_rows, waves, atomics)
    g = torch.Generator(device=cuda).manual_seed(n_in + k)
    tr = torch.randint(-32768, 32768, (n_in // 16, n_out // 16, 16 * k), dtype=torch.int16, device=cuda, generator=g)
    sign = lambda n: (torch.randint(0, 2, (n,), device=cuda, generator=g) * 2 - 1).half()
    suh, svh = sign(n_in), sign(n_out)
    bias = torch.randn(n_out, device=cuda, generator=g).half()
    print(f"one row k={k} {n_in}->{n_out}", flush=True)
    for scale in (1.0, 1e-5):
        x = (torch.randn((1, n_in), device=cuda, generator=g) * scale).half()
        _check(cuda, x, tr, k, cb, suh, svh, bias * scale, n_in, n_out)


def _check(cuda, x, tr, k, cb, suh, svh, bias, n_in, n_out):
    from ponyexl3_amd import ops

    y = ops.linear_forward(x, tr, k, cb, suh, svh, bias)
    assert torch.equal(y, ops.linear_forward(x, tr, k, cb, suh, svh, bias))
    assert int(ops.sync_counters(cuda, 1).abs().sum()) == 0
    # the chain of separate kernels on the first and the last column group
    xh = ops.had128_pre(x, suh)
    for c0 in (0, n_out - 128):
        part = tr[:, c0 // 16:c0 // 16 + 8].contiguous()
        w = ops.decode_full(part, k, cb).double()
        ref = ops.had128_post((xh.reshape(1, n_in).double() @ w).half(), svh[c0:c0 + 128].contiguous(),
                              bias[c0:c0 + 128].contiguous())
        assert rel_l2(y[:, c0:c0 + 128].float().cpu().numpy(), ref.float().cpu().numpy()) <= TOL
