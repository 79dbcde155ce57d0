"""Layers of 9 to 16 rows at K <= 4 on both sides of the lines between the medium-batch and the rows kernel."""
import pytest
import torch

from conftest import rel_l2

pytestmark = pytest.mark.gpu
# fp16 rotated activations and weights, fp32 sums, fp16 output: the bar of the other layer comparisons
TOL = 1e-3


# whole reductions: 430 column groups and one fewer, 340 at 14 steps and at 15, 256 and 257 groups, 200 and 199 at 17
# steps; ranges: 6 x 80 workgroups of 16 steps, 9 and of 21 steps, 3 x 149 and 3 x 150, 96 groups (medium-batch workgroups fill the
# chip evenly), 31 steps at K = 3
@pytest.mark.parametrize("rows,k,cb,blocks,groups", [
    (16, 4, 0, 16, 430), (9, 4, 1, 16, 429), (12, 3, 2, 14, 340), (12, 4, 0, 15, 340), (13, 2, 0, 12, 256), (13, 2, 0, 12, 257),
    (16, 4, 1, 17, 200), (10, 4, 0, 17, 199), (11, 4, 0, 96, 80), (14, 4, 2, 54, 80), (12, 4, 0, 63, 160), (15, 2, 1, 33, 149),
    (15, 2, 1, 33, 150), (12, 4, 0, 56, 96), (9, 3, 0, 93, 160)])
def test_either_side_of_the_lines(cuda, rows, k, cb, blocks, groups):
    from ponyexl3_amd import ops

    n_in, n_out = 128 * blocks, 128 * groups
    g = torch.Generator(device=cuda).manual_seed(rows + groups)
    tr = torch.randint(-32768, 32768, (n_in // 16, n_out // 16, 16 * k), dtype=torch.int16, device=cuda, generator=g)
    sign = lambda n: (torch.randint(0, 2, (n,), device=cuda, generator=g) * 2 - 1).half()
    suh, svh = sign(n_in), sign(n_out) * n_in**-0.5
    bias = torch.randn(n_out, device=cuda, generator=g).half()
    x = torch.randn((rows, n_in), device=cuda, generator=g).half()
    print(f"rows={rows} k={k} {n_in}->{n_out}", flush=True)
    y = ops.linear_forward(x, tr, k, cb, suh, svh, bias)
    assert torch.equal(y, ops.linear_forward(x, tr, k, cb, suh, svh, bias))
    assert int(ops.sync_counters(cuda, 1).abs().sum()) == 0
    # the chain of separate kernels on the first, a middle and the last column group
    xh = ops.had128_pre(x, suh).reshape(rows, n_in).double()
    for c0 in (0, groups // 2 * 128, n_out - 128):
        w = ops.decode_full(tr[:, c0 // 16:c0 // 16 + 8].contiguous(), k, cb).double()
        ref = ops.had128_post((xh @ w).half(), svh[c0:c0 + 128].contiguous(), bias[c0:c0 + 128].contiguous())
        assert rel_l2(y[:, c0:c0 + 128].float().cpu().numpy(), ref.float().cpu().numpy()) <= TOL
