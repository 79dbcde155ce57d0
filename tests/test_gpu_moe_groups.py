"""Slots of a routing table grouped by expert through the list that one workgroup makes of it."""
import numpy as np
import pytest
import torch

from conftest import rel_l2

pytestmark = pytest.mark.gpu
# two chains of fp16 casts with fp32 sums in other orders, and the down projection's unsummed halves in one
# of them up to 23 tokens: the bar of the other chain comparisons
TOL = 1e-3


def _switch(E, D, H, k, cb, seed, device):
    from ponyexl3_amd import EXL3SwitchGLU

    g = torch.Generator(device=device).manual_seed(seed)
    tr = lambda a, b: torch.randint(-32768, 32768, (a // 16, b // 16, 16 * k), dtype=torch.int16, device=device, generator=g)
    sg = lambda *s, c=1.0: ((torch.randint(0, 2, s, device=device, generator=g) * 2 - 1) * c).half()
    return EXL3SwitchGLU(gu_trellis=tr(D, E * 2 * H), gu_suh=sg(E, 2, D), gu_svh=sg(E, 2 * H, c=0.8 * D**-0.5),
                         dn_trellis=tr(H, E * D), dn_suh=sg(E, H), dn_svh=sg(E, D, c=0.8 * H**-0.5), k=k, cb=cb)


# groups of one to four rows, a slot past the last group, 256 and 512 slots (whole passes of the workgroup's
# threads) and one more, the largest list and the first call that has none, experts beyond the 64 and 256 that a
# wave and a workgroup scan at once, D and H of blocks that leave waves idle
@pytest.mark.parametrize("tokens,top_k,E,D,H,k,hot", [(7, 3, 3, 256, 128, 4, False), (43, 6, 65, 640, 128, 3, True),
                                                      (64, 4, 30, 256, 640, 4, False), (128, 4, 300, 128, 128, 4, True),
                                                      (171, 3, 257, 256, 128, 5, False), (256, 4, 700, 128, 128, 4, True),
                                                      (205, 5, 20, 128, 256, 2, False)])
def test_grouped_slots_against_the_launch_chain(cuda, tokens, top_k, E, D, H, k, hot):
    from ponyexl3_amd import ops

    m = _switch(E, D, H, k, 1, tokens, cuda)
    rng = np.random.default_rng(tokens)
    idx = np.stack([rng.permutation(E)[:top_k] for _ in range(tokens)]).astype(np.int32)
    if hot:  # an expert that every token has
        idx[:, -1] = np.where((idx == E - 1).any(1), idx[:, -1], E - 1)
    x = torch.from_numpy(rng.standard_normal((tokens, D)).astype(np.float16)).to(cuda)
    args = (x, torch.from_numpy(idx).to(cuda), m._gu_trellis, m._gu_suh, m._gu_svh, m._dn_trellis, m._dn_suh, m._dn_svh,
            k, 1)
    print(f"grouped slots tokens={tokens} top_k={top_k} E={E}", flush=True)
    y = ops.moe_forward(*args)
    assert torch.equal(y, ops.moe_forward(*args))
    assert int(ops.sync_counters(cuda, 1).abs().sum()) == 0
    ref = ops.moe_forward(*args, fused=False)
    worst = (y.double() - ref.double()).flatten(0, 1).norm(dim=1) / ref.double().flatten(0, 1).norm(dim=1)
    assert rel_l2(y.float().cpu().numpy(), ref.float().cpu().numpy()) <= TOL
    assert float(worst.max()) <= 2 * TOL  # a row of another slot or expert would be off by order one


@pytest.mark.parametrize("tokens,E,top_k,shared", [(8, 9, 4, False), (21, 60, 4, True), (33, 256, 8, True),
                                                   (57, 200, 7, False), (100, 500, 8, True)])
def test_block_with_the_list_made_behind_the_router(cuda, tokens, E, top_k, shared):
    """The last workgroup of the router's launch makes the list: the block against its parts, where a launch
    of its own makes it. Three calls, so that the arrival counter is seen to go back to zero."""
    from ponyexl3_amd import EXL3MoEBlock, ops
    from ponyexl3_amd.moe import combine_experts

    D, H = 256, 128
    switch = _switch(E + shared, D, H, 4, 0, tokens, cuda)
    g = torch.Generator().manual_seed(tokens)
    lin = lambda n: torch.nn.Linear(D, n, bias=False).half().to(cuda).requires_grad_(False)
    block = EXL3MoEBlock(lin(E), lin(1) if shared else None, switch, top_k)
    print(f"block with list tokens={tokens} E={E}", flush=True)
    for _ in range(3):
        x = torch.randn((1, tokens, D), generator=g).half().to(cuda)
        y = block(x)
        inds, scores = block.route(x)
        ref = combine_experts(switch(x, inds).float(), scores)
        assert rel_l2(y.float().cpu().numpy(), ref.cpu().numpy()) <= TOL
        assert int(ops.sync_counters(cuda, 1).abs().sum()) == 0


@pytest.mark.parametrize("tokens,top_k,E", [(24, 1, 8), (25, 1, 10), (24, 1, 2), (24, 2, 16), (64, 4, 30)])
def test_down_weights_are_rounded_from_the_prefills_sizes_on(cuda, tokens, top_k, E):
    """From 24 tokens and 2.5 slots per expert on the slot kernels are no further from the reference's arithmetic
    than the prefill, also where hardly any slots are spared: the launch chain, whose weights are rounded,
    differs by the order of fp32 sums, i.e. fp16 roundings here and there, well under the 4e-4 and more that unsummed
    halves make (2^-11 per weight)."""
    from ponyexl3_amd import ops

    D, H, k = 512, 256, 4
    m = _switch(E, D, H, k, 0, 31 * tokens + E, cuda)
    rng = np.random.default_rng(tokens + E)
    idx = torch.from_numpy(np.stack([rng.permutation(E)[:top_k] for _ in range(tokens)]).astype(np.int32)).to(cuda)
    x = torch.from_numpy(rng.standard_normal((tokens, D)).astype(np.float16)).to(cuda)
    args = (x, idx, m._gu_trellis, m._gu_suh, m._gu_svh, m._dn_trellis, m._dn_suh, m._dn_svh, k, 0)
    print(f"rounded down weights tokens={tokens} top_k={top_k} E={E}", flush=True)
    y, ref = ops.moe_forward(*args), ops.moe_forward(*args, fused=False)
    assert rel_l2(y.float().cpu().numpy(), ref.float().cpu().numpy()) <= 2.5e-4
