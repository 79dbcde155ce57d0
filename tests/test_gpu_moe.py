"""Routed MoE expert chain against the oracle's unfused per-expert chain."""
import ctypes
import os

import numpy as np
import pytest
import torch

from conftest import rel_l2

pytestmark = pytest.mark.gpu
TOL = 1e-3


def _experts(E, D, H, k, mcg, seed):
    from ponyexl3_amd import make_exl3_layer

    mk = lambda i, n_in, n_out, tag: make_exl3_layer(k=k, in_features=n_in, out_features=n_out,
                                                     seed=seed + i, mcg=mcg, key=f"e{i}.{tag}")
    gate = [mk(3 * e, D, H, "gate") for e in range(E)]
    up = [mk(3 * e + 1, D, H, "up") for e in range(E)]
    down = [mk(3 * e + 2, H, D, "down") for e in range(E)]
    return gate, up, down


def _switch(E, D, H, k):
    from ponyexl3_amd import EXL3SwitchGLU

    return EXL3SwitchGLU.from_layers(*_experts(E, D, H, k, False, 1300))


def _oracle_chain(oracle, gate, up, down, x, idx, act):
    experts = [{"gate": (g.trellis, g.suh, g.svh), "up": (u.trellis, u.suh, u.svh),
                "down": (d.trellis, d.suh, d.svh)} for g, u, d in zip(gate, up, down)]
    return oracle.moe_experts_forward(experts, x, idx, gate[0].k, gate[0].codebook_mode, act)


@pytest.mark.parametrize("tokens", [1, 3, 8])
@pytest.mark.parametrize("k,mcg,act", [(4, False, "silu"), (3, True, "silu"), (4, True, "gelu")])
def test_moe_matches_oracle(cuda, oracle, tokens, k, mcg, act):
    from ponyexl3_amd import EXL3SwitchGLU

    E, D, H, kk = 6, 256, 128, 2
    gate, up, down = _experts(E, D, H, k, mcg, 500)
    moe = EXL3SwitchGLU.from_layers(gate, up, down, activation=act)
    rng = np.random.default_rng(tokens + k)
    x = (rng.standard_normal((tokens, D)) * 0.5).astype(np.float16)
    idx = np.stack([rng.permutation(E)[:kk] for _ in range(tokens)]).astype(np.int32)
    print(f"moe tokens={tokens} k={k} act={act}", flush=True)
    y = moe(torch.from_numpy(x).to(cuda).reshape(1, tokens, D),
            torch.from_numpy(idx).to(cuda).reshape(1, tokens, kk)).cpu().numpy()
    assert y.shape == (1, tokens, kk, D)
    ref = _oracle_chain(oracle, gate, up, down, x, idx, act)
    assert rel_l2(y[0], ref) <= TOL


@pytest.mark.parametrize("tokens", [1, 8, 48])
def test_two_launch_and_five_launch_chains(cuda, oracle, tokens):
    """D and H of five Hadamard blocks each: both kernels of the two-launch chain
    run two workgroups per column block (one of them with a single active wave)
    and meet through the counters. 1 and 8 tokens take the eight-wave workgroups
    on half blocks, 48 tokens (96 slots) the four-wave ones on whole blocks.
    Checked against the oracle, against the five-launch chain, and twice in a row
    (the counters must be left at zero)."""
    from ponyexl3_amd import EXL3SwitchGLU, ops

    E, D, H, kk, k = 5, 640, 640, 2, 4
    gate, up, down = _experts(E, D, H, k, False, 700)
    moe = EXL3SwitchGLU.from_layers(gate, up, down)
    rng = np.random.default_rng(70 + tokens)
    x = (rng.standard_normal((tokens, D)) * 0.5).astype(np.float16)
    idx = np.stack([rng.permutation(E)[:kk] for _ in range(tokens)]).astype(np.int32)
    xt, it = torch.from_numpy(x).to(cuda), torch.from_numpy(idx).to(cuda)
    args = (xt, it, moe._gu_trellis, moe._gu_suh, moe._gu_svh, moe._dn_trellis, moe._dn_suh, moe._dn_svh,
            k, moe._cb)
    print(f"moe two-launch tokens={tokens}", flush=True)
    y1 = ops.moe_forward(*args, fused=True)
    y2 = ops.moe_forward(*args, fused=True)
    y5 = ops.moe_forward(*args, fused=False)
    assert torch.equal(y1, y2)
    assert int(ops.sync_counters(cuda, 1).abs().sum()) == 0
    ref = _oracle_chain(oracle, gate, up, down, x, idx, "silu")
    assert rel_l2(y1.cpu().numpy(), ref) <= TOL
    assert rel_l2(y5.cpu().numpy(), ref) <= TOL
    assert rel_l2(y1.cpu().numpy(), y5.cpu().numpy()) <= TOL


def _groups_of(ws, slots, D, H):
    """Number of groups in the list that a grouped call leaves in its workspace (behind the two buffers of rotated rows)."""
    at = sum((n * 2 + 255) // 256 * 256 for n in (slots * 2 * D, slots * H))
    return int(ws[at:at + 4].view(torch.int32)[0])


def _moe_forward(x, idx, moe, k, D, H):
    """exl3_moe_forward as ops.moe_forward with accumulators=False calls it, with a workspace that can be looked at."""
    from ponyexl3_amd import _lib, ops

    lib, p, (tokens, top_k) = _lib.load(), ops._ptr, idx.shape
    need = lib.exl3_moe_workspace_bytes(tokens, top_k, D, H)
    ws = torch.full((need,), 0xCC, dtype=torch.uint8, device=x.device)
    y = torch.empty((tokens, top_k, D), dtype=torch.float16, device=x.device)
    n = tokens * top_k * (H // 128 + D // 128)
    cnt = ops.sync_counters(x.device, n)
    _lib.check(lib.exl3_moe_forward(p(x), tokens, p(idx), top_k, p(moe._gu_trellis), p(moe._gu_suh), p(moe._gu_svh),
                                    p(moe._dn_trellis), p(moe._dn_suh), p(moe._dn_svh), moe.num_experts, D, H, k, moe._cb, 0,
                                    p(y), p(ws), need, p(cnt), n + 2, ops._stream()), "exl3_moe_forward")
    assert int(cnt.abs().sum()) == 0
    return y, ws


# few and many experts, groups of one to four rows and up to 20 of one expert, one and two workgroups a reduction; up to
# K = 4 half blocks below 4096 waves of whole ones and whole blocks from there on, from K = 5 on half blocks throughout
@pytest.mark.parametrize("tokens,top_k,E,D,H,k,whole", [
    (9, 3, 4, 384, 256, 4, False), (32, 2, 40, 384, 256, 4, False), (12, 3, 6, 640, 128, 6, False), (23, 7, 12, 256, 640, 8, False),
    (20, 8, 16, 640, 384, 4, True), (23, 7, 30, 640, 640, 3, True)])
def test_slots_grouped_by_expert_equal_ungrouped(cuda, tokens, top_k, E, D, H, k, whole):
    """With several tokens the slots of one expert share a pass over its weights, four rows at a time. Below the
    prefill's sizes the arithmetic per row is that of the per-slot kernels, so the result is bit-identical to runs that do
    not group, take the same blocks and reduce through partial rows too: one token at a time where waves take half
    blocks, and where they take whole ones the same tokens among more than 1024 slots, which no list holds."""
    moe = _switch(E, D, H, k)
    many = 1024 // top_k + 1
    rng = np.random.default_rng(tokens * 7 + E)
    x = torch.from_numpy((rng.standard_normal((many, D)) * 0.5).astype(np.float16)).to(cuda)
    idx = torch.from_numpy(np.stack([rng.permutation(E)[:top_k] for _ in range(many)]).astype(np.int32)).to(cuda)
    slots = tokens * top_k
    assert (slots * 2 * (D // 128) * (H // 128) >= 4096) == whole and (tokens < 24 or slots < 2.5 * E)
    print(f"moe grouped tokens={tokens} top_k={top_k} E={E} k={k}", flush=True)
    y, ws = _moe_forward(x[:tokens], idx[:tokens], moe, k, D, H)
    count = torch.bincount(idx[:tokens].flatten().long(), minlength=E)
    assert _groups_of(ws, slots, D, H) == int(((count + 3) // 4).sum()) < slots
    assert torch.equal(y, _moe_forward(x[:tokens], idx[:tokens], moe, k, D, H)[0])
    if whole:
        wide, ws = _moe_forward(x, idx, moe, k, D, H)
        assert _groups_of(ws, many * top_k, D, H) == -0x33333334  # 0xCCCCCCCC: no list
        assert torch.equal(y, wide[:tokens])
    else:
        for t in range(tokens):
            assert torch.equal(y[t], _moe_forward(x[t:t + 1], idx[t:t + 1], moe, k, D, H)[0][0]), f"token {t}"


@pytest.mark.parametrize("tokens,top_k,E,D,H,k", [(256, 2, 3, 384, 256, 4), (256, 2, 3, 384, 256, 6), (24, 2, 16, 384, 256, 4),
                                                  (171, 3, 257, 256, 128, 5)])
def test_rows_of_a_group_do_not_touch_each_other(cuda, tokens, top_k, E, D, H, k):
    """From the prefill's sizes on grouped calls round the down projection's weights, which no ungrouped one does: a slot's
    result is bit for bit that of a call of the same size in which the other tokens have other inputs and other experts, so
    that it sits in another group among other rows (the values themselves: test_down_weights_are_rounded_...)."""
    from ponyexl3_amd import _lib

    assert _lib.load().exl3_moe_groups_rounded(tokens, top_k, E, D, H)
    moe = _switch(E, D, H, k)
    rng = np.random.default_rng(tokens + E)
    draw = lambda: (torch.from_numpy((rng.standard_normal((tokens, D)) * 0.5).astype(np.float16)).to(cuda),
                    torch.from_numpy(np.stack([rng.permutation(E)[:top_k] for _ in range(tokens)]).astype(np.int32)).to(cuda))
    (x, idx), (x2, idx2) = draw(), draw()
    print(f"moe rounded groups tokens={tokens} top_k={top_k} E={E} k={k}", flush=True)
    y, _ = _moe_forward(x, idx, moe, k, D, H)
    kept = torch.from_numpy(rng.permutation(tokens)[:tokens // 3]).to(cuda)
    x2[kept], idx2[kept] = x[kept], idx[kept]
    assert torch.equal(_moe_forward(x2, idx2, moe, k, D, H)[0][kept], y[kept])


@pytest.mark.parametrize("tokens,top_k,E,D,H,act", [(1, 2, 4, 640, 640, 0), (1, 8, 64, 2048, 512, 0),
                                                     (3, 2, 64, 384, 256, 1), (8, 8, 256, 512, 256, 0)])
def test_accumulator_reduction_of_gate_up(cuda, oracle, tokens, top_k, E, D, H, act):
    """Every slot on its own: gate and up of a k-chunk run in one workgroup and meet the
    other chunks in 64-bit accumulators (D of five blocks: three chunks of two blocks, the
    last half empty; 16 blocks: eight chunks). Against the partial-row reduction of the
    same call (an fp16 ulp at most: same products, the sum rounded once instead of per
    row), twice in a row bit for bit, with the accumulators back at zero."""
    from ponyexl3_amd import EXL3SwitchGLU, ops

    k = 4
    rng = np.random.default_rng(tokens * 31 + E)
    if E <= 8:
        gate, up, down = _experts(E, D, H, k, False, 1500)
        moe = EXL3SwitchGLU.from_layers(gate, up, down, activation="silu" if act == 0 else "gelu")
    else:  # random stacks: many experts without building them one by one
        rnd = lambda *s: torch.from_numpy(rng.integers(-32768, 32768, size=s, dtype=np.int16)).to(cuda)
        sgn = lambda *s: torch.from_numpy(np.where(rng.random(s) > 0.5, -1.0, 1.0).astype(np.float16)).to(cuda)
        moe = EXL3SwitchGLU(gu_trellis=rnd(D // 16, E * 2 * H // 16, 16 * k), gu_suh=sgn(E, 2, D),
                            gu_svh=sgn(E, 2 * H), dn_trellis=rnd(H // 16, E * D // 16, 16 * k),
                            dn_suh=sgn(E, H), dn_svh=sgn(E, D), k=k, cb=0)
    x = torch.from_numpy((rng.standard_normal((tokens, D)) * 0.25).astype(np.float16)).to(cuda)
    idx = torch.from_numpy(np.stack([rng.permutation(E)[:top_k] for _ in range(tokens)]).astype(np.int32)).to(cuda)
    args = (x, idx, moe._gu_trellis, moe._gu_suh, moe._gu_svh, moe._dn_trellis, moe._dn_suh, moe._dn_svh, k,
            moe._cb, act)
    print(f"moe accumulators tokens={tokens} top_k={top_k} E={E} D={D} H={H}", flush=True)
    ya = ops.moe_forward(*args)
    ya2 = ops.moe_forward(*args)
    yp = ops.moe_forward(*args, accumulators=False)
    assert torch.equal(ya, ya2)
    assert int(ops.sync_counters(cuda, 1).abs().sum()) == 0
    assert rel_l2(ya.float().cpu().numpy(), yp.float().cpu().numpy()) <= 5e-4  # fp16 ulps over three casts
    if E <= 8:
        ref = _oracle_chain(oracle, gate, up, down, x.cpu().numpy(), idx.cpu().numpy(), "silu" if act == 0 else "gelu")
        assert rel_l2(ya.cpu().numpy(), ref) <= TOL


@pytest.mark.parametrize("seed", range(10))
def test_random_shapes_three_reductions_agree(cuda, seed):
    """Random small shapes (D and H from one to six Hadamard blocks, K from 2 to 8, both
    codebooks, 1..40 tokens, top-k up to 6, few or many experts, indices outside the
    expert range included: they are clamped): the two-launch chain with whatever kernels
    the library picks (accumulators / grouped slots / per-slot partial rows), the same
    with partial rows only, and the five-launch chain must agree to fp16 ulps."""
    from ponyexl3_amd import EXL3SwitchGLU, ops

    rng = np.random.default_rng(9000 + seed)
    D, H = 128 * int(rng.integers(1, 7)), 128 * int(rng.integers(1, 7))
    k = int(rng.integers(2, 9))
    cb = int(rng.integers(0, 2))
    E = int(rng.choice([2, 5, 16, 70]))
    top_k = int(rng.integers(1, min(E, 6) + 1))
    tokens = int(rng.choice([1, 2, 3, 7, 16, 40]))
    act = int(rng.integers(0, 2))
    rnd = lambda *s: torch.from_numpy(rng.integers(-32768, 32768, size=s, dtype=np.int16)).to(cuda)
    sgn = lambda *s: torch.from_numpy(np.where(rng.random(s) > 0.5, -1.0, 1.0).astype(np.float16)).to(cuda)
    gu, dn = rnd(D // 16, E * 2 * H // 16, 16 * k), rnd(H // 16, E * D // 16, 16 * k)
    gu_suh, gu_svh, dn_suh, dn_svh = sgn(E, 2, D), sgn(E, 2 * H), sgn(E, H), sgn(E, D)
    x = torch.from_numpy((rng.standard_normal((tokens, D)) * 0.25).astype(np.float16)).to(cuda)
    idx = np.stack([rng.permutation(E)[:top_k] for _ in range(tokens)]).astype(np.int32)
    if tokens > 1:
        idx[0, 0], idx[-1, -1] = -3, E + 5  # clamped to expert 0 and E - 1
    it = torch.from_numpy(idx).to(cuda)
    args = (x, it, gu, gu_suh, gu_svh, dn, dn_suh, dn_svh, k, cb, act)
    print(f"moe random seed={seed} D={D} H={H} k={k} cb={cb} E={E} top_k={top_k} tokens={tokens}", flush=True)
    y = ops.moe_forward(*args)
    y_rows = ops.moe_forward(*args, accumulators=False)
    y_five = ops.moe_forward(*args, fused=False)
    assert torch.equal(y, ops.moe_forward(*args))
    assert int(ops.sync_counters(cuda, 1).abs().sum()) == 0
    assert torch.isfinite(y.float()).all()
    ref = y_five.float().cpu().numpy()
    assert rel_l2(y.float().cpu().numpy(), ref) <= TOL
    assert rel_l2(y_rows.float().cpu().numpy(), ref) <= TOL


@pytest.mark.parametrize("tokens,act", [(40, "silu"), (200, "gelu")])
def test_prefill_path_matches_oracle_and_slot_kernels(cuda, oracle, tokens, act):
    """From 24 tokens on the pairs are sorted by expert and go through the segmented
    GEMM. Experts with no token, one token and many tokens occur; checked against
    the oracle chain and against the per-slot kernels on the same input."""
    from ponyexl3_amd import EXL3SwitchGLU, ops

    E, D, H, kk, k = 7, 256, 128, 2, 4
    gate, up, down = _experts(E, D, H, k, False, 800)
    moe = EXL3SwitchGLU.from_layers(gate, up, down, activation=act)
    rng = np.random.default_rng(80 + tokens)
    x = (rng.standard_normal((tokens, D)) * 0.5).astype(np.float16)
    # skewed routing: expert 5 never chosen, expert 6 exactly once, the rest unevenly
    p = np.array([0.45, 0.25, 0.15, 0.1, 0.05])
    idx = np.stack([rng.choice(5, size=kk, replace=False, p=p) for _ in range(tokens)]).astype(np.int32)
    idx[3, 1] = 6
    xt, it = torch.from_numpy(x).to(cuda), torch.from_numpy(idx).to(cuda)
    print(f"moe prefill tokens={tokens} act={act}", flush=True)
    y = moe(xt.reshape(1, tokens, D), it.reshape(1, tokens, kk))[0]
    assert tuple(y.shape) == (tokens, kk, D)
    ref = _oracle_chain(oracle, gate, up, down, x, idx, act)
    assert rel_l2(y.cpu().numpy(), ref) <= TOL
    slots = torch.cat([ops.moe_forward(xt[r:r + 8], it[r:r + 8], moe._gu_trellis, moe._gu_suh, moe._gu_svh,
                                       moe._dn_trellis, moe._dn_suh, moe._dn_svh, k, moe._cb,
                                       0 if act == "silu" else 1) for r in range(0, tokens, 8)])
    assert rel_l2(y.cpu().numpy(), slots.cpu().numpy()) <= TOL


@pytest.mark.parametrize("tokens,E,kk,D,H,K,cb,act,general", [
    (40, 300, 3, 640, 128, 3, 2, 0, False),    # down in four waves, 32 rows; a last block of 128 columns
    (590, 170, 8, 1152, 256, 6, 0, 1, True),   # both, 64 rows, blocks of one row and of 64; scales other than +-1
    (300, 32, 8, 1024, 768, 8, 1, 0, False),   # gate/up in four waves, down in eight
    (590, 170, 8, 640, 768, 4, 0, 0, False),   # both, with LDS for two of eight waves
])
def test_prefill_workgroups_of_four_waves(cuda, tokens, E, kk, D, H, K, cb, act, general):
    """The prefill kernels at as many row blocks as they take in workgroups of four waves, against the slot
    kernels on the same input (bar of the other prefill test)."""
    from ponyexl3_amd import _lib, ops

    lib = _lib.load()
    g = torch.Generator().manual_seed(tokens)
    bits = lambda *s: torch.randint(-32768, 32768, s, generator=g, dtype=torch.int16).to(cuda)
    def scale(size, *s):
        v = torch.randint(0, 2, s, generator=g) * 2.0 - 1.0
        return (v * size * (0.5 + torch.rand(s, generator=g) if general else 1)).half().to(cuda)
    gu, dn = bits(D // 16, 2 * E * H // 16, 16 * K), bits(H // 16, E * D // 16, 16 * K)
    gsu, gsv, dsu, dsv = scale(1, E, 2, D), scale(D**-0.5, E, 2, H), scale(1, E, H), scale(H**-0.5, E, D)
    x = (torch.randn((tokens, D), generator=g) * 0.5).half().to(cuda)
    # a few experts get most of the pairs, some one, some none
    weight = torch.rand((tokens, E), generator=g) * torch.linspace(0.3, 1, E)
    idx = weight.topk(kk, dim=1).indices.int().contiguous().to(cuda)
    y = torch.full((tokens, kk, D), float("nan"), dtype=torch.float16, device=cuda)
    need = lib.exl3_moe_prefill_workspace_bytes(tokens, kk, E, D, H)
    ws = torch.empty((need,), dtype=torch.uint8, device=cuda)
    p = ops._ptr
    print(f"prefill four waves tokens={tokens} E={E} D={D} H={H} K={K}", flush=True)
    _lib.check(lib.exl3_moe_prefill(p(x), tokens, p(idx), kk, p(gu), p(gsu), p(gsv), p(dn), p(dsu), p(dsv), E, D, H, K,
                                    cb, act, None, p(y), p(ws), need, ops._stream()), "exl3_moe_prefill")
    slots = torch.cat([ops.moe_forward(x[r:r + 8], idx[r:r + 8], gu, gsu, gsv, dn, dsu, dsv, K, cb, act)
                       for r in range(0, tokens, 8)])
    assert rel_l2(y.float().cpu().numpy(), slots.float().cpu().numpy()) <= TOL


def test_moe_equals_linear_modules(cuda):
    """The stacked chain equals the same experts run as individual EXL3Linear
    modules (fused-vs-unfused, ponyexl3/tests/test_moe_activation.py:44-65)."""
    from ponyexl3_amd import EXL3Linear, EXL3SwitchGLU

    E, D, H, kk = 4, 512, 256, 3
    gate, up, down = _experts(E, D, H, 4, False, 900)
    moe = EXL3SwitchGLU.from_layers(gate, up, down)
    g = torch.Generator().manual_seed(1)
    x = (torch.randn((2, D), generator=g) * 0.5).to(torch.float16).to(cuda)
    idx = torch.tensor([[0, 2, 3], [1, 0, 2]], dtype=torch.int32, device=cuda)
    y = moe(x.reshape(1, 2, D), idx.reshape(1, 2, kk))[0]
    for t in range(2):
        for s in range(kk):
            e = int(idx[t, s])
            gv = EXL3Linear(gate[e])(x[t : t + 1]).float()
            uv = EXL3Linear(up[e])(x[t : t + 1]).float()
            h = (torch.nn.functional.silu(gv) * uv).to(torch.float16)
            ref = EXL3Linear(down[e])(h).float()
            got = y[t, s].float()
            assert float((got - ref[0]).abs().max() / (ref.abs().max() + 1e-9)) < 5e-3


def test_bounded_wait_gives_up_visibly(cuda, monkeypatch):
    """A counters array that is not zero on entry breaks the accumulator reduction of
    gate/up: the finishing workgroup's wait for complete counts is bounded (lowered here
    through EXL3_SPIN_LIMIT so that it runs out at once), every kernel still exits, the
    slot's output is NaN, the other slots are untouched and the status word is set."""
    from ponyexl3_amd import EXL3SwitchGLU, ops

    if os.environ.get("EXL3_EXACT_WEIGHTS") == "1":
        pytest.skip("the multi-launch chains this knob selects have no accumulator reduction")
    E, D, H, kk, k = 4, 640, 256, 2, 4
    gate, up, down = _experts(E, D, H, k, False, 900)
    moe = EXL3SwitchGLU.from_layers(gate, up, down)
    rng = np.random.default_rng(9)
    xt = torch.from_numpy((rng.standard_normal((1, D)) * 0.5).astype(np.float16)).to(cuda)
    it = torch.tensor([[2, 1]], dtype=torch.int32, device=cuda)
    args = (xt, it, moe._gu_trellis, moe._gu_suh, moe._gu_svh, moe._dn_trellis, moe._dn_suh, moe._dn_svh,
            k, moe._cb)
    good = ops.moe_forward(*args, fused=True)
    ops.check_counters(cuda)
    cnt = ops.sync_counters(cuda, 1)
    try:
        # accumulator of (slot 0, gate, column 5): a count of 255 that can never come out right
        cnt.view(torch.int64)[5] = -(1 << 56)
        monkeypatch.setenv("EXL3_SPIN_LIMIT", "4")
        print("moe bounded wait", flush=True)
        bad = ops.moe_forward(*args, fused=True)
        torch.cuda.synchronize()
        assert torch.isnan(bad[0, 0].float()).all()
        assert torch.equal(bad[0, 1], good[0, 1])
        with pytest.raises(RuntimeError):
            ops.check_counters(cuda)
        monkeypatch.delenv("EXL3_SPIN_LIMIT")
        assert torch.equal(ops.moe_forward(*args, fused=True), good)  # check_counters zeroed the array
        ops.check_counters(cuda)
    finally:
        torch.cuda.synchronize()
        cnt.zero_()  # whatever happened above, the shared array is clean for the next test


def test_config4_a3b_shapes(cuda, oracle):
    """hidden 2048, 256 experts of 2048->512 / 512->2048, top-8 routing from a
    softmax over seeded router logits, at 1 and 8 tokens. Every (token, expert) slot
    is checked against the oracle's unfused expert chain
    (ponyexl3/mlx/exl3_moe.py:648-682) at rel-L2 <= 1e-3, two slots also against
    per-expert EXL3Linear chains, and the slot order against permutation
    equivariance."""
    from ponyexl3_amd import EXL3Layer, EXL3Linear, EXL3SwitchGLU, ops
    from ponyexl3_amd.moe import combine_experts, route_topk

    E, D, H, kk, k = 256, 2048, 512, 8, 4
    rng = np.random.default_rng(40_004)
    gu = rng.integers(0, 65536, size=(D // 16, E * 2 * H // 16, 16 * k), dtype=np.uint16)
    dn = rng.integers(0, 65536, size=(H // 16, E * D // 16, 16 * k), dtype=np.uint16)
    sgn = lambda shape: np.where(rng.random(shape) > 0.5, -1.0, 1.0).astype(np.float16)
    gu_suh, gu_svh, dn_suh, dn_svh = sgn((E, 2, D)), sgn((E, 2 * H)), sgn((E, H)), sgn((E, D))
    dev = lambda a: torch.from_numpy(a).to(cuda)
    moe = EXL3SwitchGLU(gu_trellis=ops.as_trellis_tensor(gu, cuda), gu_suh=dev(gu_suh), gu_svh=dev(gu_svh),
                        dn_trellis=ops.as_trellis_tensor(dn, cuda), dn_suh=dev(dn_suh), dn_svh=dev(dn_svh),
                        k=k, cb=0)
    for T in (1, 8):
        x = (rng.standard_normal((T, D)) * 0.25).astype(np.float16)
        logits = torch.from_numpy(rng.standard_normal((T, E)).astype(np.float32)).to(cuda)
        inds, scores = route_topk(logits, kk)
        assert torch.allclose(scores.sum(-1), torch.ones(T, device=cuda), atol=1e-5)
        xt = dev(x)
        print(f"config4 T={T}", flush=True)
        y = moe(xt.reshape(1, T, D), inds.reshape(1, T, kk))
        assert tuple(y.shape) == (1, T, kk, D)
        out = combine_experts(y, scores.reshape(1, T, kk))
        assert tuple(out.shape) == (1, T, D) and torch.isfinite(out.float()).all()
        # slot-order permutation equivariance
        perm = torch.randperm(kk, generator=torch.Generator().manual_seed(T)).to(cuda)
        y2 = moe(xt.reshape(1, T, D), inds[:, perm].reshape(1, T, kk))
        assert torch.equal(y2, y[:, :, perm])
        # all T * 8 slots against the oracle's chain over the selected experts
        gt = H // 16
        cut = lambda a: np.ascontiguousarray(a)
        experts = {}
        for e in sorted(set(int(v) for v in inds.cpu().numpy().ravel())):
            experts[e] = {
                "gate": (cut(gu[:, e * gt : (e + 1) * gt]), gu_suh[e, 0], gu_svh[e, :H]),
                "up": (cut(gu[:, (E + e) * gt : (E + e + 1) * gt]), gu_suh[e, 1], gu_svh[e, H:]),
                "down": (cut(dn[:, e * (D // 16) : (e + 1) * (D // 16)]), dn_suh[e], dn_svh[e]),
            }
        ref_all = oracle.moe_experts_forward(experts, x, inds.cpu().numpy(), k, 0)
        got_all = y[0].cpu().numpy()
        worst = max(float(np.linalg.norm(got_all[t, s].astype(np.float64) - ref_all[t, s].astype(np.float64))
                          / np.linalg.norm(ref_all[t, s].astype(np.float64)))
                    for t in range(T) for s in range(kk))
        print(f"config4 T={T}: worst slot rel-L2 vs oracle {worst:.2e}", flush=True)
        assert worst <= 1e-3
        # two sampled slots against stand-alone layers cut out of the stacks
        for (t, s) in [(0, 0), (T - 1, kk - 1)]:
            e = int(inds[t, s])
            mk = lambda tr, suh, svh, n_in, n_out: EXL3Linear(
                EXL3Layer(f"e{e}", n_in, n_out, k, np.ascontiguousarray(tr), suh, svh))
            gl = mk(gu[:, e * gt : (e + 1) * gt], gu_suh[e, 0], gu_svh[e, :H], D, H)
            ul = mk(gu[:, (E + e) * gt : (E + e + 1) * gt], gu_suh[e, 1], gu_svh[e, H:], D, H)
            dl = mk(dn[:, e * (D // 16) : (e + 1) * (D // 16)], dn_suh[e], dn_svh[e], H, D)
            h = (torch.nn.functional.silu(gl(xt[t : t + 1]).float()) * ul(xt[t : t + 1]).float()).to(torch.float16)
            ref = dl(h).float()[0]
            got = y[0, t, s].float()
            assert float((got - ref).norm() / ref.norm()) <= 5e-3


def test_errors(cuda):
    from ponyexl3_amd import EXL3SwitchGLU

    z = lambda *s: torch.zeros(s, dtype=torch.float16, device=cuda)
    zi = lambda *s: torch.zeros(s, dtype=torch.int16, device=cuda)
    with pytest.raises(ValueError):
        EXL3SwitchGLU(gu_trellis=zi(8, 16, 64), gu_suh=z(1, 2, 128), gu_svh=z(1, 256), dn_trellis=zi(8, 8, 64),
                      dn_suh=z(1, 128), dn_svh=z(1, 128), k=4, cb=0, activation="relu")
    with pytest.raises(ValueError):
        EXL3SwitchGLU(gu_trellis=zi(8, 8, 64), gu_suh=z(1, 2, 128), gu_svh=z(1, 256), dn_trellis=zi(8, 8, 64),
                      dn_suh=z(1, 128), dn_svh=z(1, 128), k=4, cb=0)


def test_moe_block_with_shared_expert(cuda, oracle):
    """Router (softmax, top-k, renormalise), the shared expert stacked last with a
    sigmoid gate, weighted sum: against the same composition over the oracle chain
    (ponyexl3/mlx/exl3_moe.py:790-839)."""
    from ponyexl3_amd import EXL3MoEBlock, EXL3SwitchGLU

    E, D, H, kk = 5, 256, 128, 2  # 4 routed experts + the shared one
    gate, up, down = _experts(E, D, H, 4, True, 950)
    switch = EXL3SwitchGLU.from_layers(gate, up, down)
    g = torch.Generator().manual_seed(2)
    router = torch.nn.Linear(D, E - 1, bias=False)
    shared_gate = torch.nn.Linear(D, 1, bias=False)
    with torch.no_grad():
        router.weight.copy_(torch.randn((E - 1, D), generator=g) * 0.2)
        shared_gate.weight.copy_(torch.randn((1, D), generator=g) * 0.2)
    block = EXL3MoEBlock(router.half().to(cuda), shared_gate.half().to(cuda), switch, kk).to(cuda)
    x = (torch.randn((3, D), generator=g) * 0.5).to(torch.float16)
    with torch.no_grad():
        y = block(x.to(cuda)).float().cpu().numpy()
        inds, scores = block.route(x.to(cuda).reshape(1, 3, D))
    assert y.shape == (3, D)
    inds, scores = inds[0].cpu().numpy(), scores[0].float().cpu().numpy()
    assert inds.shape == (3, kk + 1) and (inds[:, -1] == E - 1).all() and (inds[:, :kk] < E - 1).all()
    np.testing.assert_allclose(scores[:, :kk].sum(axis=1), 1.0, atol=2e-3)
    per_expert = _oracle_chain(oracle, gate, up, down, x.numpy(), inds.astype(np.int32), "silu")
    ref = (per_expert.astype(np.float32) * scores[..., None]).sum(axis=1)
    assert rel_l2(y, ref) <= 2 * TOL  # fp16 products and sum over three experts on top of the chain


@pytest.mark.parametrize("tokens,top_k,E,block_rows", [(40, 2, 7, 64), (513, 8, 256, 64), (3000, 4, 1024, 64),
                                                        (2100, 8, 16, 256), (1, 1, 1, 64)])
def test_pair_sort_kernel_equals_stable_argsort(cuda, tokens, top_k, E, block_rows):
    """Integer work, bit-exact: order / tok / sidx against torch's stable argsort, the
    row-block table against the table built from device-side torch ops (same worst-case
    length, same empty entries). Includes out-of-range ids (clamped), experts with no
    pair and more pairs than one 1024-pair scatter round."""
    from ponyexl3_amd import ops

    rng = np.random.default_rng(tokens + E)
    idx = rng.integers(0, E, size=(tokens, top_k)).astype(np.int32)
    if E > 4:
        idx[idx == 3] = 2  # expert 3 gets nothing
        idx[0, 0] = E + 5  # clamps to E - 1
        if tokens > 1:
            idx[1, 0] = -4  # clamps to 0
    it = torch.from_numpy(idx).to(cuda)
    order, tok, sidx, table = ops.moe_sort(it, E, block_rows)
    flat = it.reshape(-1).long().clamp(0, E - 1)
    ref_order = torch.argsort(flat, stable=True)
    assert torch.equal(order.long(), ref_order)
    assert torch.equal(sidx.long(), flat[ref_order])
    assert torch.equal(tok.long(), ref_order // top_k)
    ref_table = ops.segment_table(flat[ref_order], E, block_rows)
    assert tuple(table.shape) == tuple(ref_table.shape)
    assert torch.equal(table, ref_table)
    o2, t2, s2, tab2 = ops.moe_sort(it, E, block_rows)  # same answer every call
    assert torch.equal(o2, order) and torch.equal(tab2, table)


@pytest.mark.parametrize("tokens,kk,E", [(1, 1, 1), (9, 7, 3), (16, 4, 65), (65, 1, 1024), (512, 2, 7), (205, 5, 600),
                                         (683, 3, 64), (4100, 8, 257), (4097, 8, 1024)])
def test_prefill_sorts_as_the_sort_kernel(cuda, tokens, kk, E):
    """The prefill chain sorts in the launch that rotates, 256 threads to a workgroup and one per 1024 pairs: order and
    row-block table, at the front of its workspace, are those of the sort by itself (whole numbers, equal), clamped ids and
    experts without pairs included."""
    from ponyexl3_amd import _lib, ops

    lib, p = _lib.load(), ops._ptr
    D, H, K, n = 128, 128, 2, tokens * kk
    rng = np.random.default_rng(n + E)
    idx = rng.integers(0, E, size=(tokens, kk)).astype(np.int32)
    if E > 4:
        idx[idx == 3] = 2
        idx[0, 0] = E + 5
        idx[-1, -1] = -4
    idx = torch.from_numpy(idx).to(cuda)
    bits = lambda *s: torch.randint(-32768, 32768, s, dtype=torch.int16, device=cuda)
    ones = lambda *s: torch.ones(s, dtype=torch.float16, device=cuda)
    x = torch.randn((tokens, D), device=cuda).half() * 0.1
    need = lib.exl3_moe_prefill_workspace_bytes(tokens, kk, E, D, H)
    ws = torch.full((need,), 0xCC, dtype=torch.uint8, device=cuda)
    y = torch.empty((tokens, kk, D), dtype=torch.float16, device=cuda)
    w = [bits(D // 16, 2 * E * H // 16, 16 * K), ones(E, 2, D), ones(E, 2, H), bits(H // 16, E * D // 16, 16 * K), ones(E, H),
         ones(E, D)]
    print(f"prefill sort tokens={tokens} kk={kk} E={E}", flush=True)
    _lib.check(lib.exl3_moe_prefill(p(x), tokens, p(idx), kk, *map(p, w), E, D, H, K, 0, 0, None, p(y), p(ws), need,
                                    ops._stream()), "exl3_moe_prefill")
    block_rows = 32 if n <= 24 * E else 64
    order, _, _, table = ops.moe_sort(idx, E, block_rows)
    assert torch.equal(ws[:4 * n].view(torch.int32), order)
    at = (4 * n + 255) // 256 * 256
    assert torch.equal(ws[at:at + 16 * table.shape[0]].view(torch.int32).view(-1, 4), table.view(-1, 4))


@pytest.mark.parametrize("tokens", [16400, 32767, 32800])
def test_prefill_past_31_and_32_bit_offsets(cuda, tokens):
    """Rotated rows are gathered at 32-bit byte offsets, the last ones past 2^31 (16400 tokens) and up to the last row that
    such an offset reaches (32767); from 4 GiB on (32800) they are put in sorted order, behind a sort of its own, instead. The
    last tokens' rows are those of a call on them alone, up to the order of the sums (the row blocks differ)."""
    from ponyexl3_amd import _lib, ops

    if torch.cuda.mem_get_info()[0] < 40 << 30:
        pytest.skip("needs 40 GB of memory")
    lib, p = _lib.load(), ops._ptr
    kk, E, D, H, K = 4, 8, 16384, 128, 2
    assert tokens * kk * D * 2 > 1 << 31 and (tokens * kk * D * 2 > 0xFFFFFFFF) == (tokens > 32767)
    g = torch.Generator(device=cuda).manual_seed(5)
    bits = lambda *s: torch.randint(-32768, 32768, s, dtype=torch.int16, device=cuda, generator=g)
    sign = lambda size, *s: ((torch.randint(0, 2, s, device=cuda, generator=g) * 2.0 - 1.0) * size).half()
    w = [bits(D // 16, 2 * E * H // 16, 16 * K), sign(1, E, 2, D), sign(D**-0.5, E, 2, H), bits(H // 16, E * D // 16, 16 * K),
         sign(1, E, H), sign(H**-0.5, E, D)]
    x = torch.randn((tokens, D), device=cuda, generator=g, dtype=torch.float16) * 0.5
    idx = torch.rand((tokens, E), device=cuda, generator=g).topk(kk, dim=1).indices.int().contiguous()

    def run(xs, ids):
        t = xs.shape[0]
        need = lib.exl3_moe_prefill_workspace_bytes(t, kk, E, D, H)
        ws = torch.empty((need,), dtype=torch.uint8, device=cuda)
        y = torch.full((t, kk, D), float("nan"), dtype=torch.float16, device=cuda)
        _lib.check(lib.exl3_moe_prefill(p(xs), t, p(ids), kk, *map(p, w), E, D, H, K, 0, 0, None, p(y), p(ws), need,
                                        ops._stream()), "exl3_moe_prefill")
        return y

    print(f"prefill past 31-bit offsets tokens={tokens}", flush=True)
    got = run(x, idx)
    for part in (slice(0, 100), slice(tokens - 100, tokens)):
        ref = run(x[part].contiguous(), idx[part].contiguous())
        assert rel_l2(got[part].float().cpu().numpy(), ref.float().cpu().numpy()) <= TOL
    assert bool(torch.isfinite(got).all())


@pytest.mark.parametrize("tokens,k", [(40, 4), (200, 8)])  # row blocks of 32 and of 64
@pytest.mark.parametrize("kind", ["general", "spikes", "small"])
def test_prefill_rotation_with_general_scales(cuda, tokens, k, kind):
    """The gate/up kernel of the prefill chain rotates the GLU's output for the down projection;
    scales that are not +-1 need fp32 products: past the fp16 range (a spike of 1.5e4 per block)
    they are finite, small ones keep all bits. Its result, the last part of the workspace,
    against the separate launches, fp16 roundings of the same values up to the order of the
    sums in gate and up; the experts with plain signs in between keep theirs."""
    from ponyexl3_amd import EXL3SwitchGLU, _lib, ops

    E, D, H, kk = 7, 256, 384, 2
    moe = EXL3SwitchGLU.from_layers(*_experts(E, D, H, k, True, 5100))
    rng = np.random.default_rng(tokens)
    sign = lambda *s: np.where(rng.random(s) > 0.5, -1.0, 1.0)
    dn_suh = sign(E, H) * (rng.uniform(0.5, 2, (E, H)) if kind != "spikes" else 1.0)
    if kind == "spikes":
        dn_suh[:, ::128] *= 1.5e4
    elif kind == "small":
        dn_suh *= 1e-3
    dn_suh[E // 2] = sign(H)
    moe._dn_suh = torch.from_numpy(dn_suh.astype(np.float16)).to(cuda)
    moe._gu_suh = torch.from_numpy((sign(E, 2, D) * rng.uniform(0.5, 2, (E, 2, D))).astype(np.float16)).to(cuda)
    x = torch.from_numpy((rng.standard_normal((tokens, D)) * 0.05).astype(np.float16)).to(cuda)
    idx = torch.from_numpy(np.stack([rng.permutation(E)[:kk] for _ in range(tokens)]).astype(np.int32)).to(cuda)
    lib, n = _lib.load(), tokens * kk
    total = lib.exl3_moe_prefill_workspace_bytes(tokens, kk, E, D, H)
    ws = torch.zeros((total,), dtype=torch.uint8, device=cuda)
    y = torch.empty((tokens, kk, D), dtype=torch.float16, device=cuda)
    p = ops._ptr
    print(f"prefill rotation tokens={tokens} k={k} {kind}", flush=True)
    _lib.check(lib.exl3_moe_prefill(p(x), tokens, p(idx), kk, p(moe._gu_trellis), p(moe._gu_suh), p(moe._gu_svh),
                                    p(moe._dn_trellis), p(moe._dn_suh), p(moe._dn_svh), E, D, H, k, moe._cb, 0, None,
                                    p(y), p(ws), total, ops._stream()), "exl3_moe_prefill")
    got = ws[total - (n * H * 2 + 255) // 256 * 256:][:n * H * 2].view(torch.float16).view(n, H)
    order, tok, sidx, table = ops.moe_sort(idx, E, 64)
    xg = ops.had128_rows(x, moe._gu_suh[:, 0], False, in_index=tok, scale_index=sidx)
    xu = ops.had128_rows(x, moe._gu_suh[:, 1], False, in_index=tok, scale_index=sidx)
    g = ops.gemm_grouped(xg, moe._gu_trellis, k, moe._cb, 0, H // 16, E, table, 64)
    u = ops.gemm_grouped(xu, moe._gu_trellis, k, moe._cb, E * H // 16, H // 16, E, table, 64)
    ref = ops.moe_glu_rows(g, u, sidx, moe._gu_svh, moe._dn_suh, 0)
    assert bool(torch.isfinite(ref).all()) and bool(torch.isfinite(got).all())
    if kind == "spikes":
        assert float(ref.abs().max()) * 128 ** 0.5 > 65504  # products past the fp16 range did occur
    assert rel_l2(got.float().cpu().numpy(), ref.float().cpu().numpy()) <= TOL


@pytest.mark.parametrize("tokens,D", [(257, 2048), (251, 2176)])
def test_large_prefill_equals_its_halves(cuda, tokens, D):
    """Rotations of 8 MB of pair rows and more take another way to memory; each token's rows are those
    of a call on half the tokens, up to the order of the sums (the row blocks may differ)."""
    from ponyexl3_amd import EXL3SwitchGLU, _lib, ops

    E, H, kk, k = 7, 128, 4, 4
    moe = EXL3SwitchGLU.from_layers(*_experts(E, D, H, k, True, 5200))
    rng = np.random.default_rng(tokens)
    scale = moe._gu_suh.clone()
    scale[E // 2, 1, 128:256] *= 1.5  # a block with general scales
    x = torch.from_numpy((rng.standard_normal((tokens, D)) * 0.05).astype(np.float16)).to(cuda)
    idx = torch.from_numpy(np.stack([rng.permutation(E)[:kk] for _ in range(tokens)]).astype(np.int32)).to(cuda)
    lib, p = _lib.load(), ops._ptr
    assert tokens * kk * D * 4 >= 8 << 20

    def run(xs, ids):
        t = xs.shape[0]
        total = lib.exl3_moe_prefill_workspace_bytes(t, kk, E, D, H)
        ws = torch.empty((total,), dtype=torch.uint8, device=cuda)
        y = torch.empty((t, kk, D), dtype=torch.float16, device=cuda)
        _lib.check(lib.exl3_moe_prefill(p(xs), t, p(ids), kk, p(moe._gu_trellis), p(scale), p(moe._gu_svh),
                                        p(moe._dn_trellis), p(moe._dn_suh), p(moe._dn_svh), E, D, H, k, moe._cb, 0, None,
                                        p(y), p(ws), total, ops._stream()), "exl3_moe_prefill")
        return y

    print(f"large prefill tokens={tokens} D={D}", flush=True)
    got, half = run(x, idx), tokens // 2
    ref = torch.cat([run(x[:half].contiguous(), idx[:half].contiguous()), run(x[half:].contiguous(), idx[half:].contiguous())])
    for a, b in ((got[:half], ref[:half]), (got[half:], ref[half:])):
        assert rel_l2(a.float().cpu().numpy(), b.float().cpu().numpy()) <= TOL


@pytest.mark.parametrize("act", [0, 1])
def test_glu_rows_kernel_equals_separate_launches(cuda, act):
    """Finish gate/up + GLU + down rotation in one launch against the per-row
    Hadamard launches around torch's GLU (same casts: fp16 after every stage)."""
    from ponyexl3_amd import ops

    rng = np.random.default_rng(17 + act)
    N, H, E = 300, 384, 9
    g = torch.from_numpy((rng.standard_normal((N, H)) * 2).astype(np.float16)).to(cuda)
    u = torch.from_numpy((rng.standard_normal((N, H)) * 2).astype(np.float16)).to(cuda)
    sidx = torch.from_numpy(np.sort(rng.integers(0, E, size=N)).astype(np.int32)).to(cuda)
    sgn = lambda *s: torch.from_numpy(np.where(rng.random(s) > 0.5, -1, 1).astype(np.float16)).to(cuda)
    gu_svh, dn_suh = sgn(E, 2 * H), sgn(E, H)
    got = ops.moe_glu_rows(g, u, sidx, gu_svh, dn_suh, act)
    gf = ops.had128_rows(g, gu_svh[:, :H], True, scale_index=sidx).float()
    uf = ops.had128_rows(u, gu_svh[:, H:], True, scale_index=sidx).float()
    a = torch.nn.functional.gelu(gf, approximate="tanh") if act else torch.nn.functional.silu(gf)
    ref = ops.had128_rows((a * uf).to(torch.float16), dn_suh, False, scale_index=sidx)
    diff = (got.float() - ref.float()).abs().max()
    # expf / tanhf of the kernel vs torch's: an fp16 ulp of h here and there
    assert float(diff) <= 4e-3 * float(ref.float().abs().max())
    with pytest.raises(ValueError):
        ops.moe_glu_rows(g, u[:, :256], sidx, gu_svh, dn_suh, act)


def test_silu_over_the_range_of_halfs(cuda):
    """SiLU where its power over- and underflows: gate values from 2^-12 to the fp16 limit and past it (infinite),
    both signs, against float64. A block's rotation spreads an infinite or undefined value over the whole block; the
    others are within two fp16 roundings (of h and of the result, 2^-11 each) of the largest h times sqrt(128)."""
    from ponyexl3_amd import ops

    rng = np.random.default_rng(23)
    N, H, E = 192, 512, 5
    g = torch.from_numpy(rng.standard_normal((N, H)).astype(np.float16)).to(cuda)
    u = torch.from_numpy(rng.standard_normal((N, H)).astype(np.float16)).to(cuda)
    sidx = torch.from_numpy(np.sort(rng.integers(0, E, size=N)).astype(np.int32)).to(cuda)
    gu_svh = torch.ones((E, 2 * H), dtype=torch.float16)
    size = 2.0 ** rng.uniform(-12, 15, (E, H // 128, 128))
    size[:, 2:] = 2.0 ** rng.uniform(-3, 8, (E, H // 128 - 2, 128))  # (nothing infinite there)
    gu_svh[:, :H] = torch.from_numpy(size.reshape(E, H).astype(np.float16))
    gu_svh[:, H:] = 2.0 ** -9
    gu_svh, dn_suh = gu_svh.to(cuda), torch.ones((E, H), dtype=torch.float16, device=cuda)
    got = ops.moe_glu_rows(g, u, sidx, gu_svh, dn_suh, 0).double().cpu().view(N, -1, 128)
    gf = ops.had128_rows(g, gu_svh[:, :H], True, scale_index=sidx).double().cpu()
    uf = ops.had128_rows(u, gu_svh[:, H:], True, scale_index=sidx).double().cpu()
    h = (gf / (1 + torch.exp(-gf)) * uf).view(N, -1, 128)
    ref = ops.had128_rows(h.view(N, H).to(torch.float16).to(cuda), dn_suh, False, scale_index=sidx).double().cpu().view(N, -1, 128)
    ok = torch.isfinite(h).all(-1)
    assert (~ok).any() and ok[:, 2:].all() and float(gf[torch.isfinite(gf)].abs().max()) > 4e4
    assert torch.equal(torch.isfinite(got).all(-1), ok) and not torch.isfinite(got[~ok]).any()
    bound = 2 * 2.0 ** -11 * 128 ** 0.5 * h.abs().amax(-1, keepdim=True)
    assert ((got - ref).abs() <= bound)[ok].all()


@pytest.mark.parametrize("tokens,E,top_k,norm,fp32", [(1, 1, 1, True, False), (5, 63, 8, True, False),
                                                      (3, 64, 64, False, True), (130, 65, 4, True, True),
                                                      (7, 257, 6, False, False), (4, 1024, 16, True, False)])
@pytest.mark.parametrize("shared", [False, True])
def test_route_kernel_against_torch(cuda, tokens, E, top_k, norm, fp32, shared):
    """Softmax, top-k (ties: lowest expert first) and weights against torch in float64,
    on coarse logits so that ties do occur, also at the k-th place."""
    from ponyexl3_amd import _lib, ops

    g = torch.Generator().manual_seed(E + top_k)
    logits = (torch.randn((tokens, E), generator=g) * 4).round() / 4
    sl = torch.randn((tokens, 1), generator=g)
    dt = torch.float32 if fp32 else torch.float16
    ld, sd = logits.to(dt).to(cuda), sl.to(dt).to(cuda)
    slots = top_k + shared
    idx = torch.full((tokens, slots), -1, dtype=torch.int32, device=cuda)
    scores = torch.zeros((tokens, slots), dtype=torch.float16, device=cuda)
    print(f"route tokens={tokens} E={E} k={top_k}", flush=True)
    rc = _lib.load().exl3_moe_route(ops._ptr(ld), int(fp32), ops._ptr(sd) if shared else None, tokens, E, top_k,
                                    int(norm), ops._ptr(idx), ops._ptr(scores), ops._stream())
    _lib.check(rc, "exl3_moe_route")
    order = torch.argsort(-logits, dim=-1, stable=True)[:, :top_k]
    w = torch.gather(torch.softmax(logits.double(), dim=-1), 1, order)
    if norm:
        w = w / w.sum(dim=-1, keepdim=True)
    assert torch.equal(idx[:, :top_k].cpu().long(), order)
    torch.testing.assert_close(scores[:, :top_k].cpu().double(), w, rtol=1e-3, atol=1e-6)
    if shared:
        assert (idx[:, top_k] == E).all()
        torch.testing.assert_close(scores[:, top_k].cpu().double(), torch.sigmoid(sd.cpu().double())[:, 0],
                                   rtol=1e-3, atol=1e-6)


@pytest.mark.parametrize("tokens,E,top_k,D", [(1, 4, 4, 8), (5, 64, 2, 128), (33, 129, 8, 520), (70, 256, 8, 2048),
                                              (9, 600, 64, 2056)])
def test_route_kernel_with_the_shared_gate(cuda, tokens, E, top_k, D):
    """exl3_moe_route_shared: the table of exl3_moe_route, and behind it sigmoid(fp16(x . w)). The logit's error
    is that of an fp32 sum of D terms, in any order, and of its fp16 rounding; the sigmoid's slope is at most
    1/4; expf and the quotient add a few units of 2^-23, the fp16 result half of 2^-10."""
    from ponyexl3_amd import _lib, ops

    g = torch.Generator().manual_seed(tokens + E)
    logits = torch.randn((tokens, E), generator=g).half().to(cuda)
    x, w = torch.randn((tokens, D), generator=g).half(), (torch.randn((D,), generator=g) * D**-0.5).half()
    xd, wd = x.to(cuda), w.to(cuda)
    idx = torch.full((tokens, top_k + 1), -1, dtype=torch.int32, device=cuda)
    scores = torch.zeros((tokens, top_k + 1), dtype=torch.float16, device=cuda)
    want_idx, want = torch.empty_like(idx[:, :top_k]).contiguous(), torch.empty_like(scores[:, :top_k]).contiguous()
    lib = _lib.load()
    print(f"route shared tokens={tokens} E={E} top_k={top_k} D={D}", flush=True)
    _lib.check(lib.exl3_moe_route_shared(ops._ptr(logits), ops._ptr(xd), D, ops._ptr(wd), tokens, E, top_k, 1,
                                         ops._ptr(idx), ops._ptr(scores), ops._stream()), "exl3_moe_route_shared")
    _lib.check(lib.exl3_moe_route(ops._ptr(logits), 0, None, tokens, E, top_k, 1, ops._ptr(want_idx), ops._ptr(want),
                                  ops._stream()), "exl3_moe_route")
    assert torch.equal(idx[:, :top_k], want_idx) and torch.equal(scores[:, :top_k], want)
    assert bool((idx[:, top_k] == E).all())
    xw = x.double() * w.double()
    exact, spread = xw.sum(-1), xw.abs().sum(-1)
    bound = 0.25 * (D * 2.0**-24 * spread + 2.0**-11 * exact.abs() + 2.0**-25) + 2.0**-11 + 2.0**-21
    assert bool(((scores[:, top_k].cpu().double() - torch.sigmoid(exact)).abs() <= bound).all())
    assert lib.exl3_moe_route_shared(ops._ptr(logits), ctypes.c_void_p(xd.data_ptr() + 2), D, ops._ptr(wd), tokens, E, top_k, 1,
                                     ops._ptr(idx), ops._ptr(scores), ops._stream()) == _lib.EXL3_E_BAD_SHAPE


@pytest.mark.parametrize("tokens,shared", [(1, False), (9, True), (30, True), (67, False)])
def test_moe_block_native_chain_equals_its_parts(cuda, tokens, shared):
    """Slot kernels, slot kernels with shared passes and the sorted prefill chain with the
    weighted sum in its last kernel: the block against route, experts and sum one by one."""
    from ponyexl3_amd import EXL3MoEBlock, EXL3SwitchGLU
    from ponyexl3_amd.moe import combine_experts

    E, D, H, kk = 9, 384, 128, 3
    gate, up, down = _experts(E, D, H, 4, True, 4200)
    switch = EXL3SwitchGLU.from_layers(gate, up, down)
    g = torch.Generator().manual_seed(tokens)
    lin = lambda n: torch.nn.Linear(D, n, bias=False).half().to(cuda).requires_grad_(False)
    block = EXL3MoEBlock(lin(E - shared), lin(1) if shared else None, switch, kk)
    x = (torch.randn((1, tokens, D), generator=g) * 0.2).half().to(cuda)
    print(f"moe block tokens={tokens}", flush=True)
    y = block(x)
    inds, scores = block.route(x)
    ref = combine_experts(switch(x, inds).float(), scores)
    assert y.shape == x.shape and y.dtype == torch.float16
    assert rel_l2(y.float().cpu().numpy(), ref.cpu().numpy()) <= TOL


@pytest.mark.parametrize("tokens,E,kk,prefill", [(33, 30, 2, False), (120, 40, 1, False), (40, 6, 4, True)])
def test_shared_gate_is_computed_here_for_many_tokens(cuda, monkeypatch, tokens, E, kk, prefill):
    """Past the tokens of the router's kernel the router's product is its module's; the shared gate's single column is not, on
    the slot kernels either: one linear product is called, and the result is that of the parts."""
    from ponyexl3_amd import EXL3MoEBlock, EXL3SwitchGLU
    from ponyexl3_amd.moe import combine_experts

    D, H = 256, 128
    switch = EXL3SwitchGLU.from_layers(*_experts(E + 1, D, H, 4, True, 4600))
    assert switch._use_prefill(tokens, kk + 1) == prefill
    lin = lambda n: torch.nn.Linear(D, n, bias=False).half().to(cuda).requires_grad_(False)
    block = EXL3MoEBlock(lin(E), lin(1), switch, kk)
    x = torch.randn((1, tokens, D), generator=torch.Generator().manual_seed(tokens)).half().to(cuda)
    linear, widths = torch.nn.functional.linear, []
    monkeypatch.setattr(torch.nn.functional, "linear", lambda a, w, *r: (widths.append(w.shape[0]), linear(a, w, *r))[1])
    print(f"shared gate tokens={tokens}", flush=True)
    y = block(x)
    assert widths == [E]
    inds, scores = block.route(x)
    ref = combine_experts(switch(x, inds).float(), scores)
    assert rel_l2(y.float().cpu().numpy(), ref.cpu().numpy()) <= TOL


def test_slot_kernels_take_more_tokens_than_a_gate_grid(cuda):
    """One token more than a launch of the gate's kernel holds, kept off the prefill by a line that the caller moved: the
    shared gate's column goes through its module and every token has the result of a small call."""
    from ponyexl3_amd import EXL3MoEBlock, EXL3SwitchGLU

    D, tokens = 128, 16 * 65535 + 1
    switch = EXL3SwitchGLU.from_layers(*_experts(2, D, 128, 4, True, 4650))
    switch.prefill_min_tokens = 1 << 30
    lin = lambda n: torch.nn.Linear(D, n, bias=False).half().to(cuda).requires_grad_(False)
    block = EXL3MoEBlock(lin(1), lin(1), switch, 1)
    base = torch.randn((1021, D), generator=torch.Generator().manual_seed(4)).half().to(cuda)
    print(f"slot kernels tokens={tokens}", flush=True)
    ref = block(base).float()
    y = block(base.repeat(-(-tokens // 1021), 1)[:tokens])
    for part in y.split(1021):
        want = ref[: len(part)]
        assert (part.float() - want).norm() <= TOL * want.norm()


@pytest.mark.parametrize("tokens", [2, 67])
def test_moe_block_reaches_replaced_parts(cuda, tokens):
    """A router replaced on the instance and hooks on all modules see the call, and the result
    is that of the parts."""
    from ponyexl3_amd import EXL3MoEBlock, EXL3SwitchGLU

    E, D, H, kk = 5, 256, 128, 2
    switch = EXL3SwitchGLU.from_layers(*_experts(E, D, H, 4, True, 4400))
    lin = torch.nn.Linear(D, E, bias=False).half().to(cuda).requires_grad_(False)
    block = EXL3MoEBlock(lin, None, switch, kk)
    x = (torch.randn((1, tokens, D), generator=torch.Generator().manual_seed(tokens)) * 0.2).half().to(cuda)
    y = block(x)
    seen = []
    handle = torch.nn.modules.module.register_module_forward_hook(lambda m, i, o: seen.append(type(m).__name__))
    try:
        y2 = block(x)
    finally:
        handle.remove()
    assert seen == ["Linear", "EXL3SwitchGLU", "EXL3MoEBlock"]
    assert rel_l2(y2.float().cpu().numpy(), y.float().cpu().numpy()) <= TOL
    last = torch.tensor([E - 1, E - 2], dtype=torch.int32, device=cuda)
    block.route = lambda x3: (last.expand(1, tokens, kk).contiguous(),
                              torch.full((1, tokens, kk), 0.5, dtype=torch.float16, device=cuda))
    y3 = block(x)
    ref = switch(x, last.expand(1, tokens, kk).contiguous()).float().mean(dim=-2)
    assert rel_l2(y3.float().cpu().numpy(), ref.cpu().numpy()) <= TOL


@pytest.mark.parametrize("tokens", [2, 67])
def test_moe_block_with_callables_for_modules(cuda, tokens):
    """Gates, the shared expert's included, and the experts may be any callables."""
    from ponyexl3_amd import EXL3MoEBlock, EXL3SwitchGLU

    E, D, H, kk = 5, 256, 128, 2
    switch = EXL3SwitchGLU.from_layers(*_experts(E, D, H, 4, True, 4800))
    lin = lambda n: torch.nn.Linear(D, n, bias=False).half().to(cuda).requires_grad_(False)
    gate, shared = lin(E - 1), lin(1)
    x = (torch.randn((1, tokens, D), generator=torch.Generator().manual_seed(tokens)) * 0.2).half().to(cuda)
    ref = EXL3MoEBlock(gate, shared, switch, kk)(x).float().cpu().numpy()
    call = lambda m: lambda *a: m(*a)
    for g, s in ((gate, call(shared)), (call(gate), shared), (call(gate), call(shared))):
        assert rel_l2(EXL3MoEBlock(g, s, switch, kk)(x).float().cpu().numpy(), ref) <= TOL
    block = EXL3MoEBlock(gate, shared, switch, kk)
    del block.switch_mlp
    block.switch_mlp = call(switch)
    assert rel_l2(block(x).float().cpu().numpy(), ref) <= TOL


@pytest.mark.parametrize("tokens", [2, 67])
def test_moe_block_takes_any_alignment(cuda, tokens):
    """x, or a scale vector of the stack, as a contiguous view off the 16-byte grid: the gate's
    product goes through the module and the experts through the slot kernels."""
    from ponyexl3_amd import EXL3MoEBlock, EXL3SwitchGLU

    E, D, H, kk = 5, 256, 128, 2
    stack = _experts(E, D, H, 4, True, 4600)
    lin = torch.nn.Linear(D, E, bias=False).half().to(cuda).requires_grad_(False)
    block = EXL3MoEBlock(lin, None, EXL3SwitchGLU.from_layers(*stack), kk)
    x = (torch.randn((1, tokens, D), generator=torch.Generator().manual_seed(tokens)) * 0.2).half().to(cuda)
    ref = block(x).float().cpu().numpy()

    def shifted(t):
        s = torch.empty(t.numel() + 2, dtype=t.dtype, device=t.device)[2:].view(t.shape).copy_(t)
        assert s.is_contiguous() and s.data_ptr() % 16
        return s

    print(f"block off the grid tokens={tokens}", flush=True)
    assert rel_l2(block(shifted(x)).float().cpu().numpy(), ref) <= TOL
    for name in ("_gu_svh", "_dn_suh"):
        other = EXL3SwitchGLU.from_layers(*stack)
        setattr(other, name, shifted(getattr(other, name)))
        assert rel_l2(EXL3MoEBlock(lin, None, other, kk)(x).float().cpu().numpy(), ref) <= TOL


def test_prefill_keeps_no_memory(cuda):
    """The sorted chain's rotated rows are gone when the call's result is: chunks of growing and
    shrinking size leave what is allocated as it was, as do the experts called alone."""
    from ponyexl3_amd import EXL3MoEBlock, EXL3SwitchGLU

    E, D, H, kk = 5, 512, 128, 4
    switch = EXL3SwitchGLU.from_layers(*_experts(E, D, H, 4, True, 4700))
    lin = torch.nn.Linear(D, E, bias=False).half().to(cuda).requires_grad_(False)
    block = EXL3MoEBlock(lin, None, switch, kk)
    x = torch.randn((1, 1500, D), generator=torch.Generator().manual_seed(1)).half().to(cuda)
    first = block(x[:, :30])  # router, scratch and library handles of this stream exist
    del first
    held = torch.cuda.memory_allocated()
    for tokens in (200, 700, 1500, 400):
        assert switch._use_prefill(tokens, kk)
        print(f"prefill memory tokens={tokens}", flush=True)
        y = block(x[:, :tokens])
        inds, scores = block.route(x[:, :tokens])
        z = switch(x[:, :tokens], inds)
        del y, z, inds, scores
        assert torch.cuda.memory_allocated() == held


@pytest.mark.parametrize("name", ["_gu_suh", "_gu_svh", "_dn_suh", "_dn_svh", "_gu_trellis"])
def test_stack_of_another_type_is_refused(cuda, name):
    """Before any launch: the kernels read fp16 scales and 16-bit words at these addresses."""
    from ponyexl3_amd import EXL3SwitchGLU

    switch = EXL3SwitchGLU.from_layers(*_experts(2, 128, 128, 4, True, 4900))
    setattr(switch, name, getattr(switch, name).float())
    with pytest.raises(ValueError):
        switch(torch.zeros((1, 1, 128), dtype=torch.float16, device=cuda),
               torch.zeros((1, 1, 1), dtype=torch.int32, device=cuda))


def test_moe_block_under_autocast_and_with_tangents(cuda):
    """The router's product, softmax and sum are torch's where something watches or changes
    torch operations: bf16 logits and an fp32 sum under autocast, a tangent through the weights
    of the sum in forward mode, a subclass of x that reaches the gate."""
    from ponyexl3_amd import EXL3MoEBlock, EXL3SwitchGLU

    E, D, H, kk, tokens = 5, 256, 128, 2, 3
    switch = EXL3SwitchGLU.from_layers(*_experts(E, D, H, 4, True, 4500))
    lin = torch.nn.Linear(D, E, bias=False).half().to(cuda).requires_grad_(False)
    block = EXL3MoEBlock(lin, None, switch, kk)
    x = (torch.randn((1, tokens, D), generator=torch.Generator().manual_seed(8)) * 0.2).half().to(cuda)

    def parts():
        inds, scores = block.route(x)
        return (switch(x, inds) * scores[..., None]).sum(dim=-2)

    with torch.autocast("cuda", dtype=torch.bfloat16):
        assert torch.equal(block(x), parts()) and block(x).dtype == parts().dtype == torch.float32
    with torch.autograd.forward_ad.dual_level():
        out = block(torch.autograd.forward_ad.make_dual(x, torch.ones_like(x)))
        assert torch.autograd.forward_ad.unpack_dual(out).tangent is not None

    class Sub(torch.Tensor):
        seen = []

        @classmethod
        def __torch_function__(cls, func, types, args=(), kwargs=None):
            Sub.seen.append(func)
            return super().__torch_function__(func, types, args, kwargs or {})

    block(x.as_subclass(Sub))
    assert torch.nn.functional.linear in Sub.seen


@pytest.mark.parametrize("tokens,E,D", [(1, 1, 128), (1, 256, 2048), (3, 15, 384), (16, 16, 1152), (17, 257, 640),
                                        (32, 33, 2176)])
@pytest.mark.parametrize("shared", [False, True])
def test_gate_kernel_against_float64(cuda, tokens, E, D, shared):
    """Router logits and the shared gate's: fp16 roundings of the exact products, up to
    the fp32 sums."""
    from ponyexl3_amd import _lib, ops

    g = torch.Generator().manual_seed(D + E)
    x = torch.randn((tokens, D), generator=g).half()
    w = (torch.randn((E + 1, D), generator=g) / D ** 0.5).half()
    xd, wd = x.to(cuda), w.to(cuda)
    logits = torch.full((tokens, E), float("nan"), dtype=torch.float16, device=cuda)
    sl = torch.full((tokens,), float("nan"), dtype=torch.float16, device=cuda)
    print(f"gate tokens={tokens} E={E} D={D}", flush=True)
    rc = _lib.load().exl3_moe_gate(ops._ptr(xd), tokens, D, ops._ptr(wd), E, ops._ptr(wd[E]) if shared else None,
                                   ops._ptr(logits), ops._ptr(sl) if shared else None, ops._stream())
    _lib.check(rc, "exl3_moe_gate")
    ref = x.double() @ w.double().T
    torch.testing.assert_close(logits.cpu().double(), ref[:, :E], rtol=6e-4, atol=1e-5)
    if shared:
        torch.testing.assert_close(sl.cpu().double(), ref[:, E], rtol=6e-4, atol=1e-5)


@pytest.mark.parametrize("tokens,E,D,H,top_k", [(1, 1, 128, 128, 1), (1, 8, 256, 768, 8), (2, 64, 1152, 256, 5),
                                                (3, 255, 2048, 512, 8), (5, 256, 640, 640, 7), (4, 300, 384, 256, 6),
                                                (40, 16, 256, 384, 4), (9, 32, 256, 128, 4)])
@pytest.mark.parametrize("shared", [False, True])
def test_decode_call_equals_its_parts(cuda, tokens, E, D, H, top_k, shared):
    _decode_call_and_parts(cuda, tokens, E, D, H, top_k, shared, 4)


# around the line between single and grouped slots, where that one expert of the table is a shared one (which only the one call
# knows) must not choose the kernels: accumulators against partial rows, and from K = 5 on half blocks against whole ones
@pytest.mark.parametrize("tokens,E,D,H,top_k,k", [(8, 64, 1024, 256, 6, 4), (8, 128, 640, 256, 8, 6), (10, 256, 1024, 256, 8, 6),
                                                  (11, 256, 1024, 256, 8, 4), (12, 256, 1024, 256, 8, 6), (14, 256, 1024, 256, 8, 4),
                                                  (13, 256, 1152, 512, 8, 8), (11, 256, 2048, 512, 8, 4)])
def test_decode_call_equals_its_parts_beside_the_grouping_line(cuda, tokens, E, D, H, top_k, k):
    _decode_call_and_parts(cuda, tokens, E, D, H, top_k, True, k)


def _decode_call_and_parts(cuda, tokens, E, D, H, top_k, shared, k):
    """exl3_moe_decode against exl3_moe_route, exl3_moe_forward and exl3_moe_combine, bit for bit, in every form
    of the slot kernels (accumulators with the routing inside, more experts than it ranks there, grouped slots,
    several partial rows of down), on coarse logits so that ties occur; twice, so that the counters
    are shown to come back to zero."""
    from ponyexl3_amd import _lib, ops

    lib = _lib.load()
    g = torch.Generator(device=cuda).manual_seed(E + D + tokens)
    rnd = lambda *s: torch.randn(s, device=cuda, generator=g)
    n = E + shared
    cb = E % 2
    tr = lambda a, b: torch.randint(-32768, 32768, (a // 16, b // 16, 16 * k), dtype=torch.int16, device=cuda, generator=g)
    gu, dn = tr(D, n * 2 * H), tr(H, n * D)
    gu_suh, gu_svh = rnd(n, 2, D).sign().half(), (rnd(n, 2 * H).sign() / D ** 0.5).half()
    dn_suh, dn_svh = rnd(n, H).sign().half(), (rnd(n, D).sign() / H ** 0.5).half()
    x = rnd(tokens, D).half()
    logits, sl = ((rnd(tokens, E) * 4).round() / 4).half(), rnd(tokens).half()
    kk = top_k + shared
    weights = [ops._ptr(t) for t in (gu, gu_suh, gu_svh, dn, dn_suh, dn_svh)]
    idx, scores = torch.zeros((tokens, kk), dtype=torch.int32, device=cuda), torch.zeros((tokens, kk), device=cuda).half()
    rows, out = torch.zeros((tokens, kk, D), device=cuda).half(), torch.zeros((tokens, D), device=cuda).half()
    ws = torch.zeros(lib.exl3_moe_workspace_bytes(tokens, kk, D, H), dtype=torch.uint8, device=cuda)
    n_cnt = lib.exl3_moe_decode_counters(tokens, kk, D, H)
    cnt = torch.zeros(n_cnt, dtype=torch.int32, device=cuda)
    sp = ops._ptr(sl) if shared else None
    print(f"moe decode tokens={tokens} E={E} D={D} H={H} top_k={top_k} shared={shared}", flush=True)
    _lib.check(lib.exl3_moe_route(ops._ptr(logits), 0, sp, tokens, E, top_k, 1, ops._ptr(idx), ops._ptr(scores),
                                  ops._stream()), "route")
    _lib.check(lib.exl3_moe_forward(ops._ptr(x), tokens, ops._ptr(idx), kk, *weights, n, D, H, k, cb, 0, ops._ptr(rows),
                                    ops._ptr(ws), ws.numel(), ops._ptr(cnt), n_cnt, ops._stream()), "forward")
    _lib.check(lib.exl3_moe_combine(ops._ptr(rows), ops._ptr(scores), tokens, kk, D, ops._ptr(out), ops._stream()),
               "combine")
    want = [t.clone() for t in (idx, scores, rows, out)]
    for _ in range(2):
        for t in (idx, scores, rows, out):
            t.fill_(-1)
        rc = lib.exl3_moe_decode(ops._ptr(x), tokens, ops._ptr(logits), sp, E, top_k, 1, *weights, n, D, H, k, cb, 0,
                                 ops._ptr(idx), ops._ptr(scores), ops._ptr(rows), ops._ptr(out), ops._ptr(ws),
                                 ws.numel(), ops._ptr(cnt), n_cnt, ops._stream())
        _lib.check(rc, "decode")
        for got, ref in zip((idx, scores, rows, out), want):
            assert torch.equal(got, ref)
        assert int(cnt.abs().sum()) == 0
    assert not torch.isnan(out.float()).any()
    assert lib.exl3_moe_decode(ops._ptr(x), tokens, ops._ptr(logits), sp, E, top_k, 1, *weights, n, D, H, k, cb, 0,
                               ops._ptr(idx), ops._ptr(scores), ops._ptr(rows), ops._ptr(out), ops._ptr(ws),
                               ws.numel(), ops._ptr(cnt), n_cnt - 1, ops._stream()) != 0


@pytest.mark.parametrize("pairs,E", [(2048, 9), (2049, 1), (2049, 257), (3073, 1024), (32768, 3), (32769, 300),
                                     (65600, 64)])
def test_pair_sort_in_several_parts(cuda, pairs, E):
    """Sizes at which the sort changes from one workgroup to several, with a last one that holds one pair, and
    from one round of 64 pairs per wave to two."""
    test_pair_sort_kernel_equals_stable_argsort(cuda, pairs, 1, E, 64)
