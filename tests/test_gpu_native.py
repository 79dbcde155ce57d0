"""Folded fp16 engine (public weight through the prefill kernels) against the
oracle's public-weight reconstruction and the exact EXL3 module."""
import numpy as np
import pytest
import torch

from conftest import rel_l2

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("k,mcg,mul1,n_in,n_out", [(4, False, False, 256, 384), (3, True, False, 384, 256),
                                                   (6, False, True, 128, 640)])
def test_public_weight_matches_oracle(cuda, oracle, k, mcg, mul1, n_in, n_out):
    """W_pub from identity activations vs diag(suh).H.W.H.diag(svh) in fp32
    (ponyexl3/ref/reconstruct.py:26-49). The prefill path rounds to fp16 after the
    input transform and after the GEMM, hence a tolerance, not equality."""
    from ponyexl3_amd import make_exl3_layer, native

    layer = make_exl3_layer(k=k, in_features=n_in, out_features=n_out, seed=500 + k, mcg=mcg, mul1=mul1)
    cb = int(layer.codebook_mode)
    ref = oracle.reconstruct_public_weights(layer.trellis, layer.suh, layer.svh, k, cb)
    w = native.public_weight(layer, device=cuda)
    assert w.dtype == torch.float16 and tuple(w.shape) == (n_in, n_out)
    assert rel_l2(w.cpu().numpy(), ref) < 1e-3
    # chunked = whole: stripes of 128 columns are independent
    parts = list(native.public_weight_chunks(layer, chunk_cols=128, device=cuda))
    assert len(parts) == n_out // 128
    assert torch.equal(torch.cat(parts, dim=1), w)
    with pytest.raises(ValueError):
        list(native.public_weight_chunks(layer, chunk_cols=100, device=cuda))


def test_public_weight_equals_identity_through_the_module(cuda):
    """The fold is the module applied to the identity. Both round the same fp32 sums to
    fp16; the module's prefill path adds the 128 terms of the output Hadamard on the
    matrix pipe, the fold in butterfly order, so a result that sits on a rounding boundary
    can come out one fp16 step apart."""
    from ponyexl3_amd import EXL3Linear, make_exl3_layer, native

    layer = make_exl3_layer(k=4, in_features=256, out_features=256, seed=9)
    eye = torch.eye(256, dtype=torch.float16, device=cuda)
    fold, module = native.public_weight(layer, device=cuda).float(), EXL3Linear(layer)(eye).float()
    step = torch.maximum(fold.abs(), module.abs()) * 2.0 ** -10 + 2.0 ** -24  # one fp16 step at that size
    assert bool(((fold - module).abs() <= step).all())
    assert float((fold != module).float().mean()) < 0.01


@pytest.mark.parametrize("k,cb,n_in,n_out", [(1, 0, 128, 128), (2, 1, 384, 1152), (5, 2, 128, 256),
                                             (7, 0, 640, 128), (8, 1, 256, 384)])
def test_public_weight_slices_and_transpose(cuda, oracle, k, cb, n_in, n_out):
    """One block, one block row, one block column, general scale vectors and none:
    against the oracle; a slice and the transposed form hold the same bits."""
    from ponyexl3_amd import ops

    rng = np.random.default_rng(40 + k)
    tr = rng.integers(0, 65536, size=(n_in // 16, n_out // 16, 16 * k), dtype=np.uint16)
    suh = (rng.standard_normal(n_in) * 0.7).astype(np.float16)
    svh = (rng.standard_normal(n_out) * 0.02).astype(np.float16)
    trt, s, v = ops.as_trellis_tensor(tr, cuda), torch.from_numpy(suh).to(cuda), torch.from_numpy(svh).to(cuda)
    print(f"public weight k={k} cb={cb} {n_in}x{n_out}", flush=True)
    w = ops.public_weight(trt, k, cb, s, v)
    assert rel_l2(w.cpu().numpy(), oracle.reconstruct_public_weights(tr, suh, svh, k, cb)) < 1e-3
    assert torch.equal(ops.public_weight(trt, k, cb, s, v, transposed=True), w.T)
    last = ops.public_weight(trt, k, cb, s, v[-128:].contiguous(), tn_offset=n_out // 16 - 8)
    assert torch.equal(last, w[:, -128:])
    one_in, one_out = np.ones(n_in, np.float16), np.ones(n_out, np.float16)
    plain = ops.public_weight(trt, k, cb)
    assert rel_l2(plain.cpu().numpy(), oracle.reconstruct_public_weights(tr, one_in, one_out, k, cb)) < 1e-3


@pytest.mark.parametrize("cb", [0, 1, 2])
@pytest.mark.parametrize("k", range(1, 9))
def test_public_weight_against_decoded_weights(cuda, k, cb):
    """One block, and more blocks than start together (each asks for the words of one 1024 places on): the
    bit-exact decoded weights under both transforms in 64 bits, with the two fp16 casts. A sum of 128 in fp32 is off by
    up to 2^-20, which moves fewer than one cast in a hundred by a step of 2^-11: 2^-14 of the norm; 2^-13 asked."""
    from ponyexl3_amd import ops

    g = torch.Generator(device=cuda).manual_seed(8 * cb + k)
    i = torch.arange(128, device=cuda)
    parity = (i[:, None] & i[None, :]).cpu().apply_(lambda v: bin(v).count("1") & 1).to(cuda)
    had = (1 - 2 * parity).double()
    for n_in, n_out in ((128, 128), (384, 128 * 345)):
        print(f"public weight k={k} cb={cb} {n_in}x{n_out}", flush=True)
        tr = torch.randint(-32768, 32768, (n_in // 16, n_out // 16, 16 * k), dtype=torch.int16, device=cuda, generator=g)
        suh = torch.randn(n_in, device=cuda, generator=g).half()
        svh = (0.02 * torch.randn(n_out, device=cuda, generator=g)).half()
        w = ops.decode_full(tr, k, cb).double().view(n_in // 128, 128, n_out // 128, 128).transpose(1, 2)
        q = (suh.float() * 0.08838834764831845).half().double().view(n_in // 128, 1, 128, 1)
        y = (q * had.matmul(w)).half().double()
        z = (y.matmul(had) * 0.08838834764831845 * svh.double().view(1, n_out // 128, 1, 128)).half()
        ref = z.transpose(1, 2).reshape(n_in, n_out).double()
        for transposed in (False, True):
            got = ops.public_weight(tr, k, cb, suh, svh, transposed=transposed).double()
            got = got.T if transposed else got
            assert float((got - ref).norm() / ref.norm()) < 2.0 ** -13


@pytest.mark.parametrize("bias", [False, True])
def test_folded_linear_tracks_exact_layer(cuda, oracle, bias):
    from ponyexl3_amd import make_exl3_layer, native

    layer = make_exl3_layer(k=4, in_features=512, out_features=384, seed=31, mcg=True, bias=bias)
    lin = native.folded_linear_from_exl3(layer, device=cuda)
    assert isinstance(lin, torch.nn.Linear) and lin.weight.dtype == torch.float16
    assert tuple(lin.weight.shape) == (384, 512) and (lin.bias is not None) == bias
    rng = np.random.default_rng(3)
    x = rng.standard_normal((5, 512)).astype(np.float16)
    y = lin(torch.from_numpy(x).to(cuda)).cpu().numpy()
    ref = oracle.linear_forward(layer.trellis, 4, int(layer.codebook_mode), layer.suh, layer.svh, x,
                                bias=layer.bias)
    assert rel_l2(y, ref) < 2e-3


@pytest.mark.parametrize("bias", [False, True])
def test_folded_linear_is_a_whole_module(cuda, bias):
    """The fold builds its Linear without Linear.__init__: the same attributes, parameters and state as a
    module built the usual way, usable and copyable like one."""
    import copy

    from ponyexl3_amd import make_exl3_layer, native

    layer = make_exl3_layer(k=4, in_features=256, out_features=128, seed=5, bias=bias)
    lin = native.folded_linear_from_exl3(layer, device=cuda)
    ref = torch.nn.Linear(256, 128, bias=bias, device=cuda, dtype=torch.float16)
    assert type(lin) is torch.nn.Linear and set(lin.__dict__) == set(ref.__dict__) and repr(lin) == repr(ref)
    assert [n for n, _ in lin.named_parameters()] == [n for n, _ in ref.named_parameters()]
    ref.load_state_dict(lin.state_dict())
    x = torch.randn((3, 256), device=cuda).half()
    assert torch.equal(lin(x), ref(x)) and torch.equal(copy.deepcopy(lin)(x), ref(x))
    assert not any(p.requires_grad for p in lin.parameters())


def test_public_weight_argument_errors(cuda):
    from ponyexl3_amd import make_exl3_layer, ops

    layer = make_exl3_layer(k=4, in_features=128, out_features=256, seed=6)
    tr = ops.as_trellis_tensor(layer.trellis, cuda)
    suh, svh = torch.from_numpy(layer.suh).to(cuda), torch.from_numpy(layer.svh).to(cuda)
    bad = [(tr, 9, 0), (tr, 3, 0), (tr.view(-1), 4, 0), (tr.cpu(), 4, 0), (tr.int(), 4, 0), ("x", 4, 0), (tr, 4, 7)]
    for args in bad:
        with pytest.raises(ValueError):
            ops.public_weight(*args)
    for kw in ({"suh": suh[:64]}, {"svh": suh}, {"suh": suh.float()}, {"svh": svh.cpu()}, {"tn_offset": -1},
               {"tn_offset": 17}, {"tn_count": -1}, {"tn_count": 4}, {"tn_offset": 8, "tn_count": 16}, {"suh": [1.0]}):
        with pytest.raises(ValueError):
            ops.public_weight(tr, 4, 0, **kw)
    assert ops.public_weight(tr, 4, 0, tn_offset=16).shape == (128, 0)
