"""Folded fp16 engine: the public weight of an EXL3 layer as a plain
``torch.nn.Linear`` (``fold16``).

The EXL3 forward is linear in x, so both Hadamard transforms and both sign/scale
vectors fold into ``W_pub = diag(suh) . H . W_inner . H . diag(svh)``. The reference
(``ponyexl3/mlx/native.py:49-85``) pushes an fp16 identity through its prefill
forward, so that the folded weight carries exactly the runtime's cast points; here
one kernel decodes the trellis and applies both transforms block by block with the
same cast points (``exl3_public_weight``).

Only the fold itself is provided: it is the fp16 materialisation of the decode path.
The reference's lossy engines around it (w8a16 / w4a16 re-quantization with MLX's
affine group quantizer, the fused SwiGLU module and the per-layer error report,
``native.py:88-264``) are alternative engines, not part of the EXL3 path.
"""

from __future__ import annotations

import torch

from . import ops
from .layer import EXL3Layer
from .linear import layer_runtime

# One stripe of output columns at a time (multiple of 128), native.py:45.
PUBLIC_CHUNK_COLS = 8192


def public_weight_chunks(layer: EXL3Layer, *, chunk_cols: int = PUBLIC_CHUNK_COLS, device="cuda"):
    """Yield ``W_pub[:, n0:n1]`` fp16 chunks with all transforms folded in
    (``public_weight_chunks``, ponyexl3/mlx/native.py:49-70)."""
    if chunk_cols % 128 != 0:
        raise ValueError("chunk_cols must be a multiple of 128")
    rt = layer_runtime(layer, device)
    n_out = layer.out_features
    for n0 in range(0, n_out, chunk_cols):
        n = min(chunk_cols, n_out - n0)
        svh = None if rt.svh is None else rt.svh[n0:n0 + n].contiguous()
        yield ops.public_weight(rt.trellis, rt.k, rt.cb, rt.suh, svh, n0 // 16, n // 16)


def public_weight(layer: EXL3Layer, *, device="cuda") -> torch.Tensor:
    """Full ``(in, out)`` fp16 public weight (``public_weight_mlx``, native.py:73-75)."""
    rt = layer_runtime(layer, device)
    return ops.public_weight(rt.trellis, rt.k, rt.cb, rt.suh, rt.svh)


def folded_linear_from_exl3(layer: EXL3Layer, *, device="cuda") -> torch.nn.Linear:
    """Exact fold: ``torch.nn.Linear`` holding the fp16 public weight, no
    requantization (``folded_linear_from_exl3``, native.py:78-85)."""
    rt = layer_runtime(layer, device)
    # Linear.__init__ without its default initialisation, which costs 22 us of host time (35 with a bias)
    # even on the meta device, where the fold of a small layer takes 5-10 us. 512 x 512: 44 -> 11 us per call.
    lin = torch.nn.Linear.__new__(torch.nn.Linear)
    torch.nn.Module.__init__(lin)
    lin.in_features, lin.out_features = layer.in_features, layer.out_features
    weight = ops.public_weight(rt.trellis, rt.k, rt.cb, rt.suh, rt.svh, transposed=True)
    lin.register_parameter("weight", torch.nn.Parameter(weight, requires_grad=False))
    lin.register_parameter("bias", None if layer.bias is None else
                           torch.nn.Parameter(rt.bias.clone(), requires_grad=False))
    return lin
