"""Which MoE calls go to the prefill chain and which to the slot kernels (no GPU needed)."""
import os
import subprocess
import sys

import pytest

from conftest import ROOT

_CODE = """
import sys
sys.path.insert(0, sys.argv[1])
import torch
from ponyexl3_amd import EXL3SwitchGLU
m = EXL3SwitchGLU.__new__(EXL3SwitchGLU)
torch.nn.Module.__init__(m)
m.input_dims, m.hidden_dims = 1024, 256
for name, value in eval(sys.argv[2]).items():
    setattr(EXL3SwitchGLU, name, value)
for tokens, top_k, m.num_experts in ((23, 8, 8), (24, 4, 32), (32, 4, 32), (24, 5, 48), (60, 1, 24), (200, 2, 64), (129, 4, 100), (128, 4, 100), (30, 2, 40)):
    print(int(m._use_prefill(tokens, top_k)))
"""


# per call: fewer tokens than the prefill's; 3, 4 and 2.5 rows an expert; top-1; 6.25; 516 and 512 slots; 1.5 rows an expert
@pytest.mark.parametrize("env,attributes,want", [
    ({}, {}, "0 0 0 0 0 1 1 0 0"),
    # calls of the prefill's sizes reach the slot kernels only where those round the down weights as it does
    ({"EXL3_MOE_GROUP": "0"}, {}, "0 1 1 1 1 1 1 1 0"),
    ({"EXL3_EXACT_WEIGHTS": "1"}, {}, "0 1 1 1 1 1 1 1 0"),
    ({}, {"prefill_min_tokens": 16}, "1 0 0 0 0 1 1 0 0"),
    ({}, {"prefill_min_rows_per_expert": 1.0, "prefill_min_tokens": 20}, "1 0 0 0 0 1 1 0 1"),
    ({}, {"prefill_min_rows_per_expert": 1000.0}, "0 0 0 0 0 0 1 0 0"),
    ({}, {"grouped_max_slots": 100}, "0 0 1 1 0 1 1 1 0"),
    ({}, {"grouped_max_slots": 1024}, "0 0 0 0 0 1 0 0 0"),
])
def test_route_of_moe_calls(env, attributes, want):
    run = subprocess.run([sys.executable, "-c", _CODE, ROOT, repr(attributes)], env=dict(os.environ, **env), capture_output=True,
                         text=True, check=True, timeout=120)
    assert run.stdout.split() == want.split()
