"""GPU tests at the edges of single kernel paths, against the CPU oracle (bit for bit)."""

import pytest
import torch

import cabi
import cases
from nanoep_amd import Buffer, EPConfig
from oracle import nanoep_oracle as oracle
from test_gpu_buffer_api import assert_dispatch_result, assert_same_bits
from test_gpu_cabi_parity import run_dispatch_combine

pytestmark = pytest.mark.gpu


# The prefetch workgroups of the slot-order walk also touch their segment's list lines and weights: list
# shares that start inside a line, windows cut short by the batch's end, lists far shorter than their
# segments (most choices masked), more lines than prefetch wavefronts (short rows, 32 choices).
@pytest.mark.parametrize(
    "tokens,hidden,experts,topk,kind",
    [(257, 256, 9, 3, "dropout"), (1025, 512, 16, 5, "sparse"), (4097, 256, 40, 32, "dropout"), (65, 7168, 256, 8, "masked"),
     (2049, 2816, 3, 1, "sparse")],
)
def test_list_and_weight_lines_of_ragged_windows(device, tokens, hidden, experts, topk, kind):
    run_dispatch_combine(device, cases.routing(kind, tokens, experts, topk, seed=tokens), hidden, experts, 1, True, True, True)
