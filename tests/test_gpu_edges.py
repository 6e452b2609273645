"""GPU tests at the edges of single kernel paths, against the CPU oracle (bit for bit)."""

import pytest
import torch

import cabi
import cases
from nanoep_amd import Buffer, EPConfig
from oracle import nanoep_oracle as oracle
from test_gpu_buffer_api import assert_dispatch_result, assert_same_bits
from test_gpu_cabi_parity import assert_layout, run_dispatch_combine

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


# The layout's three plans (1: every workgroup counts the batch, 2: histogram rows summed by every
# workgroup, 3: histogram rows scanned by one) at the edges of its blocks, rows and wavefront chunks: batches one
# token around a block, choices whose chunks leave lanes idle, experts around a strip of 64 and beyond the
# threads of a workgroup, histogram rows of several blocks (short rows, long batches).
@pytest.mark.parametrize("launches", [1, 2, 3])
@pytest.mark.parametrize(
    "tokens,experts,topk,hidden,alignment",
    [(1, 2, 2, 256, 1), (31, 63, 5, 1024, 4), (32, 64, 8, 1024, 1), (33, 65, 10, 1024, 16), (64, 3, 1, 7168, 1), (65, 256, 8, 7168, 128),
     (127, 40, 32, 512, 1), (129, 33, 17, 2048, 2), (257, 1030, 6, 4096, 8), (513, 8, 3, 512, 3), (700, 3839, 4, 512, 1),
     (9000, 300, 7, 256, 1), (16385, 17, 8, 512, 128)],
)
def test_layout_plans_at_their_edges(device, tuning, launches, tokens, experts, topk, hidden, alignment):
    tuning("LAYOUT_LAUNCHES", launches)
    idx = cases.routing("dropout", tokens, experts, topk, seed=tokens + topk)
    for expand in (True, False):
        metadata, counts = cabi.layout(idx.to(device), experts, alignment, expand, hidden=hidden)
        assert_layout(metadata, counts, oracle.layout(idx, experts, alignment), expand, hidden)


# One bad token anywhere in the batch is found by every plan: an id in another half of its 64 bits, a
# duplicate in the token's first and last choice, in the first and last block.
@pytest.mark.parametrize("launches", [1, 2, 3])
@pytest.mark.parametrize("token", [0, 127, 128, 771])
@pytest.mark.parametrize("bad,status", [(-2, 1), (24, 1), ((1 << 32) + 3, 1), (None, 2)])
def test_every_layout_plan_reports_bad_routing(device, tuning, launches, token, bad, status):
    tuning("LAYOUT_LAUNCHES", launches)
    idx = cases.routing("random", 772, 24, 5, seed=9)
    idx[token, 4] = idx[token, 0] if bad is None else bad
    _, counts = cabi.layout(idx.to(device), 24, 1, True, raise_on_routing=False)
    assert counts[3] == status
