"""Large batches, bit-exact to the oracle (needs an MI355X).

From 512 tokens the down launch adds a slot's first eight 32-channel tiles into
one partial. The widths and budgets give slots on both sides of that (none, one
tile, eight, more), skewed routing and padded rows slots outside the tiles, and
hidden sizes outputs past a wave's 256.
"""

import pytest
import torch

from calibration_free_moe.reader.budget import compile_budget
from tests.synthetic import make_layer
from tests.test_gpu_parity import assert_parity, build, run_both

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("tokens", [511, 512, 600])
@pytest.mark.parametrize("hidden,width,top_k,rank,retention", [
    (256, 512, 2, 16, 0.6), (384, 320, 3, 0, 0.5), (256, 64, 4, 32, 0.1), (1152, 288, 2, 32, 1.0),
])
def test_large_batches_bit_exact(tokens, hidden, width, top_k, rank, retention):
    layer = make_layer(hidden=hidden, width=width, experts=6, top_k=top_k, rank=max(rank, 8),
                       tokens=tokens, seed=400 + hidden + width, zipf=1.2)
    plan = compile_budget(hidden_size=hidden, expert_width=width, top_k=top_k, retention=retention,
                          screen_keep=1.0 if retention == 1.0 else 0.625)
    layer.weights[::7, 0] = 40.0  # slots that keep almost everything beside slots that keep nothing
    if rank == 0:
        layer.encoder, layer.decoder = None, None
    padding = torch.zeros(tokens, dtype=torch.bool)
    padding[3::50] = True
    reader = build_any(layer, plan, tokens)
    out, expected = run_both(reader, layer, plan, layer.hidden, layer.ids, layer.weights, padding)
    assert_parity(reader, out, expected, tokens, screened=retention < 1.0)


def build_any(layer, plan, tokens):
    if layer.encoder is not None:
        return build(layer, plan, tokens, selection_score="point")
    from calibration_free_moe.reader.progressive import ProgressiveReader, channel_major_down
    from tests.test_gpu_parity import DEVICE

    return ProgressiveReader(layer.gate_up.to(DEVICE), channel_major_down(layer.down.to(DEVICE)), None, None,
                             plan, tokens, sketch=(layer.codes.to(DEVICE), layer.statistics.to(DEVICE)),
                             selection_score="point")
