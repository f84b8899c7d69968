"""Large batches, bit-exact to the oracle (needs an MI355X).

From 512 tokens the down launch adds a slot's first eight 32-channel tiles into
one partial. The widths and budgets give slots on both sides of that (none, one
tile, eight, more), skewed routing and padded rows slots outside the tiles, and
hidden sizes outputs past a wave's 256.

The output launch of partials that the staged kernel cannot hold (more than 512
(slot, rank) pairs) is output_kernel while its workgroups run in one round, then
output_stream_kernel: token counts on both sides of each.
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


@pytest.mark.parametrize("hidden,top_k,rank,tokens", [
    (2048, 24, 32, 24), (2048, 24, 32, 32), (2048, 24, 32, 33), (1024, 33, 16, 63), (1024, 33, 16, 64),
    (1024, 33, 16, 65), (512, 20, 32, 64), (512, 20, 32, 128), (512, 20, 32, 129), (128, 40, 64, 17),
    (4096, 9, 64, 48), (4096, 9, 64, 49), (4096, 9, 64, 64),
])
def test_unstaged_outputs_bit_exact(hidden, top_k, rank, tokens):
    layer = make_layer(hidden=hidden, width=48, experts=top_k + 2, top_k=top_k, rank=rank, tokens=tokens,
                       seed=500 + hidden + tokens)
    layer.weights[::5, 0] = 30.0
    plan = compile_budget(hidden_size=hidden, expert_width=48, top_k=top_k, retention=0.3, screen_keep=0.625)
    padding = torch.zeros(tokens, dtype=torch.bool)
    padding[3::20] = True
    reader = build_any(layer, plan, tokens)
    out, expected = run_both(reader, layer, plan, layer.hidden, layer.ids, layer.weights, padding)
    assert_parity(reader, out, expected, tokens)


@pytest.mark.parametrize("width,experts,top_k", [(512, 32, 24), (1024, 32, 8)])
def test_output_launch_at_the_grouped_size(width, experts, top_k):
    """The output launch of 16 tokens with many partials takes little longer than
    that of 8 (1.2 times; 2.8 and 2.0 when a wave walks all of a token's partials)."""
    layer = make_layer(hidden=2048, width=width, experts=experts, top_k=top_k, rank=32, tokens=16, seed=11)
    plan = compile_budget(hidden_size=2048, expert_width=width, top_k=top_k, retention=0.4, screen_keep=0.625)
    reader = build_any(layer, plan, 16)

    def fastest(tokens):
        arguments = [v[:tokens].to(reader.native_gu.device) for v in (layer.hidden, layer.ids, layer.weights)]
        out = reader(*arguments)
        torch.cuda.synchronize()
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph):
            for _ in range(16):
                reader.launch_stage("output", *arguments, None, out)
        times = []
        for _ in range(10):
            begin, end = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
            begin.record()
            for _ in range(4):
                graph.replay()
            end.record()
            torch.cuda.synchronize()
            times.append(begin.elapsed_time(end))
        return min(times)

    assert fastest(16) < 1.6 * fastest(8)


def build_any(layer, plan, tokens):
    if layer.encoder is not None:
        return build(layer, plan, tokens, selection_score="point")
    from calibration_free_moe.reader.progressive import ProgressiveReader, channel_major_down
    from tests.test_gpu_parity import DEVICE

    return ProgressiveReader(layer.gate_up.to(DEVICE), channel_major_down(layer.down.to(DEVICE)), None, None,
                             plan, tokens, sketch=(layer.codes.to(DEVICE), layer.statistics.to(DEVICE)),
                             selection_score="point")
