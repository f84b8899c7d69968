"""Device sketch construction (cfmoe_build_sketch) against the torch build.

The HIP kernel (`build_sketch(..., device_kernel=True)`) builds the reference's
resident sketch format (sketch.py:84-150) from device weights; the default
`build_sketch` runs the torch construction on any device (the default reader
constructor uses it, test_progressive_reader.py:803-805 of the reference). The rotation is the same FP32 operations in the same order, so
the rotated values agree bit for bit; the sums behind mean|v|, the scale and
the residual run in a different order. The check therefore follows the
reference's own comparison of two sketch builds (codes exact, statistics
atol 1e-4 / rtol 1e-3, test_progressive_reader.py:803-809), with one stated
allowance: a trit may differ only where |v| lies within 2e-5 (relative) of
0.7 mean|v| computed in float64, and the statistics of such a (row, block)
are left out of the tolerance check. Shapes cover the block-paired 16-byte
tails (width 512), an odd block count (hidden 384: the last tail half is
padding), a width that is not a multiple of five, and unrotated blocks.
"""

import pytest
import torch

from calibration_free_moe.reader import _ext
from calibration_free_moe.reader.sketch import (
    ZERO_CODE,
    block_hadamard_signs,
    build_sketch,
    code_offsets,
    rotate_blocks,
    unpack_sketch,
)

pytestmark = pytest.mark.gpu

DEVICE = torch.device("cuda:0")


@pytest.mark.parametrize(
    "experts,width,hidden,rotated",
    [(4, 256, 512, True), (2, 512, 2048, True), (3, 96, 384, True), (2, 72, 256, False)],
)
def test_device_sketch_matches_torch_build(experts, width, hidden, rotated):
    generator = torch.Generator().manual_seed(experts * 1000 + width + hidden)
    weights = (torch.randn(experts, 2 * width, hidden, generator=generator) * 0.02).to(torch.bfloat16)
    signs = block_hadamard_signs(hidden, "cpu") if rotated else None
    want_codes, want_stats = build_sketch(weights, signs)
    got_codes, got_stats = build_sketch(
        weights.to(DEVICE), None if signs is None else signs.to(DEVICE), device_kernel=True
    )
    torch.cuda.synchronize()
    got_codes, got_stats = got_codes.cpu(), got_stats.cpu()
    assert got_codes.shape == want_codes.shape and got_stats.shape == want_stats.shape
    rows = 2 * width
    got_trits = unpack_sketch(got_codes, rows, hidden)
    want_trits = unpack_sketch(want_codes, rows, hidden)
    # the allowance: near-threshold coordinates, from the FP32 rotated values
    value = rotate_blocks(weights, signs).reshape(experts, rows, hidden // 128, 128).double()
    magnitude = value.abs()
    threshold = 0.7 * magnitude.mean(-1, keepdim=True)
    near = ((magnitude - threshold).abs() <= 2e-5 * threshold).reshape(experts, rows, hidden)
    differ = got_trits != want_trits
    assert not (differ & ~near).any(), "a trit differs away from the TWN threshold"
    assert int(differ.sum()) <= max(8, differ.numel() // 10000)
    # every byte without a flipped trit is identical (padding bytes included)
    assert int((got_codes != want_codes).sum()) <= int(differ.sum())
    # statistics [E, 2 I, blocks, 2] to the reference's tolerance, outside
    # the (row, block) cells that hold a flipped trit
    flipped = differ.reshape(experts, rows, hidden // 128, 128).any(-1)
    clean = ~flipped
    torch.testing.assert_close(got_stats.float()[clean], want_stats.float()[clean],
                               rtol=1e-3, atol=1e-4)


def test_default_build_on_the_device_is_the_torch_construction():
    """Without device_kernel, device weights get the torch construction: the
    same codes as the build on the host, and statistics to the reference's
    tolerance (its reductions run in the device's order)."""
    generator = torch.Generator().manual_seed(77)
    weights = (torch.randn(3, 2 * 96, 384, generator=generator) * 0.02).to(torch.bfloat16)
    signs = block_hadamard_signs(384, "cpu")
    want_codes, want_stats = build_sketch(weights, signs)
    got_codes, got_stats = build_sketch(weights.to(DEVICE), signs.to(DEVICE))
    torch.cuda.synchronize()
    assert torch.equal(got_codes.cpu(), want_codes)
    torch.testing.assert_close(got_stats.cpu(), want_stats, atol=1e-4, rtol=1e-3)


@pytest.mark.parametrize(
    "experts,width,hidden,offset",
    # one tile of code columns holds 160 channels: a part of one, one, one and
    # a channel, with rows and signs that start at odd elements; one block (an
    # odd count's tail), and the largest widths
    [(2, 33, 128, 1), (2, 160, 384, 3), (1, 161, 640, 5), (1, 2048, 256, 0), (1, 80, 4096, 7)],
)
def test_device_sketch_tiles_and_offsets(experts, width, hidden, offset):
    """Tile edges and views at any element offset."""
    generator = torch.Generator().manual_seed(width + offset)
    flat = (torch.randn(offset + experts * 2 * width * hidden, generator=generator) * 0.02).bfloat16()
    weights = flat[offset:].view(experts, 2 * width, hidden)
    signs = block_hadamard_signs(hidden, "cpu")
    want_codes, want_stats = build_sketch(weights, signs)
    device_signs = torch.cat([torch.zeros(offset, dtype=torch.int8), signs]).to(DEVICE)[offset:]
    got_codes, got_stats = build_sketch(
        flat.to(DEVICE)[offset:].view(experts, 2 * width, hidden), device_signs, device_kernel=True
    )
    torch.cuda.synchronize()
    value = rotate_blocks(weights, signs).reshape(experts, 2 * width, hidden // 128, 128).double()
    threshold = 0.7 * value.abs().mean(-1, keepdim=True)
    near = (value.abs() - threshold).abs() <= 2e-5 * threshold
    differ = (unpack_sketch(got_codes.cpu(), 2 * width, hidden)
              != unpack_sketch(want_codes, 2 * width, hidden)).reshape(near.shape)
    assert not (differ & ~near).any()
    assert int((got_codes.cpu() != want_codes).sum()) <= int(differ.sum())
    clean = ~differ.any(-1)
    torch.testing.assert_close(got_stats.cpu().float()[clean], want_stats.float()[clean],
                               rtol=1e-3, atol=1e-4)


@pytest.mark.parametrize(
    "experts,width,hidden,rotated",
    # runs of 16 bytes (four blocks to a workgroup: fewer, four, five, and a
    # workgroup that is short of blocks), 32, 64 and more than a tile; odd block
    # counts, whose last tail rows have no second block, with and without a body
    [(2, 3, 128, True), (3, 5, 384, False), (2, 16, 640, True), (1, 40, 512, True), (2, 33, 1152, True),
     (2, 41, 384, True), (1, 80, 256, False), (2, 160, 128, True), (1, 176, 384, True)],
)
def test_device_sketch_writes_every_byte_and_no_other(experts, width, hidden, rotated):
    """The C entry on buffers that hold 0xff, between guard bytes: every code
    byte is written (121 where no channel's trits lie), every statistic, and
    nothing on either side."""
    generator = torch.Generator().manual_seed(7 * width + hidden)
    weights = (torch.randn(experts, 2 * width, hidden, generator=generator) * 0.02).bfloat16()
    signs = block_hadamard_signs(hidden, "cpu") if rotated else None
    want_codes, want_stats = build_sketch(weights, signs)
    guard, statistics = 256, 2 * want_stats.numel()
    codes = torch.full((2 * guard + want_codes.numel(),), 0xFF, dtype=torch.uint8, device=DEVICE)
    stats = torch.full((2 * guard + statistics,), 0xFF, dtype=torch.uint8, device=DEVICE)
    rows = weights.to(DEVICE)
    device_signs = None if signs is None else signs.to(DEVICE)
    _ext.check(_ext.library().cfmoe_build_sketch(
        experts, width, hidden, rows.data_ptr(), None if signs is None else device_signs.data_ptr(),
        codes.data_ptr() + guard, stats.data_ptr() + guard, torch.cuda.current_stream().cuda_stream))
    torch.cuda.synchronize()
    for buffer in (codes, stats):
        assert bool((buffer[:guard] == 0xFF).all()) and bool((buffer[-guard:] == 0xFF).all())
    got = codes[guard:-guard].cpu().view(experts, -1)
    padding = torch.ones(got.shape[1], dtype=torch.bool)
    padding[code_offsets(2 * width, hidden).flatten()] = False
    assert bool((got[:, padding] == ZERO_CODE).all())
    differ = unpack_sketch(got, 2 * width, hidden) != unpack_sketch(want_codes, 2 * width, hidden)
    assert int(differ.sum()) <= max(2, differ.numel() // 10000)  # (near the threshold)
    assert int((got != want_codes).sum()) <= int(differ.sum())
    # 0xffff is a NaN: no statistic is one
    got_stats = stats[guard:-guard].cpu().view(torch.float16).view(experts, hidden // 128, 2, 2 * width)
    clean = ~differ.reshape(experts, 2 * width, hidden // 128, 128).any(-1)
    torch.testing.assert_close(got_stats.permute(0, 3, 1, 2).float()[clean], want_stats.float()[clean],
                               rtol=1e-3, atol=1e-4)


def test_narrow_sketch_does_not_pay_for_a_wide_tile():
    """A width of 16 fills 8 of a workgroup's 64 code columns: it takes less time
    than the 160 channels that fill them all (half of it; as long when every
    workgroup walks 64 columns)."""
    signs = block_hadamard_signs(2048, DEVICE)

    def fastest(width):
        weights = torch.randn(128, 2 * width, 2048, device=DEVICE).mul_(0.02).bfloat16()
        times = []
        for _ in range(8):
            begin, end = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
            begin.record()
            for _ in range(20):
                build_sketch(weights, signs, device_kernel=True)
            end.record()
            torch.cuda.synchronize()
            times.append(begin.elapsed_time(end))
        return min(times)

    assert fastest(16) < 0.75 * fastest(160)


def test_device_sketch_of_more_experts_than_a_launch_holds():
    """8 388 608 workgroups of 512 threads are 2^32, one more than a launch can
    hold: the experts past them come from a second one."""
    pattern = (torch.randn(97, 2, 128, generator=torch.Generator().manual_seed(5)) * 0.02).bfloat16().to(DEVICE)
    want_codes, want_stats = build_sketch(pattern, device_kernel=True)
    repeats = (1 << 23) // 97 + 1
    codes, stats = build_sketch(pattern.repeat(repeats, 1, 1), device_kernel=True)
    for begin in range(0, repeats, 1 << 13):
        part = codes.view(repeats, 97, -1)[begin : begin + (1 << 13)]
        assert bool((part == want_codes).all())
    assert torch.equal(stats.reshape(repeats, 97, -1), want_stats.reshape(1, 97, -1).expand(repeats, -1, -1))
