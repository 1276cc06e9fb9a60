"""The sums of the adaptive sink decision where a token range or a thread's columns can end badly: similarities against
float64 means.  bf16: two cosines and their sum, each rounded once (2^-9 of at most 1, 1 and 2), the means before them
(2^-9 of a column each, which a cosine over 128 columns and more averages out) - 1e-2 as for every call; fp32 1e-5."""
import pytest
import torch

from oracle import sdv2_oracle as oracle

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize(
    "heads,grid,sink,dtype",
    [
        (16, (1, 1, 1), 2, torch.bfloat16),       # one token: seven of the eight ranges empty
        (17, (1, 3, 3), 1, torch.bfloat16),       # ranges of two tokens, the last of one; three column groups a thread
        (3, (1, 16, 16), 3, torch.bfloat16),      # a token for every thread row of every range
        (2, (1, 43, 48), 5, torch.bfloat16),      # 258 tokens to a range: two more than one trip takes
        (48, (1, 5, 13), 2, torch.bfloat16),
        (49, (1, 5, 13), 3, torch.bfloat16),      # four column groups a thread
        (2, (1, 33, 32), 2, torch.float32),       # 132 tokens to a range: more than one trip takes in fp32
    ],
)
@pytest.mark.parametrize("kept", [False, True])
def test_similarities_at_the_edges(gpu_device, heads, grid, sink, dtype, kept):
    from streamdiffusionv2_amd import ops, rope

    rows, tokens = 2, grid[1] * grid[2]
    gen = torch.Generator().manual_seed(heads * 1000 + tokens)
    draw = lambda n, base: (torch.randn(rows, n, heads, 128, generator=gen) * 0.5 + base).to(dtype)
    base = torch.randn(1, 1, heads, 128, generator=gen)
    k, v = draw(tokens, base), draw(tokens, -base)
    ck = torch.cat([draw(tokens, base * (1 - 0.4 * j)) for j in range(sink + 1)], 1)
    cv = torch.cat([draw(tokens, base * (0.4 * j - 1)) for j in range(sink + 1)], 1)
    starts = [3, 0]
    roped = oracle.causal_rope_apply(k, [grid] * rows, oracle.build_freqs(), starts).type_as(v)
    means = lambda t, n: t[:, :n * tokens].double().reshape(rows, n, tokens, -1).mean(2)
    cos = lambda a, b: torch.cosine_similarity(a, b, dim=-1)
    want = (cos(means(ck, sink), means(roped, 1)) + cos(means(cv, sink), means(v, 1))) / 2
    table = ops.device_freqs(rope.build_freqs(), gpu_device)
    args = [t.to(gpu_device) for t in (k, v, ck, cv)]
    more = {}
    if kept:
        sums = ops.new_sink_frame_sums(rows, heads, sink, gpu_device)
        more = dict(frame_sums=sums, planned_frames=[-1] * rows)
        ops.sink_similarity(*args, table, grid[1:], starts, sink, -2.0, stale_frames=[(1 << sink) - 1] * rows, **more)
        more["stale_frames"] = [0] * rows
    sim, refresh = ops.sink_similarity(*args, table, grid[1:], starts, sink, 1.5, **more)
    torch.cuda.synchronize()
    assert (sim.cpu().double() - want).abs().max().item() <= (1e-2 if dtype == torch.bfloat16 else 1e-5), (sim.cpu(), want)
    assert refresh.cpu().tolist() == sim.argmin(dim=1).cpu().tolist()
