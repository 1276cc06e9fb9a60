"""fp32 attention in shares of the key tiles: the arithmetic of the shares on the
CPU, the assembly, and results against the fp32 oracle where a share or the rows
past the last query tile can end badly.  Both sides sum L products in fp32 in different
orders on N(0,1) inputs: 5e-5 at most and 5e-6 on average, as for every fp32 call."""
import os
import shutil
import subprocess

import pytest
import torch

from oracle import sdv2_oracle as oracle
from streamdiffusionv2_amd import build_ext

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_every_tile_has_one_owner(tmp_path):
    if shutil.which("g++") is None:
        pytest.skip("no g++")
    exe = str(tmp_path / "f32_plan_check")
    subprocess.run(["g++", "-std=c++17", "-O2", "-Wall", "-Werror", f"-I{build_ext.CSRC}",
                    os.path.join(ROOT, "tests", "c_abi", "f32_plan_check.cpp"), "-o", exe], check=True)
    run = subprocess.run([exe], capture_output=True, text=True, timeout=120)
    assert run.returncode == 0 and "2000 plans" in run.stdout, run.stdout


def test_places_for_the_pieces():
    from streamdiffusionv2_amd import _capi

    need = _capi.lib().sdv2_swa_attn_f32_workspace_bytes
    # tickets, and two places of four blocks (32 x 128 sums, 32 maxima, 32 sums of weights) for each of 512 workgroups
    assert need(1, 1560, 12, 6240) == 65536 + 2 * 512 * 4 * 32 * (128 + 2) * 4
    assert need(1, 64, 1, 32) == 0 and need(64, 65536, 64, 640) == 0        # one tile; more items than tickets
    assert need(65535, 1 << 30, 65535, 640) == 0


@pytest.mark.gpu
@pytest.mark.parametrize(
    "rows,S,H,L,lens,block",
    [
        (1, 160, 3, 1040, None, 0),               # one block past a whole tile: 4 waves over 33 tiles of keys
        (2, 129, 2, 999, [999, 5], 0),            # one row in it, a row shorter than a piece
        (1, 192, 3, 1000, None, 0),               # two blocks, two waves each
        (2, 190, 2, 700, [700, 33], 95),          # the mask inside the chunk, in the rest and in the whole tile
        (1, 224, 2, 640, None, 0),                # three blocks: a tile with an idle wave
        (1, 31, 40, 96, None, 0),                 # fewer key tiles than waves
        (1, 33, 1, 8192, None, 0),                # the most pieces, of two blocks alone
        (1, 128, 1, 8192, None, 0),               # the most pieces of a whole tile
        (3, 896, 12, 160, None, 0),               # whole items, uncut
        (1, 1300, 24, 330, None, 0),              # more than one item to a workgroup
        (3, 160, 2, 300, [0, 300, 64], 0),        # a row without keys: zeros
    ],
)
def test_shares_match_the_oracle(gpu_device, rows, S, H, L, lens, block):
    from streamdiffusionv2_amd import ops

    torch.manual_seed(31)
    q, k, v = torch.randn(rows, S, H, 128), torch.randn(rows, L, H, 128), torch.randn(rows, L, H, 128)
    starts = [max(0, n - S) for n in lens] if block else None
    full = lens or [L] * rows
    live = [r for r in range(rows) if full[r] > 0]
    pick = lambda t: t[live]
    mask = ([starts[r] for r in live], block) if block else ()
    if block:
        live = [r for r in live if full[r] >= S]
        mask = ([starts[r] for r in live], block)
    want = oracle.attention_fp32_reference(pick(q), pick(k), pick(v), [full[r] for r in live], *mask)
    sl = torch.tensor(full, dtype=torch.int32, device=gpu_device)
    kw = dict(chunk_key_start=starts, mask_block_tokens=block) if block else {}
    args = [t.to(gpu_device) for t in (q, k, v)]
    got, again = ops.swa_attention(*args, sl, **kw), ops.swa_attention(*args, sl, **kw)
    torch.cuda.synchronize()
    assert torch.equal(got, again)
    err = (got.cpu()[live] - want).abs()
    assert torch.isfinite(got).all() and err.max().item() <= 5e-5 and err.mean().item() <= 5e-6, err.max().item()
    for r in range(rows):
        if full[r] == 0:
            assert not got[r].any()
