"""sdv2_linear in its tiles of 192 and more rows: which products take one round, what the compiler made of those loops,
and their results at the edges of the tiles."""
import ctypes as C
import os
import re
import shutil
import subprocess

import pytest
import torch

from streamdiffusionv2_amd import _capi, build_ext, ops
from test_attention_isa import instructions, registers
from test_linear import ROOT, _check


def test_which_products_are_one_round():
    lib = _capi.lib()
    for m, n, k, squares, want in ((1560, 4608, 1536, 0, 1), (1560, 5120, 5120, 0, 1), (1792, 5120, 64, 0, 1), (1793, 5120, 64, 0, 0),
                                   (1560, 5120, 5120, 1, 0), (1536, 5120, 64, 1, 1), (1280, 5120, 5120, 1, 1),
                                   (96, 5120, 5120, 0, 0), (97, 5120, 5120, 0, 1), (1, 5120, 2048, 0, 1), (9360, 1536, 1536, 0, 0), (1560, 15360, 5120, 0, 0), (0, 64, 64, 0, 0), (16, 96, 64, 0, 0), (16, 64, 96, 0, 0)):
        assert lib.sdv2_linear_one_round(m, n, k, squares) == want, (m, n, k, squares)


@pytest.mark.skipif(shutil.which("g++") is None, reason="no g++")
def test_the_tile_a_product_takes(tmp_path):
    """Measured (us, weights cold): within 5 % of the fastest tile, among them products whose row tiles differ in how full they
    are.  With sums of squares never the tile of 160 columns."""
    measured = [
        ((352, 4352, 4352), {(160, 64): 27.28, (96, 128): 37.27, (160, 128): 37.42}),
        ((359, 5120, 5120), {(160, 64): 32.98, (96, 128): 46.67, (160, 128): 45.28}),
        ((320, 6144, 6144), {(160, 64): 49.95, (96, 128): 43.41}),
        ((508, 6144, 6144), {(128, 128): 62.45, (160, 128): 53.06}),
        ((1561, 3712, 3712), {(224, 128): 48.21, (256, 128): 43.44}),
        ((1567, 5120, 5120), {(224, 160): 72.81}),
        ((256, 1536, 1536), {(64, 64): 7.76}),
    ]
    exe = str(tmp_path / "linear_tile_check")
    subprocess.run(["g++", "-std=c++17", "-O2", "-Wall", "-Werror", f"-I{build_ext.CSRC}",
                    os.path.join(ROOT, "tests", "c_abi", "linear_tile_check.cpp"), "-o", exe], check=True)
    asked = [*(size + (0,) for size, _ in measured), (1567, 5120, 5120, 1), (64, 96, 64, 0)]
    run = subprocess.run([exe, *(str(x) for a in asked for x in a)], capture_output=True, text=True, timeout=60)
    got = [tuple(int(x) for x in line.split()) for line in run.stdout.splitlines()]
    for (size, times), tile in zip(measured, got):
        assert times[tile] <= 1.05 * min(times.values()), (size, tile)
    assert got[-2][1] != 160 and got[-1] == (0, 0)


def test_nothing_touches_a_fragment_on_its_way():
    """(as for the smaller tiles: from an LDS read to the wait behind it no instruction names the registers it will land in;
    the loops are walked twice, so that what is on its way at their end meets their beginning)"""
    out = os.path.join(ROOT, "build", "isa_check")
    os.makedirs(out, exist_ok=True)
    path = os.path.join(out, "linear_wide.s")
    cmd = [build_ext.hipcc_path(), *build_ext.HIPCC_FLAGS, f"-I{os.path.join(ROOT, 'include')}", f"-I{build_ext.CSRC}",
           "-S", "--cuda-device-only", str(build_ext.CSRC / "linear_wide.hip"), "-o", path]
    res = subprocess.run(cmd, capture_output=True, text=True)
    assert res.returncode == 0, res.stderr[-2000:]
    lines = open(path).read().split("\n")
    starts = [i for i, l in enumerate(lines) if re.match(r"^_Z\S*linear_kernel\S*:", l)]
    assert len(starts) == 4
    for start in starts:
        body = lines[start:next(i for i in range(start, len(lines)) if lines[i].strip().startswith(".Lfunc_end"))]
        products = [i for i, l in enumerate(body) if "v_mfma" in l]
        # from the first fragments asked for (behind the barrier ahead of the loop) to the wait behind the loop
        first = next(i for i, l in enumerate(body) if "ds_read_b128" in l)
        top = max(i for i in range(products[0]) if re.match(r"^\.LBB", body[i]))
        name = body[top].split(":")[0]
        back = next(i for i in range(products[-1], len(body)) if re.search(r"s_cbranch\w*\s+" + re.escape(name) + r"\b", body[i]))
        end = next(i for i in range(back, len(body)) if "lgkmcnt(0)" in body[i])
        assert first < top and not any(re.match(r"^\.LBB", l) for l in body[top + 1:back])        # one block
        flying, reads = set(), 0
        for mn, ops_ in instructions(body[first:back + 1] + body[top:back + 1] + body[back + 1:end + 1]):
            if mn == "s_waitcnt" and "lgkmcnt(0)" in ops_[0]:
                flying = set()
            elif mn.startswith("ds_read_b128"):
                assert not (registers(ops_[0]) | registers(ops_[1])) & flying, (mn, ops_)
                flying |= registers(ops_[0])
                reads += 1
            else:
                assert not any(registers(o) & flying for o in ops_), (mn, ops_)
        assert reads >= 50 and not flying
    text = "\n".join(lines)
    assert not re.search(r"\bscratch_(load|store)", text)
    assert max(int(x) for x in re.findall(r"\.vgpr_count:\s+(\d+)", text)) <= 256


@pytest.mark.gpu
@pytest.mark.parametrize("m,n,k,tile", [
    (5601, 1280, 192, (256, 128)), (6399, 1280, 64, (256, 128)),                            # fewer stages than lie in LDS
    (3841, 1536, 320, (192, 128)), (4032, 1536, 128, (192, 128)),
    (4256, 1536, 1536, (224, 128)), (4033, 1536, 192, (224, 128)), (1560, 4608, 256, (224, 128)), (1569, 4608, 128, (256, 128)),
    (1560, 5120, 320, (224, 160)), (1792, 5120, 64, (224, 160)), (1569, 5120, 128, (224, 160)), (1570, 5120, 192, (224, 160)),
])
def test_wide_products(gpu_device, m, n, k, tile):
    print(f"linear {m} x {n} x {k}", flush=True)
    assert (m + tile[0] - 1) // tile[0] * (n // tile[1]) <= 256 and _capi.lib().sdv2_linear_one_round(m, n, k, 0)
    gen = torch.Generator(device=gpu_device).manual_seed(m + n + k)
    x, w, b = (torch.randn(*s, generator=gen, device=gpu_device).bfloat16() for s in ((m, k), (n, k), (n,)))
    wide = torch.randn(m, k + 72, generator=gen, device=gpu_device).bfloat16()
    for xx, bb, squared in ((x, b, False), (wide[:, 8:k + 8], None, tile[1] % 64 == 0)):
        out = torch.full((m + 3, n + 8), 7.0, device=gpu_device).bfloat16()                # rows and columns that are not its own
        squares = torch.full((m + 1, n // 32), -1.0, device=gpu_device)
        p = _capi.LinearParams(xx.data_ptr(), w.data_ptr(), bb.data_ptr() if bb is not None else None, out.data_ptr(),
                               xx.stride(0), k, n + 8, m, n, k, _capi.DTYPE_BF16, torch.cuda.current_stream().cuda_stream)
        p.row_squares = squares.data_ptr() if squared else None
        _capi.check(_capi.lib().sdv2_linear(C.byref(p)), "sdv2_linear")
        torch.cuda.synchronize()
        _check(out[:m, :n], xx, w, bb)
        assert (out[m:] == 7).all() and (out[:, n:] == 7).all()
        if squared:                                        # 32 terms in fp32, 2^-24 each
            want = out[:m, :n].double().pow(2).view(m, n // 32, 32).sum(-1)
            assert ((squares[:m].double() - want).abs() <= 32 * 2.0 ** -24 * want).all() and (squares[m:] == -1).all()


@pytest.mark.gpu
@pytest.mark.parametrize("m,n,k,squared", [
    (97, 2176, 2176, True), (300, 2176, 2176, False), (352, 3712, 3712, True), (464, 3712, 3712, True), (820, 3712, 3712, False),
    (352, 5120, 5120, True), (640, 5120, 5120, True), (1080, 5120, 5120, True), (1560, 5120, 5120, False), (130, 15360, 5120, False),
])
def test_long_contractions(gpu_device, m, n, k, squared):
    """Past 2048: all of the width of a model of 17, 29 and 40 heads, against 64 bits, with sums of squares or without."""
    print(f"linear {m} x {n} x {k}", flush=True)
    assert _capi.lib().sdv2_linear_one_round(m, n, k, squared)
    gen = torch.Generator(device=gpu_device).manual_seed(m + n + k)
    x, w, b = (torch.randn(*s, generator=gen, device=gpu_device).bfloat16() for s in ((m, k), (n, k), (n,)))
    with torch.no_grad():
        out = ops.linear_or_none(x, w, b, row_squares=squared)
        again = ops.linear_or_none(x, w, b)
    if squared:                                            # 32 terms in fp32, 2^-24 each
        out, squares = out
        want = out.double().pow(2).view(m, n // 32, 32).sum(-1)
        assert ((squares.double() - want).abs() <= 32 * 2.0 ** -24 * want).all()
    assert torch.equal(out, again)
    _check(out, x, w, b)
