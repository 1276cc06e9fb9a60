"""Attention with equal shares of the key tiles (num_splits = SDV2_SPLITS_EVEN):
the integer arithmetic of the shares on the CPU, what the compiler made of the
kernel, and its results against the fp32 oracle where a share can end badly -
around a query tile of 256 rows, a block of 32, a key tile of 64, with rows of
different lengths, with the mask inside the chunk, and with scores that force
the running-maximum pass."""
import os
import re
import shutil
import subprocess

import pytest
import torch

from oracle import sdv2_oracle as oracle
from streamdiffusionv2_amd import _capi, build_ext, ops
from test_attention_isa import early_reads, instructions

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
EVEN = 1 << 20


def test_every_tile_has_one_owner(tmp_path):
    if shutil.which("g++") is None:
        pytest.skip("no g++")
    exe = str(tmp_path / "even_plan_check")
    subprocess.run(["g++", "-std=c++17", "-O2", "-Wall", "-Werror", f"-I{build_ext.CSRC}",
                    os.path.join(ROOT, "tests", "c_abi", "even_plan_check.cpp"), "-o", exe], check=True)
    run = subprocess.run([exe], capture_output=True, text=True, timeout=120)
    assert run.returncode == 0 and "3000 plans" in run.stdout, run.stdout


def test_which_calls_get_equal_shares():
    lib = _capi.lib()
    for shape, plan in (((1, 1560, 40, 9360), EVEN), ((4, 4680, 12, 18720), EVEN),
                        ((1, 256, 12, 1536), lib.sdv2_swa_attn_default_splits(1, 256, 12, 1536)),
                        ((1, 1560, 12, 9360), lib.sdv2_swa_attn_default_splits(1, 1560, 12, 9360)),
                        ((0, 1560, 12, 9360), 1)):
        assert lib.sdv2_swa_attn_plan(*shape) == plan, shape
    # tickets, and two results of 256 x 128 floats and 256 log-sum-exps for each of 256 workgroups, whatever the shape
    assert lib.sdv2_swa_attn_workspace_bytes(1, 1560, 40, 9360, EVEN) == 65536 + 512 * 256 * (128 + 1) * 4
    assert lib.sdv2_swa_attn_workspace_bytes(64, 65536, 64, 640, EVEN) == 0          # more query tiles than tickets


def test_calls_that_equal_shares_make_slower_keep_their_ranges():
    """Chunks whose last query tile holds few rows: the rest of every pair takes longer in shares, and its idle waves leave
    the tile kernels more power.  (Measured 5 to 11 % slower in equal shares.)"""
    lib = _capi.lib()
    for shape in ((3, 257, 12, 7471), (1, 528, 40, 6336), (1, 544, 40, 6528), (2, 783, 12, 4698), (1, 320, 40, 22155),
                  (2, 770, 12, 4620)):
        assert lib.sdv2_swa_attn_plan(*shape) == lib.sdv2_swa_attn_default_splits(*shape), shape


def test_masked_calls_are_planned_with_their_mask():
    """The mask inside the chunk leaves items of several lengths, which are handed out without whole rounds: over many (row,
    head) pairs that took 9 to 19 % more than the key ranges, over few it takes less."""
    lib = _capi.lib()
    for shape, block in (((4, 2574, 40, 10296), 1716), ((4, 3120, 40, 6240), 1560), ((4, 2142, 40, 14994), 1428),
                         ((2, 4896, 40, 34272), 1632), ((3, 3000, 40, 9000), 1000), ((2, 3120, 40, 9360), 1560)):
        assert lib.sdv2_swa_attn_plan_masked(*shape, block, 1) == lib.sdv2_swa_attn_default_splits(*shape), shape
    for shape, block in (((1, 3807, 12, 11421), 1269), ((3, 1995, 12, 3990), 1330), ((1, 2652, 12, 18564), 1768)):
        assert lib.sdv2_swa_attn_plan_masked(*shape, block, 1) == EVEN, shape
    for shape in ((1, 3807, 12, 11421), (4, 3120, 40, 6240), (0, 1, 1, 1)):
        for block in (0, -1, shape[1], 1 << 30):                                # no mask
            assert lib.sdv2_swa_attn_plan_masked(*shape, block, 1) == lib.sdv2_swa_attn_plan(*shape), (shape, block)
    assert lib.sdv2_swa_attn_plan_masked(1, 3807, 12, 3000, 1269, 1) == lib.sdv2_swa_attn_plan(1, 3807, 12, 3000)
    # a descriptor is the mask's own: starts on the device, different ones, or no mask at all are planned apart
    q, k = (torch.empty(2, n, 40, 128, dtype=torch.bfloat16, device="meta") for n in (2331, 16317))
    assert ops._starts_alike([5, 5]) and ops._starts_alike((7,))
    assert not ops._starts_alike([5, 6]) and not ops._starts_alike(None) and not ops._starts_alike(torch.zeros(2)) \
        and not ops._starts_alike([0] * 17) and not ops._starts_alike([])
    splits = [_capi.AttnParams.from_buffer_copy(ops._attn_layout(q, k, k, None, 0, False, False, block, alike)[0]).num_splits
              for block, alike in ((0, False), (1554, True), (1554, False))]
    assert splits == [EVEN, lib.sdv2_swa_attn_default_splits(2, 2331, 40, 16317), EVEN]


def test_equal_shares_that_are_refused():
    """(every refusal comes before the first HIP call)"""
    import ctypes as C

    lib = _capi.lib()

    def params(**more):
        p = _capi.AttnParams(q=256, k_cache=512, v_cache=768, out=1024, rows=1, q_tokens=512, heads=2, head_dim=128,
                             max_seq_len=640, num_splits=EVEN)
        for st in (p.q_stride, p.k_stride, p.v_stride, p.out_stride):
            st.row, st.token, st.head = 1 << 20, 256, 128
        for name, value in more.items():
            setattr(p, name, value)
        return C.byref(p)

    assert lib.sdv2_swa_attn_fwd(params()) == _capi.SDV2_ERR_WORKSPACE
    assert lib.sdv2_swa_attn_fwd(params(workspace=4096, workspace_bytes=65536)) == _capi.SDV2_ERR_WORKSPACE
    assert lib.sdv2_swa_attn_fwd(params(rope_freqs=2048)) == _capi.SDV2_ERR_UNSUPPORTED
    assert lib.sdv2_swa_attn_fwd(params(rows=64, q_tokens=65536, heads=64)) == _capi.SDV2_ERR_UNSUPPORTED
    assert lib.sdv2_swa_attn_fwd(params(num_splits=EVEN | 2)) == _capi.SDV2_ERR_INVALID_ARG
    assert lib.sdv2_swa_attn_fwd_static(params()) == _capi.SDV2_ERR_INVALID_ARG


def test_the_streaming_loop_keeps_its_promises():
    out = os.path.join(ROOT, "build", "isa_check")
    os.makedirs(out, exist_ok=True)
    path = os.path.join(out, "swa_attn_fwd_even.s")
    cmd = [build_ext.hipcc_path(), *build_ext.HIPCC_FLAGS, f"-I{os.path.join(ROOT, 'include')}", f"-I{build_ext.CSRC}",
           "-S", "--cuda-device-only", str(build_ext.CSRC / "swa_attn_fwd_even.hip"), "-o", path]
    res = subprocess.run(cmd, capture_output=True, text=True)
    assert res.returncode == 0, res.stderr[-2000:]
    lines = open(path).read().split("\n")
    starts = [i for i, l in enumerate(lines) if re.match(r"^_Z\S*swa_attn_fwd_even_kernel\S*:", l)]
    assert len(starts) == 2                       # without and with the mask inside the chunk
    for start in starts:
        end = next(i for i in range(start, len(lines)) if lines[i].strip().startswith(".Lfunc_end"))
        body = lines[start:end]
        problems, n_mfma = early_reads(instructions(body))
        assert n_mfma >= 256 and not problems, problems[:10]
        first = next(i for i, l in enumerate(body) if "matrix pipe drained, site 1" in l)
        last = next(i for i, l in enumerate(body) if "matrix pipe drained, site 0" in l)
        loop = next(i for i in range(first, last) if "Loop Header" in body[i])
        hot = body[loop:last]
        assert sum("v_mfma_f32_16x16x32_bf16" in l for l in hot) >= 128
        assert not [l.strip() for l in hot if re.search(r"\bscratch_(load|store)", l)]
    assert max(int(x) for x in re.findall(r"\.vgpr_count:\s+(\d+)", "\n".join(lines))) <= 256


def _close(got, want):
    err = (got.float().cpu() - want).abs()
    assert err.max().item() <= 2e-2 and err.mean().item() <= 2e-3, (err.max().item(), err.mean().item())


def _inputs(rows, S, H, L, scale=1.0):
    gen = torch.Generator().manual_seed(1000 * S + L)
    q, k, v = (torch.randn(rows, n, H, 128, generator=gen) for n in (S, L, L))
    return (q * scale).bfloat16(), (k * scale).bfloat16(), v.bfloat16()


def _twice(q, k, v, lens, dev, **kw):
    """The result, the same bits both times; the tickets are left at zero."""
    from streamdiffusionv2_amd import ops

    ws = ops.new_workspace(dev, _capi.lib().sdv2_swa_attn_workspace_bytes(q.shape[0], q.shape[1], q.shape[2], k.shape[1], EVEN))
    out = [ops.swa_attention(q.to(dev), k.to(dev), v.to(dev), lens, num_splits=EVEN, workspace=ws, **kw) for _ in range(2)]
    torch.cuda.synchronize()
    assert torch.equal(out[0], out[1])
    assert not ws[:65536].any()
    return out[0]


@pytest.mark.gpu
@pytest.mark.parametrize("rows,S,H,L", [
    (1, 256, 2, 1), (1, 256, 1, 64), (1, 255, 1, 65), (1, 20, 3, 700),      # one query tile, a tile that is not whole, a block
    (1, 257, 3, 1100), (2, 288, 2, 640), (1, 289, 2, 129), (1, 384, 2, 333), (1, 385, 2, 700),      # rows past the last whole tile
    (1, 512, 12, 127), (3, 1040, 4, 515), (2, 777, 5, 2000),                # shares of less than a tile, of about one, of several
    (5, 600, 40, 130),                                                      # every workgroup takes a query tile whole first
])
def test_against_the_oracle(gpu_device, rows, S, H, L):
    print(f"equal shares: {rows} x {S} x {H} against {L}", flush=True)
    q, k, v = _inputs(rows, S, H, L)
    _close(_twice(q, k, v, None, gpu_device), oracle.attention_fp32_reference(q, k, v, [L] * rows))


@pytest.mark.gpu
def test_rows_of_different_lengths(gpu_device):
    q, k, v = _inputs(4, 600, 3, 1000)
    lens = [1000, 1, 64, 517]
    got = _twice(q, k, v, torch.tensor(lens, dtype=torch.int32, device=gpu_device), gpu_device)
    _close(got, oracle.attention_fp32_reference(q, k, v, lens))


@pytest.mark.gpu
@pytest.mark.parametrize("device_starts", [False, True])
@pytest.mark.parametrize("rows,S,L,block,starts", [
    (1, 800, 1500, 100, [700]), (1, 777, 777, 259, [0]), (2, 544, 1200, 32, [656, 656]), (2, 544, 1200, 300, [0, 600]),
    (1, 600, 650, 1, [17]),
])
def test_mask_inside_the_chunk(gpu_device, rows, S, L, block, starts, device_starts):
    q, k, v = _inputs(rows, S, 5, L)
    where = torch.tensor(starts, dtype=torch.int32, device=gpu_device) if device_starts else starts
    got = _twice(q, k, v, None, gpu_device, chunk_key_start=where, mask_block_tokens=block)
    _close(got, oracle.attention_fp32_reference(q, k, v, [L] * rows, starts, block))


@pytest.mark.gpu
@pytest.mark.parametrize("block", [0, 300])
def test_scores_of_several_hundred(gpu_device, block):
    """Pieces of an item whose exponent references differ by hundreds, some redone with a running maximum; a piece that
    goes on from the last key to the first must not take hidden keys for all there is."""
    q, k, v = _inputs(1, 600, 4, 900, scale=14.0)
    kw = dict(chunk_key_start=[300], mask_block_tokens=block) if block else {}
    want = oracle.attention_fp32_reference(q, k, v, [900], *(([300], block) if block else ()))
    _close(_twice(q, k, v, None, gpu_device, **kw), want)


@pytest.mark.gpu
def test_a_layer_call_is_planned_again_when_the_mask_changes(gpu_device):
    from streamdiffusionv2_amd import ring, rope

    heads, grid, S, cap = 40, (3, 20, 52), 3120, 9360
    cache = ring.new_kv_cache(1, 2, cap, heads, 1, device=gpu_device)[0]
    q = torch.empty(2, S, heads, 128, device=gpu_device, dtype=torch.bfloat16)
    launcher = ops.LayerLauncher(cache["k"], cache["v"], cache["global_end_index"], cache["local_end_index"],
                                 ops.device_freqs(rope.build_freqs(), gpu_device), grid, q, rope_in_attention=False)
    ranges = _capi.lib().sdv2_swa_attn_default_splits(2, S, heads, cap)
    for start, block, want in ((S, 0, EVEN), (S, 1560, ranges), (2 * S, 1560, ranges), (S, 0, EVEN)):
        launcher.patch(q, q, q, [4, 4], ring.AppendPlan([start] * 2, [cap] * 2, [cap] * 2), None, block)
        assert launcher.at.num_splits == want and bool(launcher.workspace_need) == (want != 1), (start, block)


@pytest.mark.gpu
def test_cut_items_lose_nothing(gpu_device):
    """Error against 64 bits of a call whose query tiles are nearly all cut, and of the same call whole: the pieces meet
    in fp32, which adds some 2^-22 to the 2^-9 of the bf16 result - 1 % of room for the other exponent references."""
    from streamdiffusionv2_amd import ops

    q, k, v = (t.to(gpu_device) for t in _inputs(2, 1024, 40, 2000))       # (whole: 320 query tiles on the same matrix instructions)
    want = torch.empty(q.shape, dtype=torch.float64, device=gpu_device)
    for row in range(2):
        for h in range(40):
            s = q[row, :, h].double() @ k[row, :, h].double().t().contiguous() * 128 ** -0.5
            want[row, :, h] = s.softmax(-1) @ v[row, :, h].double()
    err = [((ops.swa_attention(q, k, v, None, num_splits=n).double() - want).norm() / want.norm()).item() for n in (1, EVEN)]
    assert err[1] <= 1.01 * err[0], err


@pytest.mark.gpu
def test_equal_shares_in_a_graph(gpu_device):
    """Recorded once, replayed on new inputs between eager calls of another shape on the same workspace."""
    from streamdiffusionv2_amd import ops

    q, k, v = (t.to(gpu_device) for t in _inputs(1, 700, 6, 1300))
    q2, k2, v2 = (t.to(gpu_device) for t in _inputs(2, 300, 4, 800))
    ops.swa_attention(q, k, v, num_splits=EVEN)
    other = ops.swa_attention(q2, k2, v2, num_splits=EVEN)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        out = ops.swa_attention(q, k, v, num_splits=EVEN)
    for i in range(4):
        q.copy_(q.roll(i + 1, 1))
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, ops.swa_attention(q, k, v, num_splits=EVEN))
        assert torch.equal(other, ops.swa_attention(q2, k2, v2, num_splits=EVEN))


def test_calls_left_whole():
    """Two ranges become one where tiles of four blocks make one round; what is not cut in two stays as it is."""
    lib = _capi.lib()
    for shape, plan in (((2, 1083, 12, 2166), 1), ((1, 672, 40, 2016), 1), ((3, 754, 12, 2262), 1), ((1, 1024, 24, 2048), 2),
                        # (plans of two counts: three ranges, or two, and one more for some pairs)
                        ((4, 567, 12, 10958), 3 | 3 << 8), ((2, 565, 24, 7152), 3 | 3 << 8), ((3, 343, 24, 3632), 2 | 4 << 8),
                        ((1, 1560, 12, 9360), 3), ((1, 756, 12, 4536), 4), ((1, 1560, 40, 9360), EVEN), ((1, 256, 12, 1536), 1)):
        assert lib.sdv2_swa_attn_plan(*shape) == plan, (shape, lib.sdv2_swa_attn_plan(*shape))
        if plan == 1:
            assert lib.sdv2_swa_attn_default_splits(*shape) == 1 and lib.sdv2_swa_attn_workspace_bytes(*shape, 0) == 0


def test_masked_calls_left_whole():
    """With the mask two ranges lose less to one, whichever entry asks: of shapes that stay whole without it, some do not."""
    lib = _capi.lib()
    for shape, block, ranges in (((1, 687, 40, 1374), 343, 1), ((4, 447, 12, 1341), 149, 1), ((2, 1278, 12, 2556), 426, 2),
                                 ((1, 2055, 12, 2950), 1027, 2)):
        assert lib.sdv2_swa_attn_default_splits(*shape) == 1
        for alike in (0, 1):
            assert lib.sdv2_swa_attn_plan_masked(*shape, block, alike) == ranges, shape
            for even in (False, True):
                assert ops._library_plan(lib, *shape, even, block, bool(alike)) == ranges, shape


@pytest.mark.gpu
@pytest.mark.parametrize("rows,S,H,L,block", [(2, 1278, 12, 2556, 426), (1, 687, 40, 1374, 343)])
def test_a_masked_shape_has_one_plan(gpu_device, rows, S, H, L, block):
    """The same ranges, and so the same bits, from every entry that chooses them."""
    import ctypes as C

    print(f"masked, one plan: {rows} x {S} x {H} against {L}, block {block}", flush=True)
    torch.manual_seed(31)
    q, k, v = (torch.randn(rows, n, H, 128).bfloat16().to(gpu_device) for n in (S, L, L))
    starts, lib = [L - S] * rows, _capi.lib()
    mask = dict(chunk_key_start=starts, mask_block_tokens=block)
    ranges = lib.sdv2_swa_attn_plan_masked(rows, S, H, L, block, 1)
    want = ops.swa_attention(q, k, v, num_splits=ranges, **mask)
    assert torch.equal(ops.swa_attention(q, k, v, **mask), want)
    assert torch.equal(ops.swa_attention(q, k, v, static_scratch=True, **mask), want)
    # the library's own choice behind the C entries, with a workspace and with none
    p = _capi.AttnParams.from_buffer_copy(ops._attn_layout(q, k, v, None, ranges, False, False, block, True)[0])
    whole = ops.swa_attention(q, k, v, num_splits=1, **mask)
    host = (C.c_int64 * rows)(*starts)
    ws = ops.new_workspace(gpu_device, max(1, lib.sdv2_swa_attn_workspace_bytes(rows, S, H, L, 2)))
    p.num_splits, p.mask_block_tokens, p.chunk_key_start_host = 0, block, C.cast(host, C.POINTER(C.c_int64))
    p.q, p.k_cache, p.v_cache = q.data_ptr(), k.data_ptr(), v.data_ptr()
    p.stream = torch.cuda.current_stream().cuda_stream
    for entry, workspace, expected in ((lib.sdv2_swa_attn_fwd_static, None, want), (lib.sdv2_swa_attn_fwd, ws, want),
                                       (lib.sdv2_swa_attn_fwd, None, whole)):
        out = torch.empty_like(q)
        p.out, p.workspace, p.workspace_bytes = out.data_ptr(), None if workspace is None else workspace.data_ptr(), \
            0 if workspace is None else workspace.numel()
        _capi.check(entry(C.byref(p)), "masked, one plan")
        torch.cuda.synchronize()
        assert torch.equal(out, expected)
