"""sdv2_linear, the projections of a chunk as the library's own product: which
calls take it and which keep the vendor's, what the compiler made of its loop,
and its results at the edges of every tile it has."""
import os
import re
import subprocess

import pytest
import torch

from streamdiffusionv2_amd import _capi, build_ext, ops
from test_attention_isa import instructions, registers

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_which_sizes_are_preferred():
    lib = _capi.lib()
    for m, n, k, want in ((1560, 1536, 1536, 1), (256, 4608, 1536, 1), (3120, 1536, 1536, 1), (1, 64, 64, 1),
                          (9360, 1536, 1536, 0), (1560, 4608, 1536, 0), (1560, 5120, 1536, 0),      # more than one round of tiles
                          (256, 5120, 5120, 0),                                                     # a long contraction
                          (0, 64, 64, 0), (16, 96, 64, 0), (16, 64, 96, 0)):
        assert lib.sdv2_linear_preferred(m, n, k) == want, (m, n, k)


def test_what_is_refused():
    """(every refusal comes before the first HIP call)"""
    import ctypes as C

    lib = _capi.lib()

    def status(**more):
        args = dict(x=256, weight=512, out=1024, x_row_stride=128, weight_row_stride=128, out_row_stride=64, m=8, n=64, k=128)
        args.update(more)
        return lib.sdv2_linear(C.byref(_capi.LinearParams(**args)))

    assert lib.sdv2_linear(None) == _capi.SDV2_ERR_INVALID_ARG
    assert status(m=0) == _capi.SDV2_OK
    for bad in (dict(n=96), dict(k=96), dict(dtype=_capi.DTYPE_F32), dict(n=0), dict(k=-64), dict(m=1 << 31)):
        assert status(**bad) == _capi.SDV2_ERR_UNSUPPORTED, bad
    for bad in (dict(m=-1), dict(x=None), dict(out=1032), dict(bias=4), dict(x_row_stride=120), dict(weight_row_stride=132),
                dict(out_row_stride=56), dict(x_row_stride=1 << 23)):
        assert status(**bad) == _capi.SDV2_ERR_INVALID_ARG, bad


def test_calls_that_keep_the_module_s_own_product():
    """Whatever else is going on: autograd, tracing, a function mode, vmap - and tensors on the CPU."""
    with torch.no_grad():
        assert ops._plain_call()
        assert ops.linear_or_none(torch.ones(2, 64).bfloat16(), torch.ones(64, 64).bfloat16(), None) is None
        seen = []
        torch.vmap(lambda t: (seen.append(ops._plain_call()), t)[1])(torch.ones(2, 2))
        torch.jit.trace(lambda t: (seen.append(ops._plain_call()), t * 2)[1], torch.ones(2), check_trace=False)
        with torch.overrides.TorchFunctionMode():
            seen.append(ops._plain_call())
        with torch.utils._python_dispatch.TorchDispatchMode():
            seen.append(ops._plain_call())
        with torch.autograd.forward_ad.dual_level():
            seen.append(ops._plain_call())
        torch.set_autocast_enabled("cuda", True)
        seen.append(ops._plain_call())
        torch.set_autocast_enabled("cuda", False)
        assert seen and not any(seen), seen
    assert not ops._plain_call()


def test_hooked_and_patched_layers_are_called_themselves():
    from streamdiffusionv2_amd.attention import _unwatched

    layer = torch.nn.Linear(64, 64)
    assert _unwatched(layer)
    handle = layer.register_forward_hook(lambda *a: None)
    assert not _unwatched(layer)
    handle.remove()
    handle = torch.nn.modules.module.register_module_forward_pre_hook(lambda *a: None)
    assert not _unwatched(layer)
    handle.remove()
    layer.forward = lambda x: x
    assert not _unwatched(layer)
    assert not _unwatched(type("Adapter", (torch.nn.Linear,), {})(64, 64))


def test_nothing_touches_a_fragment_on_its_way():
    """LDS reads are issued a step ahead of their wait, as assembly: until that wait no instruction may name the
    registers they will land in (a copy the compiler put there would copy what was in them before)."""
    out = os.path.join(ROOT, "build", "isa_check")
    os.makedirs(out, exist_ok=True)
    path = os.path.join(out, "linear.s")
    cmd = [build_ext.hipcc_path(), *build_ext.HIPCC_FLAGS, f"-I{os.path.join(ROOT, 'include')}", f"-I{build_ext.CSRC}",
           "-S", "--cuda-device-only", str(build_ext.CSRC / "linear.hip"), "-o", path]
    res = subprocess.run(cmd, capture_output=True, text=True)
    assert res.returncode == 0, res.stderr[-2000:]
    lines = open(path).read().split("\n")
    starts = [i for i, l in enumerate(lines) if re.match(r"^_Z\S*linear_kernel\S*:", l)]
    assert len(starts) == 6
    for start in starts:
        body = lines[start:next(i for i in range(start, len(lines)) if lines[i].strip().startswith(".Lfunc_end"))]
        # basic blocks, and where each goes
        blocks, label, after = {}, "", {}
        for line in body:
            name = re.match(r"^(\.LBB\d+_\d+|; %bb\.\d+):", line)
            if name:
                after.setdefault(label, []).append(name.group(1))
                label = name.group(1)
            blocks.setdefault(label, []).append(line)
            jump = re.match(r"\s+(s_c?branch\w*|s_endpgm)\s*(\S*)", line)
            if jump and jump.group(2):
                after.setdefault(label, []).append(jump.group(2))
            if jump and jump.group(1) in ("s_branch", "s_endpgm"):
                label = f"dead {len(blocks)}"
        # registers on their way at the start of each block, until nothing changes
        at_start, todo, reads = {"": frozenset()}, [""], 0
        while todo:
            label = todo.pop()
            flying = set(at_start[label])
            for mn, ops_ in instructions(blocks.get(label, [])):
                if mn == "s_waitcnt" and "lgkmcnt(0)" in ops_[0]:
                    flying = set()
                elif mn.startswith("ds_read_b128"):
                    assert not (registers(ops_[0]) | registers(ops_[1])) & flying, (mn, ops_)
                    flying |= registers(ops_[0])
                    reads += 1
                else:
                    assert not any(registers(o) & flying for o in ops_), (mn, ops_)
            for to in after.get(label, []):
                if to not in at_start or not flying <= at_start[to]:
                    at_start[to] = frozenset(flying | at_start.get(to, frozenset()))
                    todo.append(to)
        assert reads >= 12
    text = "\n".join(lines)
    assert not re.search(r"\bscratch_(load|store)", text)
    assert max(int(x) for x in re.findall(r"\.vgpr_count:\s+(\d+)", text)) <= 256


def _check(got, x, w, b):
    """bf16 rounding of a sum of k products in fp32.  bf16 has 8 significant bits: a result in [2^e, 2^(e+1)) is rounded
    by at most half of 2^(e-7), 2^-8 of its magnitude.  Before that, 2^-23 of the sum of magnitudes per addition."""
    x, w = x.double(), w.double()
    want = x @ w.t().contiguous() + (b.double() if b is not None else 0)
    bound = want.abs() * 2.0 ** -8 + (x.abs() @ w.t().abs().contiguous()) * (x.shape[-1] * 2.0 ** -23)
    assert ((got.double() - want).abs() <= bound).all()


@pytest.mark.gpu
@pytest.mark.parametrize("m,n,k", [
    (1, 64, 64), (7, 128, 128), (64, 64, 448), (65, 192, 512), (100, 1536, 1536),          # 64 x 64; fewer stages than fit, and more
    (960, 1536, 384), (865, 1536, 448), (1560, 1536, 320), (1600, 1536, 64),               # 96 x 64; 160 x 64
    (1500, 1792, 256), (2000, 2048, 320), (2048, 2048, 64),                                # 96 x 128; 128 x 128
    (3120, 1536, 1536), (3041, 1536, 64), (3200, 1536, 192),                               # 160 x 128
    (1560, 4608, 192), (3000, 3072, 128),                                                  # more than a round
])
def test_products(gpu_device, m, n, k):
    import ctypes as C

    print(f"linear {m} x {n} x {k}", flush=True)
    gen = torch.Generator(device=gpu_device).manual_seed(m + n + k)
    x, w, b = (torch.randn(*s, generator=gen, device=gpu_device).bfloat16() for s in ((m, k), (n, k), (n,)))
    wide = torch.randn(m, k + 72, generator=gen, device=gpu_device).bfloat16()
    for xx, bb in ((x, b), (wide[:, 8:k + 8], None)):
        out = torch.full((m + 3, n + 8), 7.0, device=gpu_device).bfloat16()                # rows and columns that are not its own
        p = _capi.LinearParams(xx.data_ptr(), w.data_ptr(), bb.data_ptr() if bb is not None else None, out.data_ptr(),
                               xx.stride(0), k, n + 8, m, n, k, _capi.DTYPE_BF16, torch.cuda.current_stream().cuda_stream)
        _capi.check(_capi.lib().sdv2_linear(C.byref(p)), "sdv2_linear")
        torch.cuda.synchronize()
        _check(out[:m, :n], xx, w, bb)
        assert (out[m:] == 7).all() and (out[:, n:] == 7).all()


@pytest.mark.gpu
def test_infinities_and_nans_stay_in_their_row(gpu_device):
    x = torch.randn(200, 256, device=gpu_device).bfloat16()
    w = torch.randn(128, 256, device=gpu_device).bfloat16()
    x[3, 5], x[170, 0], x[199, 255] = float("inf"), float("nan"), float("-inf")
    with torch.no_grad():
        got = ops.linear_or_none(x, w, None)
    bad = [3, 170, 199]
    ok = torch.ones(200, dtype=torch.bool, device=gpu_device)
    ok[bad] = False
    assert not got[bad].isfinite().any() and got[ok].isfinite().all()
    _check(got[ok], x[ok], w, None)


def test_layouts_that_stay_with_the_caller():
    """Rows further apart than the kernel's offsets reach (sdv2_linear refuses them), and what is no product."""
    w = torch.empty(64, 64, dtype=torch.bfloat16)
    flat = torch.empty((1 << 22) + 72, dtype=torch.bfloat16)
    for step, want in ((1 << 22, True), ((1 << 22) + 8, False), (68, False), (0, False)):
        assert (ops._linear_layout(flat.as_strided((2, 64), (step, 1)), w, False) is not None) == want, step
    assert ops._linear_layout(flat[:64], w, False) is None and ops._linear_layout(flat[:32].view(1, 32), w, False) is None
    assert ops._linear_layout(flat[:0].view(0, 64), w, False) is None


def test_results_are_contiguous_whatever_the_strides_of_ones():
    t = torch.empty(4096).as_strided((1, 4, 2, 128), (3, 256, 128, 1))
    assert t.is_contiguous() and ops._empty_as(t).stride() == (1024, 256, 128, 1)
    assert ops._empty_as(t.transpose(1, 2)).stride() == (1024, 512, 128, 1)


@pytest.mark.filterwarnings("ignore:Named tensors")
def test_results_have_no_names():
    assert ops._empty_as(torch.zeros(2, 3, names=("a", "b"))).names == (None, None)


@pytest.mark.gpu
@pytest.mark.filterwarnings("ignore:Sparse CSR")
def test_sparse_operands_stay_with_the_caller(gpu_device):
    """(they have no strides to look at)"""
    x, w = torch.randn(256, 128, device=gpu_device).bfloat16(), torch.eye(128, device=gpu_device).bfloat16()
    with torch.no_grad():
        assert ops.linear_or_none(x, w, None) is not None
        for sparse in (w.to_sparse_csr(), w.to_sparse()):
            assert ops.linear_or_none(x, sparse, None) is None and ops.linear_or_none(sparse, w, None) is None


@pytest.mark.gpu
def test_a_bias_of_another_length_stays_with_the_caller(gpu_device):
    x, w = torch.randn(32, 64, device=gpu_device).bfloat16(), torch.randn(128, 64, device=gpu_device).bfloat16()
    bias = torch.randn(128, device=gpu_device).bfloat16()
    with torch.no_grad():
        _check(ops.linear_or_none(x, w, bias), x, w, bias)
        assert ops.linear_or_none(x, w, bias[:1]) is None and ops.linear_or_none(x, w, bias[:64]) is None


@pytest.mark.gpu
def test_the_modules_take_it(gpu_device):
    """A chunk's q, k, v and o, of a strided input too; one product for q, k and v gives the bits of three (every element
    is the same sum in the same order, whatever the tile)."""
    from streamdiffusionv2_amd.attention import CausalWanSelfAttention, _linear

    torch.manual_seed(8)
    mod = CausalWanSelfAttention(1536, 12).to(gpu_device).bfloat16()
    wide = torch.randn(2, 300, 1536 * 2, device=gpu_device).bfloat16()
    for x in (wide[..., :1536], wide[:, :, 1536:].contiguous()):
        with torch.inference_mode():
            assert ops.linear_or_none(x, mod.o.weight, mod.o.bias) is not None
            _check(_linear(mod.o, x).flatten(0, 1), x.flatten(0, 1), mod.o.weight, mod.o.bias)
            for got, layer in zip(mod.project_qkv(x), (mod.q, mod.k, mod.v)):
                assert torch.equal(got, _linear(layer, x))
        assert ops.linear_or_none(x, mod.o.weight, mod.o.bias) is None            # autograd on
