"""The text cross-attention's query norm inside the attention: the projection leaves sums of squares of 32 columns of its
rows, the attention normalises the raw query as it reads it."""
import ctypes as C

import pytest
import torch

from oracle import sdv2_oracle as oracle
from streamdiffusionv2_amd import _capi


def test_which_calls_fold_the_norm():
    folds = _capi.lib().sdv2_swa_attn_folds_norm
    assert folds(2, 1560, 12, 512) == 1 and folds(2, 1560, 12, 77) == 1 and folds(2, 1560, 12, 704) == 1
    assert folds(2, 1560, 12, 705) == 0                    # 12 key tiles: another kernel
    assert folds(1, 256, 12, 512) == 0                     # few query blocks: the waves share them
    assert folds(0, 1560, 12, 512) == folds(1, 1560, 12, 0) == folds(1, 1560, 0, 512) == 0


def test_what_is_refused():
    """(every refusal comes before the first HIP call)"""
    lib = _capi.lib()

    def status(**more):
        p = _capi.AttnParams(q=256, k_cache=512, v_cache=768, out=1024, rows=2, q_tokens=1560, heads=12, head_dim=128,
                             max_seq_len=512, q_norm_weight=4096, q_row_squares=8192, q_norm_eps=1e-6)
        stride = _capi.Stride3(1560 * 1536, 1536, 128)
        p.q_stride = p.k_stride = p.v_stride = p.out_stride = stride
        for name, value in more.items():
            setattr(p, name, value)
        return lib.sdv2_swa_attn_fwd(C.byref(p))

    invalid, unsupported = _capi.SDV2_ERR_INVALID_ARG, _capi.SDV2_ERR_UNSUPPORTED
    assert status(q_norm_weight=None) == invalid and status(q_inv_rms=4096) == invalid
    assert status(q_norm_weight=4104) == invalid and status(q_row_squares=8196) == invalid
    assert status(q_norm_eps=-1.0) == invalid and status(q_norm_eps=float("nan")) == invalid
    assert status(mask_block_tokens=520, chunk_key_start=4096) == invalid
    assert status(max_seq_len=705) == unsupported and status(rows=1, q_tokens=256) == unsupported
    linear = _capi.LinearParams(x=256, weight=512, out=1024, x_row_stride=64, weight_row_stride=64, out_row_stride=64, m=64,
                                n=64, k=64, dtype=_capi.DTYPE_BF16, row_squares=4098)
    assert lib.sdv2_linear(C.byref(linear)) == invalid


@pytest.mark.gpu
@pytest.mark.parametrize("m,n,k", [(65, 64, 64), (250, 192, 128), (1000, 1536, 256), (1560, 1536, 1536), (3120, 1536, 64), (5000, 1536, 128)])
def test_row_squares(gpu_device, m, n, k):
    """Against the squares of the stored product in float64: 32 terms in fp32, 2^-24 each."""
    torch.manual_seed(9)
    x, w = torch.randn(m, k, device=gpu_device).bfloat16(), torch.randn(n, k, device=gpu_device).bfloat16()
    out = torch.empty(m, n, device=gpu_device, dtype=torch.bfloat16)
    plain = torch.empty_like(out)
    squares = torch.full((m, n // 32), float("nan"), device=gpu_device)
    for dst, sums in ((out, squares.data_ptr()), (plain, None)):
        p = _capi.LinearParams(x.data_ptr(), w.data_ptr(), None, dst.data_ptr(), k, k, n, m, n, k, _capi.DTYPE_BF16,
                               torch.cuda.current_stream().cuda_stream)
        p.row_squares = sums
        _capi.check(_capi.lib().sdv2_linear(C.byref(p)), "sdv2_linear")
    torch.cuda.synchronize()
    want = out.double().pow(2).view(m, n // 32, 32).sum(-1)
    assert torch.equal(out, plain)
    assert ((squares.double() - want).abs() <= 32 * 2.0 ** -24 * want).all()


@pytest.mark.gpu
@pytest.mark.parametrize("rows,S,heads,L,lens", [(2, 1560, 12, 512, None), (1, 3000, 7, 77, None), (2, 1023, 17, 704, [704, 65]),
                                                 (3, 900, 12, 300, [300, 0, 1])])
def test_folded_norm_matches_the_oracle(gpu_device, rows, S, heads, L, lens):
    from streamdiffusionv2_amd import ops

    torch.manual_seed(10)
    width = heads * 128
    raw, weight = torch.randn(rows, S, width).mul(3).bfloat16(), torch.rand(width).add(0.5).bfloat16()
    k, v = torch.randn(rows, L, heads, 128).bfloat16(), torch.randn(rows, L, heads, 128).bfloat16()
    assert _capi.lib().sdv2_swa_attn_folds_norm(rows, S, heads, L)
    xf = raw.float()
    q = (xf * torch.rsqrt(xf.pow(2).mean(-1, keepdim=True) + 1e-6)).bfloat16() * weight
    squares = xf.pow(2).view(rows, S, width // 32, 32).sum(-1).to(gpu_device)
    sl = None if lens is None else torch.tensor(lens, dtype=torch.int32, device=gpu_device)
    got = ops.swa_attention(raw.view(rows, S, heads, 128).to(gpu_device), k.to(gpu_device), v.to(gpu_device), sl,
                            q_row_squares=(weight.to(gpu_device), squares, 1e-6))
    plain = ops.swa_attention(q.view(rows, S, heads, 128).to(gpu_device), k.to(gpu_device), v.to(gpu_device), sl)
    torch.cuda.synchronize()
    # The row's 1 / rms is the same fp32 number but for its last bits: a query element is the same bf16 number or, near a
    # tie, its neighbour.  The same kernel runs on both; a neighbour here and there moves a score by some 2^-9 of it.
    err = (got.float() - plain.float()).abs()
    assert torch.isfinite(got.float()).all() and err.max().item() <= 2e-2 and err.mean().item() <= 1e-5, (err.max(), err.mean())
    live = [r for r in range(rows) if lens is None or lens[r] > 0][:1]
    want = oracle.attention_fp32_reference(q.view(rows, S, heads, 128)[live], k[live], v[live], [L if lens is None else lens[r] for r in live])
    err = (got.cpu()[live].float() - want.float()).abs()
    assert err.max().item() <= 2e-2 and err.mean().item() <= 2e-3, (err.max(), err.mean())


@pytest.mark.gpu
def test_module_folds_only_what_nobody_watches(gpu_device, monkeypatch):
    from streamdiffusionv2_amd import attention, ops

    torch.manual_seed(11)
    module = attention.WanT2VCrossAttention(1536, 12).to(gpu_device).bfloat16()
    x, text = (torch.randn(2, n, 1536, device=gpu_device).bfloat16() for n in (1560, 512))
    norms = []
    plain = ops.rms_norm_or_none
    monkeypatch.setattr(ops, "rms_norm_or_none", lambda t, *a: (norms.append(tuple(t.shape)), plain(t, *a))[1])
    query = (2, 1560, 1536)
    with torch.no_grad():
        cache = {"is_init": False}
        first, later = module(x, text, None, cache), module(x, text, None, cache)
        assert torch.equal(first, later) and query not in norms
        assert torch.equal(module(x, text, None), first)
        handle = module.norm_q.register_forward_hook(lambda *_: None)
        watched = module(x, text, None, cache)
        handle.remove()
        assert norms.count(query) == 1
        assert (watched.float() - first.float()).abs().max() <= 2e-2 * max(1.0, first.float().abs().max().item())
        short = module(x[:1, :256], text[:1], None)            # another kernel: the norm's own launch
        assert (1, 256, 1536) in norms and torch.isfinite(short.float()).all()
        # keys that are not bf16, from projections that have no weight of their own: cast, as without the fold
        module.norm_k.float()
        inner = module.v
        module.v = torch.nn.Sequential(inner)
        mixed = module(x, text, None)
        module.norm_k.bfloat16()
        module.v = inner
        assert norms.count(query) == 1 and (mixed.float() - first.float()).abs().max() <= 2e-2 * max(1.0, first.float().abs().max().item())
    module(x, text, None).sum()                                # autograd: the module's own expression
    assert norms.count(query) == 1


@pytest.mark.gpu
@pytest.mark.parametrize("rows,S,heads,L,lens", [(1, 200, 40, 100, None), (2, 97, 63, 65, [65, 3]), (1, 161, 64, 77, None),
                                                 (1, 129, 67, 64, None)])
def test_folded_norm_of_many_heads(gpu_device, rows, S, heads, L, lens):
    """Sums of more heads than one trip brings (40), of as many as a wave's part of LDS holds (64), and of more; few rows, so
    that the last block of a query tile is short."""
    test_folded_norm_matches_the_oracle(gpu_device, rows, S, heads, L, lens)
