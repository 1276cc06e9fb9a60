"""Operator-level Python surface over the sdv2kv C ABI.

``flash_attn_with_kvcache`` keeps the four-argument call the reference makes
(models/wan/causal_model.py:353-358); ``kv_append_rope`` is the fused
replacement for causal_rope_apply + the per-row slice writes (:253-266,
:321-342).  PyTorch supplies device memory and the current stream only.
"""
from __future__ import annotations

import ctypes as C
from typing import Optional, Sequence, Tuple

import torch

from . import _capi

HEAD_DIM = _capi.HEAD_DIM

_DTYPES = {torch.bfloat16: _capi.DTYPE_BF16, torch.float32: _capi.DTYPE_F32}


def _require_gpu(*tensors: torch.Tensor) -> torch.device:
    dev = tensors[0].device
    for t in tensors:
        if t is None:
            continue
        if not t.is_cuda:
            raise RuntimeError(
                "sdv2kv operators run on the GPU only (tensor on %s); there is no CPU path" % t.device
            )
        if t.device != dev:
            raise RuntimeError(f"tensors on different devices: {t.device} vs {dev}")
    return dev


def _stride3(t: torch.Tensor, name: str) -> _capi.Stride3:
    if t.dim() != 4 or t.shape[-1] != HEAD_DIM:
        raise RuntimeError(f"{name}: expected [rows, tokens, heads, {HEAD_DIM}], got {tuple(t.shape)}")
    if t.shape[-1] > 1 and t.stride(-1) != 1:
        raise RuntimeError(f"{name}: last dimension must be contiguous (stride {t.stride(-1)})")
    return _capi.Stride3(t.stride(0), t.stride(1), t.stride(2))


def _stream_ptr(dev: torch.device) -> int:
    # (the handle itself; torch.cuda.current_stream() wraps it in an object first, three microseconds a call)
    index = dev.index
    return torch._C._cuda_getCurrentRawStream(torch.cuda.current_device() if index is None else index)


def _empty_as(t: torch.Tensor) -> torch.Tensor:
    """A contiguous plain tensor of t's shape, dtype and device."""
    if type(t) is torch.Tensor and t.is_contiguous() and not t.has_names():
        # (a third of the time it takes to spell them out; by itself it would take over odd strides of dimensions of one)
        return torch.empty_like(t, memory_format=torch.contiguous_format)
    return torch.empty(t.shape, dtype=t.dtype, device=t.device)


class _NoSwitch:
    def __enter__(self):
        return self

    def __exit__(self, *exc):
        return False


_NO_SWITCH = _NoSwitch()


def _on_device(dev: torch.device):
    """Context in which ``dev`` is the current device: torch's guard when it is
    another one, nothing at all (the usual case, and several microseconds less
    per call) when it already is."""
    return _NO_SWITCH if torch.cuda.current_device() == dev.index else torch.cuda.device(dev)


def _i64_array(values: Sequence[int]):
    return (C.c_int64 * len(values))(*[int(v) for v in values])


_FREQS_CACHE: dict = {}


def device_freqs(freqs: torch.Tensor, device: torch.device) -> torch.Tensor:
    """The complex128 [rows, 64] RoPE table as float64 [rows, 64, 2] on
    ``device``.  Converted once per (table, device)."""
    try:
        version = freqs._version
    except RuntimeError:            # created under torch.inference_mode(): no edit counter
        version = None
    key = (id(freqs), version, freqs.data_ptr(), device)
    hit = _FREQS_CACHE.get(key)
    if hit is not None and hit[0] is freqs:
        return hit[1]
    if freqs.dtype != torch.complex128 or freqs.dim() != 2 or freqs.shape[1] != HEAD_DIM // 2:
        raise RuntimeError(
            f"freqs must be complex128 [rows, {HEAD_DIM // 2}], got {freqs.dtype} {tuple(freqs.shape)}"
        )
    table = torch.view_as_real(freqs.detach().resolve_conj()).contiguous().to(device)
    if len(_FREQS_CACHE) > 8:
        _FREQS_CACHE.clear()
    _FREQS_CACHE[key] = (freqs, table)
    return table


def _check_norm(qk_norm, dtype, heads: int, dev) -> None:
    wq, wk, eps = qk_norm
    for w in (wq, wk):
        if w.dtype != dtype or w.numel() != heads * HEAD_DIM or not w.is_contiguous() or w.device != dev:
            raise RuntimeError(f"norm weights must be contiguous {dtype} tensors of {heads * HEAD_DIM} elements on {dev}")
    if not eps >= 0:
        raise RuntimeError("norm eps must be >= 0")


def _check_override(t: torch.Tensor, rows: int, dev) -> None:
    if t.dtype != torch.int64 or t.numel() < rows or not t.is_contiguous() or t.device != dev:
        raise RuntimeError(f"dst_start_override must be a contiguous int64 tensor with one entry per row on {dev}")


def kv_append_rope(
    q: Optional[torch.Tensor],
    k: torch.Tensor,
    v: torch.Tensor,
    k_cache: torch.Tensor,
    v_cache: torch.Tensor,
    freqs_table: torch.Tensor,
    grid: Tuple[int, int, int],
    start_frames: Sequence[int],
    dst_starts: Sequence[int],
    q_out: Optional[torch.Tensor] = None,
    global_end_index: Optional[torch.Tensor] = None,
    local_end_index: Optional[torch.Tensor] = None,
    new_global_end: Optional[Sequence[int]] = None,
    new_local_end: Optional[Sequence[int]] = None,
    qk_norm: Optional[Tuple[torch.Tensor, torch.Tensor, float]] = None,
    dst_start_override: Optional[torch.Tensor] = None,
    q_inv_rms: Optional[torch.Tensor] = None,
) -> Optional[torch.Tensor]:
    """RoPE q and k, write k' and v into the cache at ``dst_starts`` and store
    the new end indices.  Returns the roped query (``q_out`` or a new tensor).

    ``dst_start_override`` (device int64 [B], written by
    :func:`sink_similarity`) replaces ``dst_starts[i]`` where it holds a value
    >= 0.

    ``qk_norm`` = (q weight, k weight, eps) folds the WanRMSNorm of the
    projection outputs in (wan_base/modules/model.py:70-86): q and k are then
    the raw projection outputs.  With ``q_inv_rms`` (float32 [B, S] on the
    device) the kernel stores 1 / rms of every q token there and writes NO
    rotated query (returns None): :func:`swa_attention` takes the raw q with
    ``q_norm=(q weight, q_inv_rms)`` and normalises and rotates it itself.

    ``freqs_table`` is :func:`device_freqs` output.  Rows are processed in
    groups of at most 16 per launch.
    """
    dev = _require_gpu(k, v, k_cache, v_cache, freqs_table, q, q_out, global_end_index, local_end_index)
    if k.dtype not in _DTYPES:
        raise RuntimeError(f"unsupported dtype {k.dtype}")
    for t in (q, v, k_cache, v_cache, q_out):
        if t is not None and t.dtype != k.dtype:
            raise RuntimeError(f"dtype mismatch: {t.dtype} vs {k.dtype}")
    rows, tokens, heads, _ = k.shape
    if q_inv_rms is not None:
        if qk_norm is None or q is None or q_out is not None:
            raise RuntimeError("q_inv_rms goes with qk_norm and q, and replaces q_out")
        if q_inv_rms.dtype != torch.float32 or q_inv_rms.numel() != rows * tokens or not q_inv_rms.is_contiguous() \
                or q_inv_rms.device != dev:
            raise RuntimeError(f"q_inv_rms must be a contiguous float32 tensor of {rows} x {tokens} elements on {dev}")
    elif q is not None and q_out is None:
        q_out = torch.empty((rows, tokens, heads, HEAD_DIM), dtype=q.dtype, device=dev)
    for name, t in (("q", q), ("v", v), ("q_out", q_out)):
        if t is not None and tuple(t.shape) != tuple(k.shape):
            raise RuntimeError(f"{name} shape {tuple(t.shape)} differs from k {tuple(k.shape)}")
    if k_cache.shape[0] < rows or v_cache.shape != k_cache.shape or k_cache.shape[2] != heads:
        raise RuntimeError(f"cache shape {tuple(k_cache.shape)} / {tuple(v_cache.shape)} does not fit k {tuple(k.shape)}")
    if len(start_frames) != rows or len(dst_starts) != rows:
        raise RuntimeError("start_frames and dst_starts need one entry per row")
    for idx in (global_end_index, local_end_index):
        if idx is not None and (idx.dtype != torch.int64 or idx.numel() < rows or not idx.is_contiguous()):
            raise RuntimeError("end-index tensors must be contiguous int64 with one entry per row")
    if freqs_table.dtype != torch.float64 or not freqs_table.is_contiguous():
        raise RuntimeError("freqs_table must be the contiguous float64 view from device_freqs()")
    if qk_norm is not None:
        _check_norm(qk_norm, k.dtype, heads, dev)
        if q is None:
            raise RuntimeError("the fused q/k norm needs q")
    if dst_start_override is not None:
        _check_override(dst_start_override, rows, dev)

    lib = _capi.lib()
    stream = _stream_ptr(dev)
    with _on_device(dev):
        for r0 in range(0, rows, _capi.MAX_ROWS):
            r1 = min(rows, r0 + _capi.MAX_ROWS)
            p = _capi.AppendParams()
            sl = slice(r0, r1)
            if q is not None:
                p.q_in, p.q_in_stride = q[sl].data_ptr(), _stride3(q, "q")
                if q_out is not None:
                    p.q_out, p.q_out_stride = q_out[sl].data_ptr(), _stride3(q_out, "q_out")
                else:
                    p.q_inv_rms = q_inv_rms.data_ptr() + 4 * r0 * tokens
            p.k_in, p.k_in_stride = k[sl].data_ptr(), _stride3(k, "k")
            p.v_in, p.v_in_stride = v[sl].data_ptr(), _stride3(v, "v")
            p.k_cache, p.k_cache_stride = k_cache[sl].data_ptr(), _stride3(k_cache, "k_cache")
            p.v_cache, p.v_cache_stride = v_cache[sl].data_ptr(), _stride3(v_cache, "v_cache")
            p.freqs = freqs_table.data_ptr()
            p.freq_rows = freqs_table.shape[0]
            p.dtype = _DTYPES[k.dtype]
            p.rows, p.tokens, p.heads, p.head_dim = r1 - r0, tokens, heads, HEAD_DIM
            p.grid_f, p.grid_h, p.grid_w = (int(x) for x in grid)
            p.cache_tokens = k_cache.shape[1]
            sf = _i64_array(start_frames[r0:r1])
            ds = _i64_array(dst_starts[r0:r1])
            p.start_frame = C.cast(sf, C.POINTER(C.c_int64))
            p.dst_start = C.cast(ds, C.POINTER(C.c_int64))
            if global_end_index is not None or local_end_index is not None:
                if new_global_end is None or new_local_end is None:
                    raise RuntimeError("new_global_end/new_local_end are required with the index tensors")
                ng = _i64_array(new_global_end[r0:r1])
                nl = _i64_array(new_local_end[r0:r1])
                p.new_global_end = C.cast(ng, C.POINTER(C.c_int64))
                p.new_local_end = C.cast(nl, C.POINTER(C.c_int64))
                if global_end_index is not None:
                    p.global_end_index = global_end_index.data_ptr() + 8 * r0
                if local_end_index is not None:
                    p.local_end_index = local_end_index.data_ptr() + 8 * r0
            p.stream = stream
            if qk_norm is not None:
                p.q_norm_weight, p.k_norm_weight = qk_norm[0].data_ptr(), qk_norm[1].data_ptr()
                p.norm_eps = float(qk_norm[2])
            if dst_start_override is not None:
                p.dst_start_override = dst_start_override.data_ptr() + 8 * r0
            _capi.check(lib.sdv2_kv_append_rope(C.byref(p)), "sdv2_kv_append_rope")
    return q_out


def causal_rope_apply(x: torch.Tensor, grid_sizes, freqs: torch.Tensor, start_frame=0, rope_cache=None) -> torch.Tensor:
    """The reference's ``causal_rope_apply`` (causal_model.py:94-108) as one
    launch per run of rows with the same grid: row i of ``x`` [B, L, H, 128]
    is rotated over its first f*h*w tokens for ``grid_sizes[i]`` = (f, h, w)
    starting at frame ``start_frame`` (an int, or one entry per row); later
    tokens and rows without a grid are returned as they are.  Bit-identical to
    the reference's complex128 product rounded to ``x``'s dtype.

    ``freqs`` is the model's complex128 table or :func:`device_freqs` output.
    ``rope_cache`` (the reference's pre-expanded per-token factors) is accepted
    and not used: the kernel indexes the table itself.  The KV-cache path does
    not call this: its append rotates q and k while it writes the cache.
    """
    dev = _require_gpu(x)
    if x.dtype not in _DTYPES:
        raise RuntimeError(f"unsupported dtype {x.dtype}")
    rows, length, heads, _ = x.shape
    grids = grid_sizes.tolist() if isinstance(grid_sizes, torch.Tensor) else [list(g) for g in grid_sizes]
    grids = [tuple(int(n) for n in g) for g in grids][:rows]
    if isinstance(start_frame, torch.Tensor):
        starts = [int(s) for s in start_frame.reshape(-1).tolist()][:len(grids)]
        grids = grids[:len(starts)]                    # the reference zips the two
    else:
        starts = [int(start_frame)] * len(grids)
    for f, h, w in grids:
        if min(f, h, w) <= 0 or f * h * w > length:
            raise RuntimeError(f"grid {(f, h, w)} does not fit {length} tokens")
    table = freqs if freqs.dtype == torch.float64 and freqs.device == dev else device_freqs(freqs, dev)
    if table.dim() != 3 or tuple(table.shape[1:]) != (HEAD_DIM // 2, 2) or not table.is_contiguous():
        raise RuntimeError("freqs must be the complex128 table or the float64 view from device_freqs()")
    _stride3(x, "x")
    whole = len(grids) == rows and all(f * h * w == length for f, h, w in grids)
    out = torch.empty_like(x) if whole else x.clone()
    if out.stride() != x.stride():
        raise RuntimeError("x must be dense (its copy did not keep the strides)")

    lib = _capi.lib()
    with _on_device(dev):
        r0 = 0
        while r0 < len(grids):
            r1 = r0 + 1
            while r1 < len(grids) and r1 - r0 < _capi.MAX_ROWS and grids[r1] == grids[r0]:
                r1 += 1
            f, h, w = grids[r0]
            p = _capi.AppendParams()
            p.q_in, p.q_in_stride = x[r0:r1].data_ptr(), _stride3(x, "x")
            p.q_out, p.q_out_stride = out[r0:r1].data_ptr(), _stride3(out, "out")
            p.freqs, p.freq_rows = table.data_ptr(), table.shape[0]
            p.dtype = _DTYPES[x.dtype]
            p.rows, p.tokens, p.heads, p.head_dim = r1 - r0, f * h * w, heads, HEAD_DIM
            p.grid_f, p.grid_h, p.grid_w = f, h, w
            sf = _i64_array(starts[r0:r1])
            p.start_frame = C.cast(sf, C.POINTER(C.c_int64))
            p.stream = _stream_ptr(dev)
            _capi.check(lib.sdv2_kv_append_rope(C.byref(p)), "sdv2_kv_append_rope")
            r0 = r1
    return out


_WORKSPACES: dict = {}
_CAPTURED_WORKSPACES: list = []       # (at most one per stream and growth step of its buffer)


def _capturing(dev: torch.device) -> bool:
    return dev.type == "cuda" and torch.cuda.is_current_stream_capturing()


TICKET_BYTES = 65536          # head of an attention workspace (256 bytes for a sink-similarity one)


def new_workspace(dev: torch.device, nbytes: int) -> torch.Tensor:
    """A split-KV workspace as the library wants it: zero-filled once (its
    ticket words start at zero and every call leaves them there).  Only
    buffers made here are accepted as ``workspace=``: a ticket word that does
    not start at zero makes a split call combine early or never, silently."""
    ws = torch.zeros(max(nbytes, 1), dtype=torch.uint8, device=dev)
    ws._sdv2_workspace = True
    return ws


def reset_workspace_tickets(dev: torch.device) -> None:
    """Zero the ticket words of this stream's workspaces again.  Every call
    that completes leaves them at zero; after a launch that failed on the
    device they may not be."""
    if dev.type != "cuda" or not (_WORKSPACES or _SIM_WORKSPACES):
        return
    key = (dev, _stream_ptr(dev))
    for pool in (_WORKSPACES, _SIM_WORKSPACES):
        ws = pool.get(key)
        if ws is not None:
            ws[:TICKET_BYTES].zero_()


def _workspace(dev: torch.device, nbytes: int, pool: Optional[dict] = None, stream: Optional[int] = None) -> torch.Tensor:
    """Scratch for split-KV partials, one buffer per (device, stream), grown on
    demand and reused.  Calls on one stream run one after another, so they can
    share a buffer; calls on different streams may overlap in time and must not
    (their tickets and partial results would mix), so each stream gets its own.

    Under capture: a buffer that is there already is never freed again, however
    the pool grows (the graph writes to it at every replay); one made inside the
    capture is the graph's own and not filed (its zeros are part of the graph,
    and nothing has filled it yet)."""
    pool = _WORKSPACES if pool is None else pool
    key = (dev, _stream_ptr(dev) if stream is None else stream)
    ws = pool.get(key)
    if ws is not None and ws.numel() >= nbytes:
        if _capturing(dev) and not any(ws is kept for kept in _CAPTURED_WORKSPACES):
            _CAPTURED_WORKSPACES.append(ws)
        return ws
    ws = new_workspace(dev, nbytes)
    if not _capturing(dev):
        pool[key] = ws
    return ws


def _check_chunk_starts(starts, rows: int, q_tokens: int, max_seq_len: int) -> None:
    if starts is None or len(starts) != rows:
        raise RuntimeError("mask_block_tokens needs chunk_key_start with one entry per row")
    for x in starts:
        if x < 0 or x + q_tokens > max_seq_len:
            raise RuntimeError(f"chunk_key_start {x} puts the chunk outside the {max_seq_len}-key view")


def chunk_starts_tensor(starts, rows: int, q_tokens: int, max_seq_len: int, dev) -> torch.Tensor:
    """Per-row cache position of the chunk's own keys as the int32 device
    tensor the attention kernel reads; host values are range-checked here."""
    if isinstance(starts, torch.Tensor):
        if starts.dtype != torch.int32 or starts.numel() != rows or starts.device != dev or not starts.is_contiguous():
            raise RuntimeError("chunk_key_start must be a contiguous int32 device tensor with one entry per row")
        return starts
    _check_chunk_starts(starts, rows, q_tokens, max_seq_len)
    return torch.tensor([int(x) for x in starts], dtype=torch.int32).to(dev, non_blocking=True)


# Descriptors of the attention calls seen, everything filled in that shapes, strides and dtypes decide: checking
# and filling them costs more host time than the rest of a call, and a program has a handful of layouts.
_ATTN_LAYOUTS: dict = {}
_MAX_ATTN_LAYOUTS = 256


def _library_plan(lib, rows: int, q_tokens: int, heads: int, max_seq_len: int, even: bool, mask_block_tokens: int,
                  starts_alike: bool) -> int:
    """num_splits as the library picks it; ``even``: equal shares of the key tiles are among what it may pick."""
    plan = lib.sdv2_swa_attn_plan_masked(rows, q_tokens, heads, max_seq_len, mask_block_tokens, starts_alike)
    if plan == _capi.SPLITS_EVEN and not even:
        return lib.sdv2_swa_attn_default_splits(rows, q_tokens, heads, max_seq_len)
    return plan


def _starts_alike(starts) -> bool:
    """Do all rows' chunks start at the same key, as host values that travel in the launch's arguments say?"""
    return starts is not None and not isinstance(starts, torch.Tensor) and 0 < len(starts) <= _capi.MAX_ROWS \
        and all(x == starts[0] for x in starts)


def _attn_layout(q, k_cache, v_cache, out, num_splits: int, static_scratch: bool, rope: bool, mask_block_tokens: int = 0,
                 starts_alike: bool = False):
    """(descriptor as bytes, workspace bytes it needs, rows, query tokens, heads, keys)."""
    if q.dtype not in _DTYPES or k_cache.dtype != q.dtype or v_cache.dtype != q.dtype:
        raise RuntimeError("swa_attention takes q and both caches in one dtype, bf16 or fp32; got %s/%s/%s"
                           % (q.dtype, k_cache.dtype, v_cache.dtype))
    fp32 = q.dtype == torch.float32
    if fp32 and (rope or static_scratch):
        raise RuntimeError("fp32 attention takes rotated queries (no rope=) and no static_scratch=")
    rows, q_tokens, heads, _ = q.shape
    if k_cache.shape[0] != rows or k_cache.shape[2] != heads or v_cache.shape != k_cache.shape:
        raise RuntimeError(f"cache view {tuple(k_cache.shape)} / {tuple(v_cache.shape)} does not match q {tuple(q.shape)}")
    lib = _capi.lib()
    max_seq_len = k_cache.shape[1]
    if fp32:
        need = lib.sdv2_swa_attn_f32_workspace_bytes(rows, q_tokens, heads, max_seq_len)    # (it picks its own splits)
    else:
        if num_splits <= 0:
            # (the static entry point has no room for equal shares, and their workgroups rotate no queries)
            num_splits = _library_plan(lib, rows, q_tokens, heads, max_seq_len, not (static_scratch or rope),
                                       mask_block_tokens, starts_alike)
        need = 0 if static_scratch else lib.sdv2_swa_attn_workspace_bytes(rows, q_tokens, heads, max_seq_len, num_splits)
    p = _capi.AttnParams()
    p.q_stride = _stride3(q, "q")
    p.k_stride, p.v_stride = _stride3(k_cache, "k_cache"), _stride3(v_cache, "v_cache")
    p.out_stride = _stride3(out, "out") if out is not None else \
        _capi.Stride3(q_tokens * heads * HEAD_DIM, heads * HEAD_DIM, HEAD_DIM)
    p.rows, p.q_tokens, p.heads, p.head_dim = rows, q_tokens, heads, HEAD_DIM
    p.max_seq_len = max_seq_len
    p.num_splits = num_splits
    p.dtype = _DTYPES[q.dtype]
    return bytes(p), need, rows, q_tokens, heads, max_seq_len


def swa_attention(
    q: torch.Tensor,
    k_cache: torch.Tensor,
    v_cache: torch.Tensor,
    seq_lens: Optional[torch.Tensor] = None,
    out: Optional[torch.Tensor] = None,
    num_splits: int = 0,
    softmax_scale: Optional[float] = None,
    workspace: Optional[torch.Tensor] = None,
    chunk_key_start: Optional[torch.Tensor] = None,
    mask_block_tokens: int = 0,
    static_scratch: bool = False,
    rope: Optional[Tuple[torch.Tensor, Sequence[int], Sequence[int]]] = None,
    q_norm: Optional[Tuple[torch.Tensor, torch.Tensor]] = None,
    q_row_squares: Optional[Tuple[torch.Tensor, torch.Tensor, float]] = None,
) -> torch.Tensor:
    """out[b] = softmax(q[b] k_cache[b,:seq_lens[b]]^T * scale) v_cache[b,:seq_lens[b]].

    ``rope`` = (:func:`device_freqs` table, (grid_h, grid_w), start frame per
    row): q is the query BEFORE RoPE and is rotated inside the kernel exactly as
    :func:`kv_append_rope` would have rotated it (S must be whole frames).  A
    caller-owned ``workspace`` must come from :func:`new_workspace` (zero-filled).
    With ``q_norm`` = (q norm weight, q_inv_rms from :func:`kv_append_rope`) as
    well, q is the raw q projection and is RMS-normalised before the rotation.
    ``q_row_squares`` = (q norm weight, sums of squares of 32 columns each of q as
    :func:`linear_or_none` stores them, eps): q is a raw projection, normalised and
    not rotated, for shapes that ``sdv2_swa_attn_folds_norm`` names.

    ``static_scratch`` takes the library's allocation-free entry point
    (``sdv2_swa_attn_fwd_static``): partial results of a split call go to device
    memory the library holds itself (64 MiB per GPU, shared by all calls on
    that GPU), no workspace is sized or allocated here; with ``out`` given the
    whole call then allocates nothing.

    q [B,S,H,128] bf16; k_cache/v_cache [B,L,H,128] bf16 views with any row /
    token / head strides; seq_lens int32 [B] on the device (None = L).  All
    three may be fp32 instead (the reference's CPU-runnable configuration): the
    result is then computed in fp32 throughout, on the fp32 matrix instructions
    (q rotated beforehand, ``num_splits`` ignored).
    With ``mask_block_tokens`` = b in (0, S) and ``chunk_key_start`` (int32 [B]
    on the device, or host ints: where each row's own chunk sits in the cache)
    query token t does not see the chunk's later blocks
    [start + (t // b + 1) * b, start + S).
    """
    dev = _require_gpu(q, k_cache, v_cache, seq_lens, out, workspace)
    if out is not None and (out.dtype != q.dtype or out.shape != q.shape):
        raise RuntimeError("out must have q's dtype and shape")
    mask_block_tokens = int(mask_block_tokens)
    alike = bool(mask_block_tokens) and _starts_alike(chunk_key_start)
    key = (q.shape, q.stride(), q.dtype, k_cache.shape, k_cache.stride(), k_cache.dtype, v_cache.shape, v_cache.stride(),
           v_cache.dtype, None if out is None else out.stride(), num_splits, static_scratch, rope is None, mask_block_tokens,
           alike)
    layout = _ATTN_LAYOUTS.get(key)
    if layout is None:
        layout = _attn_layout(q, k_cache, v_cache, out, num_splits, static_scratch, rope is not None,
                              mask_block_tokens, alike)
        if len(_ATTN_LAYOUTS) >= _MAX_ATTN_LAYOUTS:
            _ATTN_LAYOUTS.clear()
        _ATTN_LAYOUTS[key] = layout
    template, need, rows, q_tokens, heads, max_seq_len = layout
    if seq_lens is not None and (seq_lens.dtype != torch.int32 or seq_lens.numel() != rows or not seq_lens.is_contiguous()):
        raise RuntimeError("seq_lens must be a contiguous int32 tensor with one entry per row")
    if out is None:
        out = _empty_as(q)

    lib = _capi.lib()
    stream = _stream_ptr(dev)
    if workspace is not None and not getattr(workspace, "_sdv2_workspace", False):
        raise RuntimeError("workspace= takes a buffer made by ops.new_workspace() (zero-filled ticket words)")
    if need and (workspace is None or workspace.numel() * workspace.element_size() < need):
        workspace = _workspace(dev, need, stream=stream)

    p = _capi.AttnParams.from_buffer_copy(template)
    p.q, p.k_cache, p.v_cache, p.out = q.data_ptr(), k_cache.data_ptr(), v_cache.data_ptr(), out.data_ptr()
    if seq_lens is not None:
        p.seq_lens = seq_lens.data_ptr()
    if softmax_scale:
        p.softmax_scale = float(softmax_scale)
    if need:
        p.workspace = workspace.data_ptr()
        p.workspace_bytes = workspace.numel() * workspace.element_size()
    p.stream = stream
    if mask_block_tokens:
        p.mask_block_tokens = mask_block_tokens
        if isinstance(chunk_key_start, torch.Tensor) or rows > _capi.MAX_ROWS:
            chunk_key_start = chunk_starts_tensor(chunk_key_start, rows, q_tokens, max_seq_len, dev)
            p.chunk_key_start = chunk_key_start.data_ptr()
        else:
            # host values travel in the launch's arguments
            _check_chunk_starts(chunk_key_start, rows, q_tokens, max_seq_len)
            key_starts = _i64_array(chunk_key_start)
            p.chunk_key_start_host = C.cast(key_starts, C.POINTER(C.c_int64))
    if rope is not None:
        table, grid_hw, start_frames = rope
        if table.dtype != torch.float64 or not table.is_contiguous() or table.device != dev:
            raise RuntimeError("rope table must be the contiguous float64 view from device_freqs() on q's device")
        if len(start_frames) != rows:
            raise RuntimeError("rope needs one start frame per row")
        frames = _i64_array(start_frames)
        p.rope_freqs, p.rope_freq_rows = table.data_ptr(), table.shape[0]
        p.rope_grid_h, p.rope_grid_w = int(grid_hw[0]), int(grid_hw[1])
        p.rope_start_frame = C.cast(frames, C.POINTER(C.c_int64))
    if q_norm is not None:
        weight, inv_rms = q_norm
        if rope is None:
            raise RuntimeError("q_norm needs rope=: the kernel normalises the raw query, then rotates it")
        if weight.dtype != q.dtype or weight.numel() != heads * HEAD_DIM or not weight.is_contiguous() or weight.device != dev:
            raise RuntimeError(f"the q norm weight must be a contiguous {q.dtype} tensor of {heads * HEAD_DIM} elements on {dev}")
        if inv_rms.dtype != torch.float32 or inv_rms.numel() != rows * q_tokens or not inv_rms.is_contiguous() \
                or inv_rms.device != dev:
            raise RuntimeError(f"q_inv_rms must be a contiguous float32 tensor of {rows} x {q_tokens} elements on {dev}")
        p.q_norm_weight, p.q_inv_rms = weight.data_ptr(), inv_rms.data_ptr()
    if q_row_squares is not None:
        weight, squares, eps = q_row_squares
        if weight.dtype != q.dtype or weight.numel() != heads * HEAD_DIM or not weight.is_contiguous() or weight.device != dev:
            raise RuntimeError(f"the q norm weight must be a contiguous {q.dtype} tensor of {heads * HEAD_DIM} elements on {dev}")
        if squares.dtype != torch.float32 or squares.numel() != rows * q_tokens * heads * HEAD_DIM // 32 \
                or not squares.is_contiguous() or squares.device != dev:
            raise RuntimeError(f"q_row_squares must be a contiguous float32 tensor of {rows} x {q_tokens} x {heads * 4} elements on {dev}")
        p.q_norm_weight, p.q_row_squares, p.q_norm_eps = weight.data_ptr(), squares.data_ptr(), eps
    with _on_device(dev):
        if static_scratch:
            _capi.check(lib.sdv2_swa_attn_fwd_static(C.byref(p)), "sdv2_swa_attn_fwd_static")
        else:
            _capi.check(lib.sdv2_swa_attn_fwd(C.byref(p)), "sdv2_swa_attn_fwd")
    return out


def query_beside_decision(rows: int, tokens: int, heads: int, norm: bool) -> bool:
    """Should the query be rotated by the sink decision's launch (``sink_similarity(query=...)``) and the append behind it
    move K and V only?  The workgroups that rotate are next to free while the decision waits on its trips to memory; where
    its sums fill the chip's bandwidth they hold those up, the more with the norm of more than sixteen heads, whose waves
    take one token at a time.  Both launches together, beside / in the append, 41 shapes each way: up to 160 000
    (token, head) pairs 0.83 to 0.97 (2 x 1560 x 12 with the norm 29.7 / 35.8 us, 1 x 3600 x 40 94.9 / 101.7); above,
    norm of more than 16 heads 0.97 to 1.14 (4 x 1560 x 40 171 / 164, 4 x 3600 x 40 320 / 291); the others 0.87 to 0.99
    up to 240 000 (4 x 3600 x 12 with the norm 96 / 110) and 0.94 to 1.05 above (8 x 1560 x 20 without 152 / 147)."""
    return rows * tokens * heads <= (160_000 if norm and heads > 16 else 240_000)


_SIM_WORKSPACES: dict = {}
_SIM_LAYOUTS: dict = {}


def _sim_layout(lib, k, v, k_cache, v_cache, freq_rows: int, grid_hw, sink_frames: int, q, q_out):
    """What a sink decision of these shapes and strides passes down whatever the pointers: the descriptor with all
    else filled in, and the bytes of its workspace and of the kept means.  (Filled anew it was 15 us of the call.)"""
    if not (k.dtype == v.dtype == k_cache.dtype == v_cache.dtype):
        raise RuntimeError("k, v and the caches must share one dtype")
    rows, tokens, heads, _ = k.shape
    if tuple(v.shape) != tuple(k.shape):
        raise RuntimeError("k and v must have one shape")
    if k_cache.shape[0] < rows or v_cache.shape != k_cache.shape or k_cache.shape[2] != heads:
        raise RuntimeError(f"cache {tuple(k_cache.shape)} does not match the chunk {tuple(k.shape)}")
    p = _capi.SinkSimParams()
    p.k_in_stride, p.v_in_stride = _stride3(k, "k"), _stride3(v, "v")
    p.k_cache_stride, p.v_cache_stride = _stride3(k_cache, "k_cache"), _stride3(v_cache, "v_cache")
    p.freq_rows = freq_rows
    if k.dtype not in _DTYPES:
        raise RuntimeError(f"unsupported dtype {k.dtype}")
    p.dtype = _DTYPES[k.dtype]
    p.rows, p.tokens, p.heads, p.head_dim = rows, tokens, heads, HEAD_DIM
    p.grid_h, p.grid_w = grid_hw
    p.sink_frames = sink_frames
    p.cache_tokens = k_cache.shape[1]
    if q is not None:
        if q.shape != k.shape or q_out.shape != k.shape or not q.dtype == q_out.dtype == k.dtype:
            raise RuntimeError("query and rotated query must have the key's shape and dtype")
        p.q_in_stride, p.q_out_stride = _stride3(q, "q"), _stride3(q_out, "rotated q")
    return p, lib.sdv2_sink_similarity_workspace_bytes(rows, tokens, heads, sink_frames), \
        lib.sdv2_sink_frame_sums_bytes(rows, heads, sink_frames)


def sink_similarity(
    k: torch.Tensor,
    v: torch.Tensor,
    k_cache: torch.Tensor,
    v_cache: torch.Tensor,
    freqs_table: torch.Tensor,
    grid_hw: Sequence[int],
    start_frames: Sequence[int],
    sink_frames: int,
    threshold: float,
    dst_start_override: Optional[torch.Tensor] = None,
    override_rows: Sequence[bool] = (),
    refresh_out: Optional[torch.Tensor] = None,
    k_norm: Optional[Tuple[torch.Tensor, float]] = None,
    frame_sums: Optional[torch.Tensor] = None,
    stale_frames: Sequence[int] = (),
    planned_frames: Sequence[int] = (),
    query: Optional[Tuple[torch.Tensor, torch.Tensor, Optional[torch.Tensor]]] = None,
    k_inv_rms: Optional[torch.Tensor] = None,
):
    """Adaptive sink refresh decision (causal_model.py:284-299) for a
    one-frame chunk, before its append.

    With ``dst_start_override`` (device int64 [B]) the decision is also handed
    to the append that follows on the stream: row i gets the start of the
    refreshed sink frame when it refreshes and ``override_rows[i]`` says the
    row is about to evict, else -1.  ``refresh_out`` (int32 [B]) receives the
    decision instead of a new device tensor; it may be PINNED host memory, which
    the kernel then writes directly (valid on the host once the stream has
    passed this call).

    ``k_norm`` = (k norm weight, eps): k is the raw k projection and its
    RMSNorm is applied inside, as :func:`kv_append_rope` with ``qk_norm`` does.

    ``frame_sums`` (from :func:`new_sink_frame_sums`) keeps the means of the
    cached sink frames between calls, so that only the new chunk is read:
    ``stale_frames[i]`` is a bit mask of the sink frames of row i whose means
    must be taken from the cache again (written behind this operator's back,
    or never summed), ``planned_frames[i]`` the sink frame the append that
    follows writes to by the host's plan, or -1.

    ``query`` = (q, rotated q, q norm weight or None), bf16: the chunk's query is
    rotated (and normalised) in the same launch, by workgroups the decision has no
    use for; with ``k_norm``, ``k_inv_rms`` (float32 [B, S]) receives 1 / rms of
    every key token.  The append that follows then moves K and V only.

    k is the chunk's key BEFORE RoPE, v its value, both [B,S,H,128]; the caches
    are read as they are.  Returns (similarity float32 [B, sink_frames],
    refresh int32 [B]) on the device: refresh[i] is the sink frame of row i to
    overwrite next, or -1.
    """
    dev = _require_gpu(k, v, k_cache, v_cache, freqs_table)
    lib = _capi.lib()
    q, q_out, q_weight = query if query is not None else (None, None, None)
    grid_hw, sink_frames = (int(grid_hw[0]), int(grid_hw[1])), int(sink_frames)      # (a key of values, whatever they came in)
    like = (k.shape, v.shape, k_cache.shape, v_cache.shape, k.stride(), v.stride(), k_cache.stride(), v_cache.stride(),
            k.dtype, v.dtype, k_cache.dtype, v_cache.dtype, grid_hw, sink_frames, freqs_table.shape[0])
    if query is not None:
        like += (q.shape, q_out.shape, q.stride(), q_out.stride(), q.dtype, q_out.dtype)
    layout = _SIM_LAYOUTS.get(like)
    if layout is None:
        if len(_SIM_LAYOUTS) >= _MAX_ATTN_LAYOUTS:
            _SIM_LAYOUTS.clear()
        layout = _SIM_LAYOUTS[like] = _sim_layout(lib, k, v, k_cache, v_cache, freqs_table.shape[0], grid_hw, sink_frames, q, q_out)
    filled, need, kept_need = layout
    rows, tokens, heads = filled.rows, filled.tokens, filled.heads
    ws = _workspace(dev, need, _SIM_WORKSPACES)      # (zero-filled: its ticket words start at zero)
    similarity = torch.empty((rows, sink_frames), dtype=torch.float32, device=dev)
    if refresh_out is None:
        refresh = torch.empty((rows,), dtype=torch.int32, device=dev)
    else:
        refresh = refresh_out
        on_device = refresh.device == dev or (refresh.device.type == "cpu" and refresh.is_pinned())
        if refresh.dtype != torch.int32 or refresh.numel() < rows or not refresh.is_contiguous() or not on_device:
            raise RuntimeError(f"refresh_out must be a contiguous int32 tensor with one entry per row, on {dev} or pinned")

    p = _capi.SinkSimParams.from_buffer_copy(filled)
    p.k_in, p.v_in, p.k_cache, p.v_cache = k.data_ptr(), v.data_ptr(), k_cache.data_ptr(), v_cache.data_ptr()
    p.freqs = freqs_table.data_ptr()
    p.threshold = float(threshold)
    p.start_frame = _i64_array(start_frames)
    p.similarity, p.refresh = similarity.data_ptr(), refresh.data_ptr()
    p.workspace, p.workspace_bytes = ws.data_ptr(), ws.numel()
    p.stream = _stream_ptr(dev)
    if dst_start_override is not None:
        _check_override(dst_start_override, rows, dev)
        if len(override_rows) != rows:
            raise RuntimeError("override_rows needs one flag per row")
        p.dst_start_override = dst_start_override.data_ptr()
        p.override_rows = sum(1 << i for i, flag in enumerate(override_rows) if flag)
    if k_norm is not None:
        weight, eps = k_norm
        if weight.dtype != k.dtype or weight.numel() != heads * HEAD_DIM or not weight.is_contiguous() \
                or weight.device != dev:
            raise RuntimeError(f"the k norm weight must be a contiguous {k.dtype} tensor of {heads * HEAD_DIM} elements on {dev}")
        p.k_norm_weight, p.norm_eps = weight.data_ptr(), float(eps)
    if frame_sums is not None:
        if frame_sums.device != dev or not frame_sums.is_contiguous() \
                or frame_sums.numel() * frame_sums.element_size() < kept_need:
            raise RuntimeError(f"frame_sums must be a contiguous buffer of at least {kept_need} bytes on {dev}")
        if len(stale_frames) != rows or len(planned_frames) != rows:
            raise RuntimeError("frame_sums needs stale_frames and planned_frames with one entry per row")
        p.frame_sums = frame_sums.data_ptr()
        p.stale_frames = (C.c_uint32 * rows)(*[int(x) & 0xffffffff for x in stale_frames])
        p.planned_frame = (C.c_int32 * rows)(*[int(x) for x in planned_frames])
    if query is not None:
        if q.device != dev or q_out.device != dev:
            raise RuntimeError(f"query and rotated query must lie on {dev}")
        if (q_weight is None) != (k_norm is None):
            raise RuntimeError("the q and k norms are folded in together")
        p.q_in, p.q_out = q.data_ptr(), q_out.data_ptr()
        if q_weight is not None:
            _check_norm((q_weight, *k_norm), q.dtype, heads, dev)
            p.q_norm_weight = q_weight.data_ptr()
    if k_inv_rms is not None:
        if k_inv_rms.dtype != torch.float32 or k_inv_rms.numel() < rows * tokens or not k_inv_rms.is_contiguous() \
                or k_inv_rms.device != dev:
            raise RuntimeError(f"k_inv_rms must be a contiguous float32 tensor with one entry per token on {dev}")
        p.k_inv_rms = k_inv_rms.data_ptr()
    with _on_device(dev):
        _capi.check(lib.sdv2_sink_similarity(C.byref(p)), "sdv2_sink_similarity")
    return similarity, refresh


def new_sink_frame_sums(rows: int, heads: int, sink_frames: int, dev) -> torch.Tensor:
    """The buffer :func:`sink_similarity` keeps the sink frames' means in
    between calls (everything in it starts out stale)."""
    n = _capi.lib().sdv2_sink_frame_sums_bytes(rows, heads, sink_frames)
    return torch.empty(max(n // 4, 1), dtype=torch.float32, device=dev)


class KernelTimer:
    """A start/stop pair of the library's timing events (a measurement hook,
    include/sdv2kv_profile.h).  Armed for a kernel (:meth:`arm`, or
    ``LayerLauncher.set_timers``) it is recorded in the dispatch of this
    thread's next launch of that kernel, so :meth:`elapsed_ms` is the kernel's
    duration as a profiler reports it, without the gap separate stream events
    add."""

    def __init__(self):
        lib = _capi.lib()
        self.start, self.stop = C.c_void_p(), C.c_void_p()
        _capi.check(lib.sdv2_event_create(C.byref(self.start)), "sdv2_event_create")
        _capi.check(lib.sdv2_event_create(C.byref(self.stop)), "sdv2_event_create")

    def arm(self, kernel: int) -> None:
        """Time this thread's next launch of ``kernel`` (``_capi.KERNEL_*``)."""
        _capi.check(_capi.lib().sdv2_profile_time_next(kernel, self.start, self.stop), "sdv2_profile_time_next")

    def elapsed_ms(self) -> float:
        ms = C.c_float()
        _capi.check(_capi.lib().sdv2_event_elapsed_ms(self.start, self.stop, C.byref(ms)), "sdv2_event_elapsed_ms")
        return ms.value

    def close(self) -> None:
        lib = _capi.lib()
        for e in (self.start, self.stop):
            if e:
                lib.sdv2_event_destroy(e)
        self.start, self.stop = C.c_void_p(), C.c_void_p()

    def __del__(self):
        try:
            self.close()
        except Exception:
            pass


class LayerLauncher:
    """Pre-built launch descriptors for one layer's (append, attention) pair.

    A chunk step calls the path once per transformer block, every time with the
    same cache, shapes and strides; only the slot, the RoPE frame, the index
    values and the q/k/v pointers change.  Building the two C structs from
    scratch costs more host time than the kernels take on the GPU, so they are
    built once per (cache, shape) and patched per call.
    """

    def __init__(self, k_cache, v_cache, global_end_index, local_end_index, freqs_table, grid, q_like, k_like=None,
                 v_like=None, qk_norm=None, rope_in_attention=True):
        k_like = q_like if k_like is None else k_like
        v_like = q_like if v_like is None else v_like
        rows, tokens, heads, _ = q_like.shape
        if tuple(k_like.shape) != tuple(q_like.shape) or tuple(v_like.shape) != tuple(q_like.shape):
            raise RuntimeError("q, k and v must have one shape")
        if rows > _capi.MAX_ROWS:
            raise RuntimeError(f"LayerLauncher handles at most {_capi.MAX_ROWS} rows")
        if q_like.dtype != torch.bfloat16:
            raise RuntimeError("LayerLauncher is the bf16 fast path")
        dev = _require_gpu(k_cache, v_cache, global_end_index, local_end_index, freqs_table, q_like)
        self.dev = dev
        self.rows, self.tokens, self.heads = rows, tokens, heads
        self.in_shape = q_like.shape
        self.in_strides = (q_like.stride(), k_like.stride(), v_like.stride())
        self.cache_shape = k_cache.shape
        self.cache_strides = (k_cache.stride(), v_cache.stride())
        self.cache_ptrs = (k_cache.data_ptr(), v_cache.data_ptr(), global_end_index.data_ptr(), local_end_index.data_ptr())
        self.k_cache, self.v_cache = k_cache, v_cache
        self.lib = _capi.lib()
        # Where the query is rotated.  rope_in_attention: where it is consumed,
        # inside the attention kernel; the append then moves K and V only (and, with
        # the q / k norm folded in, leaves 1 / rms per q token in ``q_inv_rms``).
        # Otherwise (what RingKVPath does) by the append, which hands the attention
        # the rotated copy: a third more bytes for the append, once per query and
        # spread over the chip, against 3.5 us of table reads and double arithmetic
        # at the start of every attention workgroup, once per key range of the query
        # (whole layer call at 3120 queries x 12 heads against themselves: 103 -> 97 us;
        # 1560 x 40 against 9360 keys: 332 -> 322 us).
        self.rope_in_attention = bool(rope_in_attention)
        # The rotated query of the last patched call, a tensor of that call's own: a second thread
        # may append on the same stream between this call's two launches, and a graph that captured
        # them keeps the memory in its pool.  (None when the attention rotates.)
        self.roped_q = None
        # Set for the next call by one whose sink decision has made them: the rotated query, and 1 / rms of the key
        # tokens with the norm folded in (which that caller holds).
        self.rotated = None
        self.q_inv_rms = torch.empty((rows, tokens), dtype=torch.float32, device=dev) \
            if self.rope_in_attention and qk_norm is not None else None
        self.sf = (C.c_int64 * rows)()
        self.ds = (C.c_int64 * rows)()
        self.ng = (C.c_int64 * rows)()
        self.nl = (C.c_int64 * rows)()

        ap = _capi.AppendParams()
        ap.k_in_stride = _stride3(k_like, "k")
        ap.v_in_stride = _stride3(v_like, "v")
        roped_stride = _capi.Stride3(tokens * heads * HEAD_DIM, heads * HEAD_DIM, HEAD_DIM)
        if not self.rope_in_attention:
            ap.q_in_stride = _stride3(q_like, "q")
            ap.q_out_stride = roped_stride
        elif self.q_inv_rms is not None:
            ap.q_in_stride = _stride3(q_like, "q")
            ap.q_inv_rms = self.q_inv_rms.data_ptr()
        ap.k_cache, ap.k_cache_stride = k_cache.data_ptr(), _stride3(k_cache, "k_cache")
        ap.v_cache, ap.v_cache_stride = v_cache.data_ptr(), _stride3(v_cache, "v_cache")
        ap.freqs, ap.freq_rows = freqs_table.data_ptr(), freqs_table.shape[0]
        ap.dtype = _capi.DTYPE_BF16
        ap.rows, ap.tokens, ap.heads, ap.head_dim = rows, tokens, heads, HEAD_DIM
        self.grid = ap.grid_f, ap.grid_h, ap.grid_w = tuple(int(x) for x in grid)
        ap.cache_tokens = k_cache.shape[1]
        ap.start_frame = C.cast(self.sf, C.POINTER(C.c_int64))
        ap.dst_start = C.cast(self.ds, C.POINTER(C.c_int64))
        ap.global_end_index = global_end_index.data_ptr()
        ap.local_end_index = local_end_index.data_ptr()
        ap.new_global_end = C.cast(self.ng, C.POINTER(C.c_int64))
        ap.new_local_end = C.cast(self.nl, C.POINTER(C.c_int64))
        self.norm_args = None
        if qk_norm is not None:
            _check_norm(qk_norm, q_like.dtype, heads, dev)
            self.norm_args = ap.q_norm_weight, ap.k_norm_weight, ap.norm_eps = \
                qk_norm[0].data_ptr(), qk_norm[1].data_ptr(), float(qk_norm[2])
            # held (their memory, whatever becomes of a module's parameter): the descriptor keeps the addresses
            self.norm_weights = tuple(w.detach() for w in qk_norm[:2])
        self.ap, self.ap_ref = ap, C.byref(ap)
        self.freqs_table = freqs_table

        at = _capi.AttnParams()
        if self.rope_in_attention:
            at.q_stride = _stride3(q_like, "q")
            at.rope_freqs, at.rope_freq_rows = freqs_table.data_ptr(), freqs_table.shape[0]
            at.rope_grid_h, at.rope_grid_w = int(grid[1]), int(grid[2])
            at.rope_start_frame = C.cast(self.sf, C.POINTER(C.c_int64))
            if self.q_inv_rms is not None:
                at.q_norm_weight, at.q_inv_rms = self.norm_args[0], self.q_inv_rms.data_ptr()
        else:
            at.q_stride = roped_stride
        at.k_cache, at.k_stride = k_cache.data_ptr(), _stride3(k_cache, "k_cache")
        at.v_cache, at.v_stride = v_cache.data_ptr(), _stride3(v_cache, "v_cache")
        at.rows, at.q_tokens, at.heads, at.head_dim = rows, tokens, heads, HEAD_DIM
        at.chunk_key_start_host = C.cast(self.ds, C.POINTER(C.c_int64))       # (where the append puts the chunk's keys)
        self.at, self.at_ref = at, C.byref(at)
        self.span, self.mask_plan = -1, None
        self.workspace_need, self.workspace = 0, None
        at.out_stride = roped_stride                 # contiguous, like the rotated query
        self.forced_splits = 0                       # 0 = the library's own choice
        self.timers = (None, None)

    def matches(self, q, k, v, kv_cache, freqs_table, qk_norm=None) -> bool:
        shape, strides, bf16 = self.in_shape, self.in_strides, torch.bfloat16
        if freqs_table is not self.freqs_table or q.shape != shape or k.shape != shape or v.shape != shape \
                or q.stride() != strides[0] or k.stride() != strides[1] or v.stride() != strides[2] \
                or q.dtype != bf16 or k.dtype != bf16 or v.dtype != bf16:
            return False
        if self.norm_args != (None if qk_norm is None else (qk_norm[0].data_ptr(), qk_norm[1].data_ptr(), qk_norm[2])):
            return False
        kc, vc = kv_cache["k"], kv_cache["v"]
        return self.cache_ptrs == (kc.data_ptr(), vc.data_ptr(), kv_cache["global_end_index"].data_ptr(),
                                   kv_cache["local_end_index"].data_ptr()) \
            and kc.shape == self.cache_shape and (kc.stride(), vc.stride()) == self.cache_strides

    def patch(self, q, k, v, start_frames, plan, seq_lens: Optional[torch.Tensor] = None,
              mask_block_tokens: int = 0, dst_start_override: Optional[torch.Tensor] = None) -> torch.Tensor:
        """Fill in what changes from call to call and allocate the output
        [rows, S, H, 128]; nothing is launched."""
        ap, at = self.ap, self.at
        stream = _stream_ptr(self.dev)
        if dst_start_override is not None:
            _check_override(dst_start_override, self.rows, self.dev)
        ap.dst_start_override = dst_start_override.data_ptr() if dst_start_override is not None else None
        at.mask_block_tokens = mask_block_tokens
        if mask_block_tokens:
            _check_chunk_starts(plan.dst_start, self.rows, self.tokens, plan.max_seq_len)
        self.sf[:] = start_frames
        self.ds[:] = plan.dst_start
        self.ng[:] = plan.new_global_end
        self.nl[:] = plan.new_local_end
        ap.k_in, ap.v_in = k.data_ptr(), v.data_ptr()
        if self.rope_in_attention:
            at.q = q.data_ptr()
            if self.q_inv_rms is not None:
                ap.q_in = q.data_ptr()
        elif self.rotated is not None:
            (self.roped_q, inv_rms), self.rotated = self.rotated, None
            at.q = self.roped_q.data_ptr()
            ap.q_in = ap.q_out = ap.q_norm_weight = None
            ap.k_inv_rms = inv_rms.data_ptr() if inv_rms is not None else None
        else:
            # (a caller that fills in its own calls may bring the same memory in another form)
            alike = q.shape == self.in_shape and q.dtype == torch.bfloat16 and q.device == self.dev
            self.roped_q = _empty_as(q) if alike else torch.empty(self.in_shape, dtype=torch.bfloat16, device=self.dev)
            ap.q_in = q.data_ptr()
            ap.q_out = at.q = self.roped_q.data_ptr()
            if self.norm_args is not None:
                ap.q_norm_weight, ap.k_inv_rms = self.norm_args[0], None
        ap.stream = at.stream = stream
        span = plan.max_seq_len
        mask_plan = (mask_block_tokens, _starts_alike(plan.dst_start)) if mask_block_tokens else None
        if span != self.span or mask_plan != self.mask_plan:
            self.span, self.mask_plan = span, mask_plan
            at.max_seq_len = span
            at.num_splits = self.forced_splits or _library_plan(
                self.lib, self.rows, self.tokens, self.heads, span, not self.rope_in_attention, *(mask_plan or (0, False)))
            self.workspace_need = self.lib.sdv2_swa_attn_workspace_bytes(self.rows, self.tokens, self.heads, span,
                                                                         at.num_splits)
        if self.workspace_need:
            # this stream's; may have been regrown by another shape (and, by another thread's call, between here
            # and the launch: the one this call carries is held)
            self.workspace = ws = _workspace(self.dev, self.workspace_need, stream=stream)
            at.workspace, at.workspace_bytes = ws.data_ptr(), ws.numel()
        out = torch.empty(self.in_shape, dtype=torch.bfloat16, device=self.dev) if self.rope_in_attention else _empty_as(self.roped_q)
        at.out = out.data_ptr()
        at.seq_lens = seq_lens.data_ptr() if seq_lens is not None else None
        return out

    def set_timers(self, append: Optional[KernelTimer] = None, attention: Optional[KernelTimer] = None) -> None:
        """Attach (or, with None, detach) kernel timers for the next launches."""
        self.timers = (append, attention)

    def run_append(self) -> None:
        if self.timers[0] is not None:
            self.timers[0].arm(_capi.KERNEL_APPEND)
        _capi.check(self.lib.sdv2_kv_append_rope(self.ap_ref), "sdv2_kv_append_rope")

    def run_attention(self) -> None:
        if self.timers[1] is not None:
            self.timers[1].arm(_capi.KERNEL_ATTENTION)
        _capi.check(self.lib.sdv2_swa_attn_fwd(self.at_ref), "sdv2_swa_attn_fwd")

    def launch(self, q, k, v, start_frames, plan, seq_lens: Optional[torch.Tensor] = None,
               mask_block_tokens: int = 0, dst_start_override: Optional[torch.Tensor] = None) -> torch.Tensor:
        """Append + attention for one call; returns the attention output
        [rows, S, H, 128]."""
        out = self.patch(q, k, v, start_frames, plan, seq_lens, mask_block_tokens, dst_start_override)
        with _on_device(self.dev):
            self.run_append()
            self.run_attention()
        return out


def flash_attn_with_kvcache(q, k_cache, v_cache, cache_seqlens=None):
    """Same call as the reference makes on flash_attn_interface
    (causal_model.py:353-358): defaults mean causal=False and scale 1/sqrt(D)."""
    if cache_seqlens is not None and cache_seqlens.dtype != torch.int32:
        cache_seqlens = cache_seqlens.to(torch.int32)
    return swa_attention(q, k_cache, v_cache, cache_seqlens)


# the reference's own fallback operator has the same four arguments and result
# (causal_model.py:111-157); with this package both names are one kernel
attention_with_kvcache_fallback = flash_attn_with_kvcache


def flash_attention(q, k, v, q_lens=None, k_lens=None, dropout_p=0.0, softmax_scale=None, q_scale=None,
                    causal=False, window_size=(-1, -1), deterministic=False, dtype=torch.bfloat16, version=None):
    """The reference's generic attention entry (wan_base/modules/attention.py,
    ``flash_attention``) for the cases the cached inference path uses:
    cross-attention of a chunk against the cached text keys / values
    (wan_base/modules/model.py:192), i.e. no causal mask, no window, no dropout,
    every query row valid.  k / v may be ``expand``-ed views (row stride 0, as
    causal_stream_inference.py:227-228 makes them).  Inputs that are not bf16
    are computed in bf16 and the result is returned in q's dtype, as the
    reference does with its ``dtype`` argument."""
    if causal or tuple(window_size) != (-1, -1) or dropout_p or q_lens is not None:
        raise NotImplementedError("flash_attention here covers the cached inference path: "
                                  "causal=False, window_size=(-1, -1), dropout_p=0, q_lens=None")
    if dtype != torch.bfloat16:
        raise NotImplementedError("the attention kernel computes in bf16")
    out_dtype = q.dtype
    scale = None
    if q_scale is not None or softmax_scale is not None:
        scale = (q_scale if q_scale is not None else 1.0) * \
                (softmax_scale if softmax_scale is not None else HEAD_DIM ** -0.5)
    if k_lens is not None:
        k_lens = k_lens.to(device=q.device, dtype=torch.int32).contiguous()
    if out_dtype != torch.bfloat16:
        q = q.to(torch.bfloat16)
    if k.dtype != torch.bfloat16:
        k = k.to(torch.bfloat16)
    if v.dtype != torch.bfloat16:
        v = v.to(torch.bfloat16)
    if q.stride(-1) != 1:
        q = q.contiguous()
    out = swa_attention(q, k, v, k_lens, softmax_scale=scale)
    return out if out_dtype == torch.bfloat16 else out.to(out_dtype)


_RELAYOUT_LAYOUTS: dict = {}


def _relayout_layout(dst, src) -> bytes:
    """The descriptor of such a pair of tensors, but for what changes from call to call."""
    if src.dtype not in _DTYPES or dst.dtype != src.dtype:
        raise RuntimeError(f"unsupported dtype pair {dst.dtype} / {src.dtype}")
    if tuple(dst.shape) != tuple(src.shape):
        raise RuntimeError(f"shape mismatch: {tuple(dst.shape)} vs {tuple(src.shape)}")
    rows, tokens, heads, _ = src.shape
    p = _capi.RelayoutParams()
    p.src_stride, p.dst_stride = _stride3(src, "src"), _stride3(dst, "dst")
    p.dtype = _DTYPES[src.dtype]
    p.rows, p.heads, p.head_dim, p.tokens = rows, heads, HEAD_DIM, tokens
    return bytes(p)


def _relayout_params(dst, src, dst_indices, src_indices, global_end_shift):
    dev = _require_gpu(dst, src, *(dst_indices or ()), *(src_indices or ()))
    key = (src.shape, dst.shape, src.stride(), dst.stride(), src.dtype, dst.dtype)
    layout = _RELAYOUT_LAYOUTS.get(key)
    if layout is None:
        layout = _relayout_layout(dst, src)
        if len(_RELAYOUT_LAYOUTS) >= _MAX_ATTN_LAYOUTS:
            _RELAYOUT_LAYOUTS.clear()
        _RELAYOUT_LAYOUTS[key] = layout
    if (dst_indices is None) != (src_indices is None):
        raise RuntimeError("index tensors are handed over as two pairs or not at all")
    p = _capi.RelayoutParams.from_buffer_copy(layout)
    p.src, p.dst = src.data_ptr(), dst.data_ptr()
    if dst_indices is not None:
        rows = src.shape[0]
        for idx in (*dst_indices, *src_indices):
            if idx.dtype != torch.int64 or idx.numel() < rows or not idx.is_contiguous():
                raise RuntimeError("end-index tensors must be contiguous int64 with one entry per row")
        p.dst_global_end_index, p.dst_local_end_index = (t.data_ptr() for t in dst_indices)
        p.src_global_end_index, p.src_local_end_index = (t.data_ptr() for t in src_indices)
        p.global_end_shift = int(global_end_shift)
    p.stream = _stream_ptr(dev)
    return p, dev


def cache_relayout(
    dst: torch.Tensor,
    src: torch.Tensor,
    dst_indices: Optional[Tuple[torch.Tensor, torch.Tensor]] = None,
    src_indices: Optional[Tuple[torch.Tensor, torch.Tensor]] = None,
    global_end_shift: int = 0,
    timer: Optional["KernelTimer"] = None,
) -> None:
    """``dst[...] = src[...]`` for two [rows, cap, heads, 128] tensors in any
    stride order, plus, with both index pairs (global_end_index,
    local_end_index) given, ``dst_global = src_global + global_end_shift`` and
    ``dst_local = src_local`` in the same launch: one side of the block
    hand-off of streamv2v/communication/kv_cache_manager.py:66-82."""
    p, dev = _relayout_params(dst, src, dst_indices, src_indices, global_end_shift)
    if timer is not None:
        timer.arm(_capi.KERNEL_RELAYOUT)
    with _on_device(dev):
        _capi.check(_capi.lib().sdv2_cache_relayout(C.byref(p)), "sdv2_cache_relayout")


def cache_relayout_pair(
    dst: Tuple[torch.Tensor, torch.Tensor],
    src: Tuple[torch.Tensor, torch.Tensor],
    dst_indices: Optional[Tuple[torch.Tensor, torch.Tensor]] = None,
    src_indices: Optional[Tuple[torch.Tensor, torch.Tensor]] = None,
    global_end_shift: int = 0,
) -> None:
    """:func:`cache_relayout` of two tensors, the indices with the first: K and
    V of a block, one launch when both have the same shape and dtype."""
    first, dev = _relayout_params(dst[0], src[0], dst_indices, src_indices, global_end_shift)
    second, dev_second = _relayout_params(dst[1], src[1], None, None, 0)
    if dev_second != dev:
        raise RuntimeError(f"tensors on different devices: {dev} vs {dev_second}")
    with _on_device(dev):
        _capi.check(_capi.lib().sdv2_cache_relayout_pair(C.byref(first), C.byref(second)), "sdv2_cache_relayout_pair")


def _norm_rows(t: torch.Tensor):
    """(rows, elements between rows) of a tensor [..., width] whose rows are
    contiguous and evenly spaced, else None."""
    width = t.shape[-1]
    if t.is_contiguous():
        return t.numel() // width, width
    if width > 1 and t.stride(-1) != 1:
        return None
    rows = t.numel() // width
    if t.dim() == 1 or rows <= 1:
        return rows, width
    step = expect = None
    for size, stride in zip(reversed(t.shape[:-1]), reversed(t.stride()[:-1])):
        if size == 1:
            continue
        if step is None:
            step = expect = stride
        elif stride != expect:
            return None
        expect *= size
    if step is None or step < width or step % 8 != 0:
        return None
    return rows, step


def _norm_input(x: torch.Tensor, weight: torch.Tensor):
    """:func:`_norm_rows` of x if :func:`rms_norm` can take it, else None."""
    width = x.shape[-1] if x.dim() else 0
    if not (x.is_cuda and x.dtype in _DTYPES and weight.dtype == x.dtype and weight.device == x.device
            and width > 0 and width % HEAD_DIM == 0 and width // HEAD_DIM <= 64 and weight.numel() == width
            and weight.is_contiguous() and x.data_ptr() % 16 == 0 and weight.data_ptr() % 16 == 0):
        return None
    return _norm_rows(x)


def rms_norm_supported(x: torch.Tensor, weight: torch.Tensor) -> bool:
    """Can :func:`rms_norm` take this input?  (A device tensor of a dtype the
    library knows; rows of a multiple of 128 up to 8192 contiguous elements, 16-byte
    aligned and evenly spaced; a contiguous weight of the same dtype.)"""
    return _norm_input(x, weight) is not None


def rms_norm_or_none(x: torch.Tensor, weight: torch.Tensor, eps: float) -> Optional[torch.Tensor]:
    """:func:`rms_norm`, or None for an input it does not take."""
    rows = _norm_input(x, weight)
    return None if rows is None else _launch_norm(x, weight, eps, torch.empty(x.shape, dtype=x.dtype, device=x.device),
                                                  rows, x.shape[-1])


def rms_norm(x: torch.Tensor, weight: torch.Tensor, eps: float, out: Optional[torch.Tensor] = None) -> torch.Tensor:
    """WanRMSNorm.forward (wan_base/modules/model.py:77-86) over the last
    dimension of x [..., width] in one launch: float32 normalisation, back to
    x's dtype, times the weight - the bits the torch expression gives on the
    CPU.  x may be a slice of a wider tensor (rows ``width`` contiguous
    elements, a common distance apart); ``out`` defaults to a new contiguous
    tensor and may be x itself."""
    dev = _require_gpu(x, weight)
    x_rows = _norm_input(x, weight)
    if x_rows is None:
        raise RuntimeError(f"rms_norm takes bf16 / fp32 rows of a multiple of 128 up to 8192 contiguous, 16-byte aligned, "
                           f"evenly spaced elements with a contiguous weight of the same dtype and width, got x "
                           f"{tuple(x.shape)} {x.dtype} strides {x.stride()}, weight {tuple(weight.shape)} {weight.dtype}")
    if out is None:
        out = torch.empty(x.shape, dtype=x.dtype, device=dev)
    elif out.shape != x.shape or out.dtype != x.dtype or out.device != dev:
        raise RuntimeError("out must have x's shape, dtype and device")
    out_rows = _norm_rows(out)
    if out_rows is None or out.data_ptr() % 16:
        raise RuntimeError("out: rows must be contiguous, 16-byte aligned and evenly spaced")
    return _launch_norm(x, weight, eps, out, x_rows, out_rows[1])


def _launch_norm(x, weight, eps, out, x_rows, out_step):
    dev = x.device
    p = _capi.RmsNormParams(x.data_ptr(), out.data_ptr(), weight.data_ptr(), x_rows[1], out_step, x_rows[0], x.shape[-1],
                            _DTYPES[x.dtype], eps, _stream_ptr(dev))
    with _on_device(dev):
        _capi.check(_capi.lib().sdv2_rms_norm(C.byref(p)), "sdv2_rms_norm")
    return out


def _plain_call() -> bool:
    """Nothing watches or rewrites tensor operations: no autograd (either mode), autocast, tracing or compilation, no
    mode that wants to see them."""
    return not (torch.is_grad_enabled() or torch.is_autocast_enabled("cuda") or torch.compiler.is_compiling()
                or torch.jit.is_tracing() or torch.autograd.forward_ad._current_level >= 0
                or torch._C._len_torch_dispatch_stack() or torch._C._len_torch_function_stack()
                or torch._C._functorch.maybe_current_level() is not None)


_PLAIN_TENSORS = (torch.Tensor, torch.nn.Parameter)
_LINEAR_LAYOUTS: dict = {}
_MAX_LINEAR_STRIDE = 1 << 22           # elements between x's rows, as sdv2_linear takes them
_FOLDS_NORM: dict = {}


def _linear_layout(x: torch.Tensor, weight: torch.Tensor, row_squares: bool):
    """(descriptor as bytes, but for what changes from call to call, shape of the result, shape of the sums) of a product
    of such tensors, or None where it is not the library's."""
    if weight.dim() != 2 or x.dim() < 2 or x.numel() == 0:
        return None
    n, k = weight.shape
    if x.shape[-1] != k:
        return None
    m = x.numel() // k
    rows = _norm_rows(x)
    if rows is None or rows[1] > _MAX_LINEAR_STRIDE or not _capi.lib().sdv2_linear_one_round(m, n, k, row_squares):
        return None
    lead = tuple(x.shape[:-1])
    return bytes(_capi.LinearParams(None, None, None, None, rows[1], k, n, m, n, k, _capi.DTYPE_BF16)), (*lead, n), (*lead, n // 32)


def linear_or_none(x: torch.Tensor, weight: torch.Tensor, bias: Optional[torch.Tensor],
                   row_squares: bool = False):
    """``x weight^T + bias`` by the library's kernel where that is the faster one
    (``sdv2_linear_one_round``: bf16, a chunk's worth of rows), else None: the
    caller's nn.Linear, for everything the kernel does not take too.  With
    ``row_squares`` the result comes with the sums of squares of every 32 columns
    of its rows, float32 [..., n / 32]."""
    bf16 = torch.bfloat16
    if not (x.is_cuda and x.dtype == bf16 and weight.dtype == bf16 and type(x) in _PLAIN_TENSORS
            and type(weight) in _PLAIN_TENSORS and x.layout is weight.layout is torch.strided and _plain_call()):
        return None
    key = (x.shape, x.stride(), weight.shape, row_squares)
    layout = _LINEAR_LAYOUTS.get(key, _LINEAR_LAYOUTS)
    if layout is _LINEAR_LAYOUTS:                   # (not seen yet)
        if len(_LINEAR_LAYOUTS) >= _MAX_ATTN_LAYOUTS:
            _LINEAR_LAYOUTS.clear()
        layout = _LINEAR_LAYOUTS[key] = _linear_layout(x, weight, row_squares)
    if layout is None:
        return None
    template, out_shape, squares_shape = layout
    dev = x.device
    x_ptr, weight_ptr = x.data_ptr(), weight.data_ptr()
    if weight.device != dev or not weight.is_contiguous() or x_ptr % 16 or weight_ptr % 16:
        return None
    p = _capi.LinearParams.from_buffer_copy(template)
    if bias is not None:
        if not (type(bias) in _PLAIN_TENSORS and bias.dtype == bf16 and bias.device == dev and bias.shape == weight.shape[:1]
                and bias.is_contiguous()):
            return None
        p.bias = bias_ptr = bias.data_ptr()
        if bias_ptr % 8:
            return None
    out = _empty_as(x) if x.shape == out_shape else torch.empty(out_shape, dtype=bf16, device=dev)
    p.x, p.weight, p.out, p.stream = x_ptr, weight_ptr, out.data_ptr(), _stream_ptr(dev)
    if row_squares:
        squares = torch.empty(squares_shape, dtype=torch.float32, device=dev)
        p.row_squares = squares.data_ptr()
    with _on_device(dev):
        _capi.check(_capi.lib().sdv2_linear(C.byref(p)), "sdv2_linear")
    return (out, squares) if row_squares else out


def folds_query_norm(q_shape, max_seq_len: int, weight: torch.Tensor, device) -> bool:
    """Does the attention of a query [B, S, heads * 128] against max_seq_len keys take the raw projection and
    normalise it itself (``swa_attention(q_row_squares=)``)?"""
    rows, tokens, width = q_shape
    if not (device.type == "cuda" and width % HEAD_DIM == 0 and type(weight) in _PLAIN_TENSORS and _plain_call()
            and weight.dtype == torch.bfloat16 and weight.is_contiguous() and weight.device == device
            and weight.numel() == width and weight.data_ptr() % 16 == 0):
        return False
    key = (rows, tokens, width, max_seq_len)
    folds = _FOLDS_NORM.get(key)
    if folds is None:
        if len(_FOLDS_NORM) >= _MAX_ATTN_LAYOUTS:
            _FOLDS_NORM.clear()
        folds = _FOLDS_NORM[key] = bool(_capi.lib().sdv2_swa_attn_folds_norm(rows, tokens, width // HEAD_DIM, max_seq_len))
    return folds


def copy_bytes(dst: torch.Tensor, src: torch.Tensor) -> None:
    """Plain 16-byte-vector copy with the library's own kernel (used to scale
    hardware counters against a transfer of known size)."""
    dev = _require_gpu(dst, src)
    n = src.numel() * src.element_size()
    if dst.numel() * dst.element_size() != n or not dst.is_contiguous() or not src.is_contiguous():
        raise RuntimeError("copy_bytes needs contiguous tensors of equal byte size")
    with _on_device(dev):
        _capi.check(_capi.lib().sdv2_copy_bytes(dst.data_ptr(), src.data_ptr(), n, _stream_ptr(dev)), "sdv2_copy_bytes")
