"""One decode position through a transformer block in four to six HIP launches.

Drop-in for the reference's `app/engine/fusedlayer.py` (`decode_block`,
`install`, `stats`, `HEAD_DIM`, `CHUNK`):

    [rms_norm + wqkv] -> [qk norm + rope + KV write + attention (+ merge)]
        -> wo(+x) -> [rms_norm + w1, w3 as silu(w1) * w3] -> w2(+h)

The bracketed steps are single launches: the norm runs in the matmul's
prologue with the standalone kernel's exact arithmetic (`nf4gemv.
matmul_fused`), w1/w3 stream through the same waves with the gate in the
epilogue, and the attention workgroups apply the head norms and rotary to
QKV themselves (`ttsp_attn_decode_qkv`; a cache longer than one 64-position
chunk adds a merge launch). With a cache of at most one chunk (the fast
transformer's), the attention and wo are one launch: every wo workgroup
computes the small attention itself (`ttsp_attn_nf4_gemv`). The results are
bit-identical to the reference's ten-launch order (reference:
fusedlayer.py:212-269).

`qk_rope_kv` does the head norms, rotary and KV-cache write for every head in
one launch; attention is split-K over CHUNK-position slices of the cache (one
workgroup per KV head and slice, the chunk's K/V staged in LDS, log-sum-exp
merge); the residual adds and the SwiGLU gate ride on the NF4 matmul's store.
Rounding follows the fork: wherever it produces a 16-bit tensor, so does this
(reference: fusedlayer.py:56-159, 212-269). Every reduction has a fixed order,
so a step's output is a deterministic function of its inputs.

Only a single position (B = S = 1) takes this path. Several positions (a
prompt prefill) take `prefill_block`: the same block as NF4 GEMMs with the
residual adds and the SwiGLU gate in their epilogues, the fork's norms and
rotary as HIP kernels, and the whole causal attention in one launch
(`fastpath.prefill_attention`) - seven GEMM launches, four norm/rotary
launches and one attention launch around the fork's q/k head norms. The
reference has no fused prefill block (it declines S > 1, fusedlayer.py:198)
and runs the unpatched block; the results agree with that order up to the
roundings the epilogues keep (tests compare the layer output).
"""

from __future__ import annotations

import logging

from ttspipe_amd import _lib

logger = logging.getLogger(__name__)

HEAD_DIM = 128
#: Cache positions per attention workgroup (the kernel's ACHUNK).
CHUNK = 64

_stats = {"fused": 0, "fallback": 0, "prefill": 0}
_installed = False


def stats() -> dict:
    return {**_stats, "ready": _lib.gpu_present() and _installed}


def _eligible(a, ff, x, mask, input_pos) -> bool:
    import torch

    from ttspipe_amd import nf4gemv

    if x.dim() != 3 or x.shape[0] != 1 or x.shape[1] != 1:
        return False
    if x.dtype not in (torch.float16, torch.bfloat16) or x.device.type != "cuda" or not x.is_contiguous():
        return False
    cache, nkv = a.kv_cache, a.n_local_heads
    if mask is None or input_pos is None or input_pos.numel() != 1 or cache is None:
        return False
    if input_pos.dtype != torch.long or input_pos.device != x.device:
        return False
    if a.head_dim != HEAD_DIM or a.n_head % nkv or a.n_head // nkv > 16:
        return False
    kc, vc = cache.k_cache, cache.v_cache
    if kc.dtype != x.dtype or vc.dtype != x.dtype or not (kc.is_contiguous() and vc.is_contiguous()):
        return False
    if kc.shape[0] != 1 or kc.shape[1] != nkv or kc.shape[3] != HEAD_DIM:
        return False
    for linear in (a.wqkv, a.wo, ff.w1, ff.w2, ff.w3):
        if getattr(linear, "bias", None) is not None or not nf4gemv.prepare(linear):
            return False
    return True


def decode_block(block, x, freqs_cis, mask, input_pos, *, workspace=None):
    """`TransformerBlock.forward` for one position, or None if it cannot.

    `workspace` (optional) is a dict of preallocated buffers from
    `make_workspace`, which lets a captured graph run without allocating.
    """
    import torch

    from ttspipe_amd import fusedops, nf4gemv

    if not _lib.gpu_present():
        return None
    a, ff = block.attention, block.feed_forward
    if not _eligible(a, ff, x, mask, input_pos):
        return None
    ftype = _lib.dtype_code(freqs_cis.dtype) if freqs_cis is not None else None
    if ftype is None or not freqs_cis.is_contiguous() or freqs_cis.numel() != HEAD_DIM:
        return None
    nh, nkv = a.n_head, a.n_local_heads
    kc, vc = a.kv_cache.k_cache, a.kv_cache.v_cache
    max_len = kc.shape[2]
    nchunk = -(-min(mask.shape[-1], max_len) // CHUNK)
    ws = workspace if workspace is not None else _Workspace(nh, nkv, x, ff.w1.out_features, nchunk)
    dt = _lib.dtype_code(x.dtype)
    lib = _lib.lib()
    st = _lib.stream()

    an = block.attention_norm
    qkv = nf4gemv.matmul_fused(a.wqkv, x, norm_weight=an.weight, eps=an.eps, out=ws["qkv"])
    if qkv is None:  # the unfused pair: norm, then matmul
        xn = fusedops.rms_norm(x, an.weight, an.eps, out=ws["xn"])
        qkv = None if xn is None else nf4gemv.matmul(a.wqkv, xn, out=ws["qkv"])
        if qkv is None:
            return None
    qn = getattr(a, "q_norm", None) if a.attention_qk_norm else None
    kn = getattr(a, "k_norm", None) if a.attention_qk_norm else None
    eps = float(qn.eps if qn is not None and qn.eps is not None else 1e-6)
    if nchunk == 1:
        h = _attn_wo(a, qkv, qn, kn, eps, freqs_cis, ftype, input_pos, x, ws, nchunk, dt, st)
        if h is not None:  # attention and wo (+ residual) in one launch (short caches)
            return _ffn(block, h, ws, x.shape)
    rc = lib.ttsp_attn_decode_qkv(
        qkv.data_ptr(), _lib.ptr(None if qn is None else qn.weight), _lib.ptr(None if kn is None else kn.weight),
        eps, freqs_cis.data_ptr(), ftype, input_pos.data_ptr(), kc.data_ptr(),
        vc.data_ptr(), ws["pm"].data_ptr(), ws["pl"].data_ptr(), ws["pacc"].data_ptr(),
        ws["y"].data_ptr(), nh, nkv, max_len, nchunk, float(HEAD_DIM**-0.5), dt, st)
    _lib.check(rc, "ttsp_attn_decode_qkv")
    h = nf4gemv.matmul(a.wo, ws["y"], epi=nf4gemv.EPI_RESIDUAL, operand=x, out=ws["h"])
    if h is None:
        raise RuntimeError("decode_block: a prepared layer declined mid-block")
    return _ffn(block, h, ws, x.shape)


def _attn_wo(a, qkv, qn, kn, eps, freqs_cis, ftype, input_pos, x, ws, nchunk, dt, st):
    """`ttsp_attn_nf4_gemv`: the attention of a cache of at most one chunk and
    wo with the residual in one launch (every GEMV workgroup recomputes the
    small attention), or None where it does not apply (the two-launch form
    runs; both give the same bits)."""
    from ttspipe_amd import nf4gemv

    fast = getattr(a.wo, "_nf4_fast", None)
    nh, nkv = a.n_head, a.n_local_heads
    max_len = a.kv_cache.k_cache.shape[2]
    D = x.shape[-1]
    if fast is None or nchunk != 1 or nh > 8 or max_len > CHUNK or nkv * max_len > 128:
        return None
    if fast["K"] != nh * HEAD_DIM or fast["M"] != D or x.numel() != D or not x.is_contiguous():
        return None
    h = ws["h"]
    rc = _lib.lib().ttsp_attn_nf4_gemv(
        qkv.data_ptr(), _lib.ptr(None if qn is None else qn.weight), _lib.ptr(None if kn is None else kn.weight),
        eps, freqs_cis.data_ptr(), ftype, input_pos.data_ptr(), a.kv_cache.k_cache.data_ptr(),
        a.kv_cache.v_cache.data_ptr(), nh, nkv, max_len, float(HEAD_DIM**-0.5),
        fast["w"], fast["a8"], fast["amax"], fast["code2"], fast["offset"], fast["lut"].data_ptr(),
        h.data_ptr(), x.data_ptr(), nf4gemv.EPI_RESIDUAL, D, fast["bs"], fast["bs2"], dt, st)
    _lib.check(rc, "ttsp_attn_nf4_gemv")
    nf4gemv._stats["fast"] += 1
    return h


def _ffn(block, h, ws, shape):
    """The block's second half: norm + w1/w3 (SwiGLU) and w2 with the residual."""
    from ttspipe_amd import fusedops, nf4gemv

    ff, fn = block.feed_forward, block.ffn_norm
    g = nf4gemv.matmul_fused(ff.w1, h, norm_weight=fn.weight, eps=fn.eps, module3=ff.w3, out=ws["g"])
    if g is None:  # the unfused chain: norm, w1, w3 with the gate epilogue
        hn = fusedops.rms_norm(h, fn.weight, fn.eps, out=ws["hn"])
        g1 = None if hn is None else nf4gemv.matmul(ff.w1, hn, out=ws["g1"])
        g = None if g1 is None else nf4gemv.matmul(ff.w3, hn, epi=nf4gemv.EPI_SILU_GATE, operand=g1, out=ws["g"])
    out = ws.get("out")
    out = None if g is None else nf4gemv.matmul(ff.w2, g, epi=nf4gemv.EPI_RESIDUAL, operand=h, out=out)
    if g is None or out is None:
        raise RuntimeError("decode_block: a prepared layer declined mid-block")
    _stats["fused"] += 1
    return out.view(shape)


class _Workspace(dict):
    """The buffers of one `decode_block` call, each allocated when first asked
    for (the common route takes seven of the eleven)."""

    def __init__(self, nh, nkv, x, inter, nchunk):
        D, HD = x.shape[-1], HEAD_DIM
        self._kind = x.dtype, x.device
        # name: (shape, fp32)
        self._shapes = {
            "xn": ((1, 1, D), False), "qkv": ((1, (nh + 2 * nkv) * HD), False), "q": ((nh * HD,), False),
            "pm": ((nh * nchunk,), True), "pl": ((nh * nchunk,), True), "pacc": ((nh * nchunk * HD,), True),
            "y": ((1, 1, nh * HD), False), "h": ((1, D), False), "hn": ((1, 1, D), False), "g1": ((1, inter), False),
            "g": ((1, 1, inter), False),
        }

    def __missing__(self, name):
        import torch

        shape, fp32 = self._shapes[name]
        dtype, device = self._kind
        t = self[name] = torch.empty(shape, dtype=torch.float32 if fp32 else dtype, device=device)
        return t


def make_workspace(block, x, nchunk: int, *, with_out: bool = False) -> dict:
    """Buffers one `decode_block` call uses (reusable across calls of the same shape)."""
    import torch

    a, ff = block.attention, block.feed_forward
    lazy = _Workspace(a.n_head, a.n_local_heads, x, ff.w1.out_features, nchunk)
    ws = {name: lazy[name] for name in lazy._shapes}
    if with_out:
        ws["out"] = torch.empty((1, x.shape[-1]), dtype=x.dtype, device=x.device)
    return ws


def _block_classes():
    from ttspipe_amd.llama import TransformerBlock

    classes = [TransformerBlock]
    try:
        from fish_speech.models.text2semantic.llama import TransformerBlock as ForkBlock

        classes.append(ForkBlock)
    except Exception:  # noqa: BLE001
        pass
    return classes


def _prefill_eligible(block, x, mask, input_pos) -> bool:
    import torch

    from ttspipe_amd import nf4gemv

    a, ff = block.attention, block.feed_forward
    if x.dim() != 3 or x.shape[0] != 1 or x.shape[1] < 2:
        return False
    if x.dtype not in (torch.float16, torch.bfloat16) or x.device.type != "cuda" or not x.is_contiguous():
        return False
    if mask is None or input_pos is None or input_pos.numel() != x.shape[1] or a.kv_cache is None:
        return False
    if a.head_dim != HEAD_DIM or a.n_head % a.n_local_heads:
        return False
    for linear in (a.wqkv, a.wo, ff.w1, ff.w2, ff.w3):
        if getattr(linear, "bias", None) is not None or not nf4gemv.prepare(linear):
            return False
    return True


def _attend_in_parts(q, kc, vc, input_pos, nh, nkv, parts):
    """A long causal span's attention, `parts` of its rows a launch (each row
    sees the cache up to its own position, so later parts' rows, which are in
    the cache already, change nothing); (1, nh, S, 128), or None."""
    import torch

    from ttspipe_amd import fastpath

    n = q.shape[2]
    out = torch.empty(1, n, nh * HEAD_DIM, dtype=q.dtype, device=q.device)
    for r0, r1, width in parts:
        if fastpath.prefill_attention(q[:, :, r0:r1], kc[:, :, :width], vc[:, :, :width], None, nh, nkv, HEAD_DIM,
                                      out=out[:, r0:r1], positions=input_pos[r0:r1]) is None:
            return None
    return out.view(1, n, nh, HEAD_DIM).transpose(1, 2)


def prefill_block(block, x, freqs_cis, mask, input_pos):
    """`TransformerBlock.forward` for several positions (B = 1, S > 1), or None.
    The block of `prefill_block_chain` without a carried norm."""
    r = prefill_block_chain(block, x, freqs_cis, mask, input_pos)
    return None if r is None else r[0]


def prefill_block_chain(block, x, freqs_cis, mask, input_pos, *, xn=None, next_norm=None, causal=False,
                        attend=None):
    """`(out, out_n)`: the block's output for several positions (B = 1, S > 1)
    and, with `next_norm` (an RMSNorm module), `next_norm(out)` for the next
    block (else None, and None for a span of up to `nf4gemv.FUSED_MAX_ROWS`
    rows, whose next block folds that norm into its wqkv GEMV); None when the
    block declines.
    `xn`, if given, is this block's `attention_norm(x)` (a previous call's
    `out_n`), whose launch is then skipped; where the split-K reduce of wo and
    w2 serves the shape it writes the following RMSNorm too
    (`nf4gemv.matmul_norm`), bit for bit the separate launch. `causal`: the
    caller's promise that the mask is the causal one (row i allows keys
    0 .. input_pos[i], all below the mask's width); a span of up to
    `fastpath.CAUSAL_ROWS_MAX` rows then attends row by row as the decode
    step does (`fastpath.causal_rows_attention`), and a longer one computes
    the mask from `input_pos` in the attention kernel; neither reads it.
    `attend` (with `causal`): `(first row, end row, window)` of each attention
    launch, in order and covering the rows, each over the first `window` cache
    positions; default one launch over the mask's width.

    The fork's block in its own order with the prefill kernels: RMSNorm,
    wqkv GEMM, q/k head norms + rotary + KV-cache write for every row in one
    launch (the decode step's kernel over rows, which also adds a K-split
    wqkv's partial sums; the fork's modules when the cache or tables do not
    fit it), one-launch causal attention, wo GEMM with
    the residual add in its epilogue, RMSNorm, w1 and w3 GEMMs with the
    SwiGLU gate (one launch where it serves the shape, else w3's epilogue), w2 GEMM with
    the residual add (reference: the
    unfused block the reference runs for S > 1, fastpath.py:207-271 and
    fusedlayer.py:198).
    """
    import torch

    from ttspipe_amd import fastpath, fusedops, nf4gemv
    from ttspipe_amd.llama import apply_rotary_emb

    if not _lib.gpu_present() or not _prefill_eligible(block, x, mask, input_pos):
        return None
    a, ff = block.attention, block.feed_forward
    bsz, n, _ = x.shape
    nh, nkv, hd = a.n_head, a.n_local_heads, a.head_dim
    an, fn = block.attention_norm, block.ffn_norm
    # a span of up to FUSED_MAX_ROWS rows takes the GEMV with each row's
    # RMSNorm folded in, as the decode step does: no norm launch runs
    fold = n <= nf4gemv.FUSED_MAX_ROWS
    wide = attend is not None  # merged spans: the products keep their order of sums
    qkv = None
    if xn is None and fold:
        qkv = nf4gemv.matmul_fused(a.wqkv, x, norm_weight=an.weight, eps=an.eps)
    if qkv is None and xn is None:
        xn = fusedops.rms_norm(x, an.weight, an.eps)
        if xn is None:
            return None
    kc, vc = a.kv_cache.k_cache, a.kv_cache.v_cache
    max_len = kc.shape[2]
    ftype = _lib.dtype_code(freqs_cis.dtype)
    rows_ok = (ftype is not None and freqs_cis.is_contiguous() and freqs_cis.numel() == n * hd
               and input_pos.dtype == torch.long and input_pos.is_contiguous() and kc.is_contiguous()
               and vc.is_contiguous() and kc.dtype == x.dtype and tuple(kc.shape) == (1, nkv, max_len, hd))
    # a K-split wqkv hands its fp32 partial sums straight to the head-norm /
    # rotary / KV kernel, which adds them as the split's own reduce would
    part = None
    if qkv is None and rows_ok and a.wqkv._nf4_fast["M"] == (nh + 2 * nkv) * hd:
        part = nf4gemv.matmul_partials(a.wqkv, xn, span=True, wide=wide)
    if part is None and qkv is None:
        qkv = nf4gemv.matmul(a.wqkv, xn, wide=wide)
        if qkv is None:
            return None
    y = None
    if causal and rows_ok and part is None and n <= fastpath.CAUSAL_ROWS_MAX:
        # a short causal span: the head norms, rotary and KV write inside the
        # row-by-row attention launch (the decode step's form, no mask reads)
        qn, kn = (a.q_norm, a.k_norm) if a.attention_qk_norm else (None, None)
        y = fastpath.causal_rows_attention_qkv(qkv, None if qn is None else qn.weight,
                                               None if kn is None else kn.weight,
                                               float(qn.eps) if qn is not None else 0.0, freqs_cis, input_pos, kc,
                                               vc, nh, nkv, mask.shape[-1])
    if y is None and rows_ok:
        # head norms, rotary and the KV write for every row in one launch
        q = torch.empty(bsz, n, nh, hd, dtype=x.dtype, device=x.device)
        qn, kn = (a.q_norm, a.k_norm) if a.attention_qk_norm else (None, None)
        eps = float(qn.eps) if qn is not None else 0.0
        qw, kw = _lib.ptr(None if qn is None else qn.weight), _lib.ptr(None if kn is None else kn.weight)
        if part is not None:
            work, splits = part
            rc = _lib.lib().ttsp_qk_rope_kv_rows_partials(
                work.data_ptr(), splits, qw, kw, eps, freqs_cis.data_ptr(), ftype, input_pos.data_ptr(),
                q.data_ptr(), kc.data_ptr(), vc.data_ptr(), nh, nkv, max_len, n, _lib.dtype_code(x.dtype),
                _lib.stream())
            _lib.check(rc, "ttsp_qk_rope_kv_rows_partials")
        else:
            rc = _lib.lib().ttsp_qk_rope_kv_rows(
                qkv.data_ptr(), qkv.shape[-1], qw, kw, eps, freqs_cis.data_ptr(), ftype, input_pos.data_ptr(),
                q.data_ptr(), kc.data_ptr(), vc.data_ptr(), nh, nkv, max_len, n, _lib.dtype_code(x.dtype),
                _lib.stream())
            _lib.check(rc, "ttsp_qk_rope_kv_rows")
        q_rows = q
        q, k, v = q.transpose(1, 2), kc, vc
    elif y is None:
        q, k, v = qkv.split([nh * hd, nkv * hd, nkv * hd], dim=-1)
        q, k, v = q.view(bsz, n, nh, hd), k.view(bsz, n, nkv, hd), v.view(bsz, n, nkv, hd)
        if a.attention_qk_norm:
            q, k = a.q_norm(q), a.k_norm(k)
        fq = fusedops.rope(q, freqs_cis)
        fk = fusedops.rope(k, freqs_cis) if fq is not None else None
        if fk is None:
            fusedops.note_rope_fallback()
            fq, fk = apply_rotary_emb(q, freqs_cis), apply_rotary_emb(k, freqs_cis)
        q, k, v = (t.transpose(1, 2) for t in (fq, fk, v))
        k, v = a.kv_cache.update(input_pos, k, v)
    if y is None and causal and rows_ok:
        # a short causal span: each row as the decode step attends (no mask reads)
        y = fastpath.causal_rows_attention(q_rows, kc, vc, input_pos, nh, nkv, mask.shape[-1])
    if y is None:
        if mask.shape[-1] < k.shape[2]:
            k, v = k[:, :, : mask.shape[-1]], v[:, :, : mask.shape[-1]]
        if causal and rows_ok and attend is not None:
            y = _attend_in_parts(q, kc, vc, input_pos, nh, nkv, attend)
        # a causal span's mask follows from its positions: computed in the kernel, not read
        if y is None:
            y = fastpath.prefill_attention(q, k, v, mask, nh, nkv, hd, positions=input_pos if causal else None)
        if y is None:
            y = fastpath.decode_attention(q, k, v, mask, nh, nkv, hd)
        y = y.transpose(1, 2).contiguous().view(bsz, n, nh * hd)
    hh = nf4gemv.matmul_norm(a.wo, y, fn.weight, fn.eps, epi=nf4gemv.EPI_RESIDUAL, operand=x, span=True, wide=wide)
    if hh is not None:
        h, hn = hh
    else:
        h = nf4gemv.matmul(a.wo, y, epi=nf4gemv.EPI_RESIDUAL, operand=x, wide=wide)
        hn = None
    u = None
    if hh is None and fold and h is not None:  # w1 and w3 with the FFN norm folded in: one launch, else two
        u = nf4gemv.matmul_fused(ff.w1, h, norm_weight=fn.weight, eps=fn.eps, module3=ff.w3)
        if u is None:
            g = nf4gemv.matmul_fused(ff.w1, h, norm_weight=fn.weight, eps=fn.eps)
            if g is not None:
                u = nf4gemv.matmul_fused(ff.w3, h, norm_weight=fn.weight, eps=fn.eps, epi=nf4gemv.EPI_SILU_GATE,
                                         operand=g)
    if u is None and hn is None and h is not None:
        hn = fusedops.rms_norm(h, fn.weight, fn.eps)
    # w1 and w3 with the SwiGLU gate in one launch where it serves the shape, else two
    if u is None and hn is not None:
        u = nf4gemv.matmul_swiglu(ff.w1, ff.w3, hn, wide=wide)
    if u is None and hn is not None:
        g = nf4gemv.matmul(ff.w1, hn, wide=wide)
        u = None if g is None else nf4gemv.matmul(ff.w3, hn, epi=nf4gemv.EPI_SILU_GATE, operand=g, wide=wide)
    oo = None
    if u is not None and next_norm is not None:
        oo = nf4gemv.matmul_norm(ff.w2, u, next_norm.weight, next_norm.eps, epi=nf4gemv.EPI_RESIDUAL, operand=h,
                                 span=True, wide=wide)
    if oo is not None:
        out, out_n = oo
    else:
        out = None if u is None else nf4gemv.matmul(ff.w2, u, epi=nf4gemv.EPI_RESIDUAL, operand=h, wide=wide)
        out_n = None
        if out is not None and next_norm is not None and not fold:  # (a short span's next block folds it)
            out_n = fusedops.rms_norm(out, next_norm.weight, next_norm.eps)
    if out is None:
        raise RuntimeError("prefill_block: a GEMM declined after the KV cache was written")
    _stats["prefill"] += 1
    return out, out_n


def spans_keep_order(block, next_norm=None) -> bool:
    """Whether `prefill_block_chain` gives 512-row spans the same bits run
    together (`attend`: 512 rows a launch) as one by one: where the attention
    kernel takes the heads and every product of 1024 to 2048 rows adds its K as
    its 512-row form in the block does."""
    from ttspipe_amd import nf4gemv

    a, ff = block.attention, block.feed_forward
    lib = _lib.lib()
    if a.head_dim != HEAD_DIM or a.n_head // a.n_local_heads > lib.ttsp_prefill_max_groups():
        return False

    def keeps(linear, summed: bool, norm=None) -> bool:
        # summed: the block adds the partial sums of ttsp_nf4_gemm_splits itself (with the next norm); else `matmul`
        if not nf4gemv.prepare(linear):
            return False
        M, K = linear._nf4_fast["M"], linear._nf4_fast["K"]
        if summed and norm is not None:
            summed = M <= nf4gemv.NORM_MAX_M and M % 8 == 0 and norm.weight.data_ptr() % 16 == 0
        parts = lib.ttsp_nf4_gemm_splits(M, K, 512)
        if not summed or parts == 1:
            parts = lib.ttsp_nf4_gemm_tile_splits(M, K, 512)
        return lib.ttsp_nf4_gemm_span_splits(M, K) == parts

    return (keeps(a.wqkv, True) and keeps(a.wo, True, block.ffn_norm) and keeps(ff.w1, False) and keeps(ff.w3, False)
            and keeps(ff.w2, next_norm is not None, next_norm))


def install() -> bool:
    """Patch `TransformerBlock.forward`: one-position calls go to `decode_block`,
    multi-position calls to `prefill_block`, anything either declines to the
    block's own forward."""
    global _installed
    if not _lib.gpu_present():
        return False
    _lib.load()
    for cls in _block_classes():
        if getattr(cls, "_fused_patched", False):
            continue
        original = cls.forward

        def forward(self, x, freqs_cis, mask, input_pos=None, _original=original):
            out = decode_block(self, x, freqs_cis, mask, input_pos)
            if out is None and x.dim() == 3 and x.shape[1] > 1:
                out = prefill_block(self, x, freqs_cis, mask, input_pos)
            if out is not None:
                return out
            if x.shape[1] == 1:
                _stats["fallback"] += 1
            return _original(self, x, freqs_cis, mask, input_pos)

        cls.forward = forward
        cls._fused_patched = True
        cls._fused_original_forward = original
    _installed = True
    return True
