"""Fused lm_head + log-prob: hidden states and the vocabulary projection weight go in, per-token
log-prob / entropy / logsumexp come out, and the ``[T, V]`` logits are never written to memory.

The reference has no such function: ``GPTModel.output_layer`` materialises the logits and
``compute_log_probs`` (``mindspeed_rl/utils/compute.py:29-51``) reads them back.  This is the
forward-only form, which serves ``compute_log_prob`` / ``compute_ref_log_prob`` (two of the three
vocabulary sweeps of a GRPO iteration).
"""
import ctypes

import torch

from . import _lib, vocab_ops

# Cells that a scoring pass's result may have beyond the rows for these to be found with their cells (score_windows):
# the two tables of them take 8 bytes a cell, 32 MiB here, which a result of one long response among many short ones
# would make twice the memory of a pass without gaining more than before.  us and MiB a pass, flagged rows / this
# way, 64-wide hidden states: 64 x 4 096 cells 88, 2 / 46, 5; 2 048 x 2 048 87, 33 / 60, 69; 512 x 16 384 88, 64 / 52, 131;
# 1 024 x 32 768 150, 257 / 90, 519.
_EXTRA_CELLS = 1 << 22

# (name, start, end, rows) appended per call when set to a list, like vocab_ops.kernel_events
kernel_events = None


def _timed(name, rows, dev, *args):
    """_lib.call with HIP events around it when kernel_events is a list."""
    if kernel_events is None:
        _lib.call(name, *args)
        return
    start, end = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
    stream = torch.cuda.current_stream(dev)
    start.record(stream)
    _lib.call(name, *args)
    end.record(stream)
    kernel_events.append((name, start, end, rows))


def lmhead_logprob(hidden, weight, labels, inv_temperature=1.0, want_entropy=True, row_active=None):
    """``hidden`` ``[..., H]`` bf16, ``weight`` ``[V, H]`` bf16 (``nn.Linear`` layout), ``labels``
    ``[...]`` int32/int64 -> ``(logp, entropy, lse)`` fp32 shaped like ``labels`` (entropy is zeros
    if not wanted).  No autograd: use it under ``torch.no_grad()`` for old / reference log-probs.
    ``row_active`` (bool / integer, shaped like ``labels``): only rows with a non-zero flag are
    projected and scored, the others return 0 in all three outputs (one host synchronisation reads
    the number of active rows)."""
    if row_active is not None:
        if tuple(row_active.shape) != tuple(labels.shape):
            raise ValueError("row_active must have the shape of labels")
        dev = _lib.require_device(hidden, weight, labels, row_active)
        hdim, n_all = hidden.shape[-1], labels.numel()
        flags = row_active.reshape(-1)
        if flags.dtype is not torch.uint8:
            flags = (flags != 0).view(torch.uint8)
        rows = _LiveRows(flags.contiguous(), _lib.U8, 1, n_all, dev)
        out = torch.zeros if rows.n == 0 else torch.empty
        full = out((3, n_all), dtype=torch.float32, device=dev)
        if rows.n > 0:
            if hidden.dtype != torch.bfloat16 or weight.dtype != torch.bfloat16:
                raise TypeError("hidden and weight must be bfloat16")
            flat = hidden.detach().reshape(-1, hdim)
            if flat.shape[0] < n_all:           # rows behind the last label count as little as inactive ones
                raise ValueError("labels shape %s does not match hidden leading shape %s"
                                 % (tuple(labels.shape), tuple(hidden.shape[:-1])))
            lab = _lib.index_column(labels, dev)
            h, y, _ = rows.gather(flat, lab, None)
            part = torch.empty((3, rows.n), dtype=torch.float32, device=dev)
            _forward(h, weight, y, inv_temperature, part[0], part[1] if want_entropy else None, part[2])
            if not want_entropy:
                part[1].zero_()
            rows.spread_scalars(part, full)
        return tuple(full[k].view(labels.shape) for k in range(3))
    dev = _lib.require_device(hidden, weight, labels)
    if hidden.dtype != torch.bfloat16 or weight.dtype != torch.bfloat16:
        raise TypeError("hidden and weight must be bfloat16")
    hdim = hidden.shape[-1]
    if weight.dim() != 2 or weight.shape[1] != hdim:
        raise ValueError("weight must have shape (vocab, hidden_dim)")
    lead = hidden.shape[:-1]
    if tuple(labels.shape) != tuple(lead):
        raise ValueError("labels shape %s does not match hidden leading shape %s" % (tuple(labels.shape), tuple(lead)))
    h = hidden.detach().reshape(-1, hdim).contiguous()
    lab = _lib.index_column(labels, dev)
    n_tokens = h.shape[0]
    logp = torch.empty(n_tokens, dtype=torch.float32, device=dev)
    lse = torch.empty(n_tokens, dtype=torch.float32, device=dev)
    ent = torch.empty(n_tokens, dtype=torch.float32, device=dev) if want_entropy else None
    _forward(h, weight, lab, inv_temperature, logp, ent, lse)
    ent_out = ent.view(lead) if want_entropy else torch.zeros(lead, dtype=torch.float32, device=dev)
    return logp.view(lead), ent_out, lse.view(lead)


def score_windows(hidden, weight, labels, windows, inv_temperature, want_entropy):
    """A scoring pass from the hidden states: ``(log_probs, entropy)`` ``[B, L]`` of the rows of ``windows`` (a
    :class:`packing.ResponseWindows`), or None where that is not the way and :func:`lmhead_logprob` takes the flagged
    rows (or refuses them).  One launch finds the rows and their cells, one gathers them, and the forward leaves its
    results in the cells: flags, count, positions, spread and cut were six launches more.  us a pass, before -> now:
    9 477 rows x 18 840 x 640 271 -> 255, 1 944 x 42 384 x 1 344 239 -> 220, 9 134 x 14 968 x 1 344 341 -> 326."""
    if not (hidden.is_cuda and hidden.dtype is weight.dtype is torch.bfloat16 and weight.dim() == 2
            and weight.shape[1] == hidden.shape[-1] and tuple(labels.shape) == tuple(hidden.shape[:-1])):
        return None
    if not (0 < windows.n_seq <= windows.MAX_CELL_SEQS and windows.width > 0 and windows.n_rows > 0):
        return None
    cells = windows.n_seq * windows.width
    if cells > windows.n_rows + _EXTRA_CELLS or cells > 0x7fffffff or vocab_ops._transformed():
        return None
    dev = _lib.require_device(hidden, weight, labels, windows.prompt)
    found = windows.cells(want_entropy)
    if found is None:
        return None
    slot, index, p_live, p_cell, logp, ent = found
    (n,) = slot.read(ctypes.c_int64, 1, _lib.stream(dev))
    if n > 0:
        flat = hidden.detach().reshape(-1, hidden.shape[-1])
        h, y, _ = _gather_rows(p_live, n, flat, _lib.index_column(labels, dev), None, dev)
        _forward(h, weight, y, inv_temperature, logp, ent if want_entropy else None, None, p_cell)
    return logp, ent


def _gather_rows(p_index, n, table, labels, ops, dev):
    """Rows index[0 .. n - 1] of `table` [., W] (W whole 16-byte vectors), of `labels` and - unless None - of `ops`
    [., 8] fp32."""
    table = table.contiguous()
    if table.data_ptr() % 16:
        table = table.clone()
    out = torch.empty((n, table.shape[1]), dtype=table.dtype, device=dev)
    lab = torch.empty(n, dtype=labels.dtype, device=dev)
    few = None if ops is None else torch.empty((n, 8), dtype=torch.float32, device=dev)
    _lib.call("mrl_move_rows", p_index, n, _lib.ptr(table), _lib.ptr(out), table.shape[1] * table.element_size(),
              _lib.ptr(ops), _lib.ptr(few), 0 if ops is None else 32, _lib.ptr(labels), _lib.ptr(lab), labels.element_size(),
              _lib.stream(dev))
    return out, lab, few


def _forward(h, weight, lab, inv_temperature, logp, ent, lse, p_cells=None):
    """The forward of dense rows into the given outputs (ent None: not wanted), or into cells of them."""
    dev, w = h.device, weight.detach().contiguous()
    if w.dim() != 2 or w.shape[1] != h.shape[1]:
        raise ValueError("weight must have shape (vocab, hidden_dim)")
    (n_tokens, hdim), vocab = h.shape, w.shape[0]
    ws_bytes = _lib.load().mrl_lmhead_workspace_bytes(n_tokens, vocab)
    workspace = torch.empty(max(ws_bytes, 16), dtype=torch.uint8, device=dev)
    name = "mrl_lmhead_logprob_fwd" if p_cells is None else "mrl_lmhead_logprob_fwd_cells"
    outputs = (_lib.ptr(logp), _lib.ptr(ent), _lib.ptr(lse)) if p_cells is None else (p_cells, _lib.ptr(logp), _lib.ptr(ent))
    args = (_lib.ptr(h), _lib.ptr(w), n_tokens, vocab, hdim, _lib.ptr(lab), _lib.dtype_code(lab),
            float(inv_temperature), *outputs, _lib.ptr(workspace), ws_bytes, _lib.stream(dev))
    if kernel_events is None:
        _lib.call(name, *args)
    else:
        start, end = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
        stream = torch.cuda.current_stream(dev)
        start.record(stream)
        _lib.call(name, *args)
        end.record(stream)
        kernel_events.append(("mrl_lmhead_logprob_fwd", start, end, n_tokens))


class _LiveRows:
    """The rows with a non-zero flag: how many (one host read), which, and moves there and back."""

    def __init__(self, flags, dtype, stride, n, dev):
        self.dev, self.n_all = dev, n
        blocks = (n + 1023) // 1024
        index = torch.empty(2 * n + blocks, dtype=torch.int32, device=dev)
        self.live, self.place = index[:n], index[n:2 * n]
        args = (flags if isinstance(flags, int) else _lib.ptr(flags), dtype, stride, n,
                index.data_ptr(), index.data_ptr() + 4 * n, index.data_ptr() + 8 * n)
        slot = _lib.HostWords.take(dev, 8) if n > 0 else None
        if slot is not None:
            slot.launch("mrl_live_rows", *args, slot.addr, _lib.stream(dev))
            (self.n,) = slot.read(ctypes.c_int64, 1, _lib.stream(dev))
        else:
            total = torch.empty(1, dtype=torch.int64, device=dev)
            _lib.call("mrl_live_rows", *args, _lib.ptr(total), _lib.stream(dev))
            self.n = int(total.item()) if n > 0 else 0

    def gather(self, table, labels, ops):
        """The live rows of the tables, see :func:`_gather_rows`."""
        return _gather_rows(_lib.ptr(self.live), self.n, table, labels, ops, self.dev)

    def spread(self, table, out, terms, p_terms_out):
        """Back to all rows, zeros in the others: `table` [n_live, W] to `out`, `terms` [n_live, 8] to an address."""
        _lib.call("mrl_move_rows", _lib.ptr(self.place), self.n_all, _lib.ptr(table), _lib.ptr(out),
                  table.shape[1] * table.element_size(), _lib.ptr(terms), p_terms_out, 32, None, None, 0,
                  _lib.stream(self.dev))

    def spread_scalars(self, part, full):
        _lib.call("mrl_spread_scalars", _lib.ptr(part), self.n, part.shape[0], _lib.ptr(self.place), self.n_all,
                  _lib.ptr(full), _lib.stream(self.dev))


def _round_up(x, to):
    return (x + to - 1) // to * to


class _FusedLmHeadLoss(torch.autograd.Function):
    """(hidden, weight) -> (loss, out[8]) with dHidden and dWeight produced during the forward.

    The rows are processed in chunks: ``logits_c = hidden_c @ weight^T`` (``mrl_lmhead_logits``),
    the fused sweep turns the chunk into dlogits in place (one read, one write), then
    ``dHidden_c = dlogits_c @ weight`` and ``dWeight += dlogits_c^T @ hidden_c``
    (``mrl_lmhead_logprob_bwd_chunk``, fp32 accumulation across chunks in stream order).  All three
    products run on the hand-written bf16 MFMA kernels; only ``chunk_rows x V`` logits exist at any
    time."""

    @staticmethod
    def forward(ctx, hidden, weight, labels, batch, cfg):
        from .loss import _FusedOperands
        dev = _lib.require_device(hidden, weight, labels)
        hdim = hidden.shape[-1]
        h2d = hidden.detach().reshape(-1, hdim).contiguous()
        w = weight.detach().contiguous()
        n_rows, vocab = h2d.shape[0], w.shape[0]
        lab = labels.reshape(-1)
        if lab.dtype not in (torch.int32, torch.int64):
            lab = lab.to(torch.int64)
        lab = lab.contiguous()
        n_seq, width = batch["responses"].shape[0], batch["responses"].shape[-1]
        layout, padded_s = (0, 0) if cfg["packed"] else (1, hidden.shape[1])
        chunk_cap = max(1, min(int(cfg["chunk_rows"]), max(n_rows, 1)))
        ops = _FusedOperands(dev, batch, cfg, n_rows, n_seq, width, layout, padded_s, _lib.BF16, vocab, chunk_cap)
        stream = _lib.stream(dev)
        ops.prepare(stream)
        row_ops = ops.rows[:max(n_rows, 1) * 8]
        # Rows whose mask is zero (prompts, padding, masked tokens) add nothing to the loss, to dWeight or
        # to their own dHidden: when they are more than a twentieth of the rows, the live rows are gathered
        # and only they go through the products.  The row count sizes the products, so it is read back (one
        # host synchronisation per call; compact_rows=False avoids it).
        live = None
        if cfg["compact_rows"] and n_rows > 0:
            live = _LiveRows(ops.p_ops + 12, _lib.F32, 8, n_rows, dev)
            if live.n * 20 > n_rows * 19:
                live = None
        all_rows, h_all = n_rows, h2d
        p_ops, p_terms = ops.p_ops, ops.p_terms
        if live is not None:
            n_rows = live.n
            h2d, lab, row_ops = live.gather(h_all, lab, row_ops.view(-1, 8))
            row_terms = torch.empty((max(n_rows, 1), 8), dtype=torch.float32, device=dev)
            p_ops, p_terms = row_ops.data_ptr(), row_terms.data_ptr()
        chunk = max(1, min(chunk_cap, n_rows))
        # the chunk of logits: rows padded to whole k-steps of the dHidden product; the padding columns, up to 56, are
        # zeroed once and never written (they meet rows of the weight that read as zero).  Zeroing the whole chunk
        # took 146 us of 9.7 ms at 5 519 x 99 760 x 3 712.
        v_pad = _round_up(vocab, 64)
        logits = torch.empty((chunk, v_pad), dtype=h2d.dtype, device=dev)
        if v_pad != vocab:
            logits[:, vocab:].zero_()
        d_hidden = torch.empty_like(h2d)
        # dWeight leaves the last chunk's product as bf16; fp32 sums exist only between chunks.  In a step of one
        # chunk dHidden may be cut along the vocabulary and dWeight along the tokens, which groups their fp32 sums
        # by the number of rows; in several neither is, so that dHidden does not depend on the chunking.
        one_chunk = n_rows <= chunk
        d_weight = torch.empty((vocab, hdim), dtype=w.dtype, device=dev) if n_rows > 0 else torch.zeros_like(w)
        d_weight32 = None if one_chunk else torch.empty((vocab, hdim), dtype=torch.float32, device=dev)
        cut_bytes = _lib.load().mrl_lmhead_bwd_workspace_bytes(n_rows, vocab, hdim) if one_chunk else 0
        cut = torch.empty(cut_bytes, dtype=torch.uint8, device=dev) if cut_bytes else None
        esz = h2d.element_size()
        for c0 in range(0, n_rows, chunk):
            rows = min(n_rows, c0 + chunk) - c0
            h_c = h2d.data_ptr() + c0 * hdim * esz
            _timed("mrl_lmhead_logits", rows, dev, h_c, _lib.ptr(w), rows, vocab, hdim, _lib.ptr(logits), v_pad, stream)
            # the first sweep finds the workspace cleared by the prepare step, the others clear it themselves
            vocab_ops._timed_call(
                "mrl_fused_logprob_loss", rows, dev, _lib.ptr(logits), _lib.dtype_code(logits), rows, vocab, v_pad,
                lab.data_ptr() + c0 * lab.element_size(), _lib.dtype_code(lab), cfg["inv_temperature"],
                p_ops + c0 * 32, 0 if ops.old is None else 1, cfg["clip_lo"], cfg["clip_hi"], cfg["kl_penalty"],
                cfg["kl_coef"], cfg["entropy_coeff"], cfg["loss_scale"], ops.p_applied, _lib.ptr(logits), v_pad,
                None, ops.p_ent + c0 * 4 if ops.p_ent is not None else None, p_terms + c0 * 32, ops.workspace,
                ops.ws_bytes, 1 if c0 == 0 else 0, stream)
            _timed("mrl_lmhead_logprob_bwd_chunk", rows, dev, h_c, _lib.ptr(w), _lib.ptr(logits), v_pad, rows, vocab, hdim,
                   d_hidden.data_ptr() + c0 * hdim * esz, _lib.ptr(d_weight), _lib.ptr(d_weight32), 1 if c0 == 0 else 0,
                   1 if c0 + rows == n_rows else 0, _lib.ptr(cut), cut_bytes, stream)
        if live is not None:
            compact_dh = d_hidden
            d_hidden = torch.empty_like(h_all)
            live.spread(compact_dh, d_hidden, row_terms, ops.p_terms)
        ops.reduce(stream)
        applied = ops.applied
        ctx.save_for_backward(d_hidden, d_weight, applied)
        ctx.meta = (tuple(hidden.shape), cfg.get("scale_state"))
        ctx.handed_out = False
        ctx.mark_non_differentiable(ops.out)
        ctx.set_materialize_grads(False)
        return ops.loss, ops.out

    @staticmethod
    def backward(ctx, g_loss, _g_out):
        from .loss import _deliver_eager_grads
        if g_loss is None:
            return None, None, None, None, None
        d_hidden, d_weight, applied = ctx.saved_tensors
        shape, state = ctx.meta
        d_hidden, d_weight = _deliver_eager_grads(ctx, (d_hidden, d_weight), applied, state, g_loss)
        return d_hidden.view(shape), d_weight, None, None, None


def fused_lmhead_policy_loss(hidden, weight, batch, *, packed, seqlens=None, cu_seqlens=None, mask=None,
                             ref_log_prob=None, clip_low, clip_high, kl_penalty=None, kl_coef=0.0, entropy_coeff=0.0,
                             token_level_loss=True, loss_scale=1.0, inv_temperature=1.0, expected_upstream=None,
                             scale_state=None, chunk_rows=32768, compact_rows=True, sent=None):
    """Policy loss straight from the hidden states: ``hidden`` is packed ``[1, T, H]`` (or padded
    ``[B, S, H]``) bf16, ``weight`` the ``[V, H]`` bf16 lm_head weight; ``batch`` as for
    :func:`mindspeed_rl_amd.fused_logprob_policy_loss` (``labels, responses, response_length,
    prompt_length, advantages``, optional ``old_log_prob``).  Returns ``(loss, out)``; ``backward()``
    yields dHidden and dWeight.  Full ``[T, V]`` logits are never materialised: at most
    ``chunk_rows x V`` exist at a time.  ``hidden_dim`` must be a multiple of 64, ``V`` of 8 and at
    most ``mrl_fused_max_vocab`` (311 296); fp16 operands are not taken.  With ``compact_rows`` (default) rows without a live response token
    skip the GEMMs when they are more than 5 % of all rows; finding them costs one host
    synchronisation per call."""
    if kl_penalty is None:
        kl_code = _lib.KL_NONE
    elif kl_penalty in _lib.KL_BY_NAME:
        kl_code = _lib.KL_BY_NAME[kl_penalty]
    else:
        raise NotImplementedError
    if hidden.dtype != torch.bfloat16 or weight.dtype != torch.bfloat16:
        raise TypeError("hidden and weight must both be bfloat16")
    if hidden.shape[-1] % 64 != 0 or weight.shape[0] % 8 != 0:
        raise ValueError("hidden_dim must be a multiple of 64 and the vocabulary of 8")
    cfg = dict(packed=bool(packed), seqlens=seqlens, cu=cu_seqlens, mask=mask, ref_log_prob=ref_log_prob,
               clip_lo=float(1.0 - clip_low), clip_hi=float(1.0 + clip_high), kl_penalty=kl_code,
               kl_coef=float(kl_coef), entropy_coeff=float(entropy_coeff), seq_mean=0 if token_level_loss else 1,
               loss_scale=float(loss_scale), inv_temperature=float(inv_temperature),
               expected_upstream=None if expected_upstream is None else float(expected_upstream),
               scale_state=scale_state, chunk_rows=int(chunk_rows), compact_rows=bool(compact_rows), sent=sent)
    return _FusedLmHeadLoss.apply(hidden, weight, batch["labels"], batch, cfg)
