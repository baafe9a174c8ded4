"""PPO's value side: KL-penalised token rewards, GAE, masked whitening and the critic loss.

Host-side mirror of ``AdaptiveKLController``, the arithmetic inside ``apply_kl_penalty`` and
``compute_gae_advantage_return`` (``mindspeed_rl/trainer/utils/compute_utils.py:33-48,80-97,107-149``),
``masked_var`` / ``masked_whiten`` (``mindspeed_rl/utils/torch_functional.py:62-106``) and
``CriticLossFunc`` (``mindspeed_rl/models/loss/critic_loss_func.py``), with the reference's names,
signatures and error behaviour; the arithmetic runs in the kernels of ``csrc/value_path.hip``.
"""
import ctypes
from typing import Dict, Tuple

import numpy as np
import torch

from . import _lib
from .loss import BaseLossFunc, LossFuncFactory, _dynamic_scale, _mask_args
from .packing import postprocess_packed_seqs, truncate_middle_and_pad


class AdaptiveKLController:
    """Reference: ``trainer/utils/compute_utils.py:33-48``."""

    def __init__(self, init_kl_coef, target_kl, horizon):
        self.value = init_kl_coef
        self.target = target_kl
        self.horizon = horizon

    def update(self, current_kl, n_steps):
        proportional_error = np.clip(current_kl / self.target - 1, -0.2, 0.2)
        mult = 1 + proportional_error * n_steps / self.horizon
        self.value *= mult


def _f32(t, dev):
    """Outside of autograd (what the kernels get is the address)."""
    if t.dtype is torch.float32 and t.is_contiguous() and t.device == dev:
        return t
    return _lib.dense(t.detach(), torch.float32, dev)


def kl_token_level_rewards(old_log_prob, ref_log_prob, response_length, rm_scores, beta, penalty="kl"):
    """The arithmetic of ``apply_kl_penalty`` (``compute_utils.py:80-97``) for one padded batch:
    ``(token_level_rewards [B, L], current_kl)`` where the reward of sample ``i`` is its score at the
    last response token minus ``beta`` times the masked KL penalty, and ``current_kl`` (a python
    float, the value handed to ``kl_ctrl.update``) is the batch mean of the per-sample masked means."""
    if penalty not in _lib.KL_BY_NAME:
        raise NotImplementedError
    dev = _lib.require_device(old_log_prob, ref_log_prob)
    old, ref = _f32(old_log_prob, dev), _f32(ref_log_prob, dev)
    batch, width = old.shape
    lens = _lib.index_column(response_length, dev)
    scores = _f32(torch.as_tensor(rm_scores), dev)
    if lens.numel() != batch or scores.numel() != batch:
        raise ValueError("response_length and rm_scores need one entry per sample")
    rewards = torch.empty_like(old)
    args = (_lib.ptr(old), _lib.ptr(ref), _lib.ptr(lens), _lib.dtype_code(lens), _lib.ptr(scores), batch, width,
            _lib.KL_BY_NAME[penalty], float(beta), _lib.ptr(rewards))
    slot = _lib.HostWords.take(dev, 4 * batch) if batch > 0 else None
    # the host waits for the kernel either way: the mean of `batch` numbers is taken where they land
    if slot is not None:
        slot.launch("mrl_kl_token_rewards", *args, slot.addr, _lib.stream(dev))
        row_kl = slot.read_doubles_of(batch, _lib.stream(dev))
    else:
        row_kl = torch.empty(batch, dtype=torch.float32, device=dev)
        _lib.call("mrl_kl_token_rewards", *args, _lib.ptr(row_kl), _lib.stream(dev))
        row_kl = row_kl.cpu().double()
    return rewards, torch.mean(row_kl, dim=0).float().item()


def _whiten(values, mask, shift_mean):
    dev = _lib.require_device(values, mask)
    x = _f32(values, dev)
    m, _ = _mask_args(mask.expand_as(values) if mask.shape != values.shape else mask, None, dev)
    out = torch.empty_like(x)
    info = torch.empty(3, dtype=torch.float64, device=dev)
    _lib.call("mrl_masked_whiten", _lib.ptr(x), _lib.ptr(m), _lib.dtype_code(m), x.numel(), 1 if shift_mean else 0,
              _lib.ptr(out), _lib.ptr(info), _lib.stream(dev))
    return out, info


def masked_var(values, mask, unbiased=True):
    """Reference: ``torch_functional.py:62-87``; a 0-d fp32 tensor.  ``unbiased=False`` undoes the
    Bessel correction the kernel applies."""
    _, info = _whiten(values, mask, True)
    count, _, var = info.cpu().tolist()
    if unbiased and count == 0:
        raise ValueError("At least one element in the mask has to be 1.")
    if not unbiased and count > 1:
        var = var * (count - 1) / count
    return torch.tensor(var, dtype=torch.float32, device=values.device)


def masked_whiten(values, mask, shift_mean=True):
    """Reference: ``torch_functional.py:90-106``."""
    out, info = _whiten(values, mask, shift_mean)
    if info[0].item() == 0:
        raise ValueError("At least one element in the mask has to be 1.")
    return out.view(values.shape)


def compute_gae_advantage_return(token_level_rewards, values, eos_mask, gamma, lam):
    """Reference: ``compute_utils.py:107-149``.  The reverse scan runs over the full width (the mask
    only enters the whitening) with the reference's fp32 operation order, so ``returns`` and the
    advantages before whitening are bit-identical to the torch loop."""
    dev = _lib.require_device(token_level_rewards, values, eos_mask)
    rewards, vals = _f32(token_level_rewards, dev), _f32(values, dev)
    if rewards.dim() != 2 or rewards.shape != vals.shape:
        raise ValueError("token_level_rewards and values must both be [batch, response_length]")
    batch, width = rewards.shape
    mask, _ = _mask_args(eos_mask.expand_as(rewards) if eos_mask.shape != rewards.shape else eos_mask, None, dev)
    adv = torch.empty_like(rewards)
    ret = torch.empty_like(rewards)
    small = torch.empty(3 + 3 * batch, dtype=torch.float64, device=dev)     # info, then the rows' moments
    # `gamma * lam` as python evaluates it inside the reference's `gamma * lam * lastgaelam`: in double
    # for python floats (the config's values), in the tensors' own precision for 0-dim tensors
    decays = float(gamma), float(gamma * lam)
    # whether the mask is empty is all that the host waits for: its rows' sums leave before the scan has ended (whole
    # numbers, so their sum has no order)
    slot = _lib.HostWords.take(dev, 8 * batch) if batch > 0 and mask.dtype is not torch.float32 else None
    launch = _lib.call if slot is None else slot.launch
    launch("mrl_gae_whiten_host", _lib.ptr(rewards), _lib.ptr(vals), _lib.ptr(mask), _lib.dtype_code(mask), batch, width,
           *decays, _lib.ptr(adv), _lib.ptr(ret), small.data_ptr(), slot.addr if slot is not None else None,
           small.data_ptr() + 24, 24 * batch, _lib.stream(dev))
    count = sum(slot.read(ctypes.c_double, batch, _lib.stream(dev))) if slot is not None else small[0].item()
    if count == 0:
        raise ValueError("At least one element in the mask has to be 1.")
    return adv, ret


class _ValueLoss(torch.autograd.Function):
    """vpreds [B, L] -> (scaled loss, out[4]) through mrl_value_loss_fwd / _bwd."""

    @staticmethod
    def forward(ctx, vpreds, returns, values, mask, lens, clip, loss_scale):
        dev = _lib.require_device(vpreds, returns, values, mask, lens)
        vp = vpreds.to(torch.float32).contiguous()
        ret, val = _f32(returns, dev), _f32(values, dev)
        batch, width = vp.shape
        out = torch.empty(4, dtype=torch.float32, device=dev)
        loss = torch.empty((), dtype=torch.float32, device=dev)     # autograd outputs must not alias
        ws_bytes = _lib.load().mrl_value_loss_workspace_bytes(batch)
        workspace = torch.empty(ws_bytes, dtype=torch.uint8, device=dev)
        _lib.call("mrl_value_loss_fwd_split", _lib.ptr(vp), _lib.ptr(ret), _lib.ptr(val), _lib.ptr(mask),
                  _lib.dtype_code(mask) if mask is not None else _lib.F32, _lib.ptr(lens),
                  _lib.dtype_code(lens) if lens is not None else _lib.I32, batch, width, float(clip), float(loss_scale),
                  _lib.ptr(out), _lib.ptr(loss), _lib.ptr(workspace), ws_bytes, _lib.stream(dev))
        ctx.save_for_backward(vp, ret, val, mask, lens, out)
        ctx.scalars = (float(clip), float(loss_scale))
        ctx.in_dtype = vpreds.dtype
        ctx.mark_non_differentiable(out)
        return loss, out

    @staticmethod
    def backward(ctx, g_loss, _g_out):
        vp, ret, val, mask, lens, out = ctx.saved_tensors
        dev = vp.device
        batch, width = vp.shape
        upstream = g_loss.to(torch.float32).reshape(1).contiguous()
        g = torch.empty_like(vp)
        _lib.call("mrl_value_loss_bwd", _lib.ptr(vp), _lib.ptr(ret), _lib.ptr(val), _lib.ptr(mask),
                  _lib.dtype_code(mask) if mask is not None else _lib.F32, _lib.ptr(lens),
                  _lib.dtype_code(lens) if lens is not None else _lib.I32, batch, width, *ctx.scalars, _lib.ptr(out),
                  _lib.ptr(upstream), _lib.ptr(g), _lib.stream(dev))
        return g.to(ctx.in_dtype), None, None, None, None, None, None


class _CriticLoss(torch.autograd.Function):
    """The value head's output [B, S, 1] -> (scaled loss, out[4]) through mrl_critic_loss_fwd_slope / _bwd: the response
    windows are read and their gradients written where they lie.  The head's output is not kept: the caller may
    overwrite it before the backward."""

    @staticmethod
    def forward(ctx, head, prompt, lens, returns, values, clip, loss_scale, sent):
        dev = _lib.require_device(head, prompt, lens, returns, values)
        head = head.contiguous()
        ret, val = _f32(returns, dev), _f32(values, dev)
        (batch, padded, _), width = head.shape, ret.shape[1]
        out = torch.empty(4, dtype=torch.float32, device=dev)
        loss = torch.empty((), dtype=torch.float32, device=dev)     # autograd outputs must not alias
        slope = torch.empty_like(ret)
        ws_bytes = _lib.load().mrl_value_loss_workspace_bytes(batch)
        workspace = torch.empty(ws_bytes, dtype=torch.uint8, device=dev)
        clip, loss_scale = float(clip), float(loss_scale)
        slot = _lib.HostWords.take(dev, 16) if sent is not None else None
        launch = _lib.call if slot is None else slot.launch
        launch("mrl_critic_loss_fwd_slope_host", _lib.ptr(head), batch, padded, _lib.ptr(prompt), _lib.dtype_code(prompt),
               _lib.ptr(lens), _lib.dtype_code(lens), _lib.ptr(ret), _lib.ptr(val), width, clip, loss_scale,
               _lib.ptr(slope), _lib.ptr(out), _lib.ptr(loss), slot.addr if slot is not None else None,
               _lib.ptr(workspace), ws_bytes, _lib.stream(dev))
        if slot is not None:
            sent.append(slot)
        ctx.save_for_backward(slope, prompt, lens, out)
        ctx.meta = (tuple(head.shape), loss_scale)
        ctx.mark_non_differentiable(out)
        ctx.set_materialize_grads(False)
        return loss, out

    @staticmethod
    def backward(ctx, g_loss, _g_out):
        if g_loss is None:
            return (None,) * 8
        slope, prompt, lens, out = ctx.saved_tensors
        shape, loss_scale = ctx.meta
        dev = slope.device
        upstream = _lib.dense(g_loss, torch.float32, dev)
        g = torch.empty(shape, dtype=torch.float32, device=dev)
        _lib.call("mrl_critic_loss_bwd_slope", _lib.ptr(slope), shape[0], shape[1], _lib.ptr(prompt), _lib.dtype_code(prompt),
                  _lib.ptr(lens), _lib.dtype_code(lens), slope.shape[1], loss_scale, _lib.ptr(out), _lib.ptr(upstream),
                  _lib.ptr(g), _lib.stream(dev))
        return g, None, None, None, None, None, None, None


def value_loss(vpreds, returns, values, response_mask=None, response_length=None, *, cliprange_value,
               loss_scale=1.0):
    """Clipped value loss: ``(loss_scale * vf_loss, out)`` with ``out = [scaled loss, vf_loss,
    vf_clipfrac, sum(mask)]`` on the device; differentiable with respect to ``vpreds`` ``[B, L]``."""
    dev = _lib.require_device(vpreds)
    if vpreds.dim() != 2:
        raise ValueError("vpreds must be [batch, response_length]")
    mask, lens = _mask_args(response_mask, response_length, dev)
    return _ValueLoss.apply(vpreds, returns, values, mask, lens, cliprange_value, loss_scale)


@LossFuncFactory.register_loss("ray_ppo", "critic")
class CriticLossFunc(BaseLossFunc):
    """Reference: ``critic_loss_func.py:14-111``."""

    def __init__(self):
        super(CriticLossFunc, self).__init__()
        self.cliprange_value = 0.5

    def add_loss_meta_info(self, meta_info: Dict):
        if meta_info is None:
            return
        if "cliprange_value" in meta_info.keys():
            self.cliprange_value = float(meta_info["cliprange_value"])

    @staticmethod
    def _get_policy_loss_input(batch: Dict[str, torch.Tensor]):
        if "responses" not in batch:
            raise ValueError("The responses is None")
        values = batch["values"] if "values" in batch else None
        returns = batch["returns"] if "returns" in batch else None
        response_length = batch["response_length"]
        from .packing import generate_mask
        response_mask = generate_mask(batch["responses"], response_length)
        return response_mask, values, returns, response_length

    @staticmethod
    def _get_compute_vpreds(output: torch.Tensor, batch: Dict[str, torch.Tensor]):
        if "responses" not in batch:
            raise ValueError("The responses is None")
        responses = batch["responses"]
        truncate_lengths = torch.cat([batch["prompt_length"], batch["prompt_length"] + batch["response_length"]],
                                     dim=1) - 1
        return truncate_middle_and_pad(responses, output, truncate_lengths)

    def _reads_windows_in_place(self, output, batch):
        """The value head's own layout, fp32 [B, S, 1] with [B, 1] lengths and [B, L] operands that belong to
        it: what the loss kernels read without a copy of the windows."""
        if type(self)._get_compute_vpreds is not CriticLossFunc._get_compute_vpreds:
            return False                    # a subclass cuts them itself
        if not (output.is_cuda and output.dim() == 3 and output.shape[2] == 1 and output.dtype is torch.float32):
            return False
        shape = tuple(batch["responses"].shape)
        columns = (batch["prompt_length"], batch["response_length"])
        rows = (batch.get("returns"), batch.get("values"))
        return (len(shape) == 2 and shape[0] == output.shape[0] and shape[1] > 0
                and all(tuple(c.shape) == (shape[0], 1) and c.dtype in (torch.int32, torch.int64) for c in columns)
                and all(t is not None and tuple(t.shape) == shape for t in rows))

    def compute_loss(self, output: torch.Tensor, batch: Dict[str, torch.Tensor], forward_only=False,
                     non_loss_data=True, **kwargs) -> Tuple[torch.Tensor, Dict]:
        if kwargs.get("use_remove_padding", False):
            output = postprocess_packed_seqs(output=output, seqlens_in_batch=kwargs.get("seqlens_in_batch", None),
                                             cu_seqlens_padded=kwargs.get("cu_seqlens_padded", None),
                                             seq_len=kwargs.get("seq_len", None))
        if not forward_only and "responses" in batch and self._reads_windows_in_place(output, batch):
            sent = []
            loss, out = _CriticLoss.apply(output, batch["prompt_length"].contiguous(), batch["response_length"].contiguous(),
                                          batch["returns"], batch["values"], self.cliprange_value,
                                          _dynamic_scale(batch, forward_only, kwargs), sent)
            return loss, self._statistics(out, sent)
        vpreds = self._get_compute_vpreds(output, batch)
        if forward_only:
            return vpreds
        if "responses" not in batch:
            raise ValueError("The responses is None")
        scale = _dynamic_scale(batch, forward_only, kwargs)
        # the mask is (j < response_length), evaluated inside the kernel
        loss, out = value_loss(vpreds.reshape(vpreds.shape[0], vpreds.shape[1]), batch.get("returns"),
                               batch.get("values"), None, batch["response_length"],
                               cliprange_value=self.cliprange_value, loss_scale=scale)
        return loss, self._statistics(out)

    @staticmethod
    def _statistics(out, sent=()):
        # the slot that the kernel left them in, else one device-to-host copy for both statistics
        host = sent[0].read(ctypes.c_float, 4, _lib.stream(out.device)) if sent else out.detach().cpu().tolist()
        return {"critic/vf_loss": abs(host[1]), "critic/vf_clipfrac": host[2]}

    @staticmethod
    def _compute_value_loss(vpreds, returns, values, response_mask, cliprange_value):
        """``(vf_loss, vf_clipfrac)`` as 0-d tensors (``critic_loss_func.py:82-111``)."""
        vp = vpreds.squeeze()
        if vp.dim() == 1:
            vp = vp.unsqueeze(0)
        loss, out = value_loss(vp, returns.reshape(vp.shape), values.reshape(vp.shape),
                               response_mask.reshape(vp.shape), None, cliprange_value=cliprange_value)
        return loss, out[2]
