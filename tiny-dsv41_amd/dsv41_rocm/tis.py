"""Decoupled Token-TIS and GRPO losses on MI355X: the drop-ins for ``decoupled_token_tis_loss``
and ``grpo_loss``.

Reference (paths relative to the Tiny-DSV41 tree):

* ``dsv41_train/rl/algorithm.py:249-346`` — ``decoupled_token_tis_loss(policy_log_probs,
  native_old_log_probs, behavior_log_probs, advantages, clip_eps=0.2, is_cap=2.0)``: the
  loss ``mean_r(-mean_i(w * min(r A, clamp(r) A)))`` with detached weights
  ``w = f32(min(cap, exp(f64(old - behavior))))`` and ``r = exp(current - old)``, plus a
  metric dict; its argument checks and ``ValueError`` messages (``:268-312``).
* ``dsv41_train/rl/algorithm.py:169-246`` — ``grpo_loss(policy_log_probs, behavior_log_probs,
  advantages, clip_eps=0.2, ref_log_probs=None, kl_beta=0.0)``: the mean over responses of
  ``-mean(min(r A, clamp(r) A))`` plus ``kl_beta`` times the mean of the importance-weighted
  k3 KL, with its metric dict and checks.
* ``dsv41_train/rl/distributed_grpo.py:197-222`` — ``aggregate_token_tis_metrics``, the
  pooling of per-response metric rows; one call here over many responses returns the pooled
  values directly.

libdsv41hip.so computes the loss, its gradient with respect to ``current`` and every metric
in two launches with fixed reduction orders; the metrics come back in one host copy
(the reference takes one per metric).  ``current`` stays differentiable.
"""

from __future__ import annotations

import ctypes
import math
from typing import Sequence

import numpy as np
import torch

from . import _lib

METRIC_KEYS = (
    "loss", "policy_loss", "response_count", "token_count", "is_cap", "is_weight_sum",
    "is_weight_square_sum", "is_weight_mean", "is_weight_min", "is_weight_max", "is_raw_weight_sum",
    "is_raw_weight_min", "is_raw_weight_max", "is_clipped_tokens", "is_clipped_fraction",
    "is_dropped_weight_mass", "is_dropped_weight_mass_fraction", "is_token_weight_ess",
    "is_token_weight_ess_fraction", "native_old_minus_behavior_mean", "native_old_minus_behavior_max_abs",
    "native_ppo_ratio_mean", "native_ppo_clip_fraction",
)

# per-response status bits (include/dsv41_rocm.h) in the reference's check order, with its messages
_CHECKS = (
    (0x1, "policy log probabilities contains non-finite values"),
    (0x2, "policy log probabilities must be nonpositive"),
    (0x4, "native-old log probabilities contains non-finite values"),
    (0x8, "native-old log probabilities must be nonpositive"),
    (0x10, "behavior log probabilities contains non-finite values"),
    (0x20, "behavior log probabilities must be nonpositive"),
    (0x40, "raw rollout importance weights contains non-finite values"),
    (0x80, "raw rollout importance weights underflowed"),
    (0x100, "training rollout importance weights contains non-finite values"),
    (0x200, "training rollout importance weights underflowed"),
    (0x400, "native PPO ratios contains non-finite values"),
    (0x800, "native PPO ratios underflowed"),
    (0x1000, "each policy log-probability tensor must be a nonempty vector"),
    (0x2000, "advantages contains non-finite values"),
    (0x4000, "response offsets must be nondecreasing and within the token count"),
)


def _vector(value, like):
    """A detached float32 vector on like's device."""
    if type(value) is torch.Tensor and value.dtype == torch.float32 and value.device == like.device:
        return value.detach()  # (also where no gradient is required: a forward-mode tangent ends here too)
    return torch.as_tensor(value, dtype=torch.float32, device=like.device).detach()


def _upload(lengths, advantages, device):
    """The responses' offsets (int64 [R + 1]) and advantages (float32 [R]) on the device, in one
    copy where the advantages are on the host."""
    offsets = np.zeros(len(lengths) + 1, dtype=np.int64)
    np.cumsum(lengths, out=offsets[1:])
    if advantages.device.type != "cpu":
        return torch.from_numpy(offsets).to(device), advantages.to(device).contiguous()
    cut = offsets.nbytes
    host = torch.empty(cut + 4 * len(lengths), dtype=torch.uint8, device="cpu", pin_memory=True)
    view = host.numpy()
    view[:cut] = offsets.view(np.uint8)
    view[cut:] = advantages.contiguous().numpy().view(np.uint8)
    both = host.to(device, non_blocking=True)  # (torch keeps the pinned block until the copy is over)
    return both[:cut].view(torch.int64), both[cut:].view(torch.float32)


def _report(n_metrics, R, device):
    """Metrics (float64) and statuses (int32 [R]) in one block, so that they come back in one copy."""
    block = torch.empty(8 * n_metrics + 4 * R, dtype=torch.uint8, device=device)
    return block, block.data_ptr(), block.data_ptr() + 8 * n_metrics


def _read_report(block, n_metrics):
    host = block.cpu().numpy()
    return host[:8 * n_metrics].view(np.float64).tolist(), host[8 * n_metrics:].view(np.int32)


def _run(current, old, behavior, advantages, offsets, clip_eps, is_cap, want_grad):
    R = advantages.numel()
    dev = current.device
    loss = torch.empty((), dtype=torch.float32, device=dev)
    grad = torch.empty_like(current) if want_grad else None
    report, metrics, status = _report(len(METRIC_KEYS), R, dev)
    d = _lib.TokenTisDesc()
    d.struct_size = ctypes.sizeof(_lib.TokenTisDesc)
    d.n_responses, d.n_tokens = R, current.numel()
    d.offsets = offsets.data_ptr()
    d.current, d.native_old, d.behavior = current.data_ptr(), old.data_ptr(), behavior.data_ptr()
    d.advantages = advantages.data_ptr()
    d.clip_eps, d.is_cap = clip_eps, is_cap
    d.out_loss, d.out_metrics, d.out_status = loss.data_ptr(), metrics, status
    d.out_grad = grad.data_ptr() if grad is not None else None
    lib = _lib.load()
    ws_bytes = lib.dsv41_token_tis_workspace_bytes(ctypes.byref(d))
    ws = torch.empty(max(ws_bytes, 1), dtype=torch.uint8, device=dev)
    with torch.cuda.device(dev):
        rc = lib.dsv41_token_tis_run(ctypes.byref(d), ws.data_ptr(), ws_bytes, torch.cuda.current_stream(dev).cuda_stream)
    _lib.check(rc)
    return loss, grad, report


class _TokenTIS(torch.autograd.Function):
    @staticmethod
    def forward(ctx, current, old, behavior, advantages, offsets, clip_eps, is_cap):
        loss, grad, report = _run(current, old, behavior, advantages, offsets, clip_eps, is_cap, True)
        ctx.save_for_backward(grad)
        ctx.mark_non_differentiable(report)
        return loss, report

    @staticmethod
    def backward(ctx, g_loss, g_report):
        (grad,) = ctx.saved_tensors
        return grad * g_loss, None, None, None, None, None, None


def decoupled_token_tis_loss(
    policy_log_probs: Sequence[torch.Tensor],
    native_old_log_probs: Sequence,
    behavior_log_probs: Sequence,
    advantages,
    clip_eps: float = 0.2,
    is_cap: float = 2.0,
) -> tuple[torch.Tensor, dict[str, float]]:
    """Same arguments, checks, loss and metric dict as algorithm.py:249-346; the per-token
    work runs on the GPU holding ``policy_log_probs``."""
    if not math.isfinite(clip_eps) or not 0 <= clip_eps < 1:
        raise ValueError("clip_eps must be finite and in [0, 1)")
    if not math.isfinite(is_cap) or is_cap <= 0:
        raise ValueError("is_cap must be finite and positive")
    size = len(policy_log_probs)
    if size == 0 or len(native_old_log_probs) != size or len(behavior_log_probs) != size:
        raise ValueError("current, native-old and behavior require the same nonzero response count")
    advantage_values = torch.as_tensor(advantages, dtype=torch.float32).detach()
    if advantage_values.ndim != 1 or len(advantage_values) != size:
        raise ValueError("one scalar advantage is required per response")
    if not bool(torch.isfinite(advantage_values).all()):
        raise ValueError("advantages contains non-finite values")
    currents, olds, behaviors, lengths = [], [], [], []
    for index, current in enumerate(policy_log_probs):
        if not isinstance(current, torch.Tensor) or current.ndim != 1 or current.numel() == 0:
            raise ValueError("each policy log-probability tensor must be a nonempty vector")
        current = current.float()
        old = _vector(native_old_log_probs[index], current)
        behavior = _vector(behavior_log_probs[index], current)
        if old.shape != current.shape or behavior.shape != current.shape:
            raise ValueError("native-old, behavior and policy response lengths must match")
        currents.append(current)
        olds.append(old)
        behaviors.append(behavior)
        lengths.append(current.numel())
    dev = currents[0].device
    if dev.type != "cuda":
        raise ValueError("log probabilities must be on the GPU (libdsv41hip has no CPU path)")
    offsets, adv = _upload(lengths, advantage_values, dev)
    cur = torch.cat(currents)
    old = torch.cat(olds).contiguous()
    beh = torch.cat(behaviors).contiguous()
    if torch.is_grad_enabled() and cur.requires_grad:
        loss, report = _TokenTIS.apply(cur.contiguous(), old, beh, adv, offsets, clip_eps, is_cap)
    else:
        loss, _, report = _run(cur.detach().contiguous(), old, beh, adv, offsets, clip_eps, is_cap, False)
    values, st = _read_report(report, len(METRIC_KEYS))  # the one host copy
    for bits in st[st != 0].tolist():
        if bits:
            for bit, message in _CHECKS:
                if bits & bit:
                    raise ValueError(message)
    m = dict(zip(METRIC_KEYS, values))
    if not math.isfinite(m["loss"]):
        raise ValueError("Token-TIS loss contains non-finite values")
    if not math.isfinite(m["is_raw_weight_sum"]):
        raise ValueError("summed raw rollout importance weights contains non-finite values")
    if not math.isfinite(m["is_token_weight_ess"]):
        raise ValueError("token weight ESS contains non-finite values")
    m["is_cap"] = float(is_cap)
    return loss, m


GRPO_METRIC_KEYS = ("loss", "policy_loss", "kl", "clip_fraction", "importance_ratio", "approx_kl")

_GRPO_CHECKS = (
    (0x1, "policy log probabilities contains non-finite values"),
    (0x2, "behavior log probabilities contains non-finite values"),
    (0x4, "importance ratios (reduce policy lag or learning rate) contains non-finite values"),
    (0x8, "reference log probabilities contains non-finite values"),
    (0x10, "importance-weighted reference KL contains non-finite values"),
    (0x20, "each policy log-probability tensor must be a nonempty vector"),
    (0x40, "advantages contains non-finite values"),
    (0x80, "response offsets must be nondecreasing and within the token count"),
)


def _run_grpo(current, behavior, reference, advantages, offsets, clip_eps, kl_beta, want_grad):
    R = advantages.numel()
    dev = current.device
    loss = torch.empty((), dtype=torch.float32, device=dev)
    grad = torch.empty_like(current) if want_grad else None
    report, metrics, status = _report(len(GRPO_METRIC_KEYS), R, dev)
    d = _lib.GrpoDesc()
    d.struct_size = ctypes.sizeof(_lib.GrpoDesc)
    d.n_responses, d.n_tokens = R, current.numel()
    d.offsets = offsets.data_ptr()
    d.current, d.behavior = current.data_ptr(), behavior.data_ptr()
    d.reference = reference.data_ptr() if reference is not None else None
    d.advantages = advantages.data_ptr()
    d.clip_eps, d.kl_beta = clip_eps, kl_beta
    d.out_loss, d.out_metrics, d.out_status = loss.data_ptr(), metrics, status
    d.out_grad = grad.data_ptr() if grad is not None else None
    lib = _lib.load()
    ws_bytes = lib.dsv41_grpo_workspace_bytes(ctypes.byref(d))
    ws = torch.empty(max(ws_bytes, 1), dtype=torch.uint8, device=dev)
    with torch.cuda.device(dev):
        rc = lib.dsv41_grpo_run(ctypes.byref(d), ws.data_ptr(), ws_bytes, torch.cuda.current_stream(dev).cuda_stream)
    _lib.check(rc)
    return loss, grad, report


class _Grpo(torch.autograd.Function):
    @staticmethod
    def forward(ctx, current, behavior, reference, advantages, offsets, clip_eps, kl_beta):
        loss, grad, report = _run_grpo(current, behavior, reference, advantages, offsets, clip_eps, kl_beta, True)
        ctx.save_for_backward(grad)
        ctx.mark_non_differentiable(report)
        return loss, report

    @staticmethod
    def backward(ctx, g_loss, g_report):
        (grad,) = ctx.saved_tensors
        return grad * g_loss, None, None, None, None, None, None


def grpo_loss(
    policy_log_probs: Sequence[torch.Tensor],
    behavior_log_probs: Sequence,
    advantages,
    clip_eps: float = 0.2,
    ref_log_probs: Sequence | None = None,
    kl_beta: float = 0.0,
) -> tuple[torch.Tensor, dict[str, float]]:
    """Same arguments, checks, loss and metric dict as algorithm.py:169-246; the per-token
    work runs on the GPU holding ``policy_log_probs``."""
    if not math.isfinite(clip_eps) or not 0 <= clip_eps < 1:
        raise ValueError("clip_eps must be finite and in [0, 1)")
    if not math.isfinite(kl_beta) or kl_beta < 0:
        raise ValueError("kl_beta must be finite and nonnegative")
    size = len(policy_log_probs)
    if size == 0 or len(behavior_log_probs) != size:
        raise ValueError("policy and behavior must contain the same nonzero number of responses")
    advantage_values = torch.as_tensor(advantages, dtype=torch.float32).detach()
    if advantage_values.ndim != 1 or len(advantage_values) != size:
        raise ValueError("one scalar advantage is required per response")
    if not bool(torch.isfinite(advantage_values).all()):
        raise ValueError("advantages contains non-finite values")
    if ref_log_probs is not None and len(ref_log_probs) != size:
        raise ValueError("one reference log-probability vector is required per response")
    if kl_beta and ref_log_probs is None:
        raise ValueError("positive kl_beta requires reference log probabilities")
    currents, behaviors, references, lengths = [], [], [], []
    for index, current in enumerate(policy_log_probs):
        if current.ndim != 1 or current.numel() == 0:
            raise ValueError("each policy log-probability tensor must be a nonempty vector")
        current = current.float()
        behavior = _vector(behavior_log_probs[index], current)
        if behavior.shape != current.shape:
            raise ValueError("behavior and policy response lengths must match")
        if kl_beta:
            reference = ref_log_probs[index].to(device=current.device, dtype=torch.float32).detach()
            if reference.shape != current.shape:
                raise ValueError("reference and policy response lengths must match")
            references.append(reference)
        currents.append(current)
        behaviors.append(behavior)
        lengths.append(current.numel())
    dev = currents[0].device
    if dev.type != "cuda":
        raise ValueError("log probabilities must be on the GPU (libdsv41hip has no CPU path)")
    offsets, adv = _upload(lengths, advantage_values, dev)
    cur = torch.cat(currents)
    beh = torch.cat(behaviors).contiguous()
    ref = torch.cat(references).contiguous() if kl_beta else None
    if torch.is_grad_enabled() and cur.requires_grad:
        loss, report = _Grpo.apply(cur.contiguous(), beh, ref, adv, offsets, clip_eps, kl_beta)
    else:
        loss, _, report = _run_grpo(cur.detach().contiguous(), beh, ref, adv, offsets, clip_eps, kl_beta, False)
    values, st = _read_report(report, len(GRPO_METRIC_KEYS))
    for bits in st[st != 0].tolist():
        if bits:
            for bit, message in _GRPO_CHECKS:
                if bits & bit:
                    raise ValueError(message)
    m = dict(zip(GRPO_METRIC_KEYS, values))
    if not math.isfinite(m["loss"]):
        raise ValueError("GRPO loss contains non-finite values")
    return loss, m
