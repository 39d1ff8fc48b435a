"""Dense KV compression: score -> normalise -> protect window -> top-k -> gather.

The reference's ``TriAttentionCompressor`` (triattention/vllm/core/compressor.py:27-421)
with ``CompressionState`` (core/state.py:23-196) and the dense helpers of
core/utils.py:433-502.  Ordinary device tensors go through one library call from the scores
to the gathered rows (``ops.dense_compress``); what that call does not take (gradients wanted,
a scoring mode or dtype of its own, rows that are not 16-byte multiples) is put together from the
scoring and top-k kernels and torch's normalisation and gather.  NaN scores rank alike both ways (above
+inf, or lowest with the sign set); only the sign of the NaN that a normalised row with infinite scores and
no NaN, or with NaN of both signs, turns into differs: there torch's depends on the order of its reduction.
"""
from __future__ import annotations

from typing import Dict, Optional, Tuple

import torch

from .. import ops
from . import stats as stats_mod
from .config import TriAttentionConfig
from .scoring import compute_scores


def normalize_scores(scores: torch.Tensor, eps: float = 1e-8) -> torch.Tensor:
    """z-score along the last axis, unbiased std, std < eps -> 1 (core/utils.py:466-480)."""
    mean = scores.mean(dim=-1, keepdim=True)
    std = scores.std(dim=-1, keepdim=True)
    return (scores - mean) / torch.where(std < eps, torch.ones_like(std), std)


def protect_window_tokens(scores: torch.Tensor, window_size: int) -> torch.Tensor:
    """Last ``window_size`` tokens -> +inf (core/utils.py:483-502)."""
    if window_size <= 0:
        return scores
    out = scores.clone()
    out[..., -window_size:] = float("inf")
    return out


def gather_kv_by_indices(kv_tensor: torch.Tensor, indices: torch.Tensor, dim: int = 2) -> torch.Tensor:
    """[B, H, T, D] gathered along T by [B, k] or [B, H, k] indices (core/utils.py:433-463)."""
    if indices.ndim == 2:
        b, k = indices.shape
        idx = indices.view(b, 1, k, 1).expand(b, kv_tensor.shape[1], k, kv_tensor.shape[3])
    elif indices.ndim == 3:
        idx = indices.unsqueeze(-1).expand(*indices.shape, kv_tensor.shape[3])
    else:
        raise ValueError(f"Unsupported indices shape: {indices.shape}")
    return torch.gather(kv_tensor, dim=dim, index=idx)


class CompressionState:
    """Per-request counters that decide when to compress (core/state.py:23-196):
    trigger at budget + divide_length, compress down to budget."""

    def __init__(self, config: TriAttentionConfig):
        self.config = config
        self.reset()

    def reset(self) -> None:
        self.absolute_position = 0
        self.compression_count = 0
        self.prefill_length = 0
        self.tokens_in_round = 0
        self.current_cache_len = 0
        self.last_prune_step = 0

    def initialize(self, seq_len: int) -> None:
        self.current_cache_len = self.prefill_length = self.absolute_position = seq_len

    def append_tokens(self, n: int) -> None:
        self.current_cache_len += n
        self.absolute_position += n
        self.tokens_in_round += n

    def should_compress(self, current_len: int) -> bool:
        if self.absolute_position == 0:
            self.initialize(current_len)
            effective = current_len
        else:
            new_tokens = current_len - self.absolute_position
            if new_tokens > 0:
                self.append_tokens(new_tokens)
            effective = self.current_cache_len
        if self.config.protect_prefill:
            effective = max(0, effective - self.prefill_length)
        return effective >= self.config.kv_budget + self.config.divide_length

    def update_after_compression(self, new_cache_len: int) -> None:
        self.current_cache_len = new_cache_len
        self.last_prune_step = self.absolute_position
        self.tokens_in_round = 0
        self.compression_count += 1

    def get_effective_budget(self) -> int:
        if self.config.protect_prefill:
            return max(0, self.config.kv_budget - self.prefill_length)
        return self.config.kv_budget

    def get_round_start(self) -> int:
        return self.absolute_position

    def to_dict(self) -> dict:
        return {k: getattr(self, k) for k in ("absolute_position", "compression_count", "prefill_length",
                                              "tokens_in_round", "current_cache_len", "last_prune_step")}


class TriAttentionCompressor:
    def __init__(self, config: TriAttentionConfig):
        self.config = config
        self.state = CompressionState(config)
        self.metadata: Optional[Dict] = None
        self.head_stats: Optional[Dict] = None
        self.inv_freq = self.omega = self.freq_scale_sq = self.offsets = None
        self.trig_cache = None      # kept for attribute compatibility; the HIP scorer needs no table cache
        self._initialized = False

    def _lazy_init(self) -> None:
        """core/compressor.py:70-117."""
        if self._initialized:
            return
        cfg = self.config
        if cfg.stats_path is None:
            raise ValueError("stats_path must be specified in TriAttentionConfig.")
        self.metadata, self.head_stats = stats_mod.load_frequency_stats(
            cfg.stats_path, device=cfg.device, dtype=cfg.compute_dtype, num_kv_heads=cfg.num_kv_heads,
            model_path=cfg.model_path)
        if cfg.head_dim is None:
            cfg.head_dim = self.metadata["head_dim"]
        if cfg.num_kv_heads is None:
            cfg.num_kv_heads = self.metadata["num_kv_heads"]
        if cfg.num_layers is None:
            cfg.num_layers = self.metadata["num_layers"]
        if "rope_style" in self.metadata:
            cfg.rope_style = str(self.metadata["rope_style"])
        self.inv_freq = stats_mod.resolve_inv_freq(self.metadata, cfg.head_dim, cfg.model_path).to(cfg.device)
        self.omega = self.inv_freq
        f = cfg.head_dim // 2
        self.freq_scale_sq = torch.zeros(cfg.num_layers, cfg.num_kv_heads, f, device=cfg.device,
                                         dtype=cfg.compute_dtype)
        for layer in range(cfg.num_layers):
            entry = self.head_stats.get(layer)
            if entry is not None and "freq_scale_sq" in entry:
                self.freq_scale_sq[layer] = entry["freq_scale_sq"]
        self.offsets = stats_mod.geometric_offsets(cfg.offset_max_length).to(cfg.device)
        self._initialized = True

    def _compute_scores(self, key_states: torch.Tensor, layer_idx: int) -> torch.Tensor:
        if layer_idx not in self.head_stats:
            raise ValueError(f"No stats found for layer {layer_idx}")
        return compute_scores(key_states=key_states, cache_positions=None, head_stats=self.head_stats[layer_idx],
                              omega=self.omega, offsets=self.offsets, freq_scale_sq=self.freq_scale_sq[layer_idx],
                              config=self.config, round_start=self.state.get_round_start(),
                              trig_cache=self.trig_cache)

    def _select_topk(self, scores: torch.Tensor, k: int) -> torch.Tensor:
        """Indices of the k largest along the last axis, ascending (core/compressor.py:388-409
        leaves their order undefined)."""
        flat = scores.reshape(-1, scores.shape[-1]).to(torch.float32).contiguous()
        keep = ops.topk_rows(flat, k)[:, :k].to(torch.long)
        return keep.reshape(*scores.shape[:-1], k)

    def _one_call_args(self, keys: torch.Tensor, values: torch.Tensor, layer_idx: int):
        """The fp32 statistics (q_mean_complex, q_abs_mean, freq_scale_sq) for ``ops.dense_compress``, or None
        where the step has to take the general way: everything that call would not do in the same way --
        gradients, forward-mode tangents, transformed or traced tensors, which only torch's gather carries; scores
        per layer or of a narrower type; a layout or a budget outside the kernels' range -- and every
        argument that the general way refuses."""
        cfg = self.config
        h, t, d = keys.shape[1:]
        if type(self) is not TriAttentionCompressor or not self.__dict__.keys().isdisjoint(("_compute_scores", "_select_topk")):
            return None                       # (a step of its own in a subclass or on the instance)
        if (type(keys) is not torch.Tensor or type(values) is not torch.Tensor or values.ndim != 4
                or not keys.is_cuda or values.device != keys.device or keys.device.index != torch.cuda.current_device()
                or keys.dtype not in (torch.bfloat16, torch.float16) or values.shape[:3] != keys.shape[:3]
                or keys.shape[0] != 1 or d not in (64, 128, 256) or h > 256):
            return None
        if ((torch.is_grad_enabled() and (keys.requires_grad or values.requires_grad))
                or torch.autograd.forward_ad._current_level >= 0 or torch.jit.is_tracing()
                or torch._C._functorch.is_functorch_wrapped_tensor(keys)
                or torch._C._functorch.is_functorch_wrapped_tensor(values)
                or values.is_conj() or values.is_neg()):
            return None
        if (cfg.topk_dtype != torch.float32 or cfg.pruning_mode == "per_layer" or cfg.score_aggregation not in ("mean", "max")
                or cfg.rope_style not in ("half", "interleaved") or not 0 < cfg.kv_budget <= t or t < 2):
            return None
        ks, vs, row = keys.stride(), values.stride(), values.shape[3] * values.element_size()
        if (ks[3] != 1 or vs[3] != 1 or ks[1] % 8 or ks[2] % 8 or ks[1] < d or row == 0 or row % 16
                or (vs[1] * values.element_size()) % 16 or (vs[2] * values.element_size()) % 16
                or keys.data_ptr() % 16 or values.data_ptr() % 16):
            return None
        entry = self.head_stats.get(layer_idx)
        if entry is None or "q_abs_mean" not in entry:
            return None
        stats = (entry["q_mean_complex"], entry["q_abs_mean"], self.freq_scale_sq[layer_idx])
        f = d // 2
        if tuple(stats[0].shape) != (h, f, 2) or tuple(stats[1].shape) != (h, f) or tuple(stats[2].shape) != (h, f):
            return None
        if self.omega.numel() != f or self.offsets.numel() > 32 or not -2**31 <= self.state.get_round_start() < 2**31:
            return None
        dev = keys.device
        return tuple(x if x.dtype is torch.float32 and x.device == dev and x.is_contiguous()
                     else x.to(device=dev, dtype=torch.float32).contiguous() for x in (*stats, self.omega, self.offsets))

    def compress(self, key_states: torch.Tensor, value_states: torch.Tensor,
                 cache_positions: Optional[torch.Tensor] = None, layer_idx: int = 0
                 ) -> Tuple[torch.Tensor, torch.Tensor, torch.Tensor]:
        """core/compressor.py:279-346; batch size 1 only, as in the reference."""
        self._lazy_init()
        b, h, t, d = key_states.shape
        if b > 1:
            raise ValueError(f"TriAttention currently only supports batch_size=1 for compression. Got batch_size={b}.")
        if not self.state.should_compress(t):
            return key_states, value_states, torch.arange(t, device=key_states.device)
        one_call = self._one_call_args(key_states, value_states, layer_idx)
        if one_call is not None:
            cfg = self.config
            keys, values, keep = ops.dense_compress(
                key_states, value_states, *one_call, budget=cfg.kv_budget, round_start=int(self.state.get_round_start()),
                window_size=cfg.window_size, normalize=bool(cfg.sparse_normalize_scores),
                aggregation=cfg.score_aggregation, rope_style=cfg.rope_style, disable_mlr=bool(cfg.disable_mlr),
                disable_trig=bool(cfg.disable_trig))
            self.state.update_after_compression(keys.shape[2])
            return keys, values, keep
        scores = self._compute_scores(key_states, layer_idx)
        if self.config.sparse_normalize_scores:
            scores = normalize_scores(scores)
        if self.config.window_size > 0:
            scores = protect_window_tokens(scores, self.config.window_size)
        keep = self._select_topk(scores, self.config.kv_budget)
        keys = gather_kv_by_indices(key_states, keep, dim=2)
        values = gather_kv_by_indices(value_states, keep, dim=2)
        self.state.update_after_compression(keys.shape[2])
        return keys, values, keep

    def reset(self) -> None:
        self.state.reset()

    def get_state(self) -> Dict:
        return self.state.to_dict()
