"""Transformers attention backend: dense, V1 and mean-corrected sparse prefill on MI355X.

Drop-in for the reference ``attention.py``: same ``METHODS``, the same
``AttentionBackend`` constructor, ``configure``, ``forward`` signature, stage
names, profiling and capture hooks, and the same registration as transformers'
``"sdpa"`` attention function (attention.py:57). Prefill of the sparse methods
runs entirely in gfx950 HIP kernels:

  descriptor  spx_block_pool           bf16 mean K, fp32 descriptors, K / V tiles
  selector    spx_v1_route             V1 score + normalise + threshold selection
              spx_selector_scores      (mean_balanced / cgf_mean / dispersion_mean)
  indices     spx_protected_selection  (new selectors; V1 selection is fused above)
  mean        spx_tile_mean_query +    rescue-token choice (rescue methods only)
              spx_rescue_choice
  exact       spx_exact_attention      block-sparse flash attention
              spx_sparse_attention_mean  same, with the mean tail and the
                                         logaddexp merge fused in (mean methods)
              spx_sparse_attention_rescue  same, with the rescue tail fused in

so the reference's separate "merge" stage (and, for the mean methods, its "mean"
stage) takes no time here and is reported as 0 ms. Dense prefill uses
``F.scaled_dot_product_attention`` exactly as the reference does
(attention.py:179-189); ``dense_impl="hip"`` routes dense prefill through the
HIP kernel with implicit all-causal block lists instead. A decode step (one query
row, bf16, head dim 128 or 256) runs in spx_decode_attention; every other
non-prefill call goes to SDPA as in the reference.
"""

from __future__ import annotations

import torch
from torch.autograd import forward_ad
import torch.nn.functional as F

from . import _lib, kernels
from .kernels import BlockDescriptors
from .upstream import flashprefill_native_forward as upstream

try:
    # torch has no public way to ask for the transforms and modes around a call
    from torch.overrides import _get_current_function_mode_stack as _function_modes
    from torch.utils._device import DeviceContext
    _dispatch_modes = torch._C._len_torch_dispatch_stack
    _transform_level = torch._C._functorch.maybe_current_level
    forward_ad._current_level
except (ImportError, AttributeError):
    _function_modes = None     # a torch without these: decode steps stay with SDPA
# the C calls behind public functions where there are any (0.4 us less each)
_current_device = getattr(torch._C, "_cuda_getDevice", torch.cuda.current_device)
_is_tracing = getattr(torch._C, "_is_tracing", torch.jit.is_tracing)

try:  # transformers is optional: the backend also runs standalone
    from transformers.modeling_utils import ALL_ATTENTION_FUNCTIONS
except Exception:  # pragma: no cover - depends on the environment
    ALL_ATTENTION_FUNCTIONS = None

METHODS = (
    "dense",
    "fp_v1",
    "mean_native",
    "mean_balanced",
    "cgf_mean",
    "dispersion_mean",
    "fp_v1_rescue",
    "fp_v1_rescue_v2",
)
V1_ROUTED_METHODS = {"fp_v1", "mean_native", "fp_v1_rescue", "fp_v1_rescue_v2"}
RESCUE_METHODS = {"fp_v1_rescue", "fp_v1_rescue_v2"}
MEAN_METHODS = {
    "mean_native",
    "mean_balanced",
    "cgf_mean",
    "dispersion_mean",
}
STAGE_NAMES = ("descriptor", "selector", "indices", "exact", "mean", "merge", "attention")


def _blocks(sequence: int, block_size: int) -> int:
    return (sequence + block_size - 1) // block_size


def _layer_shapes_match(query, key, value) -> bool:
    """Whether K and V have the shape that Q implies. One set of sizes describes all
    buffers of AttentionBackend._prefill; any other call takes the stage functions, which
    size each buffer by its own tensor and refuse what does not fit."""
    if query.dim() != 4 or key.shape != value.shape:
        return False
    batch, q_heads, sequence, head_dim = query.shape
    kv_heads = key.shape[1]
    return (0 not in query.shape and kv_heads > 0 and q_heads % kv_heads == 0
            and tuple(key.shape) == (batch, kv_heads, sequence, head_dim))


def _decode_shapes_fit(query, key, value) -> bool:
    """Whether spx_decode_attention runs tensors of these [batch, head, sequence, dim]
    shapes: one query row, nothing empty (an empty query included: the kernel has no grid
    for it), no more keys than it counts."""
    batch, q_heads, rows, head_dim = query
    k_batch, kv_heads, keys, k_dim = key
    return (rows == 1 and (head_dim == 128 or head_dim == 256) and key == value
            and k_batch == batch > 0 and k_dim == head_dim and kv_heads > 0 and q_heads > 0
            and 0 < keys <= 1 << 30 and q_heads % kv_heads == 0 and batch * q_heads <= 65535)


def _reads_in_place(tensors, device) -> bool:
    """Whether spx_decode_attention reads these tensors' storage as it is: plain bf16
    tensors of this device index, no lazy negation, 16-byte rows."""
    for x in tensors:
        if type(x) is not torch.Tensor or x.get_device() != device \
                or x.dtype is not torch.bfloat16 or x.dim() != 4 or x.is_neg():
            return False
        batch, heads, rows, dim = x.stride()
        if dim != 1 or (batch | heads | rows) & 7 or x.data_ptr() & 15:
            return False
    return True


def _decode_kernel_takes(query, key, value, scaling) -> bool:
    """Whether a non-prefill call is a decode step of spx_decode_attention: one query
    row per head of plain bf16 GPU tensors in a layout it reads in place, and nothing
    around the call that SDPA honours and a raw kernel cannot (autograd in either
    mode, autocast, tracing and function transforms, a backend pin without flash).
    SDPA runs one workgroup per head (28/4 heads: 1156 us behind 32K tokens, 150 behind
    4K); at 130 tokens both are bound by the host's launches, so the length does not
    decide."""
    if (_function_modes is None or torch.compiler.is_compiling() or _is_tracing()
            or _transform_level() is not None or _dispatch_modes() or forward_ad._current_level >= 0
            or torch.is_autocast_enabled("cuda") or not torch.backends.cuda.flash_sdp_enabled()):
        return False
    for mode in _function_modes():
        if type(mode) is not DeviceContext:      # a default device: factories only
            return False
    return (isinstance(scaling, (int, float)) and query.is_cuda
            and _reads_in_place((query, key, value), _current_device())
            and _decode_shapes_fit(query.shape, key.shape, value.shape)
            and not (torch.is_grad_enabled() and (query.requires_grad or key.requires_grad
                                                  or value.requires_grad)))


class AttentionBackend:
    """Reference: attention.py:37-369."""

    def __init__(
        self,
        alpha: float = 0.08,
        sink_blocks: int = 2,
        window_blocks: int = 4,
        last_full_blocks: int = 2,
        block_size: int = 128,
        selector_chunk_tiles: int = 8,
        register: bool = True,
        dense_impl: str = "sdpa",
    ):
        if dense_impl not in ("sdpa", "hip"):
            raise ValueError(f"dense_impl must be 'sdpa' or 'hip', got {dense_impl!r}")
        self.method = "dense"
        self.alpha = alpha
        self.sink_blocks = sink_blocks
        self.window_blocks = window_blocks
        self.last_full_blocks = last_full_blocks
        self.block_size = block_size
        self.selector_chunk_tiles = selector_chunk_tiles
        self.dense_impl = dense_impl
        self.record = False
        self.profile_records = []
        self.capture_callback = None
        # When a list, every attention-kernel launch appends its (start, end)
        # torch.cuda.Event pair, recorded on the launch stream (benchmarks).
        self.kernel_events = None
        if register and ALL_ATTENTION_FUNCTIONS is not None:
            ALL_ATTENTION_FUNCTIONS["sdpa"] = self.forward

    def configure(self, method: str, alpha: float | None = None):
        if method not in METHODS:
            raise ValueError(f"unknown method {method!r}; choose from {METHODS}")
        self.method = method
        if alpha is not None:
            self.alpha = alpha

    def _stage(self, record, name, function):
        if not self.record:
            return function()
        start = torch.cuda.Event(enable_timing=True)
        end = torch.cuda.Event(enable_timing=True)
        start.record()
        result = function()
        end.record()
        record["events"][name] = (start, end)
        return result

    # ------------------------------------------------------------ pooling

    def _pool(self, k, v, want_kbar: bool, want_descriptors: bool, want_tiles: bool):
        """One spx_block_pool launch -> (bf16 mean K, descriptors, (key tiles,
        value tiles))."""
        device = _lib.require_gpu(k, v)
        batch, sequence, kv_heads, head_dim = k.shape
        blocks = _blocks(sequence, self.block_size)
        kbar = torch.empty(batch, blocks, kv_heads, head_dim, dtype=torch.bfloat16,
                           device=device) if want_kbar else None
        desc = kernels.empty_descriptors(batch, blocks, kv_heads, head_dim, device) \
            if want_descriptors else None
        tiles = (torch.empty(batch, kv_heads, blocks, self.block_size, head_dim,
                             dtype=torch.bfloat16, device=device),
                 torch.empty(batch, kv_heads, blocks, head_dim, self.block_size,
                             dtype=torch.bfloat16, device=device)) if want_tiles else None
        _lib.call(
            "spx_block_pool", _lib.ptr(k), _lib.strides(k), _lib.ptr(v), _lib.strides(v),
            batch, sequence, kv_heads, head_dim, self.block_size, _lib.ptr(kbar),
            _lib.ptr(desc.mean_k if desc else None), _lib.ptr(desc.mean_v if desc else None),
            _lib.ptr(desc.var_k if desc else None), _lib.ptr(desc.sigma_v if desc else None),
            _lib.ptr(desc.counts if desc else None), _lib.ptr(tiles[0] if tiles else None),
            _lib.ptr(tiles[1] if tiles else None), _lib.stream(device))
        return kbar, desc, tiles

    # ---------------------------------------------------------- selection

    def _route_v1(self, q, k, v, scale, record, want_descriptors, want_tiles,
                  want_scores=False):
        kbar, descriptors, tiles = self._stage(
            record, "descriptor",
            lambda: self._pool(k, v, True, want_descriptors, want_tiles))
        batch, sequence, q_heads, head_dim = q.shape
        blocks = kbar.shape[1]
        device = q.device
        scores = torch.empty(batch, blocks, blocks, q_heads, dtype=torch.float32,
                             device=device) if want_scores else None
        indices = torch.empty(batch, blocks, blocks, q_heads, dtype=torch.int64, device=device)
        counts = torch.empty(batch, blocks, q_heads, dtype=torch.int32, device=device)
        selected = torch.empty(batch, blocks, blocks, q_heads, dtype=torch.bool, device=device)

        def route():
            _lib.call(
                "spx_v1_route", _lib.ptr(q), _lib.strides(q), _lib.ptr(kbar), _lib.strides(kbar),
                batch, sequence, q_heads, k.shape[2], head_dim, self.block_size, float(scale),
                float(self.alpha), int(self.sink_blocks), int(self.window_blocks),
                int(self.last_full_blocks), _lib.ptr(scores), _lib.ptr(indices),
                _lib.ptr(counts), _lib.ptr(selected), _lib.stream(device))

        self._stage(record, "selector", route)
        return kbar, descriptors, tiles, scores, indices, counts, selected

    def _v1_selection(self, q, k, scale, record, descriptors_needed, return_auxiliary=False):
        """Reference attention.py:77-108: descriptors (fp32 only when a value
        tensor is given) + bf16 mean K -> V1 scores -> selection -> mask."""
        q = _lib.kernel_view(q)
        k = _lib.kernel_view(k)
        v = descriptors_needed if isinstance(descriptors_needed, torch.Tensor) else None
        if v is not None:
            v = _lib.kernel_view(v)
        kbar, descriptors, _, scores, indices, counts, selected = self._route_v1(
            q, k, v if v is not None else k, scale, record, v is not None, False,
            want_scores=return_auxiliary)
        if return_auxiliary:
            return descriptors, kbar, scores, indices, counts, selected
        return descriptors, indices, counts, selected

    def _new_selection(self, q, k, v, scale, record, want_tiles=False):
        """Reference attention.py:110-152 (plus the attention tiles of the pooling pass)."""
        _, descriptors, tiles = self._stage(
            record, "descriptor", lambda: self._pool(k, v, False, True, want_tiles))
        batch, sequence, q_heads, _ = q.shape
        blocks = descriptors.mean_k.shape[1]
        if self.alpha == 0:
            scores = torch.zeros(batch, blocks, blocks, q_heads, dtype=torch.float32,
                                 device=q.device)
        else:
            scores = self._stage(
                record, "selector",
                lambda: kernels.selector_scores(q, descriptors, scale, self.method,
                                                self.block_size, self.selector_chunk_tiles))
        indices = torch.empty(batch, blocks, blocks, q_heads, dtype=torch.int64, device=q.device)
        counts = torch.empty(batch, blocks, q_heads, dtype=torch.int32, device=q.device)
        selected = self._stage(
            record, "indices",
            lambda: kernels.protected_selection(scores, self.alpha, self.sink_blocks,
                                                self.window_blocks, self.last_full_blocks,
                                                indices, counts))
        return descriptors, tiles, indices, counts, selected

    # --------------------------------------------------------- attention

    def _attention(self, q, k, tiles, indices, counts, scale, descriptors: BlockDescriptors | None,
                   rescue=None, want_lse=True):
        """One attention-kernel launch: exact blocks, plus the block-mean tail
        (``descriptors``) or the rescue tail (``rescue`` = (choice, remainder,
        descriptors-or-None, v)) in the same online softmax. Returns (output, lse);
        lse is None when not wanted (the layer discards it, and the kernel then
        skips its stores)."""
        device = q.device
        batch, sequence, q_heads, head_dim = q.shape
        output = torch.empty(batch, sequence, q_heads, head_dim, dtype=q.dtype, device=device)
        lse = (torch.empty(batch, sequence, q_heads, dtype=torch.float32, device=device)
               if want_lse else None)
        common_head = (_lib.ptr(q), _lib.strides(q), _lib.ptr(tiles[0]), _lib.ptr(tiles[1]),
                       _lib.ptr(indices), _lib.strides(indices), _lib.ptr(counts),
                       _lib.strides(counts))
        # zeroed counters of the kernel's persistent grid (work items taken in turn); None
        # for launches that run faster with a workgroup per item
        queue = _lib.work_queue(batch, sequence, q_heads, k.shape[2], head_dim, device)
        common_tail = (batch, sequence, q_heads, k.shape[2], head_dim, self.block_size,
                       float(scale), _lib.ptr(output), _lib.strides(output), _lib.ptr(lse),
                       _lib.strides(lse), _lib.ptr(queue), _lib.stream(device))
        if head_dim in upstream._ATTENTION_CONFIGS:   # what attention_tile_sizes() reports
            upstream._flash_forward.best_config = upstream._ATTENTION_CONFIGS[head_dim]
        events = None
        if self.kernel_events is not None:
            events = (torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True))
            events[0].record()
        if rescue is not None:
            choice, remainder, rdesc, values = rescue
            _lib.call("spx_sparse_attention_rescue", *common_head, _lib.ptr(choice),
                      _lib.ptr(values), _lib.strides(values),
                      _lib.ptr(rdesc.mean_k if rdesc else None),
                      _lib.ptr(rdesc.mean_v if rdesc else None), int(remainder), *common_tail)
        elif descriptors is None:
            _lib.call("spx_exact_attention", *common_head, *common_tail)
        else:
            _lib.call("spx_sparse_attention_mean", *common_head, _lib.ptr(descriptors.mean_k),
                      _lib.ptr(descriptors.mean_v), _lib.ptr(descriptors.counts), *common_tail)
        if events is not None:
            events[1].record()
            self.kernel_events.append(events)
        return output, lse

    def _dense_hip(self, q, k, v, scale):
        _, _, tiles = self._pool(k, v, False, False, True)
        return self._attention(q, k, tiles, None, None, scale, None, want_lse=False)

    def _prefill(self, q, k, v, scale):
        """One prefill layer of any method as bare launches, nothing between the stages
        but pointers: all intermediate buffers are parts of one allocation, and what the
        method does not read (the selection mask of the V1 route, unused moments) is not
        written. The stage functions above do the same launches through tensors, for
        profiles, captures and callers of the stages; their dozen allocations and views
        kept layers of up to 1100 tokens bound by the host (52 us of Python per layer,
        28/4 heads; here 30)."""
        method, block_size = self.method, self.block_size
        batch, sequence, q_heads, head_dim = q.shape
        kv_heads = k.shape[2]
        blocks = _blocks(sequence, block_size)
        device = q.device
        stream = _lib.stream(device)
        shape = (batch, sequence, q_heads, kv_heads, head_dim, block_size)
        selector = method in kernels.SELECTORS
        v1 = method in V1_ROUTED_METHODS
        rescue = method in RESCUE_METHODS
        size = 0

        def take(nbytes):
            nonlocal size
            offset, size = size, size + ((nbytes + 255) & ~255)
            return offset

        vectors = batch * blocks * kv_heads * head_dim
        entries = batch * blocks * blocks * q_heads
        tile_bytes = 2 * vectors * block_size
        key_tiles, value_tiles = take(tile_bytes), take(tile_bytes)
        kbar = take(2 * vectors) if v1 else None
        moments = method in MEAN_METHODS or method == "fp_v1_rescue_v2"
        mean_k = mean_v = counts = var_k = sigma_v = None
        if moments:
            mean_k, mean_v, counts = take(4 * vectors), take(4 * vectors), take(4 * blocks)
        if selector:
            var_k, sigma_v = take(4 * vectors), take(4 * batch * blocks * kv_heads)
            nbytes = _lib.load().spx_selector_workspace_bytes(batch, sequence, kv_heads, head_dim)
            split = take(max(nbytes, 0))
            scores, mask = take(4 * entries), take(entries)
        if rescue:
            qmean, choice = take(4 * batch * blocks * q_heads * head_dim), take(entries)
        indices = list_counts = None
        if method != "dense":
            indices, list_counts = take(8 * entries), take(4 * batch * blocks * q_heads)
        space = torch.empty(size, dtype=torch.uint8, device=device)
        base = space.data_ptr()

        def at(offset):
            return None if offset is None else base + offset

        four, three = _lib.STRIDES[4], _lib.STRIDES[3]
        qs, ks, vs = _lib.strides(q), _lib.strides(k), _lib.strides(v)
        qp, kp, vp = q.data_ptr(), k.data_ptr(), v.data_ptr()
        entry_strides = four(blocks * blocks * q_heads, blocks * q_heads, q_heads, 1)
        rules = (int(self.sink_blocks), int(self.window_blocks), int(self.last_full_blocks))
        _lib.call("spx_block_pool", kp, ks, vp, vs, batch, sequence, kv_heads, head_dim, block_size,
                  at(kbar), at(mean_k), at(mean_v), at(var_k), at(sigma_v), at(counts),
                  at(key_tiles), at(value_tiles), stream)
        if v1:
            _lib.call("spx_v1_route", qp, qs, at(kbar),
                      four(blocks * kv_heads * head_dim, kv_heads * head_dim, head_dim, 1), *shape,
                      scale, float(self.alpha), *rules, None, at(indices), at(list_counts), None,
                      stream)
        elif selector:
            if nbytes < 0:
                raise ValueError(
                    f"selector_scores: unsupported shape {tuple(q.shape)} (head_dim 128 or 256)")
            _lib.call("spx_selector_scores", qp, qs, at(mean_k), at(var_k), at(sigma_v), at(counts),
                      *shape, _lib.SELECTOR_IDS[method], scale, at(split), at(scores),
                      entry_strides, stream)
            _lib.call("spx_protected_selection", at(scores), entry_strides, batch, blocks, blocks,
                      q_heads, float(self.alpha), *rules, at(mask), at(indices), at(list_counts),
                      stream)
        if rescue:
            _lib.call("spx_tile_mean_query", qp, qs, batch, sequence, q_heads, head_dim, block_size,
                      at(qmean), stream)
            _lib.call("spx_rescue_choice", at(qmean), at(key_tiles), *shape, at(choice), stream)
        output = torch.empty(batch, sequence, q_heads, head_dim, dtype=q.dtype, device=device)
        queue = _lib.work_queue(batch, sequence, q_heads, kv_heads, head_dim, device)
        if head_dim in upstream._ATTENTION_CONFIGS:   # what attention_tile_sizes() reports
            upstream._flash_forward.best_config = upstream._ATTENTION_CONFIGS[head_dim]
        head = (qp, qs, at(key_tiles), at(value_tiles), at(indices),
                entry_strides if indices is not None else None, at(list_counts),
                three(blocks * q_heads, q_heads, 1) if indices is not None else None)
        tail = (*shape, scale, output.data_ptr(), _lib.strides(output), None, None, _lib.ptr(queue),
                stream)
        if rescue:
            _lib.call("spx_sparse_attention_rescue", *head, at(choice), vp, vs, at(mean_k),
                      at(mean_v), int(moments), *tail)
        elif moments:
            _lib.call("spx_sparse_attention_mean", *head, at(mean_k), at(mean_v), at(counts), *tail)
        else:
            _lib.call("spx_exact_attention", *head, *tail)
        return output

    @staticmethod
    def _decode(query, key, value, scale):
        """One query row per head against the whole cache -> [B, 1, Hq, D]."""
        batch, q_heads, _, head_dim = query.shape
        _, kv_heads, sequence, _ = key.shape
        nbytes = _lib.load().spx_decode_workspace_bytes(batch, sequence, q_heads, kv_heads, head_dim)
        workspace = query.new_empty(nbytes, dtype=torch.uint8) if nbytes else None
        output = query.new_empty(batch, 1, q_heads, head_dim)
        _lib.call("spx_decode_attention", _lib.ptr(query), _lib.strides(query), _lib.ptr(key),
                  _lib.strides(key), _lib.ptr(value), _lib.strides(value), batch, sequence,
                  q_heads, kv_heads, head_dim, scale, _lib.ptr(workspace), _lib.ptr(output),
                  _lib.stream(query.device))
        return output

    def forward(
        self,
        module,
        query,
        key,
        value,
        attention_mask,
        scaling,
        dropout=0.0,
        **kwargs,
    ):
        """Reference attention.py:154-339. query [B, Hq, S, D], key / value
        [B, Hkv, S, D] -> (output [B, S, Hq, D], None)."""
        record = {
            "layer": getattr(module, "layer_idx", None),
            "method": self.method,
            "events": {},
            "accounting": None,
        }
        overall_start = overall_end = None
        if self.record:
            overall_start = torch.cuda.Event(enable_timing=True)
            overall_end = torch.cuda.Event(enable_timing=True)
            overall_start.record()

        is_prefill = query.shape[2] == key.shape[2]
        if not is_prefill and _decode_kernel_takes(query, key, value, scaling):
            output = self._decode(query, key, value, float(scaling))
        elif (self.method == "dense" and self.dense_impl == "sdpa") or not is_prefill:
            output = F.scaled_dot_product_attention(
                query, key, value, attn_mask=None, dropout_p=0.0, is_causal=is_prefill,
                scale=scaling, enable_gqa=True,
            ).transpose(1, 2).contiguous()
            if self.record and is_prefill:
                record["accounting"] = self._dense_accounting(query)
        elif (not self.record and self.capture_callback is None and self.kernel_events is None
              and not (self.alpha == 0 and self.method in kernels.SELECTORS)
              and _layer_shapes_match(query, key, value)):
            _lib.require_gpu(query, key, value)
            output = self._prefill(_lib.kernel_view(query.transpose(1, 2)),
                                   _lib.kernel_view(key.transpose(1, 2)),
                                   _lib.kernel_view(value.transpose(1, 2)), float(scaling))
        elif self.method == "dense":
            q = _lib.kernel_view(query.transpose(1, 2))
            k = _lib.kernel_view(key.transpose(1, 2))
            v = _lib.kernel_view(value.transpose(1, 2))
            output, _ = self._stage(record, "exact", lambda: self._dense_hip(q, k, v, float(scaling)))
            if self.record:
                record["accounting"] = self._dense_accounting(query)
        else:
            _lib.require_gpu(query, key, value)
            q = _lib.kernel_view(query.transpose(1, 2))
            k = _lib.kernel_view(key.transpose(1, 2))
            v = _lib.kernel_view(value.transpose(1, 2))
            scale = float(scaling)
            capture_v1 = self.capture_callback is not None and self.method == "fp_v1"
            if self.method in V1_ROUTED_METHODS:
                kbar, descriptors, tiles, scores, indices, counts, selected = self._route_v1(
                    q, k, v, scale, record,
                    self.method in ("mean_native", "fp_v1_rescue_v2"), True,
                    want_scores=capture_v1)
            else:
                descriptors, tiles, indices, counts, selected = self._new_selection(
                    q, k, v, scale, record, want_tiles=True)
                kbar = scores = None

            if capture_v1:
                self.capture_callback(
                    layer=int(module.layer_idx), q=q, k=k, v=v, mean_k=kbar, scores=scores,
                    indices=indices, counts=counts, selected=selected, scale=scale)

            mean_desc = descriptors if self.method in MEAN_METHODS else None
            rescue = None
            if self.method in RESCUE_METHODS:
                # the rescue-token choice is timed as the "mean" stage (the non-exact
                # tail path of the profile schema, attention.py:306-307); the tail
                # itself runs inside the attention kernel
                choice = self._stage(
                    record, "mean",
                    lambda: kernels.rescue_choice(q, tiles[0], self.block_size))
                rescue = (choice, self.method == "fp_v1_rescue_v2", descriptors, v)
            output, _ = self._stage(
                record, "exact",
                lambda: self._attention(q, k, tiles, indices, counts, scale, mean_desc, rescue,
                                        want_lse=False))
            if self.record:
                q_tile, k_tile = upstream.attention_tile_sizes()
                score_tile = upstream.score_tile_size() if self.method in V1_ROUTED_METHODS else None
                record["accounting"] = kernels.selection_accounting(
                    selected, q.shape[1], q_tile, k_tile, self.method, score_tile, self.block_size)

        if self.record and is_prefill:
            overall_end.record()
            record["events"]["attention"] = (overall_start, overall_end)
            self.profile_records.append(record)
        return output, None

    @staticmethod
    def _dense_accounting(query):
        sequence = query.shape[2]
        pairs = query.shape[0] * query.shape[1] * sequence * (sequence + 1) // 2
        return {
            "effective_exact_token_pair_ratio": 1.0,
            "exact_token_pairs": pairs,
            "causal_token_pairs": pairs,
            "legacy_block_density": 1.0,
            "selected_block_entries": None,
            "causal_block_entries": None,
            "exact_physical_qk_tiles": None,
            "mean_proxy_entries": 0,
            "selector_proxy_entries": 0,
            "mean_executed_logit_entries": 0,
            "mean_executed_value_entries": 0,
            "selector_executed_dot_entries": 0,
            "selector_physical_qk_tiles": None,
            "q_tile_size": None,
            "k_tile_size": None,
            "score_k_tile_size": None,
        }

    # ---------------------------------------------------- profile / capture

    def start_profile(self):
        self.profile_records.clear()
        self.record = True

    def start_capture(self, callback):
        """Attach a synchronous V1-prefill diagnostic callback."""
        self.capture_callback = callback

    def finish_capture(self):
        self.capture_callback = None

    def finish_profile(self):
        self.record = False
        torch.cuda.synchronize()
        rows = []
        for record in self.profile_records:
            row = {"layer": record["layer"], "method": record["method"]}
            for name in STAGE_NAMES:
                event = record["events"].get(name)
                row[f"{name}_ms"] = event[0].elapsed_time(event[1]) if event else 0.0
            for key, value in (record["accounting"] or {}).items():
                row[key] = value.item() if isinstance(value, torch.Tensor) else value
            rows.append(row)
        self.profile_records.clear()
        return rows
