"""Calls into the kernel library: tensors to raw pointers, the current stream, error codes
to exceptions.  Shapes were checked in `ops`; what is checked here is that tensors live
on the GPU, since a host pointer handed to a kernel faults the device."""
from __future__ import annotations

import ctypes
import functools
from ctypes import c_float, c_int, c_longlong, c_void_p
from types import SimpleNamespace

import numpy as np
import torch

from wllm_amd.kernels.attention_plan import PROMPT_ROWS, AttentionPlan, build_work_items, count_tile_items, prompt_kernel_pays
from wllm_amd.kernels import ops
from wllm_amd.kernels.ops import gate_args
from wllm_amd.kernels.library import door, load
from wllm_amd.kernels.staging import pack_int32


class KernelError(RuntimeError):
    """A kernel launch failed or a kernel refused its operands."""


# torch's own shortcut to the current stream's handle (what its compiled kernels call)
_raw_current_stream = getattr(torch._C, "_cuda_getCurrentRawStream", None)


_ptr = ops._address


_SIGNATURES = {
    "wllm_gemm_residual": [c_void_p, c_void_p, c_int, c_void_p, c_void_p, c_int, c_int, c_int, c_void_p],
    "wllm_qkv_rope": [c_void_p, c_void_p, c_int, c_void_p, c_void_p, c_void_p, c_void_p, c_void_p, c_void_p, c_longlong,
                      c_int, c_int, c_int, c_int, c_int, c_int, c_void_p],
    "wllm_rms_norm": [c_void_p, c_void_p, c_int, c_int, c_longlong, c_void_p, c_void_p, c_void_p, c_void_p, c_int, c_int,
                      c_int, c_float, c_float, c_void_p],
    "wllm_rope_cache_write": [c_void_p, c_int, c_void_p, c_int, c_longlong, c_void_p, c_void_p, c_void_p, c_void_p,
                              c_void_p, c_longlong, c_int, c_int, c_int, c_int, c_int, c_int, c_void_p],
    "wllm_gemm_skinny_gated": [c_void_p, c_void_p, c_int, c_void_p, c_int, c_int, c_int, c_int, c_float, c_float, c_float, c_int,
                               c_int, c_void_p],
    "wllm_gemm_skinny_gated_norm": [c_void_p, c_void_p, c_int, c_void_p, c_float, c_float, c_void_p, c_int, c_void_p, c_int,
                                    c_int, c_int, c_int, c_float, c_float, c_float, c_void_p],
    "wllm_tile_weight": [c_void_p, c_void_p, c_int, c_int, c_void_p],
    "wllm_paged_attention_generic": [c_void_p, c_void_p, c_int, c_void_p, c_void_p, c_void_p, c_void_p, c_void_p,
                                     c_void_p, c_void_p, c_void_p, c_int, c_int, c_int, c_int, c_int, c_int, c_int, c_int,
                                     c_float, c_int, c_int, c_float, c_void_p, c_void_p],
    "wllm_paged_attention_generic_chunk_keys": [],
    "wllm_paged_attention_mfma": [c_void_p, c_void_p, c_void_p, c_void_p, c_int, c_void_p, c_void_p, c_int, c_void_p, c_int, c_void_p, c_void_p,
                                  c_void_p, c_void_p, c_void_p, c_void_p, c_int, c_int, c_int, c_int, c_int, c_float,
                                  c_int, c_int, c_float, c_int, c_void_p, c_void_p],
    "wllm_paged_attention_mfma_f32": [c_void_p, c_void_p, c_void_p, c_void_p, c_void_p, c_int, c_void_p, c_int, c_void_p, c_void_p,
                                      c_void_p, c_void_p, c_void_p, c_int, c_int, c_int, c_int, c_int, c_float, c_int, c_int,
                                      c_float, c_void_p, c_void_p],
    "wllm_paged_attention_prefill_f32": [c_void_p, c_void_p, c_void_p, c_void_p, c_int, c_int, c_void_p, c_void_p, c_void_p,
                                         c_void_p, c_void_p, c_void_p, c_int, c_int, c_int, c_int, c_int, c_float, c_int,
                                         c_int, c_float, c_void_p, c_void_p],
    "wllm_paged_attention_prefill": [c_void_p, c_void_p, c_void_p, c_void_p, c_int, c_int, c_void_p, c_void_p, c_void_p,
                                     c_void_p, c_void_p, c_void_p, c_int, c_int, c_int, c_int, c_int, c_float, c_int,
                                     c_int, c_float, c_int, c_void_p, c_void_p],
    "wllm_paged_attention_prompt": [c_void_p, c_void_p, c_void_p, c_void_p, c_int, c_int, c_void_p, c_void_p, c_void_p,
                                    c_void_p, c_void_p, c_void_p, c_int, c_int, c_int, c_int, c_int, c_float, c_int,
                                    c_int, c_float, c_int, c_void_p, c_void_p],
    "wllm_gemm_tile": [c_void_p, c_void_p, c_void_p, c_void_p, c_int, c_int, c_int, c_int, c_int, c_float, c_float, c_float,
                       c_void_p],
    "wllm_gemm_wide": [c_void_p, c_void_p, c_void_p, c_void_p, c_int, c_int, c_int, c_int, c_int, c_int, c_float, c_float,
                       c_float, c_void_p],
    "wllm_gemm_stream": [c_void_p, c_void_p, c_int, c_void_p, c_void_p, c_int, c_int, c_int, c_int, c_int, c_int, c_float, c_float,
                         c_float, c_void_p],
    "wllm_gemm_block": [c_void_p, c_void_p, c_void_p, c_void_p, c_int, c_int, c_int, c_int, c_int, c_int, c_float, c_float, c_float, c_int,
                        c_int, c_void_p],
    "wllm_split_sum": [c_void_p, c_void_p, c_int, c_longlong, c_int, c_void_p],
    "wllm_gemm_generic": [c_void_p, c_void_p, c_void_p, c_int, c_void_p, c_int, c_void_p, c_int, c_int, c_int, c_void_p],
    "wllm_tile_weight_f32": [c_void_p, c_void_p, c_int, c_int, c_void_p],
    "wllm_gemm_f32_segments": [c_int, c_int, c_int],
    "wllm_argmax_rows": [c_void_p, c_void_p, c_void_p, c_int, c_int, c_void_p],
    "wllm_gemm_pieces": [c_void_p, c_void_p, c_int, c_void_p, c_void_p, c_int, c_int, c_int, c_int, c_int, c_int, c_void_p],
    "wllm_gemm_skinny": [c_void_p, c_void_p, c_int, c_void_p, c_int, c_void_p, c_int, c_int, c_int, c_int, c_int,
                         c_void_p],
    "wllm_sample_rows": [c_void_p, c_void_p, c_void_p, c_void_p, c_void_p, c_void_p, c_void_p, c_int, c_int, c_void_p],
    "wllm_sample_rows_split": [c_void_p, c_void_p, c_void_p, c_void_p, c_void_p, c_void_p, c_void_p, c_void_p, c_int,
                               c_int, c_int, c_void_p],
    "wllm_sample_split_row_words": [],
    "wllm_gemm_skinny_joined": [c_void_p, c_void_p, c_int, c_void_p, c_int, c_int, c_int, c_int, c_int, c_void_p],
}


class HipBackend:
    def __init__(self):
        if not torch.cuda.is_available():
            raise KernelError("no GPU is visible; the kernels run on gfx950 only and there is no other path")
        raw = load()
        self._door = door()
        if self._door is not None:
            global _ptr
            ops.use_native(self._door)
            _ptr = ops._address
            self._on_gpu = self._door.make_on_gpu(KernelError)
        self._device_index = torch.cuda.current_device()
        self._partial_o = None
        self._slots_of = {}                # device -> workgroups of the prompt kernel it runs at once
        self._gemm_partials = None
        self._argmax_scratch = None
        self._sample_scratch = None
        self._partial_ml = None
        self._generic_partial_o = None
        self._registered: dict = {}
        self.library_events = None      # a list: every library product is bracketed by a pair of timing events
        self.lib = SimpleNamespace(raw=raw)        # the entry points by name, and the library itself
        for name, argtypes in _SIGNATURES.items():
            setattr(self.lib, name, self._entry(getattr(raw, name), argtypes))

    @staticmethod
    def _on_gpu(*tensors) -> None:      # (a backend with the native module has its)
        for t in tensors:
            if t is not None and not t.is_cuda:
                raise KernelError("a kernel operand is not on the GPU")

    _CODES = {c_void_p: "p", c_int: "i", c_longlong: "l", c_float: "f"}

    def _entry(self, fn, argtypes):
        """What calls the function `fn`, a ctypes library's, with arguments of these types: an entry of the native module, or,
        without the module and for types or numbers of arguments that it has no room for, `fn` itself."""
        fn.argtypes, fn.restype = argtypes, c_int
        codes = [self._CODES.get(a) for a in argtypes]
        if self._door is None or None in codes or len(codes) > 48 or codes.count("f") > 8 or len(codes) - codes.count("f") > 40:
            return fn
        return self._door.Entry(ctypes.cast(fn, c_void_p).value, "".join(codes))

    def _stream(self) -> int:
        # the raw handle of torch's current stream on this process's GPU, asked for at every launch
        if _raw_current_stream is not None:
            return _raw_current_stream(self._device_index)
        return torch.cuda.current_stream().cuda_stream

    @staticmethod
    def _check(code: int, what: str) -> None:
        if code == -1:
            raise KernelError(f"{what}: the kernel does not take these sizes")
        if code != 0:
            raise KernelError(f"{what}: HIP error {code}")

    def run_registered(self, op, args, kwargs) -> None:
        """An operation that a part registered (`ops.register_op`): its entry point is looked up once in
        its library, given its signature, and launched on the current stream (a part's own through ctypes: its launch may hand it
        whatever ctypes takes)."""
        fn = self._registered.get(op.name)
        if fn is None or fn[0] is not op:
            lib = op.library() if op.library is not None else getattr(self.lib, "raw", self.lib)
            entry = getattr(lib, op.entry_point)
            if op.own:
                entry = self._entry(entry, op.argtypes)
            else:
                entry.argtypes = op.argtypes
                entry.restype = c_int
            fn = self._registered[op.name] = (op, entry)
        self._on_gpu(*[a for a in args if isinstance(a, torch.Tensor)])
        if kwargs:
            self._on_gpu(*[a for a in kwargs.values() if isinstance(a, torch.Tensor)])
        stream = self._stream() if op.own else c_void_p(self._stream())
        self._check(op.launch(fn[1], stream, *args, **kwargs), op.name)

    def rms_norm(self, x, weight, eps, offset, out, delta, rows, delta_bias=None):
        self._on_gpu(x, weight, out, delta, rows, delta_bias)
        splits, stride = 1, 0
        if delta is not None and delta.dim() == 3:
            splits, stride = delta.shape[0], delta.shape[1] * delta.shape[2]
        self._check(self.lib.wllm_rms_norm(
            _ptr(x), _ptr(delta), int(delta is not None and delta.dtype == torch.bfloat16), splits, stride,
            _ptr(delta_bias), _ptr(weight), _ptr(rows), _ptr(out), int(out.dtype == torch.bfloat16), out.shape[0], x.shape[1], eps,
            offset, self._stream()), "rms_norm")

    def rope_and_cache_write(self, qkv, bias, positions, inv_freq, slots, cache, num_heads, num_kv_heads, head_dim,
                             rotary_dim, page_size, parts=None):
        self._on_gpu(qkv, bias, positions, inv_freq, slots, cache, parts)
        splits, stride = (parts.shape[0], parts.shape[1] * parts.shape[2]) if parts is not None else (0, 0)
        self._check(self.lib.wllm_rope_cache_write(
            _ptr(qkv), int(qkv.dtype == torch.bfloat16), _ptr(parts), splits, stride, _ptr(bias), _ptr(positions),
            _ptr(inv_freq), _ptr(slots),
            _ptr(cache), cache.shape[0] if cache is not None else 0, qkv.shape[0], num_heads, num_kv_heads, head_dim,
            rotary_dim, page_size, self._stream()), "rope_and_cache_write")

    RESIDUAL_MAX_K = 4096

    def linear_residual_takes(self, rows: int, dtype, out_features: int, in_features: int) -> bool:
        """The product that adds into the residual stream: bfloat16, at most 16 rows, whole bands of
        16 columns.  Its workgroups are the bands; with a long K axis there are too few of them for the
        weight to stream from all compute units, and the split product with its norm kernel is faster."""
        return (dtype == torch.bfloat16 and 1 <= rows <= 16 and out_features % 16 == 0 and in_features % 32 == 0
                and in_features <= self.RESIDUAL_MAX_K)

    def linear_residual(self, x, weight, tiles, residual, sumsq):
        self._on_gpu(x, weight, tiles, residual, sumsq)
        w, tiled = (tiles, 1) if tiles is not None else (weight, 0)
        self._check(self.lib.wllm_gemm_residual(_ptr(x), _ptr(w), tiled, _ptr(residual), _ptr(sumsq), x.shape[0],
                                                weight.shape[0], x.shape[1], self._stream()), "linear_residual")

    @staticmethod
    def qkv_rope_takes(rows: int, dtype, in_features: int, head_dim: int, rotary_dim: int) -> bool:
        """The fused projection, rotation and cache write: bfloat16, at most 32 tokens, heads of a
        multiple of 32 that are rotated whole."""
        return (dtype == torch.bfloat16 and 1 <= rows <= 32 and in_features % 32 == 0 and head_dim % 32 == 0
                and rotary_dim == head_dim)

    def qkv_rope(self, x, weight, tiles, qkv, bias, positions, inv_freq, slots, cache, num_heads, num_kv_heads,
                 head_dim, page_size):
        self._on_gpu(x, weight, tiles, qkv, bias, positions, inv_freq, slots, cache)
        w, tiled = (tiles, 1) if tiles is not None else (weight, 0)
        self._check(self.lib.wllm_qkv_rope(
            _ptr(x), _ptr(w), tiled, _ptr(bias), _ptr(positions), _ptr(inv_freq), _ptr(slots), _ptr(qkv), _ptr(cache),
            cache.shape[0] if cache is not None else 0, x.shape[0], x.shape[1], num_heads, num_kv_heads, head_dim,
            page_size, self._stream()), "qkv_rope")

    @staticmethod
    def mfma_attention_takes(dtype, head_dim: int, page_size: int) -> bool:
        """The matrix-core kernels: bfloat16 or float32 (each with the instruction of its own type), head sizes
        32..256 in steps of 32, pages of a multiple of 4."""
        return (dtype in (torch.bfloat16, torch.float32) and head_dim % 32 == 0 and 32 <= head_dim <= 256
                and page_size % 4 == 0)

    @staticmethod
    def portions_beside(head_dim: int, page_size: int) -> bool:
        """Whether a step's prompt portions run in one launch with its decoded tokens: the sizes of the portions' kernel that loads
        into shared memory (`attention_portion.h`).  The blocks of 128 rows of long prompts fill the device by themselves."""
        return head_dim in (64, 128, 256) and page_size >= 8 and page_size & (page_size - 1) == 0

    # Decoded tokens' items (of 16 rows by 128 keys) from which on a step's portions run by themselves, unless they are as much work.  Together
    # a compute unit runs two of the decoded tokens' workgroups instead of three: as long as they are some rounds that is less than the portions' own
    # launch, of many rounds it is up to a tenth.  us, apart and together, a portion of 448 tokens over 896 keys: 8 heads of 256 on one beside 128 of
    # 1,500 keys (1,189 items) 62.7 / 49.4, 16 on as many beside 8 of 2,048 and 256 of 300 (1,584 and 9,392) 70 / 64 and 211 / 224, 32 of 128 on eight
    # beside 60 of 1,500 and 128 of 4,000 (4,464 and 24,512) 81 / 80 and 332 / 347, 40 of 64 on as many beside 8 of 2,048 and 60 of 4,000 (3,960 and
    # 57,440) 50 / 43 and 337 / 366; one of 448 over 3,000 beside 128 of 1,500 (64 of 64 on eight, 9,512) 133 / 111.
    MANY_DECODED_ITEMS = 8192

    @classmethod
    def portions_pay_beside(cls, prefill, prefill_rows: int, num_items: int) -> bool:
        """Whether a step's portions gain by running in its decoded tokens' launch (see above): `prefill` are their items, whose tiles of 16
        rows by their keys are compared with the decoded tokens' of 128 keys."""
        if num_items < cls.MANY_DECODED_ITEMS:
            return True
        return int((prefill[:, 4] - prefill[:, 3]).sum()) * (prefill_rows // 16) >= 128 * num_items

    # Up to how many (items of 16 rows by 128 keys) x (elements of a head) float32 prompt portions are tiles: these take a time in
    # proportion, the blocks of 64 rows hardly less for few of them than for the 256 that give every compute unit one.
    # Tiles against blocks, heads of 256: 309 items 27 and 67 us, 1,280 61 and 75, 1,631 73 and 77, 2,080 89 and 79, 2,304 92 and
    # 91 (16 heads on as many) or 88 (8 on one), 2,560 104 and 112 or 105 and 104, 3,616 137 and 118; heads of 128: 2,304 items 50 and
    # 63, 2,616 56 and 69, 3,616 70 and 78, 4,032 80 and 81, 4,776 88 and 81.
    F32_TILE_WORK = 1 << 19

    def plan_paged_attention(self, host_q_len, host_ctx_len, num_heads, num_kv_heads, head_dim, page_size, window,
                             dtype, device):
        # `window`: w > 0 a sliding window, 0 none, -c < 0 chunks of c positions (the kernels' own convention)
        if not self.mfma_attention_takes(dtype, head_dim, page_size):
            return None
        group, slots_of_device = num_heads // num_kv_heads, self._workgroup_slots(device)
        if (dtype == torch.bfloat16 and head_dim == 256 and page_size >= 16 and page_size & (page_size - 1) == 0
                and prompt_kernel_pays(host_q_len, host_ctx_len, group, num_kv_heads, window)):
            items, reduces, slots, prefill, prefill_rows = build_work_items(
                host_q_len, host_ctx_len, group, num_kv_heads, window, page_size, PROMPT_ROWS, slots_of_device // 2, slots_a_unit=1)
        else:
            items, reduces, slots, prefill, prefill_rows = build_work_items(
                host_q_len, host_ctx_len, group, num_kv_heads, window, page_size, workgroup_slots=slots_of_device)
        if dtype == torch.float32 and prefill.shape[0] and \
                count_tile_items(host_q_len, host_ctx_len, group, num_kv_heads, window) * head_dim < self.F32_TILE_WORK:
            # float32 and little work: tiles of 16 rows fill the device better than the blocks of 64 rows would
            items, reduces, slots, prefill, prefill_rows = build_work_items(
                host_q_len, host_ctx_len, group, num_kv_heads, window, page_size, workgroup_slots=slots_of_device,
                tiles_only=True)
        flat = np.concatenate([items.reshape(-1), reduces.reshape(-1), prefill.reshape(-1)])
        dev = pack_int32([flat], device)[0]
        n_i, n_r, n_p = items.shape[0], reduces.shape[0], prefill.shape[0]
        self._ensure_partials(slots, head_dim, device)
        a, b = n_i * 8, (n_i + n_r) * 8
        return AttentionPlan(dev[:a].view(n_i, 8), dev[a:b].view(n_r, 8) if n_r else None, n_i, n_r, slots,
                             self._partial_o, self._partial_ml, dev[b:].view(n_p, 8) if n_p else None, n_p,
                             prefill_rows, together=bool(n_p and n_i) and self.portions_pay_beside(prefill, prefill_rows, n_i))

    def _workgroup_slots(self, device) -> int:
        """Workgroups of the kernel for prompt portions that the device runs at once: two a compute unit."""
        key = torch.device(device)
        if key not in self._slots_of:
            self._slots_of[key] = 2 * torch.cuda.get_device_properties(key).multi_processor_count
        return self._slots_of[key]

    def static_attention_plan(self, segments, num_heads, num_kv_heads, head_dim, page_size, window, dtype, device,
                              max_context: int, max_total_keys: int):
        """A plan of fixed shape for a captured decode graph of `segments` requests of one token."""
        if not self.mfma_attention_takes(dtype, head_dim, page_size):
            return None
        from wllm_amd.kernels.attention_plan import KEY_CHUNK, StaticAttentionPlan, row_tiles
        group = num_heads // num_kv_heads
        fixed = -(-max_context // KEY_CHUNK)
        max_slots = (max_total_keys // KEY_CHUNK + 2 * segments) * num_kv_heads * row_tiles(1, group)
        return StaticAttentionPlan(segments, group, num_kv_heads, window, fixed, max_slots, head_dim, device)

    def _ensure_partials(self, slots: int, head_dim: int, device) -> None:
        need = max(1, slots) * 16 * head_dim
        if self._partial_o is None or self._partial_o.numel() < need or self._partial_o.device != torch.device(device):
            self._partial_o = torch.empty(need, dtype=torch.float32, device=device)
        need = max(1, slots) * 16 * 2
        if self._partial_ml is None or self._partial_ml.numel() < need or self._partial_ml.device != torch.device(device):
            self._partial_ml = torch.empty(need, dtype=torch.float32, device=device)

    GENERIC_PARTIAL_FLOATS = 1 << 25       # 128 MiB of partial results for the general attention kernel

    def paged_attention(self, qkv, cache, block_tables, token_segment, seg_q_start, seg_q_len, seg_ctx_len, out,
                        num_heads, num_kv_heads, head_dim, page_size, scale, window, max_q_len, max_ctx_len,
                        plan=None, softcap=0.0, exact_weights=False, chunk=0, sinks=None):
        self._on_gpu(qkv, cache, block_tables, token_segment, seg_q_start, seg_q_len, seg_ctx_len, out, sinks)
        if chunk:
            # the kernels take one integer for the mask: w > 0 a sliding window, -c < 0 chunks of c positions
            window = -int(chunk)
        q_stride = qkv.shape[1]         # a row begins with the query heads; this many elements lie between two rows
        if plan is not None:
            if not self.mfma_attention_takes(qkv.dtype, head_dim, page_size):
                raise KernelError("paged_attention: a plan was given for sizes the matrix-core kernel does not take")
            if qkv.dtype == torch.float32:
                if plan.num_prefill:
                    self._check(self.lib.wllm_paged_attention_prefill_f32(
                        _ptr(qkv), _ptr(cache), _ptr(block_tables), _ptr(plan.prefill_items), plan.num_prefill,
                        plan.prefill_rows, _ptr(seg_q_start), _ptr(seg_q_len), _ptr(seg_ctx_len), _ptr(out),
                        _ptr(plan.partial_o), _ptr(plan.partial_ml), num_heads, num_kv_heads, head_dim, page_size,
                        block_tables.shape[1], scale, window, q_stride, softcap, _ptr(sinks), self._stream()),
                        "paged_attention (prompt portions, matrix cores, float32)")
                if plan.num_items == 0 and plan.num_reduce == 0:
                    return
                self._check(self.lib.wllm_paged_attention_mfma_f32(
                    _ptr(qkv), _ptr(cache), _ptr(block_tables), _ptr(plan.items), _ptr(plan.live_items), plan.num_items,
                    _ptr(plan.reduce_items), plan.num_reduce, _ptr(seg_q_start), _ptr(seg_q_len), _ptr(out),
                    _ptr(plan.partial_o), _ptr(plan.partial_ml), num_heads, num_kv_heads, head_dim, page_size,
                    block_tables.shape[1], scale, window, q_stride, softcap, _ptr(sinks), self._stream()),
                    "paged_attention (matrix cores, float32)")
                return
            together = plan.together and plan.prefill_rows != PROMPT_ROWS and self.portions_beside(head_dim, page_size)
            if plan.num_prefill and not together:
                prefill = self.lib.wllm_paged_attention_prompt if plan.prefill_rows == PROMPT_ROWS else self.lib.wllm_paged_attention_prefill
                self._check(prefill(
                    _ptr(qkv), _ptr(cache), _ptr(block_tables), _ptr(plan.prefill_items), plan.num_prefill,
                    plan.prefill_rows,
                    _ptr(seg_q_start), _ptr(seg_q_len), _ptr(seg_ctx_len), _ptr(out), _ptr(plan.partial_o),
                    _ptr(plan.partial_ml), num_heads, num_kv_heads,
                    head_dim, page_size, block_tables.shape[1], scale, window, q_stride, softcap, int(exact_weights),
                    _ptr(sinks), self._stream()), "paged_attention (prompt portions, matrix cores)")
            if plan.num_items == 0 and plan.num_reduce == 0:
                return
            self._check(self.lib.wllm_paged_attention_mfma(
                _ptr(qkv), _ptr(cache), _ptr(block_tables), _ptr(plan.prefill_items) if together else None,
                plan.num_prefill if together else 0, _ptr(plan.items), _ptr(plan.live_items), plan.num_items, _ptr(plan.reduce_items),
                plan.num_reduce, _ptr(seg_q_start), _ptr(seg_q_len), _ptr(seg_ctx_len), _ptr(out),
                _ptr(plan.partial_o), _ptr(plan.partial_ml), num_heads, num_kv_heads, head_dim, page_size,
                block_tables.shape[1], scale, window, q_stride, softcap, int(exact_weights), _ptr(sinks), self._stream()),
                "paged_attention (matrix cores)")
            return
        if head_dim % 4 or head_dim > 256:
            raise KernelError(f"paged_attention: head_dim {head_dim} is not a multiple of 4 up to 256")
        # The general kernel cuts a token's keys into chunks and leaves the chunks of a token that has
        # several in a buffer for a second kernel.  The buffer is made once at a fixed size (captured
        # graphs hold its address); the tokens of a step run in as many launches as it takes.
        longest = block_tables.shape[1] * page_size
        max_ctx_len = min(max_ctx_len, longest) if max_ctx_len > 0 else longest
        chunks = -(-max_ctx_len // self.lib.wllm_paged_attention_generic_chunk_keys())
        per_token = num_heads * chunks * (head_dim + 2)
        if per_token > self.GENERIC_PARTIAL_FLOATS:
            raise KernelError(f"paged_attention: one token of {num_heads} heads over {max_ctx_len} keys needs "
                              f"{per_token} floats of partial results, {self.GENERIC_PARTIAL_FLOATS} are reserved")
        if self._generic_partial_o is None or self._generic_partial_o.device != qkv.device:
            self._generic_partial_o = torch.empty(self.GENERIC_PARTIAL_FLOATS, dtype=torch.float32, device=qkv.device)
        partial_tokens = self.GENERIC_PARTIAL_FLOATS // per_token
        partial_ml = self._generic_partial_o[partial_tokens * num_heads * chunks * head_dim:]
        self._check(self.lib.wllm_paged_attention_generic(
            _ptr(qkv), _ptr(cache), int(qkv.dtype == torch.bfloat16), _ptr(block_tables), _ptr(token_segment),
            _ptr(seg_q_start), _ptr(seg_q_len), _ptr(seg_ctx_len), _ptr(out), _ptr(self._generic_partial_o),
            _ptr(partial_ml), partial_tokens, max_ctx_len, qkv.shape[0], num_heads, num_kv_heads,
            head_dim, page_size, block_tables.shape[1], scale, window, q_stride, softcap, _ptr(sinks), self._stream()),
            "paged_attention")

    @staticmethod
    @functools.lru_cache(maxsize=4096)
    def skinny_split(n: int, k: int) -> int:
        """Over how many workgroups the K axis of a few-row product is split: enough that about
        2,000 wavefronts stream weights at once, a function of the weight's shape only."""
        tiles = -(-n // 16)
        splits = 1
        while tiles * splits < 1536 and k % (splits * 2) == 0 and (k // (splits * 2)) % 32 == 0 \
                and k // (splits * 2) >= 256:
            splits *= 2
        return splits

    # The kernel whose wavefronts meet (`gemm_pieces.hip`, which has the figures).  Where a split product goes to a consumer as a
    # stack of partial sums: (pieces of the K axis, bands of 16 columns a workgroup), or (0, 0).  A workgroup a compute unit at
    # most: its time goes by its bytes of w, at about 26 KB a us, and by x, which several workgroups read (half its bytes, at 24 rows);
    # every piece costs the consumer 0.6 us a launch (a norm of 8 to 64 rows after a product 2.4 us with 2 pieces, 3.2 with 4, 4.3 with
    # 8, 6.6 with 16).  A piece is a quarter as long a chain of sums as it has keys, in whole steps of 64: no longer than a piece of
    # `skinny_split`, or by 32 keys at most where four wavefronts share the steps unevenly.  So no exactness is lost: of 39 sizes, those of the longer chains among
    # them, every sum of pieces was nearer to 64 bits than that of `skinny_split`'s (root mean square, 2,304 keys to 2,048 columns 1.05e-7 and 1.07e-7, 5,632 1.17e-7
    # and 1.27e-7, 16,384 1.93e-7 and 1.99e-7; 4,096 in 2 pieces, which the bound rules out, 1.34e-7 and 1.15e-7).  A function of the weight's shape only, so that a row's sum does not depend on the rows beside it.
    @staticmethod
    @functools.lru_cache(maxsize=4096)
    def piece_split(n: int, k: int) -> tuple:
        best, least = (0, 0), None
        if HipBackend.skinny_split(n, k) == 1 or (n + 15) * k >= 1 << 31 or k >= 1 << 24:
            return best
        for bands in (1, 2, 3):
            groups, pieces = -(-n // (16 * bands)), 2
            while groups * pieces <= HipBackend.COMPUTE_UNITS and k % (64 * pieces) == 0 and k // pieces >= 256 and pieces <= 16:
                cost = (16 * bands + 12) * 2 * (k // pieces) / 26000 + 0.6 * pieces
                if 4 * pieces >= HipBackend.skinny_split(n, k) and (least is None or cost < least):
                    best, least = (pieces, bands), cost
                pieces *= 2
        # Two workgroups a compute unit, where that halves the pieces of `skinny_split` (us with the norm, 8 / 24 / 64 rows, that kernel, `gemm_stream.hip` and this
        # one: 1,152 keys to 6,145 columns 14.2 / 15.9 / 20.7, 13.8 / 15.9 / 20.7 and 13.0 / 14.0 / 19.6; 1,024 to 8,192 11.3 / 12.9 / 16.5, 10.8 / 12.2 / 15.3 and
        # 9.1 / 9.9 / 14.5; 2,048 to 8,192 14.4 / 15.2 / 19.4, 13.3 / 14.1 / 17.5 and 12.0 / 12.8 / 17.6; to 9,216 21.8 / 23.5 / 28.7, 21.4 / 23.3 / 27.6 and 19.4 / 21.5 / 27.4;
        # to 10,304 23.3 / 24.5 / 30.1, 22.6 / 24.4 / 29.5 and 21.0 / 23.2 / 28.9).  As many pieces gain nothing (512 to 6,400 7.9 / 8.7 / 10.8, 7.8 / 8.5 / 10.4 and 7.3 / 8.1 / 11.8;
        # 1,024 to 12,288 22.0 / 23.9 / 26.4, 20.8 / 21.9 / 24.7 and 19.9 / 21.8 / 27.6).
        if least is None and n <= 48 * HipBackend.COMPUTE_UNITS and 512 <= k <= 2048 and k % 128 == 0 and HipBackend.skinny_split(n, k) > 2:
            best = (2, 3)
        return best

    @staticmethod
    def crowded_bands(n: int, rows: int) -> int:
        """Bands a workgroup where there are two workgroups a compute unit and more: three, or, where three would leave a part of a second round
        or no room for two workgroups (their rings, from 33 rows on), two (us with the norm, three and two: 2,048 keys to 8,192 columns at 8 / 24 / 40 / 64 rows
        12.9 / 14.5 / 17.4 / 19.8 and 12.0 / 12.8 / 14.6 / 17.6; to 10,304 21.0 / 23.2 / 26.0 / 28.9 and 21.3 / 23.4 / 25.0 / 30.6).  A row's bits are the same."""
        return 2 if n <= 8192 or 32 < rows <= 48 else 3

    # splits * N stays below 3072 * 16 by the rule of `skinny_split`; 64 rows of float32 of that
    GEMM_PARTIAL_FLOATS = 3072 * 16 * 64

    def _gemm_partial(self, count: int, device) -> torch.Tensor:
        """The buffer of split sums.  It is allocated once at its largest size and never again,
        because captured graphs hold its address."""
        if count > self.GEMM_PARTIAL_FLOATS:
            raise KernelError(f"split-sum buffer: {count} floats needed, {self.GEMM_PARTIAL_FLOATS} reserved")
        if self._gemm_partials is None or self._gemm_partials.device != device:
            self._gemm_partials = torch.empty(self.GEMM_PARTIAL_FLOATS, dtype=torch.float32, device=device)
        return self._gemm_partials

    SKINNY_CHUNK = {1: 1024, 2: 512, 3: 256, 4: 256}     # K elements of x staged at a time, by row tiles
    GATED_CHUNK = {1: 256, 2: 256, 3: 256, 4: 256}       # the same per half of K in the gated product

    @staticmethod
    def skinny_takes(dtype, rows: int, in_features: int) -> bool:
        return dtype == torch.bfloat16 and rows <= 64 and in_features % 32 == 0

    # The tiled matrix-core product (`gemm_tile.hip`) for the rows of a mixed step or a large decode
    # batch, where the tiles of 256 further down do not take the product.  Measured against the library's product it is ahead where the output has few columns and
    # the K axis is long, so that the library's tiles leave compute units idle and a split of the K axis
    # fills them (the down projection: 1.3 to 1.6 times as fast at 128 to 1,024 rows), and for the gated
    # product, which it writes once, up to 256 rows (at 512 rows it takes 84 us in a mixed step where
    # the library's product and the activation kernel take 69).  With these two the decode step of 256
    # requests is 5% and the stress workload 2% faster.  The projections of the attention block are not cut:
    # the rotation and the norm that then add the pieces lose more than the product gains (`block_tile` has them).
    TILE_MAX_ROWS = 1024
    F32_FEW_ROWS = 64         # rows up to which the float32 product streams its weights a band a wavefront
    TILE_LONG_K = 8192
    TILE_GATED_MAX_ROWS = 256

    @staticmethod
    @functools.lru_cache(maxsize=4096)
    def tile_splits(n: int, k: int, rows: int = 128) -> int:
        """Over how many workgroups the tiled product splits the K axis: a function of the weight's
        shape up to 640 rows (a row's sums still change with the step's rows where `wide_splits` takes the product).
        More rows fill the machine with fewer pieces, and every piece is a stack of partial sums to
        write and to read: halved while the launch has more than 640 workgroups (the down projection
        of 2,048 x 16,384 with the norm after it, 4 pieces against 8: 78 against 92 us at 1,024 rows,
        70 against 80 at 896, 68 against 70 at 768, but 67 against 64 at 640; that of 3,072 x 24,576:
        184 us with 2 pieces against 215 with 8 at 1,024 rows, 155 with 4 against 164 at 768)."""
        tiles = -(-n // 128)
        splits = 1
        while tiles * splits * 2 < 256 and k % (128 * splits) == 0 and k // (2 * splits) >= 512:
            splits *= 2
        row_tiles = -(-rows // 128)
        while splits > 2 and row_tiles > 5 and tiles * row_tiles * splits > 640:
            splits //= 2
        return splits

    def tile_takes(self, dtype, rows: int, out_features: int, in_features: int) -> bool:
        return (dtype == torch.bfloat16 and 64 < rows <= self.TILE_MAX_ROWS and in_features >= self.TILE_LONG_K
                and in_features % 64 == 0 and self.tile_splits(out_features, in_features, rows) > 1
                and max(rows, out_features) * in_features * 2 < 2 ** 32)

    # The product in tiles of 256 x 256 (`gemm_wide.hip`), a workgroup a compute unit, against the library's product and
    # the tiles of 128 x 128, with the pass that follows each (the activation kernel; the norm that adds the pieces).
    # It is ahead wherever its tiles fill the rounds of 256 compute units: the gated product of 2,048 keys to 2 x 16,384
    # columns at 384 / 768 / 1,500 / 2,048 / 7,777 rows 56 / 101 / 157 / 211 / 753 us against 58 / 106 / 183 / 234 / 880, to 2 x 4,096
    # columns at 1,500 / 2,048 / 3,001 rows 43 / 49 / 88 against 50 / 61 / 93; where a round is less than 0.7 full the others are
    # (to 2 x 16,384 at 257 / 640 rows 55 / 98 against 51 / 95, to 2 x 4,096 at 512 / 1,024 rows 36 / 39 against 26 / 38).  At most 256
    # rows are bound by the weights: there the tile's whole height pays where tiles of 128, two a compute unit, no longer run all at
    # once, from one more than half a tile a compute unit on (weights from HBM, to 2 x 20,480 columns at 129 / 192 / 256 rows 50 / 54 / 57 us against 72 /
    # 75 / 83, 3,072 keys to 2 x 24,576 78 / 81 / 87 against 104 / 115 / 131; but to 2 x 16,384 48 / 50 / 53 against 46 / 46 / 50).  Both have the same bits there.
    WIDE_TILE = 256
    COMPUTE_UNITS = 256
    WIDE_FULL = 0.7

    @classmethod
    def wide_gated_takes(cls, rows: int, columns: int, k: int) -> bool:
        """Whether the gated product of `columns` output columns goes in tiles of 256 rows (of x, and of both streams' weights)."""
        if rows <= 128 or columns < 1 or k < 64 or k % 64 != 0 or max(rows, 2 * columns) * k * 2 >= 2 ** 32:
            return False
        tiles = -(-rows // cls.WIDE_TILE) * -(-columns // (cls.WIDE_TILE // 2))
        if rows <= cls.WIDE_TILE:
            return tiles > cls.COMPUTE_UNITS // 2
        rounds = -(-tiles // cls.COMPUTE_UNITS)
        return rows * columns * 2 >= cls.WIDE_FULL * rounds * cls.COMPUTE_UNITS * cls.WIDE_TILE ** 2

    @classmethod
    def wide_takes(cls, rows: int, n: int, k: int) -> bool:
        """Whether a product rounded to bfloat16 goes in tiles of 256 x 256 instead of to the library.  The library is ahead where
        the columns fill its tiles (2,048 keys to 8,192 columns at 1,500 / 2,048 rows: 44 / 52 us against 46 / 53); where they are no
        multiple of 128 it falls back (to 10,304 columns at 1,024 / 1,500 / 4,096 rows 51 / 62 / 180 against 45 / 52 / 144; to 5,160
        at 3,001 rows 64 against 52), unless the rounds of tiles are less than 0.6 full (to 10,304 at 768 rows 38 against 44)."""
        if rows <= 128 or n % 128 == 0 or k < 64 or k % 64 != 0 or max(rows, n) * k * 2 >= 2 ** 32:
            return False
        rounds = -(-(-(-rows // cls.WIDE_TILE) * -(-n // cls.WIDE_TILE)) // cls.COMPUTE_UNITS)
        return rows * n >= 0.6 * rounds * cls.COMPUTE_UNITS * cls.WIDE_TILE ** 2

    # Tiles of the products of one round (`gemm_block.hip`, which has the figures; of 65 rows on, to 2,048 columns up to 3,072): rows of x, rows of w, and the time of a
    # launch that fills at most one round of workgroups, us and us a stage of 64 keys.  (256 rows: only the gated product has them.)
    BLOCK_TILES = ((64, 64, 2.9, 0.27), (128, 64, 3.2, 0.37), (192, 64, 3.6, 0.42), (128, 128, 4.0, 0.51), (192, 128, 4.6, 0.58), (256, 128, 4.6, 0.75))

    @classmethod
    @functools.lru_cache(maxsize=4096)
    def _one_round(cls, rows: int, n: int, k: int, pieces: int = 1, gated: bool = False):
        """The quickest tile of which one round of a workgroup a compute unit is enough, and how many make it; None if none is."""
        if rows <= 64 or n < 1 or k < 64 * pieces or k % 64 != 0 or max(rows, 2 * n if gated else n) * k * 2 >= 2 ** 32:
            return None
        best = None
        for tm, tn, launch, stage in cls.BLOCK_TILES:
            tiles = -(-rows // tm) * -(-n // (tn // 2 if gated else tn)) * pieces
            time = launch + stage * -(-k // (64 * pieces))
            if tiles <= cls.COMPUTE_UNITS and (gated or tm <= 192) and (best is None or time < best[0]):
                best = (time, tm, tn, tiles)
        return best[1:] if best is not None else None

    @classmethod
    def block_gated_tile(cls, rows: int, columns: int, k: int):
        """The tile of a gated product of `columns` output columns, or None: where one round is enough, up to 256 rows, and beyond where the tiles of
        256 x 256 do not take it.  us, tiles of 128 and here, 2,048 keys to 2 x 16,384 columns at 100 / 164 / 256 rows 37.0 / 44.3 / 48.7 and 35.3 / 37.4 /
        42.1; to 2 x 4,096 24.1 / 23.7 / 24.6 and 13.2 / 16.1 / 17.6, at 300 / 512 rows the library's product with the activation's pass 27.6 / 29.2 and
        19.7 / 23.9.  One and a half rounds lose (to 2 x 24,576 at 164 rows 57 and 64).  Beyond 256 rows and 2,048 keys few tiles are a chain of stages on a
        part of the machine, where the library cuts the K axis (with the activation's pass, 4,096 keys to 2 x 250 columns at 300 / 1,024 / 1,200 rows 14 /
        18 / 23 and 19 / 19 / 20, 3,072 to 2 x 128 at 1,024 / 1,200 12 / 18 and 15 / 16): from more than 64 tiles on, of more than 3,072 keys 128.
        Up to 256 rows all have the same bits; beyond, gate and up stay float32 up to the activation, which the library rounds before it."""
        if k > 4096 or (rows > cls.WIDE_TILE and cls.wide_gated_takes(rows, columns, k)):
            return None
        found = cls._one_round(rows, columns, k, gated=True)
        if found is None or (rows > cls.WIDE_TILE and k > 2048 and found[2] <= (64 if k <= 3072 else 128)):
            return None
        return found[:2]

    @classmethod
    def block_split_tile(cls, rows: int, n: int, k: int, pieces: int):
        """The tile of a stack of `pieces` partial sums, or None: where one round is enough, up to 256 rows (16,384 keys to 2,048 columns in 8 pieces at 65 /
        128 / 164 / 256 rows 20.9 / 21.9 / 24.7 / 28.0 us, in tiles of 128, two a compute unit, 26.2 / 26.6 / 26.5 / 28.7).  The same bits."""
        found = cls._one_round(rows, n, k, pieces) if rows <= 256 else None
        return found[:2] if found is not None else None

    @classmethod
    def block_tile(cls, rows: int, n: int, k: int):
        """The tile in which a product rounded to bfloat16 goes instead of to the library, or None: the quickest of which one round of a
        workgroup a compute unit is enough.

        Chosen by what a pass takes, not by the launch alone.  Alone (weights from HBM, us, library and here) the tiles are ahead where they fill
        much of a round (2,048 keys to 2,048 columns at 333 / 900 / 1,200 / 1,800 / 2,300 rows 13 / 16 / 23 / 24 / 29 and 11.7 / 14.8 / 17 / 20 / 26, at
        3,001 28 and 28) and behind by up to an eighth where the library's own are whole and these few (128 and 768 rows 11 / 14 and 12.1 / 15.5, 384 to
        3,072 columns 14 and 15.4), by up to a third at few columns (256 rows to 64 / 16 columns 9.9 / 8.1 and 11.5 / 10.5), by more at more keys
        (4,096 to 2,048 at 128 / 256 rows 13 / 16 and 21 / 21).  But a call of the library costs the host 19 us where a launch costs 6, and steps of up to
        some 300 rows wait for the host.  Passes of one prompt, us, the library always / where the tiles of 64 x 64 fill less than half of the round or
        larger ones less than four fifths / this rule: Tokuvik's 100 / 256 / 500 / 768 rows 4,690 / 4,369 / 3,508, 4,788 / 3,978 / 3,604, 5,000 / 4,632 / 4,591, 6,055 / 5,992 / 5,955,
        Gemma-2B's 100 / 500 / 768 2,203 / 2,225 / 2,089, 3,281 / 3,249 / 3,211, 4,364 / 4,330 / 4,283; in eleven designs at 70 to 1,000 rows this rule is
        the quickest or within 1%.  More than 512 rows to few columns, and more than 3,072 keys where the tiles fill less than nine tenths of
        the round, are the library's, which cuts the K axis: there the pass is the GPU's."""
        if k > 4096 or (n < 1024 and rows > 512):
            return None
        found = cls._one_round(rows, n, k)
        return found[:2] if found is not None and (k <= 3072 or found[2] >= 0.9 * cls.COMPUTE_UNITS) else None

    @classmethod
    def wide_splits(cls, n: int, k: int, rows: int) -> int:
        """Over how many workgroups the product in tiles of 256 splits a long K axis (1: another kernel is better): as many
        pieces as make one round of workgroups, at least 512 keys each and 16 at most.  So they go by the rows, in tiles of 256 (16,384 keys to
        2,048 columns: 8 pieces in tiles of 128 up to 256 rows, 16 up to 512, 10 up to 768, 8 up to 1,024), and a row's sum has other
        bits in a step of another number of tiles.  One number up to 640 rows would cost 10% at 512 rows there and half as much again for 24,576 keys to
        3,072 columns.  Product and norm, 16,384 keys to 2,048
        columns at 512 / 1,024 / 1,500 / 2,048 / 3,001 / 4,096 rows 50 / 73 / 102 / 124 / 193 / 221 us against 55 / 91 in tiles of 128
        (up to 1,024 rows) and 66 / 104 / 120 / 153 / 199 / 239 with the library's; 24,576 to 3,072 at 160 / 512 / 1,024 / 2,048 rows
        52 / 84 / 136 / 268 against 63 / 128 / 239 and 151 / 275 / 282 / 421.  More tiles than half a round leave one piece, and the
        library is mostly ahead (5,000 rows: 280 against 329); fewer than 168 workgroups leave too much of the machine idle (256
        rows to 2,048 columns: 40 against 33 in tiles of 128), and a K axis of 4,096 is too short for what its pieces cost (2,048
        rows: 54 against 48)."""
        if rows <= 128 or n < 1 or k < cls.TILE_LONG_K or k % 64 != 0 or max(rows, n) * k * 2 >= 2 ** 32:
            return 1
        tiles = -(-rows // cls.WIDE_TILE) * -(-n // cls.WIDE_TILE)
        splits = min(16, cls.COMPUTE_UNITS // tiles, k // 512)
        return splits if splits > 1 and tiles * splits >= 168 else 1

    @staticmethod
    def _odd(x: torch.Tensor, weight: torch.Tensor) -> bool:
        """Operands that begin at no multiple of 16 bytes: the loads of the tiles of 128 do not take them, a variant of the tiles of 256
        does, with the same bits in the same pieces."""
        return (x.data_ptr() | weight.data_ptr()) % 16 != 0

    def linear_splits(self, rows, out_features, in_features, dtype) -> int:
        if self.skinny_takes(dtype, rows, in_features):
            return self.piece_split(out_features, in_features)[0] or self.skinny_split(out_features, in_features)
        if dtype == torch.bfloat16 and self.wide_splits(out_features, in_features, rows) > 1:
            return self.wide_splits(out_features, in_features, rows)
        if self.tile_takes(dtype, rows, out_features, in_features):
            return self.tile_splits(out_features, in_features, rows)
        if dtype == torch.float32 and rows <= self.F32_FEW_ROWS:
            return self.lib.wllm_gemm_f32_segments(rows, out_features, in_features)
        return 1

    def tile_weight(self, weight, tiles) -> None:
        self._on_gpu(weight, tiles)
        if weight.dtype == torch.float32:
            self._check(self.lib.wllm_tile_weight_f32(_ptr(weight), _ptr(tiles), weight.shape[0], weight.shape[1],
                                                      self._stream()), "tile_weight (float32)")
            return
        self._check(self.lib.wllm_tile_weight(_ptr(weight), _ptr(tiles), weight.shape[0], weight.shape[1], self._stream()),
                    "tile_weight")

    @staticmethod
    def joined_takes(rows: int, n: int, splits: int, k: int) -> bool:
        """Where a split product whose sum the caller wants itself runs as one launch, the pieces of the K axis meeting
        inside a workgroup (a wavefront each, at most 16).  There every band of 16 columns reads x for itself, so with
        more rows and more columns the two launches that stage x once win: 2,048 keys to 2,568 columns 9.1 against 5.0 us
        at 8 rows, 10.3 against 7.2 at 24, but to 2,048 columns 10.9 against 12.2 at 64; to 10,304 columns 13.9
        against 11.1 at 8 and 15.8 against 16.3 at 24; in two pieces (768 keys to 2,048 columns) 9.9 against 6.7 at 64.
        And with more keys, to 2,048 columns: at 8 rows of 8,192 keys 13.1 against 11.3, of 12,288 14.7 against 16.5; at 16 of
        6,144 12.3 against 11.5, of 8,192 13.4 against 14.0; at 24 of 4,096 12.0 against 11.3, of 6,144 12.8 against 15.3.  (What
        `piece_split` takes comes here only with operands at odd addresses, in its pieces.)"""
        if k > 8192 or rows * k > 98304:
            return False
        return 1 < splits <= 16 and (rows <= 16 or n <= 8192 and (rows <= 32 or rows <= 64 and splits == 2))

    # The kernel of at most 64 rows that brings everything through shared memory (`gemm_stream.hip`, which has the figures): split
    # sums of more columns than `piece_split` takes, and gated products of more rows than two tiles of 16.  Its loads are of 16 bytes.
    @staticmethod
    def stream_takes(x_address: int, w_address: int, rows: int, w_rows: int, k: int, splits: int) -> bool:
        return ((x_address | w_address) % 16 == 0 and k % (64 * splits) == 0 and rows <= 64 and 0 < w_rows * k < 1 << 31
                and rows * k < 1 << 31)

    def _skinny(self, x, weight, out, tiles=None) -> None:
        m, k = x.shape
        n = weight.shape[0]
        pieces, bands = self.piece_split(n, k)
        splits = pieces or self.skinny_split(n, k)
        w, tiled = (tiles, 1) if tiles is not None else (weight, 0)
        whole = out.dim() == 2
        if splits > 1:
            px, pw = x.data_ptr(), w.data_ptr()
            if pieces and (px | pw) % 16 == 0:
                # A whole sum meets inside the workgroups, as many bands each as leave a compute unit one, or, of a long K axis, in a
                # second launch.  us, inside and in two: 2,048 keys to 2,568 columns at 8 / 64 rows 5.1 / 7.8 and 6.7 / 8.9; 4,096 to 2,048
                # 7.9 / 12.2 and 7.8 / 10.3; 5,632 to 2,048 at 8 / 24 rows 10.4 / 11.9 and 8.5 / 9.2.  (The kernels below: 4.9 / 11.1, 6.9 / 14.8 and 9.7 / 15.4.)
                inside = whole and k < 4096
                if inside:
                    bands = min(3, -(-n // (16 * self.COMPUTE_UNITS)))
                elif n > 16 * 3 * self.COMPUTE_UNITS // 2:
                    bands = self.crowded_bands(n, m)
                sums = self._gemm_partial(pieces * m * n, x.device) if whole and not inside else out
                rounded = inside and out.dtype == torch.bfloat16
                self._check(self.lib.wllm_gemm_pieces(px, pw, tiled, None if rounded else sums.data_ptr(),
                                                      out.data_ptr() if rounded else None, m, n, k, pieces, inside, bands, self._stream()),
                            "linear (at most 64 rows, wavefronts' sums joined)")
                if whole and not inside:
                    self._check(self.lib.wllm_split_sum(_ptr(sums), _ptr(out), int(out.dtype == torch.bfloat16), m * n, pieces,
                                                        self._stream()), "linear (sum of partial sums)")
                return
            if not (whole and self.joined_takes(m, n, splits, k)) and self.stream_takes(px, pw, m, n, k, splits):
                sums = self._gemm_partial(splits * m * n, x.device) if whole else out
                self._check(self.lib.wllm_gemm_stream(px, pw, tiled, None, sums.data_ptr(), m, n, k, n, splits, 0, 0.0, 0.0, 0.0,
                                                      self._stream()), "linear (at most 64 rows, partial sums)")
                if whole:
                    self._check(self.lib.wllm_split_sum(_ptr(sums), _ptr(out), int(out.dtype == torch.bfloat16), m * n, splits,
                                                        self._stream()), "linear (sum of partial sums)")
                return
        chunk = self.SKINNY_CHUNK[min(4, -(-m // 16))]
        if not whole:           # the caller adds the partial sums later
            self._check(self.lib.wllm_gemm_skinny(_ptr(x), _ptr(w), tiled, c_void_p(0), 0, _ptr(out), m, n, k, splits,
                                                  chunk, self._stream()), "linear (few rows, partial sums)")
            return
        if self.joined_takes(m, n, splits, k):
            self._check(self.lib.wllm_gemm_skinny_joined(_ptr(x), _ptr(w), tiled, _ptr(out), int(out.dtype == torch.bfloat16),
                                                         m, n, k, splits, self._stream()), "linear (few rows, pieces of K joined)")
            return
        partial = self._gemm_partial(splits * m * n, x.device) if splits > 1 else None
        self._check(self.lib.wllm_gemm_skinny(_ptr(x), _ptr(w), tiled, _ptr(out), int(out.dtype == torch.bfloat16),
                                              _ptr(partial), m, n, k, splits, chunk, self._stream()),
                    "linear (few rows, matrix cores)")

    def linear(self, x, weight, out, tiles=None):
        self._on_gpu(x, weight, out, tiles)
        m, k = x.shape
        if x.dtype == torch.bfloat16:
            if self.skinny_takes(x.dtype, m, k):
                self._skinny(x, weight, out, tiles)
                return
            n, wide = weight.shape[0], self.wide_splits(weight.shape[0], k, m)
            splits = wide if wide > 1 else self.tile_splits(n, k, m) if self.tile_takes(x.dtype, m, n, k) else 1
            # many rows and a long K axis: a tiled product, its K axis in pieces whose sums the caller adds, or a kernel
            # here in their order (without room for them the kernels below make the product)
            stack = out if out.dim() == 3 else None
            if splits > 1 and stack is None:
                stack = ops.scratch_or_none(lambda: torch.empty((splits, m, n), dtype=torch.float32, device=x.device))
            if stack is not None:
                odd = self._odd(x, weight)
                block = self.block_split_tile(m, n, k, splits) if wide == 1 and not odd else None
                if block is not None:
                    self._check(self.lib.wllm_gemm_block(_ptr(x), _ptr(weight), None, _ptr(stack), m, n, k, n, splits, 0, 0.0, 0.0, 0.0,
                                                         *block, self._stream()), "linear (tiles in one round, partial sums)")
                elif wide > 1 or odd:
                    self._check(self.lib.wllm_gemm_wide(_ptr(x), _ptr(weight), None, _ptr(stack), m, n, k, n, splits, 0, 0.0, 0.0,
                                                        0.0, self._stream()), "linear (tiles of 256, partial sums)")
                else:
                    self._check(self.lib.wllm_gemm_tile(_ptr(x), _ptr(weight), None, _ptr(stack), m, n, k, splits, 0, 0.0, 0.0,
                                                        0.0, self._stream()), "linear (tiles, partial sums)")
                if out.dim() == 2:
                    self._check(self.lib.wllm_split_sum(_ptr(stack), _ptr(out), int(out.dtype == torch.bfloat16), m * n, splits,
                                                        self._stream()), "linear (sum of partial sums)")
                return
            if k % 32 == 0 and out.dtype == torch.float32 and self.skinny_split(weight.shape[0], k) == 1:
                # float32 results from bfloat16 operands (logits at many rows): the few-row kernel with a
                # workgroup per 64 rows, placed so that the weights come from HBM once
                self._skinny(x, weight, out, tiles)
                return
            if k % 32 == 0 and out.dtype == torch.float32:
                for r in range(0, m, 64):
                    self._skinny(x[r:r + 64], weight, out[r:r + 64], tiles)
                return
            block = self.block_tile(m, n, k) if out.dtype == torch.bfloat16 else None
            if block is not None and not self._odd(x, weight):
                self._check(self.lib.wllm_gemm_block(_ptr(x), _ptr(weight), _ptr(out), None, m, n, k, n, 1, 0, 0.0, 0.0, 0.0, *block,
                                                     self._stream()), "linear (tiles in one round)")
                return
            if out.dtype == torch.bfloat16 and self.wide_takes(m, n, k):
                self._check(self.lib.wllm_gemm_wide(_ptr(x), _ptr(weight), _ptr(out), None, m, n, k, n, 1, 0, 0.0, 0.0, 0.0,
                                                    self._stream()), "linear (tiles of 256)")
                return
            if out.dtype == torch.bfloat16 and m > 64:
                # many rows: the library's matrix-core product (float32 accumulation)
                if self.library_events is not None:     # a measurement asked for the library's share of a step
                    begin, end = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
                    begin.record()
                    torch.mm(x, weight.t(), out=out)
                    end.record()
                    self.library_events.append((begin, end))
                    return
                torch.mm(x, weight.t(), out=out)
                return
        # float32, few rows, a long K axis: the segments of K are summed by wavefronts of their own
        if x.dtype == torch.float32 and m <= self.F32_FEW_ROWS:
            n = weight.shape[0]
            segments = self.lib.wllm_gemm_f32_segments(m, n, k)
            if out.dim() == 3:      # the caller adds the segments' sums later
                self._check(self.lib.wllm_gemm_generic(_ptr(x), _ptr(weight), _ptr(tiles), 0, c_void_p(0), 0, _ptr(out), m, n, k,
                                                       self._stream()), "linear (float32, partial sums)")
                return
            if segments > 1 and segments * m * n > self.GEMM_PARTIAL_FLOATS:
                # more partial sums than the buffer holds: some rows at a time; a row's sums do not
                # depend on the rows beside it
                rows = self.GEMM_PARTIAL_FLOATS // (segments * n)
                if rows < 1:
                    raise KernelError(f"linear: {segments} segments of {n} columns need more than the "
                                      f"{self.GEMM_PARTIAL_FLOATS} floats of the split-sum buffer for one row")
                for r in range(0, m, rows):
                    self._generic(x[r:r + rows], weight, out[r:r + rows], segments, tiles)
                return
            self._generic(x, weight, out, segments, tiles)
            return
        # float32, more rows: the kernel says whether it cuts the K axis over workgroups; without room for the segments' sums
        # (256 MiB at most) it runs uncut, with the same bits
        n, partial = weight.shape[0], None
        segments = self.lib.wllm_gemm_f32_segments(m, n, k) if x.dtype == out.dtype == torch.float32 else 1
        if segments > 1:
            partial = ops.scratch_or_none(lambda: torch.empty(segments * m * n, dtype=torch.float32, device=x.device))
        self._generic(x, weight, out, 1, partial=partial)

    def _generic(self, x, weight, out, segments: int, tiles=None, partial=None) -> None:
        m, n = x.shape[0], weight.shape[0]
        if segments > 1:
            partial = self._gemm_partial(segments * m * n, x.device)
        self._check(self.lib.wllm_gemm_generic(
            _ptr(x), _ptr(weight), _ptr(tiles) if x.dtype == torch.float32 else c_void_p(0), int(x.dtype == torch.bfloat16),
            _ptr(out), int(out.dtype == torch.bfloat16),
            _ptr(partial), m, n, x.shape[1], self._stream()), "linear")

    def gated_linear_writes_band(self, rows: int, dtype, in_features: int) -> bool:
        """True where `gated_linear` runs a kernel that writes rows of any stride: the few-row product, and
        the activation kernel where the product and the activation are two kernels."""
        if self.skinny_takes(dtype, rows, in_features) and in_features % 64 == 0:
            return True        # the few-row kernel takes a row stride for its result
        return not (dtype == torch.bfloat16 and 64 < rows <= self.TILE_GATED_MAX_ROWS and in_features % 64 == 0)

    def gated_linear(self, x, weight, out, activation, scratch, tiles=None):
        self._on_gpu(x, weight, out, scratch, tiles)
        m, k = x.shape
        w, tiled = (tiles, 1) if tiles is not None else (weight, 0)
        if 32 < m <= 64 and x.dtype == torch.bfloat16:
            px, pw, n = x.data_ptr(), w.data_ptr(), out.shape[1]
            if self.stream_takes(px, pw, m, 2 * n, k, 2):
                number, *shape = gate_args(activation)
                self._check(self.lib.wllm_gemm_stream(px, pw, tiled, out.data_ptr(), None, m, n, k, out.stride(0), 1, 1 + number, *shape,
                                                      self._stream()), "gated_linear (at most 64 rows)")
                return
        if self.skinny_takes(x.dtype, m, k) and k % 64 == 0:
            self._check(self.lib.wllm_gemm_skinny_gated(
                _ptr(x), _ptr(w), tiled, _ptr(out), m, out.shape[1], k, *gate_args(activation),
                self.GATED_CHUNK[-(-m // 16)], out.stride(0) if m > 1 else out.shape[1], self._stream()),
                "gated_linear (few rows, matrix cores)")
            return
        n = out.shape[1]
        tiles_of_128 = (x.dtype == torch.bfloat16 and 64 < m <= self.TILE_GATED_MAX_ROWS and k % 64 == 0
                        and max(m, 2 * n) * k * 2 < 2 ** 32)
        block = self.block_gated_tile(m, n, k) if x.dtype == torch.bfloat16 else None
        if block is not None and not self._odd(x, weight):
            number, *shape = gate_args(activation)
            self._check(self.lib.wllm_gemm_block(_ptr(x), _ptr(weight), _ptr(out), None, m, n, k, out.stride(0), 1, 1 + number, *shape, *block,
                                                 self._stream()), "gated_linear (tiles in one round)")
            return
        if x.dtype == torch.bfloat16 and self.wide_gated_takes(m, n, k) or tiles_of_128 and self._odd(x, weight):
            number, *shape = gate_args(activation)
            self._check(self.lib.wllm_gemm_wide(_ptr(x), _ptr(weight), _ptr(out), None, m, n, k, out.stride(0), 1, 1 + number,
                                                *shape, self._stream()), "gated_linear (tiles of 256)")
            return
        if tiles_of_128:
            # some hundred rows: the tiled product with the activation in its registers
            number, *shape = gate_args(activation)
            self._check(self.lib.wllm_gemm_tile(_ptr(x), _ptr(weight), _ptr(out), None, m, n, k, 1, 1 + number, *shape,
                                                self._stream()),
                        "gated_linear (tiles)")
            return
        # (the tile-major copy of a stacked float32 matrix is that of the one matrix it is; a bfloat16 one's
        # halves are tiled each by itself, which only the gated kernels above read)
        self.linear(x, weight, scratch, tiles if x.dtype == torch.float32 else None)
        ops.call("gated_activation", scratch, out, activation)

    def activated_linear(self, x, weight, out, name, tiles=None, paired_tiles=None):
        self._on_gpu(x, weight, out, tiles, paired_tiles)
        m, k = x.shape
        n = weight.shape[0]
        half = n // 2
        # the kernels that make a gated product's two streams make the two halves of these columns
        if name == "squared_relu" and n % 2 == 0 and x.dtype == torch.bfloat16:
            number = len(ops.ACTIVATIONS) + 1
            w, tiled = (paired_tiles, 1) if paired_tiles is not None else (weight, 0)
            if 32 < m and self.stream_takes(x.data_ptr(), w.data_ptr(), m, n, k, 2):
                self._check(self.lib.wllm_gemm_stream(_ptr(x), _ptr(w), tiled, _ptr(out), None, m, half, k, n, 1, 1 + number, 0.0, 0.0,
                                                      0.0, self._stream()), "activated_linear (at most 64 rows)")
                return
            if self.skinny_takes(x.dtype, m, k) and k % 64 == 0 and out.data_ptr() % 8 == 0:
                self._check(self.lib.wllm_gemm_skinny_gated(
                    _ptr(x), _ptr(w), tiled, _ptr(out), m, half, k, number, 0.0, 0.0, 0.0, self.GATED_CHUNK[-(-m // 16)], n,
                    self._stream()), "activated_linear (few rows, matrix cores)")
                return
            tiles_of_128 = 64 < m <= self.TILE_GATED_MAX_ROWS and k % 64 == 0 and max(m, n) * k * 2 < 2 ** 32
            block = self.block_gated_tile(m, half, k)
            if block is not None and not self._odd(x, weight):
                self._check(self.lib.wllm_gemm_block(_ptr(x), _ptr(weight), _ptr(out), None, m, half, k, n, 1, 1 + number, 0.0, 0.0, 0.0, *block,
                                                     self._stream()), "activated_linear (tiles in one round)")
                return
            if self.wide_gated_takes(m, half, k) or tiles_of_128 and self._odd(x, weight):
                self._check(self.lib.wllm_gemm_wide(_ptr(x), _ptr(weight), _ptr(out), None, m, half, k, n, 1, 1 + number, 0.0, 0.0,
                                                    0.0, self._stream()), "activated_linear (tiles of 256)")
                return
            if tiles_of_128:
                self._check(self.lib.wllm_gemm_tile(_ptr(x), _ptr(weight), _ptr(out), None, m, half, k, 1, 1 + number, 0.0, 0.0,
                                                    0.0, self._stream()), "activated_linear (tiles)")
                return
        self.linear(x, weight, out, tiles)
        ops.call("activation", out, out, name)

    @staticmethod
    def gated_linear_norm_takes(rows: int, dtype, in_features: int) -> bool:
        """The gated product with the norm folded into its load of x: bfloat16, at most 16 rows,
        input size a multiple of 512 (whole chunks of 256 keys per half of the K axis)."""
        return dtype == torch.bfloat16 and 1 <= rows <= 16 and in_features % 512 == 0

    def gated_linear_norm(self, x, weight, out, activation, tiles=None):
        self._on_gpu(x.residual, x.sumsq, x.weight, weight, out, tiles)
        w, tiled = (tiles, 1) if tiles is not None else (weight, 0)
        self._check(self.lib.wllm_gemm_skinny_gated_norm(
            _ptr(x.residual), _ptr(x.sumsq), x.sumsq.shape[1], _ptr(x.weight), x.eps, x.offset, _ptr(w), tiled,
            _ptr(out), x.shape[0], out.shape[1], x.shape[1], *gate_args(activation), self._stream()),
            "gated_linear (norm on load)")

    ARGMAX_ROWS = 4096       # rows per launch; the scratch (64 words a row) is allocated once

    def argmax_rows(self, logits, out):
        self._on_gpu(logits, out)
        if self._argmax_scratch is None or self._argmax_scratch.device != logits.device:
            self._argmax_scratch = torch.empty(self.ARGMAX_ROWS * 64, dtype=torch.int32, device=logits.device)
        for r in range(0, logits.shape[0], self.ARGMAX_ROWS):
            rows = min(self.ARGMAX_ROWS, logits.shape[0] - r)
            self._check(self.lib.wllm_argmax_rows(_ptr(logits[r:r + rows]), _ptr(out[r:r + rows]),
                                                  _ptr(self._argmax_scratch), rows, logits.shape[1], self._stream()),
                        "argmax_rows")

    SAMPLE_SPLIT_ROWS = 256     # up to this many rows each row is spread over many workgroups

    def sample_rows(self, logits, params, seeds, penalty_ids, penalty_offsets, out_tokens, out_logprobs,
                    truncations=True):
        self._on_gpu(logits, params, seeds, penalty_ids, penalty_offsets, out_tokens, out_logprobs)
        rows, vocab = logits.shape
        if rows <= self.SAMPLE_SPLIT_ROWS:
            # a decode step's few rows: one workgroup a row would leave the chip idle
            if self._sample_scratch is None or self._sample_scratch.device != logits.device:
                words = self.lib.wllm_sample_split_row_words()
                self._sample_scratch = torch.empty(self.SAMPLE_SPLIT_ROWS * words, dtype=torch.int64,
                                                   device=logits.device)
            self._check(self.lib.wllm_sample_rows_split(
                _ptr(logits), _ptr(params), _ptr(seeds), _ptr(penalty_ids), _ptr(penalty_offsets), _ptr(out_tokens),
                _ptr(out_logprobs), _ptr(self._sample_scratch), rows, vocab, int(bool(truncations)), self._stream()),
                "sample_rows (rows spread over workgroups)")
            return
        self._check(self.lib.wllm_sample_rows(
            _ptr(logits), _ptr(params), _ptr(seeds), _ptr(penalty_ids), _ptr(penalty_offsets), _ptr(out_tokens),
            _ptr(out_logprobs), rows, vocab, self._stream()), "sample_rows")
