"""The GPT-2 block's linear layers for the decode harness, on libvmi_gpt2_layer.so (include/vmi_gpt2_layer.h).

Counterpart of the torch modules around the reference's call pair — ln_1 -> c_attn, c_proj + residual,
ln_2 -> c_fc -> GELU -> c_proj + residual (vllmini/model/gpt2.py:14-15, 117-128, 130-135, GPT2Block.forward): one
hand-written gfx950 kernel family (csrc/gpt2_layer.hip) that runs each linear layer of a decode step — LayerNorm in front,
bias / GELU / residual add behind — as ONE launch; and prompts whole: attention that also writes the pages
(csrc/gpt2_prompt.hpp), norms, and every launch of all layers from one call (`prompts()`).  There is no torch fallback: a missing
library or an unsupported shape raises.
"""
from __future__ import annotations

import ctypes
import os
import threading
from typing import Optional, Tuple

import numpy as np
import torch

from . import build as _build
from .staging import PinnedBuffer

ABI_VERSION = 1
EPI_BIAS, EPI_BIAS_GELU, EPI_BIAS_RESIDUAL, EPI_BIAS_KV_CACHE = 0, 1, 2, 3

_vp, _i32, _i64 = ctypes.c_void_p, ctypes.c_int32, ctypes.c_int64


class Prompts(ctypes.Structure):
    """vmi_gpt2_prompts."""
    _fields_ = [(n, t) for t, names in (
        (_vp, "layers wte wpe ln_f_g ln_f_b input_ids position_ids tiles block_tables last_rows x qkv attended hidden out key_cache value_cache"),
        (_i64, "kv_block_stride kv_head_stride"),
        (_i32, "num_layers num_heads head_size num_tokens num_prompts num_tiles tile_rows table_ld block_size device"),
        (ctypes.c_float, "eps scale")) for n in names.split()]


SIGNATURES = {
    "vmi_gpt2_linear_f16": (ctypes.c_int, [_vp, _i64, _vp, _vp, _vp, _vp, ctypes.c_float, _vp, _i64, _vp, _i64,
                                           _i32, _i32, _i32, _i32, _i32, _i32, _vp]),
    "vmi_gpt2_linear_qkv_cache_f16": (ctypes.c_int, [_vp, _i64, _vp, _vp, _vp, _vp, ctypes.c_float, _vp, _i64, _i32, _i32, _i32,
                                                     _vp, _vp, _vp, _i32, _i32, _i32, _i64, _i64, _i32, _vp]),
    "vmi_gpt2_embed_f16": (ctypes.c_int, [_vp, _vp, _vp, _vp, _vp, _i32, _i32, _i32, _vp]),
    "vmi_gpt2_linear_slabs": (_i32, [_i32, _i32, _i32, _i32, _i32]),
    "vmi_gpt2_head_fits": (_i32, [_i32, _i32]),
    "vmi_gpt2_head_f16": (ctypes.c_int, [_vp, _i64, _vp, _vp, _vp, ctypes.c_float, _vp, _vp, _i64, _i32, _i32, _i32, _i32, _vp]),
    "vmi_gpt2_step_inputs": (ctypes.c_int, [_vp, _vp, _i64, _i32, _i32, _i32, _vp, _vp, _i32, _i32, _vp]),
    "vmi_gpt2_prompt_attention_f16": (ctypes.c_int, [_vp, _i64, _vp, _i64, _vp, _i32, _i32, _i32, _i32, ctypes.c_float, _vp, _vp,
                                                     _vp, _i32, _i32, _i64, _i64, _i32, _vp]),
    "vmi_gpt2_linear_tiles_f16": (ctypes.c_int, [_vp, _vp, _vp, _vp, _vp, _i32, _i32, _i32, _i32, _i32, _vp]),
    "vmi_gpt2_add_norm_f16": (ctypes.c_int, [_vp, _vp, _vp, _vp, _vp, ctypes.c_float, _vp, _i32, _i32, _i32, _vp]),
    "vmi_gpt2_prompts_f16": (ctypes.c_int, [ctypes.POINTER(Prompts), _vp]),
    "vmi_gpt2_prompts_in_tiles": (_i32, [_i32, _i32]),
    "vmi_gpt2_argmax_f16": (ctypes.c_int, [_vp, _i64, _i32, _i32, _vp, _i32, _vp]),
    "vmi_gpt2_sample_top_k_f16": (ctypes.c_int, [_vp, _i64, _i32, _i32, _i32, ctypes.c_float, _vp, _vp, _i32, _vp]),
    "vmi_gpt2_linear_kernel_name": (ctypes.c_char_p, [_i32, _i32, _i32, _i32, _i32]),
    "vmi_gpt2_layer_last_error": (ctypes.c_char_p, []),
    "vmi_gpt2_layer_abi_version": (_i32, []),
    "vmi_gpt2_layer_target_arch": (ctypes.c_char_p, []),
}

_lock = threading.Lock()
_lib = None


class LayerLibraryError(RuntimeError):
    """libvmi_gpt2_layer.so is missing / stale / does not match the header."""


def load() -> ctypes.CDLL:
    global _lib
    if _lib is None:
        with _lock:
            if _lib is None:
                path = _build.LAYER_LIB_PATH
                if not os.path.exists(path):
                    raise LayerLibraryError(f"{path} not found: build it with `python -m vllmini_amd.build` "
                                            "(or __graft_entry__.build()).  The native layers have no torch fallback; "
                                            "GPT2PagedDecoder(native_layers=False) is the torch-module harness.")
                try:
                    lib = ctypes.CDLL(path)
                except OSError as e:
                    raise LayerLibraryError(f"cannot load {path}: {e}") from e
                for name, (restype, argtypes) in SIGNATURES.items():
                    try:
                        fn = getattr(lib, name)
                    except AttributeError as e:
                        raise LayerLibraryError(f"{path} does not export {name}: it is of older sources, build it with `python -m vllmini_amd.build` (or `make layer`)") from e
                    fn.restype, fn.argtypes = restype, argtypes
                if lib.vmi_gpt2_layer_abi_version() != ABI_VERSION:
                    raise LayerLibraryError(f"{path}: ABI {lib.vmi_gpt2_layer_abi_version()}, expected {ABI_VERSION}: build it with `python -m vllmini_amd.build` (or `make layer`)")
                _lib = lib
    return _lib


def supports(M: int, N: int, K: int) -> bool:
    """Whether linear() takes this shape (K % 32 == 0, N % 16 == 0, K <= 4608)."""
    return load().vmi_gpt2_linear_kernel_name(M, N, K, 0, 0) is not None


def kernel_name(M: int, N: int, K: int, ln: bool = False, epilogue: int = EPI_BIAS) -> Optional[str]:
    s = load().vmi_gpt2_linear_kernel_name(M, N, K, int(ln), epilogue)
    return s.decode() if s else None


class PackedWeight:
    """An nn.Linear weight [N, K] re-laid as the MFMA tiles the kernels read (include/vmi_gpt2_layer.h, w_layout 1):
    tile[s][t][kc * 16 + r][e] = w[16 s + r][32 t + 8 kc + e].  Weights are static, so the harness packs each once."""

    def __init__(self, weight: torch.Tensor):
        N, K = weight.shape
        if N % 16 or K % 32 or weight.dtype != torch.float16:
            raise RuntimeError("pack_weight: half [N, K] with N % 16 == 0 and K % 32 == 0")
        self.shape = (N, K)
        self.tiles = weight.view(N // 16, 16, K // 32, 4, 8).permute(0, 2, 3, 1, 4).contiguous()


def pack_weight(weight: torch.Tensor) -> PackedWeight:
    return PackedWeight(weight)


def linear(x: torch.Tensor, weight, bias: Optional[torch.Tensor] = None, *,
           ln: Optional[Tuple[torch.Tensor, torch.Tensor, float]] = None, gelu: bool = False,
           residual: Optional[torch.Tensor] = None, out: Optional[torch.Tensor] = None) -> torch.Tensor:
    """out = epilogue(LN?(x) @ weight.T + bias): x [M, K] half (last dim contiguous), weight [N, K] half contiguous
    (nn.Linear layout) or its pack_weight() form, ln = (gamma, beta, eps) for a LayerNorm over K in front, gelu / residual [M, N] behind (not both).
    `out` may be `residual` itself.  Launches on torch's current stream; never synchronises."""
    lib = load()
    packed = isinstance(weight, PackedWeight)
    wshape = weight.shape
    if packed:
        weight = weight.tiles
    if x.device.type != "cuda":
        raise RuntimeError("gpt2_layer.linear: there is no CPU path")
    if x.dtype != torch.float16 or weight.dtype != torch.float16:
        raise RuntimeError("gpt2_layer.linear: float16 tensors only")
    if gelu and residual is not None:
        raise RuntimeError("gpt2_layer.linear: gelu and residual are alternative epilogues")
    if x.dim() != 2 or len(wshape) != 2 or x.shape[1] != wshape[1] or x.stride(1) != 1 or not weight.is_contiguous():
        raise RuntimeError("gpt2_layer.linear: x [M, K] with unit stride in K, weight [N, K] contiguous")
    M, K = x.shape
    N = wshape[0]
    if out is None:
        out = torch.empty((M, N), dtype=torch.float16, device=x.device)
    if out.shape != (M, N) or out.stride(1) != 1 or out.dtype != torch.float16:
        raise RuntimeError("gpt2_layer.linear: out [M, N] half with unit stride in N")
    if out.data_ptr() == x.data_ptr():
        # a workgroup stores its columns of `out` while others still read the rows of `x`: only the RESIDUAL may alias out
        raise RuntimeError("gpt2_layer.linear: out must not alias x (out may alias the residual)")
    for t, what in ((bias, "bias"), (ln[0] if ln else None, "ln gamma"), (ln[1] if ln else None, "ln beta")):
        if t is not None and (t.dtype != torch.float16 or not t.is_contiguous() or t.device != x.device):
            raise RuntimeError(f"gpt2_layer.linear: {what} must be a contiguous half tensor on x's device")
    if residual is not None and (residual.shape != (M, N) or residual.stride(1) != 1 or residual.dtype != torch.float16):
        raise RuntimeError("gpt2_layer.linear: residual [M, N] half with unit stride in N")
    epi = EPI_BIAS_GELU if gelu else EPI_BIAS_RESIDUAL if residual is not None else EPI_BIAS
    stream = torch.cuda.current_stream(x.device).cuda_stream
    rc = lib.vmi_gpt2_linear_f16(x.data_ptr(), x.stride(0), weight.data_ptr(), bias.data_ptr() if bias is not None else None,
                                 ln[0].data_ptr() if ln else None, ln[1].data_ptr() if ln else None,
                                 float(ln[2]) if ln else 0.0, residual.data_ptr() if residual is not None else None,
                                 residual.stride(0) if residual is not None else 0, out.data_ptr(), out.stride(0),
                                 M, N, K, epi, int(packed), x.device.index or 0, stream)
    if rc != 0:
        raise RuntimeError(lib.vmi_gpt2_layer_last_error().decode("utf-8", "replace"))
    return out


def linear_tiles(x: torch.Tensor, weight: PackedWeight, bias: Optional[torch.Tensor] = None, *, gelu: bool = False,
                 residual: Optional[torch.Tensor] = None) -> torch.Tensor:
    """linear() for hundreds of rows and more (rows and residual contiguous, K a multiple of 64, no norm in front): a new tensor."""
    lib = load()
    if x.device.type != "cuda":
        raise RuntimeError("gpt2_layer.linear_tiles: there is no CPU path")
    if gelu and residual is not None:
        raise RuntimeError("gpt2_layer.linear_tiles: gelu and residual are alternative epilogues")
    if not isinstance(weight, PackedWeight) or weight.tiles.device != x.device:
        raise RuntimeError("gpt2_layer.linear_tiles: a packed weight on x's device")
    if x.dim() != 2 or x.dtype != torch.float16 or x.shape[1] != weight.shape[1] or not x.is_contiguous():
        raise RuntimeError("gpt2_layer.linear_tiles: x half [M, K], contiguous")
    M, (N, K) = x.shape[0], weight.shape
    for t, shape, what in ((bias, (N,), "bias [N]"), (residual, (M, N), "residual [M, N]")):
        if t is not None and (t.dtype != torch.float16 or t.shape != shape or not t.is_contiguous() or t.device != x.device):
            raise RuntimeError(f"gpt2_layer.linear_tiles: {what} half, contiguous, on x's device")
    out = torch.empty((M, N), dtype=torch.float16, device=x.device)
    epi = EPI_BIAS_GELU if gelu else EPI_BIAS_RESIDUAL if residual is not None else EPI_BIAS
    _check(lib.vmi_gpt2_linear_tiles_f16(x.data_ptr(), weight.tiles.data_ptr(), bias.data_ptr() if bias is not None else None,
                                         residual.data_ptr() if residual is not None else None, out.data_ptr(), M, N, K, epi, x.device.index or 0,
                                         torch.cuda.current_stream(x.device).cuda_stream))
    return out


def linear_qkv_cache(x: torch.Tensor, weight, bias: Optional[torch.Tensor], key_cache: torch.Tensor, value_cache: torch.Tensor,
                     slot_mapping: torch.Tensor, num_heads: int, *, ln: Optional[Tuple[torch.Tensor, torch.Tensor, float]] = None,
                     out: Optional[torch.Tensor] = None) -> torch.Tensor:
    """The q / k / v projection with cache_ops.reshape_and_cache's copy done by the producing kernel: returns qkv [M, 3E] and
    writes every row's k and v into the float16 paged caches at slot_mapping[m] (rows with a negative slot are skipped) — the
    same bytes the reference's call (gpt2.py:44, 81-89) writes from the k / v views of qkv, one launch earlier."""
    lib = load()
    packed = isinstance(weight, PackedWeight)
    wshape = weight.shape
    if packed:
        weight = weight.tiles
    if x.device.type != "cuda":
        raise RuntimeError("gpt2_layer.linear_qkv_cache: there is no CPU path")
    M, K = x.shape
    N = wshape[0]
    E = N // 3
    if N != 3 * E or E % num_heads or x.dtype != torch.float16 or weight.dtype != torch.float16 or x.stride(1) != 1 \
            or wshape[1] != K or not weight.is_contiguous():
        raise RuntimeError("gpt2_layer.linear_qkv_cache: x [M, K] half, weight [3E, K] half contiguous, E = heads * head_size")
    D = E // num_heads
    if key_cache.dtype != torch.float16 or value_cache.dtype != torch.float16 or key_cache.dim() != 5 or value_cache.dim() != 4 \
            or key_cache.shape[4] != 8 or key_cache.shape[1] != num_heads or key_cache.shape[2] * 8 != D \
            or value_cache.shape[1:3] != (num_heads, D) or key_cache.shape[3] != value_cache.shape[3] \
            or not key_cache[0].is_contiguous() or not value_cache[0].is_contiguous() \
            or key_cache.stride(0) != value_cache.stride(0):
        raise RuntimeError("gpt2_layer.linear_qkv_cache: float16 caches in the reference layout [NB, H, D/8, bs, 8] / [NB, H, D, bs]")
    if slot_mapping.dtype != torch.int64 or slot_mapping.shape != (M,) or not slot_mapping.is_contiguous():
        raise RuntimeError("gpt2_layer.linear_qkv_cache: slot_mapping int64 [M]")
    if out is None:
        out = torch.empty((M, N), dtype=torch.float16, device=x.device)
    if out.shape != (M, N) or out.stride(1) != 1 or out.dtype != torch.float16:
        raise RuntimeError("gpt2_layer.linear_qkv_cache: out [M, 3E] half with unit stride in N")
    for t, what in ((bias, "bias"), (ln[0] if ln else None, "ln gamma"), (ln[1] if ln else None, "ln beta")):
        if t is not None and (t.dtype != torch.float16 or not t.is_contiguous() or t.device != x.device):
            raise RuntimeError(f"gpt2_layer.linear_qkv_cache: {what} must be a contiguous half tensor on x's device")
    stream = torch.cuda.current_stream(x.device).cuda_stream
    rc = lib.vmi_gpt2_linear_qkv_cache_f16(x.data_ptr(), x.stride(0), weight.data_ptr(), bias.data_ptr() if bias is not None else None,
                                           ln[0].data_ptr() if ln else None, ln[1].data_ptr() if ln else None,
                                           float(ln[2]) if ln else 0.0, out.data_ptr(), out.stride(0), M, K, int(packed),
                                           key_cache.data_ptr(), value_cache.data_ptr(), slot_mapping.data_ptr(), num_heads, D,
                                           key_cache.shape[3], key_cache.stride(0), key_cache.stride(1), x.device.index or 0, stream)
    if rc != 0:
        raise RuntimeError(lib.vmi_gpt2_layer_last_error().decode("utf-8", "replace"))
    return out


def _check(rc: int) -> None:
    if rc != 0:
        raise RuntimeError(load().vmi_gpt2_layer_last_error().decode("utf-8", "replace"))


def pack_head(weight: torch.Tensor) -> PackedWeight:
    """A vocabulary's weight [V, E] for head(): packed, zero rows up to a multiple of 16."""
    V, E = weight.shape
    padded = torch.zeros(((V + 15) // 16 * 16, E), dtype=weight.dtype, device=weight.device)
    padded[:V] = weight
    packed = PackedWeight(padded)
    packed.shape = (V, E)
    return packed


HEAD_MAX_ROWS = 16


def head_fits(rows: int, width: int) -> bool:
    """Whether head() takes that many rows of that width."""
    return bool(load().vmi_gpt2_head_fits(rows, width))


def head(x: torch.Tensor, weight: PackedWeight, ln: Optional[Tuple[torch.Tensor, torch.Tensor, float]] = None) -> torch.Tensor:
    """Logits [M, V] of few rows x [M, E] behind the final norm (None: as they are), weight from pack_head()."""
    lib = load()
    if x.device.type != "cuda":
        raise RuntimeError("gpt2_layer.head: there is no CPU path")
    (V, E), M = weight.shape, x.shape[0]
    if x.dim() != 2 or x.dtype != torch.float16 or x.shape[1] != E or x.stride(1) != 1 or weight.tiles.device != x.device or weight.tiles.numel() < (V + 15) // 16 * 16 * E:
        raise RuntimeError("gpt2_layer.head: x half [M, E], unit column stride, and pack_head()'s weight beside it")
    if ln is not None:
        for t in ln[:2]:
            if t.dtype != torch.float16 or t.shape != (E,) or not t.is_contiguous() or t.device != x.device:
                raise RuntimeError("gpt2_layer.head: the norm's weight and bias half [E], contiguous, on x's device")
    out = torch.empty((M, V), dtype=torch.float16, device=x.device)
    _check(lib.vmi_gpt2_head_f16(x.data_ptr(), x.stride(0), None, ln[0].data_ptr() if ln else None, ln[1].data_ptr() if ln else None, ln[2] if ln else 0.0,
                                 weight.tiles.data_ptr(), out.data_ptr(), V, M, V, E, x.device.index or 0, torch.cuda.current_stream(x.device).cuda_stream))
    return out


def step_inputs(host: PinnedBuffer, dev: torch.Tensor, head: int, rows: int, ld: int, used: int, ids: Optional[torch.Tensor], ids_out: torch.Tensor) -> None:
    """The first `head` bytes of `host` into `dev`, behind them the first `used` of the `ld` int32 of each of `rows` rows; ids (if any) into the start of ids_out."""
    if not dev.is_contiguous() or min(host.tensor.numel(), dev.numel() * dev.element_size()) < head + rows * ld * 4:
        raise RuntimeError("gpt2_layer.step_inputs: host and device memory hold the head and the rows")
    if ids is not None and not (ids.dtype == ids_out.dtype == torch.int64 and ids.is_contiguous() and ids_out.is_contiguous() and ids.device == dev.device == ids_out.device
                                and ids.numel() <= ids_out.numel()):
        raise RuntimeError("gpt2_layer.step_inputs: int64 ids beside what they are copied to")
    with torch.cuda.device(dev.device):
        _check(load().vmi_gpt2_step_inputs(host.tensor.data_ptr(), dev.data_ptr(), head, rows, ld, used, ids.data_ptr() if ids is not None else None, ids_out.data_ptr(),
                                           ids.numel() if ids is not None else 0, dev.device.index or 0, torch.cuda.current_stream(dev.device).cuda_stream))
        host.read()


def embed(input_ids: torch.Tensor, position_ids: torch.Tensor, wte: torch.Tensor, wpe: torch.Tensor,
          out: Optional[torch.Tensor] = None) -> torch.Tensor:
    """wte[input_ids] + wpe[position_ids] in one launch (gpt2.py: inputs_embeds + position_embeds): int64 ids [T], half tables."""
    lib = load()
    T, E = input_ids.shape[0], wte.shape[1]
    if input_ids.device.type != "cuda":
        raise RuntimeError("gpt2_layer.embed: there is no CPU path")
    if input_ids.dtype != torch.int64 or position_ids.dtype != torch.int64 or position_ids.shape != (T,) \
            or not input_ids.is_contiguous() or not position_ids.is_contiguous() or wte.dtype != torch.float16 \
            or wpe.dtype != torch.float16 or wpe.shape[1] != E or not wte.is_contiguous() or not wpe.is_contiguous():
        raise RuntimeError("gpt2_layer.embed: int64 ids / positions [T], contiguous half tables [V, E] / [P, E]")
    if out is None:
        out = torch.empty((T, E), dtype=torch.float16, device=wte.device)
    _check(lib.vmi_gpt2_embed_f16(input_ids.data_ptr(), position_ids.data_ptr(), wte.data_ptr(), wpe.data_ptr(), out.data_ptr(),
                                  T, E, wte.device.index or 0, torch.cuda.current_stream(wte.device).cuda_stream))
    return out


ADD_NORM_MAX_WIDTH = 4096


def add_norm(x: torch.Tensor, ln: Tuple[torch.Tensor, torch.Tensor, float], add: Optional[torch.Tensor] = None,
             rows: Optional[torch.Tensor] = None) -> torch.Tensor:
    """x += add in place (if given), then layer_norm(x) — of x[rows] where given — as a new tensor; half [., E], contiguous, one launch."""
    lib = load()
    if x.device.type != "cuda":
        raise RuntimeError("gpt2_layer.add_norm: there is no CPU path")
    E = x.shape[-1]
    if x.dim() != 2 or x.dtype != torch.float16 or not x.is_contiguous() or (add is not None and (rows is not None or add.shape != x.shape
                                                                             or add.dtype != torch.float16 or not add.is_contiguous()
                                                                             or add.device != x.device)):
        raise RuntimeError("gpt2_layer.add_norm: half [T, E], contiguous; add of the same shape, not together with rows")
    if rows is not None and (rows.dtype != torch.int32 or rows.dim() != 1 or not rows.is_contiguous() or rows.device != x.device):
        raise RuntimeError("gpt2_layer.add_norm: rows int32 [M]")
    for t in ln[:2]:
        if t.dtype != torch.float16 or t.shape != (E,) or not t.is_contiguous() or t.device != x.device:
            raise RuntimeError("gpt2_layer.add_norm: gamma and beta half [E] on x's device")
    M = x.shape[0] if rows is None else rows.shape[0]
    out = torch.empty((M, E), dtype=torch.float16, device=x.device)
    _check(lib.vmi_gpt2_add_norm_f16(x.data_ptr(), add.data_ptr() if add is not None else None, rows.data_ptr() if rows is not None else None,
                                     ln[0].data_ptr(), ln[1].data_ptr(), float(ln[2]), out.data_ptr(), M, E, x.device.index or 0,
                                     torch.cuda.current_stream(x.device).cuda_stream))
    return out


PROMPT_HEAD_SIZES, PROMPT_BLOCK_SIZE = (64, 128), 16      # what prompt_attention is built for


def prompt_tiles(lens, num_heads: int, head_size: int) -> Tuple[np.ndarray, int]:
    """How prompt_attention's launch is cut: int32 [n, 4] (prompt, its first packed row, first position, length), the longest walks over
    keys first, and the positions of a tile.  64 of them, a row tile a wave.  Heads of 128 take 128 (a key tile read from LDS serves two
    row tiles of a wave) where that leaves two workgroups for every compute unit: 16 heads, 40 prompts of 500 tokens 165.8 -> 145.4 us,
    4 of 900 57.7 -> 49.5, but 16 of 128 13.9 -> 14.7 (256 workgroups).  Heads of 64 lose by it at every size: 12 heads, 40 of 500
    52.3 -> 54.3, 24 of up to 512 23.4 -> 26.7, one of 900 15.9 -> 24.0."""
    lens = np.asarray(lens, dtype=np.int64)
    rows = 128 if head_size == 128 and int((-(-lens // 128)).sum()) * num_heads >= 512 else 64
    per = -(-lens // rows)
    prompt = np.repeat(np.arange(len(lens)), per)
    at = (np.arange(int(per.sum())) - np.repeat(np.cumsum(per) - per, per)) * rows
    tiles = np.stack([prompt, (np.cumsum(lens) - lens)[prompt], at, lens[prompt]], axis=1).astype(np.int32)
    return np.ascontiguousarray(tiles[np.argsort(-np.minimum(at + rows, lens[prompt]), kind="stable")]), rows


def prompt_attention(qkv: torch.Tensor, tiles: torch.Tensor, tile_rows: int, key_cache: torch.Tensor, value_cache: torch.Tensor,
                     block_table: torch.Tensor, num_heads: int, scale: float, out: Optional[torch.Tensor] = None) -> torch.Tensor:
    """Causal attention of whole prompts from the rows of their projection, qkv [T, 3E] half, and cache_ops.reshape_and_cache of those
    rows, in one launch.  tiles: prompt_tiles() on the device; block_table int32 [prompts, n]: the blocks of every prompt."""
    lib = load()
    if qkv.device.type != "cuda":
        raise RuntimeError("gpt2_layer.prompt_attention: there is no CPU path")
    T, E = qkv.shape[0], qkv.shape[1] // 3
    D = E // num_heads
    if qkv.dtype != torch.float16 or qkv.stride(1) != 1 or qkv.shape[1] != 3 * num_heads * D or D not in PROMPT_HEAD_SIZES:
        raise RuntimeError(f"gpt2_layer.prompt_attention: qkv half [T, 3E] of heads of {PROMPT_HEAD_SIZES}")
    if key_cache.dtype != torch.float16 or value_cache.dtype != torch.float16 or key_cache.dim() != 5 or value_cache.dim() != 4 \
            or tuple(key_cache.shape[1:]) != (num_heads, D // 8, PROMPT_BLOCK_SIZE, 8) \
            or tuple(value_cache.shape[1:]) != (num_heads, D, PROMPT_BLOCK_SIZE) or not key_cache[0].is_contiguous() \
            or not value_cache[0].is_contiguous() or key_cache.stride(0) != value_cache.stride(0):
        raise RuntimeError("gpt2_layer.prompt_attention: float16 caches in the reference layout [NB, H, D/8, 16, 8] / [NB, H, D, 16]")
    if tiles.dtype != torch.int32 or tiles.dim() != 2 or tiles.shape[1] != 4 or not tiles.is_contiguous() or tile_rows not in ((64, 128) if D == 128 else (64,)) \
            or block_table.dtype != torch.int32 or block_table.dim() != 2 or block_table.stride(1) != 1 \
            or any(t.device != qkv.device for t in (tiles, block_table, key_cache, value_cache)):
        raise RuntimeError("gpt2_layer.prompt_attention: tiles int32 [n, 4], block_table int32 [prompts, blocks], all on qkv's device")
    if out is None:
        out = torch.empty((T, E), dtype=torch.float16, device=qkv.device)
    if out.shape != (T, E) or out.stride(1) != 1 or out.dtype != torch.float16 or out.device != qkv.device:
        raise RuntimeError("gpt2_layer.prompt_attention: out [T, E] half with unit stride in E")
    _check(lib.vmi_gpt2_prompt_attention_f16(qkv.data_ptr(), qkv.stride(0), out.data_ptr(), out.stride(0), tiles.data_ptr(), tiles.shape[0],
                                             tile_rows, num_heads, D, float(scale), key_cache.data_ptr(), value_cache.data_ptr(),
                                             block_table.data_ptr(), block_table.stride(0), PROMPT_BLOCK_SIZE, key_cache.stride(0),
                                             key_cache.stride(1), qkv.device.index or 0,
                                             torch.cuda.current_stream(qkv.device).cuda_stream))
    return out


# a layer's weights in the order of vmi_gpt2_layer_weights (matrices as pack_weight() lays them out)
LAYER_WEIGHTS = ("ln_1.weight", "ln_1.bias", "attn.c_attn.weight", "attn.c_attn.bias", "attn.c_proj.weight", "attn.c_proj.bias", "ln_2.weight", "ln_2.bias",
                 "mlp.c_fc.weight", "mlp.c_fc.bias", "mlp.c_proj.weight", "mlp.c_proj.bias")


def takes_weights(tensors) -> bool:
    """Whether prompts() and add_norm() can read these by address: half, contiguous, 16-byte aligned, on one device."""
    return all(t.dtype == torch.float16 and t.is_contiguous() and t.device == tensors[0].device and t.data_ptr() % 16 == 0 for t in tensors)


def prompts(weights, ends, input_ids: torch.Tensor, position_ids: torch.Tensor, last_rows: torch.Tensor, tiles: torch.Tensor, tile_rows: int,
            block_tables: torch.Tensor, key_cache: torch.Tensor, value_cache: torch.Tensor, num_heads: int, head_size: int, eps: float,
            scale: float) -> torch.Tensor:
    """All layers over whole prompts, issued from one native call: the normed last rows [prompts, E].  weights: the layers' tensors, LAYER_WEIGHTS
    each, one layer behind the other; ends: wte, wpe, ln_f weight and bias (all such as takes_weights() allows); the others as prompt_attention and
    embed take them, block_tables [layers, prompts, blocks]."""
    T, E, n, dev = input_ids.shape[0], num_heads * head_size, last_rows.shape[0], input_ids.device
    layers = len(weights) // len(LAYER_WEIGHTS)
    if input_ids.dtype != torch.int64 or position_ids.dtype != torch.int64 or position_ids.shape != (T,) or last_rows.dtype != torch.int32 \
            or tiles.dtype != torch.int32 or tiles.dim() != 2 or tiles.shape[1] != 4 or block_tables.dtype != torch.int32 \
            or tuple(block_tables.shape[:2]) != (layers, n) or any(not t.is_contiguous() or t.device != dev for t in (
                input_ids, position_ids, last_rows, tiles, block_tables)):
        raise RuntimeError("gpt2_layer.prompts: int64 ids and positions [T], int32 last rows, tiles [n, 4] and tables [layers, prompts, blocks]")
    if key_cache.dtype != torch.float16 or value_cache.dtype != torch.float16 or key_cache.device != dev or value_cache.device != dev \
            or tuple(key_cache.shape[1:]) != (num_heads, head_size // 8, PROMPT_BLOCK_SIZE, 8) \
            or tuple(value_cache.shape[1:]) != (num_heads, head_size, PROMPT_BLOCK_SIZE) or not key_cache[0].is_contiguous() \
            or not value_cache[0].is_contiguous() or key_cache.stride(0) != value_cache.stride(0):
        raise RuntimeError("gpt2_layer.prompts: float16 caches in the reference layout [NB, H, D/8, 16, 8] / [NB, H, D, 16]")
    work = torch.empty((T, 9 * E), dtype=torch.float16, device=dev)      # x, qkv, attended, hidden
    out = torch.empty((n, E), dtype=torch.float16, device=dev)
    at, w = work.data_ptr(), (ctypes.c_void_p * len(weights))(*[t.data_ptr() for t in weights])
    a = Prompts(ctypes.addressof(w), *[t.data_ptr() for t in (*ends, input_ids, position_ids, tiles, block_tables, last_rows)],
                at, at + 2 * T * E, at + 8 * T * E, at + 10 * T * E, out.data_ptr(), key_cache.data_ptr(), value_cache.data_ptr(),
                key_cache.stride(0), key_cache.stride(1), layers, num_heads, head_size, T, n, tiles.shape[0], tile_rows, block_tables.shape[2],
                PROMPT_BLOCK_SIZE, dev.index or 0, eps, scale)
    _check(load().vmi_gpt2_prompts_f16(ctypes.byref(a), torch.cuda.current_stream(dev).cuda_stream))
    return out


def argmax(logits: torch.Tensor, out: Optional[torch.Tensor] = None) -> torch.Tensor:
    """torch.argmax(logits, -1) for half logits [B, V] (first maximum on ties), one workgroup per row."""
    lib = load()
    if logits.device.type != "cuda":
        raise RuntimeError("gpt2_layer.argmax: there is no CPU path")
    if logits.dim() != 2 or logits.dtype != torch.float16 or logits.stride(1) != 1:
        raise RuntimeError("gpt2_layer.argmax: half logits [B, V] with unit stride in V")
    B, V = logits.shape
    if out is None:
        out = torch.empty((B,), dtype=torch.int64, device=logits.device)
    _check(lib.vmi_gpt2_argmax_f16(logits.data_ptr(), logits.stride(0), B, V, out.data_ptr(), logits.device.index or 0,
                                   torch.cuda.current_stream(logits.device).cuda_stream))
    return out


def sample_top_k(logits: torch.Tensor, top_k: int = 50, temperature: float = 1.0,
                 generator: Optional[torch.Generator] = None, uniform: Optional[torch.Tensor] = None) -> torch.Tensor:
    """Scheduler.sample_next_token (scheduler.py:144-153) for a batch in one launch: logits / temperature -> the top_k largest ->
    softmax -> one draw per row, by inverse CDF over the top_k in descending order at `uniform` (default: torch.rand from
    `generator`).  Same distribution as topk + softmax + multinomial, not the same stream of draws.  int64 [B]."""
    lib = load()
    if logits.device.type != "cuda":
        raise RuntimeError("gpt2_layer.sample_top_k: there is no CPU path")
    if logits.dim() != 2 or logits.dtype != torch.float16 or logits.stride(1) != 1:
        raise RuntimeError("gpt2_layer.sample_top_k: half logits [B, V] with unit stride in V")
    B, V = logits.shape
    if uniform is None:
        uniform = torch.rand(B, device=logits.device, generator=generator)
    if uniform.dtype != torch.float32 or uniform.shape != (B,) or not uniform.is_contiguous():
        raise RuntimeError("gpt2_layer.sample_top_k: uniform float32 [B]")
    out = torch.empty((B,), dtype=torch.int64, device=logits.device)
    _check(lib.vmi_gpt2_sample_top_k_f16(logits.data_ptr(), logits.stride(0), B, V, min(top_k, V), float(temperature),
                                         uniform.data_ptr(), out.data_ptr(), logits.device.index or 0,
                                         torch.cuda.current_stream(logits.device).cuda_stream))
    return out

