"""Python face of libslm_latent.so (include/slm_latent.h): the dense 16- / 32-bit ops and latent attention.

Everything runs on torch's current stream and is hipGraph-capturable.  Shapes are checked here, on the host;
there is no fallback: a missing library or a CPU tensor raises.
"""
from __future__ import annotations

import ctypes as C
from typing import List, Optional, Tuple

import numpy as np
import torch

from . import _lib
from ._lib import SLM_BF16, SLM_F32, SlmError, latent_check
from .kernels import current_stream_handle as _stream, reserve_workspace

# rows up to which a bf16 product of row-major weights is streamed
STREAM_MAX_ROWS = 32
# rows from which the tile kernel may do a stored product of row-major weights
TILE_MIN_ROWS = 129
# the same of weights in the streamed layout (stream_layout()), where the product reduces or activates in its epilogue
STREAM_LAYOUT_MAX_ROWS = 128
# clamped GLU: y = g * sigmoid(alpha * g) * (u + shift)
GLU_ALPHA, GLU_SHIFT = 1.702, 1.0


def _code(t: torch.Tensor) -> int:
    if t.dtype == torch.bfloat16:
        return SLM_BF16
    if t.dtype == torch.float32:
        return SLM_F32
    raise SlmError(f"unsupported dtype {t.dtype}: bfloat16 / float32 only")


def _p(t: Optional[torch.Tensor]):
    if t is None:
        return None
    if not t.is_cuda:
        raise SlmError("libslm_latent needs GPU tensors (no CPU fallback)")
    return t.data_ptr()


def _need(ok: bool, what: str) -> None:
    if not ok:
        raise SlmError(what)


def _i32(t: torch.Tensor, n: int, what: str) -> None:
    _need(t.dtype == torch.int32 and t.is_contiguous() and t.numel() >= n, f"{what}: contiguous int32 [>= {n}]")


def arrays_to_device(arrays, device) -> List[torch.Tensor]:
    """Contiguous int32 numpy arrays as tensors on the device, in one copy that nobody waits for: a copy out of pageable memory waits for all that
    the stream has to do, and the device then for the host."""
    if torch.device(device).type != "cuda":
        return [torch.from_numpy(a).to(device) for a in arrays]
    _need(not torch.cuda.is_current_stream_capturing(), "a step's plan is made of host data: it can't be captured")
    _need(all(a.dtype == np.int32 for a in arrays), "plans are int32")
    at, total = [], 0
    for a in arrays:
        at.append(total)
        total += (a.size + 3) // 4 * 4   # (each on 16 bytes)
    host = torch.empty(total, dtype=torch.int32, pin_memory=True)   # (torch's host pool keeps it until the copy is done)
    flat = host.numpy()
    for i, a in zip(at, arrays):
        flat[i:i + a.size] = a.reshape(-1)
    dev = host.to(device, non_blocking=True)
    return [dev[i:i + a.size].view(a.shape) for i, a in zip(at, arrays)]


class TanhNorm:
    """tanh(alpha x) * weight + bias in place of a norm's statistics; given to residual_norm() as its weight."""
    __slots__ = ("alpha", "weight", "bias")

    def __init__(self, alpha: float, weight: torch.Tensor, bias: torch.Tensor):
        self.alpha, self.weight, self.bias = float(alpha), weight, bias


class Slabs:
    """fp32 split-K partial sums [n, rows, ld] that residual_norm() adds up."""
    __slots__ = ("t",)

    def __init__(self, t: torch.Tensor):
        self.t = t


def residual_norm(resid: torch.Tensor, out: Optional[torch.Tensor], weight, eps: float,
                  delta=None, embed=None, row_index: Optional[torch.Tensor] = None, mult: float = 1.0,
                  row_shift: int = 0, clear: Optional[torch.Tensor] = None) -> None:
    """resid (fp32 [rows, width]) += mult * delta (a [rows, >= width] tensor or Slabs), or
    resid = mult * (table[tokens] (+ pos[positions])) for embed = (tokens, table, positions, pos); then
    out = rms_norm(resid) * weight, or a TanhNorm given as weight, zero padded to out's width.  weight = None: the sum only.
    row_index: out row r is the norm of stream row row_index[r] + row_shift; nothing is added.  clear (int32, with embed): set to zero."""
    a = _lib.ResidualNormArgs()
    rows, width = resid.shape
    _need(resid.dtype == torch.float32 and resid.is_contiguous(), "residual_norm: resid is contiguous fp32")
    ref = out if out is not None else (delta if isinstance(delta, torch.Tensor) else None)
    a.resid, a.width, a.eps, a.delta_mult = _p(resid), width, float(eps), float(mult)
    if embed is not None:
        tokens, table, positions, pos = embed
        _i32(tokens, rows, "tokens")
        _need(table.dim() == 2 and table.stride(1) == 1 and table.size(1) >= width, "residual_norm: embedding table")
        a.mode, a.tokens, a.embed, a.ld_embed = _lib.RN_EMBED, _p(tokens), _p(table), table.stride(0)
        ref = table
        if pos is not None:
            _i32(positions, rows, "positions")
            _need(pos.is_contiguous() and pos.size(1) == width and pos.dtype == table.dtype, "residual_norm: position table")
            a.positions, a.pos_table = _p(positions), _p(pos)
    elif isinstance(delta, Slabs):
        t = delta.t
        _need(t.dtype == torch.float32 and t.is_contiguous() and t.dim() == 3 and t.size(1) == rows and t.size(2) >= width,
              "residual_norm: slabs are fp32 [n, rows, >= width]")
        a.mode, a.slabs, a.n_slabs, a.ld_delta, a.slab_stride = _lib.RN_SLABS, _p(t), t.size(0), t.size(2), t.stride(0)
    elif delta is not None:
        _need(delta.size(0) == rows and delta.size(1) >= width and delta.stride(1) == 1, "residual_norm: delta [rows, >= width]")
        _need(out is None or out.dtype == delta.dtype, "residual_norm: dtypes")
        a.mode, a.delta, a.ld_delta = _lib.RN_ADD, _p(delta), delta.stride(0)
    else:
        a.mode = _lib.RN_PLAIN
        if row_index is not None:
            _need(out is not None, "residual_norm: row_index needs an output")
            rows = out.size(0)
            _i32(row_index, rows, "row_index")
            a.row_index, a.row_shift = _p(row_index), row_shift
    a.rows = rows
    if clear is not None:
        _need(embed is not None and clear.dtype == torch.int32 and clear.is_contiguous() and clear.device == resid.device, "residual_norm: clear")
        a.clear, a.n_clear = _p(clear), clear.numel()
    if isinstance(weight, TanhNorm):
        t, weight = weight, weight.weight
        _need(t.bias.dtype == torch.float32 and t.bias.numel() == width and t.bias.is_contiguous(), "norm bias: fp32 [width]")
        a.norm, a.norm_alpha, a.bias = _lib.NORM_TANH, t.alpha, _p(t.bias)
    if weight is not None:
        _need(weight.dtype == torch.float32 and weight.numel() == width and weight.is_contiguous(), "norm weight: fp32 [width]")
        _need(out.size(0) == rows and out.stride(1) == 1 and out.size(1) >= width, "residual_norm: out [rows, >= width]")
        a.weight, a.out, a.ld_out = _p(weight), _p(out), out.size(1)
        _need(out.stride(0) == out.size(1), "residual_norm: out rows are contiguous")
    a.dtype = _code(ref) if ref is not None else SLM_F32
    latent_check(_lib.latent_lib().slm_residual_norm(C.byref(a), _stream()), "slm_residual_norm")


def wanted_rows(params, T: int):
    """Which stream rows a step's logits are of: None for every row (each sequence brings one), else (index tensor, what to add to it):
    params.logit_rows, by default the last row of every sequence."""
    if params.logit_rows is not None:
        return params.logit_rows, 0
    q_cu = params.q_cu_seq_lens
    if params.q_max_seq_len == 1 and T == q_cu.numel() - 1 > 0:
        return None
    return (q_cu[1:], -1) if q_cu.is_contiguous() else (q_cu[1:] - 1, 0)


def _linear_args(x, w, M, N, K) -> "_lib.LinearArgs":
    a = _lib.LinearArgs()
    a.x, a.w, a.M, a.N, a.K = _p(x), _p(w), M, N, K
    a.alpha, a.batch, a.n_splits, a.dtype = 1.0, 1, 1, _code(w)
    return a


def _run_linear(a) -> None:
    latent_check(_lib.latent_lib().slm_linear(C.byref(a), _stream()), "slm_linear")


def _check_xw(x, w) -> Tuple[int, int, int]:
    _need(x.dim() == 2 and w.dim() == 2 and x.dtype == w.dtype and x.size(1) == w.size(1) and x.stride(1) == 1 and
          w.is_contiguous(), "linear: x [M, K], w [N, K] contiguous, one dtype")
    return x.size(0), w.size(0), w.size(1)


def streams_rows(x: torch.Tensor) -> bool:
    """Does the weight-streaming kernel serve this row count (32-bit: always)?"""
    return x.dtype == torch.float32 or x.size(0) <= STREAM_MAX_ROWS


def stream_layout(w: torch.Tensor, glu: bool = False) -> Optional[torch.Tensor]:
    """W [N, K] once more in the order slm_linear_stream reads it (include/slm_latent.h), made at load: what products of
    few rows run on.  The row-major tensor stays for products of many.  glu: W = [gate | up].  None where that kernel has
    no form (32-bit weights, gate halves that are no multiple of 32) and for weights that no kernel reads yet (a model
    loaded on the host).  It is a copy of w as it is now: once w is changed in place (its version counter tells; inference
    tensors have none and are not followed) products are w's own again, until a new layout is made."""
    N, K = w.shape
    if w.dtype != torch.bfloat16 or K % 64 or N % 16 or (glu and N % 64) or not w.is_cuda or not w.is_contiguous() or w.data_ptr() % 16:
        return None
    out = torch.empty((N + 63) // 64, K // 64, 4, 2, 64, 8, dtype=w.dtype, device=w.device)
    with torch.cuda.device(w.device):   # (a model may be built before its device is made the current one)
        latent_check(_lib.latent_lib().slm_stream_layout(_p(out), _p(w), N, K, int(glu), _stream()), "slm_stream_layout")
    if not w.is_inference():
        out.copy_of, out.copy_version = w, w._version
    return out


def spare_memory(device: torch.device) -> int:
    """Half of what is left of the device's memory."""
    if device.type != "cuda":
        return 0
    return (torch.cuda.mem_get_info(device)[0] + torch.cuda.memory_reserved(device) - torch.cuda.memory_allocated(device)) // 2


def lay_out(holders, spare: Optional[int] = None) -> None:
    """Makes the streamed layouts of holders' weights (STREAMED: attribute of the layout, of the weight, gate and up?), in their
    order, as many as fit into `spare` bytes and can be had; products of the others run on the weights alone."""
    for holder in holders:
        for name, weight, glu in holder.STREAMED:
            w = getattr(holder, weight)
            size = (w.size(0) + 63) // 64 * 64 * w.size(1) * w.element_size()
            setattr(holder, name, None)
            if spare is not None and size > spare:
                continue
            try:
                setattr(holder, name, stream_layout(w, glu))
            except torch.OutOfMemoryError:
                spare = 0
                continue
            if spare is not None and getattr(holder, name) is not None:
                spare -= size


def layout_is_current(layout: torch.Tensor, w: torch.Tensor) -> bool:
    of = getattr(layout, "copy_of", None)
    return of is None or (of.data_ptr() == w.data_ptr() and of._version == layout.copy_version)


def copied_weights(layouts) -> List[torch.Tensor]:
    """The weights behind layouts (None among them) that can be followed."""
    return [t.copy_of for t in layouts if hasattr(t, "copy_of")]


def slab_rows(layout: Optional[torch.Tensor]) -> int:
    """Rows up to which a product with this streamed layout (None, or of a weight that has changed: row-major weights only) is left as slabs."""
    if layout is None or not layout_is_current(layout, getattr(layout, "copy_of", None)):
        return STREAM_MAX_ROWS
    return STREAM_LAYOUT_MAX_ROWS


def _stream_args(x, w, layout, M, N, K, rows) -> "Optional[_lib.LinearArgs]":
    """Arguments of slm_linear_stream, or None where it does not serve the call."""
    if layout is None or M > rows or x.stride(0) < K or x.stride(0) % 8 or x.data_ptr() % 16:   # (rows that overlap: the vendor's)
        return None
    if not layout_is_current(layout, w):
        return None
    _need(layout.is_contiguous() and layout.dtype == x.dtype and layout.numel() == (N + 63) // 64 * 64 * K, "linear: streamed layout of w")
    a = _linear_args(x, w, M, N, K)
    a.w, a.ldx, a.ldw = _p(layout), x.stride(0), K
    return a


def _run_stream(a) -> None:
    latent_check(_lib.latent_lib().slm_linear_stream(C.byref(a), _stream()), "slm_linear_stream")


def _store_rows(N: int, K: int) -> int:
    """Rows up to which a product that is only stored is streamed.  Without slabs its workgroups are its columns': from 33
    rows the vendor GEMM, which splits K for itself, is level or ahead under 8192 columns (6752 x 4096, 64 rows: 17.8 us
    against 21.8) and a little above where K is long (vendor / streamed, 64 rows: 8192 x 2048 13.7 / 12.4, x 4096 18.6 / 21.9, x 8192
    32.7 / 41.0; 9216 x 4096 26.4 / 22.5, x 8192 40.2 / 42.1; 12288 x 8192 44.8 / 43.1).  Above 64 rows it is far ahead for
    narrow products; of the widest up to 96 rows it is 2 to 3 us behind (12608 x 4096, 85 rows 29.0 / 25.7; 12288 x 2048, 96 rows 17.2 / 15.3), which this
    line doesn't follow, and level from there on (16896 x 4096, 128 rows 42.1 / 43.0; 64 rows 39.6 / 33.9)."""
    return 64 if N >= 8192 and K <= 2048 + 5 * (N - 8192) // 2 else STREAM_MAX_ROWS


class StepTickets:
    """What the products of one step that are cut in K count their arrivals by: `words`, cleared by the residual_norm() of the embedding that they
    follow.  Streamed products share the first ones, which each of them leaves at zero; a tile product takes some of its own."""
    __slots__ = ("words", "at")

    def __init__(self, words: torch.Tensor):
        self.words, self.at = words, _lib.STREAM_TICKETS

    def take(self) -> Optional[torch.Tensor]:
        """Counters of the next tile product; None: none left (it clears some itself)."""
        at, self.at = self.at, self.at + _lib.GEMM_COUNTERS
        return self.words[at:self.at] if self.at <= self.words.numel() else None


def step_tickets(rows: int, width: int, products: int, device) -> Optional[StepTickets]:
    """For a step of so many rows of a stream of that width and at most so many tile products (None: nothing is cut)."""
    if rows <= 16 or (rows <= STREAM_MAX_ROWS and width < 4096):   # (join_count)
        return None
    n = 0 if rows < TILE_MIN_ROWS else min(products, 240)
    return StepTickets(torch.empty(_lib.STREAM_TICKETS + n * _lib.GEMM_COUNTERS, dtype=torch.int32, device=device))


def _check_counters(t: torch.Tensor, n: int, device) -> None:
    _need(t.dtype == torch.int32 and t.is_contiguous() and t.numel() >= n and t.device == device, "linear: counters")


def join_count(N: int, K: int, rows: int) -> int:
    """Slices of K of a product that is only stored and cut in one launch; 1: not cut.  As many as give every CU a workgroup of 64 columns, ten steps
    of 64 each at least: joining them costs 2 to 4 us.  us, vendor / whole / cut, 64 and 128 rows: 6752 x 4096 in 2 18.9 / 22.6 / 17.7, 26.4 / 28.2 / 22.8;
    6464 x 2048 in 2 13.2 / 12.3 / 10.7, 15.4 / 16.0 / 13.9; 3664 x 2048 in 3 12.1 / 11.7 / 9.1, 14.7 / 15.4 / 11.8; 4096 x 4096 in 4 15.1 / 21.4 / 12.0, 24.4 /
    27.5 / 15.0; 2048 x 8192 in 8 22.3 / 37.7 / 13.2, 21.2 / 49.0 / 16.4; 8192 x 8192 in 2 35.0 / 44.4 / 30.0, 49.6 / 53.1 / 38.8; 512 x 4096 in 6 14.1 / 19.5 /
    8.6, 14.4 / 25.9 / 11.3; short ones are whole (6464 x 1024 11.9 / 7.6 / 7.9, 12.6 / 9.9 / 10.4).  Between half and five eighths of the CUs long ones are
    cut in three for workgroups of 128 columns (9216 x 4096 25.7 / 22.9 / 19.9, 30.3 / 28.9 / 26.5), wider ones are whole (12608 x 4096 25.7 / 24.5 / 26.1).  Up to
    32 rows only long products gain (6752 x 4096 15.9 / 15.3 / 13.7, 3664 x 2048 11.7 / 8.2 / 8.1)."""
    if not 16 < rows <= STREAM_LAYOUT_MAX_ROWS or N > 32 * _lib.STREAM_TICKETS or (rows <= STREAM_MAX_ROWS and K < 4096):
        return 1
    panels = (N + 63) // 64
    if 128 < panels <= 160 and K >= 4096:
        return 3
    return max(1, min(8, 256 // panels, K // 640))


def _joined(a, n: int, words: torch.Tensor, device) -> bool:
    """The stored product in n slices of K; False: no memory for them."""
    L = _lib.latent_lib()
    _check_counters(words, _lib.STREAM_TICKETS, device)
    a.n_splits = n
    try:   # (the launch's own: products of other streams have theirs)
        ws = torch.empty(L.slm_linear_stream_join_bytes(C.byref(a)), dtype=torch.uint8, device=device)
    except torch.OutOfMemoryError:
        a.n_splits = 1
        return False
    latent_check(L.slm_linear_stream_join(C.byref(a), ws.data_ptr(), ws.numel(), words.data_ptr(), _stream()), "slm_linear_stream_join")
    return True


def _tile_pays(M: int, N: int, K: int, glu: bool) -> bool:
    """Is a product that the tile kernel takes its own, or the vendor's?  us by the device, vendor / tiles, where they are the vendor's:
    129 - 160 rows of large weights, whose one row of tiles reads them slower (28672 x 4096 GLU 59 / 74, from 161 rows 67 / 65; of the largest up to 192
    rows: 16384 x 8192, 170 rows, 75 / 93), and
    256 x 256 tiles that fill whole rounds of the chip (4096 x 4096, K 2048 49 / 53, 4096 89 / 94; 4096 x 16384 x 4096 363 / 388).
    Short and narrow products are up to 8 us longer by the device (207 x 512 x 2048 8.5 / 15.8, 207 x 4096 x 4096 17.5 / 20.6) and stay here all the same: steps
    with prompts run eagerly, and the vendor product takes 8 us more of the host for each (18 / 10).  Steps of four layers with one prompt of
    150 - 300 tokens, all their products by the vendor / here: 2b 847 / 580 and 836 / 618, 8b 975 / 903 and 1189 / 1065."""
    if 128 < M <= (192 if N * K >= 1 << 27 else 160) and N * K >= 1 << 26:
        return False
    return glu or M <= 1024 or K < 1024 or -(-M // 256) * -(-N // 256) % 256 != 0


def _gemm(x: torch.Tensor, w: torch.Tensor, out: torch.Tensor, glu=None, tile: int = -1, slices: int = 0, tickets: Optional[StepTickets] = None) -> bool:
    """out = x w^T, or with glu = (limit, alpha, shift) the clamped GLU of its halves, by the tile kernel for many rows.  tickets: step_tickets(),
    cleared.  False: shapes and strides that it does not take."""
    M, (N, K), dtype = x.size(0), w.shape, x.dtype
    half, ldx, ldw, ldy = dtype == torch.float16, x.stride(0), w.stride(0), out.stride(0)
    if (not (half or dtype == torch.bfloat16) or w.dtype != dtype or out.dtype != dtype or not N or not K or K % 64 or N % (32 if glu else 16) or
            ldx < K or (ldx | ldw | ldy) % 8 or (x.data_ptr() | w.data_ptr() | out.data_ptr()) % 16 or max(M * ldx, N * ldw) > 1 << 30 or max(M, N) > 1 << 24):
        return False
    limit, alpha, shift = glu or (0.0, 0.0, 0.0)
    # (in the order of the fields: a third of what setting them one by one takes)
    a = _lib.LinearArgs(_p(x), _p(w), _p(out), None, M, N, K, ldx, ldw, ldy, 0, 0, 0, 0, 1.0, limit, alpha, shift, 1, 1, _lib.LIN_GLU if glu else _lib.LIN_STORE,
                         _lib.SLM_F16 if half else SLM_BF16)
    L = _lib.latent_lib()
    need, ws = L.slm_gemm_workspace_bytes(C.byref(a), tile, slices), None
    if need:
        try:   # (its own: products of other streams have theirs; without it no tile is cut)
            ws = torch.empty(need, dtype=torch.uint8, device=x.device)
        except torch.OutOfMemoryError:
            need = 0
    counters = tickets.take() if need and tickets is not None else None
    if counters is not None:
        _check_counters(counters, _lib.GEMM_COUNTERS, x.device)
        latent_check(L.slm_gemm_counted(C.byref(a), ws.data_ptr(), need, counters.data_ptr(), tile, slices, _stream()), "slm_gemm_counted")
        return True
    latent_check((L.slm_gemm_half if half else L.slm_gemm)(C.byref(a), ws.data_ptr() if ws is not None else None, need, tile, slices, _stream()), "slm_gemm")
    return True


gemm = _gemm   # (for other modules)


def linear(x: torch.Tensor, w: torch.Tensor, out: Optional[torch.Tensor] = None, layout: Optional[torch.Tensor] = None,
           tickets: Optional[StepTickets] = None) -> torch.Tensor:
    """x [M, K] W[N, K]^T -> [M, N] of the same dtype.  layout: stream_layout(w); tickets: step_tickets(), cleared."""
    M, N, K = _check_xw(x, w)
    if out is None:
        out = torch.empty(M, N, dtype=x.dtype, device=x.device)
    _need(out.shape == (M, N) and out.stride(1) == 1 and out.dtype == x.dtype, "linear: out [M, N]")
    n = join_count(N, K, M) if tickets is not None else 1
    # (with tickets what is not cut is short or wide, and streamed: us, vendor / whole, 96 and 128 rows: 12608 x 4096 30.5 / 27.7, 32.3 / 30.9; 16384 x 4096
    # 38.2 / 31.1, 38.8 / 34.9; 10240 x 2048 16.8 / 14.9, 18.2 / 16.8)
    a = _stream_args(x, w, layout, M, N, K, _store_rows(N, K) if tickets is None else STREAM_LAYOUT_MAX_ROWS)
    if a is not None:
        a.ldy, a.y, a.epilogue = out.stride(0), _p(out), _lib.LIN_STORE
        if n == 1 or not _joined(a, n, tickets.words, x.device):
            _run_stream(a)
        return out
    if not streams_rows(x):
        # (of row-major weights stored products of up to 128 rows are the vendor's, whose small tiles leave fewer CUs idle)
        return out if M >= TILE_MIN_ROWS and _tile_pays(M, N, K, False) and _gemm(x, w, out, tickets=tickets) else torch.mm(x, w.t(), out=out)
    a = _linear_args(x, w, M, N, K)
    a.ldx, a.ldw, a.ldy, a.y, a.epilogue = x.stride(0), K, out.stride(0), _p(out), _lib.LIN_STORE
    _run_linear(a)
    return out


def linear_f32(x: torch.Tensor, w: torch.Tensor, alpha: float = 1.0, layout: Optional[torch.Tensor] = None) -> torch.Tensor:
    """alpha * x W^T as fp32 (logits).  layout: stream_layout(w)."""
    M, N, K = _check_xw(x, w)
    out = torch.empty(M, N, dtype=torch.float32, device=x.device)
    s = _stream_args(x, w, layout, M, N, K, M)
    a = s if s is not None else _linear_args(x, w, M, N, K)
    a.ldx, a.ldw, a.ldy, a.y, a.epilogue, a.alpha = x.stride(0), K, N, _p(out), _lib.LIN_F32, float(alpha)
    (_run_linear if s is None else _run_stream)(a)
    return out


def stream_split_count(n_out: int, k: int, rows: int) -> int:
    """Slabs of a streamed product: as many as give every CU a workgroup of 64 columns, at least 8 steps of 64 each (a slab
    is written and read: 4096 x 14336, 128 rows, 4 against 8 slabs 30.4 us against 28.3, and 1 us less behind it).  Above 32 rows a step is
    0.3 to 0.5 us long, so short products of few columns take 4 steps each (with the norm behind them, 100 rows, before / after / vendor
    product: 512 x 512 10.0 / 8.1 / 7.6, 2048 x 896 13.4 / 10.0 / 10.3, 1024 x 1536
    10.7 / 9.5 / 10.1, 4096 x 768 13.2 / 11.4 / 10.9; more columns leave no CUs for it: 5504 x 640 13.3 / 13.3 / 10.9), and large ones
    above 64 rows two workgroups a CU, which hide each other's waits (with the norm, 128 rows, 2 / 4 / 8 slabs: 8192 x 8192 38.1 / 36.3 / 46.6,
    8192 x 14336 63.1 / 55.3 / 67.6)."""
    panels = (n_out + 63) // 64
    wgs = 512 if rows > 64 and n_out > 4096 and k >= (8192 if n_out <= 8192 else 4096) else 256
    step = 256 if rows > STREAM_MAX_ROWS and ((k < 2048 and n_out <= 2048) or (k < 1024 and n_out <= 4096)) else 512
    return max(1, min(8, wgs // panels, k // step))


def glu_split_count(n_out: int, k: int, rows: int) -> int:
    """Slabs of a streamed product in front of the GLU; 1: the GLU is its epilogue.  A workgroup of that form walks all of K, 0.29 us a
    step of 64 up to 64 rows and 0.43 above, however few columns there are; slabs share it out for one launch more (epilogue / slabs /
    vendor product and GLU, us, 64 rows: 1024 x 1024 7.9 / 6.3 / 10.8, 1024 x 8192 39.0 / 10.9 / 15.9, 4096 x 4096 22.3 / 13.0 / 17.9, 8192 x 1024 8.6 / 9.9 /
    14.8; 128 rows: 512 x 512 7.2 / 7.4 / 8.8, 4096 x 4096 28.8 / 23.1 / 28.7, 8192 x 8192 62.3 / 55.6 / 66.6; by the epilogue, vendor: 14336 x 2048 26.3 / 34.5,
    14336 x 8192 89 / 118).  Up to 32 rows the epilogue is ahead of row-major weights at every size."""
    if rows <= STREAM_MAX_ROWS or (k < 1536 and n_out > 4096):
        return 1
    return stream_split_count(n_out, k, rows)


def split_count(rows: int, n_out: int, k: int) -> int:
    """Split-K slabs of a narrow product: enough workgroups for the chip, at least 4 steps of 64 per wave."""
    per = 16 if rows <= 16 else 32
    wgs = (n_out + per - 1) // per
    return max(1, min(8, 768 // max(wgs, 1), k // 1024))


def linear_slabs(x: torch.Tensor, w: torch.Tensor, layout: Optional[torch.Tensor] = None) -> Slabs:
    """x W^T left as fp32 split-K partial sums for residual_norm().  layout: stream_layout(w)."""
    M, N, K = _check_xw(x, w)
    s = _stream_args(x, w, layout, M, N, K, STREAM_LAYOUT_MAX_ROWS)
    n = split_count(M, N, K) if s is None else stream_split_count(N, K, M)
    out = torch.empty(n, M, N, dtype=torch.float32, device=x.device)
    a = s if s is not None else _linear_args(x, w, M, N, K)
    a.ldx, a.ldw, a.ldy, a.y, a.epilogue, a.n_splits = x.stride(0), K, N, _p(out), _lib.LIN_SLABS, n
    (_run_linear if s is None else _run_stream)(a)
    return Slabs(out)


def linear_glu(x: torch.Tensor, w_gate_up: torch.Tensor, out: torch.Tensor, limit: float, alpha: float = GLU_ALPHA,
               shift: float = GLU_SHIFT, layout: Optional[torch.Tensor] = None, tickets: Optional[StepTickets] = None) -> torch.Tensor:
    """out = clamped GLU of the two halves of x [gate | up]^T: the activation is the product's epilogue where a streaming kernel or
    the tile kernel runs, one more launch behind the vendor GEMM otherwise.  layout: stream_layout(w_gate_up, glu=True)."""
    M, N, K = _check_xw(x, w_gate_up)
    half = N // 2
    _need(out.shape == (M, half) and out.stride(1) == 1 and out.dtype == x.dtype, "linear_glu: out [M, N / 2]")
    s = _stream_args(x, w_gate_up, layout, M, N, K, STREAM_LAYOUT_MAX_ROWS)
    n = glu_split_count(N, K, M) if s is not None else 1
    if n > 1:
        slabs = torch.empty(n, M, N, dtype=torch.float32, device=x.device)
        s.ldy, s.y, s.epilogue, s.n_splits = N, _p(slabs), _lib.LIN_SLABS, n
        _run_stream(s)
        latent_check(_lib.latent_lib().slm_glu_slabs(_p(out), _p(slabs), M, half, n, out.stride(0), float(limit), float(alpha), float(shift),
                                                     _stream()), "slm_glu_slabs")
        return out
    if s is not None or streams_rows(x):
        a = s if s is not None else _linear_args(x, w_gate_up, M, N, K)
        a.ldx, a.ldw, a.ldy, a.y, a.epilogue = x.stride(0), K, out.stride(0), _p(out), _lib.LIN_GLU
        a.limit, a.glu_alpha, a.glu_shift = float(limit), float(alpha), float(shift)
        (_run_linear if s is None else _run_stream)(a)
    elif not (_tile_pays(M, N, K, True) and _gemm(x, w_gate_up, out, (float(limit), float(alpha), float(shift)), tickets=tickets)):
        gu = torch.mm(x, w_gate_up.t())
        clamped_glu(gu, out, limit, alpha, shift)
    return out


def clamped_glu(gate_up: torch.Tensor, out: torch.Tensor, limit: float, alpha: float = GLU_ALPHA,
                shift: float = GLU_SHIFT) -> None:
    M, N = gate_up.shape
    _need(out.shape == (M, N // 2) and gate_up.stride(1) == 1 and out.stride(1) == 1 and gate_up.dtype == out.dtype,
          "clamped_glu: gate_up [M, 2 n], out [M, n]")
    latent_check(_lib.latent_lib().slm_clamped_glu(_p(out), _p(gate_up), M, N // 2, gate_up.stride(0), out.stride(0), float(limit),
                                                   float(alpha), float(shift), _code(out), _stream()), "slm_clamped_glu")


def _heads_args(x: torch.Tensor, x_head: int, w: torch.Tensor, out: torch.Tensor, out_head: int) -> "_lib.LinearArgs":
    H, N, K = w.shape
    M = x.size(0)
    _need(x.dim() == 2 and out.dim() == 2 and out.size(0) == M and w.is_contiguous() and x.dtype == w.dtype == out.dtype and
          x.stride(1) == 1 and out.stride(1) == 1, "linear_heads: x [M, ..], w [heads, N, K], out [M, ..]")
    _need((H - 1) * x_head + K <= x.size(1) and (H - 1) * out_head + N <= out.size(1), "linear_heads: heads exceed the rows")
    a = _linear_args(x, w, M, N, K)
    a.ldx, a.ldw, a.ldy, a.y = x.stride(0), K, out.stride(0), _p(out)
    a.batch, a.x_batch, a.w_batch, a.y_batch = H, x_head, N * K, out_head
    a.epilogue = _lib.LIN_STORE
    return a


def _gated_heads(x, x_head, w, out, out_head, gate) -> "_lib.LinearArgs":
    a = _heads_args(x, x_head, w, out, out_head)
    if gate is not None:
        M, H = x.size(0), w.size(0)
        _need(gate.size(0) == M and gate.size(1) >= H and gate.stride(1) == 1 and gate.dtype == x.dtype, "linear_heads: gate")
        a.epilogue, a.gate, a.ld_gate = _lib.LIN_GATE, _p(gate), gate.stride(0)
    return a


def linear_heads(x: torch.Tensor, x_head: int, w: torch.Tensor, out: torch.Tensor, out_head: int,
                 gate: Optional[torch.Tensor] = None) -> None:
    """Per-head products: head h of `out` (columns from h * out_head) = columns from h * x_head of x times w[h]^T;
    w [heads, N, K].  gate [rows, >= heads]: the result is multiplied by sigmoid(gate[:, h])."""
    _run_linear(_gated_heads(x, x_head, w, out, out_head, gate))


def latent_append(proj: torch.Tensor, cache: torch.Tensor, q_abs: Optional[torch.Tensor], norm_weight: torch.Tensor,
                  cos_sin: torch.Tensor, positions: torch.Tensor, slots: torch.Tensor, *, heads: int, q_dim: int, q_rot: int,
                  rank: int, c_pad: int, off_c: int, off_r: int, eps: float, w_abs: Optional[torch.Tensor] = None) -> None:
    """Latent RMS norm + rotation -> cache rows; the queries' rotated part in place (and behind c_pad of q_abs).  With w_abs
    [heads, c_pad, K] the queries of q_abs's rows, absorbed, in front of it."""
    rows = proj.size(0)
    a = _lib.LatentAppendArgs()
    _need(proj.stride(1) == 1 and cache.dim() == 2 and cache.is_contiguous() and cache.dtype == proj.dtype, "latent_append: cache")
    _need(cos_sin.dtype == torch.float32 and cos_sin.is_contiguous() and norm_weight.dtype == torch.float32 and
          norm_weight.numel() == rank, "latent_append: fp32 tables")
    _i32(positions, rows, "positions")
    _i32(slots, rows, "slots")
    a.proj, a.cache, a.norm_weight, a.cos_sin = _p(proj), _p(cache), _p(norm_weight), _p(cos_sin)
    a.positions, a.slots, a.rows, a.ld_proj = _p(positions), _p(slots), rows, proj.stride(0)
    a.off_c, a.off_r, a.max_positions = off_c, off_r, cos_sin.size(0)
    a.heads, a.q_dim, a.q_rot, a.rank, a.rot = heads, q_dim, q_rot, rank, cos_sin.size(1)
    a.c_pad, a.r_pad, a.dtype, a.eps = c_pad, cache.size(1) - c_pad, _code(proj), float(eps)
    if q_abs is not None and q_abs.size(0):
        _need(q_abs.is_contiguous() and q_abs.shape[1:] == (heads, cache.size(1)) and q_abs.size(0) <= rows, "latent_append: q_abs")
        a.q_abs, a.abs_rows = _p(q_abs), q_abs.size(0)
    if w_abs is None or not a.abs_rows:
        latent_check(_lib.latent_lib().slm_latent_append(C.byref(a), _stream()), "slm_latent_append")
        return
    n = q_abs.size(0)
    x = _heads_args(proj[:n], q_dim + q_rot, w_abs, q_abs.view(n, -1), cache.size(1))
    latent_check(_lib.latent_lib().slm_latent_append_absorb(C.byref(a), C.byref(x), _stream()), "slm_latent_append_absorb")


def latent_attention(q_abs: torch.Tensor, cache: torch.Tensor, out: torch.Tensor, positions: torch.Tensor, q_cu: torch.Tensor,
                     block_table: torch.Tensor, block_cu: torch.Tensor, *, block_size: int, window: int, scale: float,
                     max_kv_len: int, n_splits: int = 0, generic: bool = False, values: Optional[tuple] = None) -> None:
    """out[row, head] = soft-max(q_abs . cache rows * scale) weighted latent over the row's visible positions.  values = (w, y, y_head, gate):
    then linear_heads() of it, w [heads, N, c_pad]; `out` is scratch."""
    rows, heads, R = q_abs.shape
    c_pad = out.size(2)
    _need(q_abs.is_contiguous() and out.is_contiguous() and out.shape[:2] == q_abs.shape[:2] and cache.size(1) == R and
          cache.is_contiguous() and cache.dtype == q_abs.dtype == out.dtype, "latent_attention: shapes")
    _i32(positions, rows, "positions")
    n = q_cu.numel() - 1
    _i32(q_cu, 2, "q_cu")
    _i32(block_cu, n + 1, "block_cu")
    _i32(block_table, 1, "block_table")
    a = _lib.LatentAttnArgs()
    a.q_abs, a.cache, a.out, a.positions = _p(q_abs), _p(cache), _p(out), _p(positions)
    a.q_cu, a.block_table, a.block_cu = _p(q_cu), _p(block_table), _p(block_cu)
    a.rows, a.batch, a.heads, a.c_pad, a.r_pad = rows, n, heads, c_pad, R - c_pad
    a.block_size, a.window, a.max_kv_len, a.n_splits = block_size, int(window), int(max_kv_len), int(n_splits)
    a.scale, a.dtype, a.generic = float(scale), _code(q_abs), int(generic)
    L = _lib.latent_lib()
    need = L.slm_latent_attn_workspace_bytes(C.byref(a))
    if need:
        ws = reserve_workspace(need, q_abs.device)
        a.workspace, a.workspace_bytes = ws.data_ptr(), ws.numel()
    if values is None:
        latent_check(L.slm_latent_attn(C.byref(a), _stream()), "slm_latent_attn")
        return
    w, y, y_head, gate = values
    v = _gated_heads(out.view(rows, -1), c_pad, w, y, y_head, gate)
    latent_check(L.slm_latent_attn_values(C.byref(a), C.byref(v), _stream()), "slm_latent_attn_values")


def latent_gather(cache: torch.Tensor, slots: torch.Tensor) -> torch.Tensor:
    """cache rows of `slots`, contiguous."""
    n = slots.numel()
    _i32(slots, n, "slots")
    out = torch.empty(n, cache.size(1), dtype=cache.dtype, device=cache.device)
    latent_check(_lib.latent_lib().slm_latent_gather(_p(out), _p(cache), _p(slots), n, cache.size(1) * cache.element_size(), _stream()),
                 "slm_latent_gather")
    return out


def latent_prefill_supported(q_dim: int, r_pad: int, v_pad: int) -> bool:
    return bool(_lib.latent_lib().slm_latent_prefill_supported(q_dim, r_pad, v_pad))


def latent_prefill(proj: torch.Tensor, ctx: torch.Tensor, kv: torch.Tensor, out: torch.Tensor, tiles: torch.Tensor, *, heads: int,
                   q_dim: int, c_pad: int, v_pad: int, gate_off: int, window: int, scale: float) -> None:
    """Causal, windowed attention of the portions' query rows over their expanded context; see slm_latent.h."""
    r_pad = ctx.size(1) - c_pad
    _need(proj.dtype == ctx.dtype == kv.dtype == out.dtype == torch.bfloat16, "latent_prefill: bfloat16")
    _need(ctx.is_contiguous() and kv.is_contiguous() and kv.shape == (ctx.size(0), heads * (q_dim + v_pad)), "latent_prefill: context")
    _need(tiles.dim() == 2 and tiles.size(1) == 6, "latent_prefill: tiles")
    _i32(tiles, tiles.numel(), "tiles")
    a = _lib.LatentPrefillArgs()
    a.q, a.ctx, a.kv, a.gate, a.out, a.tiles = _p(proj), _p(ctx), _p(kv), _p(proj), _p(out), _p(tiles)
    a.ld_q, a.ld_out, a.n_rows, a.n_ctx, a.gate_off = proj.stride(0), out.stride(0), proj.size(0), ctx.size(0), gate_off
    a.n_tiles, a.heads, a.q_dim, a.c_pad, a.r_pad, a.v_pad = tiles.size(0), heads, q_dim, c_pad, r_pad, v_pad
    a.window, a.scale = int(window), float(scale)
    latent_check(_lib.latent_lib().slm_latent_prefill(C.byref(a), _stream()), "slm_latent_prefill")
