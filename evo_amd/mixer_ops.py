"""The mixer libraries (include/evo_mi355x.h, last section) as methods of the op set: kernels of models with an fp32 residual stream, softmax
attention, decayed linear attention, latent attention, gated linear recurrence.  Storage is bf16 or fp32, taken from the tensors; the
arithmetic is fp32."""
from __future__ import annotations

import functools
import inspect
from dataclasses import dataclass
from typing import List, Optional, Sequence, Tuple

import torch

LC = 64                                     # tokens per chunk of the linear-attention kernel
ACTIVATIONS = {"silu": 1, "gelu_tanh": 2, "relu2": 3}
_DECODE_COLUMNS = (1, 2, 3, 4, 6, 8, 12, 16)   # latent widths, in units of 32, the matrix-core decode kernel is built for


def takes(method, keyword: str) -> bool:
    """Whether a method has the keyword, one of those that programs' own versions of it -- a subclass's, an op set's, a wrapper's -- need not have: they are called as before then."""
    f = getattr(method, "__func__", method)
    code = getattr(f, "__code__", None)
    if code is None or not (keyword in code.co_varnames[:code.co_argcount + code.co_kwonlyargcount] or code.co_flags & inspect.CO_VARKEYWORDS):
        return False
    return not hasattr(f, "__wrapped__") or takes(f.__wrapped__, keyword)


@dataclass
class TokenBatch:
    """Tokens of several sequences, packed one after the other.  `lens` / `past`: new and earlier tokens per sequence (host); `cu` [B + 1]
    int32, `seq` [M] int32, `pos` [M] int64, `resume` [B] int32 (sequences that go on from a cached state): on the device.  A decode step
    (`decode`: one token per cache row, positions known to the device only) has no host lengths."""
    cu: Optional[torch.Tensor]
    seq: Optional[torch.Tensor]
    pos: torch.Tensor
    resume: Optional[torch.Tensor]
    lens: List[int]
    past: List[int]
    decode: bool = False

    @staticmethod
    def of_prompts(lens: Sequence[int], past: Sequence[int], device, ops=None) -> "TokenBatch":
        lens, past = list(lens), list(past)
        B, M, device = len(lens), sum(lens), torch.device(device)
        if device.type == "cuda" and hasattr(ops, "token_batch") and 0 < B <= ops.MAX_PUT:
            cu, seq, pos, resume = ops.token_batch(lens, past, device)
            return TokenBatch(cu, seq, pos, resume, lens, past)
        host = torch.tensor([[0] + lens, [0] + past], dtype=torch.int64).to(device)       # (one copy; the rest is made on the device)
        cu = host[0].cumsum(0)
        seq = torch.repeat_interleave(torch.arange(B, device=device), host[0, 1:], output_size=M)
        pos = torch.arange(M, device=device) + (host[1, 1:] - cu[:-1])[seq]
        resume = (host[1, 1:] > 0).to(torch.int32) if any(past) else None
        return TokenBatch(cu.to(torch.int32), seq.to(torch.int32), pos, resume, lens, past)

    @staticmethod
    def of_decode(pos: torch.Tensor) -> "TokenBatch":
        return TokenBatch(None, None, pos, None, [], [], decode=True)


class Stream:
    """The fp32 residual stream x [M, D] of one pass, its storage-type copy, and at most one sublayer output that has not been added yet: for one
    row of bf16 the next layer's launch adds it (ops.postnorm_linear / postnorm_gate), the last of a pass the final norm's (ops.closing_final),
    otherwise it is added before the next layer.

    The norm of a sublayer's output y comes before the addition, x <- x + norm(y), or -- with `alpha` -- behind it, x <- norm(alpha x + y);
    norm(t) = t / rms(t) * (w_offset + w)."""

    def __init__(self, ops, ids: torch.Tensor, weight: torch.Tensor, scale: float, eps: float, w_offset: float, alpha: Optional[float] = None,
                 ids_known: bool = False, later: Optional[list] = None):
        self.ops, self.eps, self.w_offset, self.alpha = ops, eps, w_offset, alpha
        more = {"validate": False} if ids_known else {} if later is None else {"later": later}
        self.x, self.xb = ops.embed_stream(ids, weight, scale, **{k: v for k, v in more.items() if takes(ops.embed_stream, k)})
        self.open = None                                         # (y, w): still to be added
        self.spare = None                                        # the buffer the next such launch writes x to
        self.behind = False                                      # xb does not hold the current x

    def product(self, a: torch.Tensor, w: torch.Tensor) -> torch.Tensor:
        """a @ w^T of a sublayer, for `add` -- or its parts over K [parts, M, N], where the layer is summed in parts: the closing norm adds them."""
        parts = self.ops.layer_parts(a, w) if self.xb.dtype == torch.bfloat16 and w.shape[0] <= 4096 and hasattr(self.ops, "layer_parts") else None
        return self.ops.linear(a, w) if parts is None else parts

    def add(self, y: torch.Tensor, w: torch.Tensor) -> None:
        self.flush()
        self.open = (y, w)

    def _next_adds(self) -> bool:
        """Whether the next layer's launch adds the open output."""
        return self.open is not None and self.open[0].dim() == 2 and self.ops.fuse_postnorm_ok(self.open[0])

    def flush(self) -> None:
        if self.open is not None:
            y, w = self.open
            self.open = None
            if y.dim() == 3:                                     # (parts)
                self.ops.closing_parts_(self.x, self.xb, y, w, self.alpha, self.eps, self.w_offset)
                self.behind = False
                return
            if self.xb.dtype == self.x.dtype:
                self.xb = self.x
            if self.alpha is None:
                self.ops.postnorm_residual_(self.x, self.xb, y, w, self.eps, self.w_offset)
            else:
                self.ops.sum_norm_(self.x, self.xb, y, w, self.alpha, self.eps, self.w_offset)
            self.behind = False

    def input(self) -> torch.Tensor:
        """The sublayer input in the storage type."""
        self.flush()
        if self.behind:
            self.xb = self.x.to(self.xb.dtype)
            self.behind = False
        return self.xb

    def _swap(self):
        """(y, norm weight, x, where the new x goes) for a launch that adds the open output."""
        y, w = self.open
        self.open = None
        old, new = self.x, torch.empty_like(self.x) if self.spare is None else self.spare
        self.x, self.spare, self.behind = new, old, True
        return y, w, old, new

    def linear(self, w: torch.Tensor, act: Optional[str] = None) -> torch.Tensor:
        if not self._next_adds():
            return self.ops.linear(self.input(), w) if act is None else self.ops.linear_act(self.input(), w, act, w.shape[0])
        return self.ops.postnorm_linear(*self._swap(), w, self.eps, self.w_offset, alpha=self.alpha, act=act)

    def gate(self, w12: torch.Tensor, grouped: bool, act: str) -> torch.Tensor:
        if not self._next_adds():
            return self.ops.mlp_gate(self.input(), None if grouped else w12, w12g=w12 if grouped else None, act=act)
        return self.ops.postnorm_gate(*self._swap(), w12, grouped, act, self.eps, self.w_offset, alpha=self.alpha)

    def final(self, w: torch.Tensor) -> torch.Tensor:
        """The final norm; nothing reads the stream behind it."""
        if self.open is not None and hasattr(self.ops, "closing_final_ok") and self.ops.closing_final_ok(*self.open, self.x, w):
            (y, g), self.open = self.open, None
            return self.ops.closing_final(self.x, y, g, w, self.alpha, self.eps, self.w_offset)
        self.flush()
        return self.ops.rmsnorm_stream(self.x, w, self.eps, self.w_offset)


class MixerOps:
    """Mixed into HipOps (needs its `lib`, `_t`, `validate_ids`)."""

    mixer_mfma = True          # False: the any-size kernels in place of the matrix-core ones (tests, measurements)

    @staticmethod
    def _store(*tensors) -> int:
        """Checks one storage type on the device; 1 for fp32, 0 for bf16."""
        dt = tensors[0].dtype
        for t in tensors:
            if not t.is_cuda:
                raise RuntimeError(f"tensor is on {t.device}; the HIP path has no CPU fallback")
            if t.dtype != dt or dt not in (torch.float32, torch.bfloat16):
                raise RuntimeError(f"expected one storage type, fp32 or bf16, got {t.dtype} beside {dt}")
            if t.stride(-1) != 1:
                raise RuntimeError("tensor rows must be dense")
        return int(dt == torch.float32)

    @staticmethod
    def _ix(t: Optional[torch.Tensor], dtype, n: int, what: str) -> Optional[int]:
        if t is None:
            return None
        if not t.is_cuda or t.dtype != dtype or not t.is_contiguous() or t.numel() < n:
            raise RuntimeError(f"{what}: need a contiguous device {dtype} tensor of at least {n} entries")
        return t.data_ptr()

    @staticmethod
    def _dense(t: torch.Tensor, shape, what: str):
        if tuple(t.shape) != tuple(shape) or not t.is_contiguous():
            raise RuntimeError(f"{what}: need a contiguous tensor of shape {tuple(shape)}, got {tuple(t.shape)}")

    def _call(self, name: str, *args):
        from .ops import _check, _stream
        with self._t(name[4:]):
            _check(getattr(self.lib, name)(*args, _stream()), name)

    # ---- residual stream ------------------------------------------------------------------------------------------------
    def embed_stream(self, ids: torch.Tensor, weight: torch.Tensor, scale: float, validate: bool = True, later: Optional[list] = None) -> Tuple[torch.Tensor, torch.Tensor]:
        """(x fp32 [M, D] = scale * weight[ids], the same in the storage type: x itself for fp32).  `validate=False`: the caller has checked the ids; `later`: it calls
        check_ids."""
        ids = ids.reshape(-1).to(torch.int64).contiguous()
        f32 = self._store(weight)
        V, D = weight.shape
        self._dense(weight, (V, D), "embedding table")
        x = torch.empty(ids.numel(), D, dtype=torch.float32, device=weight.device)
        xb = x if f32 else torch.empty(ids.numel(), D, dtype=torch.bfloat16, device=weight.device)
        flag = None if torch.cuda.is_current_stream_capturing() or not (self.validate_ids and validate) else \
            torch.zeros(1, dtype=torch.int32, device=weight.device)
        self._call("evo_embed_stream", self._ix(ids, torch.int64, ids.numel(), "ids"), weight.data_ptr(), x.data_ptr(), None if f32 else xb.data_ptr(),
                   ids.numel(), D, V, float(scale), None if flag is None else flag.data_ptr(), f32)
        if flag is not None:
            self.raise_bad_ids(flag, V, later)
        return x, xb

    def _closing_args(self, x, xb, y, w):
        f32 = self._store(y, w, xb)
        M, D = y.shape
        self._dense(y, (M, D), "y"), self._dense(x, (M, D), "x"), self._dense(xb, (M, D), "xb"), self._dense(w, (D,), "w")
        assert x.dtype == torch.float32 and (not f32 or xb is x)
        return y.data_ptr(), w.data_ptr(), x.data_ptr(), None if f32 else xb.data_ptr(), M, D

    def postnorm_residual_(self, x: torch.Tensor, xb: torch.Tensor, y: torch.Tensor, w: torch.Tensor, eps: float, w_offset: float) -> None:
        """x += rms_norm(y) * (w_offset + w) in place; xb (the storage-type copy of x, or x itself) follows."""
        self._call("evo_postnorm_residual", *self._closing_args(x, xb, y, w), float(eps), float(w_offset), int(y.dtype == torch.float32))

    def sum_norm_(self, x: torch.Tensor, xb: torch.Tensor, y: torch.Tensor, w: torch.Tensor, alpha: float, eps: float, w_offset: float) -> None:
        """x = rms_norm(alpha x + y) * (w_offset + w) in place; xb follows."""
        self._call("evo_sum_norm", *self._closing_args(x, xb, y, w), float(alpha), float(eps), float(w_offset), int(y.dtype == torch.float32))

    def closing_parts_(self, x: torch.Tensor, xb: torch.Tensor, y: torch.Tensor, w: torch.Tensor, alpha: Optional[float], eps: float, w_offset: float) -> None:
        """sum_norm_ (`alpha` given) or postnorm_residual_ on the parts y [parts, M, D] of a dense layer (HipOps.linear_parts)."""
        n, M, D = y.shape
        assert y.dtype == torch.float32 and y.is_contiguous() and x.dtype == torch.float32 and self._store(xb, w) == 0
        self._dense(x, (M, D), "x"), self._dense(xb, (M, D), "xb"), self._dense(w, (D,), "w")
        if (x.data_ptr() | xb.data_ptr() | w.data_ptr()) % 16:   # (a norm weight cut out of a larger tensor)
            total = y[0]
            for part in y[1:]:
                total = total + part
            total = total.to(xb.dtype)
            return self.postnorm_residual_(x, xb, total, w, eps, w_offset) if alpha is None else self.sum_norm_(x, xb, total, w, alpha, eps, w_offset)
        self._call("evo_closing_parts", y.data_ptr(), n, w.data_ptr(), x.data_ptr(), xb.data_ptr(), M, D, int(alpha is not None), float(alpha or 0.0), float(eps),
                   float(w_offset))

    fuse_postnorm = True       # False: every closing norm as its own launch (tests, measurements)

    def fuse_postnorm_ok(self, y: torch.Tensor) -> bool:
        """One row: every workgroup of the next layer builds it for itself.  With more the norm's own launch is ahead (us at D = 4,096, fused : norm and layer.
        16,384 columns 24.8 : 26.9, at 2 rows 27.1 : 26.5, 4 rows 35.6 : 24.3; the gated layer of 11,008 31.7 : 33, 34.5 : 33.2, 43.2 : 30.7)."""
        M, D = y.shape
        return self.fuse_postnorm and y.dtype == torch.bfloat16 and M == 1 and D % 8 == 0 and D <= 8192

    def _postnorm_args(self, y, g, x, x_out, w):
        M, K = y.shape
        assert self._store(y, g, w) == 0
        for t, shape, what in ((y, (M, K), "y"), (g, (K,), "g"), (x, (M, K), "x"), (x_out, (M, K), "x_out"), (w, (w.shape[0], K), "w")):
            self._dense(t, shape, what)
        assert x.dtype == torch.float32 and x_out.dtype == torch.float32 and x.data_ptr() != x_out.data_ptr()
        return y.data_ptr(), g.data_ptr(), x.data_ptr(), x_out.data_ptr(), w.data_ptr()

    def postnorm_linear(self, y, g, x, x_out, w, eps: float, w_offset: float, alpha: Optional[float] = None, act: Optional[str] = None) -> torch.Tensor:
        """x_out = x + norm(y) * (w_offset + g), or norm(alpha x + y) * (w_offset + g); -> act(x_out @ w^T), one launch for up to four rows."""
        M, K = y.shape
        z = torch.empty(M, w.shape[0], dtype=y.dtype, device=y.device)
        fused = act in (None, "relu2")
        self._call("evo_postnorm_linear_small_m_bf16", *self._postnorm_args(y, g, x, x_out, w), z.data_ptr(), M, w.shape[0], K, float(alpha or 0.0),
                   int(alpha is not None), float(eps), float(w_offset), ACTIVATIONS[act] if fused and act else 0)
        if not fused:
            self.act_cols_(z, z.shape[1], act)
        return z

    def postnorm_gate(self, y, g, x, x_out, w12, grouped: bool, act: str, eps: float, w_offset: float, alpha: Optional[float] = None) -> torch.Tensor:
        """x_out as above; -> the gated MLP's first half on it, in the same launch."""
        M, K = y.shape
        I = w12.shape[0] // 2
        a = torch.empty(M, I, dtype=y.dtype, device=y.device)
        self._call("evo_postnorm_mlp_gate_small_m_bf16", *self._postnorm_args(y, g, x, x_out, w12), a.data_ptr(), M, I, K, float(alpha or 0.0),
                   int(alpha is not None), float(eps), float(w_offset), int(grouped), {"gelu": 0, "silu": 1}[act])
        return a

    def rmsnorm_stream(self, x: torch.Tensor, w: torch.Tensor, eps: float, w_offset: float) -> torch.Tensor:
        f32 = self._store(w)
        M, D = x.shape
        self._dense(x, (M, D), "x"), self._dense(w, (D,), "w")
        assert x.dtype == torch.float32 and x.is_cuda
        out = torch.empty(M, D, dtype=w.dtype, device=x.device)
        self._call("evo_rmsnorm_stream", x.data_ptr(), w.data_ptr(), out.data_ptr(), M, D, float(eps), float(w_offset), f32)
        return out

    def closing_final_ok(self, y: torch.Tensor, w: torch.Tensor, x: torch.Tensor, wf: torch.Tensor) -> bool:
        """Rows that closing_final's kernel holds in registers."""
        D = x.shape[1]
        return (D in (2048, 4096, 8192) and (y.dim() == 2 or D == 4096) and w.dtype == wf.dtype and w.is_contiguous() and wf.is_contiguous()
                and (y.data_ptr() | w.data_ptr() | x.data_ptr() | wf.data_ptr()) % 16 == 0)

    def closing_final(self, x: torch.Tensor, y: torch.Tensor, w: torch.Tensor, wf: torch.Tensor, alpha: Optional[float], eps: float, w_offset: float) -> torch.Tensor:
        """rmsnorm_stream(x', wf) of the x' that postnorm_residual_, sum_norm_ or closing_parts_ (y of three dimensions) would store; x itself stays."""
        parts = y.shape[0] if y.dim() == 3 else 0
        f32 = self._store(w, wf) if parts else self._store(y, w, wf)
        M, D = x.shape
        self._dense(y, ((parts,) if parts else ()) + (M, D), "y"), self._dense(x, (M, D), "x"), self._dense(w, (D,), "w"), self._dense(wf, (D,), "wf")
        assert x.dtype == torch.float32 and x.is_cuda and (not parts or (y.dtype == torch.float32 and y.is_cuda))
        out = torch.empty(M, D, dtype=w.dtype, device=x.device)
        self._call("evo_closing_final", y.data_ptr(), parts, w.data_ptr(), x.data_ptr(), wf.data_ptr(), out.data_ptr(), M, D, int(alpha is not None), float(alpha or 0.0),
                   float(eps), float(w_offset), f32)
        return out

    def gated_norm(self, o: torch.Tensor, g: torch.Tensor, w: torch.Tensor, eps: float) -> torch.Tensor:
        """rms_norm(o) * w * sigmoid(g); g [M, D] may be a column range of a wider matrix."""
        f32 = self._store(o, g, w)
        M, D = o.shape
        self._dense(o, (M, D), "o"), self._dense(w, (D,), "w")
        assert tuple(g.shape) == (M, D)
        out = torch.empty_like(o)
        self._call("evo_gated_norm", o.data_ptr(), g.data_ptr(), g.stride(0), w.data_ptr(), out.data_ptr(), M, D, float(eps), f32)
        return out

    def silu_gate(self, z: torch.Tensor) -> torch.Tensor:
        f32 = self._store(z)
        M, I2 = z.shape
        self._dense(z, (M, I2), "z")
        a = torch.empty(M, I2 // 2, dtype=z.dtype, device=z.device)
        self._call("evo_silu_gate", z.data_ptr(), a.data_ptr(), M, I2 // 2, f32)
        return a

    def linear_act(self, x: torch.Tensor, w: torch.Tensor, act: str, act_cols: int, b: Optional[torch.Tensor] = None) -> torch.Tensor:
        """x @ w^T (+ b) with an activation on the first `act_cols` columns; in the dense layer's epilogue for prefill-sized
        batches and, the square of relu on all columns, for decode-sized ones."""
        M, K = x.shape
        N = w.shape[0]
        if act == "relu2" and act_cols == N and self._use_small_m(x, w):
            return self._linear_small_m(x, w, b, None, act=ACTIVATIONS[act])
        if (self._take_mfma(False) and self.mfma_linear_ok(x, w) and not self._use_small_m(x, w) and act_cols % 256 == 0 and K >= 128
                and M * K * 2 < 0xffffffff and N * K * 2 < 0xffffffff):
            r = self._tail_rows(x, w)
            y = torch.empty(M, N, dtype=x.dtype, device=x.device)
            with self._t("linear_act_mfma_bf16"):
                self._dense_layer(0, x, w, y, M - r, N, K, act=ACTIVATIONS[act], b=b, act_cols=act_cols)
            if r:
                self._linear_small_m(x[M - r:], w, b, None, out=y[M - r:])
                self.act_cols_(y[M - r:], act_cols, act)
            return y
        y = self.linear(x, w, b)
        self.act_cols_(y, act_cols, act)
        return y

    def act_cols_(self, z: torch.Tensor, n: int, act: str) -> None:
        """z[:, :n] = act(z[:, :n]) in place"""
        f32 = self._store(z)
        assert z.dim() == 2 and z.shape[1] >= n
        self._call("evo_act_cols", z.data_ptr(), z.stride(0), z.shape[0], n, ACTIVATIONS[act], f32)

    # ---- decayed linear attention ---------------------------------------------------------------------------------------
    def lightning(self, z: torch.Tensor, heads: int, dk: int, dv: int, decay: torch.Tensor, log2_decay: torch.Tensor, batch: TokenBatch,
                  state: Optional[torch.Tensor] = None, seg_len: Optional[int] = None) -> torch.Tensor:
        """z [M, >= heads (2 dk + dv)] = [q | k | v | ..] -> o [M, heads dv]: after their SiLU for prompts (linear_act), before it for a decode
        step (the step applies it).  `state` [rows, heads, dk, dv] fp32 follows."""
        f32 = self._store(z)
        M = z.shape[0]
        o = torch.empty(M, heads * dv, dtype=z.dtype, device=z.device)
        assert z.shape[1] >= heads * (2 * dk + dv) and decay.numel() == heads and log2_decay.numel() == heads
        B = M if batch.decode else len(batch.lens)
        if state is not None:
            self._dense(state, (state.shape[0], heads, dk, dv), "state")
            assert state.dtype == torch.float32 and state.is_cuda and state.shape[0] >= B
        sp = None if state is None else state.data_ptr()
        dp = self._ix(decay, torch.float32, heads, "decay")
        if batch.decode:
            self._call("evo_lightning_recurrent", z.data_ptr(), z.stride(0), o.data_ptr(), sp, dp, None, None, B, heads, dk, dv, 1, f32)
            return o
        assert sum(batch.lens) == M
        cu, resume = self._ix(batch.cu, torch.int32, B + 1, "cu"), self._ix(batch.resume, torch.int32, B, "resume")
        if f32 or dk > 128 or not self.mixer_mfma:
            self._call("evo_lightning_recurrent", z.data_ptr(), z.stride(0), o.data_ptr(), sp, dp, cu, resume, B, heads, dk, dv, 0, f32)
            return o
        L = max(batch.lens)
        seg_len = seg_len or self.lightning_segment(tuple(sorted(batch.lens)), heads * ((dv + 127) // 128), dk * min(dv, 128))
        seg = torch.empty(self.segment_slots(B, M, seg_len), heads, dk, dv, dtype=torch.float32, device=z.device) if L > seg_len else None
        self._call("evo_lightning_chunk_bf16", z.data_ptr(), z.stride(0), o.data_ptr(), sp, None if seg is None else seg.data_ptr(),
                   self._ix(log2_decay, torch.float32, heads, "log2_decay"), cu, resume, B, heads, dk, dv, L, seg_len)
        return o

    @staticmethod
    @functools.lru_cache(maxsize=64)
    def lightning_segment(lens: Tuple[int, ...], columns: int, state: int, cus: int = 256) -> int:
        """Tokens per segment (whole chunks): the least of what the launches cost, for `columns` (head, value tile) pairs a sequence and `state` elements of one such tile.
        A workgroup a CU takes 5.4 us a chunk; cut sequences need another pass for their segments' states (2.2 us a chunk) and each of those crosses memory four
        times.  (us at 32 heads of 128 x 128, the rule before, segments for a workgroup per CU -> this one.  6 sequences of 1,459 to 2,500 tokens: 295 in
        segments of 1,280, 214 uncut; 5,000 and 300: 148 -> 101 in segments of 768; 3,000 and four times 300: 177 -> 102; 1,500 and three times 100: 98 -> 57;
        4,000 twice 133 as before, 311 uncut.)"""
        def us(seg, span, busy, n_cut):
            return 6.0 + 5.3 * span + (3.0 + 2.2 * busy + n_cut * state * 16 / 4.5e6 if n_cut else 0.0)
        return MixerOps.cheapest_segment(lens, columns, us, cus, 0.7 if state <= 4096 else 1.0)

    @staticmethod
    def segment_slots(B: int, rows: int, seg_len: int) -> int:
        """Workspace slots of the segments of cut sequences (csrc/mixers_common.h segment_slot): by the rows, however many sequences share the pass."""
        whole = rows // seg_len
        return whole + min(B, whole)

    @staticmethod
    def cheapest_segment(lens: Tuple[int, ...], columns: int, us, cus: int, share: float = 1.0) -> int:
        """The segment length, whole chunks of a share of the longest sequence, of least us(segment, chunks of the launch's end, chunks of cut sequences at the most of a
        CU where two workgroups share one, workgroups of cut sequences).  Several rounds of workgroups end half a workgroup late, and each costs 1.3 chunks before its
        first; `share`: what a chunk costs where small workgroups share a CU (6 sequences of 1,459 to 2,500 tokens: 32 heads of 64 x 64 uncut 129, 1,280 115, 768 96; 16 blocks
        of 64 channels 896 104, 1,280 101, 256 to 512 71).  Few columns: shares down to a workgroup per CU (us, 32 shares at the most -> as many as CUs.  Decayed linear attention, 131,072 tokens at two heads
        of 128 x 128 431 -> 164, one of 64 x 64 277 -> 113; 32,000 at four heads 130 -> 94; gated recurrence, 131,072 tokens in two blocks of 256 526 -> 310)."""
        longest = max(lens)
        chunks = sum((n + LC - 1) // LC for n in lens) * columns / cus
        best = None
        for seg in sorted({max(4 * LC, (longest + n * LC - 1) // (n * LC) * LC) for n in range(1, 33 + cus // (columns * len(lens)))}, reverse=True):
            n_wg = sum((n + seg - 1) // seg for n in lens) * columns
            cut = [n for n in lens if n > seg]
            top = min(seg, (longest + LC - 1) // LC * LC) / LC
            t = us(seg, top if n_wg <= cus else max(top, share * (chunks + 1.3 * n_wg / cus + 0.55 * top)), max(top, sum((n + LC - 1) // LC for n in cut) * columns / cus),
                   sum((n + seg - 1) // seg for n in cut) * columns)
            if best is None or t < best[0]:
                best = (t, seg)
        return best[1]

    # ---- latent attention -----------------------------------------------------------------------------------------------
    @staticmethod
    def latent_row(R: int, dr: int) -> int:
        """Elements of a cached row [latent | rotated key | zeros]: whole 32-wide steps, one or two more than a latent width the matrix-core
        decode kernel is built for, where the rotated part allows it."""
        need = (R + dr + 31) // 32
        fit = [max(need, c + 1) for c in _DECODE_COLUMNS if c * 32 >= R and need <= c + 2]
        return 32 * (min(fit) if fit else need)

    def latent_prep(self, qd: torch.Tensor, heads: int, dn: int, dr: int, R: int, norm_w: torch.Tensor, inv_freq: torch.Tensor, eps: float,
                    batch: TokenBatch, cache: Optional[torch.Tensor], want_kv: bool):
        """Rotates qd's query part in place; -> (c [M, R], kr [M, dr]) with `want_kv`; appends to the ring cache [rows, ring, row]."""
        f32 = self._store(qd, norm_w) if cache is None else self._store(qd, norm_w, cache)
        M = qd.shape[0]
        c = torch.empty(M, R, dtype=qd.dtype, device=qd.device) if want_kv else None
        kr = torch.empty(M, dr, dtype=qd.dtype, device=qd.device) if want_kv else None
        assert qd.shape[1] >= heads * (dn + dr) + R + dr and norm_w.numel() == R
        B = M if batch.decode else len(batch.lens)
        ring = rs = 0
        if cache is not None:
            rows, ring, rs = cache.shape
            self._dense(cache, (rows, ring, rs), "latent cache")
            assert rows >= B
        self._call("evo_latent_prep", qd.data_ptr(), qd.stride(0), None if c is None else c.data_ptr(), None if kr is None else kr.data_ptr(),
                   None if cache is None else cache.data_ptr(), norm_w.data_ptr(), self._ix(inv_freq, torch.float32, 0, "inv_freq"),
                   self._ix(batch.pos, torch.int64, M, "pos"), self._ix(batch.seq, torch.int32, M, "seq"),
                   self._ix(batch.cu, torch.int32, B + 1, "cu"), M, heads, dn, dr, R, 2 * inv_freq.numel(), ring, rs, float(eps), f32)
        return c, kr

    def window_attention(self, qd: torch.Tensor, kv: torch.Tensor, kr: torch.Tensor, heads: int, dn: int, dr: int, dv: int, window: int,
                         scale: float, sink: torch.Tensor, cu_q: torch.Tensor, cu_k: torch.Tensor, max_q: int) -> torch.Tensor:
        """qd rows start with the heads' [dn | dr] queries; kv rows = [keys (heads dn) | values (heads dv)]; kr [Mk, dr] -> [Mq, heads dv]."""
        nk = heads * dn
        assert kv.shape[1] == heads * (dn + dv) and kr.shape == (kv.shape[0], dr) and kr.is_contiguous() and kr.dtype == qd.dtype
        assert sink.numel() == heads and qd.shape[1] >= heads * (dn + dr)
        return self._window_attn(qd, kv[:, :nk], kv[:, nk:], kr, sink, heads, heads, 1, dn, dr, dv, window, 0, scale, 0.0, 1.0, 0.0, cu_q, cu_k, max_q)

    def _window_attn(self, q, kn, v, kr, sink, heads, kv_heads, maps, dn, dr, dv, window, keep, scale, lam, gain, eps, cu_q, cu_k, max_q):
        f32 = self._store(q, kn, v)
        B = cu_q.numel() - 1
        assert cu_k.numel() == B + 1 and kn.stride(0) == v.stride(0)
        o = torch.empty(q.shape[0], heads * dv, dtype=q.dtype, device=q.device)
        self._call("evo_window_attn", q.data_ptr(), q.stride(0), kn.data_ptr(), v.data_ptr(), kn.stride(0), None if kr is None else kr.data_ptr(),
                   o.data_ptr(), self._ix(cu_q, torch.int32, B + 1, "cu_q"), self._ix(cu_k, torch.int32, B + 1, "cu_k"),
                   self._ix(sink, torch.float32, heads, "sink"), B, heads, kv_heads, maps, dn, dr, dv, int(min(window, 1 << 29)), int(keep), int(max_q),
                   float(scale), float(lam), float(gain), float(eps), f32, int(self.mixer_mfma))
        return o

    @staticmethod
    def latent_split(B: int, heads: int, tiles: int, cus: int = 256):
        """(parts of the window, heads per workgroup) of the decode kernel: a workgroup per CU.  16 heads per workgroup get through a tile
        quicker, 32 read it once for twice the heads: the former while that leaves a workgroup at most four tiles."""
        def parts(groups):
            return max(1, min(tiles, cus // (B * groups), 32))
        n = parts((heads + 15) // 16)
        if (tiles + n - 1) // n <= 4 or heads <= 16:
            return n, 16
        return parts((heads + 31) // 32), 32

    @staticmethod
    def latent_prep_fits(qd: torch.Tensor, cache: torch.Tensor, norm_w: torch.Tensor, inv_freq: torch.Tensor, heads: int, dn: int, dr: int, R: int) -> bool:
        """What latent_decode's `prep` takes, rows of whole 16-byte pieces, and where it is ahead: not where many workgroups split the columns, whose angles are all made by the
        first of them (us, in two launches : in one.  64 heads, R = 512: 16 / 24 / 64 sequences 11.7 : 11.2, 14.3 : 15.4, 22.7 : 29.3; 16 heads at 100 14.5 : 15.6; 128
        heads, R = 256, at 100 40.8 : 35.9)."""
        ahead = R <= 256 or heads * ((qd.shape[0] + 3) // 4) * ((R + 255) // 256) <= 512
        return (ahead and qd.stride(0) % 8 == 0 and heads * (dn + dr) % 8 == 0 and R % 8 == 0 and cache.shape[2] % 8 == 0 and 0 < 2 * inv_freq.numel() <= dr and dn <= 4096
                and norm_w.dtype == qd.dtype and (qd.data_ptr() | cache.data_ptr() | norm_w.data_ptr()) % 16 == 0)

    def latent_decode(self, qd: torch.Tensor, cache: torch.Tensor, pos: torch.Tensor, wuk: torch.Tensor, wuv: torch.Tensor, sink: torch.Tensor,
                      heads: int, dn: int, dr: int, dv: int, R: int, window: int, scale: float, n_split: Optional[int] = None, prep=None) -> torch.Tensor:
        """One token per cache row against the ring cache -> [B, heads dv].  The rows are already appended by latent_prep or, with `prep` = (norm weight, inv_freq, eps),
        are appended here, by the first launch; qd's queries then stay as they are."""
        f32 = self._store(qd, cache, wuk, wuv)
        B = qd.shape[0]
        rows, ring, rs = cache.shape
        self._dense(cache, (rows, ring, rs), "latent cache")
        self._dense(wuk, (heads * dn, R), "wuk"), self._dense(wuv, (heads * dv, R), "wuv")
        assert rows >= B and qd.shape[1] >= heads * (dn + dr) and window <= ring and sink.numel() == heads
        q = torch.empty(B, heads, rs, dtype=qd.dtype, device=qd.device)
        if prep is None:
            self._call("evo_latent_absorb", qd.data_ptr(), qd.stride(0), wuk.data_ptr(), q.data_ptr(), B, heads, dn, dr, R, rs, f32)
        else:
            norm_w, inv_freq, eps = prep
            assert norm_w.dtype == qd.dtype and norm_w.is_cuda and norm_w.is_contiguous() and norm_w.numel() == R and qd.shape[1] >= heads * (dn + dr) + R + dr
            self._call("evo_latent_prep_absorb", qd.data_ptr(), qd.stride(0), wuk.data_ptr(), q.data_ptr(), cache.data_ptr(), norm_w.data_ptr(),
                       self._ix(inv_freq, torch.float32, 0, "inv_freq"), self._ix(pos, torch.int64, B, "pos"), B, heads, dn, dr, R, 2 * inv_freq.numel(), ring, rs,
                       float(eps), f32)
        group = 1
        if n_split is None:
            n_split, group = self.latent_split(B, heads, (ring + 63) // 64)
        part_o = torch.empty(B, heads, n_split, R, dtype=torch.float32, device=qd.device)
        part_ml = torch.empty(B, heads, n_split, 2, dtype=torch.float32, device=qd.device)
        self._call("evo_latent_decode", q.data_ptr(), cache.data_ptr(), self._ix(pos, torch.int64, B, "pos"), part_o.data_ptr(), part_ml.data_ptr(),
                   B, heads, R, dr, rs, ring, int(window), n_split, float(scale), f32, group if self.mixer_mfma else 0)
        o = torch.empty(B, heads * dv, dtype=qd.dtype, device=qd.device)
        self._call("evo_latent_up", part_o.data_ptr(), part_ml.data_ptr(), self._ix(sink, torch.float32, heads, "sink"), wuv.data_ptr(), o.data_ptr(),
                   B, heads, R, dv, n_split, f32, int(self.mixer_mfma))
        return o

    # ---- attention with cached keys and values ---------------------------------------------------------------------------
    def heads_prep(self, z: torch.Tensor, nq: int, nk: int, dim: int, nv: int, qk_norm, inv_freq: torch.Tensor, amp: float, unit: bool, eps: float,
                   batch: TokenBatch, cache: Optional[torch.Tensor], keep: int) -> None:
        """z rows = [nq query vectors | nk key vectors | nv values]: norms (`qk_norm`: (query weight, key weight) or None; `unit`: behind the
        rotation, without a weight) and rotation in place; keys and values go to the cache [rows, ring, row]."""
        f32 = self._store(z) if cache is None else self._store(z, cache)
        M, B = z.shape[0], z.shape[0] if batch.decode else len(batch.lens)
        assert z.shape[1] >= (nq + nk) * dim + nv
        qw, kw = qk_norm if qk_norm is not None else (None, None)
        for w in (qw, kw):
            if w is not None:
                self._store(z, w), self._dense(w, (dim,), "norm weight")
        ring = rs = 0
        if cache is not None:
            rows, ring, rs = cache.shape
            self._dense(cache, (rows, ring, rs), "key and value cache")
            assert rows >= B
        self._call("evo_heads_prep", z.data_ptr(), z.stride(0), None if cache is None else cache.data_ptr(), None if qw is None else qw.data_ptr(),
                   None if kw is None else kw.data_ptr(), self._ix(inv_freq, torch.float32, 0, "inv_freq"), self._ix(batch.pos, torch.int64, M, "pos"),
                   self._ix(batch.seq, torch.int32, M, "seq"), self._ix(batch.cu, torch.int32, B + 1, "cu"), M, nq, nk, dim, nv, 2 * inv_freq.numel(),
                   keep, ring, rs, float(amp), float(eps), int(unit), f32)

    def heads_attention(self, z: torch.Tensor, kv: torch.Tensor, heads: int, kv_heads: int, maps: int, dim: int, dv: int, window: Optional[int],
                        keep: int, scale: float, lam: float, gain: float, eps: float, cu_q: torch.Tensor, cu_k: torch.Tensor, max_q: int) -> torch.Tensor:
        """Queries at the start of z's rows against kv rows [keys | values] -> [Mq, heads dv]."""
        nk = kv_heads * maps * dim
        assert z.shape[1] >= heads * maps * dim and kv.shape[1] >= nk + kv_heads * dv
        return self._window_attn(z, kv[:, :nk], kv[:, nk:], None, None, heads, kv_heads, maps, dim, 0, dv, window or 1 << 29, keep, scale, lam, gain, eps,
                                 cu_q, cu_k, max_q)

    @staticmethod
    def heads_split(groups: int, ring: int, cus: int = 256) -> int:
        """Parts of the cache in the decode kernel: a workgroup per CU, at least 128 slots (one round of a workgroup's waves) each."""
        return max(1, min((ring + 127) // 128, (cus + groups - 1) // groups, 64))

    def heads_whole_ok(self, groups: int, ring: int, Q: int, maps: int, dim: int, dv: int, z, cache) -> bool:
        """One workgroup per (sequence, key head) walks its whole cache and writes the result itself: no parts, no merge launch.  From 256 of them on the cache had one
        part anyway; with fewer only where a whole cache is short, as parts share a long sequence among short ones (us in a graph, parts and merge : whole.  Full caches /
        lengths from all of it down to a third / one full, the others 100 tokens.  10 sequences, 16 heads of two maps of 128, values of 256: 640 slots 43 : 29, 33 : 27, 21 : 23;
        1,028 slots 56 : 43, 40 : 40, 27 : 33; 2,048 88 : 73, 58 : 65, 37 : 50.  8 key heads of four queries, 128: 20 sequences, 1,536 slots 36 : 31, 28 : 27, 17 : 19,
        2,048 46 : 41, 36 : 37, 20 : 24; 10 sequences, 1,028 slots 18 : 16, 15 : 15, 13 : 15, 1,536 23 : 27, 18 : 21, 14 : 18.  16 heads of 64: 8 sequences, 2,048 slots
        21 : 25, 16 : 19, 13 : 15, 10 of them 30 : 26, 22 : 23, 13 : 15.  200 tokens each 12 : 7 to 25 : 15)."""
        return (self.mixer_mfma and z.dtype == torch.bfloat16 and dim % 8 == 0 and dv % 8 == 0 and z.stride(0) % 8 == 0 and cache.shape[2] % 8 == 0
                and dim <= (128 if maps == 2 else 256) and dv <= 256 and maps * min(Q, 16) <= 16 and (z.data_ptr() | cache.data_ptr()) % 16 == 0
                and groups >= 80 and (groups >= 256 or ring * (maps * dim + dv + 64) <= (500000 if groups >= 160 else 330000)))

    def heads_decode(self, z: torch.Tensor, cache: torch.Tensor, pos: torch.Tensor, heads: int, kv_heads: int, maps: int, dim: int, dv: int, scale: float,
                     lam: float, gain: float, eps: float, n_split: Optional[int] = None) -> torch.Tensor:
        """One token per cache row (already appended by heads_prep) -> [B, heads dv]."""
        f32 = self._store(z, cache)
        B = z.shape[0]
        rows, ring, rs = cache.shape
        self._dense(cache, (rows, ring, rs), "key and value cache")
        assert rows >= B and z.shape[1] >= heads * maps * dim and rs >= kv_heads * (maps * dim + dv)
        groups = B * kv_heads * ((heads // kv_heads + 15) // 16)
        if n_split is None and self.heads_whole_ok(groups, ring, heads // kv_heads, maps, dim, dv, z, cache):
            o = torch.empty(B, heads * dv, dtype=z.dtype, device=z.device)
            self._call("evo_heads_decode_whole", z.data_ptr(), z.stride(0), cache.data_ptr(), self._ix(pos, torch.int64, B, "pos"), o.data_ptr(), B, heads, kv_heads,
                       maps, dim, dv, ring, rs, float(scale), float(lam), float(gain), float(eps))
            return o
        if n_split is None:
            # (fp32: one wave per part, head and sequence, 64 slots a round)
            n_split = max(1, min((ring + 63) // 64, 4096 // (B * heads * maps), 64)) if f32 else self.heads_split(groups, ring)
        part_o = torch.empty(B, heads * maps, n_split, dv, dtype=torch.float32, device=z.device)
        part_ml = torch.empty(B, heads * maps, n_split, 2, dtype=torch.float32, device=z.device)
        self._call("evo_heads_decode", z.data_ptr(), z.stride(0), cache.data_ptr(), self._ix(pos, torch.int64, B, "pos"), part_o.data_ptr(),
                   part_ml.data_ptr(), B, heads, kv_heads, maps, dim, dv, ring, rs, n_split, float(scale), f32, int(self.mixer_mfma))
        o = torch.empty(B, heads * dv, dtype=z.dtype, device=z.device)
        self._call("evo_heads_merge", part_o.data_ptr(), part_ml.data_ptr(), o.data_ptr(), B, heads, maps, dv, n_split, float(lam), float(gain), float(eps),
                   f32)
        return o

    # ---- gated linear recurrence ------------------------------------------------------------------------------------------
    @staticmethod
    def rglru_mfma_ok(W: int, blocks: int, taps: int, dtype) -> bool:
        bs = W // blocks
        return dtype == torch.bfloat16 and bs % 8 == 0 and bs <= 384 and taps <= 4

    @staticmethod
    @functools.lru_cache(maxsize=64)
    def rglru_segment(lens: Tuple[int, ...], columns: int, cus: int = 256, small: bool = False) -> int:
        """Tokens per segment, as lightning_segment: 4.4 us a chunk, and 3.9 for its gates once more where sequences are cut; the carries walk the segments one by one.
        (us at 4,096 channels in 16 blocks, the rule before, from the longest sequence alone -> this one.  4,000, 1,000 and 2,000 tokens 262 -> 144 in segments of
        1,024; 3,000 and three times 300 202 -> 113; 2,000 and three times 500 144 -> 89; 5,000 and 300 173 -> 116; 500 52 -> 44 uncut; one of 8,190 152 -> 145 and
        six of 1,459 to 2,500, uncut, 187 -> 186 are cut as they were.)"""
        def us(seg, span, busy, n_wg):
            return 8.0 + 4.4 * span + (3.0 + 3.9 * span + 0.3 * ((max(lens) + seg - 1) // seg) if seg < max(lens) else 0.0)
        return MixerOps.cheapest_segment(lens, columns, us, cus, 0.65 if small else 1.0)

    def rglru(self, z: torch.Tensor, in_b: Optional[torch.Tensor], act: bool, W: int, conv: torch.Tensor, conv_b: torch.Tensor, ra, ra_b, ri, ri_b,
              decay: torch.Tensor, batch: TokenBatch, state: Optional[torch.Tensor] = None, seg_len: Optional[int] = None) -> torch.Tensor:
        """z [M, >= 2 W] = [y | x] -> o [M, W]; `in_b` [2 W]: still to be added to z; `act`: y is before its activation.  `state`
        [rows, 1 + taps, W] fp32 follows."""
        f32 = self._store(z, conv, conv_b, ra, ra_b, ri, ri_b)
        M, nb, taps = z.shape[0], ra.shape[0], conv.shape[1]
        bs = W // nb
        for t, shape, what in ((conv, (W, taps), "conv"), (conv_b, (W,), "conv_b"), (ra, (nb, bs, bs), "ra"), (ri, (nb, bs, bs), "ri"), (ra_b, (nb, bs), "ra_b"),
                               (ri_b, (nb, bs), "ri_b")):
            self._dense(t, shape, what)
        assert z.shape[1] >= 2 * W and (in_b is None or (in_b.dtype == z.dtype and in_b.is_contiguous() and in_b.numel() >= 2 * W))
        B = M if batch.decode else len(batch.lens)
        if state is not None:
            self._dense(state, (state.shape[0], 1 + taps, W), "state")
            assert state.dtype == torch.float32 and state.is_cuda and state.shape[0] >= B
        o = torch.empty(M, W, dtype=z.dtype, device=z.device)
        head = (z.data_ptr(), z.stride(0))
        sp, bp = None if state is None else state.data_ptr(), None if in_b is None else in_b.data_ptr()
        w = (conv.data_ptr(), conv_b.data_ptr(), ra.data_ptr(), ra_b.data_ptr(), ri.data_ptr(), ri_b.data_ptr(), self._ix(decay, torch.float32, W, "decay"),
             self._ix(batch.pos, torch.int64, M, "pos"))
        fast = self.mixer_mfma and self.rglru_mfma_ok(W, nb, taps, z.dtype) and z.stride(0) % 8 == 0
        if batch.decode and fast:
            self._call("evo_rglru_step_bf16", *head, bp, o.data_ptr(), sp, *w, B, W, nb, taps, int(act))
            return o
        cu, resume = self._ix(batch.cu, torch.int32, B + 1, "cu"), self._ix(batch.resume, torch.int32, B, "resume")
        if fast and in_b is None and not act:
            assert sum(batch.lens) == M
            L = max(batch.lens)
            seg_len = seg_len or self.rglru_segment(tuple(sorted(batch.lens)), nb * ((bs + 127) // 128), small=bs <= 64)
            seg = torch.empty(self.segment_slots(B, M, seg_len), 2, W, dtype=torch.float32, device=z.device) if L > seg_len else None
            self._call("evo_rglru_chunk_bf16", *head, o.data_ptr(), sp, None if seg is None else seg.data_ptr(), *w, cu, resume, B, W, nb, taps, L, seg_len)
            return o
        ab = torch.empty(M, 2, W, dtype=torch.float32, device=z.device)
        self._call("evo_rglru_any", *head, bp, o.data_ptr(), sp, ab.data_ptr(), *w, self._ix(batch.seq, torch.int32, M, "seq"), cu, resume, M, B, W, nb, taps,
                   int(act), f32)
        return o
