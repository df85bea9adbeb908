"""hipserve op library.

``KernelOps`` calls the hand-written gfx950 kernels in ``hipserve/_C.so``
(``torch.ops.hipserve.*``) and, for the layer-list decoders, ``hipserve/_C_seq.so``, ``_C_delta.so``,
``_C_cell.so`` and ``_C_stream.so`` (``torch.ops.hipserve_seq.*`` and so on); each library is loaded at the
first use of one of its kernels. ``ReferenceOps`` is the plain-PyTorch oracle used by
the CPU plumbing engine and by the numerics tests. The choice is made ONCE, when
an engine is built for a device — never per call. On a GPU device the native
library is mandatory: a missing/unloadable ``_C.so`` raises instead of silently
falling back to PyTorch.
"""
from __future__ import annotations

import functools
import math
import os
import threading

import torch
import torch.nn.functional as F

from . import gemm
from . import reference as ref

_PKG = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
_LIB = os.path.join(_PKG, "_C.so")
# the layer-list decoders' kernels, a library (and a torch.ops namespace hipserve_<name>) per set of designs:
# seq: latent attention, minGRU, table experts; delta: window attention, delta rules, decayed linear attention;
# cell: gated parallel blocks, mLSTM, PolyNorm; stream: residual streams, lightning attention
_SEQ_LIBS = {n: os.path.join(_PKG, f"_C_{n}.so") for n in ("seq", "delta", "cell", "stream")}
_lock = threading.Lock()
_loaded = False
_loaded_seq: set = set()


def library_path() -> str:
    return _LIB


def load_library(build_if_missing: bool = False) -> str:
    """Load hipserve/_C.so into torch.ops (idempotent). Raises if unavailable."""
    global _loaded
    with _lock:
        if _loaded:
            return _LIB
        if not os.path.exists(_LIB) and build_if_missing:
            from .._build import build_kernels

            build_kernels()
        if not os.path.exists(_LIB):
            raise RuntimeError(
                f"hipserve native kernels not built ({_LIB} missing): run `python -m hipserve._build`")
        torch.ops.load_library(_LIB)
        _loaded = True
        return _LIB


def load_kernel_library(name: str) -> str:
    """Load hipserve/_C_<name>.so (a key of ``_SEQ_LIBS``) into torch.ops (idempotent); built first when it is
    missing (a few hipcc seconds)."""
    path = _SEQ_LIBS[name]
    with _lock:
        if name in _loaded_seq:
            return path
        if not os.path.exists(path):
            from .._build import build_kernels

            build_kernels(lib=name)
        torch.ops.load_library(path)
        _loaded_seq.add(name)
        return path


def load_seq_library() -> str:
    return load_kernel_library("seq")


def load_delta_library() -> str:
    return load_kernel_library("delta")


def load_cell_library() -> str:
    return load_kernel_library("cell")


def load_stream_library() -> str:
    return load_kernel_library("stream")


def core_built() -> bool:
    """True when hipserve/_C.so exists (loaded or not): callers that only PREFER a core kernel ask this, so
    that a model which can do without never triggers the core library's build."""
    return _loaded or os.path.exists(_LIB)


def native_available() -> bool:
    try:
        load_library()
        return True
    except Exception:
        return False


class NormedRows:
    """Rows [T, H] before their norm's factor: row t is to be multiplied by 1 / sqrt(sum of squares[t] / H + eps). What
    ``KernelOps.linear_update`` leaves; ``KernelOps.linear`` takes them in place of a tensor."""

    def __init__(self, rows, squares, eps: float):
        self.rows, self.squares, self.eps = rows, squares, eps
        self.shape, self.dtype, self.device = rows.shape, rows.dtype, rows.device

    def normed(self):
        return (self.rows.float() * torch.rsqrt(self.squares.sum(1, keepdim=True) / self.shape[1] + self.eps)).to(self.dtype)


class DeltaBeside:
    """A delta rule's decode step, of so many workgroups, that another kernel of the same step may take into its launch; ``taken`` says whether one has."""

    def __init__(self, args, workgroups=0):
        self.args, self.workgroups, self.taken = args, workgroups, False

    def take(self, launch) -> bool:
        self.taken = bool(launch(*self.args))
        return self.taken


class ConvBeside:
    """The update of the inputs that a gated delta rule's convolution keeps, left by a decode step (``KernelOps.gated_delta_step``) for the layer's
    last product: ``take`` runs it in that product's launch, ``finish`` on its own unless it has run."""

    def __init__(self, ops):
        self.ops, self.left = ops, None   # (kept inputs, projection, sequences, taps)

    def take(self, launch) -> bool:
        if self.left is None or not launch(*self.left):
            return False
        self.left = None
        return True

    def finish(self):
        if self.left is not None:
            self.ops._delta.conv_update(*self.left)
            self.left = None


class ExpertSteps:
    """The products of a step's experts, to be launched in their order: each beside an independent product of the same step that takes it
    into its launch (``take``), or on its own (``finish``). None of them reads or writes what such a product writes or reads."""

    def __init__(self, ops, products):
        self.ops, self.left = ops, list(products)

    def take(self, launch) -> bool:
        """Whether ``launch`` (out, x, w, slots, tile_expert, gather_k, act, pairs, tiles) has taken the next product along."""
        if not self.left:
            return False
        out, x, w, slots, tile_expert, tile, gather_k, act, pairs, tiles = self.left[0]
        if not (tile == 32 and x.dtype == torch.bfloat16 and int(act) <= 1 and pairs > 0 and tiles > 0):
            return False
        if not launch(out, x, w, slots, tile_expert, gather_k, int(act), pairs, tiles):
            return False
        del self.left[0]
        return True

    def finish(self):
        for out, x, w, slots, tile_expert, tile, gather_k, act, pairs, tiles in self.left:
            self.ops.expert_gemm(out, x, w, slots, tile_expert, tile, gather_k, act, pairs=pairs, tiles=tiles)
        self.left = []


class KernelOps:
    """gfx950 HIP kernels (all outputs written in place; graph-capturable)."""

    name = "hip"

    def __init__(self):
        self._core = None
        self._lib_ops = {}
        # the library whose copy of the shared kernels runs ("seq" / "delta" / "cell" / "stream"): a model sets it to
        # the one its mixers load anyway, so it never builds or loads another
        self.norm_library = "seq"
        # the rules of products of a few rows: arithmetic on sizes, a few us each, and a step asks for every product. What they said of
        # the last sizes is kept (a step that is not captured, of four layers and a few rows, took 20 - 40 us longer)
        (self.skinny_pays, self.skinny_parts, self.update_pays, self.update_cols, self.mingru_pays, self.expert_plan, self.latent_run,
         self.two_pay) = (
            functools.lru_cache(maxsize=4096)(rule)
            for rule in (self._skinny_pays, self._skinny_parts, self._update_pays, self._update_cols, self._mingru_pays, self._expert_plan, self._latent_run,
                         self._two_pay))

    @property
    def _op(self):
        """torch.ops.hipserve, loaded at the first use of a core kernel (a missing _C.so raises there)."""
        if self._core is None:
            load_library(build_if_missing=os.environ.get("HIPSERVE_BUILD_ON_DEMAND") == "1")
            self._core = torch.ops.hipserve
        return self._core

    def _lib(self, name: str):
        """torch.ops.hipserve_<name>, its library loaded at the first use."""
        if name not in self._lib_ops:
            load_kernel_library(name)
            self._lib_ops[name] = getattr(torch.ops, "hipserve_" + name)
        return self._lib_ops[name]

    _seq = property(lambda self: self._lib("seq"))
    _delta = property(lambda self: self._lib("delta"))
    _cell = property(lambda self: self._lib("cell"))
    _stream = property(lambda self: self._lib("stream"))

    @property
    def _latent_lib(self):
        """The library whose copy of the latent-attention kernels runs."""
        return self._lib("cell" if self.norm_library == "cell" else "seq")

    @property
    def _window_lib(self):
        """The library whose copy of the window attention, router and activation kernels runs."""
        return self._lib(self.norm_library if self.norm_library in ("cell", "stream") else "delta")

    def rmsnorm(self, out, x, w, eps, out8=None):
        """out8: (e4m3 [rows, hidden] uint8, scales fp32 [rows]) per-token FP8 copy of out."""
        self._op.rmsnorm(out, x, w, eps, *(out8 if out8 is not None else (None, None)))
        return out

    def fused_add_rmsnorm(self, out, x, residual, w, eps, out8=None):
        self._op.fused_add_rmsnorm(out, x, residual, w, eps, *(out8 if out8 is not None else (None, None)))
        return out

    def silu_and_mul(self, out, x):
        self._op.silu_and_mul(out, x)
        return out

    def gelu_and_mul(self, out, x):
        self._op.gelu_and_mul(out, x)
        return out

    def qk_rmsnorm(self, qkv, q_w, k_w, nq, nkv, D, eps):
        self._op.qk_rmsnorm(qkv, q_w, k_w, nq, nkv, D, eps)

    def fill_uniform(self, out, row0, col0, gcols, key, scale):
        self._op.fill_uniform(out, row0, col0, gcols, key, scale)
        return out

    def rope_cache(self, qkv, positions, slots, cos_sin, k_cache, v_cache, nq, nkv, D, mode):
        self._op.rope_cache(qkv, positions, slots, cos_sin, k_cache, v_cache, nq, nkv, D, mode)

    def paged_decode(self, out, q, k_cache, v_cache, block_tables, context_lens, tmp_out, tmp_ml,
                     nq, nkv, part_size, scale, window=0, out16=None):
        self._op.paged_decode(out, q, k_cache, v_cache, block_tables, context_lens, tmp_out, tmp_ml,
                              nq, nkv, part_size, scale, window, out16)
        return out

    def prefill_attention(self, out, q, k_cache, v_cache, block_tables, cu_q, ctx_lens, tiles,
                          nq, nkv, scale, window=0):
        self._op.prefill_attention(out, q, k_cache, v_cache, block_tables, cu_q, ctx_lens, tiles,
                                   nq, nkv, scale, window)
        return out

    def sample(self, out_tok, out_lp, logits, temperature, top_k, top_p, seeds, steps, two_rounds=True):
        """two_rounds=False: no row combines top-k with top-p (the multi-CU sampler's
        second fine-histogram round is then a no-op and is not launched)."""
        self._op.sample(out_tok, out_lp, logits, temperature, top_k, top_p, seeds, steps, two_rounds)

    def penalty_apply(self, logits, slot, pres, freq, rep, counts, seen):
        self._op.penalty_apply(logits, slot, pres, freq, rep, counts, seen)

    def penalty_update(self, tok, slot, counts, seen):
        self._op.penalty_update(tok, slot, counts, seen)

    def penalty_init(self, counts, seen, slots, off, n_prompt, toks):
        self._op.penalty_init(counts, seen, slots, off, n_prompt, toks)

    def top_logprobs(self, logits, nreq, out_ids, out_lp):
        self._op.top_logprobs(logits, nreq, out_ids, out_lp)

    # ---- vision tower (csrc/kernels/vision.hip)
    def layernorm(self, out, x, w, b, eps, residual=None):
        self._op.layernorm(out, x, w, b, residual, eps)
        return out

    def gelu_(self, x, tanh):
        self._op.gelu_(x, tanh)
        return x

    VISION_TILE = 128  # query rows per attention workgroup (4 waves x 32)

    def vision_meta(self, geo, nh, D):
        """(cu_seqlens, tiles) device tensors of an image batch for vision_attention."""
        import numpy as np

        cu = geo.cu_seqlens
        tiles = np.array([(s, r) for s in range(len(cu) - 1) for r in range(0, int(cu[s + 1] - cu[s]),
                                                                          self.VISION_TILE)], np.int32)
        dev = torch.device("cuda", torch.cuda.current_device())
        return (torch.from_numpy(cu.astype(np.int32)).to(dev), torch.from_numpy(tiles.reshape(-1, 2)).to(dev))

    def vision_attention(self, out, qkv, cos_sin, cu_seqlens, nh, D, scale, meta=None):
        cu, tiles = meta
        self._op.vision_attention(out, qkv, cos_sin, cu, tiles, nh, D, scale)
        return out


    # ---- layer-list decoders (csrc/kernels/seq/*.hip; bf16 or true fp32 activations)
    def scaled_add_group_rmsnorm(self, out, residual, w, groups, eps, mix=None, ls1=None, y=None, pair_slot=None,
                                 top=0, ls2=None, extra=None, table=None, ids=None):
        """``table`` / ``ids``: the rows start as table[ids] instead of what ``residual`` holds. ``mix``: [T, H], or 32-bit parts of it
        [parts, T, H] (``linear_parts``)."""
        lib = self._delta if self.norm_library == "delta" else self._seq
        lib.scaled_add_group_rmsnorm(out, residual, w, groups, eps, mix, ls1, y, pair_slot, top, ls2, extra, table, ids)
        return out

    def latent_prepare(self, cq, cache, proj, positions, slots, q_norm, kv_norm, inv_freq, q_rank, kv_rank,
                       rot_dim, eps):
        self._latent_lib.latent_prepare(cq, cache, proj, positions, slots, q_norm, kv_norm, inv_freq, q_rank, kv_rank,
                                 rot_dim, eps)

    LATENT_PREFILL_TQ = 4  # tokens per workgroup of a prompt portion (x up to 4 heads = 16 waves)
    # bf16 runs the MFMA kernel (HIPSERVE_LATENT_MFMA=0: the generic kernel, as fp32 does)
    LATENT_MFMA = os.environ.get("HIPSERVE_LATENT_MFMA", "1") != "0"
    LATENT_DECODE_RUN = 128  # keys per run of a decode row (a multiple of 32; 64 measured slower)

    def latent_query_in_place(self, dtype, kv_rank, rot_dim) -> bool:
        """True when ``latent_attention`` wants the absorbed queries as bf16 rows of the cached width
        ([heads, T, kv_rank + rot_dim], the rotary part left for it to fill) instead of fp32 [heads, T, kv_rank]."""
        return dtype == torch.bfloat16 and self.LATENT_MFMA and bool(self._latent_lib.latent_attention_mfma_ok(kv_rank, rot_dim))

    # up to 64 rows the heads' products with W_uk and W_uv run the kernel for a few rows and the latents are faster (33 rows, one
    # mixer, width 2048: 67 us and 74); from there on forming the keys is: 96 rows 105 and 163
    LATENT_PROMPT_MIN_ROWS = 65

    def latent_prompt_rows(self, dtype, sp, nfreq, cache, meta, T) -> int:
        """Where the heads' keys and values of a step are formed (``latent_prompt_attention``): an upper bound of the cache rows
        that its sequences see; 0 where the attention on the latents is the one to run: steps with decode rows, and steps that
        see more than two cache rows per token, whose keys and values cost more than they save."""
        if not (dtype == torch.bfloat16 and self.LATENT_MFMA and sp.scale > 0 and T >= self.LATENT_PROMPT_MIN_ROWS and meta.num_decode == 0
                and nfreq == 32 and cache.shape[1] & (cache.shape[1] - 1) == 0 and cache.data_ptr() % 16 == 0 and sp.key_dim % 8 == 0
                and getattr(meta, "max_q", None) and getattr(meta, "max_ctx", None) and self._latent_lib.latent_prompt_ok(sp.dim, sp.rot_dim, sp.vdim)):
            return 0
        rows = meta.seq_ctx.shape[0] * min(meta.max_ctx, meta.max_q + sp.window - 1 if sp.window > 0 else meta.max_ctx)
        return rows if rows <= 2 * T else 0

    def latent_prompt_attention(self, out, q, proj, cache, meta, inv_freq, sp, w_kv, rows, gate_off):
        """out [T, heads * vdim] of a prompt step: the ``rows`` cache rows its sequences see times ``w_kv`` (keys of all heads, values
        of all heads), then attention of every head on its own keys and the shared rotary part."""
        lib = self._latent_lib
        lat = torch.empty(rows, sp.key_dim, device=q.device, dtype=q.dtype)
        off = torch.empty(meta.seq_ctx.shape[0] + 1, device=q.device, dtype=torch.int32)
        lib.latent_gather(lat, off, cache, meta.seq_cu, meta.seq_ctx, meta.seq_bt, sp.window)
        kv = F.linear(lat[:, :sp.kv_rank], w_kv)
        lib.latent_prompt_attention(out, q, kv, lat, off, meta.seq_cu, meta.seq_ctx, meta.positions, inv_freq, proj, sp.heads, gate_off,
                                    sp.gate == "channel", sp.scale, sp.window)
        return out

    def latent_attention(self, o_lat, q_abs, q, proj, cache, meta, inv_freq, heads, dim, rot_dim, kv_rank,
                         gate_off, scale, window):
        """Prompt portions (the step's first sequences) run several tokens per workgroup, decode
        rows one token per workgroup."""
        nseq = meta.seq_ctx.shape[0]
        nd = meta.num_decode
        npf, Tp = nseq - nd, meta.num_prefill_tokens
        if (q.dtype == torch.bfloat16 and self.LATENT_MFMA and self._latent_lib.latent_attention_mfma_ok(kv_rank, rot_dim)):
            # bf16: the matrix-core kernel; decode rows split their keys into runs merged by a reduce kernel
            if q_abs.dtype == torch.bfloat16:  # the absorption GEMM wrote the rows in place (latent_query_in_place)
                qc, q_abs = q_abs, None
            else:
                qc = torch.empty(heads, q.shape[0], kv_rank + rot_dim, device=q.device, dtype=q.dtype)
            fill = True
            if npf:
                self._latent_lib.latent_attention_mfma(o_lat, qc, q_abs, q, proj, meta.positions, cache, meta.seq_cu,
                                                meta.seq_ctx, meta.seq_bt, 0, npf, Tp, inv_freq, heads, dim, rot_dim,
                                                kv_rank, gate_off, scale, window, 1, 0, None, None, 0, fill)
                fill = False
            if nd:
                span = min(window, meta.max_ctx or window) if window > 0 else meta.max_ctx
                part = self.LATENT_DECODE_RUN
                if self._latent_lib.latent_attention_dma_ok(kv_rank, rot_dim):
                    part = self.latent_run(nd, heads, -(-span // 128) * 128)   # (so that a growing context seldom asks anew)
                while -(-span // part) > 64:
                    part *= 2
                nparts = max(1, -(-span // part))
                ws_acc = ws_ml = None
                if nparts > 1:
                    ws_acc = torch.empty(nparts, heads, nd, kv_rank, device=q.device, dtype=torch.float32)
                    ws_ml = torch.empty(nparts, heads, nd, 2, device=q.device, dtype=torch.float32)
                self._latent_lib.latent_attention_mfma(o_lat, qc, q_abs, q, proj, meta.positions, cache, meta.seq_cu,
                                                meta.seq_ctx, meta.seq_bt, npf, nseq, nd, inv_freq, heads, dim, rot_dim,
                                                kv_rank, gate_off, scale, window, nparts, part, ws_acc, ws_ml, Tp, fill)
            return
        for s0, s1, rows, tq in ((0, npf, Tp, self.LATENT_PREFILL_TQ), (npf, nseq, nd, 1)):
            if s1 > s0:
                self._latent_lib.latent_attention(o_lat, q_abs, q, proj, cache, meta.seq_cu, meta.seq_ctx, meta.seq_bt,
                                           s0, s1, rows, tq, inv_freq, heads, dim, rot_dim, kv_rank, gate_off,
                                           scale, window)

    @staticmethod
    def _latent_run(rows, heads, span) -> int:
        """Keys of a run of the decode kernel that multiplies 64 at a time. ``span`` is a bound on the contexts, and a captured step's is the model's length or its
        window, whatever its contexts are: so the choice is made over contexts of the span, half of it, a quarter, .. 128 keys, by a model of each (us of a latency, of
        a run's pieces one behind the other, which take longer where a compute unit has more than one workgroup, of workgroups that find no keys, and of the merge of
        the runs). Runs of 64, longer ones up to 256 where their workgroups are more than 1024, are left only for a length that is expected to take less on
        average over the contexts and nowhere more than 6 % more.
        360 measured (rows, heads, span, contexts) of 1 - 64 rows, 16, 32, 64 heads, spans of 200 - 8192 and contexts of 60 keys up to the span, equal and mixed: 7 % less than
        with those runs on average, at most 11 % more; chosen as if contexts were as long as the span, 6 % less and up to twice as long. us of runs of 64 / 128 / 256 / 512 / 1024
        keys: 48 rows, 16 heads, span 1024, contexts of 150 13.2 / 13.8 / 15.4 / 15.4 / 13.1, of 700 28.5 / 21.1 / 22.8 / 32.6 / 38.4, of 1024 30.7 / 24.9 / 25.6 / 33.5 / 52.4; 16 rows,
        32 heads, span 8192, of 700 - / 20.3 / 20.3 / 26.5 / 32.1, of 2000 - / 30.2 / 27.0 / 34.2 / 54.1, of 8192 - / 77 / 59 / 48 / 60."""
        groups = rows * -(-heads // 16)

        def time(part, ctx):
            runs, live, pieces = -(-span // part), -(-ctx // part), -(-min(part, ctx) // 64)
            return (5.6 + 2.3 * pieces * max(1.0, groups * live / 256) + 2.7e-3 * groups * runs
                    + (1.3 + 0.07 * runs + 0.83e-3 * rows * heads * live if runs > 1 else 0.0))
        plain = 64
        while plain < 256 and groups * -(-span // plain) > 1024:
            plain *= 2
        ctxs = [span >> i for i in range(max(1, span.bit_length())) if i == 0 or span >> i >= 128]
        known, best = [time(plain, c) for c in ctxs], (float("inf"), plain)
        for part in (64, 128, 256, 512):
            times = [time(part, c) for c in ctxs]
            if all(t <= 1.06 * k for t, k in zip(times, known)):
                best = min(best, (math.prod(t / k for t, k in zip(times, known)), part))
        return best[1]

    def _mingru_pays(self, rows, width, k, f32) -> bool:
        """Whether the step in its product's epilogue is expected to take less than the faster product of the two and its launch, 2 us (1 in 32 bits)
        as the rules' times go: of 1209 sizes (1 - 64 rows, widths 256 - 8192, k 256 - 4096) the choice takes 1 % longer than the faster of the two.
        us, product and step / this: width 4096, k 2048, 1 and 48 rows 14.8 / 12.6, 20.6 / 16.4; in 32 bits width 512, k 4096, 33 rows 18.5 / 41.2."""
        apart = min(self._skinny_time(rows, 3 * width, k, False, f32), 1.2 * self._vendor_time(rows, 3 * width, k, f32))
        return self._seq.mingru_product_time(rows, width, k, f32) < apart + (1.0 if f32 else 2.0)

    def mingru_product(self, y, state, x, w, b_z, b_x, meta, beside=None) -> bool:
        """``mingru_scan`` of the product x . w^T for a step of one row per sequence; False, and nothing done, where they are two launches.
        ``beside``: an ``ExpertSteps`` whose next product may go into the launch."""
        if not (meta.max_q == 1 and x.dim() == 2 and self._skinny_ok(x, w) and self.mingru_pays(x.shape[0], y.shape[-1], w.shape[1], x.dtype == torch.float32)):
            return False
        seqs = (meta.seq_cu, meta.seq_ctx, meta.seq_state)
        if beside is None or not beside.take(lambda *e: self._seq.mingru_product_experts(y, state, x, w, b_z, b_x, *seqs, *e)):
            self._seq.mingru_product(y, state, x, w, b_z, b_x, *seqs)
        return True

    def mingru_scan(self, y, state, proj, b_z, b_x, meta):
        self._seq.mingru_scan(y, state, proj, b_z, b_x, meta.seq_cu, meta.seq_ctx, meta.seq_state, meta.max_q)

    def attn_prepare(self, proj, cache, meta, inv_freq, sp, q_norm, k_norm, eps):
        mode = 1 if sp.qk_norm else 2 if sp.head_norm else 3 if sp.unit_qk else 0
        own_kv = sp.kv_from is None   # else the layer reads another layer's cache: only q is prepared
        self._window_lib.attn_prepare(proj, cache if own_kv else None, meta.positions, meta.slot_mapping, inv_freq, sp.heads,
                                 sp.kv_heads, sp.maps, sp.dim, sp.vdim, q_norm if mode in (1, 2) else None,
                                 k_norm if mode in (1, 2) and own_kv else None, mode, sp.v_norm, eps,
                                 sp.scaling.amplitude if sp.scaling is not None else 1.0, sp.temp_coef, sp.temp_every)

    WINDOW_PREFILL_TQ = 4  # tokens per workgroup of a prompt portion (x the query heads of one key/value head)
    # the matrix-core kernels where they take the sizes (HIPSERVE_WINDOW_MFMA=0: the generic kernel)
    WINDOW_MFMA = os.environ.get("HIPSERVE_WINDOW_MFMA", "1") != "0"
    WINDOW_DECODE_RUN = 128  # keys per run of a decode row (a multiple of 32)

    def window_step(self, out, proj, cache, meta, inv_freq, sp, q_norm, k_norm, eps, gate_off, out_scale=1.0, sink_w=None, beside=None) -> bool:
        """``attn_prepare`` and ``window_attention`` of a decode step (one row per sequence) in one launch; False, and nothing done, where they
        are two. ``beside``: a ``DeltaBeside`` that may go into the launch (it says so)."""
        if not (meta.max_q == 1 and meta.num_prefill_tokens == 0 and meta.num_decode == meta.seq_ctx.shape[0] > 0 and inv_freq.numel() % 8 == 0
                and 2 * inv_freq.numel() <= sp.dim <= 128 and all(w is None or w.data_ptr() % 16 == 0 for w in (q_norm, k_norm))):
            return False
        mode, own_kv = 1 if sp.qk_norm else 2 if sp.head_norm else 3 if sp.unit_qk else 0, sp.kv_from is None
        prep = (meta.positions, meta.slot_mapping, inv_freq, own_kv, q_norm if mode in (1, 2) else None, k_norm if mode in (1, 2) and own_kv else None,
                mode, sp.v_norm, eps, sp.scaling.amplitude if sp.scaling is not None else 1.0, sp.temp_coef, sp.temp_every)
        return self._window_decode(out, proj, cache, meta, sp, gate_off, out_scale, sink_w, prep, beside)

    def _window_decode(self, out, proj, cache, meta, sp, gate_off, out_scale, sink_w, prep=None, beside=None) -> bool:
        """The decode rows of ``window_attention`` by the kernel for them; False where it does not take the sizes. ``prep``: what is between
        the cache and the table in ``window_attention_step``."""
        if sp.maps != 1 or not self.WINDOW_MFMA or not self._window_lib.window_attention_decode_ok(proj, cache, sp.dim, sp.vdim):
            return False
        nd = meta.num_decode
        span = min(sp.reach, meta.max_ctx or sp.reach) if sp.reach > 0 else meta.max_ctx
        groups = nd * sp.kv_heads * -(-(sp.heads // sp.kv_heads) // 16)   # workgroups per run
        # One run where a second launch to merge runs costs more than it spreads: few keys (200 keys of one sequence, 8 heads
        # over 2: 7.2 us, two runs 8.1; 400 keys: 9.2, four runs 8.5), or workgroups for half of the chip and no more than
        # 1024 keys (41 sequences x 4 key heads: 21.3 us, in runs of 128 24.3; 16 sequences: 16.9, in runs 13.3). Longer runs
        # where there would be many (8000 keys of one sequence, 8 key heads: runs of 256 17.6 us, of 128 22.4) or they would
        # fill the chip several times over (their unnormalised outputs are written and read once more).
        part = max(1, span)
        if span > 256 and (groups < 128 or span > 1024):
            part = self.WINDOW_DECODE_RUN
            while -(-span // part) > 32 or groups * -(-span // part) > 1024 and part < span:
                part *= 2
        nparts = max(1, -(-span // part))
        # Two launches in fp32 of 128 dims, whose registers hold one workgroup per compute unit (two without the preparation), where the compute
        # units take several: few keys each, or many key heads and rounds that two at a time halve. us, one launch / two, 8 key heads: 48 and 64
        # rows of 70 keys 20.1 / 16.1, 21.7 / 17.4, of 900 keys 86.5 / 85.3, 119 / 96.5, 8 rows in runs of 128 26.2 / 24.0; but 32 rows (256
        # workgroups) 51.9 / 62.6, 96 rows (768) 158 / 169, with 4 key heads 128 and 192 rows 92.6 / 92.4, 137 / 159. bf16 holds one either way.
        wgs = groups * nparts
        if prep is not None and proj.dtype == torch.float32 and sp.dim == 128 and wgs > 256 and (
                min(part, span) <= 128 or sp.kv_heads >= 8 and (wgs - 1) % 512 >= 256):
            return False
        ws_acc = ws_ml = None
        if nparts > 1:
            ws_acc = torch.empty(nparts, sp.heads, nd, sp.vdim, device=proj.device, dtype=torch.float32)
            ws_ml = torch.empty(nparts, sp.heads, nd, 2, device=proj.device, dtype=torch.float32)
        rest = (sp.heads, sp.kv_heads, sp.dim, gate_off, sp.scale, sp.window, sp.sink, out_scale, nparts, part, ws_acc, ws_ml,
                sp.keep_first, sp.softcap, sink_w, sp.channel_gate, sp.chunk)
        if prep is not None:
            args = (out, proj, cache, *prep, meta.seq_cu, meta.seq_ctx, meta.seq_bt, *rest)
            if beside is None or not self._window_delta_pays(sp.dim, min(part, span), beside.workgroups) or not beside.take(lambda *d: self._delta.window_delta_step(*args, *d)):
                self._window_lib.window_attention_step(*args)
        else:
            self._window_lib.window_attention_decode(out, proj, cache, meta.seq_cu, meta.seq_ctx, meta.seq_bt,
                                                     meta.seq_ctx.shape[0] - nd, meta.num_prefill_tokens, *rest)
        return True


    def window_attention(self, out, proj, cache, meta, sp, gate_off, out_scale=1.0, lam=0.0, eps=0.0, sink_w=None):
        """Prompt portions (the step's first sequences) run several tokens per workgroup, decode
        rows one token per workgroup. Two maps per head (``sp.maps`` = 2): ``lam`` weighs the second
        map, the head output is divided by its root mean square (``eps``) and scaled by 1 - ``sp.diff``.
        ``sink_w``: fp32 [heads] learned sink logits (None: 0)."""
        nseq = meta.seq_ctx.shape[0]
        nd = meta.num_decode
        npf, Tp = nseq - nd, meta.num_prefill_tokens
        diff = (sp.maps, lam, 1.0 - sp.diff, eps, sp.keep_first, sp.softcap, sink_w, sp.channel_gate, sp.chunk)
        if nd and self._window_decode(out, proj, cache, meta, sp, gate_off, out_scale, sink_w):
            nseq, nd = npf, 0   # what is left
        if (proj.dtype == torch.bfloat16 and self.WINDOW_MFMA
                and self._window_lib.window_attention_mfma_ok(sp.dim, sp.vdim, out.stride(0), out.storage_offset(), sp.maps)):
            # bf16: the matrix-core kernel; decode rows split their keys into runs merged by a reduce kernel
            args = (sp.heads, sp.kv_heads, sp.dim, sp.vdim, gate_off, sp.scale, sp.window, sp.sink, out_scale)
            if npf:
                self._window_lib.window_attention_mfma(out, proj, cache, meta.seq_cu, meta.seq_ctx, meta.seq_bt, 0, npf, Tp,
                                                *args, 1, 0, None, None, 0, *diff)
            if nd:
                # keys a row can see: its window and the kept first keys behind it, or its chunk
                reach = sp.reach
                span = min(reach, meta.max_ctx or reach) if reach > 0 else meta.max_ctx
                part = self.WINDOW_DECODE_RUN
                if span >= 16 * part:   # long runs of keys: fewer, longer runs per row (measured at 2k and 8k keys)
                    part *= 2
                while -(-span // part) > 64:
                    part *= 2
                nparts = max(1, -(-span // part))
                ws_acc = ws_ml = None
                if nparts > 1:
                    ws_acc = torch.empty(nparts, sp.heads * sp.maps, nd, sp.vdim, device=proj.device, dtype=torch.float32)
                    ws_ml = torch.empty(nparts, sp.heads * sp.maps, nd, 2, device=proj.device, dtype=torch.float32)
                self._window_lib.window_attention_mfma(out, proj, cache, meta.seq_cu, meta.seq_ctx, meta.seq_bt, npf, nseq, nd,
                                                *args, nparts, part, ws_acc, ws_ml, Tp, *diff)
            return
        if npf and (proj.dtype == torch.float32 and sp.maps == 1 and self.WINDOW_MFMA
                    and self._window_lib.window_attention_decode_ok(proj, cache, sp.dim, sp.vdim)):
            # fp32 prompts on the 32-bit matrix cores (3 prompts, 8 heads over 2 of 128: 104 -> 28 us)
            self._window_lib.window_attention_prompts_f32(out, proj, cache, meta.seq_cu, meta.seq_ctx, meta.seq_bt, 0, npf, Tp,
                                                          sp.heads, sp.kv_heads, sp.dim, gate_off, sp.scale, sp.window, sp.sink,
                                                          out_scale, sp.keep_first, sp.softcap, sink_w, sp.channel_gate, sp.chunk)
            npf = 0
        for s0, s1, rows, tq in ((0, npf, Tp, self.WINDOW_PREFILL_TQ), (nseq - nd, nseq, nd, 1)):
            if s1 > s0:
                self._window_lib.window_attention(out, proj, cache, meta.seq_cu, meta.seq_ctx, meta.seq_bt, s0, s1, rows, tq,
                                           sp.heads, sp.kv_heads, sp.dim, sp.vdim, gate_off, sp.scale, sp.window,
                                           sp.sink, out_scale, *diff)

    # bf16 prompt portions of at least this many rows run the delta rules in chunks on the (fp32) matrix cores
    # (HIPSERVE_DELTA_CHUNK=0: token by token on the scan, as fp32 does)
    DELTA_CHUNK = os.environ.get("HIPSERVE_DELTA_CHUNK", "1") != "0"
    DELTA_CHUNK_ROWS = 32
    DELTA_CHUNK_DTYPES = (torch.bfloat16,)

    def gated_delta(self, y, state, proj, conv_w, a_log, dt_bias, norm_w, decay, gate, offs, sp, eps, meta):
        """``decay`` (fp32) / ``gate``: the pre-activations that come from bottlenecks (None: columns of ``proj``);
        ``offs``: the columns of ``proj`` where the decay, the gate and beta (or the bottlenecks) start."""
        T = proj.shape[0]
        scratch = torch.empty(T * (2 * sp.kv_heads * sp.dim + 2 * sp.out_size + sp.heads * (1 + (sp.dim if sp.channel_decay else 1))) + 64,
                              device=proj.device, dtype=torch.float32)
        chunks = None
        if self.DELTA_CHUNK and proj.dtype in self.DELTA_CHUNK_DTYPES and meta.max_q >= self.DELTA_CHUNK_ROWS:
            n = self._delta.delta_chunk_floats(T, meta.seq_ctx.shape[0], sp.heads, sp.dim, sp.vdim)   # 0: not for these sizes
            chunks = torch.empty(n, device=proj.device, dtype=torch.float32) if n else None
        self._delta.gated_delta(y, state[0], state[1], proj, conv_w, a_log, dt_bias, norm_w, decay, gate, meta.seq_cu,
                                meta.seq_ctx, meta.seq_state, scratch, sp.heads, sp.kv_heads, sp.dim, sp.vdim, sp.conv, eps,
                                *offs, sp.channel_decay, sp.gate_act == "silu", chunks)

    def conv_beside(self):
        return ConvBeside(self)

    def gated_delta_step(self, y, state, proj, conv_w, a_log, dt_bias, norm_w, w_a2, w_g2, offs, sp, eps, meta, conv=None):
        """``gated_delta`` for steps in which every sequence has one row (``meta.max_q`` == 1), the bottlenecks'
        up-projections ``w_a2`` / ``w_g2`` included; ``conv``: a ``ConvBeside`` that is given the update of the convolution's kept inputs where
        that is a launch of its own (queries and keys shared by several heads)."""
        later = conv is not None and sp.heads != sp.kv_heads
        self._delta.gated_delta_step(y, state[0], state[1], proj, conv_w, a_log, dt_bias, norm_w, w_a2, w_g2, meta.seq_cu,
                                     meta.seq_ctx, meta.seq_state, sp.heads, sp.kv_heads, sp.dim, sp.vdim, sp.conv, eps,
                                     *offs, sp.channel_decay, sp.gate_act == "silu", not later)
        if later:
            conv.left = (state[1], proj, meta.seq_cu, meta.seq_ctx, meta.seq_state, sp.conv)

    DELTA_LOW_RANK = 128   # widest bottleneck that every (sequence, head) multiplies for itself

    def _delta_low_ok(self, state, proj, w2, sp, meta) -> bool:
        # Every workgroup (a head of a row) reads its 64 rows of w2 again, from its compute unit's 32 KB of cache where they fit: a launch saved
        # (1.9 us) against that. us, one launch / two: rank 64 in bf16 1024 workgroups 10.6 / 12.1, 4096 33.2 / 33.0, in fp32 2048 19.7 / 20.6, 3072
        # 28.9 / 27.8; rank 128 in bf16 2048 19.6 / 20.2, 3072 31.2 / 27.4, 16384 137 / 111, in fp32 512 7.9 / 8.7, 1024 13.1 / 12.3, 16384 176 / 117.
        per, row = 16 // proj.element_size(), w2.shape[1] * w2.element_size()
        if proj.shape[0] * sp.heads * row > (1 << 19 if row <= 256 else 1 << 18):
            return False
        return (meta.max_q == 1 and self._delta.delta_rule_step_ok(sp.dim) and w2.shape[1] % 32 == 0 and w2.shape[1] <= self.DELTA_LOW_RANK
                and proj.dtype == w2.dtype and w2.is_contiguous() and proj.stride(0) % per == 0 and all(t.data_ptr() % 16 == 0 for t in (state[0], proj, w2)))

    def delta_rule_low(self, out, state, proj, w2, a_b, w0, norm_w, sp, eps, meta, out_scale=1.0) -> bool:
        """``delta_rule`` of a decode step with the bottleneck's product (the last columns of ``proj`` times ``w2``) in its launch; False, and
        nothing done, where it is a product before it."""
        if not self._delta_low_ok(state, proj, w2, sp, meta):
            return False
        self._delta.delta_rule_step(out, state[0], proj, None, a_b, w0, norm_w, meta.seq_cu, meta.seq_ctx, meta.seq_state,
                                    sp.heads, sp.dim, eps, out_scale, w2)
        return True

    def delta_beside(self, out, state, proj, w2, a_b, w0, norm_w, sp, eps, meta, out_scale=1.0):
        """``delta_rule_low`` for ``window_step`` to take into its launch: a ``DeltaBeside``, or None where it has no such launch."""
        if not (meta.num_prefill_tokens == 0 and self._delta_low_ok(state, proj, w2, sp, meta)):
            return None
        return DeltaBeside((out, state[0], proj, a_b, w0, norm_w, meta.seq_state, sp.heads, sp.dim, eps, out_scale, w2), meta.num_decode * sp.heads)

    @staticmethod
    def _window_delta_pays(dim: int, keys: int, workgroups: int) -> bool:
        """Whether window attention over runs of so many keys takes a delta rule's workgroups into its launch. They have its LDS and waves then, up to eight of
        128 dims from 128 keys on, and many of them wait for room. Beside such runs in bf16, 24 sizes with 1000 - 2000 of
        them are 7 % faster in one launch on average, of 55 with 2000 - 8000 29 are slower, by up to 15 %: us, apart / one, 128 rows of 2 heads, 300 keys and
        32 of the rule's 43.4 / 49.7, 96 of 16 over 4, 230 and 48 50.0 / 56.1; but 128 rows of 16 over 2 of 64 dims and 48 48.9 / 45.4."""
        return not (dim == 128 and keys > 128 and workgroups >= 2048)

    def delta_rule(self, out, state, proj, wl, a_b, w0, norm_w, sp, eps, meta, out_scale=1.0):
        def aligned(*tensors):   # the kernels below read and write 16 bytes at a time
            return all(t.data_ptr() % 16 == 0 for t in tensors)
        if meta.max_q == 1 and self._delta.delta_rule_step_ok(sp.dim) and aligned(state[0]):   # decode steps: one launch
            self._delta.delta_rule_step(out, state[0], proj, wl, a_b, w0, norm_w, meta.seq_cu, meta.seq_ctx, meta.seq_state,
                                        sp.heads, sp.dim, eps, out_scale)
            return
        T, n = proj.shape[0], 0
        if self.DELTA_CHUNK and proj.dtype in self.DELTA_CHUNK_DTYPES and meta.max_q >= self.DELTA_CHUNK_ROWS and aligned(wl, a_b, w0):
            n = self._delta.delta_rule_chunk_floats(proj, meta.seq_ctx.shape[0], sp.heads, sp.dim)   # 0: not for these sizes
        chunks = torch.empty(n, device=proj.device, dtype=torch.float32) if n else None
        scratch = torch.empty(T * sp.size + 64 if n else T * 7 * sp.size, device=proj.device, dtype=torch.float32)
        self._delta.delta_rule(out, state[0], proj, wl, a_b, w0, norm_w, meta.seq_cu, meta.seq_ctx, meta.seq_state,
                             scratch, sp.heads, sp.dim, eps, out_scale, chunks)

    # ---- dense layers
    SKINNY_ROWS = 64
    GLU_ACTS = ("silu_mul", "clamped_glu")

    def _skinny_pays(self, rows: int, cols: int, k: int, glu: bool = False, f32: bool = False, act: bool = False) -> bool:
        """Whether ``skinny_linear`` is expected to be faster than the vendor's GEMM for ``rows`` x ``cols`` results (``cols`` over all
        batches), both sides in us for cold weights: ours as the kernel's choice of tiles has it (skinny_time in skinny_linear.hip), the vendor's as
        the choice between them comes out best. Over 5127 sizes (1 - 64 rows, 64 - 65536 columns, k 128 - 12288, plain and gated, 32 bits) it takes
        1.2 % longer than the faster of the two. Examples, ours / vendor: 2048 x 2048 with 1, 16, 48, 64 rows 4.0 / 11.0, 4.3 / 11.0, 7.0 / 11.1, 7.7 /
        11.7; 6144 x 2048 with 1, 16, 48 rows 7.0 / 12.5, 8.0 / 12.5, 10.2 / 13.1; 4096 x 12288 with 1, 16, 48 rows 20.4 / 22.0, 22.0 / 22.5, 33.6 /
        32.1; 512 x 8192 with 48 rows 14.9 / 11.4; 32000 x 2048 with 1, 16, 48, 64 rows 25.0 / 32.3, 27.5 / 32.7, 33.3 / 37.4, 37.5 / 34.2; in 32 bits
        1024 x 1024 with 1, 16, 48 rows 3.7 / 8.3, 3.8 / 8.8, 6.4 / 8.8; 32000 x 2048 with 1, 16, 64 rows 44 / 63, 51 / 65, 84 / 72."""
        # an activation is a launch more there (48 x 32000: 6 - 8 us)
        launch = 2.5 + 2.5e-6 * rows * cols if act and not glu else 0.0
        return self._skinny_time(rows, cols, k, glu, f32) < self._vendor_time(rows, cols, k, f32, glu) + launch

    def _skinny_time(self, rows, cols, k, glu=False, f32=False, parts=1) -> float:
        return self._moe_lib.skinny_time(rows, cols, k, glu, f32, parts)

    # [f32, gate][up to 16, 32, 48, 64 rows]: us that the vendor's product takes at least, that per 1000 k, that per doubling of more than 1024 columns;
    # us and TB/s of large weights
    VENDOR = {(False, False): ((6.58, 0.52, 0.07, 1.54, 3.04), (5.88, 0.64, 0.09, 6.1, 4.8), (3.0, 1.09, 0.02, 9.87, 5.11), (6.09, 1.47, 0.21, 6.49, 5.41)),
              (True, False): ((4.67, 1.71, 0.14, 4.79, 3.32), (3.86, 2.0, 1.5, 9.6, 6.02), (4.25, 1.98, 1.21, 6.76, 2.58), (4.34, 2.0, 1.1, 7.25, 4.82)),
              (False, True): ((6.07, 0.66, 1.22, 4.64, 5.03), (8.06, 0.84, 0.12, 8.17, 5.03), (8.81, 0.97, 0.03, 8.9, 4.27), (8.78, 1.8, 0.24, 9.17, 4.51)),
              (True, True): ((4.67, 2.0, 1.5, 7.69, 5.25), (6.04, 2.0, 1.18, 9.15, 4.51), (8.32, 1.99, 0.98, 5.85, 3.31), (6.83, 2.0, 0.89, 8.72, 4.09))}

    @staticmethod
    def _vendor_time(rows, cols, k, f32, glu=False) -> float:
        """us of the vendor's GEMM (and of the gate's launch), which are by turns a fifth above and below any smooth rule: the constants are those
        that made the fewest and smallest wrong choices beside ``skinny_time``, not the closest ones. 16-bit weights whose rows lie a multiple of
        4096 bytes apart come slower, up to k of 8192: 17 - 48 rows, TB/s at k of 1536, 2048, 2304, 3072, 3584, 4096, 5120, 6144 (mean of 16384 - 65536
        columns) 3.8, 3.7, 4.6, 4.7, 4.9, 4.2, 5.1, 4.4. A tenth of the rate is what chooses best (0.07 - 0.1 alike; 5127 sizes: 1.33 % longer than the
        faster one without it, 1.24 with it): 32000 x 2048 with 48 rows 33.3 / 37.4, 24576 x 4096 gated with 32 rows 40.1 / 49.0."""
        least, per_k, per_cols, start, rate = KernelOps.VENDOR[f32, glu][(min(rows, 64) - 1) // 16]
        if not f32 and k % 2048 == 0 and k < 8192:
            rate *= 0.91
        least += per_k * 1e-3 * k + (per_cols * math.log2(cols / 1024) if cols > 1024 else 0.0)
        return max(least, start + (4.0 if f32 else 2.0) * cols * k / 1e6 / rate)

    def _skinny_parts(self, rows, cols, k, f32=False) -> int:
        """Parts of k for a product whose 32-bit sums the next kernel adds up (1: none), or 0 where the vendor's GEMM is the one to run. A part
        more gives idle compute units a share and costs 0.15 us and what it is to write and read it (fitted), and the first one 0.7 us, which
        the update takes longer with parts in a captured step than in a loop of the two; every wave keeps a piece of 64 halves. The vendor's 1.2: it
        is the slower one by more than ``_vendor_time`` says where parts pay, many k. us with the residual update and norm behind it, cold weights,
        vendor / one / two / four parts: 1024 x 3072 with 1, 16, 48 rows 14.6 / 8.0 / 7.5 / 7.5, 15.1 / 9.7 / 8.4 / 8.1, 14.7 / 12.8 / 10.2 / 9.1; 2048
        x 2048 with 1, 16, 48 rows 14.0 / 7.9 / 7.7 / 8.3, 14.3 / 8.8 / 8.2 / 8.9, 14.3 / 10.7 / 9.6 / 10.4; 2048 x 6144 with 16, 48 rows 14.6 / 14.2
        / 11.4 / 11.8, 19.9 / 20.2 / 14.6 / 14.0; 4096 x 4096 with 24 rows 16.7 / 13.7 / 14.7 / 15.6; 4096 x 12288 with 48 rows 35.0 / 36.7 / 32.1 /
        28.8. Over 855 sizes (1 - 64 rows, 512 - 6144 columns, k 512 - 12288) the choice takes 1 % longer than the best of the four."""
        ours, parts = min((self._parts_time(rows, cols, k, f32, p), p) for p in (1, 2, 4))
        one = self._parts_time(rows, cols, k, f32, 1)
        if ours > 0.94 * one:   # no more parts for what the model cannot tell
            ours, parts = one, 1
        return parts if ours < 1.2 * self._vendor_time(rows, cols, k, f32) else 0

    def _parts_time(self, rows, cols, k, f32, p) -> float:
        if p > 1 and p * 512 > k * (2 if f32 else 1):
            return float("inf")
        return self._skinny_time(rows, cols, k, False, f32, p) + (p > 1) * 0.7 + (p - 1) * (0.15 + 0.2e-5 * rows * cols)

    def _linear_beside(self, x, w, beside, parts=1):
        """The product x . w^T in one launch with the next product of ``beside``, or None (also where they are faster apart for the numbers of their
        workgroups: expert_beside.hip). What would be ``parts`` of k without it is one, still in 32 bits: the experts fill the compute units that parts are for. From 33 rows on such a product holds a compute unit for longer than the launch saves:
        16 experts of 2048 x 1024 beside 2048 x 4096, us apart / in one launch: 32 rows 20.6 / 19.3, 48 rows 21.9 / 23.6, 64 rows 23.0 / 25.6; 8 of
        1024 x 512 beside 1024 x 2048, 40, 64 rows 7.9 / 6.4, 8.5 / 7.6."""
        if parts > 1 and x.shape[0] > 32 and w.numel() > 1 << 21:
            return None
        T, N = x.shape[0], w.shape[0]
        out = torch.empty(*((1, T, N) if parts > 1 else (T, N)), device=x.device, dtype=torch.float32 if parts > 1 else x.dtype)
        return out if beside.take(lambda *e: self._seq.skinny_linear_experts(out, x, w, *e)) else None

    def linear_parts(self, x, w, bias=None, beside=None):
        """``linear`` for a result that ``scaled_add_group_rmsnorm`` takes as ``mix``: where that is faster, 32-bit sums over parts of k,
        [parts, T, N]. ``beside``: an ``ExpertSteps`` whose next product may go into the launch."""
        if x.dim() == 2 and x.shape[0] <= self.SKINNY_ROWS and self._skinny_ok(x, w, bias):
            T, N, K = x.shape[0], w.shape[0], w.shape[1]
            parts = self.skinny_parts(T, N, K, x.dtype == torch.float32)
            if parts and bias is None and beside is not None:
                out = self._linear_beside(x, w, beside, parts)
                if out is not None:
                    return out
            if parts > 1:
                out = torch.empty(parts, T, N, device=x.device, dtype=torch.float32)
                self._moe_lib.skinny_linear_parts(out, x, w, bias)
                return out
            if parts:
                return self._skinny_linear(x, w, bias)
        return self.linear(x, w, bias)

    def _skinny_ok(self, x, w, bias=None) -> bool:
        """The shapes, types, alignment and bias that ``skinny_linear`` takes."""
        if x.dim() != w.dim() or not 0 < x.shape[-2] <= self.SKINNY_ROWS:
            return False
        per, K, stride = 16 // x.element_size(), x.shape[-1], x.stride()
        return (x.dtype in (torch.bfloat16, torch.float32) and w.dtype == x.dtype and K % per == 0 and max(K, stride[-2]) < 1 << 24
                and stride[-1] == 1 and stride[-2] % per == 0 and stride[0] % per == 0
                and x.data_ptr() % 16 == 0 and w.is_contiguous() and w.data_ptr() % 16 == 0
                and (bias is None or (bias.dtype == x.dtype and bias.shape == w.shape[:1] and bias.is_contiguous())))

    def linear(self, x, w, bias=None, out_f32=False, act=None, c0=0.0, c1=0.0, act_from=0, beside=None):
        """act(x . w^T + bias) of rows x [T, K]; ``out_f32``: a 32-bit result of 16-bit operands; ``act_from``: the first column that
        the activation applies to. A few rows run the weight-streaming kernel with the activation in its epilogue, anything else the
        vendor's GEMM and a second launch. ``beside``: an ``ExpertSteps`` whose next product may go into the launch of a plain one."""
        if isinstance(x, NormedRows):
            if self._skinny_ok(x.rows, w, bias):
                N = w.shape[0] // 2 if act in self.GLU_ACTS else w.shape[0]
                out = torch.empty(x.shape[0], N, device=x.device, dtype=torch.float32 if out_f32 else x.dtype)
                self._moe_lib.skinny_linear_normed(out, x.rows, x.squares, x.eps, w, bias, -1 if act is None else self.ACTIVATIONS[act], c0, c1, act_from)
                return out
            x = x.normed()
        if (x.dim() == 2 and x.shape[0] <= self.SKINNY_ROWS and self._skinny_ok(x, w, bias)
                and self.skinny_pays(x.shape[0], w.shape[0], w.shape[1], act in self.GLU_ACTS, x.dtype == torch.float32, act is not None)):
            if beside is not None and bias is None and act is None and not out_f32:
                out = self._linear_beside(x, w, beside)
                if out is not None:
                    return out
            return self._skinny_linear(x, w, bias, out_f32, act, c0, c1, act_from)
        if out_f32 and x.dtype != torch.float32:
            y = torch.mm(x, w.t(), out_dtype=torch.float32)
            if bias is not None:
                y += bias
        else:
            y = self._vendor_linear(x, w, bias)
        if act is None:
            return y
        if act_from:
            self.activation(y[:, act_from:], y[:, act_from:], act, c0, c1)
            return y
        out = torch.empty(*y.shape[:-1], y.shape[-1] // 2, device=y.device, dtype=y.dtype) if act in self.GLU_ACTS else y
        return self.activation(out, y, act, c0, c1)

    def in_rounds(self, x, before, cols, biased=True) -> bool:
        """Whether rows x onto ``before`` columns and so many further ones, which have no biases or some of which have (``biased``), are faster as a product each than as
        one, in rounds of tiles that they fill better."""
        if len(x.shape) != 2 or not x.shape[0] or x.dtype not in (torch.bfloat16, torch.float32):
            return False
        rows, k = x.shape
        if (isinstance(x, torch.Tensor) and x.dtype == torch.bfloat16 and before % 256 == 0 and -(-rows // 256) * before // 256 % 256 == 0
                and gemm.round_columns(rows, cols, k) > 0):
            return True   # whole rounds, and a product that is cut where rounds end
        return k >= 512 and self.two_pay(rows, before, cols, k, biased, x.dtype == torch.float32)   # (shorter ones were not measured)

    def _two_pay(self, rows, before, cols, k, biased, f32) -> bool:
        """``in_rounds`` by estimates. Up to 64 rows, by the time of the own kernel, whose workgroups over the sum of the columns may be a round that neither half starts (or the
        vendor's product is to run). Else by rounds of tiles of 256 x 256, 256 at a time: one product where it saves a round and is up to two of them, not of halves that
        fill one by themselves, or three to four; above 5000 rows two, as rounds are many. In 32 bits the vendor's tiles are smaller, and one is taken where it saves
        a round of 64 x 64. Time against two products always, of parallel mixers' widths (k 512 - 4096, 384 - 37000 columns), one product always / as chosen here: 9973
        sizes of up to 64 rows -23 / -23 %, 53 / 4 of them more than 3 % longer, up to 16 / 4; 2898 of 65 - 8192 rows -14 / -16 %, 451 / 11, up to 56 / 19 (35 us); in 32 bits 2533
        of up to 64 rows -17 / -18 %, 229 / 24, up to 38 / 11, 1001 of 65 - 2048 rows -7 / -7 %, 224 / 54, up to 50 / 50 (65 rows of k 4096). us, two / one: 4073 rows of 3840 +
        7808 x 3072 231 / 334, 3000 of 1280 + 10304 x 2048 137 / 169, 33 of 10240 + 10304 x 4096 40.8 / 46.9, 4096 of 4608 + 10256 x 2048 264 / 205."""
        both = before + cols
        if rows <= self.SKINNY_ROWS and (f32 or self.skinny_pays(rows, before, k) and self.skinny_pays(rows, cols, k)):
            apart = self._skinny_time(rows, before, k, False, f32) + self._skinny_time(rows, cols, k, False, f32)
            return self._skinny_time(rows, both, k, False, f32) > (0.975 if self.skinny_pays(rows, both, k, False, f32) else 0.925) * apart
        tile = 64 if f32 else 256
        left, right, one = (-(-rows // tile) * -(-n // tile) / 256 for n in (before, cols, both))
        saves = math.ceil(one) < math.ceil(left) + math.ceil(right)
        if f32:
            return not saves
        if not biased and gemm.round_columns(rows, both, k) > 0:
            return rows > 5000
        return rows > 5000 or not (saves and (one <= 1 or one <= 2 and max(left, right) > 1.1 or 3 < one <= 4))

    def _vendor_linear(self, x, w, bias):
        y = gemm.linear_in_rounds(x, w) if bias is None and x.dim() == 2 else None
        return F.linear(x, w, bias) if y is None else y

    def _skinny_linear(self, x, w, bias, out_f32=False, act=None, c0=0.0, c1=0.0, act_from=0):
        out = torch.empty(x.shape[0], w.shape[0] // 2 if act in self.GLU_ACTS else w.shape[0], device=x.device,
                          dtype=torch.float32 if out_f32 else x.dtype)
        self._moe_lib.skinny_linear(out, x, w, bias, -1 if act is None else self.ACTIVATIONS[act], c0, c1, act_from)
        return out

    NORM_ROWS = 32   # rows that ``linear_update`` takes

    def _update_pays(self, rows, cols, k, f32) -> bool:
        """Whether a residual update and norm go into the products around them: what their launch costs in a captured step (2.5 us, and 0.05 per
        row and 1024 columns) is weighed against k in parts (``linear_parts``), which needs it, against the loads that both products do more, and
        against what the next product, taken to be of three times the columns, loses where the vendor's GEMM would be the one to run."""
        apart = min(self._vendor_time(rows, cols, k, f32), min(self._parts_time(rows, cols, k, f32, p) for p in (1, 2, 4)))
        after = max(0.0, self._skinny_time(rows, 3 * cols, cols, False, f32) - self._vendor_time(rows, 3 * cols, cols, f32))
        return self._skinny_time(rows, cols, k, False, f32) + 0.6 + after <= apart + 2.5 + 0.05 * rows * cols / 1024

    @staticmethod
    def _update_cols(rows, cols, k, f32) -> int:
        """Columns that a workgroup of the update takes, and that a sum of squares is over: as skinny_half (skinny_linear.hip) has it for
        up to 32 rows."""
        return 8 if cols <= 2048 and k * (2 if f32 else 1) > (4096 if rows <= 8 and cols <= 1024 else 1024) else 16

    def linear_update(self, x, w, bias, residual, norm_w, eps, conv=None):
        """residual += x . w^T + bias, and the rows for the next products as ``NormedRows`` of its norm; None, and nothing done, where the
        update and norm are a launch of their own (``update_pays``). ``conv``: a ``ConvBeside`` that the launch may take, but for 17 rows and
        more of 32 bits from k 2048 on whose workgroups take 8 columns: of 1025 such sizes 633 took 1 - 11 % longer in one launch (22 rows of
        2048 x 4096, 8192 channels, 16.9 -> 18.6 us). Of 31991 others 55 took more than 1 % longer, three of them 5, 7 and 15, and all 23 % less on average."""
        T, N, K = x.shape[0], w.shape[0], w.shape[1]
        if not (0 < T <= self.NORM_ROWS and N % 64 == 0 and N <= 4096 and self.update_pays(T, N, K, x.dtype == torch.float32)
                and self._skinny_ok(x, w, bias) and residual.is_contiguous() and residual.data_ptr() % 16 == 0):
            return None
        cols = self.update_cols(T, N, K, x.dtype == torch.float32)
        rows, squares = torch.empty(T, N, device=x.device, dtype=x.dtype), torch.empty(T, N // cols, device=x.device, dtype=torch.float32)
        product = (rows, squares, residual, norm_w, x, w, bias)
        if conv is None or (x.dtype == torch.float32 and T > 16 and cols == 8 and K >= 2048) or not conv.take(lambda *c: self._delta.skinny_update_conv(*product, *c)):
            self._moe_lib.skinny_linear_update(*product)
        return NormedRows(rows, squares, eps)

    def linear_heads(self, out, x, w) -> bool:
        """out[h] = x[h] . w[h]^T for a few bf16 rows (x [heads, T, K], w [heads, N, K], out [heads, T, N], strided rows);
        False, and nothing done, where the vendor's batched GEMM is the one to run."""
        if not (x.dim() == 3 and x.dtype == torch.bfloat16 and self._skinny_ok(x, w) and self.skinny_pays(x.shape[1], w.shape[0] * w.shape[1], w.shape[2])):
            return False
        self._moe_lib.skinny_linear(out, x, w, None, -1, 0.0, 0.0)
        return True

    ACTIVATIONS = {"tanh": 0, "xielu": 1, "relu2": 2, "silu_mul": 3, "clamped_glu": 4, "softcap": 5}

    def activation(self, out, x, kind, c0=0.0, c1=0.0):
        self._window_lib.activation(out, x, self.ACTIVATIONS[kind], c0, c1)
        return out

    def add_normed(self, out, residual, y, w, eps, moe=None):
        if moe is None:
            self._delta.add_normed(out, residual, w, eps, y, None, None, None, None, 0, None, None)
        else:
            ye, pair_slot, ids, wts, E, h, shared = moe
            self._delta.add_normed(out, residual, w, eps, None, ye, pair_slot, ids, wts, E, h, shared)
        return out

    def token_shift(self, out, x, state, mu, meta):
        self._delta.token_shift(out, x, state, mu, meta.seq_cu, meta.seq_ctx, meta.seq_state)

    def wkv(self, out, state, proj, wl, w0, u, norm_w, sp, eps, meta):
        scratch = torch.empty(proj.shape[1] * (5 * sp.size + sp.heads), device=proj.device, dtype=torch.float32)
        self._delta.wkv(out, state, proj, wl, w0, u, norm_w, meta.seq_cu, meta.seq_ctx, meta.seq_state, scratch,
                        sp.heads, sp.dim, eps)

    def wkv_step(self, out, state, proj, low, w2, w0, u, norm_w, sp, eps, meta):
        """``wkv`` for steps in which every sequence has one row (``meta.max_q`` == 1), the decay bottleneck's
        tanh and up-projection included (``low``: its output before the tanh): one launch."""
        self._delta.wkv_step(out, state, proj, low, w2, w0, u, norm_w, meta.seq_cu, meta.seq_ctx, meta.seq_state,
                             sp.heads, sp.dim, eps)

    ROUTER_MAX_OUTPUTS = 256

    def route_topk(self, ids, wts, logits, correction, top, scale, E, groups=1, keep_groups=1, renorm=False,
                   score="softmax", group_top2=False):
        if logits.shape[1] > self.ROUTER_MAX_OUTPUTS or groups > 64:
            # more router outputs than a wave holds: device-side torch ops
            ref.route_topk(ids, wts, logits, correction, top, scale, E, groups, keep_groups, renorm, score, group_top2)
            return
        self._window_lib.route_topk(ids, wts, logits, correction, top, scale, E, groups, keep_groups, renorm,
                                    score == "sigmoid", group_top2)

    ROUTE_ALIGN_PAIRS, ROUTE_ALIGN_SLOTS = 256, 8192   # batches whose router and alignment run in one launch

    def route_align(self, ids, wts, slots, tile_expert, pair_slot, logits, correction, top, scale, E, nb, tile, groups=1,
                    keep_groups=1, renorm=False, score="softmax", group_top2=False):
        """``route_topk`` and ``moe_align`` (``nb`` buckets) of the choices."""
        if (ids.numel() <= self.ROUTE_ALIGN_PAIRS and slots.numel() <= self.ROUTE_ALIGN_SLOTS and nb <= 128 and groups <= 64
                and logits.shape[1] <= self.ROUTER_MAX_OUTPUTS and self._window_lib is self._moe_lib):
            self._window_lib.route_align(ids, wts, slots, tile_expert, pair_slot, logits, correction, top, scale, E, nb, tile,
                                         groups, keep_groups, renorm, score == "sigmoid", group_top2)
            return
        self.route_topk(ids, wts, logits, correction, top, scale, E, groups, keep_groups, renorm, score, group_top2)
        self.moe_align(ids.view(-1), nb, tile, slots, tile_expert, pair_slot)

    # ---- parallel blocks with gated sublayer results, mLSTM, PolyNorm (csrc/kernels/seq/gated_block.hip, mlstm.hip,
    # elementwise.hip)
    def gated_add_norms(self, out1, out2, residual, w1, w2, eps, first=None, second=None):
        """``first`` / ``second``: (y, g, b) of a sublayer, y its result rows or, for a mixture of experts,
        (ye, pair_slot, wts, shared)."""
        y1, g1, b1 = first if first is not None else (None, None, None)
        y2, g2, b2 = second if second is not None else (None, None, None)
        parts = (None, None, None, None)
        if isinstance(y2, tuple):
            parts, y2 = y2, None
        self._cell.gated_add_norms(out1, out2, residual, w1, w2, eps, y1, g1, b1, y2, g2, b2, *parts)

    def polynorm(self, out, x, coef, eps):
        self._cell.polynorm(out, x, coef, eps)
        return out

    def gate_mul(self, out, x, gate):
        self._cell.gate_mul(out, x, gate)
        return out

    def mlstm(self, out, state, proj, gates, b_if, norm_w, sp, eps, meta):
        scratch = torch.empty(proj.shape[0] * sp.heads * (2 * sp.dim + 2 * sp.vdim + 6), device=proj.device,
                              dtype=torch.float32)
        self._cell.mlstm(out, state[0], state[1], state[2], proj, gates, b_if, norm_w, meta.seq_cu, meta.seq_ctx,
                         meta.seq_state, scratch, sp.heads, sp.dim, sp.vdim, sp.gate_cap, eps, meta.max_q == 1)

    @property
    def _moe_lib(self):
        """The library whose copy of the expert alignment and expert GEMMs runs (the one the model loads anyway)."""
        return self._lib(self.norm_library)

    def moe_align(self, experts, E, tile, slots, tile_expert, pair_slot):
        if E <= 128:
            self._moe_lib.moe_align(experts, E, tile, slots, tile_expert, pair_slot)
            return
        # more experts than the alignment kernel's LDS tables hold: the same layout from device-side
        # sort / scan ops (no host round trip)
        ex = experts.long()
        P = ex.numel()
        order = torch.argsort(ex, stable=True)
        counts = torch.bincount(ex, minlength=E)
        padded = (counts + tile - 1) // tile * tile
        ends = torch.cumsum(padded, 0)
        first = torch.cumsum(counts, 0) - counts           # rank of each expert's first pair in `order`
        e_sorted = ex[order]
        pos = (ends - padded)[e_sorted] + torch.arange(P, device=ex.device) - first[e_sorted]
        slots.fill_(-1)
        slots[pos] = order.to(torch.int32)
        pair_slot[order] = pos.to(torch.int32)
        t = torch.arange(tile_expert.numel(), device=ex.device) * tile
        te = torch.searchsorted(ends, t, right=True)
        tile_expert.copy_(torch.where(te < E, te, torch.full_like(te, -1)).to(torch.int32))

    def moe_tables_align_ok(self, tables, tokens, E) -> bool:
        """Whether ``moe_table_align`` takes ``tables`` [(layers,) rows, top] in one launch, with a row of outputs per table."""
        return E <= 128 and tokens.dtype == torch.long and tokens.is_contiguous() and self._moe_lib.moe_align_small(tokens.numel() * tables.shape[-1])

    def moe_table_align(self, table, tokens, E, tile, slots, tile_expert, pair_slot, num_tiles=None, order=None, per_round=(), across=()):
        """``moe_align`` of the experts table[tokens] [T, top]: one launch for small batches. ``table`` may hold the tables of several
        layers, and ``num_tiles`` (the tiles in use) and ``order`` (for GEMMs of ``across`` tiles for each of these, or of one, that
        take ``per_round`` tiles at once, a row each; one table) be asked for, where ``moe_tables_align_ok`` says so."""
        if self.moe_tables_align_ok(table, tokens, E):
            self._moe_lib.moe_table_align(table, tokens, E, tile, slots, tile_expert, pair_slot, num_tiles, order, list(per_round), list(across))
        else:
            assert table.dim() == 2 and num_tiles is None and order is None, "the tables of several layers: small batches"
            self.moe_align(table.index_select(0, tokens).view(-1), E, tile, slots, tile_expert, pair_slot)

    def expert_gemm(self, out, x, w, slots, tile_expert, tile, gather_k, act, row_scale=None, limit=0.0, pairs=0, tiles=0):
        """act: False / 0 none, True / 1 squared ReLU, 2: w = [gate rows; up rows], out = silu(gate) * up, 3: the same
        with the gate clamped at ``limit``; ``row_scale`` fp32 [pairs] multiplies each pair's product before it;
        ``pairs``: how many (token, choice) pairs the tiles hold, where the caller knows (the choice of kernel); ``tiles``: the tiles in use are
        among the first so many, as the alignments leave them with a pair in each (the rest is not launched)."""
        self._moe_lib.expert_gemm(out, x, w, slots, tile_expert, tile, gather_k, int(act), row_scale, limit, pairs, tiles)

    def _expert_plan(self, pairs: int, experts: int, ff: int, hidden: int, may_pack: bool) -> str:
        """How a prompt's two expert products, [ff, hidden] and back, are expected to be fastest in bf16: "rows" (tiles of 32, the kernel for few rows),
        "tiles" (of 128; from 16 pairs per expert on, and below 128 of them if 7 % faster by the model than 32) or, with ``may_pack``, "packed" (the grouped GEMM
        over packed weights), in us of a model of each: a latency and the larger of the weights at 4.4 or 5.2 TB/s and what a compute unit takes in, per workgroup
        rows and columns times k; rounds of 512 columns x 128 rows for packed ones, half a round up to 64 of them, whose columns go to workgroups of their own. Of
        1000 sizes where the choice is tiles (4 - 128 experts, 512 x 512 to 4096 x 4096, 65 - 8200 tokens, even and uneven) they take 0.64 of the time of tiles of
        32 and 0.74 of packed weights' on average, and 3 - 12 % more in one of a hundred. What the bounds leave out, us: 10 - 15 pairs each gain 5 %
        on average, but 24 experts of 2048 x 4096, 13 pairs each, 162 -> 182; 6 of 896 x 4096, 74 each, 44 -> 51; 12 of 4096 x 768, 257 each, packed 89, tiles 111.
        Up to two rounds of workgroups of a long k count as 1.6 at least: 4 of 2816 x 512, 1201 each, packed 69, tiles 84.
        us rows / tiles / packed of both: 16 experts of 1024 x 2048, 87, 250, 350 pairs each 76 / 39 / -, 167 / 82 / 96, 222 / 100 / 97; 8 of 512 x 1024, 75, 175,
        1000 each 13.6 / 15.9 / -, 24 / 20 / 24, 103 / 39 / 59."""
        each = pairs / experts

        def rows(n, k):
            tiles, r = experts * max(1.0, each / 32 + 0.5), min(32.0, 8 * math.ceil(each / 8))
            return 2.2 + max(2e-6 * experts * n * k / 4.4, n / 16 * tiles * 2e-3 * k * (16 + r) / 256 / 70)

        def tiles(n, k):
            wgs = math.ceil(n / 64) * experts * max(1.0, each / 128 + (0.5 if each > 96 else 0.0))
            r = min(128.0, 32 * math.ceil(each / 32))
            rounds = max(1.0, wgs / 256, 1.6 if wgs > 256 and k >= 2048 else 0.0)   # a second one is not hidden where there are no more
            return 2.5 + max(2e-6 * experts * n * k / 5.2, rounds * 2e-3 * k * (64 + r) / (42 if wgs <= 256 else 50))

        def packed(n, k):
            t = math.ceil(n / 512) * experts * (each / 128 + 0.5)
            whole, left = divmod(t, 256)
            return 9 + whole * 24e-3 * k + (0 if left == 0 else min(24e-3 * k, 10) if whole and left <= 48 else (24e-3 if t > 64 else 12e-3) * k)

        def both(f):
            return f(ff, hidden) + f(hidden, ff)
        options = [(both(rows), "rows")] + ([(both(tiles), "tiles")] if each >= 16 and both(tiles) < (0.93 if each < 128 else 1.0) * both(rows) else [])
        options += [(both(packed), "packed")] if may_pack else []
        return min(options)[1]

    # ---- norms before and after every sublayer (csrc/kernels/seq/sandwich.hip)
    def sandwich_update(self, out, residual, w_next, eps, y=None, w_post=None, mult=1.0, table=None):
        rows, ids, scale = table if table is not None else (None, None, 1.0)
        a = a_w = b = b_w = ye = pair_slot = wts = shared = gate = None
        a_scale = b_scale = 1.0
        if isinstance(y, tuple) and len(y) == 6:
            a, a_w, b, b_w, a_scale, b_scale = y
        elif isinstance(y, tuple):
            ye, pair_slot, wts, shared, gate = y
        else:
            a = y
        self._delta.sandwich_update(out, residual, w_next, eps, w_post, mult, rows, ids, scale, a, a_w, b, b_w, a_scale,
                                    b_scale, ye, pair_slot, wts, shared, gate)
        return out

    # ---- residual streams, lightning attention (csrc/kernels/seq/streams.hip, lightning.hip)
    def stream_update(self, out, dst, src, coef, w, eps, y1=None, y2=None):
        """``src``: the streams, or (table, ids, scale): all of them equal the embedding ``scale * table[ids]``. ``y2``: a
        sublayer's result rows or, for a mixture of experts, (ye, pair_slot, wts or top, shared, gate)."""
        table = ids = None
        scale = 1.0
        if isinstance(src, tuple):
            table, ids, scale = src
            src = None
        ye = pair_slot = wts = shared = gate = None
        top = 0
        if isinstance(y2, tuple):
            ye, pair_slot, wts, shared, gate = y2
            top, wts = (wts, None) if isinstance(wts, int) else (wts.shape[1], wts)
            y2 = None
        self._stream.stream_update(out, dst, src, table, ids, scale, coef, w, eps, y1, y2, ye, pair_slot, wts, top, shared, gate)
        return out

    # bf16 prompt portions run the chunked matrix-core kernel (HIPSERVE_LIGHTNING_MFMA=0: the scan, as fp32 does)
    LIGHTNING_MFMA = os.environ.get("HIPSERVE_LIGHTNING_MFMA", "1") != "0"
    LIGHTNING_SEGMENT = 256    # tokens per segment of long portions (a multiple of 64) ...
    LIGHTNING_FILL = 1024      # ... while fewer (sequence, head, 32-column block) workgroups than this would run

    def lightning(self, out, S, proj, powers, norm_w, sp, eps, meta, out_scale=1.0):
        """Prompt portions (the step's first sequences) run the chunked kernel or the scan, decode rows the
        one-row kernel; one launch norms and gates the concatenated heads of all rows."""
        nd, nseq = meta.num_decode, meta.seq_ctx.shape[0]
        npf = nseq - nd
        T = proj.shape[0]
        mfma = (npf > 0 and self.LIGHTNING_MFMA and proj.dtype == torch.bfloat16
                and self._stream.lightning_mfma_ok(sp.dim, sp.vdim, proj.stride(0), proj.storage_offset()))
        rows = meta.num_prefill_tokens if npf and not mfma else 0   # the scan reads them as dense fp32 rows
        nseg, seg = 1, self.LIGHTNING_SEGMENT
        blocks = npf * sp.heads * -(-sp.vdim // 32)
        if mfma and meta.max_q >= 2 * seg and blocks < self.LIGHTNING_FILL:
            while blocks * -(-meta.max_q // seg) > 4 * self.LIGHTNING_FILL:
                seg *= 2
            nseg = -(-meta.max_q // seg)
        extra = npf * nseg * sp.heads * sp.dim * sp.vdim if nseg > 1 else rows * sp.heads * (2 * sp.dim + sp.vdim)
        scratch = torch.empty(T * sp.out_size + extra, device=proj.device, dtype=torch.float32)
        self._stream.lightning(out, S, proj, powers, norm_w, meta.seq_cu, meta.seq_ctx, meta.seq_state, scratch, npf,
                               meta.num_prefill_tokens, sp.heads, sp.dim, sp.vdim, eps, out_scale, mfma,
                               nseg, seg, meta.max_q)


class ReferenceOps:
    """PyTorch reference path (CPU plumbing engine / numerics oracle)."""

    name = "reference"

    def in_rounds(self, x, before, cols, biased=True) -> bool:
        return False

    def fill_uniform(self, out, row0, col0, gcols, key, scale):
        return ref.fill_uniform(out, row0, col0, gcols, key, scale)

    def rmsnorm(self, out, x, w, eps, out8=None):
        assert out8 is None, "the FP8 copy is a HIP-kernel output"
        out.copy_(ref.rmsnorm(x, w, eps))
        return out

    def fused_add_rmsnorm(self, out, x, residual, w, eps, out8=None):
        assert out8 is None, "the FP8 copy is a HIP-kernel output"
        y, r = ref.fused_add_rmsnorm(x, residual, w, eps)
        residual.copy_(r)
        out.copy_(y)
        return out

    def silu_and_mul(self, out, x):
        out.copy_(ref.silu_and_mul(x))
        return out

    def gelu_and_mul(self, out, x):
        out.copy_(ref.gelu_and_mul(x))
        return out

    def qk_rmsnorm(self, qkv, q_w, k_w, nq, nkv, D, eps):
        ref.qk_rmsnorm(qkv, q_w, k_w, nq, nkv, D, eps)

    def rope_cache(self, qkv, positions, slots, cos_sin, k_cache, v_cache, nq, nkv, D, mode):
        ref.rope_cache(qkv, positions, slots, cos_sin, k_cache, v_cache, nq, nkv, D, mode)

    def paged_decode(self, out, q, k_cache, v_cache, block_tables, context_lens, tmp_out, tmp_ml,
                     nq, nkv, part_size, scale, window=0, out16=None):
        B = context_lens.shape[0]
        D = k_cache.shape[3]
        out[:B, : nq * D].copy_(ref.paged_decode(q, k_cache, v_cache, block_tables, context_lens,
                                                 nq, nkv, scale, window).view(B, nq * D))
        return out

    def prefill_attention(self, out, q, k_cache, v_cache, block_tables, cu_q, ctx_lens, tiles,
                          nq, nkv, scale, window=0):
        D = k_cache.shape[3]
        T = int(cu_q[-1])
        out[:T, : nq * D].copy_(ref.prefill_attention(q, k_cache, v_cache, block_tables, cu_q,
                                                      ctx_lens, nq, nkv, scale, window).view(T, nq * D))
        return out

    def penalty_apply(self, logits, slot, pres, freq, rep, counts, seen):
        ref.penalty_apply(logits, slot, pres, freq, rep, counts, seen)

    def penalty_update(self, tok, slot, counts, seen):
        ref.penalty_update(tok, slot, counts, seen)

    def penalty_init(self, counts, seen, slots, off, n_prompt, toks):
        ref.penalty_init(counts, seen, slots, off, n_prompt, toks)

    def top_logprobs(self, logits, nreq, out_ids, out_lp):
        ref.top_logprobs(logits, nreq, out_ids, out_lp)

    # ---- vision tower (Qwen3-VL ViT)
    def layernorm(self, out, x, w, b, eps, residual=None):
        if residual is None:
            out.copy_(ref.layernorm(x, w, b, eps))
        else:
            y, r = ref.add_layernorm(x, residual, w, b, eps)
            residual.copy_(r)
            out.copy_(y)
        return out

    def gelu_(self, x, tanh):
        x.copy_(ref.gelu(x, tanh))
        return x

    def vision_attention(self, out, qkv, cos_sin, cu_seqlens, nh, D, scale, meta=None):
        ref.vision_rope(qkv, cos_sin, nh, D)
        out.copy_(ref.vision_attention(qkv, cu_seqlens, nh, D, scale))
        return out

    # ---- layer-list decoders (models/mixers.py)
    def scaled_add_group_rmsnorm(self, out, residual, w, groups, eps, mix=None, ls1=None, y=None, pair_slot=None,
                                 top=0, ls2=None, extra=None, table=None, ids=None):
        ref.scaled_add_group_rmsnorm(out, residual, w, groups, eps, mix, ls1, y, pair_slot, top, ls2, extra, table, ids)
        return out

    def latent_prepare(self, cq, cache, proj, positions, slots, q_norm, kv_norm, inv_freq, q_rank, kv_rank,
                       rot_dim, eps):
        ref.latent_prepare(cq, cache, proj, positions, slots, q_norm, kv_norm, inv_freq, q_rank, kv_rank, rot_dim, eps)

    def latent_attention(self, o_lat, q_abs, q, proj, cache, meta, inv_freq, heads, dim, rot_dim, kv_rank,
                         gate_off, scale, window):
        ref.latent_attention(o_lat, q_abs, q, proj, cache, meta.seq_cu, meta.seq_ctx, meta.seq_bt, inv_freq,
                             heads, dim, rot_dim, kv_rank, gate_off, scale, window)

    def latent_query_in_place(self, dtype, kv_rank, rot_dim) -> bool:
        return False

    def latent_prompt_rows(self, dtype, sp, nfreq, cache, meta, T) -> int:
        return 0

    def mingru_product(self, y, state, x, w, b_z, b_x, meta, beside=None) -> bool:
        return False

    def mingru_scan(self, y, state, proj, b_z, b_x, meta):
        ref.mingru_scan(y, state, proj, b_z, b_x, meta.seq_cu, meta.seq_ctx, meta.seq_state)

    def moe_align(self, experts, E, tile, slots, tile_expert, pair_slot):
        ref.moe_align(experts, E, tile, slots, tile_expert, pair_slot)

    def moe_tables_align_ok(self, tables, tokens, E) -> bool:
        return False

    def moe_table_align(self, table, tokens, E, tile, slots, tile_expert, pair_slot):
        ref.moe_align(table.index_select(0, tokens).view(-1), E, tile, slots, tile_expert, pair_slot)

    def expert_gemm(self, out, x, w, slots, tile_expert, tile, gather_k, act, row_scale=None, limit=0.0, pairs=0, tiles=0):
        ref.expert_gemm(out, x, w, slots, tile_expert, tile, gather_k, int(act), row_scale, limit)

    def stream_update(self, out, dst, src, coef, w, eps, y1=None, y2=None):
        ref.stream_update(out, dst, src, coef, w, eps, y1, y2)
        return out

    def lightning(self, out, S, proj, powers, norm_w, sp, eps, meta, out_scale=1.0):
        ref.lightning(out, S, proj, powers[:, 1], norm_w, sp, eps, meta.seq_cu, meta.seq_ctx, meta.seq_state, out_scale)

    def attn_prepare(self, proj, cache, meta, inv_freq, sp, q_norm, k_norm, eps):
        ref.attn_prepare(proj, cache, meta.positions, meta.slot_mapping, inv_freq, sp, q_norm, k_norm, eps)

    def window_attention(self, out, proj, cache, meta, sp, gate_off, out_scale=1.0, lam=0.0, eps=0.0, sink_w=None):
        ref.window_attention(out, proj, cache, meta.seq_cu, meta.seq_ctx, meta.seq_bt, sp, gate_off, out_scale, lam, eps,
                             sink_w)

    def gated_add_norms(self, out1, out2, residual, w1, w2, eps, first=None, second=None):
        ref.gated_add_norms(out1, out2, residual, w1, w2, eps, first, second)

    def polynorm(self, out, x, coef, eps):
        ref.polynorm(out, x, coef, eps)
        return out

    def gate_mul(self, out, x, gate):
        ref.gate_mul(out, x, gate)
        return out

    def mlstm(self, out, state, proj, gates, b_if, norm_w, sp, eps, meta):
        ref.mlstm(out, state[0], state[1], state[2], proj, gates, b_if, norm_w, sp, eps, meta.seq_cu, meta.seq_ctx,
                  meta.seq_state)

    def add_normed(self, out, residual, y, w, eps, moe=None):
        ref.add_normed(out, residual, y, w, eps, moe)
        return out

    def token_shift(self, out, x, state, mu, meta):
        ref.token_shift(out, x, state, mu, meta.seq_cu, meta.seq_ctx, meta.seq_state)

    def wkv(self, out, state, proj, wl, w0, u, norm_w, sp, eps, meta):
        ref.wkv(out, state, proj, wl, w0, u, norm_w, sp, eps, meta.seq_cu, meta.seq_ctx, meta.seq_state)

    def wkv_step(self, out, state, proj, low, w2, w0, u, norm_w, sp, eps, meta):
        t = torch.tanh(low.float()).to(low.dtype)
        wl = torch.nn.functional.linear(t.float(), w2.float())
        ref.wkv(out, state, proj, wl, w0, u, norm_w, sp, eps, meta.seq_cu, meta.seq_ctx, meta.seq_state)

    def route_topk(self, ids, wts, logits, correction, top, scale, E, groups=1, keep_groups=1, renorm=False,
                   score="softmax", group_top2=False):
        ref.route_topk(ids, wts, logits, correction, top, scale, E, groups, keep_groups, renorm, score, group_top2)

    def route_align(self, ids, wts, slots, tile_expert, pair_slot, logits, correction, top, scale, E, nb, tile, groups=1,
                    keep_groups=1, renorm=False, score="softmax", group_top2=False):
        ref.route_topk(ids, wts, logits, correction, top, scale, E, groups, keep_groups, renorm, score, group_top2)
        ref.moe_align(ids.view(-1), nb, tile, slots, tile_expert, pair_slot)

    def gated_delta(self, y, state, proj, conv_w, a_log, dt_bias, norm_w, decay, gate, offs, sp, eps, meta):
        ref.gated_delta(y, state[0], state[1], proj, conv_w, a_log, dt_bias, norm_w, decay, gate, offs, sp, eps,
                        meta.seq_cu, meta.seq_ctx, meta.seq_state)

    def conv_beside(self):
        return None

    def gated_delta_step(self, y, state, proj, conv_w, a_log, dt_bias, norm_w, w_a2, w_g2, offs, sp, eps, meta, conv=None):
        decay = gate = None
        if sp.channel_decay:
            low_a, low_g = (proj[:, o:o + w.shape[1]].float() for o, w in ((offs[0], w_a2), (offs[1], w_g2)))
            decay = torch.nn.functional.linear(low_a, w_a2.float())
            gate = torch.nn.functional.linear(low_g, w_g2.float())
        ref.gated_delta(y, state[0], state[1], proj, conv_w, a_log, dt_bias, norm_w, decay, gate, offs, sp, eps,
                        meta.seq_cu, meta.seq_ctx, meta.seq_state)

    def sandwich_update(self, out, residual, w_next, eps, y=None, w_post=None, mult=1.0, table=None):
        ref.sandwich_update(out, residual, w_next, eps, y, w_post, mult, table)
        return out

    def delta_rule_low(self, out, state, proj, w2, a_b, w0, norm_w, sp, eps, meta, out_scale=1.0) -> bool:
        return False

    def window_step(self, out, proj, cache, meta, inv_freq, sp, q_norm, k_norm, eps, gate_off, out_scale=1.0, sink_w=None, beside=None) -> bool:
        return False

    def delta_beside(self, *args):
        return None

    def delta_rule(self, out, state, proj, wl, a_b, w0, norm_w, sp, eps, meta, out_scale=1.0):
        ref.delta_rule(out, state[0], proj, wl, a_b, w0, norm_w, sp, eps, meta.seq_cu, meta.seq_ctx,
                       meta.seq_state, out_scale)

    def linear(self, x, w, bias=None, out_f32=False, act=None, c0=0.0, c1=0.0, act_from=0, beside=None):
        if out_f32 and x.dtype != torch.float32:
            x, w, bias = x.float(), w.float(), None if bias is None else bias.float()
        y = F.linear(x, w, bias)
        if act is None:
            return y
        if act_from:
            self.activation(y[:, act_from:], y[:, act_from:], act, c0, c1)
            return y
        out = y.new_empty(*y.shape[:-1], y.shape[-1] // 2) if act in KernelOps.GLU_ACTS else y
        return self.activation(out, y, act, c0, c1)

    def linear_parts(self, x, w, bias=None, beside=None):
        return self.linear(x, w, bias)

    def linear_update(self, x, w, bias, residual, norm_w, eps, conv=None):
        return None

    def linear_heads(self, out, x, w) -> bool:
        return False

    def activation(self, out, x, kind, c0=0.0, c1=0.0):
        ref.activation(out, x, kind, c0, c1)
        return out

    def sample(self, out_tok, out_lp, logits, temperature, top_k, top_p, seeds, steps, two_rounds=True):
        t, lp = ref.sample(logits, temperature, top_k, top_p, seeds, steps, bf16_row=False)
        n = t.shape[0]
        out_tok[:n].copy_(t)
        if out_lp.numel():
            out_lp[:n].copy_(lp)


def get_ops(device: torch.device | str):
    device = torch.device(device)
    if device.type == "cuda":
        return KernelOps()
    return ReferenceOps()
