"""What the runners over a HybridCache share: step buffers, the grouping of a step's rows, and the sublayers that more than one design is
made of - rotated attention over [values | keys] rows, latent attention, the gated delta rule, gated linear attention, clamped and mixture
feed-forwards - each with its options as parameters.
A design's own file holds its weight layout, its residual and the order in which its sublayers run."""
from __future__ import annotations

import os
from contextlib import contextmanager, nullcontext
from typing import Callable, Dict, Optional

import torch

from . import ops_dense as D
from .ops import upload

NO_WORK: Dict[tuple, torch.Tensor] = {}     # a step whose scans take no workspace (_scan_work)
UNIT_EPS = 1e-6     # inside the root of the delta rule's unit vectors: a constant of the mechanism, not of a checkpoint


def pad8(n: int) -> int:
    return (int(n) + 7) // 8 * 8


class HybridRunner:
    MAX_BUFFER_SETS = int(os.environ.get("I64H_MAX_BUFFER_SETS", "8"))
    ATTN_MAX_SEGMENTS = 4
    ATTN_WAVES = {64: 3072, 128: 2048, 256: 1024}     # waves a decode-sized attention launch aims at, by the width of a key head's cached part
    BUFFERS: Optional[Callable] = None                # (runner, rows, logit rows) -> the step's buffers
    SIDE_STREAM = False                               # a second stream for a sublayer that runs beside another one

    def _init_runner(self, cfg, device, dtype: str) -> None:
        if dtype not in ("bfloat16", "float32"):
            raise ValueError(f"dtype {dtype}: bfloat16 or float32")
        self.cfg, self.device, self.dtype = cfg, torch.device(device), dtype
        self.exact = dtype == "float32"
        self._bufs: Dict[tuple, object] = {}
        self._pinned: set = set()
        self._arange: Dict[int, torch.Tensor] = {}
        self.max_ff = 0      # the widest feed-forward's inner rows
        self.side = torch.cuda.Stream(device=self.device) if self.SIDE_STREAM and self.device.type == "cuda" else None

    # ---- two sublayers side by side ----
    # Eager steps of little work (rows times the square of the width, twice as much with 32-bit products) are bound by the host, and the events of a fork and its
    # meeting take 40 to 65 us of it.  Microseconds a step of two blocks, forked | not, on a host that needs 1200 to 1300 for its launches: width 1024, Vepelix
    # 600 rows 2200 | 1560, 1024 2300 | 1724, 1536 2354 | 2117, 2048 in four prompts 2450 | 2182, in one 2893 | 3074, 3072 2909 | 3005; Pukatar 1024 1696 | 1385, 1536 1784 |
    # 1698, 2048 1700 | 1808, 2285 | 2440; width 2048, 200 rows 2160 | 1610 and 1673 | 1382, 400 2160 | 2178 and 1708 | 1840, 600 2436 | 2727 and 1770 | 2142; 32-bit
    # (a block), width 1024, 600 rows 1478 | 1543 and 1197 | 1134, 1024 1716 | 1796 and 1271 | 1414.
    FORK_WORK = int(os.environ.get("I64H_FORK_WORK", "1650000000"))

    def _heavy(self, n: int) -> bool:
        return n * self.cfg.width ** 2 * (2 if self.exact else 1) >= self.FORK_WORK

    def _forks(self, n: int) -> bool:
        return self.side is not None and (self._heavy(n) or torch.cuda.is_current_stream_capturing())

    @contextmanager
    def _beside(self, n: int):
        """The launches of the body (a step of n rows) run on the side stream (of default priority), behind what the current stream holds so far and
        beside what it gets next, until _meet(n); a captured graph keeps the two branches.  Without a side stream, and in eager steps of few rows, they
        simply run here.  One level only: the body forks no further."""
        if not self._forks(n):
            yield
            return
        self.side.wait_stream(torch.cuda.current_stream())
        with torch.cuda.stream(self.side):
            yield

    def _meet(self, n: int) -> None:
        if self._forks(n):
            torch.cuda.current_stream().wait_stream(self.side)

    # ---- rows that only Linears read: their producer rounds them to bf16 once ----
    WIDE_BYTES = 0xfffffff0 - 64    # what the 32-bit offsets of the tiles on such rows reach: gathered rows, and the gate and up rows of a pair's weight
    FEW_ROWS = 2                    # up to this many rows: the forms that stream the weights past rows in 32 bits

    def _rounded(self, n: int, *widths: int) -> bool:
        """Whether a step of n rows rounds them where they are written (the values the Linears' tiles would round to: results are the same), for rows of these widths: whatever their
        number within the tiles' offsets, and below 65 as well, where the kernels of rows in bf16 are the faster ones from three rows on (64 rows, width 2048, us: 11392 columns 19.4 | 14.8, a pair of 5504 19.0 | 14.5, 2048 columns of 5504 22.5 | 16.6; steps of 64 rows 1608 | 1534, of 7
        rows and width 1024 526 | 497).  One row under 1024 x 1024 takes 3.0 | 3.4.  Short k is soon read: up to eight rows of fewer than 1024 values, and up to 16 of fewer than 512, stay
        in 32 bits.  1024 columns of 512, 3 rows 3.2 | 3.6, 8 3.4 | 3.6, 12 3.6 | 3.7, 32 5.0 | 3.9, a pair of 1344 4.1 | 4.9, 4.4 | 4.9, 4.6 | 5.0; columns of 256, 3 rows 2.8 | 3.6, 16
        3.1 | 3.6, 48 4.1 | 3.8."""
        if self.exact or n <= self.FEW_ROWS:
            return False
        top, narrow = 2 * max(n, self.max_ff + 256), 1024 if n <= 8 else 512 if n <= 16 else 0
        for w in widths:      # (asked a few times a layer by steps that wait for the host)
            if w % 64 or w < narrow or w * top >= self.WIDE_BYTES:
                return False
        return True

    def _wide_attention(self, n: int, width: int, vals: int, part: int, cache: torch.Tensor) -> bool:
        """Whether an attention over rows of `part` values a key head, the first `vals` of them summed, leaves its result (rows of `width`) in bf16: the matrix-core form
        and Linears that read it so."""
        return self._rounded(n, width) and cache.dtype == torch.bfloat16 and vals % 16 == 0 and vals <= 256 and part % 8 == 0 and part <= 320

    @staticmethod
    def _as16(t16: torch.Tensor, n: int, width: int) -> torch.Tensor:
        """The first rows of a buffer's bf16 view (which shares the memory of its fp32 rows) as a matrix."""
        return t16[: n * width].view(n, width)

    # ---- tensors by name and shape, in the two forms the kernels read ----
    def _bf(self, t: torch.Tensor) -> torch.Tensor:
        return t.to(device=self.device, dtype=torch.bfloat16).contiguous()

    def _f(self, t: torch.Tensor) -> torch.Tensor:
        return t.to(device=self.device, dtype=torch.float32).contiguous()

    @staticmethod
    def _reader(weights: Dict[str, torch.Tensor]):
        def need(name, shape):
            if name not in weights:
                raise KeyError(f"tensor '{name}' is missing")
            if tuple(weights[name].shape) != tuple(shape):
                raise ValueError(f"'{name}': shape {tuple(weights[name].shape)}, config says {tuple(shape)}")
            return weights[name]
        return need

    # ---- load-time layout ----
    def _stack(self, parts):
        """Rows of several projections as one weight, every part starting at a multiple of eight rows (rows of zeros between), so that the
        columns of a projection row can be read 16 bytes at a time; returns (weight, first column of each part)."""
        rows, offs, at = [], [], 0
        for t in parts:
            offs.append(at)
            rows.append(t.float())
            at = pad8(at + t.shape[0])
            if at > offs[-1] + t.shape[0]:
                rows.append(torch.zeros(at - offs[-1] - t.shape[0], t.shape[1]))
        return self._bf(torch.cat([r.cpu() for r in rows], 0)), offs

    def _low_rank(self, weights, need, first: str, second: str, out: int):
        """A map of two factors: the rank is the tensors' own; the second factor's columns are padded to where the first one's rows end."""
        if first not in weights or weights[first].dim() != 2:
            raise KeyError(f"tensor '{first}' is missing or is no matrix")
        r = weights[first].shape[0]
        a, b = need(first, (r, self.cfg.width)), need(second, (out, r))
        return a, self._bf(torch.nn.functional.pad(b.float(), (0, pad8(r) - r)))

    # ---- step buffers: the most recent row counts are kept, pinned sets stay for captured graphs ----
    def buffers(self, n: int, m: int):
        key = (n, m)
        B = self._bufs.pop(key, None)
        if B is None:
            B = type(self).BUFFERS(self, n, m)
            for name in ("b", "c", "rn", "act", "sact"):      # rows that may be written rounded, in the same memory
                if hasattr(B, name):
                    setattr(B, name + "16", getattr(B, name).view(torch.bfloat16))
        self._bufs[key] = B
        loose = [k for k in self._bufs if k not in self._pinned and k != key]
        for k in loose[:max(0, len(loose) + 1 - self.MAX_BUFFER_SETS)]:
            del self._bufs[k]
        return B

    def pin_buffers(self, n: int, m: int) -> None:
        self.buffers(n, m)
        self._pinned.add((n, m))

    def check_sync(self, force: bool = True):
        """No launch of these runners waits on a grid barrier: nothing to read back."""

    def snapshot_state(self):
        """The per-sequence state, for a caller that runs a step which must not count (a warm-up before a graph capture)."""
        return self.kv.snapshot()

    def restore_state(self, held) -> None:
        self.kv.restore(held)

    def _runs(self, n: int, slot_ids: torch.Tensor, tokens_per_seq, rows_are_slots: bool):
        """First rows of the runs of consecutive rows of one sequence, int32 [runs + 1] on the device, their number and the longest one's rows."""
        if rows_are_slots:
            t = self._arange.get(n)
            if t is None:
                t = self._arange[n] = torch.arange(n + 1, dtype=torch.int32, device=self.device)
            return t, n, 1
        if tokens_per_seq is None:      # (a caller that does not say how its rows are grouped: read it off the slot ids)
            s = slot_ids.tolist()
            tokens_per_seq, k = [], 0
            for j in range(1, n + 1):
                if j == n or s[j] != s[j - 1]:
                    tokens_per_seq.append(j - k)
                    k = j
        starts = [0]
        for t in tokens_per_seq:
            if int(t) > 0:
                starts.append(starts[-1] + int(t))
        if starts[-1] != n:
            raise ValueError(f"tokens_per_seq adds up to {starts[-1]} rows, the step has {n}")
        return upload(starts, torch.int32, self.device), len(starts) - 1, max(b - a for a, b in zip(starts, starts[1:]))

    def _splits(self, B, rows: int, heads: int, kv_heads: int, vals: int, width: int, ctx_hint: int, floats):
        """How many waves share a decode row's keys (about ATTN_WAVES waves in the launch, a wave keeping at least two tiles of 32 keys),
        and the workspace their partial results meet in."""
        tasks = rows * kv_heads * ((heads // kv_heads + 15) // 16)
        waves = self.ATTN_WAVES[64 if width <= 64 else (128 if width <= 128 else 256)]
        splits = max(1, min(waves // max(1, tasks), ctx_hint // 64, 64))
        if splits <= 1:
            return 1, None
        key = (rows, heads, kv_heads, vals, splits)
        ws = B.attn_ws.get(key)
        if ws is None:
            ws = B.attn_ws[key] = torch.empty(max(1, floats(splits)), dtype=torch.float32, device=self.device)
        return splits, ws

    def _scan_work(self, n: int, nseg: int, longest: int, scans, delta: bool, recs=()) -> Dict[tuple, torch.Tensor]:
        """The workspace of a step's scans by (heads, dim, vdim), for those of `scans` whose runs are worth the form that takes one, alone or (recs) from the projections.  The caller holds it for
        the step and no longer: 27 KB a tile of 16 rows and head of 128 would otherwise lie beside every kept buffer set.  Where the card has no room for
        it the scans go token by token: the same values in another order of the sums."""
        sizes = {s: D.scan_work_floats(n, nseg, s[0], s[1]) for s in scans if (D.rec_in_tiles if s in recs else D.scan_in_tiles)(n, nseg, longest, *s, delta=delta)}
        if not sizes:
            return {}
        try:
            ws = torch.empty(max(sizes.values()), dtype=torch.float32, device=self.device)
        except torch.OutOfMemoryError:
            return {}
        return {s: ws for s in sizes}      # (one after the other on one stream)

    # ---- attention over grouped key / value heads, separate keys and values in one cached row ----
    def _kattn(self, B, a, Q, O, rows, kvc, slot_ids, positions, runs, ctx_hint: int, *, bias=None, softcap: float = 0.0, window: int = 0,
               keep_first: int = 0, sink_w=None, nseg: int = 0) -> None:
        """Runs of rows that are one per sequence (a wave takes a token's query heads of one key head, the keys dealt to several waves) and
        runs of prompt portions (a wave takes 16 consecutive rows of one head), each one launch.  nseg: the step's sequences (0: not known)."""
        gs = a.vdim + a.dim
        portions = max(0, nseg - sum(r1 - r0 for r0, r1, one in runs if one)) if self.exact else 0      # (what the choice between the 32-bit forms asks)
        keys = min(ctx_hint, window + keep_first + 64) if window > 0 else ctx_hint
        for r0, r1, one_per_seq in runs:
            splits, ws = 1, None
            if one_per_seq and not self.exact:
                splits, ws = self._splits(B, r1 - r0, a.heads, a.kv_heads, a.vdim, gs, keys,
                                          lambda s: D.kattn_workspace_floats(r1 - r0, a.heads, a.kv_heads, a.vdim, s))
            D.kattn(Q[r0:r1], rows, None, kvc.block_table, slot_ids[r0:r1], positions[r0:r1], chunk=0, bias=bias, sink=sink_w is not None,
                    heads=a.heads, kv_heads=a.kv_heads, dim=a.dim, vdim=a.vdim, out=O[r0:r1], n=r1 - r0, mode=2 if one_per_seq else 3, splits=splits,
                    workspace=ws, softcap=softcap, window=window, keep_first=keep_first, sink_w=sink_w, seqs=portions)

    def _rotary_tables(self, a, d: dict) -> None:
        """Frequency tables of a rotated attention: evaluated in 64 bits on the host, rounded once to fp32."""
        d["inv_freq"], d["rot_mult"], d["v_freq"] = None, 1.0, None
        if a.rot is not None and a.rot.dims:
            fr, d["rot_mult"] = a.rot.frequencies()
            d["inv_freq"] = self._f(torch.tensor(fr, dtype=torch.float64))
        if a.rot is not None and a.rotate_values:
            d["v_freq"] = self._f(torch.tensor([a.rot.base ** (-2.0 * i / a.vdim) for i in range(a.vdim // 2)], dtype=torch.float64))

    def _rotary_attention(self, B, d, a, P, l, n, positions, slot_ids, kvc, runs, ctx_hint, out, scale: float = 1.0, nseg: int = 0) -> None:
        """Rotated attention on the projection rows P (already computed; columns d["q_off"], d["k_off"], d["v_off"]): prep -> paged
        [values | keys] rows and query rows, attention, the turn back and the head gate, out-projection (times `scale`) into `out`."""
        gs = a.vdim + a.dim
        Q = B.a[: n * a.heads * gs].view(n, a.heads * gs)
        rows = kvc.rows[l]
        D.rot_prep(P, q_off=d["q_off"], k_off=d["k_off"], v_off=d["v_off"], heads=a.heads, kv_heads=a.kv_heads, dim=a.dim, vdim=a.vdim, q_norm_w=d.get("q_norm"),
                   k_norm_w=d.get("k_norm"), eps=self.cfg.norm_eps, rot_dims=a.rot.dims if a.rot is not None else 0, interleaved=a.interleaved,
                   inv_freq=d["inv_freq"], rot_mult=d["rot_mult"], head_norm=a.qk_norm == "head", v_freq=d["v_freq"], scale=a.scale, positions=positions,
                   slot_ids=slot_ids, block_table=kvc.block_table, cache=rows, q=Q, n=n, norm_heads=a.qk_norm == "head_weight")
        behind = d["v_freq"] is not None or a.head_gate
        wide = not behind and self._wide_attention(n, a.heads * a.vdim, a.vdim, gs, rows)
        O = self._as16(B.b16, n, a.heads * a.vdim) if wide else B.b[: n * a.heads * a.vdim].view(n, a.heads * a.vdim)
        self._kattn(B, a, Q, O, rows, kvc, slot_ids, positions, runs, ctx_hint, softcap=a.softcap, window=a.window, keep_first=a.keep_first, sink_w=d.get("sink"), nseg=nseg)
        if behind:
            D.rot_post(O, heads=a.heads, vdim=a.vdim, interleaved=a.interleaved, v_freq=d["v_freq"], positions=positions,
                       gate=P if a.head_gate else None, gate_off=d.get("g_off", 0), ldg=P.shape[-1], n=n)
        self._out(None if wide else O, d["o"], out, scale, O if wide else None)

    def _out(self, a, w, out, scale: float = 1.0, a16=None) -> None:
        D.linear(a, w, out, a16=a16, exact=self.exact, epilogue=D.EPI_STORE if scale == 1.0 else D.EPI_SCALE, scale=scale)

    # ---- latent attention: one cached row per token that all heads share ----
    def _load_latent(self, p: str, m, need, d: dict) -> list:
        """Tensors of a latent attention under the prefix p behind its input projections, which are returned as parts of the layer's input
        weight, in order: queries (or their low-rank row), latent + shared key part, head gates."""
        W, bf, f, H, r = self.cfg.width, self._bf, self._f, m.heads, m.kv_rank
        # a head's score against a cached latent c is q_h . (U_h c) = (U_h^T q_h) . c: the key map transposed per head
        d["uk_t"] = bf(need(p + "uk", (H * m.dim, r)).reshape(H, m.dim, r).transpose(1, 2))      # [H, r, dim]
        d["uv"] = bf(need(p + "uv", (H * m.vdim, r)).reshape(H, m.vdim, r))                      # [H, vdim, r]
        d["c_norm"] = f(need(p + "dkv.norm", (r,)))
        d["sink"] = f(need(p + "sink", (H,))) if m.sink else None
        d["o"] = bf(need(p + "o", (W, H * m.vdim)))
        d["inv_freq"], d["rot_mult"] = None, 1.0
        if m.rot is not None:
            fr, d["rot_mult"] = m.rot.frequencies()
            d["inv_freq"] = f(torch.tensor(fr, dtype=torch.float64))
        if m.q_rank:
            d["q_norm"], d["uq"] = f(need(p + "dq.norm", (m.q_rank,))), bf(need(p + "uq", (m.q_width, m.q_rank)))
        parts = [need(p + "dq", (m.q_rank, W)) if m.q_rank else need(p + "q", (m.q_width, W)), need(p + "dkv", (r + m.rot_dim, W))]
        return parts + ([need(p + "g", (H, W))] if m.head_gate else [])

    def _latent_attention(self, B, d, m, P, l, n, positions, slot_ids, kvc, runs, ctx_hint, out) -> None:
        """Latent attention on the projection rows P (columns d["q_off"]: the queries, or their low-rank row; d["dkv_off"]: latent + shared
        key part; d["g_off"]: head gates): norms and rotation -> paged rows and query rows, queries into latent space per head, attention,
        summed latents into value space per head (times the head's gate), out-projection into `out`."""
        ex, N1 = self.exact, P.shape[-1]
        H, r, rd, qh = m.heads, m.kv_rank, m.rot_dim, m.dim + m.rot_dim
        width = r + rd
        src, q_off = P, d["q_off"]
        if m.q_rank:
            src, q_off = B.q[: n * H * qh].view(n, H * qh), 0
            D.linear(P, d["uq"], src, m=n, a_off=d["q_off"], exact=ex, in_norm_w=d["q_norm"], in_eps=self.cfg.norm_eps)
        cache = kvc.rows[l]
        Q = B.a[: n * H * width]
        D.latent_prep(P, q_off=q_off, dkv_off=d["dkv_off"], heads=H, dim=m.dim, rot_dim=rd, kv_rank=r, rot_dims=m.rot_dims, c_norm_w=d["c_norm"], eps=self.cfg.norm_eps,
                      inv_freq=d["inv_freq"], positions=positions, slot_ids=slot_ids, block_table=kvc.block_table, block_size=kvc.block, cache=cache, q=Q, n=n,
                      q_src=src if m.q_rank else None, rot_mult=d["rot_mult"])
        # queries into latent space, per head: Q[:, h, :r] = q_unrotated[:, h, :] @ U_h
        D.linear(src, d["uk_t"], Q, m=n, n=r, k=m.dim, a_off=q_off, lda=src.shape[-1], ldc=H * width, batch=H, a_batch=qh, w_batch=r * m.dim, c_batch=width, exact=ex)
        # (few rows: the value map's short k is faster over rows in 32 bits, by as much as an out-projection of 1024 loses; both, us, 8 heads of 256 to 64: 16 rows 7.0 | 7.7, 16 heads 3
        # rows 6.9 | 7.9, 12 7.9 | 8.0, 16 8.3 | 8.0, 32 heads 3 rows 9.1 | 9.1, 8 10.0 | 9.2)
        wide = self._wide_attention(n, H * r, r, width, cache) and r % 64 == 0 and self._rounded(n, H * m.vdim) and (n > 16 or H * m.vdim >= 2048)
        olat = (B.b16 if wide else B.b)[: n * H * r]
        keys = min(ctx_hint, m.window + 64) if m.window > 0 else ctx_hint
        for r0, r1, one_per_seq in runs:
            splits, ws = 1, None
            if one_per_seq and not ex:
                splits, ws = self._splits(B, r1 - r0, H, 1, r, width, keys, lambda s: D.latent_attn_workspace_floats(r1 - r0, H, r, s))
            D.latent_attn(Q[r0 * H * width: r1 * H * width], cache, kvc.block_table, slot_ids[r0:r1], positions[r0:r1], window=m.window, scale=m.scale, heads=H, kv_rank=r,
                          rot_dim=rd, out=olat[r0 * H * r: r1 * H * r], n=r1 - r0, mode=2 if one_per_seq else 3, splits=splits, workspace=ws, sink=d["sink"])
        # summed latents into value space, per head
        og = (B.c16 if wide else B.c)[: n * H * m.vdim]
        gate = dict(epilogue=D.EPI_ROW_SIGMOID, e=P, e_off=d["g_off"], lde=N1, e_batch=1) if m.head_gate else {}
        maps = dict(m=n, n=m.vdim, k=r, lda=H * r, ldc=H * m.vdim, batch=H, a_batch=r, w_batch=m.vdim * r, c_batch=m.vdim, exact=ex, **gate)
        if wide:
            D.linear(None, d["uv"], None, a16=olat, out16=og, **maps)
            D.linear(None, d["o"], out, a16=og, m=n, k=H * m.vdim, lda=H * m.vdim)
        else:
            D.linear(olat, d["uv"], og, **maps)
            D.linear(og, d["o"], out, m=n, k=H * m.vdim, lda=H * m.vdim, exact=ex)

    # ---- a recurrence's step where every row is a sequence of its own: one launch from the projections to the normed and gated rows ----
    # (The separate launches | one, us in graphs, delta rule and linear attention: 8 heads of 128, 1 row 18.5 | 7.0 and 10.2 | 5.1, 64 rows 34.6 | 14.7 and 23.1 | 11.3, 256 74 | 52 and 57 | 44,
    # 1024 271 | 250 and 220 | 201; 32 heads of 64, 64 rows 40 | 22 and 24 | 15, 1024 327 | 319 and 224 | 214; 2 heads of 32, 1 row 17 | 5.3 and 10 | 3.9, 1024 26 | 17 and 15 | 11: always the one.)
    def _recurs(self, r, P, n: int, seg, nseg: int, work, R, X, taps: int, **own) -> bool:
        """A recurrence from its projections (own: D.rec_step's operands), where every row is a sequence of its own or the scan goes in tiles of bf16 products; False: nothing was
        launched."""
        ws = work.get((r.heads, r.dim, r.vdim))
        if r.dim > D.REC_DIM or r.vdim > D.REC_DIM or r.dim % 4:
            return False
        if nseg == n and taps <= D.REC_STEP_TAPS:
            D.rec_step(P, heads=r.heads, dim=r.dim, vdim=r.vdim, n=n, exact=self.exact, **own)
            return True
        if ws is None or not self._rec_tiles_take(r, taps):
            return False
        D.rec_tiles(P, seg_start=seg, nseg=nseg, work=ws, r=R, x=X, heads=r.heads, dim=r.dim, vdim=r.vdim, n=n, **own)
        return True

    def _rec_tiles_take(self, r, taps: int) -> bool:
        """Whether prompts of a recurrence may go from the projections in tiles (taps of its convolution, 0: linear attention)."""
        # (linear attention in narrow heads has nothing to save but the decays' way through memory: 32 heads of 64, runs of 700 and 300, 55.6 us in launches of its own, 56.2 here; of 128, 16
        # heads, 2956 rows 145 and 131; the delta rule 104 and 90, 270 and 191)
        return not self.exact and max(r.dim, r.vdim) <= D.REC_DIM and r.dim % 4 == 0 and r.vdim % 4 == 0 and taps <= D.REC_TILE_TAPS and (taps > 0 or r.dim > 64)

    @staticmethod
    def _delta_recurs(r) -> bool:
        """Whether a delta rule has the form of one that goes from its projections: a decay per key channel, every head its own keys, a convolution."""
        return r.decay == "channel" and r.kv_heads == r.heads and r.conv > 1

    # ---- gated linear attention ----
    def _gated_linear(self, B, d, r, P, l, n, positions, slot_ids, kvc, seg, nseg, out, scale: float = 1.0, work=NO_WORK, longest: int = 0) -> None:
        """Gated linear attention on the projection rows P (columns d["rq_off"], d["rk_off"], d["rv_off"], d["rg_off"]: queries, keys, values, output
        gates; d["a1_off"]: the low-rank decay map's first factor).  sigmoid(z)^(1 / tau) = exp(-softplus(-z) / tau): the second factor and
        its bias are held negated, the exponent's rate is d["a_rate"]."""
        rv = r.heads * r.vdim
        wide = self._rounded(n, rv)
        Rn, Rn16 = None if wide else B.rn[: n * rv].view(n, rv), self._as16(B.rn16, n, rv) if wide else None
        R = B.r[: n * rv].view(n, rv)
        if self._recurs(r, P, n, seg, nseg, work, R, None, 0, q_off=d["rq_off"], k_off=d["rk_off"], v_off=d["rv_off"], a=d["a2"], a_off=d["a1_off"], a_bias=d["a2_b"], a_rate=d["a_rate"],
                        z_off=d["rg_off"], norm_w=d["r_norm"], eps=self.cfg.norm_eps, positions=positions, slot_ids=slot_ids, state=kvc.state[l]["gla"], out=Rn, out16=Rn16,
                        q_scale=r.dim ** -0.5):
            self._out(Rn, d["o_right"], out, scale, Rn16)
            return
        F = B.f[: n * r.heads * r.dim].view(n, r.heads * r.dim)
        D.linear(P, d["a2"], F, m=n, a_off=d["a1_off"], exact=self.exact, bias=d["a2_b"], epilogue=D.EPI_DECAY, e=d["a_rate"])
        D.gla_scan(P, f=F, q_off=d["rq_off"], k_off=d["rk_off"], f_off=0, v_off=d["rv_off"], heads=r.heads, dim=r.dim, vdim=r.vdim, seg_start=seg, nseg=nseg,
                   positions=positions, slot_ids=slot_ids, state=kvc.state[l]["gla"], out=R, n=n, q_scale=r.dim ** -0.5,
                   work=work.get((r.heads, r.dim, r.vdim)), longest=longest)
        D.gate_norm(R, d["r_norm"], Rn, groups=r.heads, eps=self.cfg.norm_eps, z=P, z_off=d["rg_off"], ldz=P.shape[-1], n=n, gate_after=True, width=rv, out16=Rn16)
        self._out(Rn, d["o_right"], out, scale, Rn16)

    # ---- gated delta rule ----
    def _gated_delta(self, B, d, r, P, l, n, positions, slot_ids, kvc, seg, nseg, single: bool, out, work=NO_WORK, longest: int = 0) -> None:
        """Gated delta rule on the projection rows P: the convolved parts q | k | v from column d["r_off"] on, the write strength's at
        d["rb_off"].  A decay per head comes from the columns d["ra_off"]; a decay per key channel (r.decay 'channel') and its output gate are
        low-rank maps whose first factors' results lie at d["a1_off"] and d["g1_off"]."""
        ex = self.exact
        st = kvc.state[l]
        C, rk, rv = r.conv_channels, r.kv_heads * r.dim, r.heads * r.vdim
        channel = r.decay == "channel"
        wide = self._rounded(n, rv)
        Rn, Rn16 = None if wide else B.c[: n * rv].view(n, rv), self._as16(B.c16, n, rv) if wide else None
        R = B.b[: n * rv].view(n, rv)
        if self._delta_recurs(r) and \
                self._recurs(r, P, n, seg, nseg, work, R, B.a[: n * rv], r.conv, q_off=d["r_off"], a=d["a2"], a_off=d["a1_off"], a_bias=d["dt_bias"], a_rate=d["a_rate"], z=d["g2"],
                             z_off=d["g1_off"], norm_w=d["r_norm"], eps=self.cfg.norm_eps, positions=positions, slot_ids=slot_ids, state=st["gdn"], out=Rn, out16=Rn16, conv_w=d["conv_w"],
                             conv=st["conv"], b_off=d["rb_off"], unit_eps=UNIT_EPS, q_scale=r.dim ** -0.5, sigmoid=r.gate == "sigmoid"):
            D.linear(Rn, d["o_right"], out, a16=Rn16, exact=ex)
            return
        X = B.a[: n * C].view(n, C)
        D.causal_conv(P, off=d["r_off"], channels=C, w=d["conv_w"], bias=None, positions=positions, slot_ids=slot_ids, state=st.get("conv"), out=X, n=n,
                      single_rows=single, seg_start=seg, nseg=nseg)
        G = B.g[: n * 2 * r.heads].view(n, 2 * r.heads)
        cols = dict(q_off=0, k_off=rk, v_off=2 * rk, heads=r.heads, kv_heads=r.kv_heads, dim=r.dim, vdim=r.vdim, n=n)
        D.gdn_gates(X, G, P, b_off=d["rb_off"], a_off=-1 if channel else d["ra_off"], a_log=None if channel else d["A_log"],
                    dt_bias=None if channel else d["dt_bias"], unit_eps=UNIT_EPS, q_scale=r.dim ** -0.5, **cols)
        F, Z, z_off, ldz = None, P, d.get("rg_off", 0), P.shape[-1]
        if channel:
            F, Z, z_off, ldz = B.f[: n * r.heads * r.dim].view(n, r.heads * r.dim), B.z[: n * rv].view(n, rv), 0, rv
            D.linear(P, d["a2"], F, m=n, a_off=d["a1_off"], exact=ex, bias=d["dt_bias"], epilogue=D.EPI_DECAY, e=d["a_rate"])
            D.linear(P, d["g2"], Z, m=n, a_off=d["g1_off"], exact=ex)
        D.gdn_scan(X, G, f=F, seg_start=seg, nseg=nseg, positions=positions, slot_ids=slot_ids, state=st["gdn"], out=R,
                   work=work.get((r.heads, r.dim, r.vdim)), longest=longest, **cols)
        D.gate_norm(R, d["r_norm"], Rn, groups=r.heads, eps=self.cfg.norm_eps, z=Z, z_off=z_off, ldz=ldz, n=n, gate_after=True, width=rv, sigmoid=r.gate == "sigmoid", out16=Rn16)
        D.linear(Rn, d["o_right"], out, a16=Rn16, exact=ex)

    # ---- mixture of experts ----
    def _load_moe(self, p: str, f, need, d: dict) -> None:
        """Router, stacked experts and shared expert of a mixture under the tensor prefix p."""
        W, bf = self.cfg.width, self._bf
        router = need(p + "router", (f.entries, W))
        if f.shared_ff and f.shared_gate:       # one more row behind the router's: the shared expert's gate
            router = torch.cat([router, need(p + "shared.sg", (1, W))], 0)
        d["router"] = bf(router)
        d["router_b"] = self._f(need(p + "router.b", (f.entries,))) if f.router_bias else None
        # per expert [gate rows; up rows], all experts stacked: one grouped launch for the pair, one for the way down
        # (a shared expert of the experts' size and activation is the first of the stack, its rows a group of all tokens)
        d["merged"] = self._shared_in_stack(f)
        names = ([p + "shared"] if d["merged"] else []) + [f"{p}e{e}" for e in range(f.experts)]
        d["gate_up"] = bf(torch.stack([torch.cat([need(x + ".gate", (f.ff, W)), need(x + ".up", (f.ff, W))], 0) for x in names]))
        d["e_down"] = bf(torch.stack([need(x + ".down", (W, f.ff)) for x in names]))
        if d["merged"]:
            d["s_gate_up"], d["s_down"] = d["gate_up"][0], d["e_down"][0]
        elif f.shared_ff:
            s = f.shared_ff
            d["s_gate_up"] = bf(torch.cat([need(p + "shared.gate", (s, W)), need(p + "shared.up", (s, W))], 0))
            d["s_down"] = bf(need(p + "shared.down", (W, s)))

    @staticmethod
    def _shared_in_stack(f) -> bool:
        return bool(f.shared_ff) and f.shared_ff == f.ff and f.shared_limit == f.limit

    @staticmethod
    def moe_buffers(B, model, n: int) -> None:
        """The step buffers of the feed-forwards on B (model.max_top == 0: no mixtures)."""
        i32, f32 = dict(dtype=torch.int32, device=model.device), dict(dtype=torch.float32, device=model.device)
        B.joined = model._joins(n)
        t, (g, act, shared) = model.max_top, model.ff_sizes[B.joined]
        B.act = torch.empty(n * max(act, 1), **f32)
        B.ey = torch.empty(n * g, model.cfg.width, **f32) if t else None   # the outputs, grouped by expert
        B.idx = torch.empty(n * max(t, 1), **i32)
        B.wgt, B.wgt_next = torch.empty(n * max(t, 1), **f32), torch.empty(n * max(t, 1), **f32)      # the choice's weights, and those of the one that follows (_moe_read)
        B.pair_token = torch.empty(n * max(g, 1), **i32)
        B.pair_row = torch.empty(n * max(t, 1), **i32)
        B.pair_wgt = torch.empty(n * max(g, 1), **f32)
        B.group_off = torch.empty(model.max_groups + 1, **i32)
        B.sgate = torch.empty(n, **f32)
        B.sync = torch.zeros(32 * (D.PLAN_ROWS // 8 + 1), **i32) if t else None      # counters of the launches that plan a step behind its norm
        B.sact = torch.empty(n * max(shared, 1), **f32)                    # the inner rows of a shared expert beside the grouped launches
        B.shared_rows = n if shared else 0

    def _moe_sizes(self, mlps) -> None:
        moes = [m for m in mlps if m is not None and m.kind == "moe"]
        self.max_top = max([m.top for m in moes] or [0])
        self.max_groups = max([m.experts + int(self._shared_in_stack(m)) for m in moes] or [0])
        dense = [m.ff for m in mlps if m is not None and m.kind == "dense"]
        self.max_ff = max(dense + [w for m in moes for w in (m.ff, m.shared_ff)] + [0])
        self.ff_sizes = {}      # by B.joined: rows a token has in the grouped Linears, its widest inner rows, the widest shared expert beside the grouped launches
        for joined in (False, True):
            inside = [joined and self._shared_in_stack(m) for m in moes]
            rows = [m.top + int(i) for m, i in zip(moes, inside)]
            self.ff_sizes[joined] = (max(rows or [0]), max(dense + [m.ff * r for m, r in zip(moes, rows)] + [0]), max([m.shared_ff for m, i in zip(moes, inside) if not i] or [0]))

    @staticmethod
    def _glu(limit: float, alpha: float) -> dict:
        """The gate / up epilogue of a feed-forward: clamped by `limit`, or silu."""
        return dict(epilogue=D.EPI_CLAMP_GLU, act_a=alpha, act_b=limit) if limit > 0 else dict(epilogue=D.EPI_SILU_MUL)

    def _load_dense(self, p: str, f, need, d: dict) -> None:
        W = self.cfg.width
        d["ff_gate_up"] = self._bf(torch.cat([need(p + "gate", (f.ff, W)), need(p + "up", (f.ff, W))], 0))
        d["ff_down"] = self._bf(need(p + "down", (W, f.ff)))

    def _act(self, buf, buf16, n: int, width: int, h16):
        """A feed-forward's inner rows: (fp32, bf16), one of them None."""
        if h16 is not None and width % 64 == 0:
            return None, self._as16(buf16, n, width)
        return buf[: n * width].view(n, width), None

    def _dense_glu(self, B, d, n, h, out, h16=None) -> None:
        """h16: the input rows in bf16, read in h's place."""
        f = d["mlp"]
        act, act16 = self._act(B.act, B.act16, n, f.ff, h16)
        D.linear(h, d["ff_gate_up"], act, a16=h16, out16=act16, exact=self.exact, **self._glu(f.limit, f.glu_alpha))
        D.linear(act, d["ff_down"], out, a16=act16, exact=self.exact)

    MOE_BESIDE = False      # the shared expert of a mixture may run on the side stream, beside the choice and the plan

    def _joins(self, n: int) -> bool:
        """Whether a shared expert in its experts' stack joins their launches in a step of n rows, but where it can run beside the choice and the plan of much work (8
        prompts of 512, width 1024: 3572 us a step joined, 3432 beside; where the whole feed-forward runs beside a mixer joined is better, 5593 and 5804)."""
        return not (self.MOE_BESIDE and self.side is not None and self._heavy(n))

    @staticmethod
    def _fills(pairs: int, experts: int) -> bool:
        """Whether the experts' rows are enough for the wide tiles, whose smallest is 64 rows high: many experts of a few rows each read rows that are not there as
        often as weights.  Microseconds of a pair's two launches, rows in fp32 | in bf16, width 2048, 768 inner: 16 experts of two, 100 tokens 37 | 39, 200
        44 | 41; 32 of two, 100 tokens 65 | 69, 320 69 | 69, 400 77 | 70; 64 of two, 200 tokens 113 | 121, 700 134 | 127; 64 of eight, 100 tokens 120 | 126, 200 136 | 126; 128 of
        eight, 100 tokens 217 | 226, 320 242 | 234; 8 of two (1792 inner), 65 tokens 48 | 45; with a shared one, 7 tokens 43 | 37, 33 58 | 54, 64 61 | 57, and of width 1024,
        896 inner, 5 tokens 13.6 | 18.2, 27 17.7 | 16.3, 64 19.1 | 16.8 (hence the rule behind this one)."""
        return experts < 16 or pairs >= 20 * experts

    @staticmethod
    def _streams(n: int, width: int, experts: int, merged: bool) -> bool:
        """Whether a mixture of few rows stays with rows in 32 bits, whose launches of at most 16 rows take 16 columns a workgroup: the second one, of `width` columns a group, has then
        about two such workgroups a CU (256) at most, where the 64 x 64 tiles of rows in bf16 leave most CUs without one.  A shared expert's group has all rows, and with more than eight
        its tile reads them less often than that (below a width of 1024, 16).  Microseconds of both launches over five draws of experts, rows in fp32 | in bf16: 8 experts of 896 and a shared one, width 1024 (576
        workgroups), 3 tokens 14.0 | 15.1, 8 17.0 | 18.1, 16 18.6 | 18.2, without it (512) 3 13.1 | 14.6, 16 15.9 | 17.5; 4 of 2048, width 1024 (256), 3 15.6 | 19.6, 16 18.2 | 22.1; 2 of
        2048, width 2048 (256), 8 17.7 | 23.8; 8 of 2752, width 1024 (512), 8 33.0 | 35.8; 4 of 1344 and a shared one, width 1536 (480), 5 20.9 | 22.9, 16 25.4 | 22.9; 8 of 512 and a shared one, width 512 (288), 12 12.2 | 13.6.  More workgroups: 4
        of 896 and a shared one, width 2048 (640), 5 23.1 | 22.2; 8 of 1024 and a shared one, width 1280 (720), 5 21.1 | 20.0."""
        return n <= (8 if merged and width >= 1024 else 16) and width * (experts + int(merged)) <= 576 * 16

    def _moe_merges(self) -> bool:
        """Whether the residual's launch sums a mixture's rows itself (i64h_streams_args.moe_y)."""
        return self.cfg.width % 4 == 0 and self.cfg.width <= 8192

    # the router's products in 32 bits in both modes (a choice between experts is not rounding's to make), inside the choice's launch
    def _route(self, B, d) -> dict:
        f = d["mlp"]
        return dict(w=d["router"], entries=f.entries, correction=d.get("correction"), groups=f.groups, keep=f.keep, top=f.top, scale=f.scale, idx=B.idx, wgt=B.wgt, bias=d["router_b"],
                    chosen_softmax=f.chosen_softmax, gate_out=B.sgate if f.shared_ff and f.shared_gate else None, sigmoid_scores=f.sigmoid_scores, raw_weights=f.raw_weights)

    def _plan(self, B, d) -> dict:
        f = d["mlp"]
        return dict(experts=f.experts, group_off=B.group_off, pair_token=B.pair_token, pair_row=B.pair_row, pair_wgt=B.pair_wgt if f.weigh_input else None,      # the weight multiplies what the expert reads, not what it returns
                    shared=d["merged"] and B.joined)

    def _routes_in_norm(self, f) -> bool:
        """Whether the launch that norms a mixture's input also chooses its experts (i64h_streams_route), and plans the step where it is small."""
        return f.entries + int(bool(f.shared_ff and f.shared_gate)) <= D.ROUTE_ENTRIES and f.groups <= 1 and self._moe_merges()

    def _moe_read(self, B, d, n, h, h16) -> dict:
        """What the launch that norms a mixture's input is to write and choose: h stays away where everybody behind it reads rows in bf16.  The launch may also sum the mixture in front,
        whose weights another row's workgroup still reads when this choice is written (they lie apart by rows only where both choose as many experts): two sets take turns."""
        f = d["mlp"]
        if not self._routes_in_norm(f):
            return dict(h=h, h16=h16)
        B.wgt, B.wgt_next = B.wgt_next, B.wgt
        bare = h16 is not None and f.entries == f.experts and self._experts_read16(d, n, d["merged"] and B.joined)
        return dict(h=None if bare else h, h16=h16, route=self._route(B, d), **(dict(plan=self._plan(B, d), sync=B.sync) if n <= D.PLAN_ROWS else {}))

    def _experts_read16(self, d, n: int, merged: bool) -> bool:
        f = d["mlp"]
        return self._fills(n * f.top, f.experts) and not self._streams(n, self.cfg.width, f.experts, merged)

    def _moe_ff(self, B, d, n, h, out, shared_out, record: Optional[dict] = None, tag: str = "", beside: bool = False, h16=None, combine: bool = True, routed: bool = False):
        """out <- the mixture of d["mlp"] on h fp32 [n, width] (h16: its rows in bf16, which the experts read); shared_out [n, width] receives the rows of a
        shared expert that is not in the experts' stack on the way (beside: on the side stream, while the routed experts run).  combine False: the
        weighted sum is left to the caller's residual launch, whose operands are returned.  routed: the launch that normed h was given _moe_read's operands."""
        f, ex, W = d["mlp"], self.exact, self.cfg.width
        E, top = f.experts, f.top
        merged = d["merged"] and B.joined
        gate = B.sgate if f.shared_ff and f.shared_gate else None
        shared = None
        if f.shared_ff and not merged:
            with self._beside(n) if beside else nullcontext():
                sact, sact16 = self._act(B.sact, B.sact16, n, f.shared_ff, h16)
                D.linear(h, d["s_gate_up"], sact, a16=h16, out16=sact16, exact=ex, **self._glu(f.shared_limit, f.glu_alpha))
                shared = D.linear(sact, d["s_down"], shared_out, a16=sact16, exact=ex)
        gate_up, e_down = (d["gate_up"], d["e_down"]) if merged or not d["merged"] else (d["gate_up"][1:], d["e_down"][1:])
        routed = routed and self._routes_in_norm(f)
        if not routed:
            D.route_topk(None, h=h, n=n, **self._route(B, d))
        if record is not None:
            record[f"{tag}.route"] = B.idx[: n * top].view(n, top).clone()
        plan = self._plan(B, d)
        if not (routed and n <= D.PLAN_ROWS):
            D.moe_plan(B.idx, n=n, top=top, wgt=B.wgt, **plan)
        # the (token, expert) pairs lie grouped by expert: one launch runs every expert over its own rows, the counts stay on the device
        x16 = h16 if self._experts_read16(d, n, merged) else None
        rows, groups = n * (top + int(merged)), E + int(merged)
        act, act16 = self._act(B.act, B.act16, rows, f.ff, x16)
        D.linear(h, gate_up, act, a16=x16, out16=act16, m=n, a_rows=B.pair_token[:rows], batch=groups, w_batch=2 * f.ff * W, exact=ex, group_off=B.group_off, row_scale=plan["pair_wgt"],
                 **self._glu(f.limit, f.glu_alpha))
        D.linear(act, e_down, B.ey[:rows], a16=act16, m=n, batch=groups, w_batch=W * f.ff, exact=ex, group_off=B.group_off)
        if shared is not None and beside:
            self._meet(n)
        if merged:
            shared = B.ey[:n]
        sums = dict(y=B.ey, pair_row=B.pair_row, wgt=None if f.weigh_input else B.wgt, h=h, shared=shared, top=top, shared_gate=gate)
        if not combine:
            return sums
        D.moe_combine(sums.pop("y"), sums.pop("pair_row"), sums.pop("wgt"), sums.pop("h"), sums.pop("shared"), out, n=n, width=W, **sums)
