"""LayeredLM: decoder-only language models whose configuration lists the layers (config.LayeredLMConfig), on the framework's engine.

The step function packs the new tokens of any set of sequences -- whole prompts, portions of prompts, single decoded tokens, of any
mix of lengths -- into one launch sequence (``md_lm_forward``); generation prefills a ragged batch that way and then decodes it in
lockstep on the shared loop (``engine.DeviceEngine._lockstep_loop``: hipGraph replay under ``compile()``, greedy or sampled on the
device).  State lives in ``state.LayeredState`` slots.
"""
from __future__ import annotations

import ctypes as C
import os
from typing import Any, Dict, List, Optional, Sequence, Tuple, Union

import torch

from . import _lib
from .config import LayeredLMConfig, load_config
from .engine import BF16, DEFAULT_MAX_TOKENS, DEFAULT_TEMPERATURE, DEFAULT_TOP_P, DeviceEngine
from .state import LayeredState
from .weights import PackedLayeredLM, read_tensors


class LayeredLM(DeviceEngine):
    def __init__(self, config: LayeredLMConfig, state_dict: Dict[str, torch.Tensor], device: Union[str, torch.device] = "cuda",
                 dtype: torch.dtype = BF16, tokenizer: Any = None, max_batch: int = 1, max_context: int = 2048, max_step_rows: int = 16384):
        """``max_batch`` slots of ``max_context`` positions are allocated at once (both grow when needed); a step of more than
        ``max_step_rows`` tokens runs as portions."""
        self.config = config
        self._init_device(device, lm_only=True)
        self.dtype = dtype
        self.tokenizer = tokenizer
        self.w = PackedLayeredLM(config, state_dict, self._device, dtype)
        self.state = LayeredState(self.w, max_batch, max_context)
        self.max_step_rows = max(1, int(max_step_rows))
        self._logits_buf: Optional[torch.Tensor] = None

    @classmethod
    def from_pretrained(cls, path: str, config: Optional[LayeredLMConfig] = None, **kwargs) -> "LayeredLM":
        """From a model folder (config.json + model.safetensors)."""
        return cls(config or load_config(path), read_tensors(os.path.join(path, "model.safetensors")), **kwargs)

    # ------------------------------------------------------------- sequences
    def open_sequence(self) -> int:
        """A slot for a new sequence (nothing in it yet)."""
        before = self.state.slots
        slot = self.state.take()
        if self.state.slots != before:
            self._graphs.clear()
        return slot

    def close_sequence(self, slot: int) -> None:
        self.state.pool.free(slot)

    def sequence_length(self, slot: int) -> int:
        return self.state.pool.length[slot]

    def _check_length(self, positions: int) -> None:
        if self.config.positions and positions > self.config.positions:
            raise ValueError(f"a sequence of {positions} tokens: the model has {self.config.positions} positions")

    def _reserve(self, positions: int) -> None:
        if positions > self.state.ctx:
            self.state.reserve(self.state.slots, positions)
            self._graphs.clear()

    # ------------------------------------------------------------------ step
    def step(self, entries: Sequence[Tuple[int, Sequence[int], Sequence[int]]], layer_out: Optional[List[torch.Tensor]] = None) -> torch.Tensor:
        """Run the next tokens of several sequences as one batch: ``entries`` = (slot, token ids, places among these tokens whose
        logits are wanted).  Returns those logits, [wanted, vocab], in the order of the entries and places.  ``layer_out`` collects
        the residual stream after every layer, fp32 [rows of the batch, width]."""
        slots = [e[0] for e in entries]
        if len(set(slots)) != len(slots):
            raise ValueError("a sequence appears twice in one step")
        for slot, ids, want in entries:
            if not 0 <= slot < self.state.slots:
                raise ValueError(f"slot {slot} does not exist")
            if len(ids) == 0:
                raise ValueError("an entry brings no tokens")
            lo, hi = min(ids), max(ids)
            if lo < 0 or hi >= self.config.vocab:
                raise ValueError(f"token id out of range [0, {self.config.vocab}): {lo if lo < 0 else hi}")
            if any(not 0 <= k < len(ids) for k in want):
                raise ValueError("a wanted place is outside the entry's tokens")
            self._check_length(self.sequence_length(slot) + len(ids))
        total = sum(len(e[1]) for e in entries)
        if total <= self.max_step_rows:
            return self._forward(entries, layer_out)
        # portions: round-robin over the entries until every token has run
        done, parts = [0] * len(entries), {}
        while any(done[i] < len(e[1]) for i, e in enumerate(entries)):
            room, portion, keys = self.max_step_rows, [], []
            for i, (slot, ids, want) in enumerate(entries):
                n = min(room, len(ids) - done[i])
                if n == 0:
                    continue
                w = [k for k in want if done[i] <= k < done[i] + n]
                portion.append((slot, ids[done[i] : done[i] + n], [k - done[i] for k in w]))
                keys += [(i, k) for k in w]
                done[i] += n
                room -= n
            for key, row in zip(keys, self._forward(portion, layer_out)):
                parts[key] = row
        rows = [parts[(i, k)] for i, e in enumerate(entries) for k in e[2]]
        return torch.stack(rows) if rows else torch.empty(0, self.config.vocab, dtype=self.dtype, device=self._device)

    def _forward(self, entries, layer_out=None) -> torch.Tensor:
        lens = [len(e[1]) for e in entries]
        n_seq, n_rows, n_want = len(entries), sum(lens), sum(len(e[2]) for e in entries)
        length = self.state.pool.length
        pos0 = [length[e[0]] for e in entries]
        max_ctx = max(p + n for p, n in zip(pos0, lens))
        self._reserve(max_ctx)
        row0 = [0]
        for n in lens:
            row0.append(row0[-1] + n)
        ctx0 = [0]
        for p, n in zip(pos0, lens):
            ctx0.append(ctx0[-1] + p + n)
        # one host array, one copy: tokens | row -> sequence | row -> position | first rows | first positions | slots | context sums | wanted rows
        host: List[int] = []
        for e in entries:
            host.extend(int(t) for t in e[1])
        for b, n in enumerate(lens):
            host.extend([b] * n)
        for p, n in zip(pos0, lens):
            host.extend(range(p, p + n))
        host.extend(row0)
        host.extend(pos0)
        host.extend(int(e[0]) for e in entries)
        host.extend(ctx0)
        host.extend(row0[b] + k for b, e in enumerate(entries) for k in e[2])
        with torch.inference_mode():
            dev = self._h2d(torch.tensor(host, dtype=torch.int32))
            at = [0]
            for n in (n_rows, n_rows, n_rows, n_seq + 1, n_seq, n_seq, n_seq + 1, n_want):
                at.append(at[-1] + n)
            ptr = [dev.data_ptr() + 4 * o for o in at]
            going = sum(p > 0 for p in pos0)
            batch = _lib.MdLmBatch(n_seq, n_rows, max(lens), going, ptr[0], ptr[1], ptr[2], ptr[3], ptr[4], ptr[5], max_ctx, ctx0[-1], ptr[6])
            logits = torch.empty(max(n_want, 1), self.w.model.head.n_pad, dtype=self.dtype, device=self._device)
            taps = None
            if layer_out is not None:
                taps = torch.empty(len(self.config.layers), n_rows, self.w.width_pad, dtype=torch.float32, device=self._device)
            ws = self._workspace(self.lib.md_lm_workspace_bytes(C.byref(self.w.model), C.byref(batch), n_want))
            st = self.state.struct()
            _lib.check(
                self.lib.md_lm_forward(
                    C.byref(self.w.model), C.byref(batch), C.byref(st), ptr[7], n_want, logits.data_ptr(), logits.shape[1],
                    taps.data_ptr() if taps is not None else None, ws.data_ptr(), ws.numel(), self._stream(),
                ),
                "md_lm_forward",
            )
        for e, n in zip(entries, lens):
            length[e[0]] += n
        if taps is not None:
            layer_out.append(taps[:, :, : self.config.width])
        return logits[:n_want, : self.config.vocab]

    # ------------------------------------------------------------ generation
    def _decode_logits(self, b: int) -> torch.Tensor:
        if self._logits_buf is None or self._logits_buf.shape[0] < b:
            self._logits_buf = torch.empty(b, self.w.model.head.n_pad, dtype=self.dtype, device=self._device)
            self._graphs.clear()
        return self._logits_buf

    def _decode_lockstep(self, first: torch.Tensor, slots: Sequence[int], max_tokens: int, suppress_id: int = -1, eos_id: Optional[int] = None,
                         check_every: int = 16, temperature: float = 0.0, top_p: float = 0.0,
                         generator: Optional[torch.Generator] = None) -> torch.Tensor:
        """int32 [steps + 1, B]: ``first`` and what each sequence goes on with (greedy, or drawn with temperature / top-p)."""
        b = first.shape[0]
        pos = [self.state.pool.length[s] for s in slots]
        max_tokens = max(0, max_tokens)
        self._reserve(max(pos) + max_tokens)
        logits = self._decode_logits(b)
        ctx = self.state.ctx
        going = sum(p > 0 for p in pos)
        ws = self._workspace(self.lib.md_lm_workspace_bytes(C.byref(self.w.model), C.byref(_lib.MdLmBatch(b, b, 1, going, max_ctx=ctx)), b), 2)
        uniforms = torch.rand(max_tokens, b, device=self._device, dtype=torch.float32, generator=generator) if temperature != 0 else None
        rows = self._h2d(torch.tensor(list(range(b + 1)) + list(slots), dtype=torch.int32))
        st = self.state.struct()

        def make_step(pos_buf):
            def one_step(tok_in, tok_out, u_row):
                batch = _lib.MdLmBatch(b, b, 1, going, tok_in.data_ptr(), rows.data_ptr(), pos_buf.data_ptr(), rows.data_ptr(), pos_buf.data_ptr(),
                                       rows.data_ptr() + 4 * (b + 1), ctx, 0, None)
                _lib.check(
                    self.lib.md_lm_decode_step(
                        C.byref(self.w.model), C.byref(batch), C.byref(st), tok_out.data_ptr(), pos_buf.data_ptr(), suppress_id,
                        logits.data_ptr(), logits.shape[1], ws.data_ptr(), ws.numel(), self._stream(),
                    ),
                    "md_lm_decode_step",
                )
                if uniforms is not None:
                    self._sample_into(logits[:b], self.config.vocab, temperature, top_p, suppress_id, u_row, tok_out)

            return one_step

        key = (tuple(slots), ctx, going, suppress_id, ws.data_ptr(), logits.data_ptr(), float(temperature), float(top_p), self.dtype)
        hist = self._lockstep_loop(first, pos, max_tokens, make_step, key, eos_id, check_every, uniforms, keep=(rows, ws, logits))
        for s in slots:
            self.state.pool.length[s] += hist.shape[0] - 1
        return hist

    def batch_generate_ids(self, prompts: Sequence[Sequence[int]], max_tokens: int = DEFAULT_MAX_TOKENS, eos_id: Optional[int] = None,
                           temperature: float = 0.0, top_p: float = DEFAULT_TOP_P, generator: Optional[torch.Generator] = None,
                           max_batch: Optional[int] = None) -> List[List[int]]:
        """Token ids for prompts of any lengths: groups of at most ``max_batch`` (default: all) are prefilled together and decoded in
        lockstep; greedy by default, ends at ``eos_id`` or after ``max_tokens``."""
        prompts = [[int(t) for t in p] for p in prompts]
        if not prompts or any(len(p) == 0 for p in prompts):
            raise ValueError("empty prompt")
        group = max(1, int(max_batch or len(prompts)))
        out: List[List[int]] = []
        for g0 in range(0, len(prompts), group):
            part = prompts[g0 : g0 + group]
            slots = [self.open_sequence() for _ in part]
            try:
                with torch.inference_mode():
                    logits = self.step([(s, p, [len(p) - 1]) for s, p in zip(slots, part)])
                    if max_tokens <= 0:
                        out += [[] for _ in part]
                        continue
                    if temperature != 0 and logits.dtype == torch.float32:
                        logits = logits.to(BF16)
                    first = self._pick(logits, temperature, top_p, generator=generator, vocab=self.config.vocab)
                    # what a sequence can still take: its last token needs no position (the shortest prompt sets the lockstep's length)
                    room = [min(max_tokens, self.config.positions - len(p) + 1) if self.config.positions else max_tokens for p in part]
                    hist = self._decode_lockstep(first, slots, max(room) - 1, eos_id=eos_id, temperature=temperature, top_p=top_p,
                                                 generator=generator)
                    out += [self._truncate(col, eos_id, n) for col, n in zip(hist.t().tolist(), room)]
            finally:
                for s in slots:
                    self.close_sequence(s)
        return out

    def batch_generate(self, prompts: Sequence[str], settings: Optional[dict] = None) -> List[str]:
        """Text in, text out (needs a tokenizer), with the framework's settings: max_tokens, temperature, top_p."""
        if self.tokenizer is None:
            raise ValueError("text prompts need a tokenizer")
        s = settings or {}
        ids = [list(self.tokenizer.encode(p).ids) for p in prompts]
        got = self.batch_generate_ids(ids, max_tokens=s.get("max_tokens", DEFAULT_MAX_TOKENS), eos_id=s.get("eos_id"),
                                      temperature=s.get("temperature", DEFAULT_TEMPERATURE), top_p=s.get("top_p", DEFAULT_TOP_P))
        return [self.tokenizer.decode(g) for g in got]

    def generate(self, prompt: str, settings: Optional[dict] = None) -> str:
        return self.batch_generate([prompt], settings)[0]
