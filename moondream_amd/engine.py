"""What every model of the framework shares on the host side: device memory arenas, streams, sampling and the lockstep decode loop.

A model derives from ``DeviceEngine``, owns its weights and its cache, and hands ``_lockstep_loop`` one device-resident decode
step; the loop (eager, or replayed from captured hipGraphs in chunks), the choice of tokens, the end-of-sequence rule and the
truncation of what a caller gets are here.
"""
from __future__ import annotations

import contextlib
import ctypes as C
import gc
from typing import Any, Callable, Dict, List, Optional, Sequence, Union

import torch

from . import _lib

BF16 = torch.bfloat16

DEFAULT_MAX_TOKENS = 768
DEFAULT_TEMPERATURE = 0.5
DEFAULT_TOP_P = 0.3


@contextlib.contextmanager
def no_collection():
    """Keeps Python's cyclic collector out of a graph capture.  A captured graph that is part of a cycle (a model whose graphs refer back to it)
    is freed by the collector, at whatever allocation that happens to run; freeing a graph synchronises the device, which a capture
    forbids: the graph's destructor then ends the process."""
    was = gc.isenabled()
    gc.disable()
    try:
        yield
    finally:
        if was:
            gc.enable()


class DeviceEngine:
    def _init_device(self, device: Union[str, torch.device], lm_only: bool = False) -> None:
        self.lib = _lib.load(lm_only=lm_only)  # raises when the HIP library has not been built
        self._device = torch.device(device)
        if self._device.type != "cuda":
            raise _lib.MoondreamHipError(f"{type(self).__name__} needs a GPU device; there is no CPU path")
        self._arenas: Dict[int, torch.Tensor] = {}
        self._graphs: Dict[Any, Any] = {}
        self.use_graphs = False

    # ------------------------------------------------------------------ infra
    @property
    def device(self) -> torch.device:
        return self._device

    def _stream(self) -> C.c_void_p:
        return C.c_void_p(torch.cuda.current_stream(self._device).cuda_stream)

    def _h2d(self, t: torch.Tensor) -> torch.Tensor:
        """Small host tensor -> device WITHOUT stalling the host: a copy from pageable memory blocks the calling thread until the
        stream has reached it (on the pipelined engine's streams: until the whole encode in front of it has run); from pinned
        memory it is queued like a kernel."""
        if t.device.type != "cpu":
            return t.to(self._device)
        with torch.inference_mode(False):
            pinned = torch.empty(t.shape, dtype=t.dtype, pin_memory=True)
        pinned.copy_(t)
        return pinned.to(self._device, non_blocking=True)

    def _workspace(self, nbytes: int, which: int = 0) -> torch.Tensor:
        """Caller-owned arenas for the C ABI.  0: encode-side stages, 1: lm_head of the
        prompt prefill, 2: the decode loop (its own arena so that a decode running on
        the decode stream never shares scratch with an encode on the encode stream)."""
        ws = self._arenas.get(which)
        if ws is None or ws.numel() < nbytes:
            ws = torch.empty(int(nbytes * 1.05) + 4096, dtype=torch.uint8, device=self._device)
            self._arenas[which] = ws
            self._graphs.clear()
        return ws

    def compile(self):
        """The reference rebinds the seam to torch.compile'd functions here
        (moondream.py:194-204).  The seam is already native; ``compile`` turns on
        hipGraph replay of the device-resident decode step."""
        self.use_graphs = True

    # --------------------------------------------------------------- sampling
    def _pick(self, logits: torch.Tensor, temperature: float, top_p: float, suppress_id: int = -1,
              generator: Optional[torch.Generator] = None, probs_out: Optional[torch.Tensor] = None,
              vocab: Optional[int] = None) -> torch.Tensor:
        """[B,V] -> int32 [B]   (reference: moondream.py:313-318,521-528).  Greedy: argmax, ties to the
        lowest id.  Otherwise temperature + top-p on the device (md_sample_top_p): the reference's
        softmax / _apply_top_p / multinomial semantics with one uniform per sequence from torch's
        generator (same distribution as torch.multinomial, different random stream).  ``vocab``: rows that are
        longer than the vocabulary (padded heads)."""
        b, v = logits.shape[0], int(vocab or logits.shape[1])
        nxt = torch.empty(b, dtype=torch.int32, device=self._device)
        if temperature == 0:
            name = "md_argmax_f32" if logits.dtype == torch.float32 else "md_argmax_bf16"
            _lib.check(getattr(self.lib, name)(logits.data_ptr(), logits.stride(0), b, v, suppress_id, nxt.data_ptr(), self._stream()), name)
            return nxt
        u = torch.rand(b, device=self._device, dtype=torch.float32, generator=generator)
        self._sample_into(logits, v, temperature, top_p, suppress_id, u, nxt, probs_out)
        return nxt

    def _sample_into(self, logits, vocab: int, temperature: float, top_p: float, suppress_id: int, u, nxt, probs_out=None) -> None:
        if logits.dtype != BF16:
            logits = logits.to(BF16)  # the sampling rule is defined on bf16 logits
        _lib.check(
            self.lib.md_sample_top_p(
                logits.data_ptr(), logits.stride(0), logits.shape[0], vocab, suppress_id, float(temperature), float(top_p), u.data_ptr(),
                nxt.data_ptr(), probs_out.data_ptr() if probs_out is not None else None,
                probs_out.stride(0) if probs_out is not None else 0, self._stream(),
            ),
            "md_sample_top_p",
        )

    @staticmethod
    def _truncate(seq: List[int], eos_id: Optional[int], max_tokens: int) -> List[int]:
        out = []
        for tok in seq:
            if (eos_id is not None and tok == eos_id) or len(out) >= max_tokens:
                break
            out.append(tok)
        return out

    # ------------------------------------------------------------ decode loop
    def _lockstep_loop(self, first: torch.Tensor, pos: Sequence[int], max_tokens: int, make_step: Callable, graph_key: tuple,
                       eos_id: Optional[int], check_every: int = 16, uniforms: Optional[torch.Tensor] = None,
                       graphs: Optional[bool] = None, keep: Sequence[torch.Tensor] = ()) -> torch.Tensor:
        """Device-resident lockstep decode: int32 [steps + 1, B], row 0 = ``first``.  ``make_step(pos_buf)`` binds a position buffer
        (device int32 [B], advanced by the step itself) and returns ``step(tok_in, tok_out, uniform_row)``, which queues one decode
        step.  ``uniforms`` [max_tokens, B]: one draw per (step, sequence) of a sampled decode.  With ``compile()`` the steps are
        replayed from a hipGraph in chunks; ``graph_key`` names everything the captured launches depend on, ``keep`` holds the tensors
        they read that nothing else keeps (a kept graph must not refer to the model: see no_collection)."""
        b = first.shape[0]
        hist = torch.zeros(max_tokens + 1, b, dtype=torch.int32, device=self._device)
        hist[0] = first
        if max_tokens == 0:
            return hist
        pos_base = self._h2d(torch.tensor(list(pos), dtype=torch.int32))

        def all_done(upto):
            return eos_id is not None and bool((hist[: upto + 1] == eos_id).any(dim=0).all())

        steps = 0
        if not (self.use_graphs if graphs is None else graphs):
            step = make_step(pos_base.clone())
            while steps < max_tokens:
                step(hist[steps], hist[steps + 1], uniforms[steps] if uniforms is not None else None)
                steps += 1
                if check_every and steps % check_every == 0 and all_done(steps):
                    break
            return hist[: steps + 1]

        # ---- hipGraph path: one graph = `chunk` consecutive steps over fixed buffers
        chunk = max(1, min(check_every or 16, max_tokens))
        while steps < max_tokens:
            n = min(chunk, max_tokens - steps)
            # a graph is replayed only on the stream (context) it was captured for: the pipelined engine's
            # decode stream and the default stream each keep their own captures
            key = ("decode", b, n, torch.cuda.current_stream(self._device).cuda_stream) + tuple(graph_key)
            entry = self._graphs.get(key)
            if entry is None:
                buf = torch.zeros(n + 1, b, dtype=torch.int32, device=self._device)
                pos_buf = torch.zeros(b, dtype=torch.int32, device=self._device)
                u_buf = torch.zeros(n, b, dtype=torch.float32, device=self._device)
                step = make_step(pos_buf)
                # eager warm-up on scratch state is not possible (KV side effects), so the
                # first chunk of a new shape runs eagerly and the graph is captured afterwards
                buf[0] = hist[steps]
                pos_buf.copy_(pos_base + steps)
                if uniforms is not None:
                    u_buf.copy_(uniforms[steps : steps + n])
                for i in range(n):
                    step(buf[i], buf[i + 1], u_buf[i])
                hist[steps + 1 : steps + n + 1] = buf[1:]
                torch.cuda.synchronize(self._device)
                g = torch.cuda.CUDAGraph()
                with no_collection(), torch.cuda.graph(g):
                    for i in range(n):
                        step(buf[i], buf[i + 1], u_buf[i])
                # the capture did not execute; nothing to undo
                self._graphs[key] = (g, buf, pos_buf, u_buf, keep)
            else:
                g, buf, pos_buf, u_buf, _ = entry
                buf[0] = hist[steps]
                pos_buf.copy_(pos_base + steps)
                if uniforms is not None:
                    u_buf.copy_(uniforms[steps : steps + n])
                g.replay()
                hist[steps + 1 : steps + n + 1] = buf[1:]
            steps += n
            if all_done(steps):
                break
        return hist[: steps + 1]
