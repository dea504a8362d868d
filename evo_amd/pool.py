"""Continuous batching of decode streams: the `semantic_design.sample_model` usage profile --
many prompts x `n_sample_per_prompt` generations of `n_tokens` each [REF semantic_design/semantic_design.py:271-360,
121-179].

The reference's `generate` batches only prompts of EQUAL length and otherwise generates one prompt at a time
[REF evo/generation.py:237-262]: a decode step streams all 12.9 GB of weights for a single token.  Here a fixed set
of `n_slots` decode streams shares every step.  Each slot owns one row of every cache tensor (KV rows, FIR history,
modal state) and its own position, held in DEVICE memory: the rotary table, the KV append and the split-K decode
attention all read per-row positions (`evo_attn_decode_bf16` dyn_pos[B]), so streams of different prompt lengths
and different ages advance together, a finished stream's slot is re-filled while the others keep going, and the
step has one shape for the whole job -- it is captured once in a hipGraph and replayed.

Prompts are prefilled with the model's parallel launches (`model.prefill_rows`), all prompts that find a slot as one packed pass where they
can share one; StripedHyena's long-convolution kernel ends every prompt with its exact modal state.  The `n_sample_per_prompt` copies of a prompt share ONE prefill, whose caches are replicated into their slots.  The
pool's own steps -- admit, advance, release -- serve callers that bring their own tokens (evo_amd/trace.py).

Sampling and scoring follow the reference wrapper verbatim (same `sample`, same shifted logits/token pairing
[REF evo/generation.py:162-167,287]), so with greedy sampling a pool run reproduces per-prompt `generate` token for token
(tests/test_pool.py).
"""
from __future__ import annotations

from collections import deque
from typing import Dict, List, Optional, Sequence, Tuple

import numpy as np
import torch

from .scoring import logits_to_logprobs, prepare_batch
from .sh.sample import sample


class DecodePool:
    def __init__(self, model, tokenizer, n_slots: int = 8, top_k: int = 4, top_p: float = 1.0,
                 temperature: float = 0.7, device: Optional[str] = None, use_graph: Optional[bool] = None):
        self.model = model
        self.tok = tokenizer
        self.n_slots = int(n_slots)
        self.top_k, self.top_p, self.temperature = top_k, top_p, temperature
        self.device = torch.device(device) if device is not None else model.device
        self.use_graph = (self.device.type == "cuda" and getattr(model, "decode_graph", False)) \
            if use_graph is None else bool(use_graph)
        self.ipd = None
        self.capacity = 0
        self._graph = None
        self.free: List[int] = []
        self.length: Dict[int, int] = {}             # live slot -> tokens its caches hold (the host's copy of self.pos)
        self.stats = {"steps": 0, "prefills": 0, "tokens": 0}

    # ------------------------------------------------------------------ cache rows
    def _allocate(self, capacity: int, n_slots: Optional[int] = None) -> None:
        """Pool-wide caches with `capacity` positions per slot (grown geometrically, outside any captured graph); live slots are kept."""
        S, dev, old = max(self.n_slots, n_slots or 0), self.device, self.ipd
        have = 0 if old is None else self.pos.numel()
        if old is not None and capacity <= self.capacity and S <= have:
            return
        if old is not None and capacity > self.capacity:
            capacity = max(capacity, 2 * self.capacity)
        self.capacity = max(capacity, self.capacity)
        self.ipd = self.model.allocate_rows(S, self.capacity, old)
        self._graph = None
        pos, ids = torch.zeros(S, dtype=torch.int64, device=dev), torch.zeros(S, 1, dtype=torch.int64, device=dev)
        if old is not None:
            pos[:have], ids[:have] = self.pos, self.ids
        self.pos, self.ids, self.n_slots = pos, ids, S
        self.free += range(have, S)

    # ------------------------------------------------------------------ steps: admit, advance, release
    def prefill(self, prompts: Sequence[torch.Tensor], want: Optional[List[List[int]]] = None):
        """Runs whole prompts ([P] ids each) -> [(logits f32 of the wanted places -- the last token by default --, caches, row)], the form
        `install` takes.  A model that packs unequal prompts runs them as one batch (model.prefill_rows)."""
        with torch.inference_mode():
            got = self.model.prefill_rows([p.reshape(-1) for p in prompts], want)
        self.stats["prefills"] += len(got)
        return [(lg.float(), ipd, row) for lg, ipd, row in got]

    def install(self, prefilled, n_tokens: int, reserve: int = 1) -> int:
        """Takes a free slot for a prefilled sequence of `n_tokens` tokens (one more slot if none is free) and returns it."""
        return self._install([prefilled], [n_tokens], reserve)[0]

    def _install(self, prefilled, n_tokens: Sequence[int], reserve: int) -> List[int]:
        """Slots for several prefilled sequences; their states move in one launch where the ops have one for it."""
        slots, pieces, ops = [], [], self.model.ops
        for n in n_tokens:
            self._allocate(max(n + reserve, self.capacity), len(self.length) + 1)
            slots.append(self.free.pop(0))
            self.length[slots[-1]] = n
        with torch.inference_mode():
            for (_, ipd, row), slot, n in zip(prefilled, slots, n_tokens):
                if hasattr(ops, "copy_rows") and hasattr(self.model, "row_pieces"):
                    pieces += self.model.row_pieces(self.ipd, slot, ipd, row, n)
                else:
                    self.model.copy_row(self.ipd, slot, ipd, row, n)
            if pieces:
                ops.copy_rows(pieces)
        if slots:
            self._put(self.pos, slots, n_tokens)                      # where the slots' next tokens sit
        return slots

    def _put(self, where: torch.Tensor, slots: Sequence[int], values) -> None:
        """where[slot] = value for host integers: a launch without a copy from host memory where the ops have one."""
        put = getattr(self.model.ops, "put_tokens", None)
        if put is not None and where.is_cuda and 0 < len(slots) <= self.model.ops.MAX_PUT:
            put(where, slots, list(values))
        else:
            where.view(-1)[torch.tensor(slots).to(self.device)] = torch.tensor(list(values), dtype=torch.int64).to(self.device)

    def admit(self, prompts: Sequence[torch.Tensor], want: Optional[List[List[int]]] = None, reserve: int = 1):
        """Starts sequences: one batch of prompts -> (slots, wanted logits f32 per prompt)."""
        prompts = [p.to(self.device) for p in prompts]
        if self.ipd is None or len(self.free) < len(prompts):
            self._allocate(max(max(p.numel() for p in prompts) + reserve, self.capacity), len(self.length) + len(prompts))
        got = self.prefill(prompts, want)
        return self._install(got, [p.numel() for p in prompts], reserve), [g[0] for g in got]

    def advance(self, tokens: Dict[int, int]) -> torch.Tensor:
        """The next token of each given slot, in one pooled step -> logits [S, V] f32 (rows of the other slots mean nothing)."""
        slots = list(tokens)
        self._put(self.ids, slots, tokens.values())
        return self._advance(slots)

    def _advance(self, slots: Sequence[int]) -> torch.Tensor:
        """self.ids holds every given slot's next token."""
        if max(self.length[s] for s in slots) >= self.capacity:
            self._allocate(2 * self.capacity)
            for s, n in self.length.items():
                self.pos[s] = n
        logits = self._step()
        for s in slots:
            self.length[s] += 1
        return logits

    def release(self, slot: int) -> None:
        """Gives a slot back; whatever it holds is overwritten by its next owner."""
        del self.length[slot]
        self.free.append(slot)

    # ------------------------------------------------------------------ one token for every slot
    def _step_eager(self) -> torch.Tensor:
        m, mha = self.model, self.ipd["mha"]
        mha.pos_tensor = self.pos
        try:
            h = m.hidden_states(self.ids, self.ipd)
            return m.ops.linear(h, m.unembed.weight, None).view(self.n_slots, m.vocab_size)
        finally:
            mha.pos_tensor = None

    def _finish(self, logits: torch.Tensor) -> torch.Tensor:
        """The step's logits in fp32, a tensor of their own; the positions move on."""
        ops = self.model.ops
        if hasattr(ops, "step_out") and logits.is_cuda and logits.dtype == torch.bfloat16 and logits.is_contiguous() and self.pos.is_contiguous():
            return ops.step_out(logits, self.pos, self.capacity - 1)
        out = logits.float()
        self._next_positions()
        return out

    def _next_positions(self) -> None:
        """(free slots drift harmlessly; a full live slot grows the caches first)"""
        if self.pos.is_cuda and hasattr(self.model.ops, "advance_positions"):
            self.model.ops.advance_positions(self.pos, self.capacity - 1)
        else:
            self.pos += 1
            self.pos.clamp_(max=self.capacity - 1)

    def _step(self) -> torch.Tensor:
        """self.ids [S,1] at positions self.pos [S] -> logits [S, V] f32 (every slot, active or not); the positions move on."""
        self.stats["steps"] += 1
        with torch.inference_mode():
            if not self.use_graph or not self.model._graph_shapes_ok(self.n_slots):
                return self._finish(self._step_eager())
            if self._graph is None:
                # The first step runs eagerly (it also warms the library handles and the M = S GEMM choices) and IS the
                # step: the caches advance in place, so nothing may run twice.  Capture records without executing.
                first = self._finish(self._step_eager())
                torch.cuda.synchronize(self.device)
                self.model._graph_prepare(self.n_slots, self.device)
                g = torch.cuda.CUDAGraph()
                with torch.cuda.graph(g):
                    out = self._step_eager()
                self._graph = (g, out)
                return first
            g, out = self._graph
            g.replay()
            return self._finish(out)

    # ------------------------------------------------------------------ the job
    def generate(self, prompts: Sequence[str], n_tokens: int = 1000, n_sample_per_prompt: int = 1,
                 prepend_bos: bool = False) -> Tuple[List[str], List[float], List[int]]:
        """Returns (generated strings, mean log-likelihood scores, index of the prompt each came from), in job
        order: prompt 0's samples first."""
        m, tok, S, dev = self.model, self.tok, self.n_slots, self.device
        if hasattr(m, "eval"):
            m.eval()
        n_tokens = int(n_tokens)
        if n_tokens < 1 or int(n_sample_per_prompt) < 1:
            raise ValueError("n_tokens and n_sample_per_prompt must be >= 1")
        prompts = list(prompts)
        if not prompts:
            return [], [], []
        if any((not isinstance(p, str)) or (len(p) == 0 and not prepend_bos) for p in prompts):
            raise ValueError("every prompt must be a non-empty string (or use prepend_bos=True)")
        encoded = [prepare_batch([p], tok, prepend_bos=prepend_bos, device=str(dev))[0] for p in prompts]
        self._allocate(max(e.shape[1] for e in encoded) + n_tokens)
        S = self.n_slots
        # job = (output index, prompt index); the copies of one prompt are adjacent so that they share a prefill
        jobs = deque((pi * n_sample_per_prompt + c, pi) for pi in range(len(prompts)) for c in range(n_sample_per_prompt))
        n_jobs = len(jobs)
        out_ids = torch.zeros(n_jobs, n_tokens, dtype=torch.long)
        out_logits = torch.zeros(n_jobs, n_tokens, m.vocab_size, dtype=torch.float32)
        job_of: Dict[int, int] = {}                                    # slot -> job
        made: Dict[int, int] = {}                                      # slot -> tokens generated
        cached_prefill: Dict[int, tuple] = {}

        def fill() -> None:
            j, pi = jobs.popleft()
            if pi not in cached_prefill:
                cached_prefill.clear()                               # keep the caches of one batch of prompts alive at a time
                ahead = [pi]
                if getattr(m, "packs_prompts", False):               # the prompts of the other free slots ride in the same pass
                    ahead += list(dict.fromkeys(p for _, p in list(jobs)[: max(0, len(self.free) - 1)] if p != pi))
                cached_prefill.update(zip(ahead, self.prefill([encoded[p] for p in ahead])))
            last_logits = cached_prefill[pi][0][-1]
            first = sample(last_logits[None], top_k=self.top_k, top_p=self.top_p, temperature=self.temperature)
            out_ids[j, 0] = int(first[0])
            out_logits[j, 0] = last_logits.cpu()
            if n_tokens == 1:
                return
            slot = self.install(cached_prefill[pi], encoded[pi].numel(), n_tokens)   # the sampled token sits behind the prompt
            self.ids[slot, 0] = first[0]
            job_of[slot], made[slot] = j, 1

        try:
            while jobs or job_of:
                while jobs and (self.free or n_tokens == 1):
                    fill()
                if not job_of:
                    continue
                active = sorted(job_of)
                logits = self._advance(active)          # [S, V]
                nxt = sample(logits, top_k=self.top_k, top_p=self.top_p, temperature=self.temperature)
                lg_cpu, nxt_cpu = logits.cpu(), nxt.cpu()
                self.ids[:, 0] = nxt
                for s in active:
                    j, k = job_of[s], made[s]
                    out_ids[j, k] = nxt_cpu[s]
                    out_logits[j, k] = lg_cpu[s]
                    made[s] = k + 1
                    self.stats["tokens"] += 1
                    if k + 1 == n_tokens:
                        del job_of[s]
                        self.release(s)
        finally:
            for s in job_of:                                          # (an interrupted job gives its slots back)
                self.release(s)

        self.last_ids, self.last_logits = out_ids, out_logits        # (kept for inspection / tests)
        seqs = list(tok.detokenize_batch(out_ids))
        lp = logits_to_logprobs(out_logits, out_ids).float().numpy()   # the reference's shifted pairing
        scores = [float(np.mean(lp[j])) for j in range(n_jobs)]
        owner = [pi for pi in range(len(prompts)) for _ in range(n_sample_per_prompt)]
        return seqs, scores, owner


def sample_many(prompts: Sequence[str], model, tokenizer, n_tokens: int = 1000, temp: float = 0.7, top_k: int = 4,
                top_p: float = 1.0, n_sample_per_prompt: int = 1, n_slots: int = 8, prepend_bos: bool = False,
                device: Optional[str] = None):
    """`semantic_design.run_model` / `sample_model` without the equal-length restriction: (prompts repeated per
    sample, generated sequences, scores)."""
    pool = DecodePool(model, tokenizer, n_slots=n_slots, top_k=top_k, top_p=top_p, temperature=temp, device=device)
    seqs, scores, owner = pool.generate(prompts, n_tokens=n_tokens, n_sample_per_prompt=n_sample_per_prompt,
                                        prepend_bos=prepend_bos)
    return [prompts[i] for i in owner], seqs, scores
