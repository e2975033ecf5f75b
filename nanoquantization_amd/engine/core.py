"""The model-independent half of the engine: leases of cache blocks and state slots, the static decode state and its
HIP graph, and the schedulers.

A model's engine subclasses EngineCore and supplies
  _prefill(ids [b, s], leases)          equal-length prompts from position 0 -> next token of each, int64 [b]
  _prefill_ragged(prompts, leases)      the same for prompts of any lengths in one pass
  _decode_step()                        one token per batch row, from and to the static device buffers below
All per-step state lives in fixed device buffers (token ids, positions, active mask, block table, state slots, step
counter, output tokens) and the step advances that state itself, so it is captured once in a HIP graph and replayed
with no host work between steps.

Scheduling.  `generate` runs one static batch of equal-length prompts.  `serve` is continuous batching over the same
decode graph: requests of any length wait in a queue, are admitted whenever a batch row, enough cache blocks and (for
models with recurrent layers) a state slot are free, decode together with whatever else is running, and give their row,
blocks and slot back when they reach their token budget or the end-of-sequence token.
"""
from __future__ import annotations

from typing import List, Optional

import numpy as np
import torch

from . import ops
from .cache import Lease, PagedKVCache, RecurrentStateCache, upload


def _offsets(fields):
    """Where fields (name, numpy type, shape) lie one after the other, each on a multiple of 256 bytes."""
    at = 0
    for _, kind, shape in fields:
        yield at
        at += -(-int(np.prod(shape)) * np.dtype(kind).itemsize // 256) * 256


class EngineCore:
    cache: PagedKVCache
    states: Optional[RecurrentStateCache] = None     # set by engines of models with recurrent layers
    step_ops = ops                                   # the module with this engine's argmax_rows and decode_advance

    def __init__(self, device: torch.device, dtype: torch.dtype, max_batch: int, max_seq_len: int, block_size: int,
                 num_blocks: Optional[int], use_graph: bool):
        self.device, self.dtype = device, dtype
        if self.device.type != "cuda":
            raise RuntimeError(f"{type(self).__name__} needs the model on a HIP device")
        self.max_batch, self.block_size = max_batch, block_size
        self.max_blocks = (max_seq_len + block_size - 1) // block_size
        self.max_ctx = self.max_blocks * block_size
        self.num_blocks = max_batch * self.max_blocks if num_blocks is None else num_blocks
        self.use_graph = use_graph
        self._graph = None
        B, dev = max_batch, self.device
        # static decode state, advanced on the device by the step itself; one buffer, so that `decode` sets it in one copy
        fields = [("s_ids", np.int64, (B,)),                    # token fed at this step
                  ("s_pos", np.int64, (B,)),                    # its position
                  ("s_step", np.int64, (1,)),                   # row of s_out the step writes
                  ("s_table", np.int32, (B, self.max_blocks)),
                  ("s_slot", np.int32, (B,)),                   # recurrent-state slot of the row
                  ("s_active", np.bool_, (B,))]                 # rows that own cache blocks
        self._state_fields = np.dtype({"names": [f[0] for f in fields], "formats": [f[1:] for f in fields],
                                       "offsets": list(_offsets(fields))})
        self._decode_state = torch.zeros(self._state_fields.itemsize, dtype=torch.uint8, device=dev)
        for name, kind, shape in fields:
            at = self._state_fields.fields[name][1]
            part = self._decode_state[at:at + int(np.prod(shape)) * np.dtype(kind).itemsize]
            setattr(self, name, part.view(getattr(torch, np.dtype(kind).name)).view(shape))
        self.s_out = torch.zeros(self.max_ctx + 1, B, dtype=torch.long, device=dev)
        self.s_logits: Optional[torch.Tensor] = None                    # logits of the last decode step [B, vocab]

    def _prefill(self, ids: torch.Tensor, leases: List[Lease]) -> torch.Tensor:
        raise NotImplementedError

    def _prefill_ragged(self, prompts: List[List[int]], leases: List[Lease]) -> torch.Tensor:
        raise NotImplementedError

    def _decode_step(self) -> None:
        raise NotImplementedError

    def _follow_weights(self) -> bool:
        """Weights that the engine keeps in a layout of its own for its steps alone, as the modules hold them now: whether any had changed."""
        return False

    # ---- leases ----------------------------------------------------------------------------------
    def acquire(self, num_blocks: int) -> Lease:
        lease = Lease(self.cache.allocate(num_blocks))
        if self.states is not None:
            try:
                lease.slot = self.states.allocate()
            except RuntimeError:
                self.cache.release(lease.blocks)
                raise
        return lease

    def release(self, lease: Lease) -> None:
        self.cache.release(lease.blocks)
        lease.blocks = []
        if self.states is not None and lease.slot >= 0:
            self.states.release(lease.slot)
            lease.slot = -1

    def _set_row(self, row: int, lease: Lease) -> None:
        blocks = lease.blocks
        self.s_table[row] = torch.tensor(blocks + [0] * (self.max_blocks - len(blocks)), dtype=torch.int32)
        self.s_slot[row] = lease.slot

    def grow(self, lease: Lease, num_tokens: int) -> None:
        """Room for `num_tokens` tokens in all: blocks are added, none are given back."""
        need = (num_tokens + self.block_size - 1) // self.block_size
        if need > self.max_blocks:
            raise ValueError(f"{num_tokens} tokens exceed max_seq_len")
        if need > len(lease.blocks):
            lease.blocks += self.cache.allocate(need - len(lease.blocks))

    # ---- decode ----------------------------------------------------------------------------------
    @torch.no_grad()
    def decode(self, rows) -> torch.Tensor:
        """One decode step for (lease, position, token) rows, at most max_batch, whose next token is given rather than
        sampled: the logits [len(rows), vocab] (valid until the next step).  Runs the step `generate` runs."""
        n = len(rows)
        if not 1 <= n <= self.max_batch:
            raise ValueError(f"{n} rows, the engine takes 1 to {self.max_batch}")
        # the whole state in one copy from pinned memory that does not wait for the step before (a copy per row and field did,
        # and took longer than a step)
        state = np.zeros((), dtype=self._state_fields)
        for i, (lease, pos, token) in enumerate(rows):
            if pos >= len(lease.blocks) * self.block_size:
                raise ValueError(f"position {pos} has no cache block")
            state["s_ids"][i], state["s_pos"][i], state["s_slot"][i] = int(token), int(pos), lease.slot
            state["s_table"][i, :len(lease.blocks)] = lease.blocks
        state["s_active"][:n] = True
        def step():
            upload(state.reshape(1).view(np.uint8), self.device, out=self._decode_state)
            self._run_decode()
        step()
        # looked at while the step runs; where something had changed the step is taken again, from the same state to the same cache slots
        if self._follow_weights():
            step()
        return self.s_logits[:n]

    def _finish_step(self, logits: torch.Tensor) -> None:
        self.s_logits = logits
        nxt = self.step_ops.argmax_rows(logits)
        # log the tokens, feed them back, move the active rows on (idle rows stay where they are), count the step
        self.step_ops.decode_advance(nxt, self.s_active, self.s_out, self.s_ids, self.s_pos, self.s_step)

    def _state(self):
        return [self.s_ids, self.s_pos, self.s_step]

    def _run_decode(self) -> None:
        if not self.use_graph:
            self._decode_step()
            return
        if self._graph is None:
            active = self.s_active.clone()
            saved = [t.clone() for t in self._state()]
            s = torch.cuda.Stream()
            s.wait_stream(torch.cuda.current_stream())
            with torch.cuda.stream(s):
                self.s_active.zero_()       # the rehearsal may write neither cache blocks nor recurrent state
                for _ in range(2):          # warm-up: workspaces and library handles exist before capture
                    self._decode_step()
                    for t, v in zip(self._state(), saved):   # the step advanced the state: put it back
                        t.copy_(v)
                self.s_active.copy_(active)
                torch.cuda.synchronize()
                g = torch.cuda.CUDAGraph()
                with torch.cuda.graph(g, stream=s):
                    self._decode_step()
            torch.cuda.current_stream().wait_stream(s)
            self._graph = g
        self._graph.replay()

    @torch.no_grad()
    def generate(self, prompts: List[List[int]], max_new_tokens: int, stats: Optional[dict] = None) -> List[List[int]]:
        """Greedy continuation of each prompt (token-id lists of equal length), `max_new_tokens` each.
        If `stats` is given it receives prefill_s / decode_s wall times (device-synchronised)."""
        import time
        n = len(prompts)
        if n == 0:
            return []
        if n > self.max_batch:
            raise ValueError(f"{n} prompts exceed max_batch={self.max_batch}")
        plen = len(prompts[0])
        if any(len(p) != plen for p in prompts):
            raise ValueError("this engine batches prompts of equal length only")
        if plen + max_new_tokens > self.max_ctx:
            raise ValueError("prompt + max_new_tokens exceeds max_seq_len")
        self._follow_weights()
        leases: List[Lease] = []
        try:
            for _ in range(n):
                leases.append(self.acquire(self.max_blocks))
            ids = torch.tensor(prompts, dtype=torch.long, device=self.device)
            torch.cuda.synchronize()
            t0 = time.perf_counter()
            nxt = self._prefill(ids, leases)
            out = [nxt.tolist()]
            t1 = time.perf_counter()
            # batch rows beyond n mirror row 0 (same token, position and table) but are marked idle:
            # they recompute row 0's token and write nothing to the cache
            rows = list(range(n)) + [0] * (self.max_batch - n)
            self.s_table.copy_(torch.tensor([l.blocks for l in leases], dtype=torch.int32)[rows])
            self.s_slot.copy_(torch.tensor([l.slot for l in leases], dtype=torch.int32)[rows])
            self.s_active.copy_(torch.tensor([True] * n + [False] * (self.max_batch - n)))
            self.s_ids.copy_(nxt[rows] if n < self.max_batch else nxt)
            self.s_pos.fill_(plen)                                   # position of the token being fed
            self.s_step.zero_()
            steps = max_new_tokens - 1
            for _ in range(steps):
                self._run_decode()
            toks = self.s_out[:steps, :n].tolist()                   # one synchronisation for the whole run
            out.extend(toks)
            if stats is not None:
                torch.cuda.synchronize()
                stats.update(prefill_s=t1 - t0, decode_s=time.perf_counter() - t1, decode_steps=max_new_tokens - 1,
                             batch=n, prompt_len=plen)
            return [[out[s][i] for s in range(len(out))] for i in range(n)]
        finally:
            for lease in leases:
                self.release(lease)

    # ---- continuous batching ---------------------------------------------------------------------------
    @torch.no_grad()
    def serve(self, requests, eos_token_id: Optional[int] = None, stats: Optional[dict] = None,
              batch_prefill: bool = False, max_prefill_tokens: int = 8192) -> List[List[int]]:
        """requests: sequence of (prompt token ids, max_new_tokens), any lengths.  Returns the greedy continuation
        of each request, in request order (cut after `eos_token_id` if one is given).  Without an end-of-sequence
        token the host reads tokens back only when the output buffer fills up or at the end; with one it reads
        them after every step.

        By default every admitted request is prefilled on its own, so its tokens do not depend on what else is
        queued or running (decode rows are independent as well).  `batch_prefill` prefills all requests admitted at
        the same moment in one pass (up to `max_prefill_tokens` prompt tokens): fewer, larger launches, but the row
        count of the prefill linears -- and with it their kernel and summation order -- then depends on the
        company a request arrives in."""
        import time
        from collections import deque
        bs = self.block_size
        for prompt, max_new in requests:
            if len(prompt) < 1 or max_new < 1:
                raise ValueError("every request needs a non-empty prompt and max_new_tokens >= 1")
            if len(prompt) + max_new > self.max_ctx:
                raise ValueError("prompt + max_new_tokens exceeds max_seq_len")
        self._follow_weights()
        out: List[List[int]] = [[] for _ in requests]
        waiting = deque(range(len(requests)))
        free_rows = list(range(self.max_batch - 1, -1, -1))
        running = {}                      # row -> [request index, tokens still to decode, lease]
        step_log = []                     # per decode step since the last read-back: [(row, request index)]
        self.s_active.zero_(); self.s_pos.zero_(); self.s_ids.zero_(); self.s_table.zero_(); self.s_step.zero_()
        torch.cuda.synchronize()
        t_start, n_steps, n_prefill, n_prefill_calls = time.perf_counter(), 0, 0, 0
        prefill_log = []                  # per prefill pass: (prompt tokens, requests, decode steps so far, seconds)

        def retire(row):
            self.release(running.pop(row)[2])
            free_rows.append(row)
            self.s_active[row] = False
            self.s_pos[row] = 0

        def read_back():
            """Tokens of the logged steps -> their requests; returns the rows whose request ended with eos."""
            ended = []
            if step_log:
                toks = self.s_out[:len(step_log)].tolist()
                for i, entries in enumerate(step_log):
                    for row, ri in entries:
                        if out[ri] and eos_token_id is not None and out[ri][-1] == eos_token_id:
                            continue            # already ended on an earlier step of this batch of steps
                        out[ri].append(toks[i][row])
                        if eos_token_id is not None and toks[i][row] == eos_token_id and row in running \
                                and running[row][0] == ri:
                            ended.append(row)
                step_log.clear()
                self.s_step.zero_()
            return ended

        try:
            while waiting or running:
                # admit while a row and the blocks for the whole request are free
                admitted = []                 # (request index, lease), prefilled together if batch_prefill
                tokens_admitted = 0
                while waiting and len(admitted) < len(free_rows):
                    ri = waiting[0]
                    prompt, max_new = requests[ri]
                    need = (len(prompt) + max_new + bs - 1) // bs
                    if need > len(self.cache.free):
                        if not running and not admitted:
                            raise RuntimeError(f"KV cache too small for request {ri}: {need} blocks wanted, "
                                               f"{len(self.cache.free)} exist free with nothing running")
                        break
                    if admitted and (not batch_prefill or tokens_admitted + len(prompt) > max_prefill_tokens):
                        break
                    waiting.popleft()
                    admitted.append((ri, self.acquire(need)))
                    tokens_admitted += len(prompt)
                if admitted:
                    if stats is not None:
                        torch.cuda.synchronize()
                        t_pf = time.perf_counter()
                    try:
                        if len(admitted) == 1:
                            ids = torch.tensor([requests[admitted[0][0]][0]], dtype=torch.long, device=self.device)
                            toks = self._prefill(ids, [admitted[0][1]]).tolist()
                        else:
                            toks = self._prefill_ragged([requests[ri][0] for ri, _ in admitted],
                                                        [lease for _, lease in admitted]).tolist()
                    except Exception:
                        for _, lease in admitted:
                            self.release(lease)
                        raise
                    n_prefill += len(admitted)
                    n_prefill_calls += 1
                    if stats is not None:       # toks.tolist() above has waited for the pass
                        prefill_log.append((tokens_admitted, len(admitted), n_steps, time.perf_counter() - t_pf))
                    for (ri, lease), tok in zip(admitted, toks):
                        prompt, max_new = requests[ri]
                        out[ri].append(tok)
                        if max_new == 1 or tok == eos_token_id:
                            self.release(lease)
                            continue
                        row = free_rows.pop()
                        running[row] = [ri, max_new - 1, lease]
                        self._set_row(row, lease)
                        self.s_ids[row] = tok
                        self.s_pos[row] = len(prompt)
                        self.s_active[row] = True
                    if waiting and free_rows and len(admitted) > 0 and not batch_prefill:
                        continue              # one prefill per pass: admit the next request before decoding
                if not running:
                    continue
                self._run_decode()
                n_steps += 1
                step_log.append([(row, r[0]) for row, r in running.items()])
                done = []
                for row, r in running.items():
                    r[1] -= 1
                    if r[1] == 0:
                        done.append(row)
                if eos_token_id is not None or len(step_log) == self.s_out.shape[0]:
                    done.extend(row for row in read_back() if row not in done)
                for row in done:
                    retire(row)
            read_back()
        finally:
            for row in list(running):
                retire(row)
        if stats is not None:
            torch.cuda.synchronize()
            wall = time.perf_counter() - t_start
            prefill_s = sum(p[3] for p in prefill_log)
            stats.update(wall_s=wall, decode_steps=n_steps, prefills=n_prefill, prefill_calls=n_prefill_calls,
                         tokens=sum(len(o) for o in out), prefill_s=prefill_s, decode_s=wall - prefill_s,
                         prefill_log=prefill_log)
        return out
