"""Model runner — builds kernel batches and executes model steps.

Owns the device, model, KV pool and (optionally) the hipGraph-captured
decode path: decode steps at a given batch size are launch-bound (dozens of
small kernels), so the runner captures one graph per padded batch-size
bucket and replays it with fresh inputs copied into static buffers
(guide: "capture launch-bound inner loops in hipGraphs").  This is the
MI355X-native replacement for the model-execution half the reference
delegates to SGLang (SURVEY §2.3 prefill/decode engine rows).
"""
from __future__ import annotations

import gc
import logging
from typing import Dict, List, Optional, Tuple

import numpy as np
import torch

from ..models.llama import PPContext, TPContext
from ..models.registry import build_model
from ..ops import place_inputs
from ..utils.upload import upload
from .batch import ForwardBatch, VarlenLayout, table_array
from .config import EngineConfig
from .sequence import Sequence

log = logging.getLogger(__name__)

GRAPH_BATCH_SIZES = (1, 2, 4, 8, 16, 24, 32, 48, 64, 96, 128, 192, 256)


class ModelRunner:
    def __init__(self, cfg: EngineConfig, tp: Optional[TPContext] = None,
                 pp: Optional[PPContext] = None):
        self.cfg = cfg
        self.device = torch.device(cfg.device)
        torch.manual_seed(cfg.seed)
        self.pp = pp or PPContext()
        self.model = build_model(cfg.model, self.device, tp, self.pp)
        self.cache = self.model.make_cache(cfg)
        self.mixed_steps = (self.model.mixed_steps if cfg.mixed_steps is None
                            else bool(cfg.mixed_steps))
        if self.mixed_steps and not self.model.mixed_steps:
            raise ValueError(f"{cfg.model.name}: mixed steps not supported")
        self.max_pages_per_seq = (cfg.max_seq_len + cfg.page_size - 1) // \
            cfg.page_size
        self._graphs: Dict[int, Tuple] = {}
        self._graph_pool = None
        # device-resident decode inputs of the last batch composition
        self._dstate: Optional[dict] = None
        log.info("model %s on %s: %d KV pages (%.1f GB pool)",
                 cfg.model.name, self.device, self.cache.num_pages,
                 self.cache.kv.numel() * self.cache.kv.element_size() / 1e9)

    # ------------------------------------------------------------------

    def _index(self, rows: List[int]) -> torch.Tensor:
        return upload([np.array(rows, dtype=np.int64)], self.device)[0]

    # one sequence's part of a varlen step: tokens at [start, start + len)
    Chunk = Tuple[Sequence, int, List[int]]

    @torch.inference_mode()
    def run_chunks(self, chunks: List[Chunk]) -> Tuple[torch.Tensor,
                                                       List[int]]:
        """One varlen forward over portions of several sequences — a full
        prompt, a cached-prefix suffix, a piece of a long prompt or (models
        with mixed steps) a single decoded token beside them.  Returns the
        last stage's hidden rows and each chunk's first row; the rows of
        single-token chunks with a past come first."""
        order = list(range(len(chunks)))
        num_decode = 0
        if self.model.mixed_steps:
            single = [len(t) == 1 and start > 0 for _, start, t in chunks]
            num_decode = sum(single)
            order.sort(key=lambda i: not single[i])
        # numpy pieces: a step of many tokens is on the GPU's critical path
        tokens: List[np.ndarray] = []
        prev: List[np.ndarray] = []
        positions: List[np.ndarray] = []
        slots: List[np.ndarray] = []
        gather: List[np.ndarray] = []
        cu = [0]
        cu_k = [0]
        first_row = [0] * len(chunks)
        starts, ends, tables = [], [], []
        any_past = any(start > 0 for _, start, _ in chunks)
        for i in order:
            seq, start, toks = chunks[i]
            end = start + len(toks)
            tokens.append(np.asarray(toks, dtype=np.int64))
            if self.model.needs_prev:
                prev += [np.array([seq.token_at(start - 1)]), tokens[-1][:-1]]
            positions.append(np.arange(start, end, dtype=np.int32))
            slots.append(seq.block_table.slots_for(start, end - start))
            first_row[i] = cu[-1]
            cu.append(cu[-1] + (end - start))
            cu_k.append(cu_k[-1] + end)
            if any_past and not self.model.varlen:
                gather.append(seq.block_table.slots_for(0, end))
            starts.append(start)
            ends.append(end)
            tables.append(seq.block_table)
        # everything the step needs from the host is one transfer
        i32 = lambda a: np.asarray(a, dtype=np.int32)   # noqa: E731
        parts = {"tokens": np.concatenate(tokens),
                 "positions": np.concatenate(positions),
                 "slots": np.concatenate(slots), "cu": i32(cu)}
        if self.model.needs_prev:
            parts["prev"] = np.concatenate(prev)
        if self.model.varlen:
            parts["starts"] = i32(starts)
            parts["state_slots"] = i32([t.state_slot for t in tables])
            parts["cu_prefill"] = i32([c - num_decode
                                       for c in cu[num_decode:]])
            if num_decode:
                parts["tables"] = table_array(tables[:num_decode])
                parts["ends"] = i32(ends[:num_decode])
        elif any_past:
            parts["cu_k"] = i32(cu_k)
            parts["gather"] = np.concatenate(gather)
        dev = dict(zip(parts, upload(list(parts.values()), self.device)))
        batch = ForwardBatch(
            mode="prefill", positions=dev["positions"],
            slot_mapping=dev["slots"], cu_seqlens=dev["cu"], cu_host=cu,
            prev_tokens=dev.get("prev"), starts=dev.get("starts"),
            state_slots=dev.get("state_slots"),
            cu_prefill=dev.get("cu_prefill"),
            block_tables=dev.get("tables"), context_lens=dev.get("ends"),
            cu_seqlens_k=dev.get("cu_k"),
            cu_k_host=cu_k if "cu_k" in dev else None,
            kv_gather_slots=dev.get("gather"))
        if self.model.varlen:
            batch.num_decode = num_decode
            batch.layout = VarlenLayout(starts, ends, tables, num_decode,
                                        self.cfg.page_size, self.device)
        # decode inputs that were left on the device are behind now
        self._dstate = None
        hidden_in = None
        if not self.pp.first:
            hidden_in = self.pp.recv_prev(
                (cu[-1], self.model.stream_width),
                self.model.stream_dtype, self.device)
        hidden = self.model.forward(dev["tokens"], batch, self.cache,
                                    hidden=hidden_in)
        if not self.pp.last:
            self.pp.send_next(hidden)
        return hidden, first_row

    def prefill(self, seqs: List[Sequence]) -> List[int]:
        """One prefill step: each sequence contributes its current chunk
        [num_prefilled, num_prefilled + chunk_len).  Only sequences whose
        chunk reaches the prompt end get a token sampled."""
        return self.mixed(seqs, [])

    @torch.inference_mode()
    def mixed(self, prefills: List[Sequence],
              decodes: List[Sequence]) -> List[int]:
        """One step of prompt chunks and decoded tokens as one batch."""
        chunks: List[ModelRunner.Chunk] = []
        sampled: List[Sequence] = []
        at: List[int] = []              # chunk of each sampled sequence
        for seq in decodes:
            sampled.append(seq)
            at.append(len(chunks))
            chunks.append((seq, seq.num_tokens - 1, [seq.last_token]))
        for seq in prefills:
            start = seq.num_prefilled
            end = start + (seq.chunk_len or
                           (seq.num_prompt_tokens - start))
            if end == seq.num_prompt_tokens:
                sampled.append(seq)
                at.append(len(chunks))
            chunks.append((seq, start, seq.prompt_tokens[start:end]))
            seq.num_prefilled = end
        hidden, first_row = self.run_chunks(chunks)
        if not sampled:
            return []
        if self.pp.last:
            last = [first_row[i] + len(chunks[i][2]) - 1 for i in at]
            logits = self.model.logits(hidden, self._index(last))
            next_dev = self.sample_device(logits, sampled)[0]
        else:
            next_dev = torch.empty(len(sampled), dtype=torch.int64,
                                   device=self.device)
        if self.pp.size > 1:
            next_dev = self.pp.broadcast_tokens(next_dev)
        next_tokens = next_dev.tolist()
        for seq, tok in zip(sampled, next_tokens):
            seq.append_token(tok)
        return next_tokens

    @torch.inference_mode()
    def feed(self, chunks: List[Chunk],
             want: List[List[int]]) -> torch.Tensor:
        """Teacher-forced step: runs the given tokens as one batch, as
        generation would (single tokens alone are a decode step), and returns
        the logits at the wanted places of each chunk, in order."""
        if all(len(t) == 1 and start > 0 for _, start, t in chunks):
            self._dstate = None
            logits = self._decode_logits([seq for seq, _, _ in chunks])
            rows = [i for i, w in enumerate(want) for _ in w]
            if rows == list(range(len(chunks))):
                return logits.clone()   # the next step writes these again
            return logits[self._index(rows)]
        hidden, first_row = self.run_chunks(chunks)
        rows = [first_row[i] + p for i, w in enumerate(want) for p in w]
        return self.model.logits(hidden, self._index(rows))

    # ------------------------------------------------------------------

    def _build_decode_state(self, seqs: List[Sequence],
                            bucket: int = 0) -> dict:
        """Device-resident decode inputs.  Valid across steps for the same
        batch composition: positions/ctx advance on-device, the block tables
        never change mid-decode (pages are reserved for prompt+max_new at
        admission — engine/scheduler.py), so the only host->device traffic
        per step is nothing at all; sampled tokens stay on-device as the
        next step's input.  With a ``bucket`` they live in the inputs of its
        captured step."""
        n, rows = len(seqs), bucket or len(seqs)
        ps = self.cfg.page_size
        # one transfer: per sequence 2 int64 and 4 int32, then the tables.
        # Padding rows decode position 0 against page 0 with ctx=1: harmless
        # work; their slot writes land in reserved scratch page 0
        fields = np.zeros(4 * rows, dtype=np.int64)
        words = fields[2 * rows:].view(np.int32).reshape(4, rows)
        positions = np.array([seq.num_tokens - 1 for seq in seqs])
        fields[:n] = [seq.last_token for seq in seqs]
        if self.model.needs_prev:
            fields[rows:rows + n] = [seq.token_at(seq.num_tokens - 2)
                                     for seq in seqs]
        bt = table_array([seq.block_table for seq in seqs])
        words[0, :n] = positions
        words[1, :n] = (bt[np.arange(n), positions // ps] * ps +
                        positions % ps)
        words[2] = 1
        words[2, :n] = positions + 1
        if self.model.stateful:
            words[3, :n] = [seq.block_table.state_slot for seq in seqs]
        fields_dev, bt_dev = upload([fields, bt], self.device)
        if bucket:
            static = self._graphs[bucket][1]
            place_inputs(static["fields"], static["bt"], fields_dev, bt_dev)
        else:
            static = dict(self._fields(fields_dev), bt=bt_dev,
                          tickets=self.model.decode_tickets(rows))
        state = {k: static[k][:n] for k in ("tokens", "prev", "positions",
                                            "slots", "ctx", "state_slots")}
        state["bt"] = static["bt"][:n]
        state["tickets"] = static["tickets"]
        if not self.model.needs_prev:
            state["prev"] = None
        if not self.model.stateful:
            state["state_slots"] = None
        state.update(ids=tuple(s.seq_id for s in seqs), fresh=True,
                     bucket=bucket)
        return state

    @staticmethod
    def _fields(fields: torch.Tensor) -> Dict[str, torch.Tensor]:
        """The parts of a step's per-sequence inputs, 4 * rows int64."""
        rows = fields.numel() // 4
        words = fields[2 * rows:].view(torch.int32).view(4, rows)
        return {"tokens": fields[:rows], "prev": fields[rows:2 * rows],
                "positions": words[0], "slots": words[1], "ctx": words[2],
                "state_slots": words[3]}

    def _decode_slots(self, state: dict) -> torch.Tensor:
        ps = self.cfg.page_size
        pos = state["positions"].long()
        page = torch.gather(state["bt"], 1,
                            (pos // ps).unsqueeze(1)).squeeze(1)
        return (page * ps + (pos % ps).to(torch.int32)).to(torch.int32)

    def _decode_logits(self, seqs: List[Sequence]) -> Optional[torch.Tensor]:
        """Forward of one decode step; logits [n, vocab] on the last stage."""
        n = len(seqs)
        ids = tuple(s.seq_id for s in seqs)
        bucket = 0
        if (not self.cfg.enforce_eager and
                self.device.type == "cuda" and
                self.pp.size == 1 and           # p2p hops: eager path
                self.model.tp.graph_safe and    # xGMI AR or no TP
                n <= GRAPH_BATCH_SIZES[-1]):
            bucket = self._graph_bucket(n)
            if bucket not in self._graphs:
                self._build_graph(bucket)
        state = self._dstate
        if state is None or state["ids"] != ids or state["bucket"] != bucket:
            state = self._build_decode_state(seqs, bucket)
            self._dstate = state
        elif not state["fresh"]:
            state["positions"] += 1
            state["ctx"] += 1
            slots = self._decode_slots(state)
            if bucket:
                state["slots"].copy_(slots)
                static = self._graphs[bucket][1]
                # the first step's tokens, its prev now, are static's own
                for key in ("prev", "tokens"):
                    if state[key] is not None:
                        static[key][:n].copy_(state[key])
            else:
                state["slots"] = slots
        state["fresh"] = False
        if bucket:
            graph, _, logits = self._graphs[bucket]
            graph.replay()
            return logits[:n]
        slots = state["slots"]
        batch = self._decode_batch(state, slots, n)
        hidden_in = None
        if not self.pp.first:
            hidden_in = self.pp.recv_prev(
                (n, self.model.stream_width),
                self.model.stream_dtype, self.device)
        hidden = self.model.forward(state["tokens"], batch, self.cache,
                                    hidden=hidden_in)
        if self.pp.last:
            return self.model.logits(hidden)
        self.pp.send_next(hidden)
        return None

    def _decode_batch(self, inputs: dict, slots: torch.Tensor,
                      n: int) -> ForwardBatch:
        return ForwardBatch(
            mode="decode", positions=inputs["positions"], slot_mapping=slots,
            block_tables=inputs["bt"], context_lens=inputs["ctx"],
            starts=inputs["positions"], state_slots=inputs["state_slots"],
            prev_tokens=inputs["prev"], tickets=inputs["tickets"],
            decode_num_splits=self.model.decode_splits(
                n, self.cfg.max_seq_len, self.cfg.page_size))

    @torch.inference_mode()
    def decode(self, seqs: List[Sequence]) -> List[int]:
        n = len(seqs)
        logits = self._decode_logits(seqs)
        state = self._dstate
        if self.pp.last:
            next_dev, next_tokens = self.sample_device(logits, seqs)
        else:
            next_dev = torch.empty(n, dtype=torch.int64, device=self.device)
        if self.pp.size > 1:
            next_dev = self.pp.broadcast_tokens(next_dev)
            next_tokens = next_dev.tolist()
        if state["prev"] is not None:
            state["prev"] = state["tokens"]
        state["tokens"] = next_dev
        for seq, tok in zip(seqs, next_tokens):
            seq.append_token(tok)
        return next_tokens

    # ------------------------------------------------------------------

    def _graph_bucket(self, n: int) -> int:
        for b in GRAPH_BATCH_SIZES:
            if n <= b:
                return b
        return GRAPH_BATCH_SIZES[-1]

    def _build_graph(self, bs: int):
        """Capture one decode step at batch size ``bs`` into a hipGraph."""
        fields = torch.zeros(4 * bs, dtype=torch.int64, device=self.device)
        static = dict(self._fields(fields), fields=fields)
        static["ctx"].fill_(1)
        static["tickets"] = self.model.decode_tickets(bs)
        static["bt"] = torch.zeros(bs, self.max_pages_per_seq,
                                   dtype=torch.int32, device=self.device)
        batch = self._decode_batch(static, static["slots"], bs)
        # warm up allocations outside capture
        torch.cuda.synchronize()
        hidden = self.model.forward(static["tokens"], batch, self.cache)
        logits = self.model.logits(hidden)
        torch.cuda.synchronize()
        graph = torch.cuda.CUDAGraph()
        # Python must not collect another engine, dropped in a cycle of
        # references, just now: freeing its pool ends a capture, and its
        # captured steps end the process
        collects = gc.isenabled()
        gc.disable()
        try:
            with torch.cuda.graph(graph, pool=self._graph_pool):
                hidden = self.model.forward(static["tokens"], batch,
                                            self.cache)
                logits = self.model.logits(hidden)
        finally:
            if collects:
                gc.enable()
        if self._graph_pool is None:
            self._graph_pool = graph.pool()
        self._graphs[bs] = (graph, static, logits)
        log.info("captured decode hipGraph for batch %d", bs)
        return self._graphs[bs]

    # ------------------------------------------------------------------

    @torch.inference_mode()
    def sample(self, logits: torch.Tensor, seqs: List[Sequence]) -> List[int]:
        return self.sample_device(logits, seqs)[1]

    @torch.inference_mode()
    def sample_device(self, logits: torch.Tensor, seqs: List[Sequence]):
        """Returns (device int64 tensor, host list) of next tokens — the
        device tensor feeds the next decode step without a host round trip."""
        temps = [seq.sampling.temperature for seq in seqs]
        if all(t == 0.0 for t in temps):
            dev = logits.argmax(dim=-1)
        else:
            t = torch.tensor([max(tt, 1e-5) for tt in temps],
                             device=logits.device).unsqueeze(1)
            probs = torch.softmax(logits / t, dim=-1)
            dev = torch.multinomial(probs, 1).squeeze(1)
        return dev, dev.tolist()
