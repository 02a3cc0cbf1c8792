"""A model as data: token table, blocks built from a `ModelSpec`, the order they
run in, final norm and output matrix.  It knows no architecture; the typed
configuration's `model_spec()` does (config/llama.py).  Reference counterpart:
LlamaModel / run_layers (src/arch/llama.rs:24-43, :146-172)."""
from __future__ import annotations

from typing import Dict, List, Mapping, Optional, Tuple

import torch

from ..cache.spec import FixedState
from ..config.spec import ModelSpec
from ..kernels import EPI_STORE_F32, kernels
from ..parts import TensorSpec, build_block, build_norm, place
from ..weights import check_tensors


class Model:
    def __init__(self, spec: ModelSpec, dtype: torch.dtype, device):
        spec.validate()
        if dtype not in (torch.float32, torch.bfloat16):
            raise ValueError(f"the engine computes in float32 or bfloat16, not {dtype}")
        self.spec, self.dtype, self.device = spec, dtype, torch.device(device)
        self.blocks = [build_block(layer, dtype) for layer in spec.layers]
        self.streams = int(spec.streams)
        # (one copy handled by arrangements that take copies is still laid out as [1, T, hidden])
        self.streamed = self.streams > 1 or any(block.takes_streams for block in self.blocks)
        if self.streamed:
            for i, block in enumerate(self.blocks):
                if not block.takes_streams:
                    raise ValueError(f"layer {i}: the arrangement {type(block).__name__} does not work on a stream kept in several copies")
        self.final_norm = build_norm(spec.final_norm, dtype) if spec.final_norm is not None else None
        self.embedding: Optional[torch.Tensor] = None
        self.head: Optional[torch.Tensor] = None
        self.wave_rates: Optional[torch.Tensor] = None
        self.pairs: Optional[torch.Tensor] = None
        self.joins: Dict[str, torch.Tensor] = {run.join_embedding: None for run in spec.schedule if run.join_embedding is not None}
        keyed = {}
        for block in self.blocks:
            for part in block.parts():
                if part.recording_signature is not None:
                    keyed.setdefault(part.recording_signature, part)
        self._keyed_parts = list(keyed.values())

    # -- weights -------------------------------------------------------------
    def tensors(self) -> Dict[str, TensorSpec]:
        s = self.spec
        out = {s.embedding_name: TensorSpec((s.vocab_size, s.hidden_size))}
        if s.head_name is not None:
            out[s.head_name] = TensorSpec((s.vocab_size, s.hidden_size))
        if s.pair_table is not None:
            out[s.pair_table.name] = TensorSpec((s.pair_table.buckets + 1, s.hidden_size))
        out.update({name: TensorSpec((s.hidden_size, 2 * s.hidden_size)) for name in self.joins})
        for block in self.blocks:
            for part in block.parts():
                out.update(part.tensors())
        if self.final_norm is not None:
            out.update(self.final_norm.tensors())
        return out

    def load(self, tensors: Mapping[str, torch.Tensor]) -> None:
        """Takes every tensor `tensors()` names; anything missing, left over or
        of another shape is reported in one error."""
        want = {n: t.shape for n, t in self.tensors().items()}
        # (a mapping that makes or reads its tensors only when asked says their shapes without doing so)
        have = tensors.shapes() if hasattr(tensors, "shapes") else {n: tuple(t.shape) for n, t in tensors.items()}
        check_tensors(have, want, ignorable=self.spec.ignorable_tensors)
        s = self.spec
        self.embedding = place(tensors[s.embedding_name], self.device, self.dtype)
        # tied: the output matrix is the token table (src/arch/llama.rs:81)
        self.head = self.embedding if s.head_name is None else place(tensors[s.head_name], self.device, self.dtype)
        if s.pair_table is not None:
            self.pairs = place(tensors[s.pair_table.name], self.device, self.dtype)
        for name in self.joins:
            self.joins[name] = place(tensors[name], self.device, self.dtype)
        if s.position_wave_base > 0:
            i = torch.arange((s.hidden_size + 1) // 2, dtype=torch.float64)
            rates = torch.pow(torch.tensor(s.position_wave_base, dtype=torch.float64), -2.0 * i / s.hidden_size)
            self.wave_rates = torch.stack([rates.float(), (rates - rates.float().double()).float()]).to(self.device)      # (as two 32-bit numbers each)
        for block in self.blocks:
            for part in block.parts():
                part.load(tensors, self.device)
        if self.final_norm is not None:
            self.final_norm.load(tensors, self.device)

    def weights(self) -> Dict[str, torch.Tensor]:
        """Every tensor of the model on the host, under its file name and in the file's layout
        (what parts fused or reordered at load is undone), in the dtype the engine keeps it in:
        what `load` would take again, and what another implementation can be given to compare."""
        s = self.spec
        out = {s.embedding_name: self.embedding.cpu()}
        if s.head_name is not None:
            out[s.head_name] = self.head.cpu()
        if s.pair_table is not None:
            out[s.pair_table.name] = self.pairs.cpu()
        out.update({name: w.cpu() for name, w in self.joins.items()})
        for block in self.blocks:
            for part in block.parts():
                out.update(part.export())
        if self.final_norm is not None:
            out.update(self.final_norm.export())
        return out

    def weight_bytes_per_step(self) -> int:
        """Bytes of weights one step reads when it uses each once (the table's rows aside):
        every tensor a part of the schedule's layers holds, the final norm's, and the output matrix."""
        seen = set()
        total = sum(part.step_weight_bytes(seen) for run in self.spec.schedule for part in self.blocks[run.layer].parts())
        total += sum(w.numel() * w.element_size() for w in self.joins.values())
        if self.final_norm is not None:
            total += self.final_norm.step_weight_bytes(seen)
        if self.head.data_ptr() not in seen:
            total += self.head.numel() * self.head.element_size()
        return total

    def graph_safe(self) -> bool:
        """Whether a step of this model may be recorded into a HIP graph (every part says so)."""
        return (all(part.graph_safe for block in self.blocks for part in block.parts())
                and (self.final_norm is None or self.final_norm.graph_safe))

    def recording_key(self, ctx) -> tuple:
        """What a recording of this step depends on beyond its sizes (its parts say)."""
        return tuple(part.recording_key(ctx) for part in self._keyed_parts)

    # -- cache ---------------------------------------------------------------
    def cache_needs(self) -> List[Tuple[object, Optional[int]]]:
        """What each run of the schedule asks for; behind them, for a model whose embedding looks at the token before, a place
        for a request's last token."""
        needs = [(self.blocks[run.layer].cache_need(), run.cache_of) for run in self.spec.schedule]
        if self.spec.pair_table is not None:
            needs.append((FixedState((1,), torch.int32), None))
        return needs

    # -- one step --------------------------------------------------------------
    def _join_rows(self, ctx):
        """(the stream's rows, the embedding's rows, both side by side) in the activation type: what a join's product reads."""
        D = self.spec.hidden_size
        both = ctx.workspace("model.join", (ctx.n_tokens, 2 * D), self.dtype)
        return both[:, :D], both[:, D:], both

    def forward(self, ctx, cache_views) -> Optional[torch.Tensor]:
        """Runs the step's T tokens through the schedule; returns float32 logits
        [n_want, vocab] at the wanted rows, or None when none is wanted."""
        k = kernels()
        T = ctx.n_tokens
        ctx.drop_streams_mix()          # (a step that ended in an error may have left one)
        if self.streamed:
            # [streams, T, hidden]: every copy starts as the embedding; blocks read and write all of them
            h = ctx.workspace("model.h", (self.streams, T, self.spec.hidden_size), torch.float32)
            k.embed_streams(h, self.embedding, ctx.tokens, self.spec.embedding_scale)
        elif self.pairs is not None:
            h = ctx.workspace("model.h", (T, self.spec.hidden_size), torch.float32)
            table = self.spec.pair_table
            k.embed_pairs(h, self.embedding, self.pairs, ctx.tokens, self.spec.embedding_scale, table.mul_prev, table.mul_cur, ctx.positions,
                          ctx.token_entry, ctx.q_starts, ctx.slots, cache_views[len(self.spec.schedule)].state,
                          copy=self._join_rows(ctx)[1] if self.joins else None)
        else:
            h = ctx.workspace("model.h", (T, self.spec.hidden_size), torch.float32)
            k.embed_rows(h, self.embedding, ctx.tokens, self.spec.embedding_scale,
                         **({} if self.wave_rates is None else {"waves": (ctx.positions, self.wave_rates)}))
            if self.joins:
                k.cast_rows(self._join_rows(ctx)[1], h)
        ctx.note_left(h, None)
        joinable = False                    # whether the rows for the next join lie ready
        for i, run in enumerate(self.spec.schedule):
            ctx.run_index = i
            block = self.blocks[run.layer]
            # the norm that reads the stream after this block: the next block's first; after the last block the
            # final norm, where it reads every row (else it reads gathered rows and runs as a kernel of its own)
            later = self.spec.schedule[i + 1] if i + 1 < len(self.spec.schedule) else None
            # (a run that takes the embeddings first changes the stream before its norm reads it: nothing to prepare)
            ctx.norm_after_block = (None if later is not None and (later.add_embedding or later.join_embedding is not None)
                                    else self.blocks[later.layer].first_norm() if later is not None
                                    else self.final_norm if ctx.wants_every_row else None)      # (None too without a final norm)
            if run.add_embedding:          # the tokens' embeddings once more, as they entered the stream at the start
                k.embed_rows(h, self.embedding, ctx.tokens, self.spec.embedding_scale, add=True)
                ctx.note_left(h, None)
            if run.join_embedding is not None:      # the stream and the embedding side by side, through one matrix
                rows, w = self._join_rows(ctx), self.joins[run.join_embedding]
                if not joinable:
                    k.cast_rows(rows[0], h)
                k.gemm(rows[2], w, h, EPI_STORE_F32, ctx.gemm_workspace(rows[2], w))
                ctx.note_left(h, None)
            before_join = later is not None and later.join_embedding is not None
            ctx.rows_after_block = self._join_rows(ctx)[0] if before_join else None
            block.forward(ctx, h, cache_views[i])
            joinable = before_join and ctx.rows_after_block is None
            ctx.rows_after_block = None
            if not block.keeps_left_current:
                ctx.note_left(h, None)
            if ctx.after_run is not None:
                ctx.flush_streams()
                ctx.after_run(i, h)
        ctx.norm_after_block = ctx.upcoming_norm = None
        if ctx.n_want == 0:
            ctx.flush_streams()
            return None
        # Norm only the wanted rows, then the output matrix: the reference norms all
        # rows and gathers after (src/arch/llama.rs:135-139), which is the same numbers.
        # (A step of few single tokens that wants them all: the last product has prepared the final norm, and the
        # output matrix's product finishes it; no norm kernel runs.)
        x = self.final_norm.deferred(ctx, h) if ctx.wants_every_row and self.final_norm is not None and not self.streamed else None
        if x is not None and not isinstance(x, torch.Tensor) and not k.product_norms_its_rows(T, self.head.shape[0], self.head.shape[1], self.dtype):
            x = None            # (rows that the output matrix's product cannot scale: the norm runs)
        if x is None:
            x = ctx.workspace("model.head_in", (ctx.n_want, self.spec.hidden_size), self.dtype)
            if self.streamed:
                # the stream is the sum of its copies: a norm that can reads them all at the wanted rows itself
                if self.final_norm is None or not self.final_norm.forward_streams(ctx, h, None, x, None if ctx.wants_every_row else ctx.want_rows):
                    raise ValueError("a stream kept in several copies needs a final norm that reads them (forward_streams)")
            elif self.final_norm is not None:
                self.final_norm.forward(ctx, h, x, ctx.want_rows)
            else:       # no norm before the output matrix: the wanted rows of the stream, in the activation type
                rows = x if self.dtype == torch.float32 else ctx.workspace("model.head_rows", x.shape, torch.float32)
                k.embed_rows(rows, h, ctx.want_rows, 1.0)
                if rows is not x:
                    k.cast(x, rows)
        logits = ctx.workspace("model.logits", (ctx.n_want, self.spec.vocab_size), torch.float32)
        k.gemm(x, self.head, logits, EPI_STORE_F32, ctx.gemm_workspace(x, self.head))
        if self.spec.logit_scale != 1.0 or self.spec.logit_softcap > 0.0:
            k.scale_softcap_rows(logits, self.spec.logit_scale, self.spec.logit_softcap)
        return logits
