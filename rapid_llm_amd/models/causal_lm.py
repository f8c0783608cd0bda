"""The generic decoder: embedding, blocks in their run order, final norm, output projection.

Built from a :class:`~rapid_llm_amd.models.spec.ModelSpec` alone; nothing here names an
architecture.  The reference's skeleton is ``CausalLM`` (rapid_llm/models/base.py:378-631):
embed (:589-591), layers (:608-612), final norm (:619-621), row selection before the vocabulary
product (:625-630), output projection (:631).
"""

from __future__ import annotations

from dataclasses import replace

import torch

from ..kernels import decode_chain, ops
from ..kernels.notes import taking_notes
from ..parts.base import (
    BLOCKS,
    EMBEDDINGS,
    FEED_FORWARDS,
    MIXERS,
    NORMS,
    OUTPUT_PROJECTIONS,
    POSITION_ENCODINGS,
    CacheNeed,
    ParamSpec,
)
from ..parts.inject import StreamMix
from ..parts.lazy import DeferredProduct, plain, run_norm, settle
from ..parts.offsets import StreamOffsetTable
from .spec import ModelSpec


# Tokens up to which a step's layers behind the second are launched from what the second launched: beyond, the device has
# more to do than the host in any model.
REPEAT_MAX_TOKENS = 2048
# The noted layer keeps its temporary tensors until all layers are launched, where a layer alone gives each back
# behind its last use: bytes of them, as estimated, up to which that is done.  A quarter of what the engine leaves for a step's
# activations, so that no step comes to need more than there is; steps that are this large are not bound by the host.
REPEAT_MAX_BYTES = 1 << 28
# Tokens times a layer's matrix elements up to which a step keeps to this package's products, where it can do without the
# library's at all: a call of that costs the host 18 us, and a layer with one cannot be launched from native code, so
# up to there the device waits for the host.  Microseconds a prompt step, with library products / without: 0.6B (15.7 M) at 200 /
# 300 / 512 / 800 / 1,024 tokens 3,612 / 1,983, 3,609 / 2,239, 3,619 / 2,579, 3,998 / 2,948, 4,058 / 3,293 (at 1,500 level); 1.7B (50.3 M) at
# 100 / 200 / 300 / 450 tokens 3,564 / 2,526, 3,414 / 2,776, 3,601 / 3,244, 3,484 / 3,632.  Recorded steps gain by fewer starts: 0.6B with 256
# requests 5,272 / 5,127, 1.7B with 192 4,358 / 4,155.
OWN_PRODUCTS_MAX = 20_000_000_000


class CausalLM:
    def __init__(self, spec: ModelSpec) -> None:
        import rapid_llm_amd.parts  # noqa: F401  registers the built-in part kinds

        self.spec = spec
        self.embed = EMBEDDINGS.create(spec.embedding.kind, **spec.embedding.params, name="embed")
        self.output = OUTPUT_PROJECTIONS.create(spec.output.kind, **spec.output.params, name="output")
        self.final_norm = NORMS.create(spec.final_norm.kind, **spec.final_norm.params, name="final_norm")
        self.order = list(spec.order())
        for li in self.order:
            if not 0 <= li < len(spec.layers):
                raise ValueError(f"run order names layer {li}; the model has {len(spec.layers)}")
        self.offsets = None
        if spec.stream_offsets is not None:
            so = spec.stream_offsets
            for place in so.places:
                if not 0 <= place < len(self.order):
                    raise ValueError(f"a stream offset names place {place} of a run order of {len(self.order)}")
            self.offsets = StreamOffsetTable(so.checkpoint_name, so.places, spec.hidden_size, name="stream_offsets")
        self.mixes = None
        if spec.stream_mixes is not None:
            sm = spec.stream_mixes
            for place in sm.places:
                if not 0 <= place < len(self.order):
                    raise ValueError(f"a stream mix names place {place} of a run order of {len(self.order)}")
            self.mixes = StreamMix(sm.checkpoint_name, sm.places, spec.hidden_size, name="stream_mix")
        self.returns: frozenset[int] = frozenset()
        if spec.stream_returns is not None:
            self.returns = frozenset(spec.stream_returns.places)
            for place in self.returns:
                if not 0 <= place < len(self.order):
                    raise ValueError(f"the embedding returns at place {place} of a run order of {len(self.order)}")
        self._chain_space: decode_chain.Space | None = None  # of the recorded steps that run all layers in one launch
        self._chain_given_up = False  # (they keep their own kernels from there on)
        self._positions: dict[str, object] = {}
        self.blocks = []
        for i, layer in enumerate(spec.layers):
            pos_key = repr((layer.position.kind, sorted(layer.position.params.items())))
            position = self._positions.get(pos_key)
            if position is None:
                position = POSITION_ENCODINGS.create(layer.position.kind, **layer.position.params)
                self._positions[pos_key] = position
            mixer = MIXERS.create(
                layer.mixer.kind, **layer.mixer.params, position=position, name=f"layers.{i}.mixer"
            )
            alone = layer.shared_norm or layer.feed_forward is None
            if alone != (layer.feed_forward_norm is None):
                raise ValueError(f"layer {i}: a feed-forward and its norm come together or not at all")
            ff = n2 = None
            if layer.feed_forward is not None:
                ff = FEED_FORWARDS.create(
                    layer.feed_forward.kind, **layer.feed_forward.params, name=f"layers.{i}.ff"
                )
            if layer.feed_forward_norm is not None:
                n2 = NORMS.create(
                    layer.feed_forward_norm.kind, **layer.feed_forward_norm.params, name=f"layers.{i}.ff_norm"
                )
            n1 = NORMS.create(layer.mixer_norm.kind, **layer.mixer_norm.params, name=f"layers.{i}.mixer_norm")
            post = {}
            if layer.mixer_post_norm is not None:
                post["mixer_post_norm"] = NORMS.create(
                    layer.mixer_post_norm.kind, **layer.mixer_post_norm.params, name=f"layers.{i}.mixer_post_norm"
                )
            if layer.feed_forward_post_norm is not None:
                if ff is None:
                    raise ValueError(f"layer {i}: a norm behind a feed-forward that is not there")
                post["feed_forward_post_norm"] = NORMS.create(
                    layer.feed_forward_post_norm.kind, **layer.feed_forward_post_norm.params,
                    name=f"layers.{i}.ff_post_norm",
                )
            self.blocks.append(
                BLOCKS.create(
                    layer.block.kind,
                    **layer.block.params,
                    mixer=mixer,
                    feed_forward=ff,
                    mixer_norm=n1,
                    feed_forward_norm=n2,
                    **post,
                )
            )

        self._kinds = [self.blocks[li] for li in self.order]

    # ---- tensors ---------------------------------------------------------------
    def all_parts(self):
        yield self.embed
        for block in self.blocks:
            yield from block.parts()
        yield self.final_norm
        yield self.output
        if self.offsets is not None:
            yield self.offsets
        if self.mixes is not None:
            yield self.mixes
        yield from self._positions.values()

    def param_specs(self) -> list[ParamSpec]:
        specs: list[ParamSpec] = []
        for part in self.all_parts():
            specs.extend(part.param_specs())
        names = [s.name for s in specs]
        if len(names) != len(set(names)):
            raise ValueError("two parts declare a parameter of the same name")
        return specs

    def bind(self, params: dict[str, torch.Tensor], runtime) -> None:
        for part in self.all_parts():
            part.bind(params, runtime)
        # a block of every kind that runs, for what depends on the sizes of a layer's matrices alone
        kinds = {}
        for li in self.order:
            block = self.blocks[li]
            plain = block.launch_signature() is not None
            kinds.setdefault(tuple(t.shape for t in block.own_tensors() if t.dim() == 2) if plain else None, block)
        self._kinds = list(kinds.values())

    def replayable(self) -> bool:
        """Whether a step of this model may be recorded into a graph: every part and every
        block says so (``Part.replayable``)."""
        return all(getattr(p, "replayable", False) for p in (*self.all_parts(), *self.blocks))

    # ---- cache -----------------------------------------------------------------
    def cache_needs(self) -> list[CacheNeed]:
        """One need per place in the run order.  ``LayerSpec.share_cache_with`` names a layer;
        it resolves to that layer's latest earlier place in the order."""
        needs: list[CacheNeed] = []
        last_place: dict[int, int] = {}
        for place, li in enumerate(self.order):
            need = self.blocks[li].mixer.cache_need()
            share = self.spec.layers[li].share_cache_with
            if share is not None:
                if share not in last_place:
                    raise ValueError(
                        f"layer {li} reads the cache of layer {share}, which has not run before it"
                    )
                need = replace(need, share_with=last_place[share])
            needs.append(need)
            last_place[li] = place
        return needs

    # ---- step ------------------------------------------------------------------
    def _chain(self, ctx, caches) -> "decode_chain.DecodeChain | None":
        """The launch of all layers of a recorded step of few tokens, where they are plain dense layers of sizes that it
        takes; made by the eager run in front of the recording and kept with the graph."""
        if "decode_only_tokens" not in ctx.static or ctx.num_tokens > decode_chain.MAX_ROWS:
            return None
        if "decode_chain" not in ctx.static:
            ctx.static["decode_chain"] = self._new_chain(ctx, caches)
        return ctx.static["decode_chain"]

    def lost_launch(self) -> bool:
        """Whether a step's launch of all layers was given up, among those that have ended.  Asked behind the wait for a step."""
        return self._chain_space is not None and self._chain_space.given_up()

    def give_up_chain(self) -> None:
        """No launch of all layers any more.  Asked for when none is under way and no recorded step holds one."""
        self._chain_space, self._chain_given_up = None, True

    def chainable(self) -> bool:
        """Whether the layers are such that one launch may run them all (``decode_chain``), whatever a step's rows are."""
        if self._chain_given_up or self.offsets is not None or self.mixes is not None or self.returns or len(self.order) < 2:
            return False
        blocks = [self.blocks[li] for li in self.order]
        first = blocks[0].launch_signature()
        # (a signature says that a block and its parts are of known classes, the same ones in every layer)
        if first is None or any(b.launch_signature() != first for b in blocks):
            return False
        if not all(p.forward_as_written() for p in (blocks[0], *blocks[0].parts())):
            return False
        mixer, ff, norms = blocks[0].mixer, blocks[0].feed_forward, (blocks[0].mixer_norm, blocks[0].feed_forward_norm)
        if not hasattr(mixer, "qkv") or not hasattr(ff, "gate_up") or not all(hasattr(n, "eps") for n in norms):
            return False
        cos = mixer.position.cos if mixer.position is not None else None
        tensors = [t for b in blocks for t in (b.mixer.qkv.weight, b.mixer.o.weight, b.feed_forward.gate_up.weight, b.feed_forward.down.weight)]
        return (
            mixer.window <= 0 and not mixer.qkv_bias and not mixer.o_bias and not ff.has_bias and not ff.limit and ff.activation == "silu"
            and (mixer.q_norm_w is None) == (mixer.k_norm_w is None)
            and all(t.dtype == torch.bfloat16 and t.is_contiguous() and t.data_ptr() % 16 == 0 for t in tensors)
            and ops.attention_prepares_queries(torch.bfloat16, mixer.d, 0 if cos is None else cos.shape[1],
                                               getattr(mixer.position, "pairing", "half_split") if cos is not None else "half_split")
            and any(decode_chain.fits(rows, mixer.hidden_size, mixer.nq, mixer.nkv, mixer.d, ff.intermediate_size, 8)
                    for rows in range(1, decode_chain.MAX_ROWS + 1))
        )

    def chain_bytes(self, span: int) -> int:
        """Bytes that the recorded steps of few tokens share for their launches (contexts of at most ``span`` keys)."""
        if not self.chainable():
            return 0
        mixer, ff = self.blocks[self.order[0]].mixer, self.blocks[self.order[0]].feed_forward
        return sum(decode_chain.space_bytes(len(self.order), mixer.hidden_size, mixer.nq, mixer.nkv, ff.intermediate_size, span))

    def _new_chain(self, ctx, caches):
        kinds = {(c.group_id, c.page_size, c.owns_pages, len(c.pages), len(c.states)) for c in caches}
        if len(kinds) != 1 or not all(c.owns_pages and not c.states and c.k is not None and c.v is not None for c in caches) or not self.chainable():
            return None
        blocks = [self.blocks[li] for li in self.order]
        mixer, ff = blocks[0].mixer, blocks[0].feed_forward
        sizes = (mixer.hidden_size, mixer.nq, mixer.nkv)
        if not decode_chain.fits(ctx.num_tokens, *sizes, mixer.d, ff.intermediate_size, caches[0].page_size, ctx.static["context_bound"]):
            return None
        columns = ctx.block_tables[caches[0].group_id].stride(0)
        if not decode_chain.takes(len(blocks), ctx.num_tokens, *sizes, ff.intermediate_size, columns, caches[0].page_size, ctx.static["context_bound"]):
            return None
        layers = [
            (b.mixer.qkv.weight, b.mixer.o.weight, b.feed_forward.gate_up.weight, b.feed_forward.down.weight, b.mixer.q_norm_w,
             b.mixer.k_norm_w, b.feed_forward_norm.weight, behind.mixer_norm.weight if behind is not None else None, c.k, c.v)
            for b, behind, c in zip(blocks, [*blocks[1:], None], caches)
        ]
        if any(t is not None and t.data_ptr() % 16 for layer in layers for t in layer):
            return None
        if self._chain_space is None:  # (one step of a runner runs at a time)
            self._chain_space = decode_chain.Space(len(layers), *sizes, ff.intermediate_size, ctx.runtime.max_seq_len, mixer.qkv.weight.device)
        return decode_chain.DecodeChain(
            layers, self._chain_space, ctx.num_tokens, *sizes, ff.intermediate_size, ctx.static["context_bound"], mixer.scale,
            (mixer.qk_norm_eps or 0.0, blocks[0].mixer_norm.eps, blocks[0].feed_forward_norm.eps),
        )

    def _alike(self, ctx, caches) -> bool:
        """Whether every layer's launches of this step are the second one's with the layer's own tensors."""
        if ctx.num_tokens > REPEAT_MAX_TOKENS or len(self.order) < 4 or "decode_only_tokens" in ctx.static:
            return False
        if self.offsets is not None or self.mixes is not None or self.returns:
            return False
        blocks = [self.blocks[li] for li in self.order]
        first = blocks[0].launch_signature()
        # (a signature says that a block and its parts are of known classes, the same ones in every layer)
        if first is None or not all(p.forward_as_written() for p in (blocks[0], *blocks[0].parts())):
            return False
        if blocks[0].calls_library(ctx.num_tokens) or any(b.launch_signature() != first for b in blocks):
            return False
        if sum(ops.product_bytes(ctx.num_tokens, t) for t in blocks[0].own_tensors() if t.dim() == 2) > REPEAT_MAX_BYTES:
            return False
        kinds = {(c.group_id, c.page_size, c.owns_pages, len(c.pages), len(c.states)) for c in caches}
        return len(kinds) == 1 and all(c.owns_pages and not c.states for c in caches)

    def _second(self, residual, delta, ctx, caches):
        """The second layer of a step whose layers are alike, and those behind it where its launches say enough: what is
        left to add, and whether that is the last layer's.  What its notes kept is given back here."""
        with taking_notes() as notes:
            left = self.blocks[self.order[1]].forward(residual, delta, ctx, caches[1])
        last = self._repeat(notes, delta, left, caches) if notes.complete else None
        return (left, False) if last is None else (last, True)

    def _repeat(self, notes, delta, left, caches):
        """The layers behind the second, launched from the notes of the second's launches; ``delta`` is what the first
        left for it, ``left`` what it left itself.  Returns what the last layer leaves, ``None`` if nothing was launched."""
        lazy = isinstance(left, DeferredProduct)
        if type(left) is not type(delta) or not (lazy or isinstance(left, torch.Tensor)):
            return None
        before, after = (delta.x, left.x) if lazy else (delta, left)
        if before.shape != after.shape or before.dtype != after.dtype:
            return None
        tables = [self.blocks[li].own_tensors() + list(cache.pages.values()) for li, cache in zip(self.order, caches)]
        kinds = [[(t.shape, t.dtype, t.is_contiguous()) for t in row] for row in tables]
        if not all(k[2] for k in kinds[0]) or any(k != kinds[0] for k in kinds[1:]) or not ops.repeat_launches(notes, tables, (before, after)):
            return None
        return DeferredProduct(self.blocks[self.order[-1]].feed_forward.last_product, after) if lazy else after

    def _own_products(self, ctx) -> bool:
        """Whether the step keeps to this package's products (``OWN_PRODUCTS_MAX``): no layer needs the library's."""
        if ctx.num_tokens <= ops.SKINNY_MAX_ROWS:
            return False
        for block in self._kinds:
            if block.launch_signature() is None:
                return False
            if ctx.num_tokens * sum(t.numel() for t in block.own_tensors() if t.dim() == 2) > OWN_PRODUCTS_MAX:
                return False
        with ops.own_products():
            return not any(block.calls_library(ctx.num_tokens) for block in self._kinds)

    def forward(self, ctx, caches) -> torch.Tensor:
        """Run the tokens of ``ctx`` through every layer (which writes their keys and values)
        and return float32 logits ``[len(ctx.logit_rows), vocab]``."""
        with ops.shared_tiles():
            if self._own_products(ctx):
                with ops.own_products():
                    return self._forward(ctx, caches)
            return self._forward(ctx, caches)

    def _forward(self, ctx, caches) -> torch.Tensor:
        residual = self.embed.forward(ctx.token_ids, ctx)
        # the embedding's output, which later places take in again (the stream itself is updated
        # in place)
        first = residual.clone() if self.mixes is not None or self.returns else None
        delta = None
        chain = self._chain(ctx, caches)
        if chain is not None:
            first_block = self.blocks[self.order[0]]
            position = first_block.mixer.position
            x = run_norm(first_block.mixer_norm, residual, None, ctx)
            delta = chain.run(x, residual, ctx.positions, ctx.token_slot, ctx.block_tables[caches[0].group_id],
                              position.cos if position is not None else None, position.sin if position is not None else None, ctx.max_position)
        for place, li in enumerate(self.order if chain is None else ()):
            if place == 1 and self._alike(ctx, caches):  # (asked while the device has the first layer to do)
                delta, whole = self._second(residual, delta, ctx, caches)
                if whole:
                    break
                continue
            block = self.blocks[li]
            if self.mixes is not None and self.mixes.at(place):
                delta = settle(residual, delta)
                if delta is not None:
                    residual.add_(delta)
                    delta = None
                residual = self.mixes.forward(residual, first)
            row = self.offsets.at(place) if self.offsets is not None else None
            again = first if place in self.returns else None
            if row is not None or again is not None:
                ops.stream_add(residual, again, row)
            if not getattr(block, "accepts_deferred", False):
                delta = settle(residual, delta)
            delta = block.forward(residual, delta, ctx, caches[place])
        if ctx.num_logit_rows == 0:
            return torch.empty((0, self.spec.vocab_size), dtype=torch.float32, device=residual.device)
        h = run_norm(self.final_norm, residual, delta, ctx, rows=ctx.logit_rows)
        return self.output.forward(h, ctx)


def model_param_specs(spec: ModelSpec) -> list[ParamSpec]:
    return CausalLM(spec).param_specs()
