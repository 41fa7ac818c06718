"""Soft-max attention through latents (``config.spec.LatentAttentionSpec``): per token the cache holds one normed latent
c [kv_rank] and one rotated key part r [rot_dim] that all heads share, instead of keys and values per head.

With h the input, per head i (D unrotated, R rotated, E value channels, C = kv_rank):
    c_q = norm(W_dq h);  q_i = (W_uq c_q)_i = [q_i^plain (D) | q_i^rot (R)];  [c' | r'] = W_dkv h;  c = norm(c');  r = rotate(r')
    score_i(t, j) = (q_i^plain(t) . Uk_i c(j) + rotate(q_i^rot(t)) . r(j)) * scale,   Uk_i = rows i of W_uk  [D, C]
    out_i(t) = sigmoid(W_g h)_i * Uv_i sum_j p_i(t, j) c(j),                          Uv_i = rows i of W_uv  [E, C]
                                                     (one gate per head, or per channel of all heads, or none)
Because q . (Uk c) = (Uk^T q) . c and Uv sum p c is linear, the attention itself runs over ONE key/value head whose key is
[c | r] and whose value is c, with queries [Uk_i^T q_i^plain | rotate(q_i^rot)]: the paged cache, its manager and the
attention kernels serve it as they serve any layer with one key/value head, key size C + R and value size C.  What is
particular to the layer are three kernels around that (``csrc/latent.hip``) and three products:
    [W_dq; W_dkv; W_g] h  ->  latent_prep (norms, rotation of r, cache write, sigmoid)  ->  W_uq c_q  ->  latent_q_absorb
    ->  attention  ->  latent_out (through Uv_i, times the gate)  ->  W_o.
(Without a query latent W_q stands in W_dq's place and gives the queries.)
Norms, angles, rotations, the gate and the scores are 32-bit whatever the model's precision.
"""

from __future__ import annotations

import torch

from ..kernels import ops
from . import registry
from .attention import TILES, TilePlan, wide_attention
from .linear import LinearWeight
from .needs import PagedNeed


# Prompt portions run over keys and values made from the latents (``csrc/latent_prompt.hip``) where they bring this many tokens
# together, and this many each on average: making a key costs what about seventy tokens save on it (a latent of 512, heads of
# 64 + 32 and 64 channels; twice as many tokens in a portion that starts a prompt, whose keys half of its tokens see).
EXPAND_TOKENS, EXPAND_TOKENS_EACH = 128, 64
EXPAND_KEYS_PER_TOKEN = 16  # keys, at most, that a portion's tokens may find for each of them
EXPAND_SCRATCH = 1 << 30  # bytes of scratch for them, at most
# How far the wide form is behind goes by its products a (query, key) pair and head over this one's, (2 C + R) / (D + R + E): 6.6 at those
# sizes, 3.4 at heads of 128 + 64 and 128, 1.8 at 64 + 32 and 64 over a latent of 128.  Below EXPAND_CLEAR, tiles too few for the GPU (one
# workgroup each walks all keys, where the wide form cuts them) and many keys are slower: 512 tokens at 7,000 keys, 8 heads over 128: 120 us,
# wide 111; 128 tokens at 1,900: 41 and 38; at 512 keys 21 and 33.
EXPAND_CLEAR, EXPAND_FULL, EXPAND_KEYS_FEW = 3.0, 256, 5
# Beside single tokens an eager step forms the wide form's queries and outputs for every row all the same, and only the attention itself
# counts: 4 portions of 64 tokens, 16 heads of 128 + 64 over 512: 29 us, wide 21; 128 tokens, 8 heads over 128: 13.3 and 12.7, 300 tokens 16.5 and 20.
EXPAND_BESIDE = 400  # tokens each, times the factor


class LatentAttention:
    graph_safe = True
    takes_layouts = True

    def __init__(self, spec, prefix: str) -> None:
        self.spec, self.prefix = spec, prefix
        self.position = registry.build("position", spec.position, prefix)
        if self.position.rotary_dim != spec.rot_dim:
            raise ValueError("the rotated part of a latent-attention head is rot_dim channels")
        if spec.rot_dim % 2:
            raise ValueError(f"rot_dim={spec.rot_dim} must be even")
        self.first: LinearWeight | None = None
        self.sink_logits: torch.Tensor | None = None
        if not spec.q_rank and spec.gate:
            raise ValueError("a latent-attention layer without a query latent has no gate per head")
        if spec.out_gate and (spec.gate or spec.q_rank):
            raise ValueError("a gate per channel stands alone, in a latent-attention layer without a query latent")

    @property
    def _n(self) -> dict:
        keys = ("dq", "dq_norm", "uq", "dkv", "dkv_norm", "uk", "uv", "g", "o")
        return {k: self.prefix + name for k, name in zip(keys, self.spec.names)}

    def wanted(self) -> dict:
        s, n = self.spec, self._n
        out = {
            n["uq"]: ((s.heads * (s.head_dim + s.rot_dim), s.q_rank or s.hidden), "linear"),
            n["dkv"]: ((s.kv_rank + s.rot_dim, s.hidden), "linear"), n["dkv_norm"]: ((s.kv_rank,), "norm"),
            n["uk"]: ((s.heads * s.head_dim, s.kv_rank), "linear"), n["uv"]: ((s.heads * s.value_dim, s.kv_rank), "linear"),
            n["o"]: ((s.hidden, s.heads * s.value_dim), "linear"),
        }
        if s.q_rank:
            out.update({n["dq"]: ((s.q_rank, s.hidden), "linear"), n["dq_norm"]: ((s.q_rank,), "norm")})
        if s.gate:
            out[n["g"]] = ((s.heads, s.hidden), "linear")
        if s.out_gate:
            out[n["g"]] = ((s.heads * s.value_dim, s.hidden), "linear")
        if s.sink_name:
            out[self.prefix + s.sink_name] = ((s.heads,), "around_zero")
        return out

    def load(self, get, dtype, device, layouts: str = "both") -> None:
        s, n = self.spec, self._n
        plain = layouts == "both"
        to = lambda name: get(name).to(device=device, dtype=dtype).contiguous()
        # one product for everything that reads the layer's input: [W_dq; W_dkv; W_g]
        # (without a query latent the queries' matrix takes the place of W_dq in it, and there is no second product)
        self.q_cols = s.q_rank or s.heads * (s.head_dim + s.rot_dim)
        rows = [to(n["dq"] if s.q_rank else n["uq"]), to(n["dkv"])] + ([to(n["g"])] if s.gate or s.out_gate else [])
        if s.out_gate:
            # (the gate's columns start, and a row ends, at a multiple of 8: the kernels read both queries and gate as columns of it)
            fill = lambda have: [torch.zeros((-have % 8, s.hidden), dtype=dtype, device=device)]
            before = rows[0].shape[0] + rows[1].shape[0]
            rows[2:2] = fill(before)
            self.gate_at = before + -before % 8
            rows += fill(rows[3].shape[0])
        self.first = LinearWeight(torch.cat(rows).contiguous(), keep_plain=plain)
        self.dq_norm, self.dkv_norm = (to(n["dq_norm"]) if s.q_rank else None), to(n["dkv_norm"])
        self.uq = LinearWeight(to(n["uq"]), keep_plain=plain) if s.q_rank else None
        if s.sink_name:
            self.sink_logits = get(self.prefix + s.sink_name).to(device=device, dtype=torch.float32).contiguous()
        # the two per-head matrices, each in the layout its kernel walks: on the matrix cores (bfloat16, sizes that fit) every
        # head's matrix as [out, in] rows; otherwise as the plain kernels of ``csrc/latent.hip`` read them
        D, R, E, C = s.head_dim, s.rot_dim, s.value_dim, s.kv_rank
        # (without a query latent the queries are columns of the first product's rows, which must then start 16 bytes apart)
        self._mfma_q = (ops.headwise_takes(dtype, C, D, D + R, C + R) and s.hidden % 8 == 0 and s.q_rank % 8 == 0
                        and (s.q_rank > 0 or self.first.n % 8 == 0))
        self._mfma_o = ops.headwise_takes(dtype, E, C, C, E)
        uk, uv = to(n["uk"]), to(n["uv"])
        # prompt portions read both as the checkpoint has them
        self._block = ops.latent_prompt_block(dtype, s.heads, D, R, E, C) if self._mfma_q and self._mfma_o else 0
        self.uk_rows = uk if self._block else None
        self.uk = uk.view(s.heads, D, C).transpose(1, 2).contiguous() if self._mfma_q else uk  # [heads, latent, dim] | [heads * dim, latent]
        self.uv = uv.view(s.heads, E, C) if self._mfma_o else uv.view(s.heads, E, C).transpose(1, 2).contiguous()  # [heads, value, latent] | [heads, latent, value]
        self.wo = LinearWeight(to(n["o"]), keep_plain=plain)
        self.position.load(get, dtype, device)
        self._factor = float(getattr(self.position, "factor", 1.0))
        self._interleaved = bool(getattr(self.position, "interleaved", False))

    def cache_need(self):
        s = self.spec
        return PagedNeed(1, s.kv_rank + s.rot_dim, s.window, s.kv_rank)

    def batch_plans(self) -> list:
        return [TILES]

    def max_positions(self) -> int | None:
        return self.position.max_positions

    def forward(self, ctx, x, cache, owns_cache: bool = True, out: torch.Tensor | None = None):
        s, pos = self.spec, self.position
        n = x.shape[0]
        if not owns_cache:
            raise ValueError("a latent-attention layer writes its own cache")
        if pos.max_positions is not None and ctx.max_position >= pos.max_positions:
            raise ValueError(f"position {ctx.max_position} is beyond the model's {pos.max_positions} positions")
        H, D, R, E, C = s.heads, s.head_dim, s.rot_dim, s.value_dim, s.kv_rank
        take = ctx.arena.take
        table = ctx.block_tables[cache.group]
        proj = self.first(x, out=take((n, self.first.n), x.dtype), arena=ctx.arena, plain_copy=not ctx.captured)
        gate = take((n, H), torch.float32) if s.gate else None
        if s.q_rank:
            cq = take((n, s.q_rank), x.dtype)
            ops.latent_prep(proj, self.dq_norm, self.dkv_norm, pos.inv_freq, self._factor, ctx.positions, ctx.token_req, table, cache.k, cache.v,
                            s.q_rank, C, R, H if s.gate else 0, s.norm_eps, cq, gate, interleaved=self._interleaved)
            q = self.uq(cq, out=take((n, H * (D + R)), x.dtype), arena=ctx.arena, plain_copy=not ctx.captured)
        else:
            # the queries are the first columns of the product; the rest of a row is [latent | rotated part]
            ops.latent_prep(proj[:, self.q_cols :], None, self.dkv_norm, pos.inv_freq, self._factor, ctx.positions, ctx.token_req, table, cache.k,
                            cache.v, 0, C, R, 0, s.norm_eps, None, None, interleaved=self._interleaved)
            q = proj[:, : self.q_cols]
        att = take((n, H * E), x.dtype)
        channel_gate = proj[:, self.gate_at : self.gate_at + H * E] if s.out_gate else None
        count, blocks = self._expands(ctx, n, cache)
        singles = TilePlan.views(ctx)[1].shape[0]
        if not count:
            self._rows(ctx, q, cache, table, gate, channel_gate, att, True)
        elif singles:
            # (the single tokens of a captured step are its first rows; elsewhere they may stand anywhere, and what is formed for the
            # portions' rows on the way is written over)
            m = singles if ctx.captured else n
            first = lambda t: t[:m] if t is not None else None
            self._rows(ctx, q[:m], cache, table, first(gate), first(channel_gate), att[:m], False)
        if count:
            scratch = take((count * blocks * self._block,), x.dtype)
            ops.latent_prompt(q, cache.k, self.uk_rows, self.uv, scratch, TilePlan.views(ctx)[0], table, pos.inv_freq, self._factor, H, D, R, E, C, count,
                              blocks, s.softmax_scale, att, window=s.window, interleaved=self._interleaved, gate=gate, channel_gate=channel_gate,
                              sink_logits=self.sink_logits)
        return self.wo(att, out=out if out is not None else take((n, s.hidden), x.dtype), arena=ctx.arena, plain_copy=not ctx.captured)

    def _expands(self, ctx, n: int, cache) -> tuple[int, int]:
        """Whether the step's prompt portions run over keys and values made from the latents: (portions, blocks of 64 keys of the longest, an
        even number), or (0, 0)."""
        s = self.spec
        chunk_tiles, decode_tiles = TilePlan.views(ctx)
        singles, page, keys = decode_tiles.shape[0], cache.k.shape[2], ctx.max_chunk_kv
        count = min(ctx.n_reqs - singles, chunk_tiles.shape[0])  # (a captured step counts the request that owns its padding too)
        tokens, blocks = n - singles, -(-keys // 128) * 2
        if not self._block or not count or page & (page - 1) or tokens < EXPAND_TOKENS or 2 * count * blocks * self._block > EXPAND_SCRATCH:
            return 0, 0
        each = tokens if ctx.captured else tokens / count
        factor = (2 * s.kv_rank + s.rot_dim) / (s.head_dim + s.rot_dim + s.value_dim)
        few = factor < EXPAND_CLEAR and -(-tokens // 64) * s.heads < EXPAND_FULL
        if each < EXPAND_TOKENS_EACH or keys > (EXPAND_KEYS_FEW if few else EXPAND_KEYS_PER_TOKEN) * tokens:
            return 0, 0
        if singles and (each * factor < EXPAND_BESIDE or (s.window and factor < 1.5)):
            return 0, 0
        return count, blocks

    def _rows(self, ctx, q, cache, table, gate, channel_gate, att, portions: bool) -> None:
        """Single tokens (and ``portions`` too) over the latents themselves: absorbed queries, one wide key/value head."""
        s, take = self.spec, ctx.arena.take
        n = q.shape[0]
        H, D, R, E, C = s.heads, s.head_dim, s.rot_dim, s.value_dim, s.kv_rank
        positions, token_req, inv_freq = ctx.positions[:n], ctx.token_req[:n], self.position.inv_freq
        q_lat, o_lat = take((n, H * (C + R)), q.dtype), take((n, H * C), q.dtype)
        if self._mfma_q:
            ops.headwise_product(q, D + R, self.uk, q_lat, C + R)
        ops.latent_q_absorb(q, None if self._mfma_q else self.uk, inv_freq, self._factor, positions, H, D, R, C, out=q_lat, interleaved=self._interleaved)
        if ops.wide_attention_takes(q.dtype, C + R, C, cache.k.shape[2]):
            wide_attention(ctx, q_lat, o_lat, cache, table, H, 1, C + R, C, s.softmax_scale, window=s.window, sink_logits=self.sink_logits, portions=portions)
        else:
            ops.attention_generic(q_lat, o_lat, cache.k, cache.v, token_req, positions, table, H, 1, C + R, s.softmax_scale, window=s.window, v_dim=C,
                                  sink_logits=self.sink_logits)
        if self._mfma_o:
            ops.headwise_product(o_lat, C, self.uv, att, E, gate=gate, channel_gate=channel_gate)
        else:
            ops.latent_out(o_lat, self.uv, gate, H, C, E, out=att, channel_gate=channel_gate)


registry.register("mixer", "latent_attention", LatentAttention)
