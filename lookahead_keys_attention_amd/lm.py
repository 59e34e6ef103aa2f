"""A small decoder-only language model around `Castle`, and its sampler.

Counterpart of the reference's training-script model (train_triton.py:73-175 `CastleLM`,
train_triton.py:56-71 sampling helpers): `depth` x [Castle attention, feed-forward], both
residual, a final RMSNorm and a logits projection.  `forward(x, return_loss, cache,
return_next_cache)` and `sample(prompt, seq_len, temperature, filter_thres)` keep the reference's
argument meaning.  With `use_triton=True` the attention layers run the HIP kernels: a prompt is
pre-filled by the parallel forward kernels, every further token by the in-place cached decode
step, one `Cache` per layer.

Differences a user can switch: `tie_embedding=True` shares the token embedding with the logits
projection (the reference keeps them separate, train_triton.py:86,111); `rotary_emb` / `prenorm`
default to the reference's choice (both on, train_triton.py:99-100).
"""
from __future__ import annotations

import contextlib
import gc
import math

import torch
import torch.nn.functional as F
from torch import nn

from . import _native, ops
from .castle import Castle, _linear, _unmodified


READ_ONCE_BYTES = 320_000_000
# The sampling kernel gives a row of logits to one workgroup, the operators below spread it over the GPU: up to this
# vocabulary the kernel is ahead at any number of rows (us per token with the random numbers, kernel / operators, 1 row and
# 64, logits of one leading digit last: 256 11 / 72 and 12 / 72; 8192 35 / 95 and 39 / 131; 20480 80 / 101 and 82 / 145,
# 88 / 102; 28672 107 / 103 and 110 / 168, 122 / 102; 131072 462 / 108 and 533 / 777).
SAMPLER_MAX_VOCABULARY = 20480


# -- sampling helpers (train_triton.py:56-71) ------------------------------------------------
def safe_log(t: torch.Tensor, eps: float = 1e-20) -> torch.Tensor:
    return t.clamp(min=eps).log()


def gumbel_noise(t: torch.Tensor, generator: torch.Generator | None = None) -> torch.Tensor:
    u = torch.rand(t.shape, dtype=t.dtype, device=t.device, generator=generator)
    return -safe_log(-safe_log(u))


def gumbel_sample(logits, temperature=1.0, dim=-1, keepdim=True, generator=None):
    """argmax(logits / temperature + Gumbel noise): a draw from softmax(logits / temperature)."""
    return (logits / max(temperature, 1e-10) + gumbel_noise(logits, generator)).argmax(dim=dim, keepdim=keepdim)


def top_k(logits: torch.Tensor, thres: float = 0.9) -> torch.Tensor:
    """Keeps the ceil((1 - thres) * vocabulary) largest logits of each row, -inf elsewhere."""
    k = math.ceil((1.0 - thres) * logits.shape[-1])
    values, index = logits.topk(k, dim=-1)
    return torch.full_like(logits, float("-inf")).scatter_(-1, index, values)


def pick_token(logits, temperature, filter_thres, generator=None):
    """(batch, n, vocabulary) logits -> (batch, 1) tokens from the last position; temperature = 0 picks the arg-max."""
    logits = top_k(logits[:, -1].float(), thres=filter_thres)
    if temperature == 0:
        return logits.argmax(dim=-1, keepdim=True)
    return gumbel_sample(logits, temperature=temperature, generator=generator)


def _runs_castle_forward(attention) -> bool:
    """True for a `Castle`, or a subclass of it, whose call does what `Castle.forward` does and nothing else."""
    return _unmodified(attention, type(attention)) and type(attention).forward is Castle.forward


def _block_parts(feed_forward):
    """(norm, linear, GELU, linear) of a block that may be taken apart: these four, the erf GELU, and nothing that wants to see a
    call of the block or of the GELU; None otherwise."""
    if not _unmodified(feed_forward, nn.Sequential):
        return None
    parts = tuple(feed_forward._modules.values())
    return parts if len(parts) == 4 and _unmodified(parts[2], nn.GELU) and parts[2].approximate == "none" else None


def token_feed_forward(feed_forward: nn.Sequential, h: torch.Tensor) -> torch.Tensor:
    """h + feed_forward(h) for a single-token step (inference), the block being [norm, linear,
    GELU, linear]: two launches of the small-M linear kernel (norm and GELU ride on the first, the
    residual on the second) when it can take them (16-bit GPU tensors), the layers themselves otherwise."""
    parts = _block_parts(feed_forward)
    if parts is None:
        return h + feed_forward(h)
    norm, up, _, down = parts
    hidden = Castle._project(up, h, True, norm=norm, activation="gelu")
    return Castle._project(down, hidden, True, residual=h)


def block_feed_forward(feed_forward: nn.Sequential, h: torch.Tensor, native: bool = True) -> torch.Tensor:
    """feed_forward(h) for the block [norm, linear, GELU, linear] over many rows: the layers themselves; of a native model
    with the two weight gradients formed in row ranges where that pays (castle._linear)."""
    parts = _block_parts(feed_forward) if native else None
    if parts is None:
        return feed_forward(h)
    norm, up, act, down = parts
    return _linear(down, act(_linear(up, norm(h))))


@contextlib.contextmanager
def _no_collection():
    """Python's cyclic garbage collector waits.  A model and the decoder kept from its last `sample` call hold each
    other, so the graph of a dropped model is destroyed by a collection; the destructor synchronises the device, which a
    capture forbids, and an error in a destructor ends the process."""
    enabled = gc.isenabled()
    gc.disable()
    try:
        yield
    finally:
        if enabled:
            gc.enable()


class GraphedDecoder:
    """One captured HIP graph of a whole single-token step of a `CastleLM` on the native path.

    A token step of a small model is a few hundred tiny launches, bound by the host; captured once
    and replayed, it costs one launch.  The cached attention step supports this through a row
    count kept in device memory (`Castle.graph_step`): the graph reads it, uses it and increments
    it, so every replay is the next step.  The graph ends at the logits; sampling stays outside.

    `caches`: the per-layer caches of a native prefill (they are consumed: the graph updates their
    buffers in place; read them back with `caches()`).  `max_len`: rows the caches must hold."""

    def __init__(self, model: "CastleLM", caches, max_len: int):
        stores = [getattr(c, "_store", None) for c in caches]
        if len(stores) != len(model.layers) or any(st is None for st in stores):
            raise RuntimeError("GraphedDecoder needs the native caches of every layer (use_triton=True on a GPU)")
        if not all(_runs_castle_forward(attention) for attention, _ in model.layers):
            raise RuntimeError("GraphedDecoder captures the attention layers' own step: hooks or a `forward` set on them would not run")
        lengths = {st.length for st in stores}
        if len(lengths) != 1:
            raise RuntimeError("the layer caches disagree about their length")
        self.length = lengths.pop()
        for st in stores:
            st.flush()   # the graph starts from complete lookahead keys
        self.stores = [st if st.capacity >= max_len else st.grown(max_len) for st in stores]
        self.base0 = self.length
        # every token goes round the rows of all layers: past what the last-level cache (256 MB) holds, with some room,
        # they are not kept there (12 layers of 16 x 8 heads x 540 rows, 420 MB: 48 tokens 22.5 -> 21.0 ms)
        loop = sum(buf[:, :, :1].numel() * min(max_len, st.capacity) * buf.element_size() for st in self.stores for buf in st.buffers)
        for st in self.stores:
            st.plan.read_once(loop > READ_ONCE_BYTES)
        self.model = model
        device = self.stores[0].buffers[0].device
        batch = self.stores[0].buffers[0].shape[0]
        self.capacity = min(st.capacity for st in self.stores)
        # while warming up and capturing, the count is out of range for every layer: such a step writes nothing
        # [row count, row count up to which the stored lookahead keys are complete]
        self.counters = torch.full((2,), max(st.capacity for st in self.stores), dtype=torch.int32, device=device)
        self.t_device, self.base_device = self.counters[:1], self.counters[1:]
        self.token = torch.zeros((batch, 1), dtype=torch.long, device=device)
        side = torch.cuda.Stream(device=device)
        side.wait_stream(torch.cuda.current_stream(device))
        with torch.cuda.stream(side), torch.no_grad():
            for _ in range(2):   # library handles and workspaces are created outside the capture
                self._step()
        torch.cuda.current_stream(device).wait_stream(side)
        self.graph = torch.cuda.CUDAGraph()
        with _no_collection(), torch.cuda.graph(self.graph), torch.no_grad():
            self.logits = self._step()
            self.t_device += 1
        self._set_counters()
        self.signature = self._signature()

    def _set_counters(self):
        self.counters.copy_(torch.tensor([self.length, self.base0], dtype=torch.int32), non_blocking=False)

    def _signature(self):
        """What the captured graph has baked in: the addresses of the weights it reads."""
        return tuple(p.data_ptr() for p in self.model.parameters())

    def fits(self, caches, max_len: int) -> bool:
        """True if `load(caches)` can reuse this graph for a generation of up to max_len rows."""
        first = getattr(caches[0], "_store", None)
        mine = self.stores[0].buffers[0]
        return (first is not None and max_len <= self.capacity and self.signature == self._signature()
                and first.buffers[0].shape[:2] == mine.shape[:2] and first.buffers[0].shape[3] == mine.shape[3]
                and first.buffers[0].dtype == mine.dtype and first.buffers[0].device == mine.device
                and first.u_half == self.stores[0].u_half)

    def takes(self, prompt, max_len: int) -> bool:
        """True if a prefill of `prompt` may write its caches straight into this decoder's buffers: they have the shape, type and
        room it needs.  (Whether the captured graph still fits is for `fits`, behind the prefill.)"""
        weight = self.model.token_emb.weight
        return (max_len <= self.capacity and all(
            st.buffers[0].shape[:2] == (prompt.shape[0], attention.heads) and st.buffers[0].shape[3] == attention.dim_head
            and st.buffers[0].dtype == weight.dtype and st.buffers[0].device == prompt.device
            and st.u_half == (weight.dtype == torch.bfloat16 and ops.LOOKAHEAD_KEYS_HALF)
            for st, (attention, _) in zip(self.stores, self.model.layers)) and len(self.stores) == len(self.model.layers))

    def load(self, caches):
        """Restarts the decoder from the caches of a new prefill: their rows are copied into the
        buffers the graph was captured on (the graph holds those addresses)."""
        stores = [getattr(c, "_store", None) for c in caches]
        if len(stores) != len(self.stores) or any(st is None for st in stores):
            raise RuntimeError("GraphedDecoder.load needs the native caches of every layer")
        length = stores[0].length
        if any(st.length != length for st in stores) or length > self.capacity:
            raise RuntimeError("these caches do not fit the buffers the graph was captured on")
        for mine, theirs in zip(self.stores, stores):
            if mine is theirs:   # the prefill went into these buffers
                continue
            theirs.flush()
            for dst, src in zip(mine.buffers, theirs.buffers):
                dst[:, :, :length].copy_(src[:, :, :length])
        self.length = self.base0 = length
        self._set_counters()

    def _step(self):
        model = self.model
        embedding = model.token_emb
        plain = _unmodified(embedding, nn.Embedding) and embedding.max_norm is None
        h = _native.host().gather_rows(embedding.weight, self.token) if plain else embedding(self.token)
        for (attention, feed_forward), store in zip(model.layers, self.stores):
            h = attention.graph_step(h, store, self.t_device, self.base_device, residual=h)
            h = token_feed_forward(feed_forward, h)
        return Castle._project(model.to_logits, h, True, norm=model.final_norm)

    def step(self, token):
        """Feeds `token` (batch, 1) and returns the logits (batch, 1, num_tokens) of the next
        position: a view of the graph's output buffer, overwritten by the next call."""
        if self.length >= self.capacity:
            raise RuntimeError(f"the graph was captured for caches of {self.capacity} rows")
        if token is not self.token:   # (whoever wrote the token into the graph's own input hands that in)
            self.token.copy_(token)
        self.graph.replay()
        self.length += 1
        return self.logits

    def caches(self):
        """The per-layer caches as they stand after the steps replayed so far."""
        for st in self.stores:
            st.length, st.base0 = self.length, self.base0
            st.flush()   # the lookahead keys complete; the graph's counters must know, or a later replay would add the pending sources twice
        self.base0 = self.length
        self._set_counters()
        return [st.as_cache() for st in self.stores]


class CastleLM(nn.Module):
    def __init__(self, *, num_tokens, dim, depth, max_seq_len=512, dim_head=64, heads=8, use_triton=True,
                 rotary_emb=True, prenorm=True, tie_embedding=False):
        super().__init__()
        self.max_seq_len = max_seq_len
        self.token_emb = nn.Embedding(num_tokens, dim)
        self.layers = nn.ModuleList()
        for _ in range(depth):
            attention = Castle(dim=dim, heads=heads, dim_head=dim_head, use_triton=use_triton,
                               rotary_emb=rotary_emb, prenorm=prenorm)
            feed_forward = nn.Sequential(
                nn.RMSNorm(dim),
                nn.Linear(dim, 4 * dim, bias=False),
                nn.GELU(),
                nn.Linear(4 * dim, dim, bias=False),
            )
            self.layers.append(nn.ModuleList([attention, feed_forward]))
        self.final_norm = nn.RMSNorm(dim)
        self.to_logits = nn.Linear(dim, num_tokens, bias=False)
        if tie_embedding:
            self.to_logits.weight = self.token_emb.weight

    def forward(self, x, return_loss=False, cache=None, return_next_cache=False):
        """x: (batch, n) token ids.  With return_loss the last position is the target of the one
        before it (shift by one) and the mean cross entropy is returned; otherwise the logits
        (batch, n, num_tokens), plus the list of per-layer caches when return_next_cache."""
        if return_loss:
            x, target = x[:, :-1], x[:, 1:]
        if cache is None and x.dim() == 2 and x.shape[1] > 1 and self._plain(x):
            return self._forward_plain(x, target if return_loss else None, return_next_cache)
        h = self.token_emb(x)
        # one token per sequence, no graph to record: the few rows of every projection go through the small-M kernel
        # (only for a model whose layers run the native kernels: one built with use_triton=False stays on
        # the PyTorch layers throughout, so it remains an independent baseline for the native one)
        native = self._native_on_gpu(h.device)
        token_step = h.shape[1] == 1 and not torch.is_grad_enabled() and native
        next_cache = []
        for index, (attention, feed_forward) in enumerate(self.layers):
            layer_cache = cache[index] if cache is not None and index < len(cache) else None
            if return_next_cache:
                attended, layer_next = attention(h, cache=layer_cache, return_next_cache=True)
                next_cache.append(layer_next)
            else:
                attended = attention(h, cache=layer_cache, return_next_cache=False)
            h = h + attended
            h = token_feed_forward(feed_forward, h) if token_step else h + block_feed_forward(feed_forward, h, native)
        logits = Castle._project(self.to_logits, h, token_step, norm=self.final_norm, native=native)
        if return_loss:
            return F.cross_entropy(logits.transpose(1, 2), target)
        return (logits, next_cache) if return_next_cache else logits

    def _plain(self, x) -> bool:
        """True if whole sequences may run as one native call per block: native layers, unmodified modules, nothing
        hooked onto any of them."""
        embedding, weight = self.token_emb, self.token_emb.weight
        if (not x.is_cuda or x.dtype != torch.long or not _unmodified(embedding, nn.Embedding) or embedding.max_norm is not None
                or embedding.padding_idx is not None or embedding.scale_grad_by_freq or embedding.sparse or weight.device != x.device
                or weight.dtype not in _native.DTYPE_CODES or not _native.is_built()):
            return False
        final, logits, dtype = self.final_norm, self.to_logits, weight.dtype
        if not (_unmodified(final, nn.RMSNorm) and _unmodified(logits, nn.Linear) and logits.bias is None and logits.weight.dtype is dtype
                and final.weight is not None and final.weight.dtype is dtype) or not len(self.layers):
            return False
        like = weight.detach()[None]   # what every block gets, as far as the blocks look at it
        for block in self.layers:
            if not _unmodified(block, nn.ModuleList) or len(block) != 2:
                return False
            attention, feed_forward = block
            if not (_unmodified(attention, Castle) and attention.use_triton and ops.kernels_support(attention.dim_head, dtype) and attention._plain(like)
                    and _block_parts(feed_forward) is not None):
                return False
            norm, up, _, down = feed_forward
            if not (_unmodified(norm, nn.RMSNorm) and norm.weight is not None and norm.weight.dtype is dtype and _unmodified(up, nn.Linear) and up.bias is None
                    and up.weight.dtype is dtype and _unmodified(down, nn.Linear) and down.bias is None and down.weight.dtype is dtype):
                return False
        return True

    def _forward_plain(self, x, target, return_next_cache, stores=None):
        """`forward` over whole sequences, one native call per block: the sum of a residual stream is formed by the
        norm that reads it next.  `stores`: where the layers' caches go, one for each."""
        host = _native.host()
        h, delta, next_cache = host.embedding(self.token_emb.weight, x), None, []
        for index, (attention, feed_forward) in enumerate(self.layers):
            results = attention._layer_native(h, return_next_cache, delta, stores[index] if stores is not None else None)
            if return_next_cache:
                *results, layer_next = results
                next_cache.append(layer_next)
            elif delta is None:
                results = (results,)
            attended, h = results if delta is not None else (results[0], h)
            norm, up, _, down = feed_forward
            delta, h = host.feed_forward(h, attended, norm.weight, norm.eps, up.weight, down.weight)
        logits = host.head(h, delta, self.final_norm.weight, self.final_norm.eps, self.to_logits.weight)
        if target is not None:
            return host.cross_entropy(logits, target)
        return (logits, next_cache) if return_next_cache else logits

    def _decoder_for(self, cache, max_len, keep=True):
        """A GraphedDecoder positioned on `cache`: the one kept from an earlier call when its graph
        still fits (same weights, batch, type; enough rows), else a newly captured one.  keep=False: captured for this
        call alone (what hooks or a replaced `forward` did meanwhile is not for other calls)."""
        kept = self.__dict__.get("_kept_decoder")
        if keep and kept is not None and kept.fits(cache, max_len):
            kept.load(cache)
            return kept
        decoder = GraphedDecoder(self, cache, max_len)
        if keep:
            self.__dict__["_kept_decoder"] = decoder   # not a module attribute: never part of the state
        return decoder

    def release_decoder(self):
        """Drops the graph (and the cache buffers it was captured on) kept from the last `sample` call."""
        self.__dict__.pop("_kept_decoder", None)

    def _unmodified(self) -> bool:
        """True if a replayed graph of a token step does what a call of every module would: no hooks, no replaced `forward`."""
        modules = [self]
        for module in modules:   # (a shared module twice is no harm; `self.modules()` takes three times as long)
            if not _unmodified(module, type(module)):
                return False
            modules += [child for child in module._modules.values() if child is not None]
        return all(_runs_castle_forward(attention) for attention, _ in self.layers)

    def _native_on_gpu(self, device) -> bool:
        return device.type == "cuda" and _native.is_built() and all(attention.use_triton for attention, _ in self.layers)

    @torch.no_grad()
    def sample(self, prompt, seq_len, temperature=1.0, filter_thres=0.9, generator=None, graph=None):
        """Extends `prompt` (batch, p) to `seq_len` tokens and returns the seq_len - p new ones.
        The prompt goes through the parallel path once; afterwards each step feeds the last token
        and the per-layer caches.  temperature = 0 picks the arg-max (no noise).
        graph: replay the token steps as one captured HIP graph (`GraphedDecoder`).  None = when
        the model runs the native kernels on a GPU, its modules are unmodified (no hooks, which a replay would not
        run) and more than a few steps follow; True insists."""
        prompt_len = prompt.shape[-1]
        steps = max(0, seq_len - prompt_len)
        if self._native_on_gpu(prompt.device):
            return self._sample_native(prompt, steps, seq_len, temperature, filter_thres, generator, graph)
        if graph:
            raise RuntimeError("graph=True needs the native kernels on a GPU")

        out, cache = prompt, None
        for _ in range(steps):
            logits, cache = self.forward(out if cache is None else out[:, -1:], cache=cache, return_next_cache=True)
            out = torch.cat((out, pick_token(logits, temperature, filter_thres, generator)), dim=-1)
        return out[..., prompt_len:]

    def _sample_native(self, prompt, steps, seq_len, temperature, filter_thres, generator, graph):
        """`sample` with the native kernels: top-k, noise and arg-max of a token are one launch (the operators for
        large vocabularies) behind the uniform numbers, which come from the generator exactly as `gumbel_noise` draws them; the token
        goes straight into the graph's input."""
        host, decoder, cache = _native.host(), None, None
        batch = prompt.shape[0]
        tokens = torch.empty((batch, steps), dtype=torch.long, device=prompt.device)
        replay = graph or graph is None and steps > 8
        kept = self.__dict__.get("_kept_decoder") if replay else None
        for i in range(steps):
            if decoder is not None:
                logits = decoder.step(decoder.token)
            else:
                if (i == 0 and kept is not None and prompt.dim() == 2 and prompt.shape[1] > 1 and kept.takes(prompt, seq_len)
                        and type(self).forward is CastleLM.forward and "forward" not in self.__dict__ and self._plain(prompt)):
                    # straight into the kept decoder's buffers: 48 copies of 8 MB (12 layers of 16 x 8 heads x 492 rows) took 340 us
                    logits, cache = self._forward_plain(prompt, None, True, kept.stores)
                else:
                    logits, cache = self.forward(prompt if cache is None else tokens[:, i - 1:i], cache=cache, return_next_cache=True)
                if i == 0 and replay:   # (looked into while the GPU works on the prompt)
                    unmodified = self._unmodified()
                    if unmodified or graph:
                        decoder = self._decoder_for(cache, seq_len, unmodified)
            if logits.shape[-1] > SAMPLER_MAX_VOCABULARY:
                tokens[:, i:i + 1] = pick_token(logits, temperature, filter_thres, generator)
                if decoder is not None:
                    decoder.token.copy_(tokens[:, i:i + 1])
                continue
            logits = logits[:, -1] if logits.dtype in _native.DTYPE_CODES else logits[:, -1].float()
            k = math.ceil((1.0 - filter_thres) * logits.shape[-1])
            uniform = None
            if temperature != 0:
                uniform = torch.rand(logits.shape, dtype=torch.float32, device=logits.device, generator=generator)
            if k < 1:   # nothing is kept: the arg-max over equal values, as the operators would have it
                tokens[:, i] = 0
                if decoder is not None:
                    decoder.token.zero_()
                continue
            host.sample_tokens(logits, uniform, k, max(temperature, 1e-10), tokens[:, i], decoder.token if decoder is not None else None)
        return tokens
