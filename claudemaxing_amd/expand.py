"""A decoder layer's NF4 weight expansions issued as one launch.

In the training step a decoder layer multiplies seven frozen NF4 weights by their fp16 expansions:
the attention's q, k and v (one product, qkv.py) and o projections and the MLP's gate, up and down
projections. Each is expanded to fp16 by the dequant kernel right before its product, in
the forward and again in the backward. Those are short launches (6-9 us each at
Qwen2.5-1.5B's shapes, of which the ramp and the drain of a launch are a large part), so the
layer issues them together, through cm_nf4_dequant_group:

* forward: the patched decoder layer calls `expand_layer` first and `drop` at its end, also when it
  raises. In between, the first consumer that asks for an expansion (`take` / `take_pair` /
  `take_rows`, called by the o and down projections' MatMulNF4, the MLP and NF4QKV instead of
  expanding) sets off the group: its own weights and those of the layer's later products that will
  take the dequant route at this token count (o and down into their own fp16 weights, gate and up
  into one [2F, K] weight, the MLP's merged product; q, k and v one under another when NF4QKV asks).
* backward: the down projection's input gradient is the first expansion of the layer's
  backward. `backward_group`, called there, finds the layer's group (recorded in its forward)
  and expands down, gate/up, o and q/k/v together the same way, for the MLP's input gradient, then
  the o projection's and NF4QKV's.

Every weight is expanded by the dequant kernel's own code (the values of dequantize_nf4, bit
for bit), and a consumer that finds nothing left for it expands its weight itself: the values
and the routes are the same with or without the grouping. Everything runs on the caller's
current stream, in order, so a captured step replays it as it runs eagerly.

What is left belongs to one pass: it is handed out on the stream it was expanded on, inside the
backward pass (autograd graph task) it was expanded in, or outside of any, and only for the very
weights it was expanded from, unmodified since. So a backward that ends early (a partial
torch.autograd.grad, an exception) leaves nothing that a later call, another stream or a graph
capture could take; the next layer's pass on the device frees it.
"""

import weakref

import torch

from . import _lib
from . import nf4_linear as _nl  # imports this module in turn: used by attribute only

_READY = {}   # device index -> _Left: what the current layer's group left
_GROUPS = {}  # down projection's packed pointer -> weak reference to its decoder layer


def _version(t):
    try:
        return t._version
    except (RuntimeError, AttributeError):  # an inference tensor has none; no tensor
        return None


def _sources(pairs):
    return [(p, s, _version(p), _version(getattr(s, "absmax", None))) for p, s in pairs]


class _Left(dict):
    """The expansions one group launch left: {key: (fp16 weight, the weights it was expanded from and
    their versions)} with key = packed pointer, ("pair", gate, up) or ("rows", q, k, v). The weights
    are held, so no other can have their address. `pending`: the layer whose forward has not asked
    for anything yet, with what its plan needs."""

    def __init__(self, device, pending=None):
        super().__init__()
        self.device, self.pending = device, pending
        self.task = torch._C._current_graph_task_id()  # -1 outside of a backward pass
        self.stream = _lib.stream(device) if device.type == "cuda" else None

    def leave(self, key, weight, pairs):
        self[key] = weight, _sources(pairs)

    def take(self, key, pairs):
        if self.task != torch._C._current_graph_task_id() or (
                self.stream is not None and self.stream != _lib.stream(self.device)):
            return None
        if self.pending is not None:
            pending, self.pending = self.pending, None
            _forward_group(self, pairs if key.__class__ is tuple and key[0] == "rows" else None,
                           *pending)
        weight, sources = self.pop(key, (None, ()))
        for (packed, state), (p, s, version, scales) in zip(pairs, sources):
            if (packed is not p or state is not s or _version(p) != version
                    or _version(getattr(s, "absmax", None)) != scales):
                return None
        return weight


def _take(device, key, pairs):
    ready = _READY.get(device.index)
    if ready is None:
        return None
    return ready.take(key, pairs) if isinstance(ready, _Left) else ready.pop(key, None)


def _nf4_module(m):
    return (isinstance(m, _nl.NF4Linear) and m.compute_dtype == torch.float16
            and not (m._forward_hooks or m._forward_pre_hooks))


def _single_route(m, tokens):
    """MatMulNF4 expands this layer's weight with the dequant kernel (not the fused GEMM) for
    `tokens` rows in fp16."""
    if not _nf4_module(m):
        return False
    state = m.quant_state
    return not (_nl.fused_pays(tokens, *state.shape) and _nl.fused_supported(m.packed, state))


def _pair_route(gp, up, tokens, x_dtype):
    """The MLP's recompute takes its merged gate/up product for `tokens` rows of an x_dtype
    input (swiglu_recompute._merged_route), through MLPInputRecompute: a call with gradients
    enabled (the MLP input of a decoder layer with trainable adapters needs its gradient)."""
    from . import swiglu_recompute as SR

    return (_nf4_module(gp) and _nf4_module(up) and gp.bias is None and up.bias is None
            and SR._frozen(gp) and SR._frozen(up)
            and SR._merged_route(tokens, gp.packed.is_cuda, x_dtype, gp, up))


def _rows_key(packed):
    return ("rows", *(p.data_ptr() for p in packed))


def _issue(left, singles, pair, rows):
    """Expand `singles` (NF4Linear modules), `pair` ((gate, up) or None) and `rows` (the (packed,
    QuantState) of q, k and v or None) in one launch, into `left`."""
    pairs, pointers = [], []
    empty = dict(dtype=torch.float16, device=left.device)
    for m in singles:
        w = torch.empty(m.quant_state.shape, **empty)
        pairs.append((m.packed, m.quant_state))
        pointers.append(w.data_ptr())
        left.leave(m.packed.data_ptr(), w, pairs[-1:])
    if pair is not None:
        gp, up = pair
        f, k = gp.quant_state.shape
        w2 = torch.empty(2 * f, k, **empty)
        pairs += [(gp.packed, gp.quant_state), (up.packed, up.quant_state)]
        pointers += [w2.data_ptr(), w2.data_ptr() + 2 * f * k]
        left.leave(("pair", gp.packed.data_ptr(), up.packed.data_ptr()), w2, pairs[-2:])
    if rows is not None:
        k = int(rows[0][1].shape[1])
        w3 = torch.empty(sum(int(state.shape[0]) for _, state in rows), k, **empty)
        pairs += rows
        at = w3.data_ptr()
        for _, state in rows:
            pointers.append(at)
            at += 2 * int(state.shape[0]) * k
        left.leave(_rows_key([packed for packed, _ in rows]), w3, rows)
    _nl.expand_to(pairs, pointers, torch.float16, left.device)


def _forward_group(left, rows, layer, tokens, x_dtype, grad, x_grad):
    """The group of a layer's forward on `tokens` rows of an x_dtype input (grad: gradients enabled;
    x_grad: the input needs one), set off by the first consumer (rows: NF4QKV's weights when it is
    that): expanded when it has at least two weights, and recorded for the backward: (o and down
    modules whose products take the dequant route, (gate, up) of the merged product or None, q/k/v
    when the backward multiplies by them too). Found anew for each pass, by the questions the
    consumers ask."""
    attn, mlp = getattr(layer, "self_attn", None), getattr(layer, "mlp", None)
    o, down = getattr(attn, "o_proj", None), getattr(mlp, "down_proj", None)
    gp, up = getattr(mlp, "gate_proj", None), getattr(mlp, "up_proj", None)
    o = o if _single_route(o, tokens) else None
    down = down if _single_route(down, tokens) else None
    pair = (gp, up) if grad and _pair_route(gp, up, tokens, x_dtype) else None
    singles = [m for m in (o, down) if m is not None]
    if grad:
        layer.__dict__.pop("_cm_expand_plan", None)
    if len(singles) + (2 if pair else 0) + (3 if rows else 0) < 2:
        return
    _issue(left, singles, pair, rows)
    if down is not None and grad:
        # the backward finds the layer (and its group: the same routes) from the down weight
        layer.__dict__["_cm_expand_plan"] = (o, down, pair, rows if x_grad else None)
        ref = _GROUPS.get(down.packed.data_ptr())
        if ref is None or ref() is not layer:
            if len(_GROUPS) > 1024:  # entries of models that are gone
                _GROUPS.clear()
            _GROUPS[down.packed.data_ptr()] = weakref.ref(layer)


def expand_layer(layer, hidden):
    """At the start of a decoder layer's forward on `hidden` (its input, [..., H] on the GPU): the
    first expansion asked for until `drop` sets off the layer's group."""
    _READY[hidden.device.index] = _Left(hidden.device, (
        layer, hidden.numel() // max(hidden.shape[-1], 1), hidden.dtype, torch.is_grad_enabled(),
        hidden.requires_grad))


def take(packed, dtype, state=None):
    """The fp16 expansion of `packed` (with its QuantState) left by the group launch, once; None when
    there is none (or `dtype` is not fp16)."""
    if dtype != torch.float16:
        return None
    return _take(packed.device, packed.data_ptr(), [(packed, state)])


def take_pair(gate_proj, up_proj):
    """The merged [2F, K] fp16 weight [Wg; Wu] left by the group launch, once; or None."""
    gate, up = gate_proj.packed, up_proj.packed
    return _take(gate.device, ("pair", gate.data_ptr(), up.data_ptr()),
                 [(p.packed, getattr(p, "quant_state", None)) for p in (gate_proj, up_proj)])


def take_rows(pairs):
    """The stacked fp16 weights of `pairs` [(packed, QuantState)] left by the group launch, once; or
    None."""
    return _take(pairs[0][0].device, _rows_key([p for p, _ in pairs]), pairs)


def backward_group(packed, dtype):
    """In the backward, for the down projection of a layer whose forward recorded a group: expand
    down, the merged gate/up weight, o and q/k/v in one launch and leave them for `take`,
    `take_pair` and `take_rows`; the down weight, or None for any other weight."""
    ref = _GROUPS.get(packed.data_ptr())
    layer = None if ref is None else ref()
    plan = None if layer is None else layer.__dict__.get("_cm_expand_plan")
    if plan is None or dtype != torch.float16:
        return None
    o, down, pair, rows = plan
    if down.packed is not packed:
        return None
    drop(packed.device)
    left = _Left(packed.device)
    _issue(left, [down] if o is None else [down, o], pair, rows)
    _READY[packed.device.index] = left
    return left[packed.data_ptr()][0]


def drop(device):
    """Forget what was left on `device` (unused expansions are freed)."""
    _READY.pop(device.index, None)
