"""BasicTransformerBlock.forward as one call into the library (kh_transformer_block_bf16).

A block is ten launches of 3 us of host time each; through the single wrappers (checks, allocations, module calls) the same
block costs 230 us, more than its GPU time for images up to 768 x 768.  What stays the same between calls (operand addresses,
shapes, flags) is laid out once per block in a KhBlockDesc and used as long as every tensor, pack, module, hook and option it
was made from is still the one in place; `run` gives None whenever the block has to take the path through its modules
(other processors, hooks, formats the descriptor does not cover, call accounting).
"""
from __future__ import annotations

import ctypes
import operator
import weakref
from ctypes import c_double, c_int64, c_uint64, c_void_p

import torch
from torch import nn

from . import _lib, layers, ops
from .lora import PooledPack, norm_key, stacked_packs


class _Linear(ctypes.Structure):   # KhLinearDesc
    _fields_ = ([(n, c_uint64) for n in ("w", "bias", "a_cat", "b_cat", "col_scale", "c1", "c2", "ca1", "ca2")]
                + [(n, c_int64) for n in ("N", "K", "R", "n_split", "r_used", "geglu", "hint_weight")] + [("eps", c_double)])


class _Block(ctypes.Structure):    # KhBlockDesc
    _fields_ = ([(n, _Linear) for n in ("qkv", "out1", "k2", "v2", "q2", "out2", "geglu", "ff")]
                + [(n, c_uint64) for n in ("n1_w", "n1_b", "n2_w", "n2_b", "n3_w", "n3_b")]
                + [(n, c_double) for n in ("n1_eps", "n2_eps", "n3_eps", "scale1", "scale2")]
                + [(n, c_int64) for n in ("heads", "folded", "fuse_xattn")])


class _Call(ctypes.Structure):     # KhBlockCall
    _fields_ = ([(n, c_void_p) for n in ("x", "ctx", "k", "v", "y", "workspace", "counters", "stats")]
                + [(n, c_int64) for n in ("B", "T", "S", "ldk", "ldv", "bsk", "bsv", "workspace_bytes", "counter_ints", "flags", "hints", "last")]
                + [("tail_hint", c_uint64 * 6)])


_addr = lambda t: 0 if t is None else t.data_ptr()


def _options():
    return layers.LN_FOLD, layers.XATTN_FUSE, layers.LORA_MODE, ops.WEIGHT_PREFETCH, ops.PREFETCH_MIN_K, ops.PREFETCH_SMALL_BYTES


class _Watch:
    """dicts[i].get(keys[i]) has to be objects[i]."""

    def __init__(self):
        self.dicts, self.keys, self.objects = [], [], []

    def expect(self, owner: dict, key: str):
        v = owner.get(key)
        self.dicts.append(owner)
        self.keys.append(key)
        self.objects.append(v)
        return v

    def holds(self) -> bool:
        return all(map(operator.is_, map(dict.get, self.dicts, self.keys), self.objects))


class _Plan:
    """The descriptor of a block without adapters, and the modules, parameters and options that it was made from.  The packed
    adapters change without these whenever a server turns to another request: they are added by _Ready."""

    def __init__(self, blk, folded: bool):
        self.options = _options()
        self.watch = _Watch()
        self.tensors = []                                  # parameters: same version, same address
        self.hooks = []                                    # hook tables that have to be empty
        self.keep = []                                     # what the addresses in the descriptor belong to
        self.linears = []                                  # (entry, layer, LayerNorm folded into it, its norm_key)
        self.ready = None
        self.desc = _Block()
        self.seen(blk, "norm1", "attn1", "norm2", "attn2", "norm3", "ff")
        self.usable = self.describe(blk, folded)
        self.versions = [t._version for t in self.tensors]
        self.addresses = [t.data_ptr() for t in self.tensors]
        if self.usable:
            for l in (self.attn1.to_q, self.attn1.to_k, self.attn1.to_v, *(l for _, l, _, _ in self.linears)):
                layers.hold_pack(l, self)

    def drop_packs(self) -> None:
        self.ready = None

    def holds(self) -> bool:
        return (self.options == _options() and self.watch.holds() and [t._version for t in self.tensors] == self.versions
                and [t.data_ptr() for t in self.tensors] == self.addresses)

    def seen(self, module, *children, params=(), plain=()):
        """Watch a module's children, parameters, plain attributes and hooks."""
        d, expect = module.__dict__, self.watch.expect
        expect(d, "forward")
        self.hooks += [module._forward_hooks, module._forward_pre_hooks]
        for n in children:
            expect(d["_modules"], n)
        for n in params:
            t = expect(d["_parameters"], n)
            if t is not None:
                self.tensors.append(t)
        for n in plain:
            expect(d, n)

    def linear(self, name: str, l, norm=None, stats=False) -> bool:
        """norm: the LayerNorm folded into this layer; stats: it leaves row statistics."""
        if type(l) is not layers.LoRALinear:
            return False
        l.prepare()
        self.seen(l, params=("weight", "bias"), plain=("_rt", "geglu", "bias"))
        _, w, b = l._rt
        if (l.__dict__.get("bias") is not None or w.dtype != torch.bfloat16 or not w.is_cuda or not w.is_contiguous() or (b is not None and not b.is_contiguous())
                or l.in_features % 64 or l.out_features % 8 or (b is not None and b.dtype != torch.bfloat16)
                or (stats and l.out_features > 128 * ops.LN_SLOTS)):
            return False
        d = getattr(self.desc, name)
        d.N, d.K, d.geglu = l.out_features, l.in_features, int(l.geglu)
        c1 = c2 = None
        if norm is not None:
            w, c1, c2 = l._ln_terms(norm)[:3]
            b, d.eps = None, norm.eps
        self.keep.append(self.weights(d, w, b, c1, c2))
        self.linears.append((name, l, norm, None if norm is None else norm_key(norm)))
        return True

    def stacked_weights(self):
        """The operands of q | k | v that do not depend on the packs, and the folded norm's key; None where the layers are not stacked."""
        got = self.qkv_weights
        if got is None:
            a, norm = self.attn1, self.norm1
            q = (a.to_q, a.to_k, a.to_v)
            if a.to_q.out_features % 128 != 0 or a.to_q.in_features % 64 != 0 or any(l.bias is not None for l in q):
                return None
            key = tuple((l.weight.data_ptr(), l.weight._version) for l in q)
            w = a._qkv_weights(key)
            nk = None if norm is None else norm_key(norm)
            got = self.qkv_weights = ((w, None, None) if norm is None else tuple(a._qkv_norm_weights(w, norm, nk, key)), nk)
        return got

    def weights(self, d: _Linear, w, b, c1, c2):
        d.w, d.bias, d.c1, d.c2 = w.data_ptr(), _addr(b), _addr(c1), _addr(c2)
        d.hint_weight = int(d.K >= ops.PREFETCH_MIN_K or w.numel() * 2 <= ops.PREFETCH_SMALL_BYTES)
        return w, b, c1, c2

    def describe(self, blk, folded: bool) -> bool:
        d = self.desc
        a1, a2, ff = blk.attn1, blk.attn2, blk.ff
        norms = (blk.norm1, blk.norm2, blk.norm3)
        if type(a1) is not layers.Attention or type(a2) not in (layers.Attention, type(None)) or type(ff) is not layers.FeedForward:
            return False
        for a in (a1,) if a2 is None else (a1, a2):
            self.seen(a, "to_q", "to_k", "to_v", "to_out", plain=("processor", "heads", "scale", "is_cross"))
            drop = a.to_out[1] if len(a.to_out) == 2 else None
            self.seen(a.to_out, "0", "1")
            if type(a.processor) is not layers.KatzAttnProcessor or type(drop) is not nn.Dropout or drop.p != 0.0:
                return False
            self.seen(drop, plain=("p",))
        geglu = ff.net[0]
        self.seen(ff, "net")
        self.seen(ff.net, "0", "2")
        if type(geglu) is not layers.GEGLU or geglu.enable_fused_geglu:
            return False
        self.seen(geglu, "proj", plain=("enable_fused_geglu",))
        if a1.is_cross or (a2 is not None and (not a2.is_cross or a2.heads != a1.heads)) or (folded and not layers.LN_FOLD):
            return False
        for i, n in enumerate(norms):
            if n is None:
                continue
            if type(n) is not layers.LayerNorm or n.weight.dtype != torch.bfloat16 or n.bias.dtype != torch.bfloat16:
                return False
            self.seen(n, params=("weight", "bias"), plain=("eps",))
            for name, v in ((f"n{i + 1}_w", n.weight.data_ptr()), (f"n{i + 1}_b", n.bias.data_ptr()), (f"n{i + 1}_eps", n.eps)):
                setattr(d, name, v)
        fold = norms if folded else (None,) * 3
        # q | k | v of the self-attention: the operands fused_qkv stacks
        q = d.qkv
        self.attn1, self.norm1 = a1, fold[0]
        for l in (a1.to_q, a1.to_k, a1.to_v):
            if type(l) is not layers.LoRALinear or l.weight.dtype != torch.bfloat16 or not l.weight.is_cuda:
                return False
            l.prepare()
            self.seen(l, params=("weight", "bias"), plain=("_rt", "bias"))
        self.qkv_weights = None
        if folded:
            q.eps = norms[0].eps
        q.N, q.K = 3 * a1.to_q.out_features, a1.to_q.in_features
        self.inner = N = a1.to_q.out_features
        if N != a1.heads * 64 or any(l.out_features != N or l.in_features != q.K for l in (a1.to_k, a1.to_v)):
            return False
        if not (self.linear("out1", a1.to_out[0], stats=folded) and self.linear("geglu", geglu.proj, fold[2])
                and self.linear("ff", ff.net[2], stats=folded)):
            return False
        if a2 is not None and not (self.linear("q2", a2.to_q, fold[1]) and self.linear("k2", a2.to_k) and self.linear("v2", a2.to_v)
                                   and self.linear("out2", a2.to_out[0], stats=folded)):
            return False
        if d.geglu.geglu != 1 or d.ff.K * 2 != d.geglu.N or d.ff.N != q.K or d.out1.N != q.K or d.out1.K != N:
            return False
        if a2 is not None and (d.q2.N != N or d.q2.K != q.K or d.k2.N != N or d.v2.N != N or d.k2.K != d.v2.K or d.out2.K != N or d.out2.N != q.K):
            return False
        d.heads, d.scale1, d.scale2 = a1.heads, a1.scale, a1.scale if a2 is None else a2.scale
        d.folded, d.fuse_xattn = int(folded), int(layers.XATTN_FUSE)
        self.width, self.cross, self.kv_width = q.K, a2 is not None, d.k2.K
        self.last_key = int(d.ff.w)
        return True


class _Ready:
    """A plan's descriptor with the packs that are in place now.  Made anew when they change and never written to after that:
    another thread may be inside the library with the previous one."""

    def __init__(self, plan: _Plan):
        self.epoch, self.packs = layers._pack_epoch, _Watch()
        self.sizes = {}                                    # (B, T, S, own_kv) -> (workspace bytes, counters)
        self.keep = []
        self.desc = _Block.from_buffer_copy(plan.desc)
        self.at = ctypes.addressof(self.desc)
        self.usable = self.fill(plan)

    def holds(self) -> bool:
        return self.epoch == layers._pack_epoch and self.packs.holds()

    def fill(self, plan) -> bool:
        expect, keep = self.packs.expect, self.keep
        attn = plan.attn1
        qkv = []
        for l in (attn.to_q, attn.to_k, attn.to_v):
            p = expect(l.__dict__, "_packed")
            qkv.append(p)
            if p is not None:
                expect(p.__dict__, "a_cat")
        split = layers.LORA_MODE == "split"
        for name, l, norm, nk in plan.linears:
            p = expect(l.__dict__, "_packed")
            if p is None:
                continue
            v, d = p.__dict__, getattr(self.desc, name)
            if p.wide or not split:
                return False
            for t in ("a_cat", "b_cat", "col_scale"):
                expect(v, t)
            at = p.addresses(nk) if type(p) is PooledPack else None
            if at is not None:                             # by address: no views are made
                d.a_cat, d.b_cat, d.col_scale, d.ca1, d.ca2 = at
                d.R, d.r_used = p.shape[0], p.r_used
                keep.append(p)
                continue
            a, b, s = p.a_cat, p.b_cat, p.col_scale
            ca1 = ca2 = None
            if norm is not None:
                a, ca1, ca2 = l._ln_terms(norm)[3:]
            self.operands(d, a, b, s, ca1, ca2, p.r_used)
        q, norm = self.desc.qkv, plan.norm1
        st, first = None, qkv[0]
        weights = plan.stacked_weights() if split and type(first) is PooledPack else None
        side_by_side = stacked_packs(qkv) if weights is not None else None
        if side_by_side is not None:
            (w, c1, c2), nk = weights
            at = [p.addresses(nk) for p in qkv]
            if None not in at:
                st = weights
                plan.weights(q, w, None, c1, c2)
                q.a_cat, q.b_cat, q.col_scale, q.ca1, q.ca2 = at[0]
                q.R, q.r_used, q.n_split = first.shape[0], max(p.r_used for p in qkv), plan.inner
                a, b, _ = side_by_side                     # (hints hold them weakly)
                if nk is not None:
                    a = first.pool[3].as_strided(a.shape, a.stride(), first.at[3])
                keep += (qkv, w, c1, c2, a, b)
                refs = (w, a, b)
        if st is None:
            st = attn._qkv_state()
            if st is None:
                return False
            w, c1, c2, a, ca1, ca2 = attn._qkv_folded(st, norm) if norm is not None else (st["w"], None, None, st.get("a"), None, None)
            keep.append(plan.weights(q, w, None, c1, c2))
            refs = (w, None, None)
            if st["R"]:
                self.operands(q, a, st["b"], st["s"], ca1, ca2, st["r_used"])
                q.n_split = plan.inner
                refs = (w, a, st["b"])
        self.first = tuple(None if t is None else weakref.ref(t) for t in refs)
        self.first_key = int(q.w)
        return True

    def operands(self, d: _Linear, a, b, s, ca1, ca2, r_used: int):
        d.a_cat, d.b_cat, d.col_scale, d.ca1, d.ca2 = a.data_ptr(), b.data_ptr(), s.data_ptr(), _addr(ca1), _addr(ca2)
        d.R, d.r_used = b.shape[1], r_used
        self.keep.append((a, b, s, ca1, ca2))

    def needs(self, B, T, S, own_kv):
        key = (B, T, S, own_kv)
        got = self.sizes.get(key)
        if got is None:
            ws, n = c_int64(), c_int64()
            _lib.check(_lib.load().kh_transformer_block_needs(self.at, B, T, S, int(own_kv), ctypes.byref(ws), ctypes.byref(n)), "kh_transformer_block_needs")
            if len(self.sizes) >= 64:
                self.sizes.clear()
            got = self.sizes[key] = (ws.value, n.value)
        return got


_plans: "weakref.WeakKeyDictionary" = weakref.WeakKeyDictionary()   # block -> [plan with separate norms, plan with folded norms]
_global_hooks = (nn.modules.module._global_forward_hooks, nn.modules.module._global_forward_pre_hooks)


def run(blk, h, ctx, stats, last: bool):
    """The block on h, or None: take the path through the modules.  Arguments as BasicTransformerBlock.forward's."""
    if (ops.CALL_LOG is not None or not h.is_cuda or h.dtype != torch.bfloat16 or h.dim() != 3 or not h.is_contiguous()
            or (stats is not None and not stats.valid) or _global_hooks[0] or _global_hooks[1]):
        return None
    folded = stats is not None
    both = _plans.get(blk)
    if both is None:
        both = _plans[blk] = [None, None]
    plan = both[folded]
    if plan is None or not plan.holds():
        plan = both[folded] = _Plan(blk, folded)
    if not plan.usable or any(plan.hooks):
        return None
    ready = plan.ready
    if ready is None or not ready.holds():
        ready = plan.ready = _Ready(plan)
        if not ready.holds():      # another thread replaced a pack meanwhile: nobody else would drop the old one
            plan.ready = None
    if not ready.usable:
        return None
    B, T, C = h.shape
    if C != plan.width or (ctx is not None) != plan.cross or (folded and stats.buf.numel() != B * T * ops.LN_SLOTS * 2):
        return None
    call = _Call()
    S, own_kv = 0, False
    if plan.cross:
        kv = blk.attn2.ctx_kv
        if kv is not None and kv[0] is ctx:
            _, k, v = kv
            S = k.shape[1]
            if k.shape != (B, S, plan.inner) or v.shape != k.shape or k.stride(2) != 1 or v.stride(2) != 1 or k.dtype != torch.bfloat16 or v.dtype != torch.bfloat16:
                return None
            call.k, call.v = k.data_ptr(), v.data_ptr()
            call.bsk, call.ldk, _ = k.stride()
            call.bsv, call.ldv, _ = v.stride()
        else:
            if not ctx.is_cuda or ctx.dtype != torch.bfloat16 or ctx.dim() != 3 or not ctx.is_contiguous() or ctx.shape[0] != B or ctx.shape[2] != plan.kv_width:
                return None
            S, own_kv = ctx.shape[1], True
            call.ctx = ctx.data_ptr()
    nbytes, ints = ready.needs(B, T, S, own_kv)
    y = torch.empty_like(h)
    ws = h.new_empty((nbytes,), dtype=torch.uint8)
    call.x, call.y, call.workspace, call.workspace_bytes = h.data_ptr(), y.data_ptr(), ws.data_ptr(), nbytes
    if folded:
        call.stats = stats.buf.data_ptr()
    call.B, call.T, call.S, call.last = B, T, S, int(last)
    ranges = ops.chain_hints(ready.first_key, ready.first, plan.last_key)
    if ranges is not None:
        call.hints = 1
        for i, r in enumerate(ranges):
            call.tail_hint[2 * i], call.tail_hint[2 * i + 1] = r
    lib, counters, call.flags = _lib.load(), 0, (1 << 8) if layers.LORA_SHRINK == "separate" else 0
    if ints and not call.flags:
        counters = ops.counters_begin(h.device, ints)
        call.counters, call.counter_ints, call.flags = counters, ints, 0 if counters else 1 << 24
    try:
        rc = lib.kh_transformer_block_bf16(ready.at, ctypes.addressof(call), ops._stream())
    finally:
        if counters:
            ops.counters_end(h.device)
    _lib.check(rc, "kh_transformer_block_bf16")
    return y


# ---- one linear ------------------------------------------------------------------------------------------------------
class _LinearReady:
    """A LoRALinear's operands, checked once, and the parameters and pack they come from (never written to after it is made)."""

    def __init__(self, l):
        l.prepare()
        params = l._parameters
        self.weight, self.bias, self.pack = params["weight"], params.get("bias"), l._packed
        self.seen = self.state()
        _, w, b = l._rt
        p = self.pack
        self.a_cat = None if p is None else p.a_cat
        self.usable = (type(l) is layers.LoRALinear and l.__dict__.get("bias") is None and w.is_cuda and w.dtype == torch.bfloat16 and w.is_contiguous()
                       and (b is None or (b.dtype == torch.bfloat16 and b.is_contiguous()))
                       and (p is None or (not p.wide and layers.LORA_MODE == "split" and l.in_features % 64 == 0)))
        if not self.usable:
            return
        d = self.desc = _Linear()
        d.N, d.K, d.geglu, d.w, d.bias = l.out_features, l.in_features, int(l.geglu), w.data_ptr(), _addr(b)
        b_cat = None
        if p is not None:
            b_cat = p.b_cat
            d.a_cat, d.b_cat, d.col_scale = p.a_cat.data_ptr(), b_cat.data_ptr(), p.col_scale.data_ptr()
            d.R, d.r_used = p.R, p.r_used
        self.keep = (w, b, b_cat, None if p is None else p.col_scale)
        self.refs = tuple(None if t is None else weakref.ref(t) for t in (w, self.a_cat, b_cat))
        self.at, self.key, self.device = ctypes.addressof(d), int(d.w), w.device
        self.N, self.K, self.R, self.width = d.N, d.K, d.R, d.N // 2 if l.geglu else d.N

    def state(self):
        w, b = self.weight, self.bias
        return (w._version, w.data_ptr(), 0) if b is None else (w._version, w.data_ptr(), b._version)

    def holds(self, l) -> bool:
        d, params, p = l.__dict__, l._parameters, self.pack
        return (d["_packed"] is p and params["weight"] is self.weight and params.get("bias") is self.bias and d.get("bias") is None and self.seen == self.state()
                and (p is None or p.a_cat is self.a_cat))


_linears: "weakref.WeakKeyDictionary" = weakref.WeakKeyDictionary()   # LoRALinear -> _LinearReady


def drop_linear(l) -> None:
    """l's pack has been replaced."""
    _linears.pop(l, None)


def run_linear(l, x, residual):
    """l on x (+ residual), or None: take the general path."""
    if ops.CALL_LOG is not None or not x.is_cuda or x.dtype is not torch.bfloat16 or not x.is_contiguous():
        return None
    r = _linears.get(l)
    if r is None or not r.holds(l):
        r = _linears[l] = _LinearReady(l)
        if not r.holds(l):         # as in run
            drop_linear(l)
    if not r.usable or (r.R and layers.LORA_MODE != "split"):
        return None
    shape = x.shape
    M = x.numel() // r.K
    if shape[-1] != r.K or M == 0:
        return None
    res = 0
    if residual is not None:
        if not residual.is_cuda or residual.dtype is not torch.bfloat16 or not residual.is_contiguous() or residual.numel() != M * r.N:
            return None
        res = residual.data_ptr()
    y = x.new_empty((*shape[:-1], r.width))
    t = x.new_empty((M, r.R)) if r.R else None
    lib, counters, flags = _lib.load(), 0, (1 << 8) if layers.LORA_SHRINK == "separate" else 0
    ranges = ops.chain_hints(r.key, r.refs, r.key)
    if ranges is not None:
        lib.kh_set_weight_prefetch(None, 0)
        for ptr, nbytes in ranges:
            lib.kh_set_weight_prefetch(ptr, nbytes)
    stream = ops._stream()
    if r.R and not flags:
        counters = ops.counters_begin(r.device, (M + 127) // 128 + 1, stream)
    try:
        rc = lib.kh_lora_linear_desc_bf16(r.at, x.data_ptr(), res, y.data_ptr(), None if t is None else t.data_ptr(), counters or None, M, flags, stream)
    finally:
        if counters:
            ops.counters_end(r.device)
    if rc:
        _lib.check(rc, "kh_lora_linear_desc_bf16")
    return y
