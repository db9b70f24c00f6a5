"""Host side of the LoRA surface: adapter registry per layer and the packed layout the kernels read.

The reference keeps one (lora_A, lora_B, alpha, rank, weight) set per adapter inside peft's Linear
wrappers and turns them on / off and scales them from the host
(set_weights_and_activate_adapters, diffusers-hf/src/diffusers/utils/peft_utils.py:238-269;
scale_lora_layers / unscale_lora_layers :103-147).  Here the ACTIVE adapters of a layer are packed
once per activation change into

    A_cat [R, in]   rows of all active A_i stacked, zero padded to R % 32 == 0
    B_cat [out, R]  columns of all active B_i side by side, zero padded
    col_scale [R]   fp32, weight_i * alpha_i / rank_i * global_scale for the columns of adapter i

so that sum_i s_i B_i A_i x is ONE rank-R product inside the fused kernel, and changing a scale only
rewrites col_scale.
"""
from __future__ import annotations

import struct
from dataclasses import dataclass, field
from typing import Dict, List, Optional, Sequence

import numpy as np
import torch

from . import ops

RANK_PAD = 64   # packed rank is padded to the K-stage depth of the GEMM that consumes it
MAX_PACKED_RANK = 128


@dataclass
class Adapter:
    """One LoRA on one layer: down = lora_A [r, in], up = lora_B [out, r]
    (LoRALinearLayer.down/up, diffusers-hf/src/diffusers/models/lora.py:210-211)."""

    down: torch.Tensor
    up: torch.Tensor
    alpha: Optional[float] = None  # network_alpha; None means alpha == rank (lora.py:227-228)
    weight: float = 1.0            # set_adapters weight

    @property
    def rank(self) -> int:
        return self.down.shape[0]

    def multiplier(self, global_scale: float = 1.0) -> float:
        a = self.rank if self.alpha is None else self.alpha
        return float(self.weight) * float(a) / float(self.rank) * float(global_scale)


@dataclass
class PackedAdapters:
    a_cat: torch.Tensor
    b_cat: torch.Tensor
    col_scale: torch.Tensor
    spans: List[tuple] = field(default_factory=list)  # (name, first column, rank)
    # Rank columns beyond the kernels' 128: further packs of at most 128 columns each (A rows / B columns of the same
    # adapters, continued).  Only LoRALinear's own forward applies them; the fused launches that stack several
    # layers' packs take the per-layer path when a layer has any.
    overflow: List["PackedAdapters"] = field(default_factory=list)
    # behind a folded LayerNorm: (norm_key of that norm, A_cat * weight, its row sums, A_cat . bias), fold_layer_norm's last three
    ln: Optional[tuple] = None

    @property
    def R(self) -> int:
        return self.a_cat.shape[0]

    @property
    def wide(self) -> bool:
        """More rank columns than one launch takes?  (Does not make a PooledPack's list.)"""
        return bool(self.__dict__.get("overflow"))

    @property
    def r_used(self) -> int:
        """Rank columns that can be non-zero (the adapters' ranks side by side), rounded up to the 16 columns of one
        MFMA step; the columns from there to R are zero padding."""
        used = max((c + r for _, c, r in self.spans), default=0)
        return min(self.R, (used + 15) // 16 * 16)


class PooledPack(PackedAdapters):
    """A layer's share of the buffers that pack_many fills for many layers.  An activation makes hundreds of these and most are only ever read by address, so
    the tensors are views that are made when somebody asks for them; one that is assigned (`moved`) takes the view's place."""

    def __init__(self, pool: Sequence[torch.Tensor], at: Sequence[int], shape: Sequence[int], names: Sequence[str], ranks: Sequence[int], used: int,
                 norm: Optional[tuple]):
        d = self.__dict__
        d["pool"], d["at"], d["shape"] = pool, at, shape           # buffers (A, B, scales, A * norm, its two terms), offsets in elements, (R, K, N)
        d["names"], d["ranks"], d["used"], d["norm"] = names, ranks, used, norm    # used: r_used of these names and ranks

    def _view(self, name: str, which: int, size: tuple, stride: tuple):
        d = self.__dict__
        v = d.get(name) if name in d else d.get("_" + name)
        return d.setdefault("_" + name, self.pool[which].as_strided(size, stride, self.at[which])) if v is None else v

    def _move(self, name: str, v) -> None:
        self.__dict__[name] = v

    @property
    def moved(self) -> bool:
        d = self.__dict__
        return "a_cat" in d or "b_cat" in d or "col_scale" in d or bool(d.get("overflow"))

    R = property(lambda self: self.shape[0] if "a_cat" not in self.__dict__ else self.a_cat.shape[0])
    r_used = property(lambda self: self.used if "spans" not in self.__dict__ else PackedAdapters.r_used.fget(self))
    a_cat = property(lambda self: self._view("a_cat", 0, (self.shape[0], self.shape[1]), (self.shape[1], 1)), lambda self, v: self._move("a_cat", v))
    b_cat = property(lambda self: self._view("b_cat", 1, (self.shape[2], self.shape[0]), (self.shape[0], 1)), lambda self, v: self._move("b_cat", v))
    col_scale = property(lambda self: self._view("col_scale", 2, (self.shape[0],), (1,)), lambda self, v: self._move("col_scale", v))

    # (lists of this pack, as a PackedAdapters has them: made when somebody asks, kept from then on)
    @property
    def overflow(self):
        return self.__dict__.setdefault("overflow", [])

    @overflow.setter
    def overflow(self, v):
        self.__dict__["overflow"] = v

    @property
    def spans(self):
        d = self.__dict__
        if "spans" not in d:
            out, c = [], 0
            for n, r in zip(self.names, self.ranks):
                out.append((n, c, r))
                c += r
            d.setdefault("spans", out)
        return d["spans"]

    @spans.setter
    def spans(self, v):
        self.__dict__["spans"] = v

    @property
    def ln(self):
        d = self.__dict__
        if d.get("ln") is None and self.norm is not None:
            R, K, _ = self.shape
            _, _, _, an, c1, c2 = self.pool
            at, c = self.at[3:]
            d.setdefault("ln", (self.norm, an.as_strided((R, K), (K, 1), at), c1.as_strided((R,), (1,), c), c2.as_strided((R,), (1,), c)))
        return d.get("ln")

    @ln.setter
    def ln(self, v):
        self.__dict__["ln"] = v

    def addresses(self, norm: Optional[tuple] = None):
        """(A, B, scales, terms 1 and 2), with a norm_key A and the terms behind that norm; None where a tensor has been moved or the norm is another one."""
        d = self.__dict__
        if self.moved or (norm is not None and norm != d["norm"]):
            return None
        pool, at = d["pool"], d["at"]
        b, s = pool[1].data_ptr() + 2 * at[1], pool[2].data_ptr() + 4 * at[2]
        if norm is None:
            return pool[0].data_ptr() + 2 * at[0], b, s, 0, 0
        if d.get("ln") is not None and d["ln"][0] != norm:
            return None
        return pool[3].data_ptr() + 2 * at[3], b, s, pool[4].data_ptr() + 4 * at[4], pool[5].data_ptr() + 4 * at[4]

    def followed_by(self, other) -> bool:
        """Do `other`'s rows lie behind this pack's in every buffer?"""
        R, K, N = self.shape
        return (type(other) is PooledPack and other.pool is self.pool and not self.moved and not other.moved and other.shape[0] == R and other.shape[1] == K
                and other.at[0] == self.at[0] + R * K and other.at[1] == self.at[1] + R * N and other.at[2] == self.at[2] + R
                and (self.norm != other.norm or self.norm is None or (other.at[3] == self.at[3] + R * K and other.at[4] == self.at[4] + R)))


def stacked_packs(packs: Sequence[PackedAdapters]):
    """A_cat, B_cat and the scales of packs that lie one behind the other in a pool, as one tensor each; None otherwise."""
    first = packs[0]
    if type(first) is not PooledPack or first.moved or not all(p.followed_by(q) for p, q in zip(packs[:-1], packs[1:])):
        return None
    R, K, _ = first.shape
    (A, B, S), n = first.pool[:3], len(packs)
    return (A.as_strided((n * R, K), (K, 1), first.at[0]), B.as_strided((sum(p.shape[2] for p in packs), R), (R, 1), first.at[1]),
            S.as_strided((n * R,), (1,), first.at[2]))


def stacked_norm_terms(packs: Sequence[PackedAdapters], norm: tuple):
    """A_cat behind a folded LayerNorm (its norm_key) and the two terms of stacked_packs' packs, as one tensor each; None where they are not in place."""
    if stacked_packs(packs) is None or any(p.addresses(norm) is None for p in packs):
        return None
    R, K, _ = packs[0].shape
    at, c = packs[0].at[3:]
    _, _, _, an, c1, c2 = packs[0].pool
    n = R * len(packs)
    return an.as_strided((n, K), (K, 1), at), c1.as_strided((n,), (1,), c), c2.as_strided((n,), (1,), c)


def interleave_geglu_rows(t: torch.Tensor) -> torch.Tensor:
    """Reorder the output-feature axis (dim 0) of a GEGLU projection tensor from
    [value(0..D) | gate(0..D)] (hidden, gate = proj(x).chunk(2, -1),
    diffusers-hf/src/diffusers/models/activations.py:148) to blocks of 32 value rows followed by
    their 32 gate rows, the order the fused GEGLU epilogue consumes."""
    two_d = t.shape[0]
    D = two_d // 2
    if two_d % 64 != 0:
        raise ValueError("GEGLU interleave needs 2*D % 64 == 0")
    v = t[:D].reshape(D // 32, 1, 32, *t.shape[1:])
    g = t[D:].reshape(D // 32, 1, 32, *t.shape[1:])
    return torch.cat([v, g], dim=1).reshape(t.shape).contiguous()


def pack_adapters(adapters: Dict[str, Adapter], active: Sequence[str], in_features: int, out_features: int,
                  dtype, device, global_scale: float = 1.0, geglu_interleave: bool = False) -> Optional[PackedAdapters]:
    """Build A_cat / B_cat / col_scale for the active adapters (in the given order). Returns None when
    nothing is active (the layer then runs as a plain Linear, like peft with adapters disabled)."""
    names = [n for n in active if n in adapters]
    if not names:
        return None
    for n in names:
        ad = adapters[n]
        if ad.down.shape != (ad.rank, in_features) or ad.up.shape != (out_features, ad.rank):
            raise ValueError(f"adapter {n!r}: down {tuple(ad.down.shape)} / up {tuple(ad.up.shape)} do not fit "
                             f"a [{out_features},{in_features}] layer")
    total = sum(adapters[n].rank for n in names)
    if total > MAX_PACKED_RANK and geglu_interleave:
        raise ValueError("more than 128 rank columns on a GEGLU projection need the plain row order: pack with "
                         "geglu_interleave=False (LoRALinear does)")
    # cut the adapters' rank rows, in order, into packs of at most MAX_PACKED_RANK columns
    packs, pieces, width = [], [], 0
    for n in names:
        r, r0 = adapters[n].rank, 0
        while r0 < r:
            take = min(r - r0, MAX_PACKED_RANK - width)
            pieces.append((n, r0, take))
            width += take
            r0 += take
            if width == MAX_PACKED_RANK:
                packs.append(pieces)
                pieces, width = [], 0
    if pieces:
        packs.append(pieces)
    built = []
    for pcs in packs:
        used = sum(t for _, _, t in pcs)
        R = (used + RANK_PAD - 1) // RANK_PAD * RANK_PAD
        a_cat = torch.zeros((R, in_features), dtype=dtype, device=device)
        b_cat = torch.zeros((out_features, R), dtype=dtype, device=device)
        col_scale = torch.zeros((R,), dtype=torch.float32, device=device)
        spans, c = [], 0
        for n, r0, take in pcs:
            ad = adapters[n]
            a_cat[c:c + take] = ad.down[r0:r0 + take].to(device=device, dtype=dtype)
            b_cat[:, c:c + take] = ad.up[:, r0:r0 + take].to(device=device, dtype=dtype)
            col_scale[c:c + take] = ad.multiplier(global_scale)
            spans.append((n, c, take))
            c += take
        if geglu_interleave:
            b_cat = interleave_geglu_rows(b_cat)
        built.append(PackedAdapters(a_cat, b_cat, col_scale, spans))
    built[0].overflow = built[1:]
    return built[0]


def norm_key(norm) -> tuple:
    """Identifies the parameters a LayerNorm has now."""
    return (id(norm), norm.weight._version, norm.bias._version, norm.weight.data_ptr())


def stacked(views: Sequence[torch.Tensor]) -> Optional[torch.Tensor]:
    """Tensors that lie one behind the other in one buffer (pack_many), as one tensor over their first axis; None otherwise."""
    first = views[0]
    at, store, rows = first.data_ptr(), first.untyped_storage().data_ptr(), 0
    for v in views:
        if v.data_ptr() != at or not v.is_contiguous() or v.shape[1:] != first.shape[1:] or v.untyped_storage().data_ptr() != store:
            return None
        at += v.numel() * v.element_size()
        rows += v.shape[0]
    return first.as_strided((rows,) + tuple(first.shape[1:]), first.stride())


_PACK_F, _UNPACK_I = struct.Struct("<f").pack, struct.Struct("<I").unpack
_PIECE_DTYPES = {torch.bfloat16: 0, torch.float16: 1, torch.float32: 2}


def pack_many_takes(layer, names: Sequence[str]) -> bool:
    """Can pack_many build this layer's pack (else: pack_adapters)?"""
    w = layer._parameters["weight"]
    K, N, adapters = layer.in_features, layer.out_features, layer.adapters
    if not w.is_cuda or w.dtype != torch.bfloat16 or K % 8 != 0 or N % 8 != 0:
        return False
    total, dev = 0, w.device
    for n in names:
        ad = adapters[n]
        down, up = ad.down, ad.up
        r, dtype = down.shape[0], down.dtype
        total += r
        if up.dtype != dtype or dtype not in _PIECE_DTYPES or down.shape != (r, K) or up.shape != (N, r):      # (a piece has one dtype)
            return False
        if down.is_cuda and (down.device != dev or not down.is_contiguous() or down.data_ptr() % 16):
            return False
        if up.is_cuda and (up.device != dev or not up.is_contiguous() or up.data_ptr() % 16):
            return False
    return 0 < total <= MAX_PACKED_RANK and (not layer.geglu or N % 64 == 0)


def pack_many(layers: Sequence, names: Sequence[Sequence[str]]) -> List[PackedAdapters]:
    """pack_adapters for many layers of one device (such as pack_many_takes accepts) in two launches (kh_lora_pack_bf16);
    adapters in host memory are uploaded with one call.  All packs of a kind share one buffer, in the order of `layers`, so
    layers that run as one launch (q / k / v of a self-attention, the context projections) find their stacked operands in place
    (`stacked`, PooledPack.followed_by).  layer.fold_norm: a function that gives the LayerNorm in front of the layer or None."""
    dev = layers[0].weight.device
    host = [t for l, ns in zip(layers, names) for n in ns for t in (l.adapters[n].down, l.adapters[n].up) if not t.is_cuda]
    keep, where = None, {}
    if host:
        keep, addresses = ops.upload_many(host, dev)
        where = {id(t): a for t, a in zip(host, addresses)}
    # One walk that leaves offsets and flat tables, then the buffers.  What an activation makes is counted: thousands of short-lived tuples and tensors
    # bring on the interpreter's full collections (125 ms for the objects of three of these models) the sooner, and views of every layer's operands
    # alone took 3 ms.
    rows, pieces, packs, n_pieces = [], [], [], 0
    at_a = at_b = at_s = at_an = at_c = 0
    b_blocks, padded, keys = [], [], {}
    pool, plain = [], []                               # plain: without the folded norms' buffers, so that a pack that needs none does not keep them
    for l, ns in zip(layers, names):
        d = l.__dict__
        K, N, ads = d["in_features"], d["out_features"], d["adapters"]
        scale, c, ranks = d["global_scale"], 0, []
        for n in ns:
            ad = ads[n]
            down, up = ad.down, ad.up
            r = down.shape[0]
            if where and not down.is_cuda:
                pa = where[id(down)]
            else:
                pa = down.data_ptr()
            if where and not up.is_cuda:
                pb = where[id(up)]
            else:
                pb = up.data_ptr()
            mult = float(ad.weight) * float(r if ad.alpha is None else ad.alpha) / float(r) * float(scale)      # Adapter.multiplier
            pieces += (pa, pb, r, c, _PIECE_DTYPES[down.dtype], _UNPACK_I(_PACK_F(mult))[0])
            ranks.append(r)
            c += r
        R = -(-c // RANK_PAD) * RANK_PAD
        g, nk = l.fold_norm(), None
        if g is not None:
            nk = keys.get(id(g))
            if nk is None:
                w = g.weight
                nk = keys[id(g)] = (norm_key(g), w.data_ptr(), g.bias.data_ptr()) if w.dtype == torch.bfloat16 and w.device == dev else ()
        rows += (at_a, at_an if nk else -1) + (nk[1:] if nk else (0, 0)) + (at_c, at_c, at_b, at_s, K, N, R, int(d["geglu"]), n_pieces, len(ns))
        packs.append(PooledPack(pool if nk else plain, (at_a, at_b, at_s, at_an, at_c), (R, K, N), tuple(ns), ranks, min(R, (c + 15) // 16 * 16), nk[0] if nk else None))
        n_pieces += len(ns)
        padded.append(R)
        b_blocks.append(-(-N // (256 // (R // 8))))
        at_a += R * K
        at_b += R * N
        at_s += R
        if nk:
            at_an += R * K
            at_c += R
    buf = lambda n, dt: torch.empty((n,), dtype=dt, device=dev)
    pool += (buf(at_a, torch.bfloat16), buf(at_b, torch.bfloat16), buf(at_s, torch.float32), buf(at_an, torch.bfloat16), buf(at_c, torch.float32), buf(at_c, torch.float32))
    plain += pool[:3]
    base = [t.data_ptr() for t in pool]
    table = np.array(rows, dtype=np.int64).reshape(-1, 14)
    folded = table[:, 1] >= 0
    for col, which, size in ((0, 0, 2), (1, 3, 2), (4, 4, 4), (5, 5, 4), (6, 1, 2), (7, 2, 4)):    # offsets -> addresses
        table[:, col] = base[which] + size * table[:, col]
    for col in (1, 4, 5):
        table[~folded, col] = 0
    start = lambda counts: np.concatenate([np.zeros(1, np.int32), np.cumsum(counts, dtype=np.int32)])
    ops.lora_pack(table, np.array(pieces, dtype=np.int64).reshape(-1, 6), start(padded), start(b_blocks), dev)
    del keep    # stream-ordered: the launches above are enqueued
    return packs


def rescale_many(rows, device) -> None:
    """rescale_ for many packs on one GPU in one launch; rows: (col_scale, first column, columns, value)."""
    ops.lora_rescale(np.array([(t.data_ptr(), c, r, struct.unpack("<I", struct.pack("<f", v))[0]) for t, c, r, v in rows], dtype=np.int64), device)


def rescale_(packed: PackedAdapters, adapters: Dict[str, Adapter], global_scale: float = 1.0) -> None:
    """Rewrite col_scale only (scale_lora_layers / set_adapters weight change); A_cat/B_cat stay put."""
    for pk in [packed, *packed.overflow]:
        for n, c, r in pk.spans:
            pk.col_scale[c:c + r] = adapters[n].multiplier(global_scale)


# ---- per-block adapter scales -------------------------------------------------------------------------------------
# A per-adapter weight may be one number or a nested description of the UNet's transformers (the surface of
# diffusers-hf/src/diffusers/loaders/unet_loader_utils.py:41-141):
#     {"down": 2, "mid": 3, "up": {"block_0": 4, "block_1": [5, 6, 7]}}
# "mid" is one number; "down" / "up" are a number for the whole half, or a dict per block ("block_<i>") whose value is
# a number for the block or a list with one number per transformer of the block; whatever is left out counts as 1.
# The result maps the module path of every transformer ("up_blocks.1.attentions.2") to its number.

def _transformer_slots(blocks_with_transformer, transformer_per_block):
    """(user spelling, module path, half, block index, transformer index) of every Transformer2DModel, the order the
    reference's result dict has: mid, then up, then down."""
    slots = [("mid", "mid_block.attentions.0", "mid", None, None)]
    for half in ("up", "down"):
        for blk in blocks_with_transformer[half]:
            for j in range(transformer_per_block[half]):
                slots.append((f"{half}.block_{blk}.{j}", f"{half}_blocks.{blk}.attentions.{j}", half, blk, j))
    return slots


def _scale_of_slot(spec: dict, half: str, blk, j):
    node = spec.get(half, 1)
    if half == "mid":
        return node
    if isinstance(node, dict):
        node = node[f"block_{blk}"]      # a per-block dict must name every block that has transformers (KeyError)
    if isinstance(node, list):
        node = node[j]
    return node


def expand_lora_scales_for_one_adapter(scales, blocks_with_transformer: Dict[str, List[int]],
                                       transformer_per_block: Dict[str, int], module_names: Optional[Sequence[str]] = None):
    """Number in, number out; nested description in, {transformer module path: scale} out (see above).
    module_names: when given, every transformer path must occur inside at least one of them (the reference checks
    against the state-dict keys, unet_loader_utils.py:135-139), else ValueError."""
    for what, d in (("blocks_with_transformer", blocks_with_transformer), ("transformer_per_block", transformer_per_block)):
        if set(d) != {"down", "up"}:
            raise ValueError(f"{what} needs to be a dict with keys `'down' and `'up'`")
    if not isinstance(scales, dict):
        return scales
    out = {}
    for user_name, path, half, blk, j in _transformer_slots(blocks_with_transformer, transformer_per_block):
        if module_names is not None and not any(path in m for m in module_names):
            raise ValueError(f"Can't set lora scale for layer {user_name}. It either doesn't exist in this unet or "
                             "it has no attentions.")
        out[path] = _scale_of_slot(scales, half, blk, j)
    return out


def module_weight(weight_for_adapter, module_name: str) -> float:
    """The scale of one module: the float itself, or the first expanded layer name contained in the module's name
    (get_module_weight, diffusers-hf/src/diffusers/utils/peft_utils.py:241-249)."""
    if not isinstance(weight_for_adapter, dict):
        return float(weight_for_adapter)
    for layer_name, w in weight_for_adapter.items():
        if layer_name in module_name:
            return float(w)
    raise RuntimeError(f"No LoRA weight found for module {module_name}.")


def _fold_terms(m: torch.Tensor, gamma: torch.Tensor, beta):
    g = gamma.detach().double()
    md = m.detach().double()
    mp = (md * g).to(m.dtype)
    s1 = mp.double().sum(dim=1)
    s2 = md @ beta.detach().double() if beta is not None else torch.zeros_like(s1)
    return mp.contiguous(), s1, s2


def fold_norm_into_weight(weight: torch.Tensor, bias, gamma: torch.Tensor, beta):
    """(W', c1, c2) of fold_layer_norm: they depend on the weights and the norm only."""
    wp, c1, c2 = _fold_terms(weight, gamma, beta)
    if bias is not None:
        c2 = c2 + bias.detach().double()
    return wp, c1.float().contiguous(), c2.float().contiguous()


def fold_norm_into_adapters(a_cat: torch.Tensor, gamma: torch.Tensor, beta):
    """(A', ca1, ca2) of fold_layer_norm."""
    ap, ca1, ca2 = _fold_terms(a_cat, gamma, beta)
    return ap, ca1.float().contiguous(), ca2.float().contiguous()


def fold_layer_norm(weight: torch.Tensor, bias, gamma: torch.Tensor, beta, a_cat=None):
    """The operands of a linear whose LayerNorm (weight gamma, bias beta over the input features) is folded into the GEMM
    (kh_lora_linear_norm_bf16):  LN(x) W^T + b = rstd * (x W'^T - mean * c1) + c2.
    Returns (W', c1, c2, A', ca1, ca2): W' = W * gamma per input column (rounded to the weight's dtype), c1 the row sums
    of the rounded W', c2 = b + W beta; A' / ca1 / ca2 the same for the stacked adapter A matrices (None without)."""
    return (*fold_norm_into_weight(weight, bias, gamma, beta),
            *(fold_norm_into_adapters(a_cat, gamma, beta) if a_cat is not None else (None, None, None)))
