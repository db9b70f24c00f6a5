"""Kernel variants at the sizes where they can go wrong: edges of tiles, remainders, the smallest and largest of a range."""
import pytest
import torch

from helpers import assert_close_rel, bf16_round
from oracle import ops as O

pytestmark = pytest.mark.gpu

BF = torch.bfloat16


def dev():
    return torch.device("cuda:0")


def say(*a):
    print(*a, flush=True)


@pytest.mark.parametrize("M,N,K,R", [(1, 1, 4, 0), (64, 64, 32, 32), (65, 63, 36, 4), (31, 130, 100, 36), (200, 70, 644, 128), (129, 640, 640, 32)])
def test_lora_linear_f32_matrix_kernel(M, N, K, R):
    """lora_linear in fp32: ragged tiles in every dimension, column counts that are no multiple of 4, all K remainders."""
    from katz_amd import ops

    say("lora_linear, fp32", M, N, K, R)
    g = torch.Generator().manual_seed(M + N)
    x, w, b, res = (torch.randn(*s, generator=g) for s in ((M, K), (N, K), (N,), (M, N)))
    A, Bm = (torch.randn(R, K, generator=g) * 0.1, torch.randn(N, R, generator=g) * 0.1) if R else (None, None)
    d = dev()
    on = lambda t: None if t is None else t.to(d)
    y = ops.lora_linear(on(x), on(w), on(b), on(A), on(Bm), torch.full((R,), 1.5, device=d) if R else None, residual=on(res))
    torch.cuda.synchronize()
    ref = O.lora_linear(x.double(), w.double(), b.double(), [(A.double(), Bm.double(), 1.5)] if R else [], res.double()).float()
    assert_close_rel(y, ref, 1e-5, "fp32 linear")


@pytest.mark.parametrize("M,N,K,R", [(1, 1, 4, 0), (64, 64, 32, 32), (65, 63, 36, 4), (31, 130, 100, 36), (200, 70, 644, 128), (300, 1280, 640, 32), (129, 65, 64, 0)])
def test_lora_linear_split_f32(M, N, K, R):
    """kh_lora_linear_split_f32 (the fp32 instruction, no planes: the shrink without workgroups that split) at ragged tiles in every dimension, column
    counts that are no multiple of 4 and all K remainders, behind a T and in front of a guard that it must not touch, against 64 bits.

    Bound, elementwise and relative to the sum of the magnitudes of the summands: a truncation of 2^-23 for every two columns of K and R
    (the matrix instruction adds two), one rounding per term behind them; the same once more for T."""
    from katz_amd import _lib, ops

    say("kh_lora_linear_split_f32", M, N, K, R)
    lib, d, g = _lib.load(), dev(), torch.Generator(device="cuda").manual_seed(M + N + K)
    rn = lambda *s, std=1.0: torch.randn(*s, generator=g, device=d) * std
    x, w, b, res = rn(M, K), rn(N, K, std=K ** -0.5), rn(N), rn(M, N)
    A, B, sc = (rn(R, K, std=0.1), rn(N, R, std=0.1), torch.full((R,), 1.5, device=d)) if R else (None, None, None)
    t, y = torch.full((M * R + 32,), 7.0, device=d), torch.full((M * N + 32,), 7.0, device=d)
    p = lambda z: None if z is None else z.data_ptr()
    rc = lib.kh_lora_linear_split_f32(p(x), p(w), p(b), p(A), p(B), p(sc), p(t) if R else None, p(res), p(y), M, N, K, R, ops._stream())
    assert rc == 0
    torch.cuda.synchronize()
    assert (t[M * R:] == 7).all() and (y[M * N:] == 7).all()
    f = lambda z: z.double()
    ref, mag = f(x) @ f(w).T + f(b) + f(res), f(x).abs() @ f(w).abs().T + f(b).abs() + f(res).abs()
    if R:
        want = 1.5 * f(x) @ f(A).T
        assert ((f(t[:M * R].view(M, R)) - want).abs() <= (K / 2 + 10) * 2.0 ** -23 * 1.5 * (f(x).abs() @ f(A).abs().T)).all()
        ref += want @ f(B).T
        mag += 1.5 * (f(x).abs() @ f(A).abs().T) @ f(B).abs().T
    assert ((f(y[:M * N].view(M, N)) - ref).abs() <= (K + R + 14) * 2.0 ** -23 * mag).all()


def test_lora_linear_f32_of_few_rows_on_many_columns():
    """lora_linear takes the form without planes where they do not pay: its bits."""
    from katz_amd import _lib, ops

    M, N, K, R = 100, 5120, 64, 32
    say("lora_linear, fp32, few rows", M, N, K, R)
    lib, d, g = _lib.load(), dev(), torch.Generator(device="cuda").manual_seed(3)
    assert lib.kh_lora_linear_planes_f32_bytes(N, K, R) > 0 and lib.kh_lora_linear_planes_f32_pays(M, N, K, R) == 0
    x, w, A, B = (torch.randn(*s, generator=g, device=d) for s in ((M, K), (N, K), (R, K), (N, R)))
    sc, t, y = torch.full((R,), 0.5, device=d), torch.empty(M, R, device=d), torch.empty(M, N, device=d)
    assert lib.kh_lora_linear_split_f32(x.data_ptr(), w.data_ptr(), None, A.data_ptr(), B.data_ptr(), sc.data_ptr(), t.data_ptr(), None, y.data_ptr(),
                                        M, N, K, R, ops._stream()) == 0
    assert torch.equal(ops.lora_linear(x, w, None, A, B, sc), y)


@pytest.mark.parametrize("M,N,K,R", [(1, 5, 4, 4), (64, 80, 32, 0), (65, 81, 36, 32), (300, 1280, 100, 36), (1300, 1284, 68, 4), (8200, 640, 640, 32)], ids=str)
def test_lora_linear_f32_on_bf16_planes(M, N, K, R):
    """kh_lora_linear_planes_f32 on each of its tiles, ragged in every dimension, against 64 bits.

    Bound, elementwise and relative to the sum of the magnitudes of the summands: the three products left out, each at most 2^-24 of its
    factors' product (2^-23 is allowed for); seven truncations of 2^-23 in a stage's sum of its own; one rounding of 2^-24 per stage of 32 columns and per term
    behind them; the same once more for T."""
    from katz_amd import _lib, ops

    say("lora_linear_planes_f32", M, N, K, R)
    d, g = dev(), torch.Generator(device="cuda").manual_seed(M + N + K)
    rn = lambda *s, std=1.0: torch.randn(*s, generator=g, device=d) * std
    x, w, b, res = rn(M, K), rn(N, K, std=K ** -0.5), rn(N), rn(M, N)
    A, B, sc = (rn(R, K, std=0.1), rn(N, R, std=0.1), torch.full((R,), 1.5, device=d)) if R else (None, None, None)
    assert _lib.load().kh_lora_linear_planes_f32_bytes(N, K, R) > 0
    y = ops.lora_linear(x, w, b, A, B, sc, residual=res)
    f = lambda t: t.double()
    ref, mag = f(x) @ f(w).T + f(b) + f(res), f(x).abs() @ f(w).abs().T + f(b).abs() + f(res).abs()
    if R:
        ref += 1.5 * (f(x) @ f(A).T) @ f(B).T
        mag += 1.5 * (f(x).abs() @ f(A).abs().T) @ f(B).abs().T
    assert ((f(y) - ref).abs() <= (2 * (3 + 7) + K / 32 + 4) * 2.0 ** -23 * mag).all()


@pytest.mark.parametrize("where,e", [("x", -108), ("x", -118), ("w", -122), ("x", -126), ("b", -119), ("one", -122)])
def test_lora_linear_f32_of_small_operands(where, e):
    """Operands whose lower bf16 planes would be subnormal or vanish keep their 24 bits: all of x, W or B_cat at 2^e, or one column of x at 2^e that
    meets weights of 2^100, among others of ordinary size.  The bound of test_lora_linear_f32_on_bf16_planes with the sixteen truncations of the
    fp32 instruction in place of its seven, and the place of the last subnormal bit (2^-149) per summand."""
    from katz_amd import ops

    say("lora_linear_f32, small operands", where, e)
    d, g = dev(), torch.Generator(device="cuda").manual_seed(-e)
    M, N, K, R = 200, 240, 128, 32
    rn = lambda *s, std=1.0: torch.randn(*s, generator=g, device=d) * std
    x, w, A, B, sc = rn(M, K), rn(N, K), rn(R, K, std=0.1), rn(N, R), torch.ones(R, device=d)
    small = lambda t: (t.double() * 2.0 ** e).float()
    if where == "x":
        x = small(x)
    elif where == "w":
        w, B = small(w), small(B)
    elif where == "b":
        w.zero_()
        B = small(B)
    else:
        small_one = small(x[77:79, 5])
        x *= 2.0 ** -24
        x[:, 5] = 0
        x[77:79, 5], w[:, 5] = small_one, w[:, 5] * 2.0 ** 100
    y = ops.lora_linear(x, w, None, A, B, sc)
    f = lambda t: t.double()
    ref, mag = f(x) @ f(w).T + (f(x) @ f(A).T) @ f(B).T, f(x).abs() @ f(w).abs().T + (f(x).abs() @ f(A).abs().T) @ f(B).abs().T
    assert ((f(y) - ref).abs() <= (2 * (3 + 16) + K / 32 + 4) * 2.0 ** -23 * mag + (K + R) * 2.0 ** -149).all()
    assert (f(y) - ref).norm() <= 1e-6 * ref.norm()      # (4e-7 where the fp32 instruction forms the tile)


def test_lora_linear_f32_products_left_out():
    """Single products of numbers whose planes weigh most: what is left out is at most 2^-23 of the product, the last addition cuts off as much again."""
    from katz_amd import ops

    say("lora_linear_f32, products left out")
    d, g = dev(), torch.Generator(device="cuda").manual_seed(8)
    col = torch.cat([1 + 2.0 ** -7 * (1 - 2.0 ** -7 * torch.rand(320, generator=g, device=d)), 1 + torch.rand(320, generator=g, device=d)])
    x, w = torch.zeros(640, 4, device=d), torch.zeros(640, 4, device=d)
    x[:, 1], w[:, 1] = col, col.flip(0)
    y, ref = ops.lora_linear(x, w).double(), x.double() @ w.double().T
    assert ((y - ref).abs() <= 2.0 ** -22 * ref).all(), ((y - ref).abs() / ref).max()


def test_lora_linear_f32_not_finite():
    """Infinities, NaN and sums that overflow come out as full fp32 products give them (a split infinity would be NaN)."""
    from katz_amd import ops

    say("lora_linear_planes_f32, not finite")
    d, g = dev(), torch.Generator(device="cuda").manual_seed(5)
    x, w = torch.randn(200, 640, generator=g, device=d), torch.randn(320, 640, generator=g, device=d) * 0.02
    w[:, 5] = torch.where(torch.arange(320, device=d) % 2 == 0, 0.5, -0.25)          # exact in bf16: its lower planes are zero
    x[3, 5], x[100, 5], x[50, 7], w[7, 9], x[150, 5] = float("inf"), -float("inf"), float("nan"), float("inf"), 3.4e38
    y = ops.lora_linear(x, w)
    ref = (x.double() @ w.double().T).float()
    assert torch.equal(y.isnan(), ref.isnan()) and torch.equal(y.isinf(), ref.isinf()) and torch.equal(y[y.isinf()], ref[ref.isinf()])
    ok = ref.isfinite()
    assert (y[ok] - ref[ok]).abs().le(1e-5 * ref[ok].abs() + 1e-4).all()


@pytest.mark.parametrize("lens,longest,K,N,RP", [
    ([1, 63, 64, 65, 0, 129], 129, 64, 128, 128),         # 64-row blocks, one stage, one column tile
    ([1, 63, 64, 65, 128, 200], 200, 640, 1280, 128),     # ... ten column tiles in ranges of one
    ([127, 128, 129, 1, 300, 700], 4000, 704, 640, 128),  # 128-row blocks (the caller's bound on the rows decides), eleven stages
    ([127, 128, 129, 1, 300, 700], 4000, 1280, 1664, 64),  # ... thirteen column tiles in one range
], ids=str)
def test_sgmv_fused_row_blocks(lens, longest, K, N, RP):
    """Both row blocks of kh_sgmv_fused_bf16 at the edges of segments, ranks on either side of 64, every rank row beyond the padded rank
    poisoned (it must not be read)."""
    from katz_amd import ops

    say("sgmv fused row blocks", lens, longest, K, N, RP)
    d, g = dev(), torch.Generator().manual_seed(K + N)
    ranks = [8, 64, 32, 60, 16, 100 if RP == 128 else 64]
    start = [0]
    for n in lens:
        start.append(start[-1] + n)
    x, base = bf16_round(torch.randn(start[-1], K, generator=g)), bf16_round(torch.randn(start[-1], N, generator=g))
    adapters = [(bf16_round(torch.randn(r, K, generator=g) * 0.05), bf16_round(torch.randn(N, r, generator=g) * 0.05), 0.5 + 0.1 * i) for i, r in enumerate(ranks)]
    a, b = torch.zeros(6, RP, K), torch.zeros(6, N, RP)
    pad = [-(-r // 32) * 32 for r in ranks]
    for i, (A, B, _) in enumerate(adapters):
        a[i, :ranks[i]], b[i, :, :ranks[i]] = A, B
        a[i, pad[i]:] = float("nan")
    i32 = dict(dtype=torch.int32, device=d)
    y = base.to(d, BF)
    ops.sgmv_fused_(y, x.to(d, BF), a.to(d, BF), b.to(d, BF), torch.tensor(start, **i32), torch.arange(6, **i32), torch.tensor(pad, **i32),
                    torch.tensor([s for _, _, s in adapters], device=d), longest)
    assert_close_rel(y, O.sgmv(x, start, list(range(6)), adapters, base), 2e-2, "row blocks")


@pytest.mark.parametrize("N,C,H,W,G", [(1, 32, 1, 1, 4), (2, 320, 7, 9, 32), (1, 1280, 3, 11, 32), (1, 1280, 26, 38, 32), (3, 2560, 5, 13, 32), (1, 4096, 2, 17, 512),
                                       (1, 320, 104, 152, 32)], ids=str)
def test_group_norm_statistics_pass(N, C, H, W, G):
    """kh_group_norm_bf16's statistics: pixel counts below, at and past whole batches of loads, one and two chunks of channels per thread, with
    and without the per-channel term."""
    from katz_amd import ops

    say("group norm statistics", N, C, H, W, G)
    d, g = dev(), torch.Generator().manual_seed(C + H)
    x, gamma, beta = bf16_round(torch.randn(N, C, H, W, generator=g) + 0.5), bf16_round(1 + 0.3 * torch.randn(C, generator=g)), bf16_round(torch.randn(C, generator=g))
    add = bf16_round(torch.randn(N, C, generator=g))
    xd = x.to(d, BF).contiguous(memory_format=torch.channels_last)
    for a in (None, add):
        y = ops.group_norm(xd, G, gamma.to(d, BF), beta.to(d, BF), 1e-5, "silu", add_nc=None if a is None else a.to(d, BF))
        assert_close_rel(y, O.group_norm(x if a is None else x + a[:, :, None, None], G, gamma, beta, 1e-5, "silu"), 2e-2, "group norm")


@pytest.mark.parametrize("host,dtype,ranks", [(False, torch.bfloat16, (64, 32)), (True, torch.float16, (16,)), (False, torch.float32, (4, 8, 100)), (True, torch.bfloat16, (5, 7))],
                         ids=str)
def test_packs_of_a_whole_model_in_two_launches(host, dtype, ranks):
    """set_adapters through kh_lora_pack_bf16 / kh_lora_rescale: every layer's buffers bit for bit against pack_adapters and
    fold_layer_norm, ranks that no 16-byte piece fits included; a change of weights alone keeps the buffers; switching off and
    on again; adapters in host memory (kh_upload_many) and on the GPU."""
    import katz_amd.layers as L
    from katz_amd.lora import fold_norm_into_adapters, pack_adapters
    from katz_amd.unet_2d_condition import UNet2DConditionModel, UNetConfig

    say("pack", host, dtype, ranks)
    d = dev()
    torch.manual_seed(3)
    with torch.device(d):
        unet = UNet2DConditionModel(UNetConfig.tiny())
    unet.to_runtime(d, BF)
    g = torch.Generator().manual_seed(5)
    for i, r in enumerate(ranks):
        for l in unet.lora_linears().values():
            l.add_adapter(f"a{i}", *(t.to(dtype) if host else t.to(d, dtype) for t in (torch.randn(r, l.in_features, generator=g), torch.randn(l.out_features, r, generator=g))))
    names, weights = [f"a{i}" for i in range(len(ranks))], [0.3 + 0.4 * i for i in range(len(ranks))]

    def check():
        for name, l in unet.lora_linears().items():
            ref = pack_adapters(l.adapters, names, l.in_features, l.out_features, BF, d, l.global_scale, geglu_interleave=l.geglu)
            p = l._packed
            assert torch.equal(p.a_cat, ref.a_cat) and torch.equal(p.b_cat, ref.b_cat) and torch.equal(p.col_scale, ref.col_scale), name
            assert p.spans == ref.spans and p.r_used == ref.r_used
            norm = l.fold_norm()
            assert (p.ln is not None) == (norm is not None)
            if norm is not None:
                ap, c1, c2 = fold_norm_into_adapters(p.a_cat, norm.weight, norm.bias)
                assert torch.equal(p.ln[1], ap), name
                assert torch.allclose(p.ln[2], c1, rtol=1e-6, atol=1e-6) and torch.allclose(p.ln[3], c2, rtol=1e-6, atol=1e-6), name

    unet.set_adapters(names, weights)
    check()
    where = {n: l._packed.a_cat.data_ptr() for n, l in unet.lora_linears().items()}
    unet.set_adapters(names, [w + 1 for w in weights])           # scales only: the same buffers
    check()
    assert where == {n: l._packed.a_cat.data_ptr() for n, l in unet.lora_linears().items()}
    unet.scale_lora_layers(0.5)
    check()
    unet.disable_lora()
    assert all(l._packed is None for l in unet.lora_linears().values())
    unet.enable_lora()
    check()


def test_packs_of_the_adapters_before_are_given_back():
    """All packs of an activation share a buffer per kind.  After the next activation, and after unload_lora, nothing that ran
    with them (blocks, single layers, the context projections) keeps it, without a forward in between."""
    import gc
    import weakref

    from katz_amd.unet_2d_condition import UNet2DConditionModel, UNetConfig

    say("packs given back")
    d = dev()
    torch.manual_seed(6)
    cfg = UNetConfig.tiny()
    with torch.device(d):
        unet = UNet2DConditionModel(cfg)
    unet.to_runtime(d, BF)
    linears = list(unet.lora_linears().values())
    for n in "ab":
        for l in linears:
            l.add_adapter(n, torch.randn(16, l.in_features, device=d, dtype=BF) * 0.02, torch.randn(l.out_features, 16, device=d, dtype=BF) * 0.02)
    x = torch.randn(1, 4, 16, 16, device=d, dtype=BF)
    ctx = torch.randn(1, 77, cfg.cross_attention_dim, device=d, dtype=BF)
    pooled = cfg.projection_class_embeddings_input_dim - 6 * cfg.addition_time_embed_dim
    added = dict(text_embeds=torch.randn(1, pooled, device=d, dtype=BF), time_ids=torch.ones(1, 6, device=d))

    def run():
        with torch.no_grad():
            unet(x, 500.0, ctx, added_cond_kwargs=added)
            for l in linears:
                l(torch.zeros(1, l.in_features, device=d, dtype=BF))

    unet.set_adapters(["a"])
    for change in (lambda: unet.set_adapters(["b"]), unet.unload_lora):
        run()
        run()
        packs = [l._packed for l in linears]
        size = sum(p.a_cat.numel() + p.b_cat.numel() for p in packs) * 2
        old = [weakref.ref(t) for p in packs for t in (p, p.a_cat, p.b_cat, p.col_scale)]
        del packs
        gc.collect()
        torch.cuda.synchronize()
        before = torch.cuda.memory_allocated()
        change()
        gc.collect()
        assert sum(r() is not None for r in old) == 0
        grown = torch.cuda.memory_allocated() - before
        assert grown < size // 2, (grown, size)
    run()


def test_one_adapter_with_unlike_dtypes():
    """An adapter whose matrices have two dtypes on some layers: those are packed one by one, the others together; active lists
    and packs agree on every layer."""
    from katz_amd.lora import pack_adapters
    from katz_amd.unet_2d_condition import UNet2DConditionModel, UNetConfig

    say("unlike dtypes")
    d = dev()
    torch.manual_seed(4)
    with torch.device(d):
        unet = UNet2DConditionModel(UNetConfig.tiny())
    unet.to_runtime(d, BF)
    linears = list(unet.lora_linears().values())
    for i, l in enumerate(linears):
        l.add_adapter("a", torch.randn(8, l.in_features, device=d, dtype=BF), torch.randn(l.out_features, 8, device=d, dtype=torch.float32 if i % 3 == 0 else BF))
    unet.set_adapters(["a"], [0.5])
    for l in linears:
        ref = pack_adapters(l.adapters, ["a"], l.in_features, l.out_features, BF, d, l.global_scale, geglu_interleave=l.geglu)
        assert l.active == ["a"] and torch.equal(l._packed.a_cat, ref.a_cat) and torch.equal(l._packed.b_cat, ref.b_cat)
        assert torch.equal(l._packed.col_scale, ref.col_scale)


def test_upload_many_sizes():
    """kh_upload_many: arrays smaller and larger than a staging half, empty gaps, one array, bit for bit."""
    from katz_amd import ops

    say("upload many")
    g = torch.Generator().manual_seed(1)
    for sizes in ([1], [3, 5, 1 << 20, 7], [(9 << 20) + 13, 1, (3 << 20) + 1], [257] * 300):
        src = [torch.randint(0, 256, (n,), generator=g, dtype=torch.uint8) for n in sizes]
        buf, at = ops.upload_many(src, dev())
        torch.cuda.synchronize()
        for t, a in zip(src, at):
            o = a - buf.data_ptr()
            assert torch.equal(buf[o:o + t.numel()].cpu(), t), sizes


@pytest.mark.parametrize("M,N,K,R,r_used", [(1, 640, 64, 0, 0), (31, 640, 128, 32, 16), (64, 1280, 640, 128, 96), (65, 640, 576, 64, 0), (154, 1280, 2048, 0, 0),
                                            (988, 640, 1280, 128, 0), (1976, 640, 2560, 32, 0), (129, 1280, 5120, 64, 32)])
def test_fine_tiles_give_the_bits_of_the_large_ones(M, N, K, R, r_used):
    """Codes 50 .. 53 (64 x 80, 128 x 80, 32 x 128, 64 x 128) add up like the 128 x 128 kernel (16), 54 / 55 (32 x 160, 64 x 160) like the
    64 x 160 one (40): edges of their rows, K shorter than the ring, rank columns that fill no stage."""
    from katz_amd import ops

    say("fine tiles", M, N, K, R, r_used)
    d = dev()
    g = torch.Generator().manual_seed(M + N + K + R)
    rnd = lambda *s: torch.randn(*s, generator=g).to(d, torch.bfloat16)
    x, w, b, res = rnd(M, K), rnd(N, K) * 0.03, rnd(N), rnd(M, N)
    t, bc = (rnd(M, R), rnd(N, R) * 0.05) if R else (None, None)
    if r_used:
        t[:, r_used:] = 0
        bc[:, r_used:] = 0
    for rs in (None, res):
        run = (lambda c: ops.lora_linear_pre(x, w, b, t, bc, residual=rs, tile=c, r_used=r_used)) if R else (lambda c: ops.lora_linear(x, w, b, residual=rs, tile=c))
        for codes, ref in (((50, 51, 52, 53), 16), ((54, 55), 40)):
            if ref == 40 and R % 64:
                continue
            want = run(ref)
            for c in codes:
                assert torch.equal(run(c), want), (c, rs is not None)
    ref = x.double() @ w.double().T + b.double() + (t.double() @ bc.double().T if R else 0)
    y = ops.lora_linear_pre(x, w, b, t, bc, r_used=r_used) if R else ops.lora_linear(x, w, b)
    assert ((y.double() - ref).norm() / ref.norm()).item() < 8e-3


@pytest.mark.parametrize("M,N,K,R,r_used", [(1, 640, 64, 0, 0), (33, 640, 128, 64, 16), (64, 1280, 960, 128, 96), (65, 640, 1024, 64, 0), (154, 1280, 2048, 0, 0),
                                            (31, 1280, 5120, 64, 32), (63, 320, 192, 32, 0)])
def test_narrow_tiles_give_the_bits_of_the_large_ones(M, N, K, R, r_used):
    """Codes 60 .. 62 (32 x 32, 32 x 64, 64 x 64) add up like the 128 x 128 kernel (16), 63 .. 65 like the 64 x 160 one (40): edges of their rows,
    K shorter and longer than their rings of up to 16 stages, rank columns that fill no stage."""
    from katz_amd import ops

    say("narrow tiles", M, N, K, R, r_used)
    d = dev()
    g = torch.Generator().manual_seed(M + N + K + R)
    rnd = lambda *s: torch.randn(*s, generator=g).to(d, torch.bfloat16)
    x, w, b, res = rnd(M, K), rnd(N, K) * 0.03, rnd(N), rnd(M, N)
    t, bc = (rnd(M, R), rnd(N, R) * 0.05) if R else (None, None)
    if r_used:
        t[:, r_used:] = 0
        bc[:, r_used:] = 0
    for rs in (None, res):
        run = (lambda c: ops.lora_linear_pre(x, w, b, t, bc, residual=rs, tile=c, r_used=r_used)) if R else (lambda c: ops.lora_linear(x, w, b, residual=rs, tile=c))
        for codes, ref in (((60, 61, 62), 16), ((63, 64, 65), 40)):
            if ref == 40 and R % 64:
                continue
            want = run(ref)
            for c in codes:
                assert torch.equal(run(c), want), (c, rs is not None)


@pytest.mark.parametrize("M,N,K,R,r_used,stats", [(1, 640, 64, 64, 16, False), (65, 640, 640, 64, 64, True), (300, 640, 640, 64, 64, False), (77, 1280, 2048, 64, 32, False),
                                                  (33, 1280, 128, 128, 96, False), (512, 1280, 5120, 64, 32, False), (1000, 640, 2560, 64, 16, True),
                                                  (200, 640, 2560, 128, 96, False), (700, 1280, 1280, 64, 16, True), (900, 1280, 5120, 64, 16, True)])
def test_few_rows_forms_of_the_dispatch(M, N, K, R, r_used, stats):
    """The form the sizes choose, as one launch and as two: the same bits (results and row statistics), a right result, no wait that ran out."""
    from katz_amd import ops

    say("forms of the dispatch", M, N, K, R, r_used, stats)
    d = dev()
    g = torch.Generator().manual_seed(M + N + K + R)
    rnd = lambda *s: torch.randn(*s, generator=g).to(d, torch.bfloat16)
    x, w, b, res, A, B = rnd(M, K), rnd(N, K) * 0.03, rnd(N), rnd(M, N), rnd(R, K) * 0.05, rnd(N, R) * 0.05
    A[r_used:], B[:, r_used:] = 0, 0
    s = torch.rand(R, generator=g).to(d)
    ops.split_counters_reset(d)
    out = []
    for two in (False, True):
        so = ops.row_stats_buffer(M, d).zero_() if stats else None
        out.append((ops.lora_linear_norm(x, w, b, residual=res, a_cat=A, col_scale=s, b_cat=B, r_used=r_used, two_launches=two, stats_out=so), so))
    ops.check_split_timeouts(d)
    assert torch.equal(out[0][0], out[1][0])
    y = out[0][0].double()
    if stats:
        assert torch.equal(out[0][1], out[1][1])
        got = out[0][1].double().sum(0)
        # fp32 sums of N values of size about 1: N * 2^-24 of their absolute sum at most
        assert torch.allclose(got[:, 0], y.sum(1), atol=N * N * 2.0 ** -24, rtol=0) and torch.allclose(got[:, 1], (y * y).sum(1), rtol=N * 2.0 ** -24)
    ref = x.double() @ w.double().T + b.double() + ((x.double() @ A.double().T) * s.double()) @ B.double().T + res.double()
    assert ((y - ref).norm() / ref.norm()).item() < 8e-3      # bf16 roundings of T and of the result: 2^-9 each


@pytest.mark.parametrize("M,N,K,R,r_used,stats", [(512, 1280, 5120, 128, 96, True), (512, 1280, 5120, 128, 96, False), (154, 1280, 5120, 128, 96, False),
                                                  (700, 640, 2560, 64, 64, True), (450, 1280, 2048, 128, 96, False), (1536, 640, 2560, 32, 16, False), (308, 1280, 2048, 64, 64, False)])
def test_few_rows_with_larger_pieces(M, N, K, R, r_used, stats):
    """Calls on either side of the line between a large tile beside 16 x 16 pieces of the shrink and a smaller one beside 32 x 32 pieces."""
    from katz_amd import ops

    assert ops._lib.load().kh_lora_linear_split_launches(M, N, K, R, 0, r_used // 16 << 16) == 1
    test_few_rows_forms_of_the_dispatch(M, N, K, R, r_used, stats)


@pytest.mark.parametrize("M,N,K,R,r_used,stats", [(1024, 1280, 1280, 64, 64, False), (1100, 640, 128, 64, 16, True), (3952, 640, 640, 64, 16, True), (4096, 640, 640, 64, 64, False),
                                                  (3968, 640, 64, 64, 16, False), (2048, 1280, 5120, 128, 96, True), (1985, 1280, 1280, 128, 96, False), (1537, 1280, 1280, 128, 128, False)])
def test_shrink_beside_128x128_tiles(M, N, K, R, r_used, stats):
    """One round of 128 x 128 tiles with 64 x 64 or 64 x 32 pieces of the shrink beside them, ragged last row blocks, a K loop much shorter than
    the shrink (the tiles wait for T): against the same call with T made in front, and against float64; repeated, on a T that starts as NaNs."""
    from katz_amd import ops

    say("shrink beside 128 x 128 tiles", M, N, K, R, r_used, stats)
    d = dev()
    assert ops._lib.load().kh_lora_linear_split_launches(M, N, K, R, 0, r_used // 16 << 16) == 1
    g = torch.Generator().manual_seed(M + N + K + R)
    rnd = lambda *s: torch.randn(*s, generator=g).to(d, torch.bfloat16)
    x, w, b, res, A, B = rnd(M, K), rnd(N, K) * 0.03, rnd(N), rnd(M, N), rnd(R, K) * 0.05, rnd(N, R) * 0.05
    A[r_used:], B[:, r_used:] = 0, 0
    s = torch.rand(R, generator=g).to(d)

    def run(two):
        ops.split_counters_reset(d)
        junk = torch.full((M, R), float("nan"), device=d, dtype=torch.bfloat16)     # the next scratch of this size
        del junk
        so = ops.row_stats_buffer(M, d).zero_() if stats else None
        return ops.lora_linear_norm(x, w, b, residual=res, a_cat=A, col_scale=s, b_cat=B, r_used=r_used, two_launches=two, stats_out=so), so

    y, so = run(False)
    for _ in range(3):
        again, so2 = run(False)
        assert torch.equal(again, y) and (so is None or torch.equal(so, so2))
    ops.check_split_timeouts(d)
    y2, _ = run(True)
    assert (y != y2).float().mean().item() < 5e-3      # the shrinks add up in different orders: a few last bits of T
    ref = x.double() @ w.double().T + b.double() + ((x.double() @ A.double().T) * s.double()) @ B.double().T + res.double()
    assert ((y.double() - ref).norm() / ref.norm()).item() < 8e-3      # bf16 roundings of T and of the result: 2^-9 each


@pytest.mark.parametrize("M,N,K,R,r_used,kind", [(1024, 1000, 1024, 64, 64, "res"), (2048, 1216, 1280, 128, 96, "res stats"), (1100, 1352, 1280, 128, 96, "fold"), (3000, 968, 1024, 64, 16, ""),
                                                 (1536, 1600, 1280, 64, 64, "stats fold"), (1025, 1288, 2560, 64, 64, "")])
def test_shrink_beside_ragged_columns(M, N, K, R, r_used, kind):
    """Column counts that are no multiple of 128, the shrink inside the launch: the last column tile and the last row block ragged, row statistics and a
    folded LayerNorm, behind a T that starts as NaNs; against two launches and float64."""
    from katz_amd import ops
    from katz_amd.lora import fold_norm_into_adapters, fold_norm_into_weight

    say("shrink beside ragged columns", M, N, K, R, r_used, kind)
    d, kind = dev(), kind.split()
    if "stats" not in kind:
        assert ops._lib.load().kh_lora_linear_split_launches(M, N, K, R, 0, r_used // 16 << 16) == 1
    g = torch.Generator().manual_seed(M + N + K + R)
    rnd = lambda *s: torch.randn(*s, generator=g).to(d, BF)
    x, w, b, A, B = rnd(M, K), rnd(N, K) * 0.03, rnd(N), rnd(R, K) * 0.05, rnd(N, R) * 0.05
    A[r_used:], B[:, r_used:] = 0, 0
    s, res, ln, xn, w0, b0, A0 = torch.rand(R, generator=g).to(d), rnd(M, N) if "res" in kind else None, None, x, w, b, A
    if "fold" in kind:
        gamma, beta = 1 + 0.1 * rnd(K), 0.1 * rnd(K)
        w, c1, c2 = fold_norm_into_weight(w, b, gamma, beta)
        A, ca1, ca2 = fold_norm_into_adapters(A, gamma, beta)
        st = ops.row_stats_buffer(M, d).zero_()
        st[0, :, 0], st[0, :, 1] = x.float().sum(1), (x.float() ** 2).sum(1)
        ln, b = (st, c1, c2, ca1, ca2, 1e-5), None
        xn = torch.nn.functional.layer_norm(x.double(), (K,), gamma.double(), beta.double(), 1e-5)

    def run(two):
        ops.split_counters_reset(d)
        junk = torch.full((M, R), float("nan"), device=d, dtype=BF)     # the next scratch of this size
        del junk
        so = ops.row_stats_buffer(M, d).zero_() if "stats" in kind else None
        return ops.lora_linear_norm(x, w, b, residual=res, a_cat=A, col_scale=s, b_cat=B, r_used=r_used, two_launches=two, ln=ln, stats_out=so), so

    y, so = run(False)
    assert ops.split_counters_last(d)[:-1].gt(0).all()      # (its workgroups have counted themselves in)
    again, so2 = run(False)
    assert torch.equal(again, y) and (so is None or torch.equal(so, so2))
    ops.check_split_timeouts(d)
    y2, _ = run(True)
    assert (y != y2).float().mean().item() < 5e-3           # the shrinks add up in different orders: a few last bits of T
    if so is not None:
        got, yd = so.double().sum(0), y.double()
        # fp32 sums of N values of size about 1: N * 2^-24 of their absolute sum at most
        assert torch.allclose(got[:, 0], yd.sum(1), atol=N * N * 2.0 ** -24, rtol=0) and torch.allclose(got[:, 1], (yd * yd).sum(1), rtol=N * 2.0 ** -24)
    f = lambda t: t.double()
    ref = f(xn) @ f(w0).T + f(b0) + ((f(xn) @ f(A0).T) * f(s)) @ f(B).T + (0 if res is None else f(res))
    assert ((f(y) - ref).norm() / ref.norm()).item() < 8e-3      # bf16 roundings of T, of folded weights and of the result: 2^-9 each


@pytest.mark.parametrize("M,N,K,split,geglu", [(1976, 10240, 1280, False, True), (1793, 10240, 1024, False, True), (3952, 1920, 640, True, False), (1500, 3840, 1280, True, False),
                                               (2900, 1920, 640, False, False), (4993, 1280, 1280, False, False), (4100, 1920, 704, True, False)])
def test_one_round_and_nearly_full_rounds(M, N, K, split, geglu):
    """256 x 128 tiles between one and two rounds of 128 x 128, GEGLU on rounds of 128 x 320 tiles: the bits of the 128 x 128 kernel (code 16)."""
    from katz_amd import ops

    say("one round, nearly full rounds", M, N, K, split, geglu)
    d = dev()
    R = 128
    g = torch.Generator().manual_seed(M + N + K)
    rnd = lambda *s: torch.randn(*s, generator=g).to(d, torch.bfloat16)
    x, w, b, t, bc = rnd(M, K), rnd(N, K) * 0.1, rnd(N), rnd(M, (3 if split else 1) * R), rnd(N, R) * 0.05
    t.view(M, -1, R)[:, :, 96:] = 0
    bc[:, 96:] = 0
    run = lambda c: ops.lora_linear_pre(x, w, b, t, bc, geglu=geglu, tile=c, n_split=N // 3 if split else 0, r_used=96)
    assert torch.equal(run(0), run(16))


@pytest.mark.parametrize("B,T,S,heads", [(1, 1, 1, 1), (2, 33, 63, 3), (1, 130, 64, 2), (3, 5, 65, 2), (1, 300, 127, 1), (2, 64, 128, 2), (1, 127, 129, 3), (1, 256, 192, 2),
                                         (1, 40, 193, 2), (1, 129, 400, 1), (2, 700, 321, 20)])
def test_attention_tiles_of_keys(B, T, S, heads):
    """One, two, three and more tiles of 64 keys, partial last ones, both sizes of workgroups; k and v are column slices of one tensor whose rows behind the
    last key, and columns beside them, are NaN: nothing of those may be used."""
    from katz_amd import ops

    say("attention tiles", B, T, S, heads)
    d = dev()
    g = torch.Generator().manual_seed(B + T + S + heads)
    c = heads * 64
    q = torch.randn(B, T, c, generator=g).to(d, BF)
    kv = torch.full((B, S + 70, 2 * c + 64), float("nan"), device=d, dtype=BF)
    kv[:, :S, :2 * c] = torch.randn(B, S, 2 * c, generator=g).to(d, BF) * 2
    k, v = kv[:, :S, :c], kv[:, :S, c:2 * c]
    o = ops.attention(q, k, v, heads)
    split = lambda t: t.double().reshape(B, -1, heads, 64).transpose(1, 2)
    p = torch.softmax(split(q) @ split(k).transpose(-1, -2).contiguous() / 8, -1)
    ref = (p @ split(v)).transpose(1, 2).reshape(B, T, c)
    # the probabilities and the result are rounded to bf16: 2^-9 each
    assert ((o.double() - ref).norm() / ref.norm()).item() < 6e-3
    assert torch.equal(ops.attention(q, k, v, heads), o)


@pytest.mark.parametrize("M,N,K,R,layers", [(1, 128, 64, 0, 1), (32, 640, 128, 32, 3), (77, 1280, 2048, 64, 5), (96, 640, 640, 128, 2), (128, 128, 1280, 0, 11), (154, 1280, 2048, 128, 4),
                                            (161, 640, 192, 64, 3), (308, 1280, 256, 96, 3), (640, 640, 128, 0, 2), (641, 640, 128, 64, 2)])
def test_grouped_layers_of_few_rows(M, N, K, R, layers):
    """Layers on the same rows in one launch, T a column slice of one wide shrink result with garbage beside it: the bits of the 128 x 128 kernel
    (code 16) layer by layer, whatever the row tiles; rows behind the last stay untouched."""
    import numpy as np
    from katz_amd import ops

    say("grouped layers", M, N, K, R, layers)
    d = dev()
    g = torch.Generator().manual_seed(M + N + K + R)
    rnd = lambda *s: torch.randn(*s, generator=g).to(d, torch.bfloat16)
    x, w, b = rnd(M, K), rnd(layers, N, K) * 0.03, rnd(layers, N)
    t, bc = (rnd(M, layers * R), rnd(layers, N, R) * 0.05) if R else (None, None)
    y = torch.full((layers, M + 1, N), 7.0, device=d, dtype=torch.bfloat16)
    rows = [[w[i].data_ptr(), b[i].data_ptr() if i % 2 == 0 else 0, bc[i].data_ptr() if R else 0, t.data_ptr() + i * R * 2 if R else 0, y[i].data_ptr()] for i in range(layers)]
    ops.lora_linear_grouped(x, ops.upload_table(np.array(rows, dtype=np.int64), d), M, N, K, R, layers * R if R else 8)
    for i in range(layers):
        bias = b[i] if i % 2 == 0 else None
        want = ops.lora_linear_pre(x, w[i], bias, t[:, i * R:(i + 1) * R], bc[i], tile=16) if R else ops.lora_linear(x, w[i], bias, tile=16)
        assert torch.equal(y[i, :M], want), i
        assert bool((y[i, M] == 7.0).all())


@pytest.mark.parametrize("M,N,K,R,r_used", [(1, 160, 64, 0, 0), (129, 320, 128, 64, 48), (127, 640, 640, 128, 96), (4000, 640, 576, 0, 0), (8192, 640, 2560, 128, 80)])
def test_fine_128x160_tiles(M, N, K, R, r_used):
    """Code 59 (128 x 160, two k-slices) against the kernel whose order of sums it keeps (41), bit for bit: partial row blocks, K shorter
    than the ring, rank columns that fill no stage."""
    from katz_amd import ops

    say("fine 128 x 160", M, N, K, R, r_used)
    d = dev()
    g = torch.Generator().manual_seed(M + N + K + R)
    rnd = lambda *s: torch.randn(*s, generator=g).to(d, torch.bfloat16)
    x, w, b, res = rnd(M, K), rnd(N, K) * 0.03, rnd(N), rnd(M, N)
    t, bc = (rnd(M, R), rnd(N, R) * 0.05) if R else (None, None)
    if r_used:
        t[:, r_used:] = 0
        bc[:, r_used:] = 0
    for rs in (None, res):
        run = (lambda c: ops.lora_linear_pre(x, w, b, t, bc, residual=rs, tile=c, r_used=r_used)) if R else (lambda c: ops.lora_linear(x, w, b, residual=rs, tile=c))
        assert torch.equal(run(59), run(41)), rs is not None


@pytest.mark.parametrize("rows,N,K,stats,fold", [(33, 1280, 640, True, True), (512, 1280, 1280, True, False), (700, 640, 640, True, True), (988, 1280, 1280, False, True),
                                                 (1100, 1280, 1280, True, True), (200, 1280, 5120, True, False), (1200, 1280, 5120, True, True)])
def test_fine_tiles_with_folded_norms_do_not_depend_on_the_rows(rows, N, K, stats, fold):
    """The first rows of a call on as many rows as keep the order of the sums (larger tiles) and a call on them alone: the same
    results and row statistics, bit for bit."""
    from katz_amd import ops
    from katz_amd.lora import fold_norm_into_weight

    say("fine tiles, folded norms", rows, N, K, stats, fold)
    d = dev()
    g = torch.Generator().manual_seed(rows + N + K)
    rnd = lambda *s: torch.randn(*s, generator=g).to(d, torch.bfloat16)
    M = 2048 if N == 1280 else 6000
    x, w, b, res = rnd(M, K), rnd(N, K) * 0.03, rnd(N), rnd(M, N)
    wk, c1, c2 = fold_norm_into_weight(w, b, 1 + 0.1 * rnd(K), 0.1 * rnd(K))
    st_in = ops.row_stats_buffer(M, d).zero_()
    st_in[0, :, 0], st_in[0, :, 1] = x.float().sum(1), (x.float() ** 2).sum(1)

    def run(m):
        st = ops.row_stats_buffer(m, d) if stats else None
        ln = (st_in[:, :m].contiguous(), c1, c2, None, None, 1e-5) if fold else None
        y = ops.lora_linear_norm(x[:m], wk if fold else w, None if fold else b, residual=res[:m], ln=ln, stats_out=st)
        return y, st

    (y, st), (yl, stl) = run(rows), run(M)
    assert torch.equal(y, yl[:rows])
    if stats:
        assert torch.equal(st, stl[:, :rows])


@pytest.mark.parametrize("M,N,K,R,r_used,kind", [
    (1, 1280, 64, 32, 16, ""), (33, 640, 640, 32, 32, "res"), (154, 1280, 2048, 128, 96, ""), (129, 1280, 1280, 128, 128, "res fold"),
    (512, 1280, 1280, 64, 32, "res stats"), (31, 1280, 1280, 64, 64, "fold stats"), (988, 1280, 1280, 64, 16, "res stats fold"),
    (988, 1280, 1280, 128, 96, "res stats"), (700, 640, 640, 32, 32, "stats"), (200, 1280, 5120, 64, 16, "res stats"),
    (512, 1280, 5120, 64, 64, "res stats"), (300, 1920, 640, 32, 16, "stack fold"), (65, 3840, 1280, 64, 64, "stack"),
    (988, 1280, 1280, 64, 16, "res"), (512, 3840, 1280, 64, 32, "stack fold"), (300, 10240, 1280, 64, 16, "geglu fold"), (640, 10240, 1280, 64, 64, "geglu")])
def test_few_rows_bring_their_shrink_along(M, N, K, R, r_used, kind):
    """Fine tiles that leave CUs idle: the shrink runs on those, in 16 x 16 or 32 x 32 tiles.  One launch and two give the same bits (results
    and row statistics), columns of T that nobody writes are never read; and the result is right."""
    from katz_amd import ops
    from katz_amd.lora import fold_norm_into_adapters, fold_norm_into_weight, interleave_geglu_rows

    say("in-launch shrink of few rows", M, N, K, R, r_used, kind)
    d = dev()
    kind = kind.split()
    g = torch.Generator().manual_seed(M + N + K + R)
    rnd = lambda *s: torch.randn(*s, generator=g).to(d, torch.bfloat16)
    parts = 3 if "stack" in kind else 1
    split = N // 3 if parts == 3 else 0
    x, w, b = rnd(M, K), rnd(N, K) * 0.03, rnd(N)
    A, B = rnd(parts, R, K) * 0.05, rnd(N, R) * 0.05
    A[:, r_used:], B[:, r_used:] = 0, 0
    A, B0 = A.reshape(parts * R, K), B
    w0, b0, A0 = w, b, A
    geglu = "geglu" in kind
    if geglu:
        w, b, B = interleave_geglu_rows(w), interleave_geglu_rows(b), interleave_geglu_rows(B)
    s = torch.rand(parts * R + 1, generator=g).to(d)[1:]      # (an array that is not 16-byte aligned)
    res = rnd(M, N) if "res" in kind else None
    ln, xn = None, x
    if "fold" in kind:
        gamma, beta = 1 + 0.1 * rnd(K), 0.1 * rnd(K)
        w, c1, c2 = fold_norm_into_weight(w, b, gamma, beta)
        A, ca1, ca2 = fold_norm_into_adapters(A, gamma, beta)
        st = ops.row_stats_buffer(M, d).zero_()
        st[0, :, 0], st[0, :, 1] = x.float().sum(1), (x.float() ** 2).sum(1)
        ln, b = (st, c1, c2, ca1, ca2, 1e-5), None
        xn = torch.nn.functional.layer_norm(x.double(), (K,), gamma.double(), beta.double(), 1e-5)
    if "stats" not in kind:   # (asked for the call without statistics, which has tiles of its own)
        assert ops._lib.load().kh_lora_linear_split_launches(M, N, K, R, split, int(geglu) | r_used // 16 << 16) == 1
    ops.split_counters_reset(d)
    out = []
    for two in (False, True):
        junk = torch.full((M, parts * R), float("nan"), device=d, dtype=torch.bfloat16)     # the next scratch of this size
        del junk
        so = ops.row_stats_buffer(M, d).zero_() if "stats" in kind else None
        y = ops.lora_linear_norm(x, w, b, residual=res, a_cat=A, col_scale=s, b_cat=B, geglu=geglu, n_split=split, r_used=r_used, two_launches=two,
                                 ln=ln, stats_out=so)
        out.append((y, so))
    ops.check_split_timeouts(d)
    assert torch.equal(out[0][0], out[1][0])
    if "stats" in kind:
        assert torch.equal(out[0][1], out[1][1])
    xd, step = xn.double(), N // parts
    ref = torch.cat([xd @ w0[j * step:(j + 1) * step].double().T + b0[j * step:(j + 1) * step].double()
                     + ((xd @ A0[j * R:(j + 1) * R].double().T) * s[j * R:(j + 1) * R].double()) @ B0[j * step:(j + 1) * step].double().T for j in range(parts)], 1)
    if geglu:
        ref = ref[:, :N // 2] * torch.nn.functional.gelu(ref[:, N // 2:])
    if res is not None:
        ref = ref + res.double()
    # bf16 roundings of T, of the folded weights, of the result: 2^-9 each, two of them before a sum
    assert ((out[0][0].double() - ref).norm() / ref.norm()).item() < 8e-3


@pytest.mark.parametrize("M,N,K,R", [(65, 2560, 640, 0), (988, 10240, 1280, 64), (577, 10240, 640, 0), (2048, 5120, 640, 128), (129, 10240, 64, 0)])
def test_fine_geglu_tiles(M, N, K, R):
    """64 x 320 and 128 x 320 tiles with the GEGLU epilogue (codes 57, 58) against the 128 x 128 kernel, bit for bit."""
    from katz_amd import ops

    say("fine geglu", M, N, K, R)
    d = dev()
    g = torch.Generator().manual_seed(M + N + K)
    rnd = lambda *s: torch.randn(*s, generator=g).to(d, torch.bfloat16)
    x, w, b = rnd(M, K), rnd(N, K) * 0.2, rnd(N)
    t, bc = (rnd(M, R), rnd(N, R) * 0.05) if R else (None, None)
    run = (lambda c: ops.lora_linear_pre(x, w, b, t, bc, geglu=True, tile=c)) if R else (lambda c: ops.lora_linear(x, w, b, geglu=True, tile=c))
    want = run(16)
    for c in (57, 58, 0):
        assert torch.equal(run(c), want), c


@pytest.mark.parametrize("K", [64, 640, 1280, 2048, 5120])
@pytest.mark.parametrize("M", [1, 16, 17, 511, 1024])
def test_shrink_of_few_rows_gives_the_bits_of_many(M, K):
    """16 x 16 shrink tiles (up to 256 of them) against the 32 x 32 tiles that run at 2048 rows; with padding columns left out
    against all columns."""
    from katz_amd import ops

    say("few-row shrink", M, K)
    d = dev()
    g = torch.Generator().manual_seed(M + K)
    rnd = lambda *s: torch.randn(*s, generator=g).to(d, BF)
    x, a, cs = rnd(2048, K), rnd(64, K) * 0.02, torch.rand(64, generator=g).to(d)
    want = ops.lora_shrink(x, a, cs)
    assert torch.equal(ops.lora_shrink(x[:M], a, cs), want[:M])
    assert_close_rel(want[:M], ((x[:M].double() @ a.double().t()) * cs.double()).float(), 1e-2)
    a[16:] = 0
    w, b = rnd(3 * 128, K), rnd(3 * 128, 64)
    a3, cs3 = torch.cat([a, a * 2, a * 3]), torch.cat([cs] * 3)
    run = lambda r: ops.lora_linear_split(x[:M], w, None, a3, cs3, b, n_split=128, two_launches=True, r_used=r)
    assert torch.equal(run(16), run(0))


@pytest.mark.parametrize("M,N,K,R,r_used,n_split,entry", [(154, 1280, 2048, 128, 96, 0, "split"), (154, 1280, 2048, 128, 96, 0, "norm"), (2048, 1280, 1280, 64, 64, 0, "norm"),
                                                          (2048, 3840, 1280, 128, 96, 1280, "split"), (8192, 640, 640, 128, 96, 0, "norm"), (2048, 1280, 1280, 64, 64, 0, "xattn")])
def test_bit_24_leaves_the_counters_alone(M, N, K, R, r_used, n_split, entry):
    """With bit 24 of the flags no workgroup counts itself in or waits: counters stay as they are, and the bits are those of two launches."""
    from katz_amd import _lib, ops

    say("bit 24", M, N, K, R, r_used, n_split, entry)
    lib, d, g = _lib.load(), dev(), torch.Generator().manual_seed(M + N)
    parts = N // n_split if n_split else 1
    rnd = lambda *s, std=1.0: (torch.randn(*s, generator=g) * std).to(d, BF)
    x, w, A, B = rnd(M, K), rnd(N, K, std=0.03), rnd(parts, R, K, std=0.05), rnd(N, R, std=0.05)
    A[:, r_used:], B[:, r_used:] = 0, 0
    s, kv = torch.rand(parts * R, generator=g).to(d), rnd(2, 2, 77, N)
    p = lambda t: t.data_ptr()

    def run(flags):
        t, y = torch.zeros(M, parts * R, dtype=BF, device=d), torch.zeros(M, N, dtype=BF, device=d)
        cnt = torch.full(((M + 127) // 128 + 1,), 5, dtype=torch.int32, device=d)
        flags |= r_used // 16 << 16
        if entry == "split":
            rc = lib.kh_lora_linear_split_bf16(p(x), p(w), None, p(A), p(s), p(B), p(t), p(cnt), None, p(y), M, N, K, R, n_split, flags, ops._stream())
        elif entry == "norm":
            rc = lib.kh_lora_linear_norm_bf16(p(x), p(w), None, p(A), p(s), p(B), p(t), p(cnt), None, p(y), None, None, None, None, None, 0.0, None, M, N, K, R,
                                              n_split, flags, ops._stream())
        else:
            rc = lib.kh_lora_linear_xattn_bf16(p(x), p(w), None, p(A), p(s), p(B), p(t), p(cnt), None, None, None, None, None, 0.0, p(kv[0]), p(kv[1]), p(y), M, N, K, R,
                                               M // 2, 77, N, N, N, 77 * N, 77 * N, 0.125, flags, ops._stream())
        assert rc == 0
        torch.cuda.synchronize()
        assert (cnt == 5).all()
        return y

    assert torch.equal(run(1 << 24), run(1 << 8))


@pytest.mark.parametrize("M,N,K,R", [(154, 1280, 2048, 32), (2048, 1280, 1280, 64)])
@pytest.mark.parametrize("reset", [False, True])
def test_captured_layers_see_their_own_inputs(M, N, K, R, reset):
    """A layer in a graph of its own runs as two launches, one behind a reset in the same graph (a model's forward) with its shrink inside; either way
    every replay gives the eager result of the inputs it finds, with eager calls in between."""
    from katz_amd import ops

    say("captured layers", M, N, K, R, reset)
    d, g = dev(), torch.Generator().manual_seed(M)
    rnd = lambda *s, std=1.0: (torch.randn(*s, generator=g) * std).to(d, BF)
    xs, w, A, B = rnd(4, M, K), rnd(N, K, std=0.03), rnd(R, K, std=0.05), rnd(N, R, std=0.5)
    sc, x = torch.ones(R, device=d), torch.zeros(M, K, dtype=BF, device=d)
    call = lambda two=False: ops.lora_linear_split(x, w, None, A, sc, B, two_launches=two)
    assert ops._lib.load().kh_lora_linear_split_launches(M, N, K, R, 0, 0) == 1
    call()
    st = ops._split_counters[0]
    torch.cuda.synchronize()
    graph, before = torch.cuda.CUDAGraph(), (st.graphs.pos, st.eager.pos)
    with torch.cuda.graph(graph):
        if reset:
            ops.split_counters_reset(d)
        outs = [call() for _ in range(3)]
    if reset:
        assert st.graphs.pos == 3 * ((M + 127) // 128 + 1) and st.eager.pos == before[1]
    else:
        assert (st.graphs.pos, st.eager.pos) == before
    for v in xs:
        x.copy_(v)
        want = call(not reset)
        for o in outs:
            o.zero_()
        graph.replay()
        for o in outs:
            assert torch.equal(o, want)
    ops.check_split_timeouts(d)


def test_two_streams_of_few_row_calls():
    """Calls of few rows on two streams at once, one of them resetting: the bits of a quiet device on both."""
    from katz_amd import ops

    say("few rows on two streams")
    d, g = dev(), torch.Generator().manual_seed(4)
    M, N, K, R = 154, 1280, 2048, 64
    rnd = lambda *s, std=1.0: (torch.randn(*s, generator=g) * std).to(d, BF)
    x, w, A, B, sc = rnd(2, M, K), rnd(N, K, std=0.03), rnd(R, K, std=0.05), rnd(N, R, std=0.05), torch.ones(R, device=d)
    call = lambda i: ops.lora_linear_split(x[i], w, None, A, sc, B)
    want = [call(0), call(1)]
    torch.cuda.synchronize()
    streams, got = [torch.cuda.Stream(), torch.cuda.Stream()], ([], [])
    for n in range(60):
        for i, s in enumerate(streams):
            with torch.cuda.stream(s):
                if i and n % 5 == 0:
                    ops.split_counters_reset(d)
                got[i].append(call(i))
    torch.cuda.synchronize()
    for i in (0, 1):
        assert all(torch.equal(y, want[i]) for y in got[i])
    ops.check_split_timeouts(d)


@pytest.mark.parametrize("T,S", [(200, 333), (128, 64), (65, 1), (64, 77), (1, 130), (97, 96)])
def test_attention_waves_of_16_queries(T, S):
    """A few heads run on waves of 16 queries, hundreds on waves of 32, the numbers between on both: the same rows, the same bits, and the oracle's values."""
    from katz_amd import ops
    from oracle import ops as O

    say("attention, waves of 16 and 32 queries", T, S)
    d, g, H = dev(), torch.Generator().manual_seed(T + S), 2
    q, k, v = (torch.randn(3, n, H * 64, generator=g).to(d, BF) for n in (T, S, S))
    k[:, S // 2:] *= 8                                    # the running maximum moves
    o = ops.attention(q, k, v, H)
    assert_close_rel(o, O.attention(q.float().cpu(), k.float().cpu(), v.float().cpu(), H), 2e-2)
    blocks = (T + 127) // 128
    for units in (256 + 12, 256 + 160):                   # 128 queries each: 256 of them whole and the rest halved; all whole
        n = units // (3 * H * blocks) + 1
        more = ops.attention(*(t.repeat(n, 1, 1) for t in (q, k, v)), H)
        assert torch.equal(more.view(n, *o.shape), o.expand(n, *o.shape))


@pytest.mark.parametrize("M,N,K,R", [(1, 320, 64, 0), (95, 640, 128, 32), (160, 640, 192, 64), (161, 320, 64, 128), (193, 960, 320, 64), (385, 640, 1280, 128), (1153, 10240, 640, 64)])
def test_geglu_tiles_of_160_and_192_rows(M, N, K, R):
    """Eight computing waves of 80 or 96 rows x 80 columns: ragged rows, one to many stages, rank columns; the bits of the 128 x 128 kernel (code 16)."""
    from katz_amd import ops

    say("geglu, 160 and 192 rows", M, N, K, R)
    d, g = dev(), torch.Generator().manual_seed(M + N + K)
    rnd = lambda *s: torch.randn(*s, generator=g).to(d, torch.bfloat16)
    x, w, b = rnd(M, K), rnd(N, K) * K ** -0.5, rnd(N)
    t, bc = (rnd(M, R), rnd(N, R) * 0.05) if R else (None, None)
    run = (lambda c: ops.lora_linear_pre(x, w, b, t, bc, geglu=True, tile=c)) if R else (lambda c: ops.lora_linear(x, w, b, geglu=True, tile=c))
    want = run(16)
    for code in (57, 58, 67, 68):
        assert torch.equal(run(code), want), code


@pytest.mark.parametrize("M,N,K,ln", [(1100, 10240, 1280, True), (1300, 10240, 1280, True), (4500, 5120, 640, True), (2500, 5120, 640, False), (2048, 10240, 1280, False)])
def test_geglu_on_the_tiles_whose_rounds_take_least(M, N, K, ln):
    """What the rule chooses between 1024 and 2048 rows and at several rounds: the
    bits of the 128 x 128 kernel where nothing is folded, the oracle's arithmetic otherwise."""
    from katz_amd import ops
    from katz_amd.lora import fold_norm_into_weight

    say("geglu, chosen tiles", M, N, K, ln)
    d, g = dev(), torch.Generator().manual_seed(M + N + K)
    rnd = lambda *s: torch.randn(*s, generator=g).to(d, torch.bfloat16)
    x, w, b = rnd(M, K), rnd(N, K) * K ** -0.5, rnd(N)
    if not ln:
        assert torch.equal(ops.lora_linear(x, w, b, geglu=True), ops.lora_linear(x, w, b, geglu=True, tile=16))
        return
    gamma, beta = 1 + rnd(K) * 0.1, rnd(K) * 0.1
    wp, c1, c2 = fold_norm_into_weight(w, b, gamma, beta)
    part = torch.zeros(ops.LN_SLOTS, M, 2, device=d)
    part[0, :, 0], part[0, :, 1] = x.float().sum(1), (x.float() ** 2).sum(1)
    y = ops.lora_linear_norm(x, wp, None, geglu=True, ln=(part, c1, c2, None, None, 1e-5))
    n = torch.nn.functional.layer_norm(x.double(), (K,), gamma.double(), beta.double(), 1e-5)
    h = (n @ w.double().T + b.double()).view(M, N // 64, 2, 32)
    ref = (h[:, :, 0] * torch.nn.functional.gelu(h[:, :, 1])).reshape(M, N // 2)
    # bf16 roundings of the folded weights, of value and gate and of the product: 2^-9 each
    assert ((y.double() - ref).norm() / ref.norm()).item() < 8e-3


@pytest.mark.parametrize("M,N,K,R,split", [(1, 640, 64, 0, False), (159, 320, 128, 64, False), (193, 960, 320, 32, True), (321, 160, 640, 128, False), (1300, 3840, 1280, 128, True),
                                           (4608, 1920, 640, 0, False), (2304, 1280, 2560, 64, False), (2430, 1280, 2624, 0, False)])
def test_tiles_of_160_columns_and_many_rows(M, N, K, R, split):
    """128 / 160 / 192 x 160 tiles in the order of the 128 x 128 kernel (codes 69 to 71) and 128 x 128 with operand waves (66): its bits, ragged rows, rank columns, one to
    many stages; and those of the tile that is chosen."""
    from katz_amd import ops

    say("160 columns, many rows", M, N, K, R, split)
    d, g, P = dev(), torch.Generator().manual_seed(M + N + K), 3 if split else 1
    rnd = lambda *s: torch.randn(*s, generator=g).to(d, torch.bfloat16)
    x, w, b, res = rnd(M, K), rnd(N, K) * K ** -0.5, rnd(N), rnd(M, N)
    t, bc = (rnd(M, P * R), rnd(N, R) * 0.05) if R else (None, None)
    run = ((lambda c: ops.lora_linear_pre(x, w, b, t, bc, residual=res, tile=c, n_split=N // 3 if split and N // 3 % 128 == 0 else 0)) if R
           else (lambda c: ops.lora_linear(x, w, b, residual=res, tile=c)))
    if split and N // 3 % 128:
        t = t[:, :R].contiguous()
    want = run(16)
    for code in (69, 70, 71) + ((66,) if N % 128 == 0 else ()):
        assert torch.equal(run(code), want), code
    if M > 1024:
        assert torch.equal(run(0), want)


@pytest.mark.parametrize("Nb,H,W,Cin,Cout,stride,res", [(2, 72, 72, 64, 320, 1, False), (2, 96, 97, 64, 320, 1, True), (1, 104, 152, 128, 640, 1, True), (2, 77, 64, 64, 640, 1, False),
                                                        (3, 110, 96, 64, 960, 2, False), (5, 24, 24, 320, 1280, 1, True)])
def test_convolutions_of_many_pixels_on_tiles_by_their_rounds(Nb, H, W, Cin, Cout, stride, res):
    """Pixel counts whose 128 x 128 tiles are neither few nor whole rounds: ragged last rows, stride 2, a residual; against float64, first image
    and last rows, and the same bits twice."""
    from katz_amd import ops

    say("convolution, many pixels", Nb, H, W, Cin, Cout, stride, res)
    d, g = dev(), torch.Generator().manual_seed(H + W + Cin)
    x = torch.randn(Nb, Cin, H, W, generator=g).to(d, torch.bfloat16).contiguous(memory_format=torch.channels_last)
    w = (torch.randn(Cout, Cin, 3, 3, generator=g) * (9 * Cin) ** -0.5).to(d, torch.bfloat16)
    b = torch.randn(Cout, generator=g).to(d, torch.bfloat16)
    ref = torch.nn.functional.conv2d(x.double().cpu()[:1], w.double().cpu(), b.double().cpu(), stride=stride, padding=1)
    r = torch.randn(Nb, *ref.shape[1:], generator=g).to(d, torch.bfloat16).contiguous(memory_format=torch.channels_last) if res else None
    y = ops.conv3x3(x, ops.pack_conv3x3_weight(w), b, stride=stride, residual=r)
    # one rounding of the sum to bf16, one more of the sum with the residual: 2^-9 each
    want = ref if r is None else ref + r[:1].double().cpu()
    assert ((y[:1].double().cpu() - want).norm() / want.norm()).item() < 5e-3
    last = torch.nn.functional.conv2d(x[-1:, :, -8:].double().cpu(), w.double().cpu(), b.double().cpu(), stride=stride, padding=1)[:, :, -2:]
    want = last if r is None else last + r[-1:, :, -2:].double().cpu()
    assert ((y[-1:, :, -2:].double().cpu() - want).norm() / want.norm()).item() < 5e-3
    assert torch.equal(ops.conv3x3(x, ops.pack_conv3x3_weight(w), b, stride=stride, residual=r), y)


@pytest.mark.parametrize("Nb,H,W,Cin,Cout,stride,res", [(2, 72, 72, 64, 320, 1, False), (2, 96, 97, 64, 320, 1, True), (1, 104, 152, 128, 640, 1, True), (3, 110, 96, 64, 960, 2, False),
                                                        (2, 36, 32, 640, 1280, 1, True), (2, 36, 36, 1280, 1280, 1, False), (2, 56, 40, 384, 1280, 1, False)])
def test_convolutions_by_their_rounds_have_the_bits_of_the_large_tiles(Nb, H, W, Cin, Cout, stride, res):
    """Eight columns less leave a width that no other tile divides, so that the 128 x 128 kernel takes the convolution: the columns that both have are the same."""
    from katz_amd import ops

    say("convolution, same bits", Nb, H, W, Cin, Cout, stride, res)
    d, g = dev(), torch.Generator().manual_seed(H + W + Cin)
    x = torch.randn(Nb, Cin, H, W, generator=g).to(d, torch.bfloat16).contiguous(memory_format=torch.channels_last)
    w = (torch.randn(Cout, Cin, 3, 3, generator=g) * (9 * Cin) ** -0.5).to(d, torch.bfloat16)
    b = torch.randn(Cout, generator=g).to(d, torch.bfloat16)
    r = torch.randn(Nb, Cout, (H - 1) // stride + 1, (W - 1) // stride + 1, generator=g).to(d, torch.bfloat16).contiguous(memory_format=torch.channels_last) if res else None
    n = Cout - 8
    y = ops.conv3x3(x, ops.pack_conv3x3_weight(w), b, stride=stride, residual=r)
    y0 = ops.conv3x3(x, ops.pack_conv3x3_weight(w[:n].contiguous()), b[:n].contiguous(), stride=stride,
                     residual=None if r is None else r[:, :n].contiguous(memory_format=torch.channels_last))
    assert torch.equal(y[:, :n], y0)


@pytest.mark.parametrize("lens,longest,K,N,RP", [
    ([1, 0, 65, 200, 64, 70], 200, 576, 1280, 128),                           # ranges of one column tile, nine stages
    ([650] * 4 + [0, 30], 650, 512, 640, 64),                                 # a full ring of stages
    ([1] * 64, 1, 320, 1280, 128),                                            # as many segments as lanes, one row each
    ([3] * 65, 3, 384, 1280, 128),                                            # one more: dealt by the host
    ([700] * 12 + [1024], 1024, 128, 1664, 128),                              # 148 blocks: thirteen column tiles each, beyond the first five
    ([1500] * 16, 4096, 640, 256, 64),                                        # 128-row blocks: less than a round
    ([2100] * 16, 2100, 640, 640, 128),                                       # ... a round and sixteen blocks in ranges
    ([900, 64, 1, 300, 129, 900], 900, 448, 640, 128),                        # adapters of more than 64 in a range more than the others
    ([100, 30, 500], 200000, 128, 256, 128),                                  # a bound on the rows far above them
], ids=str)
def test_sgmv_fused_dealt_by_the_segments(lens, longest, K, N, RP):
    """Every row of every segment and every column range exactly once, whatever the lengths: against the products in float64 with t and
    the delta rounded to bf16 as the kernel rounds them.  Tolerance: a result that falls on the other side of a rounding of t (2^-9 of
    it, over sqrt(rank) terms) or of the delta and the sum (2^-8 each): 2^-7 of the largest."""
    from katz_amd import ops

    say("sgmv fused dealt", lens, longest, K, N, RP)
    d = dev()
    torch.manual_seed(K + N)
    start = [0]
    for n in lens:
        start.append(start[-1] + n)
    ranks = [32, 64, 96, 128] if RP == 128 else [32, 64]
    a, b = torch.randn(len(ranks), RP, K, device=d) * K ** -0.5, torch.randn(len(ranks), N, RP, device=d) * RP ** -0.5
    for i, r in enumerate(ranks):
        a[i, r:], b[i, :, r:] = 0, 0
    a, b = a.to(BF), b.to(BF)
    x, base = torch.randn(start[-1], K, device=d).to(BF), torch.randn(start[-1], N, device=d).to(BF)
    who = [i % len(ranks) if i % 7 != 3 else -1 for i in range(len(lens))]     # (every seventh segment has no adapter)
    who = [w if n > 0 else 10 ** 6 for w, n in zip(who, lens)]                 # (an empty one may name any)
    scale = [0.5 + 0.25 * i for i in range(len(ranks))]
    i32 = dict(dtype=torch.int32, device=d)
    y = base.clone()
    ops.sgmv_fused_(y, x, a, b, torch.tensor(start, **i32), torch.tensor(who, **i32), torch.tensor(ranks, **i32), torch.tensor(scale, device=d), longest)
    for i, w in enumerate(who):
        s, e = start[i], start[i + 1]
        if s == e or w < 0:
            assert torch.equal(y[s:e], base[s:e])
            continue
        t = (x[s:e].double() @ a[w].double().T).to(BF).double()
        delta = (scale[w] * (t @ b[w].double().T)).to(BF).double()
        ref = (base[s:e].double() + delta).to(BF).double()
        err = (y[s:e].double() - ref).abs().max()
        assert err <= 2 ** -7 * ref.abs().max(), (i, w, float(err))


@pytest.mark.parametrize("layers,lens,longest", [
    (53, [64, 1, 30, 0, 63, 40], 64),                      # 64-row blocks, four a layer (an empty segment, one without an adapter): 212, less than a round
    (62, [64, 1, 30, 63, 40], 64),                         # ... 248
    (53, [64, 1, 30, 7, 63, 40], 64),                      # five a layer, 265: a round and nine of the last two layers in ranges
    (37, [130, 1, 77, 128, 300, 0, 129], 300),             # 128-row blocks, nine a layer, 333: a layer cut by the end of the round
    (101, [200, 0, 129, 31], 200),                         # three a layer, 303
], ids=str)
def test_sgmv_fused_grouped_in_whole_rounds_and_ranges(layers, lens, longest):
    """Many layers dealt on the device, whole rounds of the CUs and what is left: each layer has the bits of its own launch, and rows without an adapter stay."""
    from katz_amd import ops

    say("sgmv fused grouped, rounds", layers, lens, longest)
    d, K, N, RP = dev(), 128, 384, 128
    torch.manual_seed(layers)
    start = [0]
    for n in lens:
        start.append(start[-1] + n)
    ranks = [32, 128, 64, 96]
    who = [i % 4 for i in range(len(lens))]
    who[2] = -1
    i32 = dict(dtype=torch.int32, device=d)
    rows, ss, sa = start[-1], torch.tensor(start, **i32), torch.tensor(who, **i32)
    rk, sc = torch.tensor(ranks, **i32), torch.tensor([0.5, 0.75, 1.0, 1.25], device=d)
    x = torch.randn(rows, K, device=d).to(BF)
    a, b = (torch.randn(layers, 4, RP, K, device=d) * K ** -0.5).to(BF), (torch.randn(layers, 4, N, RP, device=d) * RP ** -0.5).to(BF)
    for i, r in enumerate(ranks):
        a[:, i, r:], b[:, i, :, r:] = 0, 0
    base = torch.randn(layers, rows, N, device=d).to(BF)
    y, want = base.clone(), base.clone()
    ops.sgmv_fused_grouped_(list(y), x, list(a), list(b), ss, sa, rk, sc, longest)
    for l in range(layers):
        ops.sgmv_fused_(want[l], x, a[l], b[l], ss, sa, rk, sc, longest)
        assert torch.equal(y[l], want[l]), l
    assert torch.equal(y[:, start[2]:start[3]], base[:, start[2]:start[3]])
    assert not torch.equal(y[-1, start[-2]:], base[-1, start[-2]:])


def test_sgmv_fused_of_many_heavy_blocks():
    """More row blocks of adapters of more than 64 than half of a signed word's upper half counts (64 x 516 of 128 rows): every row once.  Tolerance as
    above."""
    from katz_amd import ops

    n, rows, K, N = 64, 66000, 64, 128
    say("sgmv fused, many heavy blocks", n, rows, K, N)
    d = dev()
    torch.manual_seed(1)
    a, b = (torch.randn(2, 128, K, device=d) * K ** -0.5).to(BF), (torch.randn(2, N, 128, device=d) * 128 ** -0.5).to(BF)
    a[1, 96:], b[1, :, 96:] = 0, 0
    x, base = torch.randn(n * rows, K, device=d, dtype=BF), torch.randn(n * rows, N, device=d, dtype=BF)
    i32 = dict(dtype=torch.int32, device=d)
    y = base.clone()
    ops.sgmv_fused_(y, x, a, b, torch.arange(n + 1, **i32) * rows, torch.arange(n, **i32) % 2, torch.tensor([128, 96], **i32), torch.tensor([0.5, 0.75], device=d), rows)
    for i in range(n):
        s = slice(i * rows, (i + 1) * rows)
        t = (x[s].double() @ a[i % 2].double().T).to(BF).double()
        ref = (base[s].double() + ((0.5 + 0.25 * (i % 2)) * (t @ b[i % 2].double().T)).to(BF).double()).to(BF).double()
        assert (y[s].double() - ref).abs().max() <= 2 ** -7 * ref.abs().max(), i


@pytest.mark.parametrize("shapes,r,dt", [
    ([(128, 128)], 128, torch.float16),                                        # two turns of 64 ranks
    ([(130, 260), (1, 8), (257, 1284)], 96, torch.bfloat16),                   # a turn and a half, pieces of 8 bytes, ragged tiles
    ([(64, 7), (129, 131)], 20, torch.float16),                                # element by element, rank in no whole piece
    ([(8, 16)] * 70 + [(200, 136)] + [(16, 8)] * 70, 8, torch.bfloat16),       # more layers than lanes
], ids=lambda v: str(v)[:40])
def test_merge_tiles(shapes, r, dt):
    """kh_lora_merge_grouped_bf16 at the edges of tiles, of turns over the rank and of the search for a tile's layer, against float64: one
    rounding to bf16 (2^-9 relative) and r products in fp32 (2^-24 r of the sum of their sizes)."""
    from katz_amd import ops

    say("merge tiles", shapes[:3], r, dt)
    d = dev()
    torch.manual_seed(r)
    w = [torch.randn(n, k, device=d).to(BF) for n, k in shapes]
    up = [torch.randn(n, r, device=d).to(dt) for n, _ in shapes]
    down = [torch.randn(r, k, device=d).to(dt) for _, k in shapes]
    scales = [0.5 + i / len(shapes) for i in range(len(shapes))]
    was = [x.clone() for x in w]
    ops.lora_merge_grouped(w, up, down, scale=0.3, layer_scales=scales)
    for x, x0, u, v, s in zip(w, was, up, down, scales):
        ref = x0.double() + 0.3 * s * (u.double() @ v.double())
        size = x0.double().abs() + 0.3 * s * (u.double().abs() @ v.double().abs())
        assert ((x.double() - ref).abs() <= ref.abs() * 2 ** -8 + size * (r + 4) * 2 ** -23).all(), tuple(x.shape)
