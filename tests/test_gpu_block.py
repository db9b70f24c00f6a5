"""A transformer block as one library call against the same block through its modules, bit for bit."""
import pytest
import torch

pytestmark = pytest.mark.gpu


def dev():
    return torch.device("cuda:0")


def say(*a):
    print("[block]", *a, flush=True)


def make(width, ranks, depth=2):
    from katz_amd.layers import LoRALinear, Transformer2DModel

    torch.manual_seed(width + len(ranks))
    m = Transformer2DModel(width // 64, 64, width, depth, 2048).to(dev(), torch.bfloat16).eval()
    for l in m.modules():
        if isinstance(l, LoRALinear):
            for i, r in enumerate(ranks):
                l.add_adapter(f"a{i}", torch.randn(r, l.in_features, device=dev(), dtype=torch.bfloat16) * 0.02,
                              torch.randn(l.out_features, r, device=dev(), dtype=torch.bfloat16) * 0.02)
            l.set_active([f"a{i}" for i in range(len(ranks))], [0.8, 0.6][:len(ranks)])
    return m


def both(monkeypatch, f):
    """f's result with the library call (which must have been taken) and without."""
    from katz_amd import block, layers

    taken, real = [], block.run

    def watch(*a):
        y = real(*a)
        taken.append(y is not None)
        return y

    with monkeypatch.context() as mp:
        mp.setattr(block, "run", watch)
        got = f()
        mp.setattr(layers, "BLOCK_CALL", False)
        want = f()
    assert torch.equal(got, want)
    return taken


@pytest.mark.parametrize("width,B,H,W,ranks", [(1280, 2, 16, 16, ()), (1280, 1, 26, 38, (16,)), (640, 2, 19, 13, (64, 32)), (640, 1, 1, 1, (128,)),
                                               (1280, 2, 32, 32, (8,))])
@torch.no_grad()
def test_block_call_gives_the_modules_bits(monkeypatch, width, B, H, W, ranks):
    say("block call", width, B, H, W, ranks)
    m = make(width, ranks)
    blk = m.transformer_blocks[0]
    ctx = torch.randn(B, 77, 2048, device=dev(), dtype=torch.bfloat16)
    h = torch.randn(B, H * W, width, device=dev(), dtype=torch.bfloat16)
    x = torch.randn(B, width, H, W, device=dev(), dtype=torch.bfloat16).contiguous(memory_format=torch.channels_last)
    assert both(monkeypatch, lambda: blk(h, ctx)) == [True]                  # its norms as launches of their own
    assert both(monkeypatch, lambda: m(x, ctx)) == [True, True]              # norms folded, statistics from block to block
    wide = torch.randn(B, 77, 3 * width, device=dev(), dtype=torch.bfloat16)
    for a in (b.attn2 for b in m.transformer_blocks):
        a.ctx_kv = (ctx, wide[..., :width], wide[..., 2 * width:])           # projected elsewhere, strided
    assert both(monkeypatch, lambda: m(x, ctx)) == [True, True]


@torch.no_grad()
def test_block_call_follows_every_change(monkeypatch):
    from katz_amd.layers import LoRALinear

    m = make(640, (32,), depth=1)
    blk = m.transformer_blocks[0]
    ctx = torch.randn(1, 77, 2048, device=dev(), dtype=torch.bfloat16)
    x = torch.randn(1, 640, 8, 8, device=dev(), dtype=torch.bfloat16).contiguous(memory_format=torch.channels_last)
    run = lambda: m(x, ctx)
    linears = [l for l in m.modules() if isinstance(l, LoRALinear)]
    seen = [run()]

    def changed(taken=True):
        assert both(monkeypatch, run) == [taken]
        seen.append(run())
        assert not torch.equal(seen[-1], seen[-2])

    blk.ff.net[2].weight.mul_(1.5)                                           # in place
    changed()
    blk.attn1.to_k.weight = torch.nn.Parameter(blk.attn1.to_k.weight * 0.5, requires_grad=False)
    changed()
    blk.norm2.bias.add_(0.5)
    changed()
    for l in linears:                                                        # a scale: the packs stay
        l.set_active(["a0"], [3.0])
    changed()
    for l in linears:
        l.set_active([])
    changed()
    blk.attn1.to_out[0] = LoRALinear(640, 640).to(dev(), torch.bfloat16)     # another module
    changed()
    hook = blk.attn2.to_q.register_forward_hook(lambda mod, args, out: out * 2)
    x_h = torch.randn(1, 64, 640, device=dev(), dtype=torch.bfloat16)
    assert both(monkeypatch, lambda: blk(x_h, ctx)) == [False]               # hooks are called: through the modules
    hook.remove()
    assert both(monkeypatch, run) == [True]


@pytest.mark.parametrize("rows,K,N,geglu,ranks,residual", [(1, 640, 640, False, (8,), True), (154, 2048, 1280, False, (64, 32), False), (300, 1280, 10240, True, (16,), False),
                                                           (77, 40, 72, False, (), True), (154, 2048, 640, False, (32,), "no bias"), (65, 1280, 1280, False, (128, 64), True)])
@torch.no_grad()
def test_single_linear_call(monkeypatch, rows, K, N, geglu, ranks, residual):
    from katz_amd import layers

    say("single linear", rows, K, N, geglu, ranks, residual)
    bf = dict(device=dev(), dtype=torch.bfloat16)
    l = layers.LoRALinear(K, N, geglu=geglu, bias=residual != "no bias").to(dev(), torch.bfloat16)
    for i, r in enumerate(ranks):
        l.add_adapter(f"a{i}", torch.randn(r, K, **bf) * 0.02, torch.randn(N, r, **bf) * 0.02)
    x, res = torch.randn(2, rows, K, **bf), torch.randn(2, rows, N, **bf) if residual is True else None

    def check():
        y = l(x, residual=res)
        with monkeypatch.context() as mp:
            mp.setattr(layers, "BLOCK_CALL", False)
            assert torch.equal(y, l(x, residual=res))
        return y

    seen = [check()]
    for change in (lambda: l.set_active([f"a{i}" for i in range(len(ranks))]), lambda: l.weight.mul_(2.0), lambda: l.bias is not None and l.bias.add_(1.0), lambda: l.set_active([])):
        change()
        seen.append(check())
    assert not torch.equal(seen[1], seen[2]) and (l.bias is None or not torch.equal(seen[2], seen[3]))
    with pytest.raises(ValueError, match="does not match x"):
        l(x[..., :-8].contiguous())


def _inputs(width, B=1, side=8):
    bf = dict(device=dev(), dtype=torch.bfloat16)
    return torch.randn(B, width, side, side, **bf).contiguous(memory_format=torch.channels_last), torch.randn(B, 77, 2048, **bf)


@torch.no_grad()
def test_block_call_steps_aside_for_another_processor(monkeypatch):
    from katz_amd.layers import KatzAttnProcessor

    say("another processor")
    m = make(640, (16,), depth=1)
    a, (x, ctx) = m.transformer_blocks[0].attn2, _inputs(640)
    plain = m(x, ctx)
    calls = []

    class Doubles(KatzAttnProcessor):
        def __call__(self, attn, h, **kw):
            calls.append(1)
            return super().__call__(attn, h, **kw) * 2

    old = a.get_processor()
    for proc in (Doubles(), KatzAttnProcessor()):
        a.set_processor(proc)
        assert both(monkeypatch, lambda: m(x, ctx)) == [type(proc) is KatzAttnProcessor]
    assert len(calls) == 2 and torch.equal(m(x, ctx), plain)
    a.set_processor(Doubles())
    assert not torch.equal(m(x, ctx), plain)
    a.set_processor(old)


@torch.no_grad()
def test_calls_follow_the_adapter_mode(monkeypatch):
    """LORA_MODE "fused" runs the adapters inside each tile (no library call for a whole block or linear); back to "split"."""
    from katz_amd import layers

    say("adapter mode")
    m = make(640, (32,), depth=1)
    x, ctx = _inputs(640)
    l, rows = m.transformer_blocks[0].attn1.to_out[0], torch.randn(77, 640, device=dev(), dtype=torch.bfloat16)
    split, one = m(x, ctx), l(rows)
    with monkeypatch.context() as mp:
        mp.setattr(layers, "LORA_MODE", "fused")
        assert both(mp, lambda: m(x, ctx)) == [False]
        fused = l(rows)
        with mp.context() as inner:
            inner.setattr(layers, "BLOCK_CALL", False)
            assert torch.equal(fused, l(rows))
    # the same sums, T rounded to bf16 in both: bf16 of the result and of T (4e-3 each), in two orders
    assert ((fused.float() - one.float()).norm() / one.float().norm()).item() < 1e-2
    assert both(monkeypatch, lambda: m(x, ctx)) == [True]
    assert torch.equal(m(x, ctx), split) and torch.equal(l(rows), one)


@torch.no_grad()
def test_a_copy_of_a_model_has_calls_of_its_own(monkeypatch):
    import copy

    from katz_amd.layers import LoRALinear

    say("copies")
    m = make(640, (16,), depth=1)
    x, ctx = _inputs(640)
    first = m(x, ctx)
    twin = copy.deepcopy(m)
    assert both(monkeypatch, lambda: twin(x, ctx)) == [True] and torch.equal(twin(x, ctx), first)
    for l in twin.modules():
        if isinstance(l, LoRALinear):
            l.set_active([])
    twin.transformer_blocks[0].ff.net[2].weight.mul_(1.5)
    assert both(monkeypatch, lambda: twin(x, ctx)) == [True] and not torch.equal(twin(x, ctx), first)
    assert both(monkeypatch, lambda: m(x, ctx)) == [True] and torch.equal(m(x, ctx), first)
    changed = twin(x, ctx)
    del m
    assert torch.equal(twin(x, ctx), changed)


@torch.no_grad()
def test_calls_on_a_second_stream():
    say("second stream")
    m = make(640, (64, 32), depth=2)
    x, ctx = _inputs(640, 2, 24)
    rows = torch.randn(154, 2048, device=dev(), dtype=torch.bfloat16)
    l = m.transformer_blocks[0].attn2.to_k
    want, one = m(x, ctx), l(rows)
    torch.cuda.synchronize()
    side = torch.cuda.Stream()
    with torch.cuda.stream(side):
        y = [m(x * s, ctx) for s in (2.0, 1.0)][1]    # inputs made on that stream: a launch elsewhere would run ahead of them
        z = l(rows * 2.0 * 0.5)
    side.synchronize()
    assert torch.equal(y, want) and torch.equal(z, one)


@torch.no_grad()
def test_two_threads_with_a_model_and_a_stream_each():
    """Forwards and changes of adapters of one model beside another's: each gives what it gives alone.  (Without the
    transformer's GroupNorm, whose scratch belongs to one stream per device.)"""
    import threading

    from katz_amd.layers import LoRALinear, RowStats

    say("two threads")
    models = [make(640, (16,), depth=1), make(640, (64, 32), depth=2)]
    inputs = [_inputs(640), _inputs(640, 2)]

    def work(i):
        m, (x, ctx) = models[i], inputs[i]
        linears = [l for l in m.modules() if isinstance(l, LoRALinear)]
        names, out = [f"a{k}" for k in range(i + 1)], []
        rows = x.permute(0, 2, 3, 1).reshape(x.shape[0], -1, 640)

        def forward():
            stats = RowStats(rows.shape[0] * rows.shape[1], dev())
            h = m.proj_in(rows, stats_out=stats)
            for blk in m.transformer_blocks:
                h = blk(h, ctx, stats=stats)
            return m.proj_out(h, residual=rows)

        with torch.no_grad():
            for k in range(6):
                for l in linears:
                    l.set_active(names if k % 2 == 0 else names[:1], [1.0 + k] * (i + 1))
                out += [forward() for _ in range(3)]
        torch.cuda.current_stream().synchronize()
        return out

    alone = [work(0), work(1)]
    torch.cuda.synchronize()
    got, errors = [None, None], []

    def thread(i):
        try:
            with torch.cuda.stream(torch.cuda.Stream()):
                got[i] = work(i)
        except BaseException as e:
            errors.append(e)

    ts = [threading.Thread(target=thread, args=(i,)) for i in range(2)]
    for t in ts:
        t.start()
    for t in ts:
        t.join(60)
    assert not errors and all(not t.is_alive() for t in ts)
    for a, g in zip(alone, got):
        assert len(a) == len(g) and all(torch.equal(u, v) for u, v in zip(a, g))
