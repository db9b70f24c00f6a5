"""Parity of the product UNet path (katz_amd.* modules on the HIP kernels) against the CPU oracle.

Tolerances: one BasicTransformerBlock -- elementwise 2e-2 relative (bf16 per-layer
contract); whole UNet step -- cosine >= 0.999 against the fp32 oracle on identical bf16-rounded weights
and inputs (BASELINE config 3's gate), plus a loose elementwise bound.
"""
import pytest
import torch

from helpers import assert_close_rel, bf16_round, cosine, katz_lora_state_dict, random_lora, round_module_to_bf16_
from oracle import blocks as OB
from oracle.unet_sdxl import UNet2DConditionModel as OracleUNet, UNetConfig as OracleCfg

pytestmark = pytest.mark.gpu
BF = torch.bfloat16


def say(*a):
    print(*a, flush=True)


def _product_from_oracle(oracle, cfg_name):
    import katz_amd.layers as L
    from katz_amd.unet_2d_condition import UNet2DConditionModel, UNetConfig

    L.SKIP_INIT = True
    try:
        prod = UNet2DConditionModel(getattr(UNetConfig, cfg_name)())
    finally:
        L.SKIP_INIT = False
    prod.load_state_dict(oracle.state_dict(), strict=True)
    return prod.to_runtime("cuda:0", BF)


def _inputs(cfg, B, H, S, seed=1):
    g = torch.Generator().manual_seed(seed)
    x = bf16_round(torch.randn(B, 4, H, H, generator=g))
    ctx = bf16_round(torch.randn(B, S, cfg.cross_attention_dim, generator=g))
    pooled = cfg.projection_class_embeddings_input_dim - 6 * cfg.addition_time_embed_dim
    added = dict(text_embeds=bf16_round(torch.randn(B, pooled, generator=g)),
                 time_ids=torch.tensor([[H * 8, H * 8, 0, 0, H * 8, H * 8]] * B, dtype=torch.float32))
    return x, ctx, added


def _to_dev(added):
    return {k: v.to("cuda:0") for k, v in added.items()}


def test_basic_transformer_block_config2():
    """hidden [2,1024,1280], context [2,77,2048], 20 heads x 64, one rank-64 LoRA
    (alpha 64, scale 1.0) on to_q/to_k/to_v/to_out.0 of both attentions and on ff GEGLU proj / out;
    weights ~N(0,0.02)."""
    from katz_amd.layers import BasicTransformerBlock

    say("config2 block")
    torch.manual_seed(0)
    ob = OB.BasicTransformerBlock(1280, 20, 64, 2048)
    with torch.no_grad():
        for n, p in ob.named_parameters():
            if p.dim() == 2:
                p.normal_(0, 0.02)
            elif "norm" in n:
                p.copy_(torch.ones_like(p) if n.endswith("weight") else torch.zeros_like(p))
            else:
                p.normal_(0, 0.02)
    round_module_to_bf16_(ob)
    lin = {n: m for n, m in ob.named_modules() if isinstance(m, OB.OracleLoRALinear)}
    assert len(lin) == 10
    lora = random_lora(lin, 64, seed=0)
    for n, (d, u) in lora.items():
        lin[n].add_adapter("a", d, u, alpha=64.0, weight=1.0)
        lin[n].active = ["a"]
    pb = BasicTransformerBlock(1280, 20, 64, 2048)
    pb.load_state_dict(ob.state_dict(), strict=True)
    pb = pb.to("cuda:0", BF).eval()
    plin = {n: m for n, m in pb.named_modules() if hasattr(m, "add_adapter")}
    for n, (d, u) in lora.items():
        plin[n].add_adapter("a", d, u, alpha=64.0)
        plin[n].set_active(["a"], [1.0])
    g = torch.Generator().manual_seed(1)
    h = bf16_round(torch.randn(2, 1024, 1280, generator=g))
    ctx = bf16_round(torch.randn(2, 77, 2048, generator=g))
    with torch.no_grad():
        ref = ob(h, ctx)
        ref_nolora_delta = None
        got = pb(h.to("cuda:0", BF), ctx.to("cuda:0", BF))
        torch.cuda.synchronize()
        assert_close_rel(got, ref, 2e-2, "BasicTransformerBlock")
        # per-layer check on the first LoRA linear with the block's real input
        n1 = torch.nn.functional.layer_norm(h, (1280,), ob.norm1.weight, ob.norm1.bias, 1e-5)
        n1b = bf16_round(n1)
        q_ref = ob.attn1.to_q(n1b)
        q_got = pb.attn1.to_q(n1b.to("cuda:0", BF))
        assert_close_rel(q_got, q_ref, 2e-2, "attn1.to_q")
        # the adapter matters: disabling it changes the output
        for m in plin.values():
            m.set_active([])
        got0 = pb(h.to("cuda:0", BF), ctx.to("cuda:0", BF))
        assert (got0.float() - got.float()).abs().max().item() > 1e-3


@pytest.fixture(scope="module")
def tiny_pair():
    torch.manual_seed(0)
    cfg = OracleCfg.tiny()
    oracle = round_module_to_bf16_(OracleUNet(cfg).eval())
    prod = _product_from_oracle(oracle, "tiny")
    return cfg, oracle, prod


def _tiny_residuals(oracle, x, ctx, added, seed):
    with torch.no_grad():
        skips, mid = oracle(x, 500, ctx, added, return_skips=True)
    g = torch.Generator().manual_seed(seed)
    down = [bf16_round(torch.randn(s.shape, generator=g) * 0.1) for s in skips]
    midr = bf16_round(torch.randn(mid.shape, generator=g) * 0.1)
    return down, midr


def test_tiny_unet_step_with_lora_and_controlnet(tiny_pair):
    cfg, oracle, prod = tiny_pair
    say("tiny unet")
    B, H = 2, 32
    x, ctx, added = _inputs(cfg, B, H, 77)
    down, midr = _tiny_residuals(oracle, x, ctx, added, 3)
    l1 = random_lora(oracle.lora_linears(), 16, seed=10, std=0.05)
    l2 = random_lora(oracle.lora_linears(), 8, seed=11, std=0.05)
    oracle.add_adapter("one", l1); oracle.add_adapter("two", l2)
    prod.load_lora_into_unet(katz_lora_state_dict(l1), adapter_name="one")
    prod.load_lora_into_unet(katz_lora_state_dict(l2), adapter_name="two")
    dev = "cuda:0"
    run_p = lambda **kw: prod(x.to(dev), torch.tensor([500.0], device=dev), ctx.to(dev), added_cond_kwargs=_to_dev(added), **kw).sample
    with torch.no_grad():
        # (a) adapters on, ControlNet residuals on
        oracle.set_adapters(["one", "two"], [0.8, 0.6]); prod.set_adapters(["one", "two"], [0.8, 0.6])
        ref = oracle(x, 500, ctx, added, down, midr)
        got = run_p(down_block_additional_residuals=[d.to(dev) for d in down], mid_block_additional_residual=midr.to(dev))
        torch.cuda.synchronize()
        assert got.shape == ref.shape
        assert cosine(got, ref) >= 0.999, cosine(got, ref)
        assert_close_rel(got, ref, 6e-2, "tiny unet, lora + controlnet")
        # (b) scale 0 == adapters disabled == no LoRA (cosine: scale 0 still runs the rank columns, with zero weights,
        # through bf16 roundings that the adapter-free launch does not have)
        prod.set_adapters(["one", "two"], [0.0, 0.0])
        g0 = run_p()
        prod.disable_lora()
        g1 = run_p()
        assert torch.equal(g1, run_p()), "the step is bit-reproducible: every convolution runs on the katz_hip kernel"
        prod.enable_lora()
        assert cosine(g0, g1) >= 0.9995
        oracle.set_adapters([], [])
        assert cosine(g0, oracle(x, 500, ctx, added)) >= 0.999
        # (c) zero residuals == no residuals
        gz = run_p(down_block_additional_residuals=[torch.zeros_like(d).to(dev) for d in down],
                   mid_block_additional_residual=torch.zeros_like(midr).to(dev))
        assert cosine(gz, g1) >= 0.9995
        # (d) two ControlNets are averaged
        oracle.set_adapters(["one"], [1.0]); prod.set_adapters(["one"], [1.0])
        down2 = [bf16_round(d * -0.5 + 0.01) for d in down]; mid2 = bf16_round(midr * 2.0)
        ref2 = oracle(x, 500, ctx, added, [(a + b) / 2 for a, b in zip(down, down2)], (midr + mid2) / 2)
        got2 = run_p(down_block_additional_residuals=[[d.to(dev) for d in down], [d.to(dev) for d in down2]],
                     mid_block_additional_residual=[midr.to(dev), mid2.to(dev)])
        assert cosine(got2, ref2) >= 0.999
        # (e) fused == unfused (diffusers-hf/tests/lora/utils.py:654-698), cross_attention_kwargs scale
        unf = run_p(cross_attention_kwargs={"scale": 0.5})
        prod.fuse_lora(0.5)
        fus = run_p()
        prod.unfuse_lora()
        assert cosine(unf, fus) >= 0.999
        oracle.set_adapters(["one"], [0.5])
        assert cosine(unf, oracle(x, 500, ctx, added)) >= 0.999
        # (f) unload restores the adapter-free model
        prod.unload_lora()
        assert cosine(run_p(), g1) >= 0.9995
        for m in oracle.lora_linears().values():
            m.adapters.clear(); m.active = []


def test_time_emb_projector_matches_per_resnet_linear(tiny_pair):
    """The batched time_emb_proj of all resnets equals each resnet's own nn.Linear on the same input (bf16 rounding of
    one GEMM against another), is handed out once per run, and follows in-place weight changes."""
    from katz_amd.layers import ResnetBlock2D

    cfg, oracle, prod = tiny_pair
    say("time emb projector")
    resnets = [m for m in prod.modules() if isinstance(m, ResnetBlock2D)]
    assert len(resnets) >= 6 and len({r.time_emb_proj.out_features for r in resnets}) >= 2
    g = torch.Generator().manual_seed(3)
    temb = torch.randn(2, resnets[0].time_emb_proj.in_features, generator=g).to("cuda:0", BF)
    with torch.no_grad():
        prod._temb_proj.run(temb)
        for r in resnets:
            assert r.temb_proj is not None and r.temb_proj.is_contiguous()
            assert_close_rel(r.temb_proj, r.time_emb_proj(temb).float().cpu(), 2e-2, "batched time_emb_proj")
        first = resnets[0]
        before = first.temb_proj.clone()
        first.time_emb_proj.weight.mul_(2.0)                     # in place: same storage, new version
        prod._temb_proj.run(temb)
        assert_close_rel(first.temb_proj, first.time_emb_proj(temb).float().cpu(), 2e-2, "after an in-place change")
        assert not torch.equal(first.temb_proj, before)
        first.time_emb_proj.weight.mul_(0.5)
        for r in resnets:
            r.temb_proj = None


def test_tiny_unet_graph_replay_matches_eager(tiny_pair):
    """The captured step reproduces eager results over several replays with fresh inputs."""
    from katz_amd.graph import GraphedUNetStep

    cfg, oracle, prod = tiny_pair
    say("tiny unet graph")
    dev = "cuda:0"
    B, H = 2, 32
    x, ctx, added = _inputs(cfg, B, H, 77, seed=5)
    down, midr = _tiny_residuals(oracle, x, ctx, added, 6)
    l1 = random_lora(oracle.lora_linears(), 16, seed=12, std=0.05)
    prod.load_lora_into_unet(katz_lora_state_dict(l1), adapter_name="g")
    prod.set_adapters(["g"], [0.7])
    with torch.no_grad():
        step = GraphedUNetStep(prod, x.to(dev), torch.tensor([500.0], device=dev), ctx.to(dev), _to_dev(added),
                               [d.to(dev) for d in down], midr.to(dev))
        for i in range(3):
            xi, ctxi, _ = _inputs(cfg, B, H, 77, seed=20 + i)
            t = torch.tensor([100.0 + 300 * i], device=dev)
            eager = prod(xi.to(dev), t, ctxi.to(dev), added_cond_kwargs=_to_dev(added),
                         down_block_additional_residuals=[d.to(dev) for d in down],
                         mid_block_additional_residual=midr.to(dev)).sample.clone()
            torch.cuda.synchronize()
            out = step(sample=xi.to(dev), timestep=t, encoder_hidden_states=ctxi.to(dev)).clone()
            torch.cuda.synchronize()
            assert cosine(out, eager) >= 0.9995, f"replay {i} differs from eager: cosine {cosine(out, eager)}"
            assert_close_rel(out, eager, 6e-2, f"graph replay {i}")
    prod.unload_lora()


def test_capture_of_a_forward_that_scales_its_adapters(tiny_pair):
    """cross_attention_kwargs={"scale": s} changes every layer's scales at the start of the forward and changes them back at its
    end; a caller may capture that.  Every replay against the eager forward, with eager work of another scale and other host
    and device allocations in between."""
    cfg, oracle, prod = tiny_pair
    say("capture of a scaled forward")
    dev = torch.device("cuda:0")
    x, ctx, added = _inputs(cfg, 2, 32, 77, seed=8)
    x, ctx, added = x.to(dev), ctx.to(dev), _to_dev(added)
    t = torch.tensor([300.0], device=dev)
    prod.load_lora_into_unet(katz_lora_state_dict(random_lora(oracle.lora_linears(), 16, seed=13, std=0.05)), adapter_name="s")
    prod.set_adapters(["s"], [0.7])
    run = lambda s: prod(x, t, ctx, added_cond_kwargs=added, cross_attention_kwargs={"scale": s}).sample
    with torch.no_grad():
        side = torch.cuda.Stream()
        side.wait_stream(torch.cuda.current_stream())
        with torch.cuda.stream(side):
            for _ in range(2):
                run(0.5)
        torch.cuda.current_stream().wait_stream(side)
        torch.cuda.synchronize()
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph):
            out = run(0.5)
        want, other = run(0.5).clone(), run(2.0).clone()
        assert not torch.equal(want, other)
        for i in range(3):
            junk = [torch.full((n,), 0x5a, dtype=torch.uint8).pin_memory() for n in (512, 4096, 1 << 16)]   # where a table might have been
            out.zero_()
            graph.replay()
            torch.cuda.synchronize()
            assert cosine(out, want) >= 0.9995 and cosine(out, want) > cosine(out, other), i
            assert_close_rel(out, want, 6e-2, f"replay {i}")
            assert torch.equal(run(2.0), other)      # the replay has put the scales back
            del junk
    prod.unload_lora()


def test_sdxl_unet_step_config3():
    """BASELINE config 3 at full size: latent [2,4,128,128], t=500, context [2,77,2048], pooled [2,1280],
    time_ids [2,6]; LoRA rank 64 scale 0.8 + rank 32 scale 0.6 on all 722 linears; 9+1 ControlNet
    residuals ~N(0,0.1).  Gate: latent cosine >= 0.999 vs the fp32 oracle."""
    say("sdxl unet config3: building oracle")
    torch.manual_seed(0)
    cfg = OracleCfg.sdxl()
    oracle = round_module_to_bf16_(OracleUNet(cfg).eval())
    prod = _product_from_oracle(oracle, "sdxl")
    x, ctx, added = _inputs(cfg, 2, 128, 77)
    l1 = random_lora(oracle.lora_linears(), 64, seed=10)
    l2 = random_lora(oracle.lora_linears(), 32, seed=11)
    oracle.add_adapter("r64", l1); oracle.add_adapter("r32", l2)
    oracle.set_adapters(["r64", "r32"], [0.8, 0.6])
    prod.load_lora_into_unet(katz_lora_state_dict(l1), adapter_name="r64")
    prod.load_lora_into_unet(katz_lora_state_dict(l2), adapter_name="r32")
    prod.set_adapters(["r64", "r32"], [0.8, 0.6])
    dev = "cuda:0"
    with torch.no_grad():
        say("sdxl unet config3: oracle skips")
        skips, mid = oracle(x, 500, ctx, added, return_skips=True)
        g = torch.Generator().manual_seed(3)
        down = [bf16_round(torch.randn(s.shape, generator=g) * 0.1) for s in skips]
        midr = bf16_round(torch.randn(mid.shape, generator=g) * 0.1)
        exp_shapes = [(320, 128)] * 3 + [(320, 64), (640, 64), (640, 64), (640, 32), (1280, 32), (1280, 32)]
        assert [(s.shape[1], s.shape[2]) for s in skips] == exp_shapes and mid.shape == (2, 1280, 32, 32)
        del skips, mid
        say("sdxl unet config3: product")
        got = prod(x.to(dev), torch.tensor([500.0], device=dev), ctx.to(dev), added_cond_kwargs=_to_dev(added),
                   down_block_additional_residuals=[d.to(dev) for d in down],
                   mid_block_additional_residual=midr.to(dev)).sample.float().cpu()
        # the same step as a HIP graph (what the benchmark times): replays are bit-identical to each other and to the
        # eager step (every replay clears the in-launch shrinks' counters with its first node)
        from katz_amd.graph import GraphedUNetStep
        say("sdxl unet config3: graph replays")
        step = GraphedUNetStep(prod, x.to(dev), torch.tensor([500.0], device=dev), ctx.to(dev), _to_dev(added),
                               [d.to(dev) for d in down], midr.to(dev))
        r1 = step().float().cpu()
        r2 = step().float().cpu()
        r3 = step().float().cpu()
        torch.cuda.synchronize()
        assert torch.equal(r1, r2) and torch.equal(r1, r3) and torch.equal(r1, got), "graph replay differs from the eager step"
        del step
        say("sdxl unet config3: oracle full step")
        ref = oracle(x, 500, ctx, added, down, midr)
    c = cosine(got, ref)
    say("sdxl unet config3 cosine", c)
    assert got.shape == (2, 4, 128, 128)
    assert c >= 0.999, c


def test_patch_on_lora_merge_matches_unmerged_adapter():
    """Katz's merge path (W += up @ down * alpha/rank as GEMMs on the GPU, keys through the key-match sidecar)
    gives the weights of the oracle's closed form and the same step output as running the adapter unmerged."""
    import katz_amd.layers as L
    from katz_amd.shm_adapters import patch_on_lora
    from katz_amd.unet_2d_condition import UNet2DConditionModel, UNetConfig
    from oracle import ops as O

    say("patch_on_lora")
    torch.manual_seed(0)
    cfg = OracleCfg.tiny()
    oracle = round_module_to_bf16_(OracleUNet(cfg).eval())
    merged = _product_from_oracle(oracle, "tiny")
    plain = _product_from_oracle(oracle, "tiny")
    lora = random_lora(oracle.lora_linears(), 16, seed=21, std=0.05)
    sd = {k: v.to(torch.float16) for k, v in katz_lora_state_dict(lora).items()}   # what the shared memory holds
    key_match = {}
    for mod in lora:
        head, _, leaf = mod.rpartition(".")
        base = (f"unet.{head}.processor.{leaf}_lora" if leaf in ("to_q", "to_k", "to_v")
                else f"unet.{mod[:-len('.to_out.0')]}.processor.to_out_lora" if mod.endswith(".to_out.0") else f"unet.{mod}.lora")
        key_match[mod + ".weight"] = {"lora_down_key": base + ".down.weight", "lora_up_key": base + ".up.weight"}
    scale = 0.75
    n = patch_on_lora(merged, sd, key_match, scale=scale)
    assert n == len(lora)
    torch.cuda.synchronize()
    params = dict(merged.named_parameters())
    for mod in list(lora)[:8] + list(lora)[-4:]:
        down, up = lora[mod]
        w0 = dict(oracle.named_parameters())[mod + ".weight"]
        ref = O.lora_merged_weight(w0, [(down.half().float(), up.half().float(), scale)])
        assert_close_rel(params[mod + ".weight"], ref, 1e-2, f"merged weight {mod}")
    # same step, adapter unmerged at the same effective scale (alpha = scale * rank)
    plain.load_lora_into_unet({k: v.float() for k, v in sd.items()},
                              network_alphas={k + ".alpha": scale * 16 for k in sd if k.endswith(".down.weight")},
                              adapter_name="a")
    plain.set_adapters(["a"], [1.0])
    x, ctx, added = _inputs(cfg, 2, 32, 77)
    dev = "cuda:0"
    with torch.no_grad():
        a = merged(x.to(dev), torch.tensor([500.0], device=dev), ctx.to(dev), added_cond_kwargs=_to_dev(added)).sample
        b = plain(x.to(dev), torch.tensor([500.0], device=dev), ctx.to(dev), added_cond_kwargs=_to_dev(added)).sample
    assert cosine(a, b) >= 0.999, cosine(a, b)


def test_reference_env_flags(monkeypatch):
    """ENABLE_FUSED_GEGLU=1 switches the feed-forward to the reference's fused arithmetic (tanh GELU, gelu.cuh:29-42),
    ENABLE_CUDA_GRAPH=1 makes forward() replay a captured graph (unet_2d_condition.py:511, :2030-2050); the other two
    switches are recorded.  Compared with the oracle evaluated with the tanh form, and with the eager product."""
    import katz_amd.layers as L
    from katz_amd.unet_2d_condition import UNet2DConditionModel, UNetConfig
    from oracle import ops as OO

    say("env flags")
    for k in ("ENABLE_FUSED_GEGLU", "ENABLE_CUDA_GRAPH", "ENABLE_FUSED_NORM_SILU", "ENABLE_CHANNELS_LAST"):
        monkeypatch.setenv(k, "1")
    torch.manual_seed(0)
    cfg = OracleCfg.tiny()
    oracle = round_module_to_bf16_(OracleUNet(cfg).eval())
    L.SKIP_INIT = True
    try:
        prod = UNet2DConditionModel(UNetConfig.tiny())
    finally:
        L.SKIP_INIT = False
    assert prod.enable_cuda_graph and prod.enable_fused_norm_silu and prod.enable_channels_last
    assert all(m.enable_fused_geglu for m in prod.modules() if isinstance(m, L.GEGLU))
    prod.load_state_dict(oracle.state_dict(), strict=True)
    prod = prod.to_runtime("cuda:0", BF)
    x, ctx, added = _inputs(cfg, 2, 16, 7, seed=9)
    down, midr = _tiny_residuals(oracle, x, ctx, added, 4)
    dev = "cuda:0"
    kw = dict(added_cond_kwargs=_to_dev(added), down_block_additional_residuals=[d.to(dev) for d in down],
              mid_block_additional_residual=midr.to(dev))
    t = torch.tensor([500.0], device=dev)
    with torch.no_grad():
        monkeypatch.setattr(OO, "geglu", lambda proj, approximate="none": OO.gelu(proj.chunk(2, -1)[1], "tanh") * proj.chunk(2, -1)[0])
        ref_tanh = oracle(x, 500, ctx, added, down, midr)
        monkeypatch.undo()
        ref_erf = oracle(x, 500, ctx, added, down, midr)
        got = prod(x.to(dev), t, ctx.to(dev), **kw).sample.clone()            # builds the graph, replays it
        got2 = prod(x.to(dev), t, ctx.to(dev), **kw).sample.clone()           # replay only
        assert len(prod._graphs) == 1
        prod.enable_cuda_graph = False
        eager = prod(x.to(dev), t, ctx.to(dev), **kw).sample
        torch.cuda.synchronize()
    assert torch.equal(got, got2) and torch.equal(got, eager)
    assert cosine(got, ref_tanh) >= 0.999 and cosine(got, ref_erf) >= 0.999   # the two forms differ below bf16 noise here
    # so that the tanh form is what ran is checked on the calls: every feed-forward went through kh_geglu_bf16(tanh)
    from katz_amd import ops
    seen = []
    real = ops.geglu
    monkeypatch.setattr(ops, "geglu", lambda proj, approximate="none": (seen.append(approximate), real(proj, approximate))[1])
    with torch.no_grad():
        prod(x.to(dev), t, ctx.to(dev), **kw)
    n_ff = sum(1 for m in prod.modules() if isinstance(m, L.GEGLU))
    assert seen == ["tanh"] * n_ff and n_ff > 0


def test_kohya_named_adapter_to_step(tiny_pair):
    """A kohya / SGM-named adapter file (lora_unet_input_blocks_4_1_..., .lora_down / .lora_up / .alpha) goes through
    convert_kohya_lora_to_diffusers -> load_lora_into_unet -> one step, against the oracle given the same matrices
    under their module names (conversion: diffusers-hf/src/diffusers/loaders/lora_conversion_utils.py:126-287)."""
    import re

    from katz_amd.lora_conversion import convert_kohya_lora_to_diffusers

    cfg, oracle, prod = tiny_pair
    say("kohya adapter -> step")

    def kohya_name(mod):   # diffusers module path -> sd-scripts name with SGM block numbering (layers_per_block = 2)
        m = re.match(r"(down_blocks|up_blocks)\.(\d+)\.attentions\.(\d+)\.(.+)", mod)
        if m:
            b, l = int(m.group(2)), int(m.group(3))
            head = f"input_blocks_{b * 3 + l + 1}_1" if m.group(1) == "down_blocks" else f"output_blocks_{b * 3 + l}_1"
            rest = m.group(4)
        else:
            head, rest = "middle_block_1", re.match(r"mid_block\.attentions\.0\.(.+)", mod).group(1)
        return "lora_unet_" + head + "_" + rest.replace(".", "_")

    rank, alpha = 16, 8.0
    lora = random_lora(oracle.lora_linears(), rank, seed=21, std=0.05)
    file_sd = {}
    for mod, (down, up) in lora.items():
        kn = kohya_name(mod)
        file_sd[kn + ".lora_down.weight"] = down
        file_sd[kn + ".lora_up.weight"] = up
        file_sd[kn + ".alpha"] = torch.tensor(alpha)
    unet_sd, alphas, rest = convert_kohya_lora_to_diffusers(file_sd)
    assert not rest and len(unet_sd) == 2 * len(lora) and len(alphas) == len(lora)
    prod.load_lora_into_unet(unet_sd, network_alphas=alphas, adapter_name="kohya")
    oracle.add_adapter("kohya", lora, alpha=alpha)
    x, ctx, added = _inputs(cfg, 2, 16, 77, seed=12)
    dev = "cuda:0"
    try:
        with torch.no_grad():
            oracle.set_adapters(["kohya"], [0.9]); prod.set_adapters(["kohya"], [0.9])
            ref = oracle(x, 500, ctx, added)
            got = prod(x.to(dev), torch.tensor([500.0], device=dev), ctx.to(dev), added_cond_kwargs=_to_dev(added)).sample
            prod.set_adapters([], [])
            base = prod(x.to(dev), torch.tensor([500.0], device=dev), ctx.to(dev), added_cond_kwargs=_to_dev(added)).sample
            torch.cuda.synchronize()
        assert cosine(got, ref) >= 0.999, cosine(got, ref)
        assert_close_rel(got, ref, 6e-2, "kohya adapter step")
        assert (got.float() - base.float()).abs().max().item() > 1e-2     # the adapter (alpha / rank = 0.5) matters
        lin = prod.lora_linears()
        assert all(m.adapters["kohya"].alpha == alpha for m in lin.values())
    finally:
        prod.unload_lora()
        for m in oracle.lora_linears().values():
            m.adapters.clear(); m.active = []
