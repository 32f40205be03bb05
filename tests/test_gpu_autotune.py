"""Plans chosen by measurement (kernels/autotune.py): every candidate plan of a product gives the product, and a runner
that times its plans before it records a step gives the plain implementation's logits."""
import numpy as np
import pytest
import torch

import helpers as H
import plain_model as pm

pytestmark = pytest.mark.gpu


def _operands(rows, n, k, seed, bias):
    g = torch.Generator().manual_seed(seed)
    d = torch.device("cuda:0")
    x = (torch.randn((rows, k), generator=g) * 0.7).bfloat16()
    w = (torch.randn((n, k), generator=g) * 0.05).bfloat16()
    b = (torch.randn((n,), generator=g) * 0.3).bfloat16() if bias else None
    return x.to(d), w.to(d), (b.to(d) if bias else None), x.double(), w.double(), (b.double() if bias else None)


@pytest.mark.parametrize("rows,n,k", [(8, 520, 1024), (24, 1536, 4480), (40, 776, 1096), (64, 1544, 2304),
                                      (128, 1536, 2048), (200, 3584, 4096)])
def test_every_candidate_plan_gives_the_product(rows, n, k):
    from ginfer_amd.kernels import ops
    from ginfer_amd.parts import linear as L
    tried = set()
    for bias in (False, True):
        for f32 in (False, True):
            for parts_ok in (False, True):
                x, w, b, xd, wd, bd = _operands(rows, n, k, rows + n + k, bias)
                ref = xd @ wd.T + (bd if bias else 0.0)
                skinny_ok = ops.gemm_skinny_supported(x, w)
                tiles_ok = ops.gemm_tiles_supported(x, w)
                key = ("linear", rows, n, k, bias, f32, parts_ok, skinny_ok, tiles_ok)
                for plan in L.linear_candidates(key):
                    y = L.run_linear_plan(plan, x, w, b, torch.float32 if f32 else None)
                    parts = plan[-1] if (plan[0] == "library" or plan[2] > 1) and plan[-1] > 1 else 1
                    if parts > 1 or plan[0] == "tiles":
                        assert y.shape == (parts, rows, n) and y.dtype == torch.float32, (plan, y.shape)
                        y = y.double().sum(0)
                    else:
                        assert y.shape == (rows, n) and y.dtype == (torch.float32 if f32 else torch.bfloat16), (plan, y.dtype)
                    err = float((y.double().cpu() - ref).abs().max() / ref.abs().max())
                    # bfloat16 results carry one rounding (2^-9 of the value); 32-bit ones only the order of the sums
                    tol = 1e-5 if (f32 or parts > 1 or plan[0] == "tiles") else 4e-3
                    assert err <= tol, "plan %s of %s: %.3g" % (plan, key, err)
                    tried.add(plan)
    assert ("library", 1) in tried and len(tried) >= 3, tried
    print("plans tried for rows %d, %d x %d: %s" % (rows, n, k, sorted(tried)))


@pytest.mark.parametrize("rows,n,k", [(8, 520, 1024), (40, 776, 1096), (64, 2304, 1536), (256, 1536, 1024)])
def test_every_candidate_plan_of_the_gated_product(rows, n, k):
    from ginfer_amd.kernels import ops
    from ginfer_amd.parts import linear as L
    x, w, _, xd, wd, _ = _operands(rows, 2 * n, k, rows + n, False)
    gate, up = xd @ wd[:n].T, xd @ wd[n:].T
    # the plain statement rounds the products to bfloat16 before the activation only where the kernels do; compare in
    # 64-bit with a tolerance of two roundings
    ref = gate * torch.sigmoid(gate) * up
    bounds = (1.5, 1.702, 1.0)
    bounded = torch.clamp(gate, max=bounds[0])
    bounded = bounded * torch.sigmoid(bounds[1] * bounded) * (torch.clamp(up, -bounds[0], bounds[0]) + bounds[2])
    for limits, want in ((None, ref), (bounds, bounded)):
        key = ("gated", rows, 2 * n, k, ops.gemm_skinny_supported(x, w), limits is None and L._transposable(x, w),
               ops.gemm_tiles_supported(x, w), limits)
        plans = L.gated_candidates(key)
        assert len(plans) >= 2 and (("tiles",) in plans) == (k % 64 == 0)
        for plan in plans:
            y = L.run_gated_plan(plan, x, w, limits)
            assert y.shape == (rows, n) and y.dtype == torch.bfloat16
            err = float((y.double().cpu() - want).abs().max() / want.abs().max())
            assert err <= 1.2e-2, "plan %s: %.3g" % (plan, err)


@pytest.mark.parametrize("rows,nh,nkv,hd,K", [(17, 4, 2, 64, 1536), (64, 4, 2, 48, 1152), (100, 3, 1, 128, 640)])
@pytest.mark.parametrize("bias", [False, True])
def test_every_way_of_the_projection(rows, nh, nkv, hd, K, bias):
    """Rotated q and the pages of k and v by every way that the tuner may keep, and that it times them all."""
    from ginfer_amd.kernels import autotune, ops
    from ginfer_amd.parts import attention
    x, w, b, xd, wd, bd = _operands(rows, (nh + 2 * nkv) * hd, K, rows + K, bias)
    with autotune.collecting() as keys:
        way, key = attention.projection_choice(x, w, bias, nh, nkv, hd, hd)
        assert way[0] == "spread" and autotune.choose(key, (w, b)) is None
    ways = attention.projection_candidates(key)
    assert [way[0] for way in ways] == {17: ["spread", "fused", "library"], 64: ["spread", "parts", "library"], 100: ["spread", "library"]}[rows]
    table = autotune.Table()
    assert autotune.tune(keys, x.device, table) == 1 and table[key] in ways and set(table.report[0][2]) == set(ways)
    positions = torch.arange(rows, dtype=torch.int32, device=x.device)
    angle = torch.arange(rows)[:, None] * (1e4 ** (-2.0 * torch.arange(hd // 2) / hd))[None]
    cos, sin = torch.cos(angle).float(), torch.sin(angle).float()
    full = (xd @ wd.T + (bd if bias else 0.0)).view(rows, nh + 2 * nkv, hd)
    lo, hi, c, s = full[..., :hd // 2], full[..., hd // 2:], cos.double()[:, None], sin.double()[:, None]
    turned = torch.cat([lo * c - hi * s, lo * s + hi * c], dim=-1)
    for way in ways:
        kp = torch.zeros((-(-rows // 8), nkv, 8, hd), dtype=torch.bfloat16, device=x.device)
        vp = torch.zeros((-(-rows // 8), nkv, hd, 8), dtype=torch.bfloat16, device=x.device)
        qkv = attention.project(way, x, w, b, positions, cos.to(x.device), sin.to(x.device), torch.arange(rows, device=x.device), kp, vp,
                                nh, nkv, hd, True)
        got = dict(q=qkv[:, :nh * hd].reshape(rows, nh, hd), k=kp.permute(0, 2, 1, 3).reshape(-1, nkv, hd)[:rows],
                   v=vp.permute(0, 3, 1, 2).reshape(-1, nkv, hd)[:rows])
        for name, want in (("q", turned[:, :nh]), ("k", turned[:, nh:nh + nkv]), ("v", full[:, nh + nkv:])):
            err = float((got[name].double().cpu() - want).abs().max() / want.abs().max())
            assert err <= 1e-2, "%s by %s: %.3g" % (name, way, err)       # the library's rows are rounded before the rotation and after it


def test_a_runner_that_times_its_plans(tmp_path):
    """Two layers of a 7B shape, 40 requests decoding side by side: the runner times the plans of its products when it
    records the step (the rules' plan for this down projection is not the fastest one), and logits stay the plain
    implementation's, in the recorded step's replays and in eager steps of the same size."""
    from ginfer_amd import ModelRunner
    from ginfer_amd.kernels import autotune
    V, live = 1500, 40
    cfg = dict(architectures=["Qwen2ForCausalLM"], num_hidden_layers=2, hidden_size=3584, num_attention_heads=28,
               num_key_value_heads=4, intermediate_size=18944, vocab_size=V, rope_theta=1e6, rms_norm_eps=1e-6,
               tie_word_embeddings=False, max_position_embeddings=512)
    folder = H.make_model_folder(tmp_path / "wide", cfg, 4, "float32")
    prompt, decoded = 18, 6
    reqs = {"r%d" % i: H.random_tokens(prompt + decoded, V, 100 + i) for i in range(live)}
    steps = [dict(entries=[dict(id=rid, tokens=ids[:prompt], want=[prompt - 1])], end=[]) for rid, ids in reqs.items()]
    for k in range(decoded):
        steps.append(dict(entries=[dict(id=rid, tokens=[ids[prompt + k]], want=[0]) for rid, ids in reqs.items()],
                          end=list(reqs) if k == decoded - 1 else []))
    runner = ModelRunner(folder, dtype="bfloat16", page_size=16, num_pages=2 * live, max_requests=live, autotune=True)
    got = H.run_steps(runner, steps)
    runner.cache.check()
    assert runner.counts["autotuned_keys"] >= 3 and runner.counts["replayed_decode"] >= 3, runner.counts
    assert isinstance(runner.plans, autotune.Table)
    keys = [key for key, _, _ in runner.plans.report]
    assert ("linear", 48, 3584, 18944, False, False, True, True, True) in keys, keys
    for key, plan, times in runner.plans.report:
        print("%s -> %s (%d plans, %.1f to %.1f us)" % (key, plan, len(times), min(times.values()), max(times.values())))
        assert runner.plans[key] == plan and plan in times
    # the plans are the runner's own: a runner built without autotune runs by the rules, whatever this one has measured
    plain = ModelRunner(folder, dtype="bfloat16", page_size=16, num_pages=2 * live, max_requests=live)
    assert plain.plans is None and not autotune.active()
    del plain
    # a second runner that is handed the first one's table finds the plans and times nothing (its first steps already run
    # by them, where the first runner's ran by the rules: the two agree up to rounding only)
    again = ModelRunner(folder, dtype="bfloat16", page_size=16, num_pages=2 * live, max_requests=live, autotune=runner.plans)
    got2 = H.run_steps(again, steps)
    assert again.counts.get("autotuned_keys", 0) == 0 and again.plans is runner.plans
    # the kept plans in recorded steps and launched kernel by kernel: the same bits (prompts run kernel by kernel in both)
    pair = [ModelRunner(folder, dtype="bfloat16", page_size=16, num_pages=2 * live, max_requests=live, autotune=runner.plans,
                        use_graphs=g, graph_mixed_steps=False) for g in (True, False)]
    a, b = (H.run_steps(r, steps) for r in pair)
    assert pair[0].counts["replayed_decode"] >= 3 and pair[1].counts["replayed_decode"] == 0
    for k in a:
        assert np.array_equal(a[k], b[k]), "replayed and launched steps differ at %s" % (k,)
    pcfg, w = pm.read_config(folder), pm.read_weights(folder, torch.float32)
    for rid in list(reqs)[:3] + list(reqs)[-2:]:
        ref = pm.forward(pcfg, w, reqs[rid]).numpy()
        for p in range(prompt - 1, prompt + decoded):
            for g in (got, got2, a):
                err = np.abs(g[(rid, p)] - ref[p]).max() / np.abs(ref).max()
                assert err <= H.TOL["bfloat16"], "request %s position %d: %.3g" % (rid, p, err)
