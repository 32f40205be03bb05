"""Decisions that are taken on the host from sizes alone: how a product is split over workgroups."""
import pytest
import torch

from ginfer_amd.parts import linear as L


def test_parts_divide_the_steps_of_k_and_leave_every_wavefront_work():
    for rows in (1, 8, 16, 17, 64):
        for n in (88, 896, 1536, 3584, 8192):
            for k in (64, 520, 1536, 3584, 8960, 18944, 29568):
                nt, parts = L._split_plan(rows, n, k)
                steps = -(-k // 64)
                assert nt in (1, 4) and 1 <= parts <= L.TUNING.max_split_k_parts
                assert parts == 1 or (steps % parts == 0 or k < L.TUNING.split_k_from) and parts * 8 <= max(steps, 8)
                assert nt == 1 or rows > 16


def test_measured_shapes_keep_their_plans():
    """The sizes the plans were measured at (1.5B and 7B shapes) keep what was found best."""
    assert L._split_plan(64, 1536, 8960) == (4, 10)
    assert L._split_plan(8, 1536, 8960) == (1, 5)
    assert L._split_plan(64, 1536, 1536) == (1, 2)
    assert L._split_plan(64, 3584, 18944) == (4, 4)
    assert L._split_plan(64, 3584, 3584) == (4, 4)
    assert L._library_split(256, 1536, 8960) == 5 and L._library_split(64, 1536, 8960) == 1
    assert L._library_split(256, 17920, 1536) == 1
    # the rows of prompt portions: four pieces up to 2,048 rows, one product beyond
    assert L._library_split(512, 1536, 8960) == 4 and L._library_split(2048, 1536, 8960) == 4
    assert L._library_split(4096, 1536, 8960) == 1 and L._library_split(2048, 1536, 1536) == 1


def test_a_long_k_of_few_rows_goes_to_the_library_in_pieces():
    """The down projections of larger models at 17 to 256 rows: the library with K in eight pieces (seven where only
    that cuts K into whole steps of 64), also where the streaming kernel could take the rows; the sizes that were
    measured as exceptions keep their own plan; small models are left as they were."""
    plan = lambda rows, n, k: L.linear_plan(rows, n, k, False, False, True, rows <= 64)
    assert plan(64, 2048, 11008) == ("library", 8) and plan(256, 2048, 11008) == ("library", 8)
    assert plan(48, 3584, 18944) == ("library", 8) and plan(256, 3584, 18944) == ("library", 8)
    assert plan(64, 5120, 27648) == ("library", 8) and plan(128, 5120, 13824) == ("library", 8)
    assert plan(64, 8192, 29568) == ("library", 7) and plan(256, 8192, 29568) == ("library", 7)
    # the fewest rows: two pieces where the library is taken anyway and K is very long, else as before
    assert plan(32, 5120, 27648) == ("library", 2) and plan(24, 8192, 29568) == ("library", 2)
    assert plan(32, 5120, 13824) == ("library", 1) and plan(32, 3584, 18944) == ("skinny", 4, 4)
    assert plan(32, 2048, 11008) == ("skinny", 4, 4)
    # about as long as wide
    assert plan(64, 5120, 5120) == ("library", 8) and plan(256, 5120, 5120) == ("library", 8)
    assert plan(64, 8192, 8192) == ("library", 1) and plan(128, 8192, 8192) == ("library", 4)
    assert plan(32, 5120, 5120) == ("library", 1)
    assert plan(64, 3584, 18944) == ("library", 8) and plan(64, 3584, 3584) == ("skinny", 4, 4)
    assert L.linear_plan(64, 3584, 18944, False, False, False, True)[0] == "skinny"     # nobody to add parts: no pieces
    assert L.linear_plan(64, 3584, 18944, True, False, True, True)[0] == "skinny"       # a bias: one product
    # the 0.5B and 1.5B shapes: as measured there
    assert plan(64, 1536, 8960) == ("skinny", 4, 10) and plan(256, 1536, 8960) == ("library", 5)
    assert plan(64, 896, 4864) == ("skinny", 1, 4) and plan(64, 1536, 1536) == ("skinny", 1, 2)
    # prompt portions of many columns: a long K in halves up to 1,024 rows
    assert plan(512, 5120, 13824) == ("library", 2) and plan(1024, 8192, 29568) == ("library", 2)
    assert plan(2048, 5120, 13824) == ("library", 1) and plan(512, 8192, 8192) == ("library", 1)
    assert plan(512, 3584, 18944) == ("library", 4) and plan(2048, 2048, 11008) == ("library", 4)
    # decode rows up to 16 fold their norms and never come here in pieces
    assert plan(16, 5120, 27648)[0] == "skinny"
    # every such plan is one the tuner would also try
    for rows, n, k in ((64, 2048, 11008), (64, 8192, 29568), (32, 5120, 27648), (128, 8192, 8192), (64, 3584, 18944)):
        key = ("linear", rows, n, k, False, False, True, rows <= 64)
        assert L.linear_candidates(key)[0] == plan(rows, n, k)


def test_products_over_tiles_in_parts_of_k():
    """The rule for a consumer that adds parts, as linear() asks for it (operands that the kernel over tiles takes)."""
    plan = lambda rows, n, k, has_bias=False, f32=False, parts_ok=True: L.linear_plan(rows, n, k, has_bias, f32, parts_ok, rows <= 64, True)
    # as many parts as keep to one round of the chip, every one with a slab, none longer than the first
    assert plan(64, 1536, 8960) == ("tiles", 1, 10) and plan(256, 1536, 8960) == ("tiles", 1, 5)
    assert plan(64, 3584, 18944) == ("tiles", 1, 4) and plan(64, 3584, 3584) == ("tiles", 1, 4)
    assert plan(128, 3584, 3584) == ("tiles", 1, 4) and plan(64, 2048, 11008) == ("tiles", 1, 8)
    for rows in (17, 48, 64, 65, 100, 128, 192, 256):
        for n, k in ((1024, 3072), (1536, 3072), (1536, 8960), (2048, 11008), (2560, 4096), (3584, 3584), (4096, 4096)):
            way, _, parts = plan(rows, n, k)
            slabs = k // 64
            assert way == "tiles" and (parts - 1) * -(-slabs // parts) < slabs
            tiles = -(-n // (64 if rows <= 64 else 128)) * -(-rows // 64)
            assert parts == 1 or (parts * tiles <= 256 and parts * 8 <= slabs)
    # outside its range, and for consumers that add no parts, the rules before it
    assert plan(16, 1536, 8960)[0] == "skinny" and plan(257, 1536, 8960) == ("library", 4)
    assert plan(64, 1536, 1536) == ("skinny", 1, 2) and plan(64, 4112, 8960)[0] == "library"
    assert plan(64, 1528, 8960) == ("skinny", 4, 10)                # 1,528 columns are no multiple of 16
    assert plan(65, 3584, 18944) == ("library", 8)                  # the rows of A are most of what is read
    assert plan(256, 2560, 9728) == ("library", 8) and plan(224, 2560, 9728)[0] == "tiles"
    assert plan(32, 896, 4864) == ("skinny", 1, 4) and plan(33, 896, 4864) == ("tiles", 1, 9)       # few rows, few columns
    assert plan(64, 3584, 18944, parts_ok=False)[0] == "skinny" and plan(64, 3584, 18944, has_bias=True)[0] == "skinny"
    assert plan(64, 3584, 18944, f32=True)[0] == "skinny"
    assert L._parts_without_gaps(140, 10) == 10 and L._parts_without_gaps(9, 4) == 3 and L._parts_without_gaps(12, 5) == 4
    assert L._parts_without_gaps(1, 1) == 1


def _plan_and_key(monkeypatch, product, operands, **kwargs):
    """(the plan that the product of these operands runs, the key by which the tuner knows it), without running it."""
    from ginfer_amd.kernels import autotune
    ran = []
    for name in ("run_linear_plan", "run_gated_plan"):
        monkeypatch.setattr(L, name, lambda plan, x, *rest: ran.append(plan) or x)
    with autotune.collecting() as keys:
        product(*operands, **kwargs)
    (plan,), (key,) = ran, keys
    return plan, key


@pytest.mark.parametrize("rows", [257, 272, 320, 384, 385])
@pytest.mark.parametrize("n,k", [(1536, 8960), (3584, 18944), (2304, 1536)])
def test_the_plan_that_runs_is_a_candidate(rows, n, k, monkeypatch):
    """The rows between those that the fixed tiles take and the most that are dealt evenly: what runs by the rules, the tuner can keep."""
    x, w = torch.empty((rows, k), dtype=torch.bfloat16), torch.empty((n, k), dtype=torch.bfloat16)
    plan, key = _plan_and_key(monkeypatch, L.linear, (x, w), parts_ok=True)
    assert (plan[0] == "tiles") == (rows <= 384 and k > 2048)
    if rows % 16 == 0:                                 # the class's own count
        assert plan in L.linear_candidates(key)


@pytest.mark.parametrize("rows", [1, 16, 32, 48, 64, 96, 128, 224, 256, 272, 384, 400, 512, 528, 2048])
def test_the_tuner_starts_from_the_plan_that_linear_and_gated_linear_run(rows, monkeypatch):
    """Whatever another plan must beat by a margin is what runs without the tuner: products whose parts are added, heads, gated products."""
    bf16 = lambda *shape: torch.empty(shape, dtype=torch.bfloat16)
    for n, k in ((1536, 8960), (3584, 18944), (1536, 1536), (896, 4864), (2304, 1528)):
        plan, key = _plan_and_key(monkeypatch, L.linear, (bf16(rows, k), bf16(n, k)), parts_ok=True)
        assert L.linear_candidates(key)[0] == plan, key
    for n, k in ((151936, 1536), (152064, 3584), (32768, 1536)):
        plan, key = _plan_and_key(monkeypatch, L.linear, (bf16(rows, k), bf16(n, k)), out_dtype=torch.float32)
        assert L.linear_candidates(key)[0] == plan, key
    for n, k in ((17920, 1536), (37888, 3584), (9728, 896), (2048, 6144), (3072, 2048), (11136, 8192)):
        for bounds in (None, (7.0, 1.702, 1.0)):
            plan, key = _plan_and_key(monkeypatch, L.gated_linear, (bf16(rows, k), bf16(n, k)), bounds=bounds)
            assert L.gated_candidates(key)[0] == plan, key


@pytest.mark.parametrize("rows", [16, 17, 48, 64, 65, 272, 512, 513])
@pytest.mark.parametrize("K,hd,rd", [(1536, 128, 128), (1152, 48, 48), (1152, 64, 32), (1096, 64, 64)])
def test_the_projection_is_one_plan_of_several(rows, K, hd, rd, monkeypatch):
    """What an attention part runs for q|k|v by the rules is what the tuner starts from, and another way that it keeps is taken."""
    from types import SimpleNamespace
    from ginfer_amd.kernels import autotune
    from ginfer_amd.parts import attention, lookup
    ran = []

    class Ran(Exception):
        pass

    def project(way, *rest):
        ran.append(way)
        raise Ran
    monkeypatch.setattr(attention, "project", project)
    position = lookup("position", "rope_neox")(theta=1e4, rotary_dim=rd, max_positions=16, device="cpu")
    part = lookup("mixer", "attention")(hidden_size=K, num_heads=4, num_kv_heads=2, head_dim=hd, qkv_bias=True, out_bias=False, window=None,
                                        position=position, scale=None, dtype=torch.bfloat16, device="cpu")
    part.bind_weights({n: torch.empty(s.shape, dtype=torch.bfloat16) for n, s in part.weight_specs().items()})
    step = SimpleNamespace(positions=None)
    cache = SimpleNamespace(slot_mapping=None, k_pages=None, v_pages=None, owner=True)
    x = torch.empty((rows, K), dtype=torch.bfloat16)
    with autotune.collecting() as keys, pytest.raises(Ran):
        part.forward(x, step, cache)
    assert (ran[0][0] == "spread") == (17 <= rows <= 512 and rd == hd and K % 64 == 0) == bool(keys)
    for key in keys:
        ways = attention.projection_candidates(key)
        assert ways[0][0] == ran[0][0] and ("library",) in ways and len(set(ways)) == len(ways) >= 2
        for way in ways:
            table = autotune.Table()
            table[key] = way
            with autotune.using(table), pytest.raises(Ran):
                part.forward(x, step, cache)
            assert ran[-1] == way


@pytest.mark.parametrize("rows", [65, 512, 513, 2048])
@pytest.mark.parametrize("K,hd,rd", [(1536, 128, 128), (1152, 48, 48), (1152, 64, 32), (1096, 64, 64)])
def test_projections_of_more_rows_than_the_streaming_kernels_take(rows, K, hd, rd, monkeypatch):
    """Steps launched kernel by kernel wait for the host: such rows go to the library without a look at the other kernels' operands, which
    would not take them whatever they are."""
    from ginfer_amd.kernels import ops
    from ginfer_amd.parts import attention
    x, w = torch.empty((rows, K + 16), dtype=torch.bfloat16), torch.empty((8 * hd, K), dtype=torch.bfloat16)
    operands = [(x[:, :K], w), (x[:, 8:K + 8], w), (x[:, 1:K + 1], w), (x[:, :K].float(), w.float()), (x[:, :K], w[:, ::1].t().contiguous().t())]
    for a, b in operands:
        assert not ops.gemm_skinny_supported(a, b) and not ops.qkv_rope_skinny_supported(a, b, hd, rd)
        assert not attention._parts_supported(a, b, hd, rd)
    asked = []
    for name in ("gemm_skinny_supported", "qkv_rope_skinny_supported"):
        monkeypatch.setattr(ops, name, lambda *args: asked.append(args))
    assert all(attention._projection_way(a, b, hd, rd) == ("library",) for a, b in operands) and not asked


def test_the_projection_is_dealt_evenly_where_that_is_faster():
    """Sizes on both sides of the lines, as measured; the tuner starts from what runs there too."""
    from ginfer_amd.kernels import autotune
    from ginfer_amd.parts import attention
    def way(rows, n, k):
        x, w = torch.empty((rows, k), dtype=torch.bfloat16), torch.empty((n, k), dtype=torch.bfloat16)
        with autotune.collecting():
            way, key = attention.projection_choice(x, w, True, n // 128 - 4, 2, 128, 128)
        assert attention.projection_candidates((key[0], rows) + key[2:])[0][0] == way[0] and ("spread",) in attention.projection_candidates(key)
        return way[0]
    spread = [(17, 2048, 1536), (512, 2048, 1536), (384, 4608, 3584), (512, 4608, 3584), (256, 10240, 8192), (300, 6144, 4096), (512, 6144, 4096),
              (448, 7168, 5120), (300, 8192, 6144), (320, 8192, 3584)]
    library = [(257, 10240, 7680), (281, 10240, 4160), (403, 7168, 4096), (418, 8192, 6912), (384, 8192, 6144), (462, 6144, 7936), (430, 6144, 4096),
               (512, 10240, 5760), (442, 12288, 8128), (500, 12288, 6720)]
    assert [way(*size) for size in spread] == ["spread"] * len(spread) and [way(*size) for size in library] == ["library"] * len(library)


def test_measured_plans_stand_before_all_rules(monkeypatch):
    monkeypatch.setattr(L.TUNING, "measured_plans", {"64,3584,18944": ("library", 2), "64,1536,8960": ("tiles", 1, 7)})
    plan = lambda rows, n, k, tiles_ok=True: L.linear_plan(rows, n, k, False, False, True, rows <= 64, tiles_ok)
    assert plan(64, 3584, 18944) == ("library", 2) and plan(50, 3584, 18944) == ("library", 2)      # classes of 16 rows
    assert plan(64, 1536, 8960) == ("tiles", 1, 7)
    assert plan(64, 1536, 8960, False) == ("skinny", 4, 10)         # operands that its kernel does not take
    assert L.linear_plan(64, 3584, 18944, True, False, True, True, True)[0] == "skinny"             # a bias: no parts


def test_a_measured_plan_is_of_its_own_size_alone(monkeypatch):
    """It stands before the even dealing too, and leaves the products of other sizes, and operands that it is not for, to the rules."""
    choice = lambda rows, n, k, skinny_ok: L.linear_choice(rows, n, k, False, False, True, skinny_ok, True)
    sizes = [(64, 1536, 8960, True), (128, 3584, 18944, False), (384, 1536, 8960, False)]
    by_rules = [choice(*size) for size in sizes]
    assert all(plan[0] == "tiles" and plan[1] != 1 for plan in by_rules)
    monkeypatch.setattr(L.TUNING, "measured_plans", {"64,1024,8192": ("library", 4), "384,1536,8960": ("library", 5), "64,1536,8960": ("skinny", 4, 10)})
    assert [choice(*size) for size in sizes] == [("skinny", 4, 10), by_rules[1], ("library", 5)]
    assert choice(64, 1536, 8960, False) == by_rules[0]


def test_the_tuner_starts_from_the_plan_that_runs():
    for rows in (16, 17, 64, 128, 256):
        for n, k in ((1536, 8960), (3584, 3584), (3072, 8192), (896, 4864), (3584, 18944)):
            for tiles_ok in (False, True):
                plans = L.linear_candidates(("linear", rows, n, k, False, False, True, rows <= 64, tiles_ok))
                assert plans[0] == L.linear_choice(rows, n, k, False, False, True, rows <= 64, tiles_ok)
                assert L.linear_plan(rows, n, k, False, False, True, rows <= 64, tiles_ok) in plans[:2]
                assert tiles_ok or not any(p[0] == "tiles" for p in plans)
                assert len(set(plans)) == len(plans) and ("library", 1) in plans
    # parts that do not divide K are candidates like any other
    assert ("tiles", 1, 5) in L.linear_candidates(("linear", 64, 3072, 8192, False, False, True, True, True))


def test_tiles_of_the_gated_product():
    """Which tiles a number of rows gets, and that the rule counts those: one place says it for both."""
    from ginfer_amd.kernels import ops
    tiles = lambda rows, n: ops.GATED_TILINGS[ops.gated_tiling(rows, n)]
    assert tiles(17, 17920) == tiles(64, 17920) == (128, 64) and tiles(64, 37888) == (256, 128)
    assert tiles(65, 17920) == tiles(128, 32768) == (128, 128) and tiles(128, 32770) == (256, 128)
    assert tiles(129, 16384) == (128, 128) and tiles(129, 17920) == tiles(256, 37888) == (128, 256)
    assert tiles(384, 8192) == (128, 128) and tiles(257, 17920) == tiles(1024, 17920) == (256, 128)
    assert tiles(1025, 17920) == tiles(4096, 17920) == (256, 256)
    for rows in range(1, 2100, 7):
        for n in (16, 8192, 17920, 37888, 70000):
            of_w, of_a = tiles(rows, n)
            assert of_a >= min(rows, 64) and (rows > 384 or of_a < 2 * rows or of_a == 64 or of_w == of_a == 128 or of_w == 256)


def test_gated_products_over_tiles_at_their_thresholds():
    """The sizes the rule was measured at: taken where the kernel was the faster, refused where the library was."""
    g = lambda rows, n, k: L.tiles_gated(rows, n, k)
    assert not g(16, 17920, 1536) and g(17, 17920, 1536) and g(64, 8192, 1024)
    assert not g(64, 8184, 1024) and not g(64, 8192, 1016) and not g(64, 12288, 3072) and not g(128, 10240, 1792)
    assert all(g(rows, n, k) for rows in (65, 96, 128) for n, k in ((17920, 1536), (22016, 2048), (27648, 5120), (28672, 4096),
                                                                     (19456, 2560), (16384, 1280), (37888, 3584), (59136, 8192)))
    # two rounds of the chip beside few rows: the library
    assert not g(129, 37888, 3584) and not g(256, 59136, 8192) and not g(128, 65792, 4096)
    assert g(256, 17920, 1536) and g(256, 12288, 3072) and g(256, 27648, 5120)
    # up to 384 rows full rounds, or a short K: the sizes where it had become up to 27 % slower than the library are refused
    assert g(300, 17920, 1536) and g(384, 37888, 3584) and g(300, 10240, 1792) and g(384, 19456, 2560)
    assert not any(g(rows, n, k) for rows in (257, 300, 384) for n, k in ((22016, 2048), (27648, 5120), (28672, 4096), (59136, 8192)))
    # ... and around 1,000 rows up to 20 %
    assert g(1000, 37888, 3584) and g(1024, 37888, 3584) and g(1000, 8192, 1024)
    assert not any(g(1000, n, k) for n, k in ((22016, 2048), (27648, 5120), (28672, 4096), (59136, 8192), (16384, 1280), (10240, 1792)))
    assert not any(g(rows, 17920, 1536) for rows in (385, 512, 700, 1000, 1025, 1500, 2048))
    # by the tiles that run: 256 x 256 from 1,025 rows on
    assert g(1025, 37888, 3584) and g(1280, 37888, 3584) and not g(1281, 37888, 3584) and not g(1536, 37888, 3584)
    assert g(1700, 17920, 1536) and g(2048, 37888, 3584) and not g(2049, 37888, 3584)


def test_gated_products_in_tiles_of_192_rows_at_their_thresholds():
    """Taken where they fill the chip's rounds better than the other tiles, refused where those, or the library, were the faster."""
    from ginfer_amd.kernels import ops
    wide = lambda rows, n, k: ops.GATED_WIDE_TILINGS.get(ops.gated_wide_tiling(rows, n, k))
    assert wide(64, 37888, 3584) == (192, 64) and wide(65, 37888, 3584) == wide(128, 37888, 3584) == (192, 128)
    assert wide(64, 32768, 3584) is None and wide(64, 49152, 1024) == (192, 64) and wide(64, 49344, 1024) is None
    assert wide(129, 17920, 1536) == wide(256, 22016, 2048) == (192, 128) and wide(256, 16384, 1280) is None and wide(256, 37888, 3584) is None
    assert wide(400, 22016, 2048) == (192, 256) and wide(400, 17920, 1536) is None and wide(384, 22016, 2048) is None
    assert all(wide(rows, 17920, 1536) == (192, 256) for rows in (1025, 1280, 1900, 2048))
    assert not any(wide(rows, 17920, 1536) for rows in (513, 1024, 1300, 1536, 1792, 4096)) and wide(2048, 22016, 2048) is None
    assert wide(1025, 28672, 4096) is None and wide(2048, 12288, 3072) == (192, 256)
    assert L.gated_plan(2048, 17920, False, True, 1536, True) == ("tiles",) and L.gated_plan(512, 17920, False, True, 1536, True) == ("transposed",)
    # 385 to 512 rows: only while K is short, shorter at 512, where the library's transposed product stands against it
    assert wide(511, 22016, 4096) == wide(400, 24576, 4096) == wide(512, 22016, 2560) == (192, 256)
    assert not any(wide(rows, n, k) for rows, n, k in ((400, 21504, 5120), (450, 24576, 8192), (511, 22016, 4160), (512, 22016, 2624), (512, 22016, 4096)))
    assert L.gated_plan(450, 24576, False, False, 8192, True) == ("library",) and L.gated_plan(512, 24576, False, True, 4096, True) == ("transposed",)
    # the weight-streaming kernel up to 32 rows, while W is small
    assert L.gated_plan(17, 17920, True, False, 1536, True) == L.gated_plan(32, 22016, True, True, 2048, True) == ("skinny",)
    assert L.gated_plan(32, 19456, True, True, 2560, True) == ("skinny",) and L.gated_plan(32, 22528, True, True, 2560, True) == ("tiles",)
    assert L.gated_plan(33, 17920, True, False, 1536, True) == L.gated_plan(17, 37888, True, False, 3584, True) == ("tiles",)


def test_gated_products_dealt_evenly():
    """A plan's tiles hold what it deals out, in one round of the chip (two for the fewest rows of the widest), and stand where they were
    measured the faster."""
    from ginfer_amd.kernels import ops
    for rows in list(range(17, 513, 9)) + [64, 65, 128, 129, 192, 193, 256, 257, 384, 512]:
        for n, k in ((16, 64), (1024, 320), (8192, 1024), (9728, 896), (17920, 1536), (22016, 2048), (37888, 3584), (59136, 8192), (131072, 128)):
            plan = ops.spread_plan(rows, n, k)
            if plan is None:
                continue
            (tm, tw, bk), m_tiles, groups = ops.SPREAD_SHAPES[plan[0]], plan[1], plan[2]
            tile_rows = -(-(-(-rows // m_tiles)) // 16) * 16
            assert tile_rows <= tm and (m_tiles - 1) * tile_rows < rows and k % bk == 0 and 1 <= groups <= n // 8
            assert -(-(n // 8) // groups) * 8 <= tw and m_tiles * groups <= (512 if rows <= 64 else 256)
    plan = ops.spread_plan
    faster = lambda plan, rows, n, k: L.spread_is_faster((plan,), rows, n, k)
    assert plan(64, 17920, 1536) == (0, 1, 256) and plan(128, 17920, 1536) == (1, 1, 256) and plan(161, 17920, 1536) == plan(256, 17920, 1536) == (3, 2, 128)
    assert plan(384, 17920, 1536) == (4, 2, 128) and plan(64, 37888, 3584) == (2, 1, 256) and plan(64, 59136, 8192) == (6, 1, 512)
    assert plan(16, 17920, 1536) is None and plan(513, 17920, 1536) is None and plan(65, 59136, 8192) is None
    assert plan(256, 22016, 2048) is None and plan(300, 10496, 3584) is None and plan(225, 9728, 896) is None and plan(256, 9088, 2880) == (7, 2, 128)
    assert plan(218, 22912, 1152) is None and plan(220, 24576, 7360) is None and plan(200, 18944, 1152) and plan(301, 8448, 2240) is None
    assert plan(385, 14336, 2048) is None and plan(512, 16384, 2048) is None and plan(384, 14336, 2048) and plan(512, 17920, 1536)
    assert faster("library", 225, 9728, 896) and faster("library", 300, 10496, 3584)      # by the other tiles
    assert plan(150, 27648, 5120) == (8, 1, 256) and plan(225, 12288, 2560) and plan(150, 3712, 2048)
    assert faster("skinny", 17, 17920, 1536) and not faster("skinny", 17, 9728, 896) and faster("skinny", 49, 3072, 2048) and not faster("skinny", 49, 2688, 512)
    assert faster("library", 400, 17920, 1536) and faster("transposed", 512, 17920, 1536) and not faster("library", 92, 2048, 6144)
    assert faster("library", 384, 11136, 8192) and not faster("library", 508, 11136, 8192) and not faster("tiles", 64, 17920, 1536)


def test_gated_products_leave_the_even_dealing_where_it_is_slower():
    """Drawn sizes on both sides of the lines: few rows of a W that the streaming kernel takes, a K that is no multiple of 128, tiles that are
    mostly room."""
    faster = lambda plan, rows, n, k: L.spread_is_faster((plan,), rows, n, k)
    assert all(faster("skinny", *size) for size in ((17, 17920, 1536), (32, 14720, 1024), (49, 2048, 6144), (64, 3072, 2048), (24, 11392, 1088)))
    assert not any(faster("skinny", *size) for size in ((34, 1792, 7488), (64, 1280, 4032), (57, 3968, 7232), (36, 1536, 4096), (48, 3072, 2048),
                                                        (20, 11264, 832), (20, 11264, 1024 - 64), (17, 11264, 768)))
    assert all(faster("library", *size) for size in ((64, 8192, 8000), (289, 5248, 4096), (197, 6912, 3584), (64, 5120, 3392), (128, 17920, 8192)))
    assert not any(faster("library", *size) for size in ((32, 4096, 8000), (17, 4224, 4544), (289, 5248, 6528), (296, 5376, 6144), (197, 6912, 7552)))


def test_the_tables_lines_hold_after_a_size_was_seen(monkeypatch):
    """Plans by size are remembered, the lines that a user sets are not passed over for that."""
    from ginfer_amd.kernels import ops
    seen = ops.spread_plan(256, 17920, 1536), ops.spread_plan(300, 10496, 3584)
    assert seen[0] and seen[1] is None
    for name, value in (("spread_up_to_rows", 512), ("spread_square_tiles", 257)):
        with monkeypatch.context() as m:
            m.setattr(L.TUNING, name, value)
            assert ops.spread_plan(300, 10496, 3584)
    assert (ops.spread_plan(256, 17920, 1536), ops.spread_plan(300, 10496, 3584)) == seen


def test_few_columns_dealt_evenly():
    """A plan's tiles hold what it deals out, its parts of K are whole slabs, and it stands where it was measured the faster."""
    from ginfer_amd.kernels import ops
    shapes = ops.SPREAD_SHAPES + ops.SPREAD_NARROW_SHAPES
    for rows in list(range(17, 513, 11)) + [64, 65, 128, 192, 256, 384, 512]:
        for n, k in ((16, 64), (896, 4864), (1536, 1536), (1536, 8960), (2048, 1536), (3584, 18944), (4608, 3584), (10240, 8192), (2048, 704)):
            for parts in (1, 2, 4, 8):
                found = ops.spread_few_columns(rows, n, k, parts)
                if found is None:
                    continue
                number, m_tiles, groups = found[1]
                (tm, tw, bk), tile_rows, of_part = shapes[number], -(-(-(-rows // m_tiles)) // 16) * 16, -(-(k // 64) // parts)
                assert tile_rows <= tm and (m_tiles - 1) * tile_rows < rows and m_tiles * groups * parts <= 256 and 1 <= groups <= n // 8
                assert -(-(n // 8) // groups) * 8 <= tw and k % bk == 0 and (parts == 1 or of_part * 64 % bk == 0) and (parts - 1) * of_part < k // 64
    assert ops.spread_few_columns(64, 2048, 1536)[1] == (10, 2, 128) and ops.spread_few_columns(65, 7168, 5120)[1] == (12, 1, 256)
    assert ops.spread_few_columns(64, 16, 64, 2) is None and ops.spread_few_columns(512, 131072, 64) is None
    def parts(rows, n, k):
        plan = L.linear_plan(rows, n, k, False, False, True, rows <= 64, True)
        return L.spread_parts(plan, rows, n, k)
    assert parts(64, 1536, 8960) == ("tiles", 320113, 8) and L._dealing(320113) == (13, 1, 32) and L._dealing(1) is None and parts(128, 3584, 18944)[2] == 8 and parts(64, 3584, 18944)[2] == 8
    assert parts(96, 1536, 1536)[2] == 2 and parts(64, 2048, 2048) and parts(17, 5120, 13824)
    assert not any(parts(rows, n, k) for rows, n, k in ((16, 1536, 8960), (48, 1536, 1536), (64, 2048, 11008), (91, 3584, 3584), (250, 4096, 14336),
                                                         (300, 2304, 1536), (385, 1536, 8960), (128, 1536, 960), (64, 1528, 8960)))
    # tiles of 128 columns that own few of them, where slabs of 128 do not divide a part
    assert not any(parts(rows, n, k) for rows, n, k in ((64, 1664, 1984), (50, 640, 1856), (31, 1152, 3904), (63, 512, 3904), (170, 1984, 5760), (203, 704, 16512),
                                                         (227, 1280, 5056), (149, 2048, 5312)))
    assert all(parts(rows, n, k) for rows, n, k in ((64, 1664, 2112), (64, 2048, 1984), (64, 1664, 1920), (31, 3072, 6208), (170, 1984, 12224), (207, 3136, 9024), (24, 2688, 4096)))
    key = ("linear", 128, 1536, 8960, False, False, True, False, True)
    assert L.linear_candidates(key)[:2] == [("tiles", L._dealing_number(14, 1, 32), 8), L.linear_plan(*key[1:])]


def test_heads_of_many_columns():
    """Where the head of 17 to 64 rows leaves the library, and that the tiles hold what its plan deals out."""
    from ginfer_amd.kernels import ops
    assert all(L.head_is_wide(rows, 151936, k) for rows in (17, 33, 64) for k in (896, 1536, 3584)) and L.head_is_wide(48, 65024, 5120)
    assert not any(L.head_is_wide(*x) for x in ((16, 151936, 1536), (65, 151936, 1536), (64, 65024, 5120), (64, 256000, 3584), (33, 24560, 1536),
                                                (33, 151936, 1500), (33, 50257, 768)))
    for n in (24576, 32768, 50304, 151936, 256000):
        shape, m_tiles, groups = ops.spread_many_columns(64, n)
        assert shape == 2 and m_tiles == 1 and groups % 256 == 0 and -(-(n // 8) // groups) * 8 <= ops.SPREAD_SHAPES[shape][1]
    key = ("linear", 64, 151936, 1536, False, True, False, True, True)
    assert L.linear_candidates(key)[:2] == [L.wide_plan(64, 151936), ("library", 1)]


def test_steps_of_a_trip():
    """Products of few rows: a short K in one way to memory, then two, then three steps at a time."""
    from ginfer_amd.kernels import build
    trip = build.load("gemm_skinny").ga_skinny_trip
    assert [trip(n) for n in range(1, 12)] == [1, 2, 3, 4, 5, 3, 4, 4, 3, 3, 3] and trip(37) == 3


def test_columns_dealt_evenly():
    """The head of few rows stays with its many small workgroups; few rows of a gate-up product have no second tile for a column or two."""
    from ginfer_amd.kernels import build
    even = build.load("gemm_skinny").ga_skinny_even_workgroups
    assert [even(M, 151936, 0) for M in (1, 4)] == [0, 0] and even(5, 151936, 0) == even(16, 151936, 0) == 2304 and even(16, 16383, 0) == 0
    assert even(1, 2047, 1) == 0 and even(1, 4096, 1) == 256 and even(8, 8960, 1) == even(1, 8960, 1) == 768 and even(1, 18944, 1) == 1280
    assert even(4, 4097, 1) == even(1, 4864, 1) == even(1, 5375, 1) == 512 and even(5, 4097, 1) == even(16, 4864, 1) == 256 and even(16, 5376, 1) == 512


def test_tokens_of_a_workgroup_of_block_means():
    """Neighbours share a workgroup only while at most one or two of them end a block."""
    from ginfer_amd.kernels import build
    tokens = build.load("pooled_attention").ga_pwa_pool_tokens
    assert [tokens(512, pool) for pool in (1, 2, 3, 4, 7, 8, 64)] == [1, 2, 2, 4, 4, 8, 8] and tokens(511, 64) == 1


def test_columns_of_a_unit_of_the_fused_projection():
    """Spread over twice the workgroups only where those are one round of the chip."""
    from ginfer_amd.kernels import build
    columns = build.load("gemm_skinny").ga_qkv_unit_columns
    assert columns(2048, 128, 2, 0) == columns(1152, 64, 2, 0) == 4 and columns(2112, 32, 2, 0) == columns(2560, 128, 2, 0) == columns(4608, 128, 2, 0) == 8
    assert columns(2048, 128, 1, 0) == 16 and columns(2048, 128, 1, 1) == 8


def test_fused_projection_of_many_columns():
    """q|k|v of more rows than a block of 16: fused, while K is short and, from 49 rows on, its workgroups make one round of the chip."""
    from ginfer_amd.parts.attention import _library_then_rotation_is_faster as library
    assert not any(library(rows, 4608, 15360) for rows in (1, 16)) and library(17, 4608, 4608) and not library(17, 4600, 4608)
    assert not any(library(rows, k, n) for rows, k, n in ((64, 3584, 4608), (64, 4096, 6144), (64, 2560, 7680), (64, 4096, 8192), (64, 1536, 24576)))
    assert not library(48, 4096, 12288) and all(library(rows, 4096, 12288) for rows in (49, 64)) and library(64, 3072, 9216) and library(64, 2048, 10240)


def test_projection_that_the_fused_kernel_does_not_take():
    """48 rows and more with a rotation over part of a head: in parts of K, while K is short and the columns few; else the library.  What the
    fused kernel takes it keeps."""
    import torch
    from ginfer_amd.kernels import ops
    from ginfer_amd.parts.attention import _projection_way as way
    rows = lambda n, k: torch.empty((n, k), dtype=torch.bfloat16)
    def at(n, cols, k, head_dim=128, rotary_dim=64):
        return way(rows(n, k), rows(cols, k), head_dim, rotary_dim)
    assert at(48, 2048, 1536) == at(64, 3584, 1536) == ("parts", 4) and at(64, 1152, 896, 64, 32) == ("parts", 2) and at(64, 1600, 1536, 80, 80) == ("parts", 4)
    assert at(47, 2048, 1536) == at(65, 2048, 1536) == at(64, 3600, 1536) == at(64, 2048, 3072) == at(64, 1152, 760) == ("library",)
    assert at(64, 2048, 1536, 128, 128) == at(1, 2048, 1536, 128, 128) == ("fused",) and at(64, 12288, 4096, 128, 128) == ("library",)
    assert at(64, 2048, 1536, 128, 60) == ("library",)                                         # pairs that are no fours
    assert way(ops.ScaledRows(rows(8, 1536), None, 0.0), rows(2048, 1536), 128, 128) == ("fused",)
    assert way(torch.empty((64, 1536)), torch.empty((2048, 1536)), 128, 64) == ("library",)    # 32-bit


def test_the_gated_product_is_one_plan_of_several():
    """The tuner starts from the plan that runs, can leave it, and tries tiles where the rule does not take them."""
    key = lambda rows, n, k, tiles_ok=True, bounds=None: ("gated", rows, n, k, rows <= 64, bounds is None and rows % 8 == 0, tiles_ok, bounds)
    assert L.gated_candidates(key(64, 17920, 1536)) == [("tiles",), ("skinny",), ("library",), ("transposed",)]
    assert L.gated_candidates(key(512, 17920, 1536)) == [("tiles",), ("library",), ("transposed",)]
    assert L.gated_candidates(key(300, 17920, 1536, False)) == [("library",)]
    assert L.gated_candidates(key(100, 17920, 1536, True, (7.0, 1.702, 1.0))) == [("tiles",), ("library",)]
    assert L.gated_plan(64, 17920, True, True, 1536, True) == ("tiles",) and L.gated_plan(64, 17920, True, True, 1536, False) == ("library",)


def test_measured_plans_can_be_set_from_json():
    from ginfer_amd.kernels.tuning import Tuning
    t = Tuning()
    t.update({"measured_plans": {"64,1024,8192": ["library", 4]}})
    assert t.measured_plans == {"64,1024,8192": ("library", 4)}


def test_nearest_divisor():
    assert L._nearest_divisor(140, 10.7, 16) == 10
    assert L._nearest_divisor(140, 5.3, 16) == 5
    assert L._nearest_divisor(296, 4.6, 16) == 4
    assert L._nearest_divisor(7, 3.0, 16) == 1          # 1 and 7 are the divisors; 1 is nearer
    assert L._nearest_divisor(24, 100.0, 3) == 3        # never above the cap


def test_rules_as_plans():
    """The rules' decisions as plans, at the sizes they were measured at."""
    # decode rows of the 1.5B shape: the streaming kernel, K in parts where the norm that follows adds them
    assert L.linear_plan(64, 1536, 8960, False, False, True, True) == ("skinny", 4, 10)
    assert L.linear_plan(8, 1536, 8960, False, False, True, True) == ("skinny", 1, 5)
    assert L.linear_plan(8, 1536, 8960, False, False, False, True) == ("skinny", 1, 1)     # nobody to add parts
    assert L.linear_plan(8, 1536, 8960, False, True, True, True) == ("skinny", 1, 1)       # float32 out: no parts
    # wide outputs go to the library from 17 rows on; prompt portions always
    assert L.linear_plan(64, 17920, 1536, False, False, False, True) == ("library", 1)
    assert L.linear_plan(16, 17920, 1536, False, False, False, True) == ("skinny", 1, 1)
    assert L.linear_plan(2048, 1536, 8960, False, False, True, False) == ("library", 4)
    assert L.linear_plan(2048, 1536, 8960, True, False, True, False) == ("library", 1)     # a bias: one product
    assert L.linear_plan(4096, 1536, 8960, False, False, True, False) == ("library", 1)
    assert L.gated_plan(8, 17920, True, True) == ("skinny",)
    assert L.gated_plan(64, 17920, True, True) == ("library",)
    assert L.gated_plan(2048, 17920, False, True) == ("transposed",)
    assert L.gated_plan(2040, 17920, False, True) == ("library",)


def test_candidates_hold_the_rules_plan_first_and_only_plans_that_fit():
    for rows in (1, 8, 16, 17, 64, 128, 256):
        for n, k in ((1536, 8960), (3584, 18944), (8192, 29568), (88, 520), (1536, 1536), (151936, 1536)):
            for has_bias in (False, True):
                for f32 in (False, True):
                    for parts_ok in (False, True):
                        skinny_ok = rows <= 64
                        key = ("linear", rows, n, k, has_bias, f32, parts_ok, skinny_ok)
                        plans = L.linear_candidates(key)
                        assert plans[0] == L.linear_plan(rows, n, k, has_bias, f32, parts_ok, skinny_ok)
                        assert len(set(plans)) == len(plans) and ("library", 1) in plans
                        for plan in plans[1:]:
                            if plan[0] == "skinny":
                                assert skinny_ok and plan[1] in (1, 4) and (plan[1] == 1 or rows > 16)
                                if plan[2] > 1:
                                    assert parts_ok and not f32 and -(-k // 64) % plan[2] == 0 and plan[2] * 8 <= -(-k // 64)
                            else:
                                if plan[1] > 1:
                                    assert parts_ok and not f32 and not has_bias
                                    assert k % plan[1] == 0 and (k // plan[1]) % 8 == 0 and k // plan[1] >= 512
    assert L.gated_candidates(("gated", 64, 17920, 1536, True, True)) == [("library",), ("skinny",), ("transposed",)]
    assert L.gated_candidates(("gated", 2048, 17920, 1536, False, True)) == [("transposed",), ("library",)]
    assert L.gated_candidates(("gated", 100, 17920, 1536, False, False)) == [("library",)]


def test_kept_plans_answer_for_their_class_of_rows():
    from ginfer_amd.kernels import autotune
    assert [autotune.rows_class(r) for r in (1, 7, 16, 17, 32, 33, 64, 65, 200)] == [1, 7, 16, 32, 32, 48, 64, 80, 208]
    assert not autotune.active() and autotune.choose(("linear", 32), ("w",)) is None
    with autotune.collecting() as seen:
        assert autotune.active()
        assert autotune.choose(("linear", 32), ("w0",)) is None and autotune.choose(("linear", 32), ("w1",)) is None
        assert autotune.choose(("gated", 32), ("w2",)) is None
    assert seen == {("linear", 32): [("w0",), ("w1",)], ("gated", 32): [("w2",)]} and not autotune.active()
    table = autotune.Table()
    table[("linear", 32)] = ("library", 2)
    assert not autotune.active() and autotune.choose(("linear", 32), ("w",)) is None      # no table is in use
    with autotune.using(table):
        assert autotune.active() and autotune.choose(("linear", 32), ("w",)) == ("library", 2)
        assert autotune.choose(("linear", 48), ("w",)) is None
        with autotune.using(None):                                                          # a runner without plans
            assert not autotune.active() and autotune.choose(("linear", 32), ("w",)) is None
    assert not autotune.active()


def test_how_many_workgroups_heads_share_a_prompts_tiles_from():
    """Fewer than a round of the chip where the heads are wide and the tiles a prompt's own; small heads, other sizes and
    recorded steps, whose tiles hold padding, wait for the full number."""
    import types
    from ginfer_amd.kernels import ops
    own, none, recorded = (types.SimpleNamespace(extra=e) for e in ({}, None, {"static_plan": {}}))
    full = ops.TUNING.prefill_fill_workgroups
    assert ops._prefill_fill(own, 128) == ops._prefill_fill(none, 128) == full // 2
    assert ops._prefill_fill(own, 256) == full * 3 // 4
    assert ops._prefill_fill(own, 64) == ops._prefill_fill(own, 112) == full
    assert all(ops._prefill_fill(recorded, d) == full for d in (64, 128, 256))


def test_keys_of_a_short_prompt_are_dealt_out_and_those_of_other_steps_are_not(monkeypatch):
    """The rule that deals a tile's keys to several workgroups: one prompt of 2,048 tokens alone in a step (one round of
    workgroups, the last tile walking twice the mean) is split, every part within the mean share, the parts of a tile
    covering its keys once; shorter and longer prompts, and steps of many requests, stay whole."""
    from ginfer_amd.kernels import ops
    tiles = ops.plan_rows([2048], [0], 32)[3]
    assert ops.key_parts(tiles, 32, 0, 4, 2) is None          # switched off in the table of thresholds: it was measured slower
    monkeypatch.setattr(ops.TUNING, "prefill_split_imbalance", 1.5)
    pieces, parts, rows, n = ops.key_parts(tiles, 32, 0, 4, 2)
    assert n == 2 and len(pieces) == len(parts) > len(tiles) and len(rows) % 32 == 0
    share = sum(range(1, 65)) * 4 / 256.0
    assert max((e - b) // 32 for b, e, _, _ in parts) <= 1.15 * share + 2
    by_tile = {}
    for t, (b, e, at, packed) in zip(pieces, parts):
        by_tile.setdefault(t, []).append((b, e, at, packed & 0xffff, packed >> 16))
    assert set(by_tile) == set(tiles)
    for t, ps in by_tile.items():
        ps.sort()
        assert ps[0][0] == 0 and ps[-1][1] == ((t[3] + t[2] - 1) // 32 + 1) * 32
        assert all(x[1] == y[0] for x, y in zip(ps, ps[1:])) and [x[3] for x in ps] == list(range(len(ps)))
        if len(ps) > 1:
            assert all(x[4] == n and x[2] == ps[0][2] for x in ps)
            assert [r[0] for r in rows[ps[0][2]:ps[0][2] + t[2]]] == list(range(t[1], t[1] + t[2]))
        else:
            assert ps[0][2] == -1
    assert [e - b for b, e, _, _ in parts] == sorted((e - b for b, e, _, _ in parts), reverse=True)      # longest walks first
    assert ops.key_parts(ops.plan_rows([1024], [0], 32)[3], 32, 0, 12, 8) is None
    assert ops.key_parts(ops.plan_rows([4096], [0], 32)[3], 32, 0, 4, 2) is None
    assert ops.key_parts(ops.plan_rows([512] * 4, [0] * 4, 32)[3], 32, 0, 4, 2) is None
    # a window bounds every tile's keys: nothing to deal out
    assert ops.key_parts(tiles, 32, 256, 4, 2) is None


def test_gates_that_add_parts_ask_for_them_beyond_few_rows(monkeypatch):
    """Side-by-side sublayers: the feed-forward's product comes whole up to the table's number of rows, and always where the gate cannot add."""
    import torch
    from types import SimpleNamespace
    from ginfer_amd.kernels.tuning import TUNING
    from ginfer_amd.parts import lookup

    def asked(rows, adds=True):
        seen = []
        part = SimpleNamespace(makes_partial_sums=True, forward=lambda n, parts_ok=False: (seen.append(parts_ok), n)[1])
        gate = SimpleNamespace(names=["a", "b"], adds_partial_sums=adds, logits=lambda n: None, add=lambda *a, **k: None)
        block = lookup("arrangement", "parallel_gated")(dict(norm=SimpleNamespace(forward=lambda r, d: r), feed_forward=part, gate=gate,
                                                             mixer=SimpleNamespace(forward=lambda n, step, cache: n)))
        block.forward(torch.zeros((rows, 4)), None, None, None)
        return seen[0]
    assert [asked(8), asked(9), asked(9, adds=False)] == [False, True, False]
    monkeypatch.setattr(TUNING, "gate_adds_parts_beyond_rows", 20)
    assert [asked(20), asked(21)] == [False, True]
