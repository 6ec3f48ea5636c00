"""The planner: the reference's choices restated (pinned by its golden plans and logic tests), and the MI355X
planner's own choices, variant codes and choice table. Host logic only, no GPU."""
import json
import os

import pytest

from fhtest import fhconv

GOLDEN = os.path.join(os.path.dirname(os.path.abspath(__file__)), "golden", "ref_conv_plans.json")


def test_reference_golden_plans_are_reproduced():
    # every conv of the 27 golden plans (crates/flyhigh-engine/tests/golden/*, 3 device classes x 9 sessions):
    # kernel, grid, packed-weight bytes, the 16 ImplicitGemmParams words, the split-K reduce and the residual add
    recs = json.load(open(GOLDEN))
    assert len(recs) == 639
    seen = set()
    for r in recs:
        c, cls = r["conv"], r["cls"]
        got = fhconv.ref_conv_steps(c["cin"], c["cout"], c["h"], c["w"], c["stride"], residual=c["residual"],
                                    coop=cls.startswith("tc"), f32_mode=cls.endswith("f32"))
        want = [(s[0], tuple(s[1]), s[2], s[3]) for s in r["steps"]]
        assert got == want, r["source"]
        seen.update(s[0] for s in want)
    # the golden plans exercise every path of the restatement
    assert {"fused", "fused2", "fdirect32", "xshift", "tconv", "tconv32", "skreduce", "binary"} <= seen


def has(lst, kind):
    return any(c & 15 == kind for c in lst)


def test_portable_candidates_for_a_wide_conv():
    # crates/flyhigh-engine/tests/logic.rs:33-45
    lst = fhconv.cand_list(False, 64, 60, 108, False)
    assert has(lst, fhconv.CAND_TILED) and has(lst, fhconv.CAND_TILED8) and has(lst, fhconv.CAND_TILED88)
    assert not has(lst, fhconv.CAND_TC) and not has(lst, fhconv.CAND_DIRECT)
    assert not has(lst, fhconv.CAND_TILED16) and not has(lst, fhconv.CAND_TILEDN8)
    for ks in (1, 2, 4):
        assert fhconv.CAND_TILED | ks << 4 in lst


def test_narrow_candidates_for_a_small_conv():
    # logic.rs:47-52
    lst = fhconv.cand_list(False, 16, 120, 216, False)
    assert has(lst, fhconv.CAND_TILED) and has(lst, fhconv.CAND_TILED16) and has(lst, fhconv.CAND_TILEDN8)
    assert not has(lst, fhconv.CAND_TILED8) and not has(lst, fhconv.CAND_TILED88)


def test_tensor_core_candidates_need_the_feature_and_direct_needs_its_shape():
    # logic.rs:54-61
    tc = fhconv.cand_list(True, 64, 60, 108, False)
    assert has(tc, fhconv.CAND_TC) and not has(tc, fhconv.CAND_DIRECT)
    direct = fhconv.cand_list(True, 64, 60, 112, True)
    assert has(direct, fhconv.CAND_TC) and has(direct, fhconv.CAND_DIRECT)
    assert has(tc, fhconv.CAND_TILED)


def test_try_all_adds_the_kernels_that_never_won():
    base = fhconv.cand_list(True, 64, 60, 112, True)
    full = fhconv.cand_list(True, 64, 60, 112, True, try_all=True)
    assert not has(base, fhconv.CAND_DIRECT64) and has(full, fhconv.CAND_DIRECT64)
    assert has(full, fhconv.CAND_TILEDM32) and has(full, fhconv.CAND_TILED8P)


def test_candidate_names():
    assert fhconv.cand_name(fhconv.CAND_TILED) == "tiled"
    assert fhconv.cand_name(fhconv.CAND_TILED | 4 << 4) == "tiled/k4"
    assert fhconv.cand_name(fhconv.CAND_DIRECT) == "direct"
    with pytest.raises(fhconv.FhcError):
        fhconv.cand_name(12)


def test_forced_split_and_env_override_in_the_reference_planner():
    # kernels.rs:157-170: a forced split (candidate nibble) is capped by the K-step count; FH_KSPLIT overrides it;
    # the partials stay under 32 MB
    steps = fhconv.ref_conv_steps(36, 36, 60, 108, 1, coop=False, cand=fhconv.CAND_TILED | 4 << 4)
    assert steps[0][1] == (1, 102, 4) and steps[1][0] == "skreduce"
    steps = fhconv.ref_conv_steps(3, 36, 120, 216, 2, coop=False, cand=fhconv.CAND_TILED | 4 << 4)
    assert steps[0][1][2] == 2  # kp 32 -> 2 K-steps
    steps = fhconv.ref_conv_steps(36, 36, 60, 108, 1, coop=False, ksplit_env=3)
    assert steps[0][1][2] == 3
    big = fhconv.ref_conv_steps(32, 32, 1088, 1920, 1, coop=False, cand=fhconv.CAND_TILED | 4 << 4)
    assert big[0][1][2] == 1 and len(big) == 1  # 4 * 32 * 2088960 * 4 bytes > 32 MB


def test_tune_table_round_trips_and_skips_garbage():
    # crates/flyhigh-engine/tests/defaults.rs:55-64, on the MI355X table (same key and text format)
    fhconv.tune_clear()
    try:
        text = "96,96,60,108,1=18\nnot a line\n36,36,180,320,1=2\n1,2,3=4\n48,48,60,108,1=x\n"
        assert fhconv.parse_tune(text) == 2
        assert fhconv.tune_get(96, 96, 60, 108, 1) == 18
        assert fhconv.tune_get(36, 36, 180, 320, 1) == 2
        assert fhconv.tune_get(48, 48, 60, 108, 1) is None
        out = fhconv.format_tune()
        assert out == "36,36,180,320,1=2\n96,96,60,108,1=18"
        fhconv.tune_clear()
        assert fhconv.parse_tune(out) == 2 and fhconv.format_tune() == out
        fhconv.tune_clear()
        assert fhconv.parse_tune("") == 0 and fhconv.parse_tune("garbage") == 0
    finally:
        fhconv.tune_clear()


# the conv layers the planner has to serve: the configs' layers and the FlyHighFG layer shapes
SHAPES = [
    (1, 136, 240, 32, 32, 3, 1), (1, 544, 960, 32, 64, 3, 2), (1, 272, 480, 64, 64, 3, 1),
    (1, 68, 120, 128, 128, 3, 1), (1, 68, 120, 128, 64, 1, 1), (1, 120, 216, 3, 36, 3, 2),
    (1, 60, 108, 36, 36, 3, 1), (1, 60, 108, 36, 72, 3, 2), (1, 30, 54, 72, 72, 3, 1), (1, 30, 54, 279, 96, 3, 1),
    (1, 30, 54, 96, 96, 3, 1), (1, 30, 54, 96, 12, 3, 1), (1, 60, 108, 155, 48, 3, 1), (1, 60, 108, 48, 48, 3, 1),
    (1, 60, 108, 48, 7, 3, 1), (1, 60, 108, 48, 5, 3, 1), (1, 60, 108, 48, 36, 3, 1), (1, 120, 216, 14, 24, 3, 1),
    (1, 120, 216, 24, 24, 3, 1), (1, 120, 216, 24, 3, 3, 1), (8, 120, 216, 3, 36, 3, 2),
]


def test_direct_kernel_where_the_channels_fit():
    # small-channel layers go to the direct kernel (weights resident), deep ones to the deep-layer kernel where the
    # input view has 16-byte channel groups, else to the chunked kernel
    assert fhconv.plan_dry(fhconv.make_desc(1, 136, 240, 32, 32))["family"] == "direct"
    assert fhconv.plan_dry(fhconv.make_desc(1, 544, 960, 32, 64, stride=2))["family"] == "direct"
    assert fhconv.plan_dry(fhconv.make_desc(1, 68, 120, 128, 64, k=1))["family"] == "direct"
    deep = fhconv.plan_dry(fhconv.make_desc(1, 30, 54, 279, 96))  # one kernel row of K per wave
    assert deep["family"] == "direct" and deep["cc"] == 288 and deep["waves"][2] == 3
    assert fhconv.plan_dry(fhconv.make_desc(1, 60, 108, 72, 36, stride=2))["family"] == "igemm"
    assert fhconv.plan_dry(fhconv.make_desc(1, 30, 54, 300, 96))["family"] == "igemm"  # 300 % 8: no DMA path
    assert fhconv.plan_dry(fhconv.make_desc(1, 30, 54, 300, 96, x_cstride=304))["family"] == "gemm"
    assert fhconv.plan_dry(fhconv.make_desc(1, 68, 120, 128, 128))["name"] == "gemm.t8x16.n48.f2x3.w4x1.c32.p2"
    d = fhconv.plan_dry(fhconv.make_desc(1, 60, 108, 36, 36))
    assert d["family"] == "direct" and d["cc"] == 64 and d["tile_channels"] == 48 and d["ntn"] == 1


# (batch, cin, cout, input channel stride): 544 x 960 tensors of 2^31 bytes and more, past the deep-layer kernel's reach
@pytest.mark.parametrize("n,cin,cout,cs", [(24, 155, 48, 160), (16, 155, 64, 160), (24, 155, 128, 160), (16, 279, 32, 288),
                                           (8, 279, 128, 288), (16, 96, 48, 160)])
def test_tensors_past_the_deep_layer_kernels_reach_keep_the_direct_kernel(n, cin, cout, cs):
    d = fhconv.make_desc(n, 544, 960, cin, cout, x_cstride=cs)
    assert n * 544 * 960 * cs * 2 >= 2 ** 31
    assert fhconv.plan_dry(d)["family"] == "direct"


# (cin, cout, n, h, w, stride), the input's and the output's (channel stride, offset), and the variant measured faster:
# one shape inside each of the planner's lines, and one past each that has a far side
MEASURED = [
    ((72, 38, 10, 167, 281, 1), (72, 0), (38, 0), "gemm.t8x16.n48.f2x3.w4x1.c32.p2"),
    ((72, 36, 10, 167, 281, 1), (72, 0), (38, 0), "gemm.t8x16.n48.f2x3.w4x1.c32.p2"),
    ((128, 16, 1, 97, 204, 1), (128, 0), (16, 0), "direct.c128.t2x4.n16"),
    ((100, 12, 3, 114, 145, 1), (103, 1), (16, 0), "direct.c128.t2x4.n16"),
    ((100, 12, 1, 122, 115, 1), (104, 0), (16, 0), "direct.c128.t1x2.n16"),
    ((128, 18, 5, 403, 363, 1), (128, 0), (22, 0), "direct.c128.t2x4.n16"),
    ((102, 18, 1, 85, 123, 1), (104, 0), (21, 1), "direct.c128.t1x2.n32"),
    ((100, 48, 5, 50, 32, 1), (103, 1), (48, 0), "direct.c128.t1x2.n48"),
    ((126, 38, 1, 82, 125, 1), (128, 0), (40, 0), "direct.c128.t2x4.n16"),
    ((102, 38, 13, 28, 37, 1), (105, 1), (41, 1), "direct.c128.t2x4.n16"),
    ((126, 36, 22, 19, 39, 1), (128, 0), (40, 0), "gemm.t8x16.n48.f2x3.w4x1.c32.p2"),
    ((24, 32, 12, 37, 56, 1), (24, 0), (34, 0), "direct.c32.t1x2.n32"),
    ((24, 18, 1, 182, 300, 1), (24, 0), (24, 0), "direct.c32.t4x2.n32"),
    ((14, 36, 10, 216, 403, 1), (17, 1), (40, 0), "direct.c32.t2x1.n48"),
    ((9, 130, 2, 102, 208, 1), (12, 2), (134, 0), "direct.c32.t4x2.n32"),
    ((16, 112, 19, 33, 24, 1), (19, 1), (115, 1), "direct.c32.t2x1.n32"),
    ((64, 24, 5, 64, 71, 1), (64, 0), (24, 0), "direct.c64.t2x1.n32"),
    ((33, 36, 11, 36, 76, 1), (35, 1), (39, 1), "direct.c64.t2x1.n48"),
    ((48, 64, 8, 175, 349, 1), (51, 1), (67, 1), "direct.c64.t2x1.n64"),
    ((64, 128, 9, 38, 58, 1), (67, 1), (128, 0), "direct.c64.t2x1.n48"),
    ((66, 7, 8, 421, 385, 1), (72, 0), (9, 1), "direct.c96.t2x4.n16"),
    ((72, 16, 8, 53, 44, 1), (72, 0), (16, 0), "direct.c96.t2x1.n16/rows"),
    ((66, 18, 18, 45, 34, 1), (72, 0), (22, 0), "direct.c96.t2x1.n32"),
    ((90, 24, 11, 143, 145, 1), (93, 1), (24, 0), "direct.c96.t4x2.n32"),
    ((90, 48, 8, 30, 42, 1), (96, 0), (48, 0), "direct.c96.t2x1.n48"),
    ((72, 36, 21, 20, 36, 1), (75, 1), (36, 0), "direct.c96.t2x1.n48"),
    ((72, 38, 2, 188, 214, 1), (72, 0), (40, 0), "gemm.t8x16.n48.f2x3.w4x1.c32.p2"),
    ((72, 52, 4, 23, 47, 1), (75, 1), (56, 0), "direct.c96.t1x2.n64"),
    ((72, 84, 4, 52, 51, 1), (72, 0), (88, 0), "gemm.t8x16.n48.f2x3.w4x1.c32.p2"),
    ((96, 160, 2, 275, 290, 1), (96, 0), (163, 1), "direct.c96.t4x2.n32"),
    ((72, 72, 2, 398, 438, 1), (75, 1), (72, 0), "direct.c96.t4x2.n32"),
    ((279, 52, 12, 31, 21, 1), (280, 0), (56, 0), "gemm.t8x16.n48.f2x3.w4x1.c32.p2"),
    ((160, 52, 1, 162, 338, 1), (160, 0), (56, 0), "gemm.t8x16.n64.f4x2.w2x2.c32.p2"),
    ((258, 256, 3, 178, 131, 1), (264, 0), (256, 0), "gemm.t8x16.n64.f4x2.w2x2.c32.p2"),
    ((288, 130, 2, 186, 220, 1), (288, 0), (136, 0), "gemm.t8x16.n48.f2x3.w4x1.c32.p2"),
    ((288, 36, 2, 175, 343, 1), (288, 0), (36, 0), "gemm.t16x16.n48.f4x3.w4x1.c32.p2"),
    ((160, 36, 1, 242, 515, 1), (160, 0), (39, 1), "gemm.t8x16.n48.f2x3.w4x1.c32.p2"),
    ((288, 16, 8, 94, 173, 1), (288, 0), (18, 0), "gemm.t8x16.n32.f4x2.w2x1.c32.p2"),
    ((128, 64, 2, 552, 683, 1), (128, 0), (64, 0), "direct.c128.t4x1.n64/p"),
    ((24, 128, 1, 595, 682, 1), (24, 0), (128, 0), "direct.c32.t8x1.n64/p"),
    ((33, 64, 4, 218, 194, 1), (40, 0), (64, 0), "direct.c64.t4x1.n64/p"),
    ((90, 56, 1, 456, 546, 1), (96, 0), (56, 0), "direct.c96.t4x1.n64/p"),
    ((160, 12, 2, 157, 117, 1), (160, 0), (16, 0), "direct.c160.t2x1.n16/rows"),
    ((130, 24, 2, 55, 50, 1), (136, 0), (26, 0), "direct.c160.t2x1.n32/rows"),
    ((279, 12, 1, 96, 66, 1), (280, 0), (12, 0), "direct.c288.t2x1.n16/rows"),
    ((288, 5, 2, 102, 139, 1), (288, 0), (8, 0), "gemm.t8x16.n48.f2x3.w4x1.c32.p2"),
    ((64, 16, 3, 10, 8, 1), (64, 0), (16, 0), "direct.c64.t1x1.n16/rows"),
    ((33, 30, 1, 9, 14, 1), (36, 2), (32, 0), "direct.c64.t1x1.n32/rows"),
    ((64, 48, 5, 10, 18, 1), (67, 1), (51, 1), "direct.c64.t1x1.n48/rows"),
    ((48, 192, 1, 10, 21, 1), (48, 0), (192, 0), "direct.c64.t1x1.n48/rows"),
    ((33, 56, 15, 9, 18, 1), (40, 0), (58, 0), "direct.c64.t1x2.n64"),
    ((90, 16, 8, 22, 23, 1), (96, 0), (19, 1), "direct.c96.t1x1.n16/rows"),
    ((90, 18, 23, 9, 8, 1), (93, 1), (22, 0), "direct.c96.t1x1.n32/rows"),
    ((66, 48, 1, 31, 56, 1), (69, 1), (48, 0), "direct.c96.t1x1.n48/rows"),
    ((72, 52, 5, 17, 29, 1), (72, 0), (54, 0), "direct.c96.t1x1.n48/rows"),
    ((96, 56, 5, 19, 35, 1), (99, 1), (56, 0), "direct.c96.t1x2.n64"),
    ((14, 144, 6, 339, 256, 2), (16, 0), (144, 0), "direct.s2.c32.t4x1.n64/p"),
    ((36, 192, 8, 219, 358, 2), (40, 0), (192, 0), "direct.s2.c64.t2x2.n64/p"),
    ((3, 128, 6, 173, 155, 2), (6, 2), (128, 0), "direct.s2.c32.t2x1.n64"),
    ((63, 72, 2, 162, 142, 2), (64, 0), (72, 0), "direct.s2.c64.t2x1.n48"),
    ((48, 98, 2, 345, 739, 2), (51, 1), (100, 0), "direct.s2.c64.t2x2.n64"),
]


@pytest.mark.parametrize("shape,xv,yv,name", MEASURED, ids=lambda v: v if isinstance(v, str) else "x".join(map(str, v)))
def test_the_planner_takes_the_measured_variant(shape, xv, yv, name):
    cin, cout, n, h, w, stride = shape
    d = fhconv.make_desc(n, h, w, cin, cout, stride=stride, x_cstride=xv[0], x_c0=xv[1], y_cstride=yv[0], y_c0=yv[1])
    assert fhconv.plan_dry(d)["name"] == name
    d.ksplit = 1  # a fixed K split keeps the one-chain K order: no resident loop
    assert not fhconv.plan_dry(d)["name"].endswith("/p")


@pytest.mark.parametrize("shape", SHAPES)
def test_mi355x_plan_covers_the_output(shape):
    n, h, w, cin, cout, k, s = shape
    p = fhconv.plan_dry(fhconv.make_desc(n, h, w, cin, cout, k=k, stride=s))
    assert p["hout"] == (h + 2 * (k == 3) - k) // s + 1 and p["wout"] == (w + 2 * (k == 3) - k) // s + 1
    tiles = -(-p["hout"] // p["tile_rows"]) * -(-p["wout"] // 16) * n
    assert p["tiles"] == tiles
    assert p["ntn"] * p["tile_channels"] >= cout > (p["ntn"] - 1) * p["tile_channels"]
    assert p["cc"] % 8 == 0 and p["cc"] * p["nchunks"] >= cin and p["cc"] * (p["nchunks"] - 1) < cin
    if p["family"] == "igemm":
        assert p["grid"][0] == tiles * p["ntn"]
        assert p["ksteps"] * 32 >= k * k * p["cc"]
    elif p["family"] == "gemm":  # deep-layer kernel: one workgroup per tile and channel tile, chunks of 32 or 64
        assert p["grid"] == [tiles, p["ntn"], 1] and k == 3 and s == 1
        assert p["cc"] in (32, 64) and p["ksteps"] * 32 == 9 * p["cc"]
    else:
        assert p["grid"][1] == p["ntn"] and 1 <= p["grid"][0] <= tiles
        assert p["cc"] % 32 == 0 and p["ksteps"] * 32 == k * k * p["cc"] and p["nchunks"] == 1
    assert p["lds"] <= 64 * 1024
    assert p["flops"] == 2 * n * p["hout"] * p["wout"] * cout * cin * k * k
    name = fhconv.variant_name(p["variant"])
    assert name == p["name"]


def test_variant_list_and_forced_variants():
    d = fhconv.make_desc(1, 68, 120, 128, 128)
    codes = fhconv.variant_list(d)
    assert len(codes) >= 4 and len(set(codes)) == len(codes)
    for code in codes:
        p = fhconv.plan_dry(fhconv.make_desc(1, 68, 120, 128, 128, variant=code))
        assert p["variant"] == code
    split = [c for c in codes if c < 128 and c >> 5]
    assert split, "a 68x120 layer has a small tile grid: split-K variants are listed"
    with pytest.raises(fhconv.FhcError):
        fhconv.plan_dry(fhconv.make_desc(1, 68, 120, 128, 128, variant=31))


@pytest.mark.parametrize("cin,cs,c0", [(130, 130, 0), (100, 102, 2), (258, 262, 4)])
def test_a_view_of_channel_pairs_takes_its_own_plans_code(cin, cs, c0):
    # the deep-layer kernel reads views of channel pairs by dword-aligned loads, so its codes are listed (and timed by
    # autotune) on them, can be forced and stay what they are when the table names them; an odd view has none
    shape, view = (2, 47, 51, cin, 68), dict(x_cstride=cs, x_c0=c0)
    fhconv.tune_clear()
    try:
        codes = {c: fhconv.variant_name(c) for c in fhconv.variant_list(fhconv.make_desc(*shape, **view))}
        deep = [c for c in codes if codes[c].startswith("gemm")]
        assert deep and fhconv.plan_dry(fhconv.make_desc(*shape, **view))["variant"] in codes
        for code in deep:
            assert fhconv.plan_dry(fhconv.make_desc(*shape, variant=code, **view))["variant"] == code
            fhconv.parse_tune(f"{cin},68,47,51,1,2,3={code}")
            assert fhconv.plan_dry(fhconv.make_desc(*shape, **view))["variant"] == code
        odd = fhconv.make_desc(*shape, variant=deep[0], x_cstride=cs + 1, x_c0=c0)
        with pytest.raises(fhconv.FhcError, match="channel pairs"):
            fhconv.plan_dry(odd)
    finally:
        fhconv.tune_clear()


# (cin, cout, n, h, w, deep-layer kernel): both sides of each line for views of channel pairs, cin + 2 channels apart
@pytest.mark.parametrize("cin,cout,n,h,w,deep", [
    (124, 144, 1, 329, 249, True), (100, 52, 1, 85, 52, False), (124, 16, 2, 100, 200, False),
    (130, 48, 4, 208, 388, True), (130, 48, 2, 61, 61, False), (160, 64, 14, 91, 144, False), (130, 72, 2, 47, 51, True),
    (288, 36, 4, 113, 130, True), (288, 12, 2, 282, 187, False), (288, 24, 2, 46, 72, False),
    (200, 60, 18, 134, 198, False), (200, 48, 18, 134, 198, True), (256, 80, 2, 134, 198, True),
    (256, 16, 2, 400, 300, False), (512, 128, 1, 64, 80, True), (512, 256, 1, 767, 683, False),
    (90, 52, 2, 134, 198, False), (90, 20, 2, 134, 198, False)])
def test_channel_pairs_take_the_deep_layer_kernel_where_it_is_faster(cin, cout, n, h, w, deep):
    d = fhconv.make_desc(n, h, w, cin, cout, x_cstride=cin + 2, y_cstride=cout + 1)  # off the resident grids
    assert (fhconv.plan_dry(d)["family"] == "gemm") == deep, fhconv.plan_dry(d)["name"]
    d.ksplit = 1  # a fixed K split keeps the choice such a view always had
    assert fhconv.plan_dry(d)["family"] != "gemm"


def test_forced_split_k_and_reference_hint():
    p = fhconv.plan_dry(fhconv.make_desc(1, 68, 120, 128, 128, ksplit=4))
    np_ = -(-128 // p["tile_channels"]) * p["tile_channels"]
    assert p["ksplit"] == 4 and p["grid"][1 if p["family"] == "igemm" else 2] == 4
    assert p["workspace_bytes"] == 4 * 68 * 120 * np_ * 4  # f32 partials [z][pixel][np]
    assert p["nchunks"] % 4 == 0
    h = fhconv.plan_dry(fhconv.make_desc(1, 68, 120, 128, 128, ref_cand=fhconv.CAND_TILED | 2 << 4))
    assert h["ksplit"] == 2
    none = fhconv.plan_dry(fhconv.make_desc(1, 68, 120, 128, 128))
    assert none["ksplit"] == 1 and none["workspace_bytes"] == 0


def test_tune_table_keys_batch_and_kernel_size():
    # the batch and the kernel size extend the reference's key: the batch-1 3x3 entry keeps the reference's 5
    # fields, a batched or 1x1 entry carries n and k, and none of them overwrites another
    fhconv.tune_clear()
    try:
        text = "48,48,60,108,1=18\n48,48,60,108,1,24,3=17\n48,48,60,108,1,1,1=130\n48,48,60,108,1,0,3=5\n" \
               "48,48,60,108,1,2,5=5\n48,48,60,108,1,2=5\n"
        assert fhconv.parse_tune(text) == 3
        assert fhconv.tune_get(48, 48, 60, 108, 1) == 18
        assert fhconv.tune_get(48, 48, 60, 108, 1, n=24) == 17
        assert fhconv.tune_get(48, 48, 60, 108, 1, k=1) == 130
        assert fhconv.tune_get(48, 48, 60, 108, 1, n=8) is None
        out = fhconv.format_tune()
        assert out == "48,48,60,108,1,1,1=130\n48,48,60,108,1,24,3=17\n48,48,60,108,1=18"
        fhconv.tune_clear()
        assert fhconv.parse_tune(out) == 3 and fhconv.format_tune() == out
        # the planner looks the descriptor's own batch up
        d1, d24 = fhconv.make_desc(1, 60, 108, 48, 48), fhconv.make_desc(24, 60, 108, 48, 48)
        codes = fhconv.variant_list(d24)
        fhconv.tune_clear()
        fhconv.parse_tune(f"48,48,60,108,1,24,3={codes[0]}\n48,48,60,108,1={codes[1]}")
        assert fhconv.plan_dry(d24)["variant"] == codes[0]
        assert fhconv.plan_dry(d1)["variant"] == codes[1]
    finally:
        fhconv.tune_clear()


def test_the_table_steers_the_planner():
    fhconv.tune_clear()
    try:
        d = fhconv.make_desc(1, 136, 240, 32, 32)
        default = fhconv.plan_dry(d)["variant"]
        other = [c for c in fhconv.variant_list(d) if c != default][0]
        fhconv.parse_tune(f"32,32,136,240,1={other}")
        assert fhconv.plan_dry(d)["variant"] == other
    finally:
        fhconv.tune_clear()


def test_tune_table_takes_variant_names():
    # a committed table names variants (stable across builds); the parser maps each name to this build's code
    fhconv.tune_clear()
    try:
        d = fhconv.make_desc(1, 60, 108, 48, 48)
        names = {fhconv.variant_name(c): c for c in fhconv.variant_list(d)}
        name = sorted(names)[0]
        assert fhconv.parse_tune(f"48,48,60,108,1={name}\n48,48,60,108,2=no.such.variant\n") == 1
        assert fhconv.tune_get(48, 48, 60, 108, 1) == names[name]
        assert fhconv.tune_get(48, 48, 60, 108, 2) is None
        assert f"48,48,60,108,1={names[name]}" in fhconv.format_tune()
        assert fhconv.plan_dry(d)["name"] == name
    finally:
        fhconv.tune_clear()


def test_committed_choice_table_parses():
    # every line of the shipped MI355X table names a variant this build has
    path = os.path.join(os.path.dirname(os.path.abspath(__file__)), "..", "flyhigh-engine_amd", "tune_mi355x.txt")
    text = open(path).read()
    fhconv.tune_clear()
    try:
        assert fhconv.parse_tune(text) == len([ln for ln in text.splitlines() if ln.strip()])
    finally:
        fhconv.tune_clear()
