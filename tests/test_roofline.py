"""The roofline accounting reads each entry point's sizes from the right argument positions:
for every entry point with a work function, the size parameters are located by name in
include/flashuma.h and the work computed from a call with distinct sizes is checked against
the formula stated for it."""
import os
import re

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
HEADER = os.path.join(ROOT, "include", "flashuma.h")


def _params(name):
    text = re.sub(r"/\*.*?\*/", "", open(HEADER).read(), flags=re.S)
    m = re.search(r"\b" + name + r"\s*\(([^)]*)\)\s*;", text)
    assert m, name
    return [p.split()[-1].lstrip("*") for p in m.group(1).split(",")]


def _args(name, **sizes):
    params = _params(name)
    args = [0] * len(params)
    for key, val in sizes.items():
        args[params.index(key)] = val
    return tuple(args)


GEMMS = {
    # entry point: (sizes, algorithmic flops)
    "fu_linear": (dict(M=1000, N=384, K=640), 2 * 1000 * 384 * 640),
    "fu_linear_batched": (dict(M=1000, N=128, K=256, batch=5), 2 * 5 * 1000 * 128 * 256),
    "fu_linear_gate": (dict(M=1000, C=128, K=768, lmax=2), 2 * 1000 * 640 * 768),
    "fu_linear_gate_bwd": (dict(M=1000, C=128, K=384, lmax=2), 2 * 1000 * 384 * 384),
    "fu_complex_linear": (dict(M=1000, Nc=256, Kc=512), 6 * 1000 * 256 * 512),
    "fu_complex_linear_gate": (dict(M=1000, Nc=256, Kc=512), 6 * 1000 * 256 * 512),
    "fu_complex_linear_gate_bwd": (dict(M=1000, Nc=128, Kc=256), 6 * 1000 * 128 * 256),
    "fu_linear_ln_silu": (dict(M=1000, N=128, K=128, batch=5, G=5), 2 * 5 * 1000 * 128 * 128),
    "fu_linear_ln_silu_bwd": (dict(M=1000, N=640, K=64, G=5), 2 * 1000 * 640 * 64),
    "fu_linear_dgrad_ln_silu_bwd": (dict(M=1000, K=1536, G=5, group=2), 2 * 1000 * 128 * 1536),
    "fu_gather_linear_gate": (dict(E=1000, C=128), 2 * 1000 * 640 * 768),
}


@pytest.mark.parametrize("name", sorted(GEMMS))
def test_gemm_work_reads_the_size_arguments(name):
    import roofline
    sizes, flops = GEMMS[name]
    nbytes, got = roofline.WORK[name](_args(name, **sizes))
    assert got == flops
    assert nbytes > 0


def test_every_work_function_names_a_declared_entry_point():
    import roofline
    text = open(HEADER).read()
    for name in roofline.WORK:
        assert re.search(r"\b" + name + r"\s*\(", text), name


def test_split_mode_accounting():
    import roofline
    args = _args("fu_linear", M=1000, N=384, K=640)
    flops = 2 * 1000 * 384 * 640
    ms = 1.0
    split = roofline.summarize([("fu_linear", args, ms)], roofline.MATMUL_SPLIT_BF16)["fu_linear"]
    fp32 = roofline.summarize([("fu_linear", args, ms)], roofline.MATMUL_FP32)["fu_linear"]
    f16 = roofline.summarize([("fu_linear", args, ms)], roofline.MATMUL_SPLIT_F16)["fu_linear"]
    rate = flops / 1e-3 / 1e12
    assert fp32["peak"] == 157.3 and abs(fp32["achieved"] - rate) < 0.01
    assert split["peak"] == 2500.0 and abs(split["achieved"] - 6 * rate) < 0.05
    assert f16["peak"] == 2500.0 and abs(f16["achieved"] - 3 * rate) < 0.05 and "fp16" in f16["matrix_op"]
    assert abs(split["fp32_tflops"] - rate) < 0.01 and abs(f16["fp32_tflops"] - rate) < 0.01
    # the gathered conv1 loader keeps the bf16 split in both split modes
    g = _args("fu_gather_linear_gate", E=1000, C=128)
    gf = roofline.summarize([("fu_gather_linear_gate", g, ms)], roofline.MATMUL_SPLIT_F16)["fu_gather_linear_gate"]
    assert "bf16" in gf["matrix_op"]


def test_roofline_frac_takes_the_larger_of_the_two_bounds():
    """roofline_frac = sum over launches of max(executed flops / matrix peak, bytes / HBM peak)
    over the measured time: equal to frac for a high-intensity GEMM, larger where the launch
    sits under the HBM slope (K = 128 with as many output columns as input)."""
    import roofline
    big = _args("fu_linear", M=245760, N=640, K=768)
    small = _args("fu_linear_batched", M=245760, N=128, K=128, batch=5)
    ms = 1.0
    r = roofline.summarize([("fu_linear", big, ms)])["fu_linear"]
    assert r["hbm_bound_launches"] == 0 and abs(r["roofline_frac"] - r["frac"]) < 1e-3
    nbytes, flops = roofline.WORK["fu_linear_batched"](small)
    t_hbm = nbytes / (roofline.HBM_PEAK_GBS * 1e9)
    t_mfma = 6 * flops / (roofline.BF16_MFMA_PEAK_TFLOPS * 1e12)
    assert t_hbm > t_mfma
    r = roofline.summarize([("fu_linear_batched", small, ms)])["fu_linear_batched"]
    assert r["hbm_bound_launches"] == 1 and abs(r["roofline_frac"] - t_hbm / 1e-3) < 1e-3


@pytest.mark.parametrize("name,sizes,per_edge", [
    ("fu_scatter_bwd", dict(E=1000, N=50, C=128), (34 + 1) * 4),
    ("fu_init_scatter_bwd", dict(E=1000, N=50, C=128), (8 + 1) * 4),
    ("fu_gather_bwd", dict(E=1000, N=50, C=128), 34 * 4),
])
def test_accumulating_calls_count_the_read_back(name, sizes, per_edge):
    import roofline
    b0, _ = roofline.WORK[name](_args(name, **sizes, accumulate=0))
    b3, _ = roofline.WORK[name](_args(name, **sizes, accumulate=3))
    assert b3 - b0 == sizes["E"] * per_edge


# entry points without a work function: set-up, graph building, queries, and node- or system-sized
# copies and norms (none of them carries a step's edge work)
UNCOUNTED = {
    "fu_version", "fu_last_error", "fu_set_matmul_mode", "fu_matmul_mode", "fu_complex_weight_split_bytes",
    "fu_complex_weight_split", "fu_linear_weight_split_bytes", "fu_linear_weight_split", "fu_radial_gather_perm",
    "fu_radial_gather_perm_lmax", "fu_rms_norm_sh_fwd", "fu_rms_norm_sh_bwd", "fu_gate_act_fwd", "fu_gate_act_bwd",
    "fu_balance_channels", "fu_balance_channels_noalloc", "fu_gather_rows", "fu_scatter_rows", "fu_edge_shifts",
    "fu_outer_sum3", "fu_morton_keys", "fu_sort_pairs_i64", "fu_invert_perm", "fu_take_i64", "fu_csr_row_ptr",
    "fu_narrow_i64_i32", "fu_nlist_bin", "fu_nlist_search", "fu_nlist_scan", "fu_nlist_limits", "fu_nlist_emit",
    "fu_wigner_ext_width"}


def test_every_entry_point_is_counted_or_named_as_not():
    """A new entry point cannot drop out of the per-kernel table silently."""
    import roofline
    from ops import _lib
    assert set(_lib.SIGNATURES) == set(roofline.WORK) | UNCOUNTED
    assert not set(roofline.WORK) & UNCOUNTED


@pytest.mark.parametrize("L,C,E", [(2, 128, 859), (3, 64, 77), (4, 256, 40)])
def test_pair_work_is_that_of_its_tiled_calls(L, C, E):
    """The pair's products are those of the tiled entry points it replaces, forward and backward; its bytes
    leave out the gated Z (forward) and g_Y and the gate sums (backward), written and read in between."""
    import roofline
    W = lambda name, **s: roofline.WORK[name](_args(name, **s))
    n = (L + 1, L, L - 1)
    fwd = [W("fu_linear_gate", M=E, C=C, K=2 * n[0] * C, lmax=L), W("fu_linear", M=E, N=n[0] * C, K=n[0] * C)]
    fwd += [W("fu_complex_linear_gate", M=E, Nc=k * C, Kc=2 * k * C) for k in n[1:]]
    fwd += [W("fu_complex_linear", M=E, Nc=k * C, Kc=k * C) for k in n[1:]]
    bwd = [W("fu_linear_gate_bwd", M=E, C=C, K=n[0] * C, lmax=L), W("fu_linear", M=E, N=2 * n[0] * C, K=(2 * L + 1) * C)]
    bwd += [W("fu_complex_linear_gate_bwd", M=E, Nc=k * C, Kc=k * C) for k in n[1:]]
    bwd += [W("fu_complex_linear", M=E, Nc=2 * k * C, Kc=k * C) for k in n[1:]]
    for name, parts in (("fu_so2_pair_fwd", fwd), ("fu_so2_pair_bwd", bwd)):
        nbytes, flops = W(name, E=E, C=C, lmax=L)
        assert flops == sum(p[1] for p in parts)
        assert 0 < nbytes < sum(p[0] for p in parts)
        rec = roofline.summarize([(name, _args(name, E=E, C=C, lmax=L), 0.1)])[name]
        assert rec["bound"] == "mfma" and "fp16" in rec["matrix_op"]


def test_few_row_and_batched_shift_work():
    import roofline
    W = lambda name, **s: roofline.WORK[name](_args(name, **s))
    assert W("fu_linear_short", M=900, N=64, K=640) == W("fu_linear", M=900, N=64, K=640)
    assert W("fu_edge_shifts_batched", E=1000, S=7) == (24000 + 7 * 44 + 8, 0)
    assert W("fu_outer_sum3_batched", E=1000, S=7) == (24000 + 7 * 44 + 8, 0)


def test_sixteen_row_tiles_are_counted_as_fp32_products():
    """fu_linear_batched on its 16-row tiles runs the fp32 matrix instructions; the line is the kernel's."""
    import roofline
    src = open(os.path.join(ROOT, "flash-uma_amd", "csrc", "gemm.hip")).read()
    assert "ROWS16_MAX_GROUPS = 512, ROWS16_MAX_BATCHED_ROWS = 512;" in src
    few, many = (_args("fu_linear_batched", M=m, N=128, K=128, batch=9) for m in (54, 8192))
    r = roofline.summarize([("fu_linear_batched", few, 1.0)])["fu_linear_batched"]
    assert r["matrix_op"] == "fp32 mfma" and r["peak"] == 157.3 and r["achieved"] == r["fp32_tflops"]
    r = roofline.summarize([("fu_linear_batched", many, 1.0)])["fu_linear_batched"]
    assert r["peak"] == 2500.0 and abs(r["achieved"] - 3 * r["fp32_tflops"]) < 0.01 + 1e-2 * r["achieved"]
    r = roofline.summarize([("fu_linear_batched", few, 1.0), ("fu_linear_batched", many, 1.0)])["fu_linear_batched"]
    assert 157.3 < r["peak"] < 2500.0 and "and" in r["matrix_op"]
