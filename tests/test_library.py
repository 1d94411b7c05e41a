"""The C ABI library: it loads without a GPU and exports every entry point
that include/fimhip.h declares; the host-side glue behaves on bad input."""
import ctypes as ct
import os
import re

import numpy as np
import pytest

from fimocn_subx_realtime_hera_apr2020_amd import fimhip, glvl, state
from helpers import golden_grid

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def declared_symbols():
    txt = open(os.path.join(ROOT, "include", "fimhip.h")).read()
    return sorted(set(re.findall(r"\b(fimhip_[a-z0-9_]+)\s*\(", txt)))


def test_header_and_python_agree():
    assert declared_symbols() == sorted(fimhip.EXPORTS)


def test_library_exports_every_declared_symbol():
    lib = fimhip.load_library()
    for s in declared_symbols():
        assert hasattr(lib, s), s


def test_host_side_pow_is_the_device_routine():
    lib = fimhip.load_library()
    assert lib.fimhip_pow(2.0, 10.0) == 1024.0
    assert b"gfx950" in lib.fimhip_version()


def test_create_rejects_bad_sizes_without_gpu_calls():
    lib = fimhip.load_library()
    gd = fimhip.GridDesc()
    gd.nip, gd.nvl, gd.ntra, gd.dt = 10, 64, 4, 240.0
    h = ct.c_void_p()
    assert lib.fimhip_create(ct.byref(gd), 0, ct.byref(h)) == -1
    gd.nip, gd.nvl = 642, 65
    assert lib.fimhip_create(ct.byref(gd), 0, ct.byref(h)) == -1
    assert lib.fimhip_create(None, 0, ct.byref(h)) == -1


def test_every_entry_rejects_a_null_handle_without_gpu_calls():
    """Every entry point that takes an instance handle returns
    FIMHIP_EINVAL (-1) for a null one, with null arrays and zero sizes, and
    touches no device (this runs without a GPU)."""
    lib = fimhip.load_library()
    no_handle = {"fimhip_create", "fimhip_ens_create", "fimhip_icos_grid", "fimhip_icos_grid_info",
                 "fimhip_pow", "fimhip_ens_kernel_count", "fimhip_ens_kernel_name", "fimhip_synth_state",
                 "fimhip_version"}
    checked = 0
    for name in fimhip.EXPORTS:
        if name in no_handle:
            continue
        f = getattr(lib, name)
        assert f.argtypes, name
        args = [0.0 if t in (ct.c_double, ct.c_float) else 0 if t in (ct.c_int, ct.c_int64, ct.c_size_t) else None
                for t in f.argtypes]
        assert f(*args) == -1, name
        checked += 1
    assert checked >= 50


def test_glvl_roundtrip(tmp_path):
    g = golden_grid(2)
    p = tmp_path / "glvl.dat"
    glvl.write_glvl(g, str(p))
    assert p.read_bytes() == open(os.path.join(ROOT, "tests", "golden", "glvl_G2.dat"), "rb").read()


def test_state_generator_is_batch_invariant():
    g = golden_grid(3)
    a = state.make_state(g.lat, g.lon, 64, 4, wind_noise=True, perturb=True, member=3)
    b = state.make_state(g.lat[:100], g.lon[:100], 64, 4, wind_noise=True, perturb=True, member=3)
    for k in ("us", "dp"):
        assert np.array_equal(a[k][:100], b[k])
    c = state.make_state(g.lat, g.lon, 64, 4, wind_noise=True, perturb=True, member=4)
    assert not np.array_equal(a["us"], c["us"])


def test_kernel_numbers_of_the_launch_shapes_stay():
    """fimhip_ens_set_tile takes a kernel's number, and launch shapes are kept
    by number or name: a kernel that goes leaves its number behind."""
    from fimocn_subx_realtime_hera_apr2020_amd import fimhip
    lib = fimhip.load_library()
    names = [lib.fimhip_ens_kernel_name(k).decode() for k in range(lib.fimhip_ens_kernel_count())]
    assert names == ["e_edgvar1", "e_edgvar3", "e_cnuity12", "e_cnuity3", "e_cnuity45", "e_trcadv12", "e_trcadv2",
                     "e_trcadv3", "e_momtum", "e_hystat", "e_massadv1", "e_massadv2", "e_trc_fct"]
    set_to = {}
    shape = type("Shape", (), dict(kernel_names=lambda self: names, h=None, lib=type("Lib", (), dict(
        fimhip_ens_set_tile=staticmethod(lambda h, k, t: set_to.update({k: t}) or 0)))()))()
    fimhip.Ensemble.set_tiles(shape, {"e_trcadv1": 5, "e_trcadv2": 3, "e_momtum": 6})
    assert set_to == {5: 5, 6: 3, 8: 6}


def test_bench_prints_a_line_that_a_logs_tail_holds():
    """Whatever the legs report, the line has the headline's keys and fits into
    2000 characters."""
    import json
    import sys
    sys.path.insert(0, ROOT)
    import bench
    leg = {"value": 1.0 / 3, "ms_per_step": 2.0 / 3, "kernels": {"k%d" % i: {"ms": 1.0 / 7} for i in range(200)}}
    out = {"metric": "m" * 70, "value": 1e10 / 3, "unit": "u", "n_gpus": 1, "steps": 20, "warmup": 5, "ms_per_step": 1.0 / 3,
           "higher_is_better": True, "scaling": "weak", "vs_baseline": None, "dtype": "f32+f64", "data": "d" * 60,
           "config": {"workload": "w" * 170, "dt_note": "n" * 200, "nip": 163842},
           "roofline": {"bound": "hbm", "achieved": 1.0 / 3, "frac": 1.0 / 7, "kernels": leg["kernels"]},
           "dominant_kernel": {"kernel": "e_trcadv12", "mean_launch_ms": 1.0 / 3}, "speedup_vs_plain_fp64": 2.0 / 3,
           "plain_fp64": leg, "ensemble": leg, "uneven_batch": {"mixed": leg, "fp64": leg},
           "hycom": dict({"n%d" % i: leg for i in range(6)}, workload="w"),
           "accuracy_96": {"rel_l2_vs_fp64": {"us": 1e-4 / 3, "vs": 2e-4 / 3}}, "cpu_baseline": leg}
    for drop in ((), ("plain_fp64", "uneven_batch", "hycom", "accuracy_96", "cpu_baseline")):
        line = bench.headline({k: None if k in drop else v for k, v in out.items()})
        assert len(json.dumps(line)) < 1900
        for k in ("metric", "value", "unit", "n_gpus", "steps", "warmup", "ms_per_step", "higher_is_better", "scaling",
                  "vs_baseline", "dtype", "data", "config"):
            assert k in line, k
        assert line["value"] == 3333333000.0 and line["config"]["nip"] == 163842


def test_incremental_build_sees_every_header():
    """A source is compiled again when a header is newer than its object: the
    list of headers is the folder's."""
    from fimocn_subx_realtime_hera_apr2020_amd import build
    assert sorted(build.HEADERS) == sorted(f for f in os.listdir(build.CSRC) if f.endswith(".h"))
