"""Which store form and block order the steps take (the headers' own rules on
the host): the lines that the measurements beside the rules draw, from both
sides.  What the forms compute is the same; tests/test_traffic.py compares
them on the GPU."""
from __future__ import annotations

import os
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
BYTES = {"f64": 8, "f32": 4, "f16": 2}
DISPATCH, RUNS_OF_8, RUNS_OF_32, CONTIGUOUS = 0, 3, 5, 31


@pytest.fixture(scope="module")
def plans(tmp_path_factory):
    exe = tmp_path_factory.mktemp("traffic") / "traffic_plan_check"
    subprocess.run(["/opt/rocm/bin/hipcc", "-O1", "-std=c++23", "--offload-arch=gfx950", "-x", "hip",
                    os.path.join(HERE, "traffic_plan_check.cpp"), "-o", str(exe)], check=True, capture_output=True,
                   timeout=300)

    def run(cases):
        """(streaming, order) of each (step, storage, (nx, ny, nz), Q, offset)."""
        text = "".join(f"{step} {BYTES[st]} {e[0]} {e[1]} {e[2]} {q} {off}\n" for step, st, e, q, off in cases)
        r = subprocess.run([str(exe)], input=text, capture_output=True, text=True, timeout=60)
        assert r.returncode == 0, r.stdout + r.stderr
        out = [tuple(int(v) for v in line.split()) for line in r.stdout.splitlines()]
        assert len(out) == len(cases)
        return [(bool(s), o) for s, o in out]

    return run


def test_planes_a_multiple_of_256_mib_apart_keep_the_dispatch_order(plans):
    apart = [("f16", (512, 512, 512)), ("f16", (1024, 1024, 128)), ("f16", (512, 512, 1024)), ("f64", (512, 512, 128))]
    others = [("f16", (256, 256, 256)), ("f16", (512, 512, 480)), ("f16", (512, 512, 256)), ("f16", (640, 640, 640)),
              ("f64", (256, 256, 256)), ("f64", (512, 512, 256))]
    cases = [("fluid", st, e, q, 0) for q in (19, 27) for st, e in apart]
    assert plans(cases) == [(True, DISPATCH)] * len(cases)
    cases = [("fluid", st, e, q, 0) for q in (19, 27) for st, e in others]
    assert plans(cases) == [(True, RUNS_OF_8)] * len(cases)
    cases = [("fluid", "f32", e, 19, 0) for e in ((512, 512, 512), (256, 256, 256), (192, 192, 192))]
    assert plans(cases) == [(True, DISPATCH)] * len(cases)


def test_2d_grids_run_contiguously_while_the_caches_hold_their_levels(plans):
    within = [("f32", (512, 512), 0, False), ("f32", (2048, 2048), 0, True), ("f32", (2048, 2048), 4, False),
              ("f16", (2880, 2880), 0, True), ("f64", (2048, 1024), 0, True), ("f64", (2093, 1026), 0, False)]
    got = plans([("fluid", st, e + (1,), 9, off) for st, e, off, _ in within])
    assert got == [(streaming, CONTIGUOUS) for *_, streaming in within]
    past = [("f32", (2048, 2112), 0, (True, RUNS_OF_8)), ("f32", (2048, 2304), 0, (True, RUNS_OF_8)),
            ("f64", (1536, 1536), 0, (True, DISPATCH)), ("f16", (3072, 3072), 0, (True, RUNS_OF_8)),
            ("f32", (2201, 2199), 0, (False, RUNS_OF_32)), ("f64", (1536, 1536), 8, (False, RUNS_OF_32))]
    assert plans([("fluid", st, e + (1,), 9, off) for st, e, off, _ in past]) == [want for *_, want in past]


def test_fused_steps_run_contiguously_only_where_their_planes_crowd_the_cache_sets(plans):
    crowded = [("f32", (2048, 2048, 1)), ("f64", (2048, 1024, 1)), ("f16", (4096, 2048, 1)), ("f16", (2880, 2880, 1)),
               ("f32", (128, 128, 128)), ("f32", (256, 256, 32)), ("f32", (112, 112, 112)), ("f64", (112, 112, 112)),
               ("f64", (256, 64, 64)), ("f16", (128, 128, 128)), ("f16", (112, 112, 224))]
    cases = [("fused", st, e, 9 if e[2] == 1 else 19, 0) for st, e in crowded]
    assert plans(cases) == [(True, CONTIGUOUS)] * len(cases)
    spread = [("f32", (1920, 1920, 1), (True, RUNS_OF_8)), ("f32", (2048, 2304, 1), (True, RUNS_OF_8)),
              ("f16", (3072, 3072, 1), (True, RUNS_OF_8)), ("f64", (1152, 1152, 1), (True, DISPATCH)),
              ("f32", (120, 120, 120), (True, DISPATCH)), ("f32", (136, 136, 136), (True, DISPATCH)),
              ("f16", (168, 168, 168), (True, RUNS_OF_8)), ("f64", (104, 104, 104), (True, RUNS_OF_8)),
              # crowded, but past the limit, or at two bytes in one or two groups
              ("f32", (2048, 4096, 1), (True, RUNS_OF_8)), ("f32", (256, 128, 128), (True, DISPATCH)),
              ("f16", (192, 256, 130), (True, RUNS_OF_8)), ("f16", (256, 256, 64), (True, DISPATCH))]
    assert plans([("fused", st, e, 9 if e[2] == 1 else 19, 0) for st, e, _ in spread]) == [want for *_, want in spread]
    cached = [("f32", (512, 512, 1)), ("f32", (1001, 701, 1)), ("f64", (64, 64, 64)), ("f32", (96, 96, 96))]
    got = plans([("fused", st, e, 9 if e[2] == 1 else 19, 0) for st, e in cached])
    assert got == [(False, CONTIGUOUS)] * 2 + [(False, RUNS_OF_32)] * 2
    # misaligned planes keep ordinary stores
    got = plans([("fused", "f32", e, 9 if e[2] == 1 else 19, 0)
                 for e in ((2049, 2047, 1), (1501, 1501, 1), (2501, 2499, 1), (129, 129, 129))])
    assert got == [(False, CONTIGUOUS)] + [(False, RUNS_OF_32)] * 3


def test_species_steps_follow_the_fluids_order_in_2d(plans):
    for step in ("reaction", "scalar"):
        cases = [("f32", (1920, 1920, 1), CONTIGUOUS), ("f32", (2048, 2048, 1), CONTIGUOUS),
                 ("f32", (2048, 2304, 1), RUNS_OF_8), ("f64", (1472, 1472, 1), DISPATCH),
                 ("f16", (3072, 3072, 1), RUNS_OF_8)]
        assert plans([(step, st, e, 9, 0) for st, e, _ in cases]) == [(True, order) for *_, order in cases], step
        assert plans([("fluid", st, e, 9, 0) for st, e, _ in cases[1:]]) == [(True, order) for *_, order in cases[1:]]
        assert plans([(step, "f32", (128, 128, 128), 19, 0), (step, "f32", (256, 128, 128), 19, 0)]) == \
            [(True, CONTIGUOUS)] * 2


def test_3d_species_steps_in_dispatch_order(plans):
    for step in ("reaction", "scalar"):
        cases = [("f64", (256, 256, 256), DISPATCH), ("f64", (256, 256, 192), DISPATCH), ("f64", (104, 104, 104), RUNS_OF_8),
                 ("f16", (320, 320, 320), DISPATCH), ("f16", (168, 168, 168), DISPATCH), ("f32", (192, 192, 192), DISPATCH),
                 ("f32", (120, 120, 120), RUNS_OF_8), ("f32", (144, 136, 144), DISPATCH),
                 ("f64", (128, 128, 128), CONTIGUOUS)]
        assert plans([(step, st, e, 19, 0) for st, e, _ in cases]) == [(True, order) for *_, order in cases], step


def test_misaligned_2d_species_steps_stream_while_that_pays(plans):
    cases = [("reaction", "f32", (1501, 1501, 1), (True, CONTIGUOUS)), ("scalar", "f32", (1801, 1799, 1), (True, CONTIGUOUS)),
             ("reaction", "f64", (1201, 1199, 1), (True, CONTIGUOUS)), ("scalar", "f32", (2049, 2047, 1), (True, CONTIGUOUS)),
             ("scalar", "f64", (1449, 1447, 1), (True, CONTIGUOUS)),
             ("reaction", "f64", (1449, 1447, 1), (False, CONTIGUOUS)), ("reaction", "f64", (1301, 1299, 1), (False, RUNS_OF_32)), ("scalar", "f64", (1501, 1499, 1), (True, DISPATCH)),
             ("reaction", "f32", (1951, 1949, 1), (False, RUNS_OF_32)), ("scalar", "f32", (2201, 2199, 1), (False, RUNS_OF_32)),
             ("scalar", "f64", (1701, 1699, 1), (False, RUNS_OF_32)), ("reaction", "f32", (1001, 701, 1), (False, CONTIGUOUS))]
    assert plans([(step, st, e, 9, 0) for step, st, e, _ in cases]) == [want for *_, want in cases]


def test_16_bit_planes_near_small_multiples_of_4_mib_keep_the_dispatch_order(plans):
    near = [(256, 256, 63), (256, 256, 64), (128, 128, 256), (256, 256, 65), (192, 256, 128), (256, 256, 95),
            (256, 256, 128), (256, 256, 160), (256, 256, 192)]
    others = [(256, 256, 62), (256, 256, 66), (256, 256, 80), (256, 256, 126), (256, 256, 176), (256, 256, 224),
              (256, 256, 256), (320, 320, 320)]
    for q in (19, 27):
        assert plans([("fluid", "f16", e, q, 0) for e in near]) == [(True, DISPATCH)] * len(near)
        assert plans([("fluid", "f16", e, q, 0) for e in others]) == [(True, RUNS_OF_8)] * len(others)
    wide = [("f64", (128, 128, 64), RUNS_OF_8), ("f32", (256, 128, 64), DISPATCH)]
    assert plans([("fluid", st, e, 19, 0) for st, e, _ in wide]) == [(True, order) for *_, order in wide]
    # slabs of 128 and 512 KiB are no planes 4 MiB apart
    slabs = [("f16", (256, 256, 256)), ("f16", (512, 512, 512)), ("f64", (256, 256, 256))]
    assert plans([("slabs", st, e, 19, 0) for st, e in slabs]) == [(True, RUNS_OF_8)] * 3
