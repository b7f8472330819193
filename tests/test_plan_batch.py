"""Which expert kernels a batch takes (`atenia_moe_hip_plan_batch`: a pure function of the layer's
dimensions and the batch size, no device needed).

The reference has one expert loop for every batch size (src/moe/layer.rs:405-443), so there is
nothing to compare the choice with; what can be held is that the plan is *defensible*: defined for
every shape, ordered in T (register-resident streaming -> mid-batch -> matrix-core tiled, never
back, per phase), and consistent with what the kernels can take.  Shapes: every layer the random
GPU suites draw (tests/test_gpu_fuzz.py), the five benchmark configurations, and two shapes of
the reference's model families (src/moe/family.rs) outside the benchmark list: Mixtral-8x22B
(d = 6144, f = 16384) and a 128-expert top-8 layer with narrow experts (f = 768).
"""
import os
import subprocess
import sys

import numpy as np
import pytest

from ateniaengine_amd import capi
from tests.test_gpu_fuzz import _cases, _mid_cases

FAMILY_ORDER = {capi.KERNELS_STREAM: 0, capi.KERNELS_MID: 1, capi.KERNELS_TILED: 2}

NAMED = [
    # E, k, d, f, f_s, weight dtype
    (8, 2, 1024, 2048, 0, capi.WEIGHT_F32),              # config 1
    (8, 2, 4096, 14336, 0, capi.WEIGHT_BF16),            # config 2
    (8, 2, 4096, 14336, 0, capi.WEIGHT_INT8_W8A16),      # config 3
    (8, 2, 4096, 14336, 0, capi.WEIGHT_INT8_PER_GROUP),
    (60, 4, 2048, 1408, 5632, capi.WEIGHT_BF16),         # config 4
    (64, 6, 2048, 1408, 2816, capi.WEIGHT_BF16),         # config 5
    (8, 2, 6144, 16384, 0, capi.WEIGHT_BF16),            # Mixtral-8x22B
    (8, 2, 6144, 16384, 0, capi.WEIGHT_INT8_W8A16),
    (128, 8, 2048, 768, 0, capi.WEIGHT_BF16),            # many narrow experts
    (128, 8, 2048, 768, 768, capi.WEIGHT_BF16),
    (256, 8, 7168, 2048, 2048, capi.WEIGHT_BF16),        # DeepSeek-V3 routed-expert shape
]


def _shapes():
    seen = []
    for p in _cases(150, 20240607) + _mid_cases(60, 20250311):
        E, k, d, f, fs, _g, _c, wd, _T, _s = p.values
        seen.append((E, k, d, f, fs, wd))
    return sorted(set(seen)) + NAMED


def _batch_sizes():
    ts = set(range(1, 701)) | {int(round(v)) for v in np.geomspace(700, 40000, 160)}
    return sorted(ts)


@pytest.mark.parametrize("E,k,d,f,fs,wd", _shapes())
def test_plan_is_defined_and_ordered_in_the_batch_size(E, k, d, f, fs, wd):
    gs = 128 if wd == capi.WEIGHT_INT8_PER_GROUP else 0
    prev = None
    for T in _batch_sizes():
        p = capi.plan_batch(E, k, d, f, fs, wd, T, group_size=gs)
        if wd == capi.WEIGHT_F32:
            assert p["up"] == p["down"] == capi.KERNELS_F32
            assert p["shared_up"] == p["shared_down"] == (capi.KERNELS_F32 if fs else -1)
            assert not (p["y_bf16"] or p["ys_bf16"] or p["tall_tiles"] or p["duo"])
            continue
        assert p["up"] in FAMILY_ORDER and p["down"] in FAMILY_ORDER, (T, p)
        assert (p["shared_up"] == -1) == (fs == 0) and (p["shared_down"] == -1) == (fs == 0), (T, p)
        # bf16 expert outputs: only bf16 layers, only behind the matrix-core down launch
        if p["y_bf16"]:
            assert wd == capi.WEIGHT_BF16 and p["down"] == capi.KERNELS_TILED, (T, p)
        if p["ys_bf16"]:
            assert p["y_bf16"] and p["shared_down"] == capi.KERNELS_TILED, (T, p)
        if p["tall_tiles"]:
            assert capi.KERNELS_TILED in (p["up"], p["down"]), (T, p)
            # a W8A16 layer has them on the bf16 copy of its int8 values only
            assert wd != capi.WEIGHT_INT8_W8A16 or p["int8_copy"], (T, p)
        if p["int8_copy"]:
            assert wd == capi.WEIGHT_INT8_W8A16 and p["up"] == p["down"] == capi.KERNELS_TILED, (T, p)
            assert fs == 0 or p["shared_up"] == p["shared_down"] == capi.KERNELS_TILED, (T, p)
            assert not p["y_bf16"], (T, p)
        if prev is not None and prev[1]["int8_copy"]:
            assert p["int8_copy"], f"back from the bf16 copy at T={T}"
        # the slab kernels take the place of the mid-batch and tiled ones on bf16 layers, both phases' row
        # tiles cut alike; outputs that travel as bf16 are then in one k range
        if p["slab"]:
            assert wd == capi.WEIGHT_BF16 and p["slab"] & 1 and not p["tall_tiles"], (T, p)
            assert p["up"] != capi.KERNELS_STREAM, (T, p)
            assert (p["slab"] == 3) == (p["down"] != capi.KERNELS_STREAM), (T, p)
        # narrow tiles: of slab phases only
        assert p["narrow"] & ~(p["slab"] | p["slab_int8"]) == 0, (T, p)
        assert p["duo"] == 0, "the two-workgroup form is off unless ATENIA_MOE_DUO_MAX_K asks for it"
        if prev is not None:
            for phase in ("up", "down"):
                assert FAMILY_ORDER[p[phase]] >= FAMILY_ORDER[prev[1][phase]], (
                    f"{phase} phase goes back from {prev[1][phase]} at T={prev[0]} to {p[phase]} at T={T}")
        prev = (T, p)
    # a large enough batch ends on the matrix cores wherever the widths allow it (K in whole 64-k
    # stages; other widths keep the streaming kernels, which take any K)
    if wd != capi.WEIGHT_F32 and d % 64 == 0 and f % 64 == 0:
        assert prev[1]["up"] == prev[1]["down"] == capi.KERNELS_TILED, prev


def test_plan_rejects_what_create_rejects():
    for bad in [dict(E=0), dict(k=0), dict(k=9), dict(d=0), dict(f=0), dict(fs=-1), dict(wd=7), dict(T=0)]:
        a = dict(E=8, k=2, d=256, f=512, fs=0, wd=capi.WEIGHT_BF16, T=16)
        a.update(bad)
        with pytest.raises(capi.MoeHipError):
            capi.plan_batch(a["E"], a["k"], a["d"], a["f"], a["fs"], a["wd"], a["T"])
    with pytest.raises(capi.MoeHipError):  # per-group scales need a group size in whole 64-k blocks
        capi.plan_batch(8, 2, 256, 512, 0, capi.WEIGHT_INT8_PER_GROUP, 16, group_size=100)


def test_plan_reports_the_slab_kernels():
    """bf16 layers with widths in whole 128s: from where the register-resident kernels end up to about one
    128-row tile for each expert; never on other storage types or widths."""
    def slab(T, E=8, k=2, d=4096, f=14336, fs=0, wd=capi.WEIGHT_BF16):
        return capi.plan_batch(E, k, d, f, fs, wd, T)["slab"]
    assert [slab(T) for T in (1, 16, 56, 64, 333, 416, 420, 4096)] == [0, 0, 0, 3, 3, 3, 0, 0]
    assert slab(333, wd=capi.WEIGHT_INT8_W8A16) == 0 and slab(333, wd=capi.WEIGHT_F32) == 0
    assert slab(333, f=14336 + 64) == 0 and slab(333, d=4096 - 64) == 0
    assert slab(333, fs=1024) == 3 and slab(333, fs=1024 + 64) == 0  # the shared expert rides along
    assert slab(997, 60, 4, 2048, 1408, 5632) == 3
    # 104 rows per expert without a shared expert, where routing that is even on average starts to give
    # experts a second tile; 117 with one or with a short K in the down phase
    for E, k, d, f in ((8, 2, 6144, 16384), (16, 2, 4096, 14336), (64, 4, 2048, 2048)):
        assert [slab(a * E // k, E, k, d, f) for a in (104, 105)] == [3, 0]
    for E, k, d, f, fs in ((60, 4, 2048, 1408, 5632), (64, 4, 2048, 2048, 2048), (128, 8, 2048, 768, 0)):
        assert [slab(a * E // k, E, k, d, f, fs) for a in (105, 117, 118)] == [3, 3, 0]
    # 190 rows per expert with a short K in the down phase
    assert [slab(T, 256, 8, 7168, 256, 256) for T in (256, 6000, 6100)] == [3, 3, 0]
    # a matrix of one expert past 2 GiB is not addressed in 32 bits
    assert slab(80, 2, 1, 32768, 32640) == 3 and slab(80, 2, 1, 32768, 32768) == 0


@pytest.mark.parametrize("knob,value,E,k,d,f,fs,T,want", [
    # the mid-batch kernel off: the tiled kernels take its place; or up to 90 rows per expert
    ("ATENIA_MOE_MID_MAX_AVG", "0", 8, 2, 4096, 14336, 0, 200, dict(up=2, down=2, slab=0)),
    ("ATENIA_MOE_MID_MAX_AVG", "90", 8, 2, 4096, 14336, 0, 333, dict(up=1, down=1, slab=0)),
    ("ATENIA_MOE_MID_MAX_AVG", "90", 60, 4, 2048, 1408, 5632, 45, dict(up=0, down=0, slab=0)),
    # the largest batch that streams, above it the tiled kernels
    ("ATENIA_MOE_STREAM_MAX_TOKENS", "30", 8, 2, 4096, 14336, 0, 64, dict(up=2, down=2, slab=0)),
    # the two-workgroup form of both phases, or of the one whose K is short enough
    ("ATENIA_MOE_DUO_MAX_K", "2048", 8, 2, 256, 512, 0, 700, dict(up=2, down=2, duo=3, slab=0)),
    ("ATENIA_MOE_DUO_MAX_K", "256", 8, 2, 256, 512, 0, 700, dict(up=2, down=2, duo=1, slab=0)),
    ("ATENIA_MOE_DUO_MAX_K", "128", 8, 2, 256, 512, 0, 700, dict(up=2, down=2, duo=0, slab=3)),
    # the per-token router: whatever the matrix cores would take from it, with more than 32 rows from 52 tokens on
    ("ATENIA_MOE_ROUTER_TOKEN_MAX", "400", 8, 2, 4096, 14336, 0, 400, dict(router=0, router_f32=0)),
    ("ATENIA_MOE_ROUTER_TOKEN_MAX", "400", 8, 2, 4096, 14336, 0, 401, dict(router=2, router_f32=2)),
    ("ATENIA_MOE_ROUTER_TOKEN_MAX", "0", 8, 2, 4096, 14336, 0, 1, dict(router=2, router_f32=2)),
    ("ATENIA_MOE_ROUTER_TOKEN_MAX", "400", 64, 6, 4096, 1408, 0, 51, dict(router=0, router_f32=0)),
    ("ATENIA_MOE_ROUTER_TOKEN_MAX", "400", 64, 6, 4096, 1408, 0, 52, dict(router=4, router_f32=4)),
    ("ATENIA_MOE_ROUTER_TOKEN_MAX", "20", 64, 6, 4096, 1408, 0, 21, dict(router=4, router_f32=4)),
])
def test_knobs_that_choose_a_kernel_are_obeyed(knob, value, E, k, d, f, fs, T, want):
    """The knobs are read once per process, so each runs in a child."""
    src = ("from ateniaengine_amd import capi; "
           f"print(capi.plan_batch({E}, {k}, {d}, {f}, {fs}, capi.WEIGHT_BF16, {T}))")
    root = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
    r = subprocess.run([sys.executable, "-c", src], cwd=root, env=dict(os.environ, **{knob: value}),
                       capture_output=True, text=True, timeout=300)
    assert r.returncode == 0, r.stderr[-2000:]
    plan = eval(r.stdout.strip().splitlines()[-1])
    assert {n: plan[n] for n in want} == want, plan


def test_plan_reads_nothing_it_has_not_set(tmp_path):
    """The same plans from a build whose uninitialised locals hold a pattern instead of what the stack held."""
    root = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
    csrc = os.path.join(root, "ateniaengine_amd", "csrc")
    subprocess.run(["make", "-C", csrc, "-j4"], check=True, capture_output=True, timeout=900)
    hipcc = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")
    obj, so = str(tmp_path / "moe_abi.o"), str(tmp_path / "libatenia_moe_hip.so")
    subprocess.run([hipcc, "--offload-arch=gfx950", "-O1", "-fPIC", "-std=c++17", "-Xarch_host",
                    "-ftrivial-auto-var-init=pattern", "-c", os.path.join(csrc, "moe_abi.hip"), "-o", obj],
                   check=True, capture_output=True, timeout=600)
    others = [os.path.join(csrc, n) for n in sorted(os.listdir(csrc)) if n.endswith(".o") and n != "moe_abi.o"]
    subprocess.run([hipcc, "--offload-arch=gfx950", "-shared", "-fPIC", "-o", so, obj] + others,
                   check=True, capture_output=True, timeout=600)
    cases = [s + (T,) for s in NAMED for T in (1, 8, 24, 40, 64, 333, 997, 4096)]
    src = ("from ateniaengine_amd import capi\n"
           f"for c in {cases!r}:\n"
           "    print(sorted(capi.plan_batch(*c, group_size=128 if c[5] == capi.WEIGHT_INT8_PER_GROUP else 0).items()))")
    got = []
    for lib in ({}, {"ATENIA_MOE_HIP_LIBRARY": so}):
        r = subprocess.run([sys.executable, "-c", src], cwd=root, env=dict(os.environ, **lib), capture_output=True,
                           text=True, timeout=300)
        assert r.returncode == 0, r.stderr[-2000:]
        got.append(r.stdout.splitlines())
    assert got[0] == got[1], [(c, a, b) for c, a, b in zip(cases, *got) if a != b][:3]


B, I = capi.WEIGHT_BF16, capi.WEIGHT_INT8_W8A16


@pytest.mark.parametrize("E,k,d,f,fs,wd,T,narrow", [
    # gate/up: a last round of wide tiles that fills more than half of the chip keeps them
    (16, 2, 2048, 1024, 1024, B, 60, 2), (32, 4, 4096, 1536, 1536, B, 56, 2), (16, 2, 4096, 1536, 0, B, 112, 0),
    (16, 4, 3072, 1536, 0, B, 110, 2), (16, 2, 7168, 1536, 0, I, 64, 0), (4, 2, 4096, 8192, 0, I, 64, 0),
    (8, 2, 4096, 7168, 0, I, 64, 0),
    # ... half of it or less does not
    (8, 2, 4096, 1408, 0, B, 112, 1), (16, 2, 7168, 1024, 0, B, 112, 1), (32, 4, 4096, 1152, 0, B, 128, 1),
    (128, 8, 4096, 512, 512, B, 128, 1), (32, 4, 4096, 1152, 0, I, 64, 1), (8, 2, 4096, 5120, 0, I, 64, 1),
    # down
    (64, 6, 2048, 1408, 2816, B, 48, 2), (64, 6, 2048, 1408, 2816, B, 160, 2), (64, 6, 2048, 1408, 2816, B, 300, 0),
    (60, 4, 2048, 1408, 5632, B, 200, 0), (16, 4, 5120, 1536, 3072, I, 64, 2),
    # by the rows of an expert, not by the batch: down tiles of more than 50 are wide, gate/up ones while twice as many
    # narrow ones do not fit one round either
    (8, 4, 4096, 896, 0, B, 100, 3), (8, 4, 4096, 896, 0, B, 160, 1), (16, 8, 2048, 768, 0, B, 100, 3),
    (16, 8, 2048, 768, 0, B, 160, 0), (8, 4, 4096, 896, 0, I, 160, 0), (16, 8, 2048, 768, 0, I, 160, 0),
])
def test_widths_of_the_slab_tiles(E, k, d, f, fs, wd, T, narrow):
    p = capi.plan_batch(E, k, d, f, fs, wd, T)
    assert p["slab" if wd == B else "slab_int8"] == 3 and p["narrow"] == narrow, p


@pytest.mark.parametrize("E,k,d,f,fs,at", [
    # batches of 36 tokens, 48, 56: phases on the slab kernels
    (64, 6, 2048, 1408, 2816, (3, 3, 3)), (256, 8, 7168, 256, 256, (3, 3, 3)), (16, 4, 5120, 1536, 3072, (3, 3, 3)),
    (16, 8, 1024, 512, 512, (3, 3, 3)),
    # few tiles, and pairs that the register-resident gate/up launch groups itself
    (4, 1, 2048, 1024, 1024, (0, 1, 3)), (8, 2, 7168, 1024, 1024, (0, 1, 3)), (16, 2, 2048, 1536, 1536, (0, 1, 3)),
    (64, 1, 4096, 1024, 1024, (0, 1, 3)),
])
def test_slab_kernels_from_36_tokens(E, k, d, f, fs, at):
    assert tuple(capi.plan_batch(E, k, d, f, fs, B, T)["slab"] for T in (36, 48, 56)) == at


@pytest.mark.parametrize("E,k,d,f,fs,wd,T,parts", [
    # the shared expert's down tiles as long as a routed expert's range of K, in small W8A16 batches
    (8, 1, 5120, 8192, 8192, I, 64, (2, 2)), (8, 2, 2048, 2048, 2048, I, 64, (4, 4)), (16, 2, 4096, 4096, 4096, I, 70, (2, 2)),
    (4, 1, 4096, 4096, 8192, I, 200, (4, 4)), (60, 4, 2048, 1408, 5632, I, 64, (1, 4)), (64, 6, 2048, 1408, 2816, I, 640, (1, 2)),
    (16, 2, 2048, 512, 512, I, 64, (1, 1)),
    # ... and in larger ones only while they are few
    (8, 1, 5120, 8192, 8192, I, 641, (2, 1)), (60, 4, 2048, 1408, 5632, I, 997, (1, 2)), (60, 4, 2048, 1408, 5632, I, 4500, (1, 1)),
    # an expert that sees several tiles' rows: fewer ranges of the routed ones too
    (8, 2, 4096, 14336, 0, I, 200, (4, 1)), (8, 2, 4096, 14336, 0, I, 500, (2, 1)),
    # bf16: by the layer alone
    (8, 1, 5120, 8192, 8192, B, 64, (2, 1)), (60, 4, 2048, 1408, 5632, B, 64, (1, 4)), (60, 4, 2048, 1408, 5632, B, 997, (1, 4)),
])
def test_k_ranges_of_the_slab_down_tiles(E, k, d, f, fs, wd, T, parts):
    p = capi.plan_batch(E, k, d, f, fs, wd, T)
    assert (p["y_parts"], p["ys_parts"]) == parts, p


@pytest.mark.parametrize("E,k,d,f,fs,first", [
    (8, 2, 4096, 14336, 0, 20), (64, 6, 2048, 1408, 2816, 20), (60, 4, 2048, 1408, 5632, 20), (128, 8, 2048, 768, 0, 20),
    (16, 2, 7168, 1536, 0, 20), (8, 2, 1024, 2048, 0, 20), (256, 8, 4096, 512, 512, 20),
    # few tiles of a long K; many experts of a long K
    (8, 4, 4096, 896, 0, 40), (8, 2, 2048, 1408, 0, 40), (16, 2, 4096, 1024, 0, 40), (64, 2, 4096, 2048, 0, 40),
    (16, 4, 6144, 10752, 0, 40), (8, 1, 4096, 1024, 1024, 48), (16, 2, 7168, 1024, 0, 80), (24, 2, 4096, 3072, 0, 80),
])
def test_first_int8_batch_on_the_slab_kernels(E, k, d, f, fs, first):
    took = [capi.plan_batch(E, k, d, f, fs, I, T)["slab_int8"] for T in range(1, 200)]
    assert took == [0] * (first - 1) + [3] * (200 - first)


@pytest.mark.parametrize("E,d,rows,want", [
    # up to eight rows: one workgroup per token, by eight tokens, by sixteen
    (8, 1024, "router", "0 to 263, 2 to 2048, 1 to 4096, 2 to 6144, 1 to 8192, 2 to 10240, 1"),
    (8, 4096, "router", "0 to 263, 2 to 2048, 1 to 4096, 2 to 6144, 1 to 8192, 2 to 10240, 1 to 12288, 2 to 14336, 1"),
    (8, 256, "router", "0 to 263, 2 to 2048, 1"), (8, 2048, "router_f32", "0 to 263, 2 to 2048, 1"),
    (8, 4096, "router_f32", "0 to 263, 2 to 2048, 1 to 4096, 2 to 6144, 1 to 8192, 2 to 10240, 1"),
    (9, 1024, "router", "0 to 512, 1"),
    # more than 32: one workgroup per token and four rows, 8 x 8, 16 x 16
    (61, 2048, "router", "0 to 16, 4 to 256, 3 to 2048, 1"), (61, 2048, "router_f32", "0 to 16, 4 to 256, 3 to 2048, 1"),
    (61, 4096, "router", "0 to 16, 4 to 256, 3 to 2048, 1"), (61, 4096, "router_f32", "0 to 19, 4 to 256, 3 to 2048, 1"),
    (40, 8192, "router", "0 to 28, 4 to 408, 3 to 2048, 1"), (40, 8192, "router_f32", "0 to 33, 4 to 408, 3 to 2048, 1"),
    (32, 2048, "router", "0 to 191, 4 to 512, 3 to 2048, 1"),
])
def test_lines_between_the_routers(E, d, rows, want):
    got, last = [], None
    for T in list(range(1, 700)) + [t + i for t in range(1024, 17000, 1024) for i in (0, 1)]:
        form = capi.plan_batch(E, min(2, E), d, 128, 0, B, T)[rows]
        if form != last:
            got += [f"{last} to {prev}"] if last is not None else []
        last, prev = form, T
    assert ", ".join(got + [str(last)]) == want
