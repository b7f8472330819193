"""Slab form of the tiled expert kernels (csrc/ffn_slab.hip): row tiles of up to 128 rows cut into
32-row groups, 256 weight rows per tile, K ranges of the down phase in separate buffers.  The routing
is fixed through the router so that the experts see exactly the row counts at which those cuts fall."""
import numpy as np
import pytest

from ateniaengine_amd import capi
from tests import synth as S
from tests.hipmem import DeviceArray, mem_free
from tests.test_gpu_parity import TOL_BF16_TOY, TOL_MODEL
from tests.test_zz_no_alloc import _run

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("counts,d,f,f_s", [
    ((128, 1, 33), 128, 128, 0),      # one stage pair of K; full tile, one row, one row past a group
    ((129, 96, 0), 384, 256, 0),      # two tiles of an expert, three groups, an expert without rows
    ((64, 65, 97), 256, 1152, 0),     # K ranges in the down phase (f = 18 stages)
    ((257, 31, 63), 256, 384, 2048),  # three tiles; the shared expert's down phase in four K ranges
    ((140, 100, 110, 90, 120), 256, 384, 2048),  # ... with more than four row tiles
    ((90, 80, 100), 640, 128, 640),   # widths that leave the last column tile partly empty
    ((129, 129, 1), 256, 256, 0),     # as many tiles as 259 rows of three experts can have
])
def test_slab_tiles_at_their_edges(ora, counts, d, f, f_s):
    E, T = len(counts), sum(counts)
    W = S.make_weights(5000 + T + d, E, d, f, f_s=f_s, gated=f_s > 0)
    W["w_router"][:] = 0.0
    W["w_router"][np.arange(E), np.arange(E)] = 1.0  # expert e reads coordinate e of the token
    oL, gL = S.build_pair(ora, W, 1, capi.CONVENTION_HUGGINGFACE_QWEN, capi.WEIGHT_BF16)
    with gL:
        x = S.make_tokens(5100 + T, T, d)
        want = np.random.default_rng(T).permutation(np.repeat(np.arange(E), counts))
        x[:, :E] = 0.0
        x[np.arange(T), want] = 4.0
        plan = gL.plan(T)
        assert plan["slab"] == 3, plan
        out = gL.forward(x).reshape(T, d)
        idx, w, got, _, _ = gL.last_routing(T)
        assert (idx[:, 0] == want).all() and tuple(got) == tuple(counts)
        sample = sorted(set(np.linspace(0, T - 1, 40).astype(int)))
        # f = 1152 is 18 stages of K, cut into two ranges while the tiles are few; the others have one range
        split = gL.last_down_split(T)
        assert (split == (2 if f == 1152 else 1)).all() and not (plan["y_bf16"] and split.max() > 1), plan
        model, slack = S.emulate_bf16_kernels(oL, x[sample], idx[sample], w[sample], with_slack=True,
                                              y_bf16=plan["y_bf16"], ys_bf16=plan["ys_bf16"],
                                              split=split[sample])
        for i, t in enumerate(sample):
            # the model's own bar: f32 summation order, plus what flips of h at a rounding midpoint move
            top = np.abs(model[i]).max()
            assert np.abs(out[t] - model[i]).max() <= TOL_MODEL * top + slack[i], (t, want[t])
            assert S.rel_err(out[t], oL.forward_f64(x[t], fixed_idx=idx[t])) <= TOL_BF16_TOY


@pytest.mark.parametrize("counts,d,f,f_s", [
    ((128, 1, 33), 128, 128, 0),      # two stages of K: fewer than are in flight
    ((129, 96, 0), 384, 256, 0),      # six and four stages, over three and four sets of registers
    ((64, 65, 97), 256, 1152, 0),     # K ranges in the down phase (f = 18 stages)
    ((257, 31, 63), 256, 384, 2048),  # three tiles; the shared expert's down phase in four K ranges
    ((90, 80, 100), 640, 128, 640),   # widths that leave the last column tile partly empty
    ((30, 20, 18), 256, 128, 2048),  # fewer routed tiles than shared ones, which follow them
    ((64, 65, 97), 256, 1152, 384),  # shared gate/up tiles that take turns with the routed ones, a down launch of one eight each
    ((64, 65, 3, 97, 40, 51), 1024, 2048, 512),  # ... in both phases
    ((30, 64, 97), 256, 1152, 1152),  # two K ranges of the routed down tiles, and of the shared expert's
    ((520, 130, 70), 2048, 512, 2048),  # more than 640 tokens: the shared expert in two ranges instead of four
    ((20, 20, 1, 20), 512, 896, 0),   # single row groups, eight and fourteen stages
    ((129, 129, 1), 256, 256, 0),     # as many tiles as 259 rows of three experts can have
])
def test_int8_slab_tiles_at_their_edges(ora, counts, d, f, f_s):
    """The same cuts on int8 weights, whose row scales are applied to the sums."""
    E, T = len(counts), sum(counts)
    W = S.make_weights(5800 + T + d, E, d, f, f_s=f_s, gated=f_s > 0, outlier_frac=0.02)
    W["w_router"][:] = 0.0
    W["w_router"][np.arange(E), np.arange(E)] = 1.0
    oL, gL = S.build_pair(ora, W, 1, capi.CONVENTION_HUGGINGFACE_QWEN, capi.WEIGHT_INT8_W8A16)
    with gL:
        x = S.make_tokens(5900 + T, T, d)
        want = np.random.default_rng(T).permutation(np.repeat(np.arange(E), counts))
        x[:, :E] = 0.0
        x[np.arange(T), want] = 4.0
        plan = gL.plan(T)
        assert plan["slab_int8"] == 3 and plan["slab"] == 0 and not plan["y_bf16"], plan
        out = gL.forward(x).reshape(T, d)
        idx, w, got, _, _ = gL.last_routing(T)
        assert (idx[:, 0] == want).all() and tuple(got) == tuple(counts)
        # K in ranges of eight stages or more, the shared expert's as long as the routed ones'
        ranges = {1152: 2, 2048: 4}.get(f, 1)
        assert (gL.last_down_split(T) == ranges).all() and plan["y_parts"] == ranges
        assert plan["ys_parts"] == (max(1, min(4, f_s * ranges // max(f, 512))) if T <= 640 else 2)
        sample = sorted(set(np.linspace(0, T - 1, 40).astype(int)))
        model, slack = S.emulate_bf16_kernels(oL, x[sample], idx[sample], w[sample], with_slack=True)
        for i, t in enumerate(sample):
            # the model's own bar: f32 summation order, plus what flips of h at a rounding midpoint move
            assert np.abs(out[t] - model[i]).max() <= TOL_MODEL * np.abs(model[i]).max() + slack[i], t
            assert S.rel_err(out[t], oL.forward_f64(x[t], fixed_idx=idx[t])) <= TOL_BF16_TOY


def test_int8_down_ranges_by_the_rows_of_an_expert(ora):
    """Experts with several row tiles have fewer K ranges."""
    E, d, f = 11, 2048, 1024
    W = S.make_weights(6300, E, d, f)
    W["w_router"][:] = 0.0
    W["w_router"][np.arange(E), np.arange(E)] = 1.0
    oL, gL = S.build_pair(ora, W, 1, capi.CONVENTION_HUGGINGFACE_QWEN, capi.WEIGHT_INT8_W8A16)
    with gL:
        for T, ranges in ((400, 2), (2400, 1)):
            x = S.make_tokens(6301 + T, T, d)
            want = np.arange(T) % E
            x[:, :E] = 0.0
            x[np.arange(T), want] = 4.0
            out = gL.forward(x).reshape(T, d)
            assert gL.plan(T)["slab_int8"] == 3 and (gL.last_down_split(T) == ranges).all()
            idx, w, _, _, _ = gL.last_routing(T)
            sample = sorted(set(np.linspace(0, T - 1, 20).astype(int)))
            model, slack = S.emulate_bf16_kernels(oL, x[sample], idx[sample], w[sample], with_slack=True)
            for i, t in enumerate(sample):
                assert np.abs(out[t] - model[i]).max() <= TOL_MODEL * np.abs(model[i]).max() + slack[i], t
                assert S.rel_err(out[t], oL.forward_f64(x[t], fixed_idx=idx[t])) <= TOL_BF16_TOY


# counts, d, f, f_s, narrow phases (1 gate/up, 2 down) of the bf16 and of the int8 layer
@pytest.mark.parametrize("wd", [capi.WEIGHT_BF16, capi.WEIGHT_INT8_W8A16])
@pytest.mark.parametrize("counts,d,f,f_s,narrow", [
    ((64, 65, 1, 33, 129, 0), 128, 128, 0, (3, 2)),  # one, two and three tiles of 64 rows, one stage pair of K
    ((32, 31, 97, 20), 640, 1152, 320 * 2, (3, 2)),  # column tiles past N, K ranges, a shared expert of two tiles
    ((60, 64, 20), 384, 256, 0, (3, 2)),
    ((65, 1, 65, 1), 256, 256, 0, (3, 2)),           # as many tiles as 132 rows of four experts can have
    ((40, 3, 7, 24, 1, 70), 256, 1792, 0, (3, 3)),
    ((60, 64, 20), 256, 6144, 0, (2, 2)),            # the down phase alone
    ((60, 64, 90), 256, 384, 0, (1, 0)),             # gate/up alone, two tiles for an expert
])
def test_narrow_slab_tiles_at_their_edges(ora, wd, counts, d, f, f_s, narrow):
    """Few tiles: 128 weight rows by 64 token rows each."""
    E, T = len(counts), sum(counts)
    W = S.make_weights(6000 + T + d, E, d, f, f_s=f_s, gated=f_s > 0)
    W["w_router"][:] = 0.0
    W["w_router"][np.arange(E), np.arange(E)] = 1.0
    oL, gL = S.build_pair(ora, W, 1, capi.CONVENTION_HUGGINGFACE_QWEN, wd)
    with gL:
        x = S.make_tokens(6100 + T, T, d)
        want = np.random.default_rng(T).permutation(np.repeat(np.arange(E), counts))
        x[:, :E] = 0.0
        x[np.arange(T), want] = 4.0
        plan = gL.plan(T)
        assert (plan["slab"] if wd == capi.WEIGHT_BF16 else plan["slab_int8"]) == 3, plan
        assert plan["narrow"] == narrow[0 if wd == capi.WEIGHT_BF16 else 1], plan
        out = gL.forward(x).reshape(T, d)
        idx, w, got, _, _ = gL.last_routing(T)
        assert (idx[:, 0] == want).all() and tuple(got) == tuple(counts)
        sample = sorted(set(np.linspace(0, T - 1, 40).astype(int)))
        model, slack = S.emulate_bf16_kernels(oL, x[sample], idx[sample], w[sample], with_slack=True,
                                              y_bf16=plan["y_bf16"], ys_bf16=plan["ys_bf16"],
                                              split=gL.last_down_split(T)[sample])
        for i, t in enumerate(sample):
            # the model's own bar: f32 summation order, plus what flips of h at a rounding midpoint move
            assert np.abs(out[t] - model[i]).max() <= TOL_MODEL * np.abs(model[i]).max() + slack[i], t
            assert S.rel_err(out[t], oL.forward_f64(x[t], fixed_idx=idx[t])) <= TOL_BF16_TOY
        # the same tokens among 60 rows for every expert, where the down tiles are wide, and gate/up's where one round
        # of narrow ones would not hold all: the same bits
        if T < 60 * E:
            more = np.concatenate([x] * E)[-60 * E:]
            wide = gL.plan(len(more))
            assert all(wide[n] == plan[n] for n in ("slab", "slab_int8", "y_bf16", "ys_bf16")), wide
            assert wide["narrow"] == (1 if wd == capi.WEIGHT_BF16 and f < 1792 else 0), wide
            assert gL.forward(more).reshape(-1, d)[-T:].tobytes() == out.tobytes()


@pytest.mark.parametrize("wd,T,d,f,f_s,parts", [
    (capi.WEIGHT_BF16, 400, 3072, 2048, 0, (4, 1)),     # the routed experts' partial buffers alone are past the 16 MiB
    (capi.WEIGHT_BF16, 400, 2048, 512, 2048, (1, 4)),   # the shared expert's
    (capi.WEIGHT_INT8_W8A16, 48, 2048, 1024, 1024, (2, 2)),    # small W8A16 batches, narrow tiles
    (capi.WEIGHT_INT8_W8A16, 40, 2048, 2048, 0, (4, 1)),
    (capi.WEIGHT_INT8_W8A16, 400, 3072, 2048, 2048, (4, 4)),   # both experts' past it
])
def test_noalloc_sums_in_the_same_k_ranges(ora, wd, T, d, f, f_s, parts):
    """A batch that fits the entry point that allocates nothing with one buffer of expert outputs runs in as
    many K ranges there as from the handle's own workspace: the outputs are the same bits."""
    E = 8
    W = S.make_weights(5300 + d, E, d, f, f_s=f_s, gated=f_s > 0)
    _, gL = S.build_pair(ora, W, 1, capi.CONVENTION_HUGGINGFACE_QWEN, wd)
    with gL:
        x = S.make_tokens(5400 + d, T, d)
        plan = gL.plan(T)
        assert plan["slab" if wd == capi.WEIGHT_BF16 else "slab_int8"] == 3 and plan["down"] == capi.KERNELS_MID, plan
        assert not plan["y_bf16"] and not plan["ys_bf16"] and (plan["y_parts"], plan["ys_parts"]) == parts, plan
        want = _run(gL, x, noalloc=False)
        _run(gL, x, noalloc=True)  # warm: one-time kernel attributes
        assert _run(gL, x, noalloc=True, watch_memory=True).tobytes() == want.tobytes()


def test_k_ranges_that_cancel_are_added_in_f32(ora):
    """Where the kernel cuts the K of every tile into ranges, the partial sums must not be rounded to bf16:
    here the two halves of K nearly cancel, so that the partial sums are some thirty times the result."""
    counts, d, f = (105, 96, 108), 256, 1152  # 9 stage pairs, two ranges
    E, T = len(counts), sum(counts)
    W = S.make_weights(5500, E, d, f)
    W["w_router"][:] = 0.0
    W["w_router"][np.arange(E), np.arange(E)] = 1.0
    for name in ("w_gate", "w_up"):
        W[name][:, f // 2:] = W[name][:, :f // 2]
    noise = np.random.default_rng(5501).standard_normal((E, d, f // 2), dtype=np.float32)
    W["w_down"][:, :, f // 2:] = -W["w_down"][:, :, :f // 2] * (1 + noise / 32)
    oL, gL = S.build_pair(ora, W, 1, capi.CONVENTION_ATENIA, capi.WEIGHT_BF16)
    with gL:
        x = S.make_tokens(5502, T, d)
        want = np.random.default_rng(T).permutation(np.repeat(np.arange(E), counts))
        x[:, :E] = 0.0
        x[np.arange(T), want] = 4.0
        plan = gL.plan(T)
        assert plan["slab"] == 3 and plan["down"] == capi.KERNELS_TILED, plan
        gL.forward(x)
        idx, *_ = gL.last_routing(T)
        assert (idx[:, 0] == want).all()
        y, _ = gL.last_expert_outputs(T)
        for t in range(0, T, 11):
            g, u, dn = (a[want[t]].astype(np.float64) for a in (oL.w_gate, oL.w_up, oL.w_down))
            gg, uu = (g @ x[t]).astype(np.float32), (u @ x[t]).astype(np.float32)
            hv = gg / (np.float32(1) + np.exp(-gg, dtype=np.float32)) * uu
            h = S.bf16_rne(hv).astype(np.float64)
            ref = dn @ h
            # one rounding of the result to bf16 at most, f32 sums of 1152 products (2^-24 of the partial
            # sum each, which is some 1 / 30 of the sum of the magnitudes), what a flip of h moves
            bar = 2.0 ** -9 * np.abs(ref) + 2.0 ** -19 * (np.abs(dn) @ np.abs(h)) + np.abs(dn) @ S._fragile_ulp(hv)
            assert (np.abs(y[t, 0] - ref) <= bar).all(), (t, (np.abs(y[t, 0] - ref) / bar).max())


def test_rows_do_not_depend_on_the_rest_of_the_batch(ora):
    """The tokens of a small batch inside a larger one that is cut into more row tiles of the routed experts
    and of a wide shared one (three and five): the same bits, before the combine and after it."""
    E, k, d, f, f_s = 16, 2, 256, 384, 2048
    W = S.make_weights(5600, E, d, f, f_s=f_s, gated=True, router_std=0.3 / np.sqrt(d))
    _, gL = S.build_pair(ora, W, k, capi.CONVENTION_HUGGINGFACE_QWEN, capi.WEIGHT_BF16)
    with gL:
        pool = S.make_tokens(5601, 600, d)
        small, large = pool[:260], np.concatenate([pool[300:], pool[:260][::-1]])
        for T in (260, 560):
            plan = gL.plan(T)
            assert plan["slab"] == 3 and not plan["y_bf16"] and not plan["ys_bf16"], plan
        out_a = gL.forward(small)
        ya, ysa = gL.last_expert_outputs(260)
        out_b = gL.forward(large)[300:][::-1]
        yb, ysb = (a[300:][::-1] for a in gL.last_expert_outputs(560))
        assert np.array_equal(ysa, ysb), "shared expert outputs depend on the batch"
        assert np.array_equal(ya, yb), "expert outputs depend on the batch"
        assert np.array_equal(out_a, out_b), "layer outputs depend on the batch"


@pytest.mark.parametrize("k", [1, 2, 3, 6, 8, 9, 17])
@pytest.mark.parametrize("d,f,parts", [(256, 1152, 2), (384, 2176, 4)])  # ranges of 4 and 5 stage pairs; of 4, 4, 4, 5
def test_combine_of_rows_in_ranges_alike(ora, d, f, parts, k):
    """Where every tile was cut into as many K ranges, whatever the number of slots: the bits of the weighted
    sum of the expert outputs, each the sum of its ranges in order."""
    E = 20
    T = 60 * E // k
    W = S.make_weights(5700 + d + k, E, d, f, f_s=128)
    oL, gL = S.build_pair(ora, W, k, capi.CONVENTION_ATENIA, capi.WEIGHT_BF16)
    with gL:
        x = S.make_tokens(5701 + k, T, d)
        plan = gL.plan(T)
        assert plan["slab"] == 3 and not plan["y_bf16"], plan
        out = gL.forward(x).reshape(T, d)
        assert (gL.last_down_split(T) == parts).all()
        idx, w, *_ = gL.last_routing(T)
        y, ys = gL.last_expert_outputs(T)
        want = np.zeros((T, d), dtype=np.float32)
        for s_ in range(k):
            want = want + w[:, s_, None] * y[:, s_, :]
        assert out.tobytes() == (want + ys).tobytes()
        g, u, dn = (np.asarray(a, np.float64) for a in (oL.w_gate, oL.w_up, oL.w_down))
        for t in range(0, T, max(1, T // 5)):  # and those sums are the expert's
            e = idx[t, k - 1]
            gg = g[e] @ x[t]
            assert S.rel_err(y[t, k - 1], dn[e] @ (gg / (1 + np.exp(-gg)) * (u[e] @ x[t]))) <= TOL_BF16_TOY


def test_workspace_of_a_large_int8_batch_holds_the_shared_outputs_once(ora):
    """Batches of several thousand tokens have the shared expert's outputs in one K range, so their workspace has one
    buffer for them."""
    E, k, d, f, f_s, T = 4, 1, 2048, 256, 512, 4600
    W = S.make_weights(6200, E, d, f, f_s=f_s, gated=True)
    _, gL = S.build_pair(ora, W, k, capi.CONVENTION_HUGGINGFACE_QWEN, capi.WEIGHT_INT8_W8A16)
    with gL:
        plan = gL.plan(T)
        assert plan["slab_int8"] == 3 and not plan["int8_copy"], plan
        x = S.make_tokens(6201, T, d)
        _run(gL, x[:8], noalloc=False)
        dx, out = DeviceArray.from_host(x), DeviceArray((T, d), np.float32)
        before = mem_free()
        gL.forward_device(dx.ptr, capi.ACT_F32, T, out.ptr)
        grown = before - mem_free()
        # rows in bf16, h of both experts, four ranges of the routed outputs, the shared ones once, rows and outputs of
        # the host entry point; a MiB for lists and logits, and the allocator's rounding
        rows = T * (2 * d + 2 * (f + f_s) + 4 * 4 * d + 4 * d + 2 * 4 * d)
        assert grown <= rows + (16 << 20), (grown, rows)
