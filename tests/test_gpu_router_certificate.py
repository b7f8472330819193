"""Routers whose sums are not exact in every order (f32 activations, bf16 ones with very small values):
the bound that follows the partial sums, and the matrix-core router on f32 activations with the bf16
copy of the rows that it leaves for the experts."""
import numpy as np
import pytest

from ateniaengine_amd import capi
from tests import synth as S
from tests.hipmem import DeviceArray
from tests.test_gpu_parity import ulp_diff

pytestmark = pytest.mark.gpu


def _rows(kind, T, d, w_router):
    rng = np.random.default_rng(T + d)
    x = rng.standard_normal((T, d))
    if kind == "wide":  # sums of a few large terms
        x *= np.exp2(rng.integers(-30, 30, size=(T, d)))
    if kind == "cancel":  # every logit is what is left of terms a thousand times larger
        u, s, vt = np.linalg.svd(np.asarray(w_router, np.float64), full_matrices=False)
        keep = vt[s > 1e-6 * s[0]]
        x -= 0.999 * (x @ keep.T) @ keep
    if kind == "tiny":  # bf16-valued, a few values small enough that no sum is exact in every order
        x[rng.random((T, d)) < 0.01] *= 1e-9
    x = x.astype(np.float32)
    return S.bf16_round_trip(x)[1] if kind == "tiny" else x


FORMS = [
    # one workgroup per token; rows in lane pieces of 4, 8 and more columns, the last ones empty
    (capi.ROUTER_TOKEN, [
        (8, 2, 4096, 48, False, "f32"), (60, 4, 2048, 16, True, "cancel"), (8, 2, 132, 30, False, "cancel"),
        (7, 2, 71, 20, False, "cancel"), (60, 4, 1024, 16, True, "tiny"), (40, 3, 520, 16, False, "wide"),
        (8, 2, 1024, 33, False, "tiny"), (31, 4, 2048, 191, False, "tiny"),
        # ... the largest batches before the matrix cores take over, with up to eight rows and with more than 32
        (8, 2, 40, 257, False, "f32"), (7, 2, 72, 258, True, "cancel"), (7, 3, 1056, 263, True, "tiny"),
        (8, 2, 4096, 259, False, "tiny"), (3, 1, 2144, 261, False, "wide"), (48, 4, 2080, 25, False, "cancel")]),
    # matrix cores, the rows dealt to workgroups: selection as a second launch
    (capi.ROUTER_SPLIT, [
        (60, 4, 2048, 997, True, "tiny"), (64, 6, 512, 300, False, "cancel"), (128, 8, 256, 130, False, "wide"),
        (64, 6, 328, 257, False, "tiny")]),
    # ... by eight rows and eight tokens: the last workgroup's rows one or the gate alone, one workgroup to a compute unit
    (capi.ROUTER_SPLIT8, [
        (60, 4, 2048, 32, True, "cancel"), (60, 4, 1024, 32, True, "tiny"),
        (60, 4, 1024, 33, True, "tiny"), (60, 4, 256, 48, True, "cancel"), (60, 4, 2048, 33, True, "tiny"),
        (60, 4, 2048, 40, True, "cancel"), (64, 6, 2048, 33, False, "f32"), (60, 4, 2048, 52, True, "f32"),
        (32, 4, 72, 192, False, "f32"), (56, 4, 1056, 20, True, "tiny"), (33, 2, 72, 29, False, "cancel"),
        (64, 6, 328, 256, False, "f32"), (200, 8, 96, 9, False, "wide"), (60, 4, 2048, 17, True, "cancel"),
        (48, 4, 2080, 26, False, "cancel")]),
    # matrix cores, one to five row blocks to a workgroup
    (capi.ROUTER_MFMA, [
        (8, 2, 256, 2100, False, "cancel"), (20, 3, 96, 2100, True, "cancel"), (40, 4, 640, 2500, False, "f32"),
        (64, 6, 1024, 2300, False, "cancel"), (79, 5, 256, 2100, True, "wide")]),
    # ... up to eight rows by eight tokens: waves of one, of an odd number and of no steps; tokens past the last one
    (capi.ROUTER_MFMA8, [
        (8, 2, 40, 265, False, "f32"), (7, 2, 72, 266, True, "cancel"), (7, 3, 1056, 271, True, "tiny"),
        (8, 2, 4096, 264, False, "tiny"), (3, 1, 2144, 269, False, "wide"), (5, 2, 328, 270, False, "tiny"),
        (8, 2, 4096, 600, False, "f32")]),
]


@pytest.mark.parametrize("form,E,k,d,T,gated,kind", [(form,) + c for form, cases in FORMS for c in cases])
def test_router_sums_that_depend_on_their_order(ora, form, E, k, d, T, gated, kind):
    # (the gate is one more row)
    assert capi.plan_batch(E + gated, k, d, 32, 32 if gated else 0, capi.WEIGHT_BF16, T)["router_f32"] == form
    W = S.make_weights(700 + E, E, d, 32, f_s=32 if gated else 0, gated=gated, router_std=1.0 / np.sqrt(d))
    W["w_router"] = S.bf16_round_trip(W["w_router"])[1]
    if gated:
        W["shared_gate"] = S.bf16_round_trip(W["shared_gate"])[1]
    conv = capi.CONVENTION_HUGGINGFACE_QWEN if gated else capi.CONVENTION_ATENIA
    oL, gL = S.build_pair(ora, W, k, conv, capi.WEIGHT_BF16)
    x = _rows(kind, T, d, W["w_router"])
    with gL:
        out = DeviceArray((T, d), np.float32, fill=0)
        dx = DeviceArray.from_host(x)
        gL.forward_device(dx.ptr, capi.ACT_F32, T, out.ptr)
        idx, w, *_ = gL.last_routing(T)
        o_idx, o_w = oL.route_tokens(x)
        assert (idx == o_idx).all(), f"{(idx != o_idx).any(axis=1).sum()} tokens routed differently"
        assert ulp_diff(w, o_w).max() <= 1
        if kind == "tiny":  # the same rows given as bf16: the same routing, the same outputs
            got = out.to_host()
            bits = DeviceArray.from_host((x.view(np.uint32) >> 16).astype(np.uint16))
            gL.forward_device(bits.ptr, capi.ACT_BF16, T, out.ptr)
            idx, w, *_ = gL.last_routing(T)
            assert (idx == o_idx).all() and ulp_diff(w, o_w).max() <= 1
            assert np.array_equal(got, out.to_host())


@pytest.mark.parametrize("wd,d,T", [(capi.WEIGHT_BF16, 72, 600), (capi.WEIGHT_INT8_W8A16, 96, 700),
                                    (capi.WEIGHT_INT8_W8A16, 128, 60), (capi.WEIGHT_BF16, 160, 2100)])
def test_bf16_copy_of_f32_rows(ora, wd, d, T):
    """The rows the experts read, padded to whole blocks of K, must be the nearest bf16 ones and zeros
    past d, whichever kernel stores them: f32 rows that hold bf16 values give the outputs of bf16 rows."""
    E, k = 40, 3
    W = S.make_weights(800 + d, E, d, 64, router_std=1.0 / np.sqrt(d))
    W["w_router"] = S.bf16_round_trip(W["w_router"])[1]
    _, gL = S.build_pair(ora, W, k, capi.CONVENTION_ATENIA, wd)
    x = S.make_tokens(810 + T, T, d, bf16=True)
    with gL:
        outs = []
        for rows, kind in ((DeviceArray.from_host(x), capi.ACT_F32),
                           (DeviceArray.from_host((x.view(np.uint32) >> 16).astype(np.uint16)), capi.ACT_BF16)):
            out = DeviceArray((T, d), np.float32, fill=0)
            gL.forward_device(rows.ptr, kind, T, out.ptr)
            outs.append(out.to_host())
    assert np.array_equal(*outs)


@pytest.mark.parametrize("E,k,d,T,gated", [(8, 2, 4096, 600, False), (60, 4, 2048, 300, True),
                                           (60, 4, 2048, 2100, True), (8, 2, 4096, 30, False)])
def test_large_products_that_cancel_keep_the_launch_short(ora, E, k, d, T, gated):
    """Two channels of large activations that cancel in every sum: the partial sums are thousands of times
    the result, about a third of the sums are flagged, and bf16 operands still give the same f32 in any order.
    A sum that falls to the reference's sequential order instead costs some 60 us, one after the other in its
    workgroup (the launches of more than 64 tokens took 95 to 170 times as long as on ordinary rows; now 5 to
    13 times)."""
    W = S.make_weights(900 + E, E, d, 32, f_s=32 if gated else 0, gated=gated, router_std=1.0 / np.sqrt(d))
    W["w_router"][:, 0] = np.sign(W["w_router"][:, 0])
    W["w_router"][:, 1] = -W["w_router"][:, 0]
    W["w_router"] = S.bf16_round_trip(W["w_router"])[1]
    if gated:
        W["shared_gate"] = S.bf16_round_trip(W["shared_gate"])[1]
    oL, gL = S.build_pair(ora, W, k, capi.CONVENTION_HUGGINGFACE_QWEN if gated else capi.CONVENTION_ATENIA,
                          capi.WEIGHT_BF16)
    x = S.make_tokens(910 + T, T, d, bf16=True)
    times = []
    with gL:
        gL.set_profiling(True)
        out = DeviceArray((T, d), np.float32, fill=0)
        for big in (0.0, 4096.0):
            x[:, :2] = big
            dx = DeviceArray.from_host((x.view(np.uint32) >> 16).astype(np.uint16))
            ms = []
            for _ in range(9):
                gL.forward_device(dx.ptr, capi.ACT_BF16, T, out.ptr)
                ms.append(gL.stage_ms()[0])
            times.append(float(np.median(ms)))
            idx, w, *_ = gL.last_routing(T)
            o_idx, o_w = oL.route_tokens(x)
            assert (idx == o_idx).all() and ulp_diff(w, o_w).max() <= 1, big
    assert times[1] <= 30 * times[0], times


@pytest.mark.parametrize("E,k,d,T,kind", [(8, 2, 40960, 300, capi.ACT_BF16), (8, 2, 33000, 250, capi.ACT_F32)])
def test_rows_of_more_than_64_pieces_are_bounded_too(ora, E, k, d, T, kind):
    """Rows of more than 32768 columns: the bound takes their pieces 64 at a time.  Where it left them out, every
    flagged sum walked the sequential order, several to a workgroup: 11 ms for the launch, 0.3 ms now."""
    W = S.make_weights(950 + E, E, d, 32, router_std=0.02)
    W["w_router"] = S.bf16_round_trip(W["w_router"])[1]
    oL, gL = S.build_pair(ora, W, k, capi.CONVENTION_ATENIA, capi.WEIGHT_BF16)
    x = S.make_tokens(960 + T, T, d, bf16=kind == capi.ACT_BF16)
    with gL:
        gL.set_profiling(True)
        out = DeviceArray((T, d), np.float32, fill=0)
        dx = DeviceArray.from_host((x.view(np.uint32) >> 16).astype(np.uint16) if kind == capi.ACT_BF16 else x)
        ms = []
        for _ in range(5):
            gL.forward_device(dx.ptr, kind, T, out.ptr)
            ms.append(gL.stage_ms()[0])
        idx, w, *_ = gL.last_routing(T)
        o_idx, o_w = oL.route_tokens(x)
        assert (idx == o_idx).all() and ulp_diff(w, o_w).max() <= 1
        assert np.median(ms) <= 3.0, ms
