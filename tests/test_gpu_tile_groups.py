"""How the 256-row tiles (csrc/ffn_tiled.hip) cut an expert's rows: pairs of 32-row groups over the tiles,
the groups of a tile over its two wave rows.  The routing is fixed through the router so that the
experts see exactly the row counts at which those cuts fall."""
import numpy as np
import pytest

from ateniaengine_amd import capi
from tests import synth as S
from tests.test_gpu_parity import TOL_BF16_TOY, TOL_MODEL

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("counts,d,f,f_s,wd", [
    ((1, 32, 33, 96, 97, 160, 200, 256, 270), 128, 128, 0, capi.WEIGHT_BF16),     # one tile of 1 .. 9 groups
    ((289, 320, 352, 353, 400, 449, 0, 512, 513, 31), 192, 320, 0, capi.WEIGHT_BF16),  # two, and one of nine
    ((64, 129, 225, 255, 577, 640, 700), 128, 640, 300, capi.WEIGHT_BF16),        # beside a shared expert
    ((65, 128, 290, 410, 600, 33, 530), 256, 192, 0, capi.WEIGHT_INT8_W8A16),     # scaled outputs
])
def test_row_groups_over_tiles_and_wave_rows(ora, counts, d, f, f_s, wd):
    E, T = len(counts), sum(counts)
    W = S.make_weights(6000 + T + d, E, d, f, f_s=f_s, gated=f_s > 0)
    W["w_router"][:] = 0.0
    W["w_router"][np.arange(E), np.arange(E)] = 1.0  # expert e reads coordinate e of the token
    oL, gL = S.build_pair(ora, W, 1, capi.CONVENTION_HUGGINGFACE_QWEN, wd)
    with gL:
        x = S.make_tokens(6100 + T, T, d)
        want = np.random.default_rng(T).permutation(np.repeat(np.arange(E), counts))
        x[:, :E] = 0.0
        x[np.arange(T), want] = 4.0
        plan = gL.plan(T)
        assert plan["up"] == capi.KERNELS_TILED and plan["down"] == capi.KERNELS_TILED, plan
        out = gL.forward(x).reshape(T, d)
        idx, w, got, _, _ = gL.last_routing(T)
        assert (idx[:, 0] == want).all() and tuple(got) == tuple(counts)
        # the first and last rows of every expert, and some in between
        rows = [np.flatnonzero(want == e) for e in range(E)]
        sample = sorted({int(t) for r in rows if len(r) for t in r[np.linspace(0, len(r) - 1, 9).astype(int)]})
        split = gL.last_down_split(T) if plan["y_bf16"] else None
        if wd == capi.WEIGHT_BF16:
            model, slack = S.emulate_bf16_kernels(oL, x[sample], idx[sample], w[sample], with_slack=True,
                                                  y_bf16=plan["y_bf16"], ys_bf16=plan["ys_bf16"],
                                                  split=None if split is None else split[sample])
        for i, t in enumerate(sample):
            if wd == capi.WEIGHT_BF16:
                # the model's own bar: f32 summation order, plus what flips of h at a rounding midpoint move
                top = np.abs(model[i]).max()
                assert np.abs(out[t] - model[i]).max() <= TOL_MODEL * top + slack[i], (t, want[t])
            assert S.rel_err(out[t], oL.forward_f64(x[t], fixed_idx=idx[t])) <= TOL_BF16_TOY
