"""Small batches whose gate/up launch groups the routed pairs by itself (wave_group_pairs, csrc/select_wave.h):
the lists it leaves and the outputs, at the edges of what it takes."""
import numpy as np
import pytest

from ateniaengine_amd import capi
from tests import synth as S
from tests.test_gpu_parity import TOL_BF16_TOY, TOL_F32, check_layer

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("wd", [capi.WEIGHT_BF16, capi.WEIGHT_INT8_W8A16, capi.WEIGHT_INT8_PER_GROUP, capi.WEIGHT_F32])
@pytest.mark.parametrize("E,k,T,f_s", [
    (2, 1, 2, 0),      # two pairs
    (16, 16, 16, 0),   # 256 pairs, every expert of every token
    (16, 16, 17, 0),   # 272: the launch of its own
    (16, 5, 51, 64),   # 255 pairs, four reads of the list, the last one short; a shared expert
    (64, 6, 8, 64),    # 48 pairs of up to 64 experts, most of them empty
    (64, 1, 48, 0),
    (33, 7, 7, 0),     # 49: the launch of its own
    (8, 4, 64, 128),   # the most rows an expert may have
    (1, 1, 64, 0),
    # the same for int8 and bf16 layers, whose larger batches take other kernels
    (16, 7, 36, 0), (16, 5, 51, 0), (8, 4, 39, 128), (1, 1, 39, 0), (64, 1, 39, 0),
])
def test_groups_and_outputs(ora, wd, E, k, T, f_s):
    d, f = 128, 128
    W = S.make_weights(6300 + E + T, E, d, f, f_s=f_s, gated=f_s > 0)
    conv = capi.CONVENTION_HUGGINGFACE_QWEN if f_s else capi.CONVENTION_ATENIA
    oL, gL = S.build_pair(ora, W, k, conv, wd)
    with gL:
        for seed in (0, 1):  # the second batch over what the first one left
            x = S.make_tokens(6400 + T + seed, T, d, bf16=wd != capi.WEIGHT_F32)
            check_layer(ora, oL, gL, x, TOL_F32 if wd == capi.WEIGHT_F32 else TOL_BF16_TOY)
            fits = T * k <= (256 if E <= 16 else 48) and gL.plan(T)["up"] in (capi.KERNELS_STREAM, capi.KERNELS_F32)
            reached = (gL.stage_launches()[1] == 0)
            assert reached == fits
        small = x[:max(1, T // 3)]  # and fewer tokens, whose lists are shorter
        check_layer(ora, oL, gL, small, TOL_F32 if wd == capi.WEIGHT_F32 else TOL_BF16_TOY)
        assert np.isfinite(gL.forward(x)).all()
