"""The host entry point on batches that travel through the handle's own page-locked rows: the same
bits as the device entry point, at the ends of a piece and of the path, and the status words with them."""
import numpy as np
import pytest

from ateniaengine_amd import capi
from tests import synth as S
from tests.hipmem import DeviceArray

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("wd,d", [(capi.WEIGHT_F32, 6), (capi.WEIGHT_F32, 1021), (capi.WEIGHT_BF16, 1024)])
def test_small_host_batches_equal_the_device_entry(ora, wd, d):
    W = S.make_weights(d, 4, d, 32, router_std=1.0 / np.sqrt(d))
    _, gL = S.build_pair(ora, W, 2, capi.CONVENTION_ATENIA, wd)
    with gL:
        for T in (1, 64, 65, 512, 513, 515, 3, 64):  # 256 KiB and 2 MiB of d = 1024, and past them
            x = S.make_tokens(T + d, T, d, bf16=wd != capi.WEIGHT_F32)
            out = DeviceArray((T, d), np.float32, fill=0)
            rows = DeviceArray.from_host(x)
            gL.forward_device(rows.ptr, capi.ACT_F32, T, out.ptr)
            want = out.to_host()
            got = np.full((T, d), np.nan, np.float32)
            gL.forward(x, got)
            assert got.tobytes() == want.tobytes(), T


@pytest.mark.parametrize("wd,d,f_s", [
    (capi.WEIGHT_BF16, 64, 0),     # one token: the down launch of two experts that also combines
    (capi.WEIGHT_BF16, 64, 32),    # ... with a shared expert, two workgroups to a strip of rows
    (capi.WEIGHT_INT8_W8A16, 128, 64),
    (capi.WEIGHT_F32, 64, 0),      # the combine by whole fours, and by single columns
    (capi.WEIGHT_F32, 6, 0), (capi.WEIGHT_F32, 1030, 10)])
@pytest.mark.parametrize("T", [1, 5, 300])
def test_small_host_batches_report_non_finite_weights(ora, T, wd, d, f_s):
    W = S.make_weights(3, 4, d, 32, f_s=f_s)
    _, gL = S.build_pair(ora, W, 2, capi.CONVENTION_ATENIA, wd)
    x = S.make_tokens(4, T, d)
    bad = x.copy()
    bad[T - 1, 5] = np.inf
    with gL:
        want = gL.forward(x)
        with pytest.raises(capi.MoeHipError):
            gL.forward(bad)
        assert gL.last_non_finite()[0] == T - 1
        assert gL.forward(x).tobytes() == want.tobytes()  # cleared, and the next call is an ordinary one
        assert gL.status()[0] == capi.OK


def test_handles_in_turn_share_their_page_locked_rows(ora):
    """Four layers that announce small batches and are called in turn hold one set of rows between them."""
    d, T, n = 1024, 512, 4  # 2 MiB each way

    def mappings():  # of the rows' size: 4 MiB and the tail, in whole pages
        with open("/proc/self/smaps") as fh:
            return sum(l.split()[1] == "4100" for l in fh if l.startswith("Size:"))

    W = S.make_weights(7, 4, d, 32)
    before = mappings()
    layers = [S.build_pair(ora, W, 2, capi.CONVENTION_ATENIA, capi.WEIGHT_BF16, max_tokens_hint=T)[1] for _ in range(n)]
    x = S.make_tokens(8, T, d)
    outs = [gL.forward(x) for gL in layers]
    held = mappings()
    assert all(o.tobytes() == outs[0].tobytes() for o in outs)
    for gL in layers:
        gL.close()
    assert held - before <= 1  # (none if a handle that is still alive left a set)


def test_calls_at_once_have_rows_of_their_own(ora):
    """Host calls on several handles from several threads: the outputs of one call alone."""
    from concurrent.futures import ThreadPoolExecutor

    d, n = 256, 6
    W = S.make_weights(17, 4, d, 64)
    layers = [S.build_pair(ora, W, 2, capi.CONVENTION_ATENIA, capi.WEIGHT_BF16)[1] for _ in range(n)]
    xs = [S.make_tokens(18 + i, 1 + 100 * i, d) for i in range(n)]
    want = [layers[0].forward(x).tobytes() for x in xs]
    with ThreadPoolExecutor(n) as pool:
        for _ in range(5):
            got = list(pool.map(lambda i: layers[i].forward(xs[i]).tobytes(), range(n)))
            assert got == want
    for gL in layers:
        gL.close()
