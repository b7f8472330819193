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


def test_page_locked_rows_only_where_the_host_entry_is_called(ora):
    """A layer made with a hint of small batches holds no page-locked rows until its host entry is called."""
    d, T, n = 1024, 512, 4  # 2 MiB each way

    def mappings():  # of the rows' size: 4 MiB and the tail, in whole pages
        with open("/proc/self/smaps") as fh:
            return sum(l.split()[1] == "4100" for l in fh if l.startswith("Size:"))

    W = S.make_weights(7, 4, d, 32)
    before = mappings()
    layers = [S.build_pair(ora, W, 2, capi.CONVENTION_ATENIA, capi.WEIGHT_BF16, max_tokens_hint=T)[1] for _ in range(n)]
    made = mappings()
    x = S.make_tokens(8, T, d)
    for gL in layers:
        gL.forward(x)
    called = mappings()
    for gL in layers:
        gL.close()
    assert (made - before, called - before, mappings() - before) == (0, n, 0)
