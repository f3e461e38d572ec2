"""GPU: the sizes at which a launch takes another kernel or a kernel another
branch (one-workgroup and sliced selection, one and several dot-product
chunks), against the oracle or a plain sort.  Bar: bit-exact."""

import numpy as np
import pytest
import torch

from oracle import oracle as O
from tests.helpers import log

pytestmark = pytest.mark.gpu

DEV = torch.device("cuda:0")


def _t(a):
    return torch.from_numpy(np.ascontiguousarray(a)).to(DEV)


# one workgroup of 1024 threads takes up to 32768 ratios, slices of 16384 more
@pytest.mark.parametrize("nb", [1, 2, 63, 1023, 1025, 32_767, 32_768, 32_769, 49_153, 70_001])
def test_thresholds_at_the_selection_sizes(nb):
    from turboadam_amd import costate as C

    log(f"thresholds nb={nb}")
    rng = np.random.default_rng(nb)
    base = np.abs(rng.standard_normal(nb)).astype(np.float32)
    two = np.where(np.arange(nb) < nb // 2, np.float32(0.5), np.float32(0.75)).astype(np.float32)
    nan = base.copy()
    nan[:: 3] = np.nan
    nan[1:: 7] = 0.0
    narrow = (np.float32(1.0).view(np.uint32) + rng.integers(0, 1 << 12, nb, dtype=np.uint32)).view(np.float32)
    for what, r in (("normal", base), ("two values", two), ("nan and zero", nan), ("narrow", narrow),
                    ("equal", np.full(nb, 0.37, np.float32))):
        for null_pct, amp_pct in ((0.1, 0.9), (0.05, 0.95), (0.0, 1.0)):
            k_lo, k_hi = O.ranks(nb, null_pct, amp_pct)
            keys = np.sort(r.view(np.uint32))
            got = [np.float32(x.item()).view(np.uint32) for x in C.compute_thresholds(_t(r), null_pct, amp_pct)]
            assert got == [keys[k_lo], keys[k_hi]], (what, null_pct)


# 8192 quarter-tile partials (of 512 elements) make one chunk of the dot products' tree
@pytest.mark.parametrize("n", [512 * 4, 512 * 1024 + 1, 512 * 8192, 512 * 8192 + 1, 512 * 8192 * 2 + 12_345])
def test_alpha_at_the_chunk_sizes(n):
    from turboadam_amd import costate as C

    log(f"alpha n={n}")
    rng = np.random.default_rng(n)
    g = rng.standard_normal(n, dtype=np.float32) * np.float32(1e-3)
    m = np.float32(0.4) * g + rng.standard_normal(n, dtype=np.float32) * np.float32(1e-4)
    delta_o = np.empty(n, np.float32)
    alpha_o = O.lib().or_decompose(O.ptr(m), O.ptr(g), n, O.ptr(delta_o))
    alpha, delta = C.decompose(_t(m), _t(g))
    assert np.float32(alpha.item()) == np.float32(alpha_o)
    assert np.array_equal(delta.cpu().numpy().view(np.uint32), delta_o.view(np.uint32))


# a tensor's last tile may hold quarters past its end, whose partial sums no kernel writes
@pytest.mark.parametrize("dt", [O.DT_F32, O.DT_BF16])
def test_step_reads_no_workspace_it_did_not_write(dt, monkeypatch):
    from tests.helpers import run_side_by_side
    from turboadam_amd import optimizer

    sizes = [1024 * 5, 1024 * 9, 4096 + 77, 512 * 9, 512 * 11 + 3, 2048 * 3, 128 * 33, 700]
    log(f"step on a workspace of NaN bytes, dtype {dt}")
    plain = optimizer._DeviceBuffers.workspace

    def poisoned(self, nbytes):
        ws = plain(self, nbytes)
        ws.fill_(255)
        return ws

    monkeypatch.setattr(optimizer._DeviceBuffers, "workspace", poisoned)
    for ef in (False, True):
        bad = run_side_by_side(sizes, [dt] * len(sizes), steps=3, error_feedback=ef)
        assert not bad, "\n".join(bad[:10])
