"""The split merge at the edges of its chunk sizes (4, 16, 32, 64 splits in one
pass, 64 at a time beyond), with splits that hold no state at the end."""
import numpy as np
import pytest

import oracle
import xqattn
from conftest import case_note
from test_gpu_fa_range_quant import _call
from test_gpu_fa_range_random import range_f64
from xqattn import workloads as wl

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("d", [128, 256])
@pytest.mark.parametrize("splits", [2, 4, 5, 16, 17, 32, 33, 64, 65, 128, 129, 256])
def test_fa_reduce_split_counts(torch_gpu, splits, d):
    hkv, n_head, origin = 1, 2, 10
    active = 32 * splits  # the fine mode's 32 rows per split
    assert xqattn.split_count(active, xqattn.SPLIT_FINE) == splits
    case_note(f"reduce {splits} splits D {d}")
    kraw = oracle.quantize(wl.F16, wl.normal(31, (active, hkv, d)))
    vraw = oracle.quantize(wl.F16, wl.normal(32, (active, hkv, d)))
    q = wl.normal(33, (3, n_head, d)) * np.float32(3.0)
    # the last row, the last row of the split before the last, and the first split alone
    positions = np.array([origin + active - 1, origin + active - 33, origin + 7], np.int32)
    got, lse = _call(torch_gpu, q, positions, kraw, vraw, hkv, wl.F16, origin, active, 1.0 / 16, xqattn.SPLIT_FINE)
    kf = oracle.dequant(wl.F16, kraw.reshape(-1, kraw.shape[-1]), d).reshape(active, hkv, d)
    vf = oracle.dequant(wl.F16, vraw.reshape(-1, vraw.shape[-1]), d).reshape(active, hkv, d)
    ref, rlse = range_f64(q, positions, n_head, kf, vf, hkv, origin, active, 1.0 / 16)
    assert np.abs(got - ref).max() < 1e-5 * np.abs(ref).max()
    assert np.abs(lse - rlse).max() < 1e-5 * np.abs(rlse).max()
    # an Inf in the last split reaches the first query alone, in full
    vraw[-1, 0, :2] = (0x00, 0x7c)
    bad, blse = _call(torch_gpu, q, positions, kraw, vraw, hkv, wl.F16, origin, active, 1.0 / 16, xqattn.SPLIT_FINE)
    assert np.isnan(bad[0]).all() and np.isnan(blse[0]).all()
    assert np.array_equal(bad[1:], got[1:]) and np.array_equal(blse[1:], lse[1:])
