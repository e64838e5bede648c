"""Pair tiles: whole queries, or 16 or 32 (query, head) pairs packed across queries
(a tile may end inside a query's heads) where that saves a round of workgroups. A
query's bits are those it has alone, and all of them are within 1e-5 of float64."""
import dataclasses

import numpy as np
import pytest

import xqattn
from conftest import case_note
from fa_cases import make_fa_case, oracle_f64, run_fa_gpu
from xqattn import workloads as wl

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("kv", [wl.Q8_0, wl.Q4_0, wl.F16, wl.E5M2], ids=lambda t: wl.TYPE_NAME[t])
@pytest.mark.parametrize("d,group,n_q", [
    (256, 6, 3),   # 18 pairs: the second tile holds two
    (256, 6, 8),   # 48: three full tiles
    (256, 5, 7),   # 35: tiles ending in queries 3 and 6
    (256, 1, 17),  # one head per KV head: 16 queries and one more
    (128, 12, 6),  # 72 over tiles of 32
    (128, 31, 3),  # 93, a group that does not divide the tile
])
def test_fa_pair_tiles(torch_gpu, kv, d, group, n_q):
    hkv, rows = 2, 403
    cfg = wl.FaConfig("pairs", n_q, hkv * group, hkv, d, rows, 1, kv, causal_prefix=rows - n_q)
    case_note(f"pair tiles {wl.TYPE_NAME[kv]} D {d} G {group} n_q {n_q}")
    case = make_fa_case(cfg, seed=41)
    got, _ = run_fa_gpu(case, torch_gpu)
    ref, _ = oracle_f64(case)
    assert np.abs(got - ref).max() < 1e-5 * np.abs(ref).max()
    for i in (0, n_q - 1):
        one = wl.FaConfig("one", 1, hkv * group, hkv, d, rows, 1, kv, causal_prefix=rows - n_q + i)
        q = np.frombuffer(case.q.buf.tobytes(), np.float32).reshape(1, n_q, hkv * group, d)
        alone = make_fa_case(one, seed=41)
        alone.q, alone.k, alone.v = wl.fa_q_tensor(q[:, i:i + 1]), case.k, case.v
        alone.mask = wl.mask_tensor(wl.fa_causal_mask(one))
        bits, _ = run_fa_gpu(alone, torch_gpu)
        assert np.array_equal(bits[:, 0], got[:, i]), f"query {i}"


@pytest.mark.parametrize("kv", [wl.Q8_0, wl.Q4_0, wl.F16, wl.E5M2], ids=lambda t: wl.TYPE_NAME[t])
@pytest.mark.parametrize("d,group,n_q,seqs", [
    (256, 6, 8, 20),   # 2 splits x 2 KV heads: 4 whole tiles are 320 workgroups, 3 packed ones 240
    (256, 5, 16, 11),  # 6 whole, 5 packed: 264, 220
    (128, 12, 8, 17),  # 4 whole, 3 packed tiles of 32: 272, 204
])
def test_fa_pair_tiles_packed(torch_gpu, kv, d, group, n_q, seqs):
    """A batch whose tiles are packed, and each of its sequences alone in whole tiles."""
    hkv, rows = 2, 403
    cfg = wl.FaConfig("packed", n_q, hkv * group, hkv, d, rows, seqs, kv, causal_prefix=rows - n_q)
    case_note(f"packed pair tiles {wl.TYPE_NAME[kv]} D {d} G {group} n_q {n_q} B {seqs}")
    case = make_fa_case(cfg, seed=43)
    got, _ = run_fa_gpu(case, torch_gpu)
    one = dataclasses.replace(cfg, B=1)
    rec = wl.record_bytes(kv, d)
    q = np.frombuffer(case.q.buf.tobytes(), np.float32).reshape(seqs, n_q, hkv * group, d)
    k, v = (np.frombuffer(t.buf.tobytes(), np.uint8).reshape(seqs, rows, hkv, rec) for t in (case.k, case.v))
    for b in (0, seqs - 1):
        alone = make_fa_case(one, seed=43)
        alone.q = wl.fa_q_tensor(q[b:b + 1])
        alone.k, alone.v = (wl.kv_tensor(x[b:b + 1].copy(), kv, d) for x in (k, v))
        alone.mask = wl.mask_tensor(wl.fa_causal_mask(one))
        bits, _ = run_fa_gpu(alone, torch_gpu)
        assert np.array_equal(bits[0], got[b]), f"sequence {b}"
        ref, _ = oracle_f64(alone)
        assert np.abs(bits - ref).max() < 1e-5 * np.abs(ref).max()
