"""Range attention over quantized storage on the matrix cores: the f32 query
enters as f16 high + low parts times a power of two per query row, so neither
its magnitude nor the other rows of its tile may matter."""
import numpy as np
import pytest

import oracle
import xqattn
from conftest import case_note
from test_gpu_fa_range_random import range_f64
from xqattn import workloads as wl

pytestmark = pytest.mark.gpu


def _call(torch, q, positions, kraw, vraw, hkv, kv, origin, active, scale, split=xqattn.SPLIT_AUTO,
          engine=xqattn.ENGINE_AUTO):
    n_q, n_head, d = q.shape
    out = torch.empty(n_q, n_head, d, dtype=torch.float32, device="cuda")
    lse = torch.empty(n_q, n_head, dtype=torch.float32, device="cuda")
    xqattn.fa_range(torch.from_numpy(q).cuda(), torch.from_numpy(positions).cuda(), n_head,
                    torch.from_numpy(kraw.reshape(-1)).cuda(), torch.from_numpy(vraw.reshape(-1)).cuda(),
                    hkv, d, kv, origin, active, scale, out, lse, split_mode=split, engine=engine)
    torch.cuda.synchronize()
    return out.cpu().numpy(), lse.cpu().numpy()


@pytest.mark.parametrize("kv", [wl.Q8_0, wl.Q4_0], ids=lambda t: wl.TYPE_NAME[t])
@pytest.mark.parametrize("d,hkv,group,n_q,active", [
    (128, 2, 1, 1, 17),     # one pair of a tile, one row past a wave slice
    (128, 2, 4, 8, 300),    # 32 pairs: two pair tiles
    (256, 4, 6, 9, 1000),   # four pair tiles, two of them ending inside a query's heads
    (256, 1, 20, 2, 515),   # a group above 16 at head dim 256: two pair tiles, four waves
])
def test_fa_range_quant_query_scale(torch_gpu, kv, d, hkv, group, n_q, active):
    n_head, origin, scale = hkv * group, 500, float(1.0 / np.sqrt(d))
    kraw = oracle.quantize(kv, wl.normal(11, (active, hkv, d)))
    vraw = oracle.quantize(kv, wl.normal(12, (active, hkv, d)))
    q = wl.normal(13, (n_q, n_head, d))
    q[0, 0, 1::2] *= np.float32(2.0 ** -20)  # small elements beside large ones
    positions = np.arange(origin + active - n_q, origin + active, dtype=np.int32)
    case_note(f"range quant {wl.TYPE_NAME[kv]} D {d} G {group} n_q {n_q}")
    got, lse = _call(torch_gpu, q, positions, kraw, vraw, hkv, kv, origin, active, scale)
    kf = oracle.dequant(kv, kraw.reshape(-1, kraw.shape[-1]), d).reshape(active, hkv, d)
    vf = oracle.dequant(kv, vraw.reshape(-1, vraw.shape[-1]), d).reshape(active, hkv, d)
    ref, rlse = range_f64(q, positions, n_head, kf, vf, hkv, origin, active, scale)
    # 2^-22 per product of the scores (|score| < 2^4 here) and of the values: 1e-5 as in the other range tests
    assert np.abs(got - ref).max() < 1e-5 * np.abs(ref).max()
    assert np.abs(lse - rlse).max() < 1e-5 * np.abs(rlse).max()
    # a power of two on Q and its inverse on the scale change no bit
    for p in (-90, 60):
        g2, l2 = _call(torch_gpu, np.ldexp(q, p).astype(np.float32), positions, kraw, vraw, hkv, kv, origin, active,
                       float(np.ldexp(np.float32(scale), -p)))
        assert np.array_equal(g2, got) and np.array_equal(l2, lse), f"Q times 2^{p}"


@pytest.mark.parametrize("bad", [np.nan, np.inf, -np.inf])
@pytest.mark.parametrize("kv", [wl.Q8_0, wl.Q4_0], ids=lambda t: wl.TYPE_NAME[t])
def test_fa_range_quant_nonfinite_query_stays_in_its_rows(torch_gpu, kv, bad):
    n_q, hkv, group, d, active, origin = 3, 2, 6, 256, 400, 0
    n_head = hkv * group
    kraw = oracle.quantize(kv, wl.normal(21, (active, hkv, d)))
    vraw = oracle.quantize(kv, wl.normal(22, (active, hkv, d)))
    q = wl.normal(23, (n_q, n_head, d))
    positions = np.array([399, -1, 399], np.int32)
    clean, clse = _call(torch_gpu, q, positions, kraw, vraw, hkv, kv, origin, active, 1.0 / 16)
    q[0, 7, 200] = bad
    q[1, 3, 5] = bad  # a query that sees no row
    got, lse = _call(torch_gpu, q, positions, kraw, vraw, hkv, kv, origin, active, 1.0 / 16)
    assert np.isnan(got[0, 7]).all() and np.isnan(lse[0, 7])
    got[0, 7], lse[0, 7] = clean[0, 7], clse[0, 7]
    assert np.array_equal(got, clean) and np.array_equal(lse, clse)


@pytest.mark.parametrize("split", [xqattn.SPLIT_NONE, xqattn.SPLIT_REFERENCE], ids=["one_split", "splits"])
@pytest.mark.parametrize("kv", [wl.Q8_0, wl.Q4_0], ids=lambda t: wl.TYPE_NAME[t])
@pytest.mark.parametrize("d,hkv,group,n_q,active", [
    (128, 2, 1, 1, 17), (128, 2, 4, 8, 300), (128, 1, 12, 2, 64), (256, 4, 6, 9, 1000), (256, 1, 20, 2, 515),
    (256, 2, 3, 1, 1),
])
def test_fa_range_quant_engines(torch_gpu, kv, d, hkv, group, n_q, active, split):
    """The vector-ALU form (f32 Q and f32 products, which AUTO leaves to ranges beyond
    the matrix cores' row indices) and the matrix-core form: both within 1e-5 of
    float64, and a query's limit inside, before and past the rows."""
    n_head, origin, scale = hkv * group, 500, float(1.0 / np.sqrt(d))
    kraw = oracle.quantize(kv, wl.normal(31, (active, hkv, d)))
    vraw = oracle.quantize(kv, wl.normal(32, (active, hkv, d)))
    q = wl.normal(33, (n_q, n_head, d))
    positions = np.arange(origin + active - n_q, origin + active, dtype=np.int32)
    if n_q > 2:
        positions[:3] = origin + active // 2, origin - 1, origin + 5 * active
    kf = oracle.dequant(kv, kraw.reshape(-1, kraw.shape[-1]), d).reshape(active, hkv, d)
    vf = oracle.dequant(kv, vraw.reshape(-1, vraw.shape[-1]), d).reshape(active, hkv, d)
    ref, rlse = range_f64(q, positions, n_head, kf, vf, hkv, origin, active, scale)
    seen = np.isfinite(rlse)
    for engine in (xqattn.ENGINE_VALU, xqattn.ENGINE_MFMA):
        case_note(f"range quant {wl.TYPE_NAME[kv]} D {d} G {group} n_q {n_q} split {split} engine {engine}")
        got, lse = _call(torch_gpu, q, positions, kraw, vraw, hkv, kv, origin, active, scale, split, engine)
        assert np.abs(got - ref).max() < 1e-5 * np.abs(ref).max()
        assert np.array_equal(np.isfinite(lse), seen)
        assert np.abs(lse[seen] - rlse[seen]).max() < 1e-5 * np.abs(rlse[seen]).max()
    auto = _call(torch_gpu, q, positions, kraw, vraw, hkv, kv, origin, active, scale, split)
    assert np.array_equal(auto[0], got) and np.array_equal(auto[1], lse), "AUTO is the matrix cores"


@pytest.mark.parametrize("split", [xqattn.SPLIT_NONE, xqattn.SPLIT_REFERENCE], ids=["one_split", "splits"])
@pytest.mark.parametrize("signs", ["mixed", "same", "one_zero", "opposite"])
@pytest.mark.parametrize("scale_bits", [0x7C00, 0xFC00, 0x7E00], ids=["inf", "neg_inf", "nan"])
@pytest.mark.parametrize("kv", [wl.Q8_0, wl.Q4_0], ids=lambda t: wl.TYPE_NAME[t])
def test_fa_range_quant_nonfinite_k_scale(torch_gpu, kv, scale_bits, signs, split):
    """An Inf or NaN block scale in one K record. The block's 32 products are +-Inf or
    NaN each: a row whose products differ in sign, or that holds a zero, scores NaN;
    one sign scores +Inf (the query's rows are poisoned) or -Inf (weight 0). Both
    engines give the oracle's pattern, and its finite rows."""
    n_q, hkv, group, d, active, origin, row, blk = 4, 2, 6, 256, 700, 50, 400, 5
    n_head, scale = hkv * group, 1.0 / 16
    kraw = oracle.quantize(kv, wl.normal(41, (active, hkv, d)))
    vraw = oracle.quantize(kv, wl.normal(42, (active, hkv, d)))
    bb = kraw.shape[-1] // (d // 32)
    rec = kraw[row, 1, blk * bb:(blk + 1) * bb]
    rec[:2] = np.frombuffer(np.uint16(scale_bits).tobytes(), np.uint8)
    q = wl.normal(43, (n_q, n_head, d))
    if signs != "mixed":
        rec[2:] = np.arange(1, 33, dtype=np.uint8) if kv == wl.Q8_0 else 0x9F  # 1 .. 32; nibbles 7 and 1
        cut = q[:, :, 32 * blk:32 * blk + 32]
        cut[:] = np.abs(cut) * (-1.0 if signs == "opposite" else 1.0)
        if signs == "one_zero":
            cut[0, :, 7] = 0.0
            rec[4] = 0 if kv == wl.Q8_0 else 0x89
    positions = np.array([origin + 699, origin + row, origin + row - 1, origin + 5000], np.int32)
    want, wlse, _ = oracle.range_attn(q, positions, n_head, kraw, vraw, hkv, d, kv, origin, active, scale,
                                      xqattn.split_count(active, split))
    bad = np.isnan(wlse)
    assert not bad[2].any() and not bad[:, :group].any()
    inf = scale_bits != 0x7E00
    skipped = inf and signs in ("same", "opposite") and (scale_bits == 0xFC00) != (signs == "opposite")
    assert bad[0, group:].all() != skipped
    for engine in (xqattn.ENGINE_VALU, xqattn.ENGINE_MFMA):
        case_note(f"K scale {scale_bits:#x} {signs} {wl.TYPE_NAME[kv]} split {split} engine {engine}")
        got, lse = _call(torch_gpu, q, positions, kraw, vraw, hkv, kv, origin, active, scale, split, engine)
        assert np.array_equal(np.isnan(lse), bad) and np.isnan(got[bad]).all()
        assert np.abs(got[~bad] - want[~bad]).max() < 1e-5 * np.abs(want[~bad]).max()
        assert np.abs(lse[~bad] - wlse[~bad]).max() < 1e-5 * np.abs(wlse[~bad]).max()
