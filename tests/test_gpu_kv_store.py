"""The KV append's units: a wave converts 256-element units, one or (large appends to
records of 16 or 32 bits per element) four of them, so records end inside units and calls inside waves.
Bytes against the oracle's quantizers."""
import numpy as np
import pytest

import oracle
import xqattn
from xqattn import workloads as wl

pytestmark = pytest.mark.gpu


def _rows(n_tok, hkv, d, seed):
    """N(0, 9) rows with blocks whose largest magnitude appears twice with either
    sign (q4_0's scale is the first one's), an all-zero block and an Inf."""
    x = wl.normal(seed, (n_tok, hkv, d)) * np.float32(3.0)
    flat = x.reshape(-1, 32)
    flat[::5] = np.rint(flat[::5])
    flat[::7, 3] = -30.0
    flat[::7, 3 + 16] = 30.0
    flat[::11, 30] = 30.5
    flat[::11, 29] = -30.5
    if len(flat) > 40:
        flat[13] = 0.0
        flat[17, 9] = np.inf
    return x


@pytest.mark.parametrize("kv_type", [wl.F16, wl.BF16, wl.E5M2, wl.Q8_0, wl.Q4_0, wl.F32])
@pytest.mark.parametrize("n_tok,hkv,d,offset", [
    (1, 1, 64, 0),       # a quarter of one unit
    (3, 1, 128, 2),      # an odd record, a plane aligned to 2 bytes
    (5, 3, 256, 0),      # a wave past the last unit
    (4100, 4, 256, 0),   # four units per wave, the last wave partly past the end
    (10931, 6, 64, 0),   # the same with four records per unit, two of them past the end
])
def test_kv_store_unit_edges(torch_gpu, kv_type, n_tok, hkv, d, offset):
    torch = torch_gpu
    x = _rows(n_tok, hkv, d, 5)
    cap = n_tok + 3
    pos = np.random.RandomState(7).permutation(cap).astype(np.int32)[:n_tok]
    pos[n_tok // 2] = -1 if n_tok > 1 else pos[0]
    rec = wl.record_bytes(kv_type, d)
    want = np.full((cap, hkv, rec), 0xA5, np.uint8)
    if kv_type in (wl.BF16, wl.F32):
        bits = oracle.f32_to_bf16(x) if kv_type == wl.BF16 else x
        for t in range(n_tok):
            if pos[t] >= 0:
                want[pos[t]] = np.ascontiguousarray(bits[t]).view(np.uint8).reshape(hkv, rec)
    else:
        oracle.kv_store(x, pos, hkv, d, kv_type, want, cap, 0)
    buf = torch.full((want.size + 64,), 0xA5, dtype=torch.uint8, device="cuda")
    dst = buf[offset:]
    xqattn.kv_store(torch.from_numpy(x).cuda(), torch.from_numpy(pos).cuda(), hkv, d, kv_type, dst, cap)
    torch.cuda.synchronize()
    got = buf.cpu().numpy()
    assert np.array_equal(got[offset:offset + want.size].reshape(want.shape), want)
    assert (got[:offset] == 0xA5).all() and (got[offset + want.size:] == 0xA5).all()
