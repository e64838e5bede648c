"""Mask rows that start in the middle of a dword (odd KV lengths, views two bytes
into a buffer): the bits of the same mask laid out on 4 bytes, at the ends of a
wave slice and of the call, with rows masked there."""
import numpy as np
import pytest

import xqattn
from conftest import case_note
from fa_cases import dst_array, make_fa_case
from xqattn import workloads as wl

pytestmark = pytest.mark.gpu


def _run(torch, case, mask, softcap=0.0):
    dev = [xqattn.DevTensor.from_host(t) for t in (case.q, case.k, case.v)]
    d = xqattn.DevTensor.empty_like_host(case.dst)
    xqattn.flash_attn_ext(*dev, mask, None, d, xqattn.fa_params(case.scale, softcap=softcap))
    torch.cuda.synchronize()
    return dst_array(case, d.to_host_bytes())


@pytest.mark.parametrize("kv", [wl.Q8_0, wl.Q4_0, wl.F16, wl.E5M2], ids=lambda t: wl.TYPE_NAME[t])
@pytest.mark.parametrize("d,hkv,group,n_q,rows", [
    (128, 1, 4, 1, 1), (128, 2, 2, 3, 17), (128, 2, 4, 8, 255), (256, 2, 6, 4, 129), (256, 1, 6, 2, 431),
    (256, 1, 20, 1, 143), (128, 2, 4, 2, 256),
])
def test_fa_mask_alignment(torch_gpu, kv, d, hkv, group, n_q, rows):
    torch = torch_gpu
    cfg = wl.FaConfig("mask", n_q, hkv * group, hkv, d, rows, 1, kv, causal_prefix=max(0, rows - n_q))
    case_note(f"mask alignment {wl.TYPE_NAME[kv]} D {d} G {group} n_q {n_q} rows {rows}")
    case = make_fa_case(cfg, seed=51)
    bits = wl.fa_causal_mask(cfg)[0].copy()
    rng = np.random.RandomState(3)
    bits[:, rng.rand(rows) < 0.2] = np.float16(-1.5).view(np.uint16)
    if rows > 2:
        bits[0, rows // 2] = bits[n_q - 1, 1] = 0xFC00
    pitch = rows + (rows & 1) + 2
    flat = np.full((n_q, pitch), 0x7E00, np.uint16)  # NaN around the rows
    flat[:, :rows] = bits
    def view(off, row_pitch, src):
        buf = torch.full((off + src.size + 8,), 0x7E00, dtype=torch.int16, device="cuda")
        buf[off:off + src.size] = torch.from_numpy(np.ascontiguousarray(src).reshape(-1).view(np.int16)).cuda()
        t = xqattn.DevTensor(wl.F16, (rows, n_q, 1, 1), (2, 2 * row_pitch, 2 * row_pitch * n_q, 2 * row_pitch * n_q), buf)
        t.t = buf[off:]
        return t
    for softcap in (0.0, 5.0):  # softcap: the rows are re-laid first
        want = _run(torch, case, view(2, pitch, flat), softcap)
        assert np.isfinite(want).all()
        odd = rows + 1 - (rows & 1) if rows & 1 else rows + 1
        tight = np.full((n_q, odd), 0x7E00, np.uint16)
        tight[:, :rows] = bits
        for off, p, src in ((0, odd, tight), (1, odd, tight), (1, pitch, flat)):
            assert np.array_equal(_run(torch, case, view(off, p, src), softcap), want), (off, p, softcap)


def test_fa_mask_misaligned_rows_far_apart(torch_gpu):
    """Two mask rows 2^31 + 2 bytes apart: beyond the 32-bit offsets the kernel reads
    masks with, so their rows are re-laid, as before."""
    torch = torch_gpu
    rows, n_q, pitch = 131, 2, (1 << 30) + 1
    cfg = wl.FaConfig("mask", n_q, 4, 2, 128, rows, 1, wl.Q8_0, causal_prefix=rows - n_q)
    case_note("mask rows 2^31 + 2 bytes apart")
    case = make_fa_case(cfg, seed=52)
    bits = np.ascontiguousarray(wl.fa_causal_mask(cfg)[0][:, :rows]).view(np.int16)
    def view(row_pitch):
        buf = torch.empty((n_q - 1) * row_pitch + rows + 9, dtype=torch.int16, device="cuda")
        for i in range(n_q):
            buf[i * row_pitch:i * row_pitch + rows] = torch.from_numpy(bits[i].copy()).cuda()
        return xqattn.DevTensor(wl.F16, (rows, n_q, 1, 1), (2, 2 * row_pitch, 2 * row_pitch * n_q, 2 * row_pitch * n_q), buf)
    assert np.array_equal(_run(torch, case, view(pitch)), _run(torch, case, view(rows + 1)))


@pytest.mark.parametrize("kv", [wl.Q8_0, wl.Q4_0, wl.F16, wl.E5M2], ids=lambda t: wl.TYPE_NAME[t])
@pytest.mark.parametrize("planes,step", [
    ("seq", 2),   # one plane per sequence, nb[3] = 2 mod 4
    ("head", 2),  # one plane per head, nb[2] = 2 mod 4
    ("row", 1),   # strides of an odd number of bytes: elements between byte boundaries of halves
    ("seq", 1),
])
def test_fa_mask_plane_strides(torch_gpu, kv, planes, step):
    """Masks whose planes lie `step` mod 4 bytes apart: the bits of the same mask on
    4-byte aligned rows. Two sequences, three queries, per-sequence or per-head planes."""
    torch = torch_gpu
    rows, n_q, heads, seqs = 141, 3, 8, 2
    cfg = wl.FaConfig("mask", n_q, heads, 2, 128, rows, seqs, kv, causal_prefix=rows - n_q)
    case_note(f"mask planes {planes} {step} mod 4 {wl.TYPE_NAME[kv]}")
    case = make_fa_case(cfg, seed=53)
    n2, n3 = (heads, 1) if planes == "head" else (1, seqs)
    rng = np.random.RandomState(5)
    bits = np.where(rng.rand(n3, n2, n_q, rows) < 0.3, np.uint16(0xFC00),
                    rng.randn(n3, n2, n_q, rows).astype(np.float16).view(np.uint16)).astype(np.uint16)
    bits[..., 7] = 0  # every query sees a row
    def view(nb1, nb2, nb3):
        buf = np.full(nb3 * n3 + 64, 0x7E, np.uint8)  # NaN between the rows
        for i3 in range(n3):
            for i2 in range(n2):
                for i in range(n_q):
                    at = i3 * nb3 + i2 * nb2 + i * nb1
                    buf[at:at + 2 * rows] = bits[i3, i2, i].view(np.uint8)
        return xqattn.DevTensor(wl.F16, (rows, n_q, n2, n3), (2, nb1, nb2, nb3), torch.from_numpy(buf).cuda())
    row = 2 * rows + 2  # a multiple of 4
    want = _run(torch, case, view(row, n_q * row, n2 * n_q * row))
    assert np.isfinite(want).all()
    nb1 = row + (step if planes == "row" else 0)
    nb2 = n_q * nb1 + (step if planes == "head" else 0)
    nb3 = n2 * nb2 + (step if planes == "seq" else 0)
    assert max(nb1 % 4 if planes == "row" else 0, nb2 % 4 if planes == "head" else 0,
               nb3 % 4 if planes == "seq" else 0) == step
    assert np.array_equal(_run(torch, case, view(nb1, nb2, nb3)), want)


def test_fa_mask_relay_many_rows(torch_gpu):
    """2^23 mask rows of 1025 elements to re-lay (softcap, rows of 2 mod 4 bytes): two
    parts a row would be 2^24 workgroups of 256 threads, one more than a launch
    holds. Every sequence reads the same Q, K, V and mask (strides of 0), so all of
    them give the bits of the call with one."""
    torch = torch_gpu
    rows, n_q, heads, d, seqs = 1025, 8, 32, 128, 32768
    cfg = wl.FaConfig("many", n_q, heads, 1, d, rows, 1, wl.F16, causal_prefix=rows - n_q)
    case_note("2^23 mask rows to re-lay")
    case = make_fa_case(cfg, seed=54)
    params = xqattn.fa_params(case.scale, softcap=5.0, split_mode=xqattn.SPLIT_NONE)
    q, k, v, m = (xqattn.DevTensor.from_host(t) for t in (case.q, case.k, case.v, case.mask))
    one = xqattn.DevTensor.empty_like_host(case.dst)
    xqattn.flash_attn_ext(q, k, v, m, None, one, params)
    many = [xqattn.DevTensor(t.type, (*t.ne[:3], seqs), (*t.nb[:3], 0), t.t) for t in (q,)]
    many += [k, v, xqattn.DevTensor(m.type, (rows, n_q, heads, seqs), (2, m.nb[1], 0, 0), m.t)]
    assert m.nb[1] == 2 * rows
    out = torch.zeros(seqs, n_q * heads * d, dtype=torch.float32, device="cuda")
    dst = xqattn.DevTensor(wl.F32, (d, heads, n_q, seqs), (4, 4 * d, 4 * d * heads, 4 * d * heads * n_q),
                           out.view(torch.uint8).reshape(-1))
    xqattn.flash_attn_ext(*many, None, dst, params)
    torch.cuda.synchronize()
    want = one.t.view(torch.int32).reshape(-1)
    assert (want != 0).any()
    for s in range(0, seqs, 1024):
        assert (out[s:s + 1024].view(torch.int32) == want).all(), f"sequences from {s}"
