"""Chunked prefill with one, two or four column tiles per workgroup (by sequences
and row type): every sequence's bits are those it has alone, where one tile runs,
for ragged lengths, padded and unaligned rows, and blocks that hold Inf or NaN."""
import numpy as np
import pytest
import torch

import xqattn
from conftest import case_note
from gdn_cases import make_gdn_case, out_array
from xqattn import workloads as wl

pytestmark = pytest.mark.gpu


def _run(case, n, b0=0, v_shift=0):
    """Sequences b0 .. b0 + n - 1 of a case; v_shift moves V off its alignment by that many bytes."""
    def part(t, d):
        per = t.nbytes // case.B
        ne = list(t.ne)
        ne[d] = n
        return wl.HostTensor(t.type, tuple(ne), t.nb, np.ascontiguousarray(t.buf[per * b0:per * (b0 + n)]))
    host = [part(t, 3) for t in (case.q, case.k, case.v, case.g, case.beta, case.state)]
    dev = [xqattn.DevTensor.from_host(t) for t in host]
    if v_shift:
        buf = torch.zeros(host[2].nbytes + 64, dtype=torch.uint8, device="cuda")
        buf[v_shift:v_shift + host[2].nbytes] = dev[2].t
        dev[2].t = buf[v_shift:]
    dst = xqattn.DevTensor.from_host(part(case.dst, 2))
    # nothing of the workspace is read before it is written (0xff: NaN in every type)
    size = xqattn.gated_delta_net_workspace(dev[0], dev[2], case.slots, xqattn.GDN_CHUNKED)
    ws = torch.full((size + 512,), 0xff, dtype=torch.uint8, device="cuda")
    xqattn.gated_delta_net(*dev, dst, case.slots, mode=xqattn.GDN_CHUNKED, workspace=ws)
    torch.cuda.synchronize()
    return out_array(type(case)(case.T, case.slots, n, *host, part(case.dst, 2)), dst.to_host_bytes())


@pytest.mark.parametrize("bf16,pad", [(True, 0), (True, 8), (True, 3), (False, 0), (False, 3)])
@pytest.mark.parametrize("tokens,slots", [(65, 1), (192, 1), (131, 4)])
def test_gdn_chunked_tiles_bits(torch_gpu, tokens, slots, bf16, pad):
    case_note(f"column tiles T {tokens} slots {slots} bf16 {bf16} pad {pad}")
    case = make_gdn_case(tokens, slots, B=8, bf16=bf16, pad=pad)
    alone = np.concatenate([_run(case, 1, b) for b in range(8)])
    ref = case.oracle_f64()
    live = np.abs(ref) < 1e20
    assert np.abs(alone - ref)[live].max() <= 1e-4 * np.abs(ref[live]).max()
    for n in (2, 3, 5, 6, 8):
        assert np.array_equal(_run(case, n), alone[:n]), f"{n} sequences"
    for shift in (2, 4) if bf16 else (4,):  # 2: V rows that take one tile
        assert np.array_equal(_run(case, 4, v_shift=shift), alone[:4]), f"V moved by {shift} bytes"


@pytest.mark.parametrize("bf16", [True, False])
def test_gdn_chunked_tiles_nonfinite_block(torch_gpu, bf16):
    """Non-finite v or state elements run their 16-column block token by token,
    whichever blocks share its workgroup; a q element far outside the chunk
    operands' range runs its whole (sequence, v-head) so."""
    def edit(v, st):
        v[1, 70, 3, 40] = np.nan
        st[2, 5, 100, 7] = np.inf
        v[3, 10, 31, 0] = -np.inf
    def qk(q, k):
        q[0, 20, 2] *= 1e5
    case_note(f"column tiles non-finite bf16 {bf16}")
    case = make_gdn_case(130, 1, B=4, bf16=bf16, vs_edit=edit, qk_edit=qk)
    alone = np.concatenate([_run(case, 1, b) for b in range(4)])
    assert np.isnan(alone).any() and np.isfinite(alone[1, :70]).all()
    got = _run(case, 4)
    assert np.array_equal(got.view(np.uint32)[~np.isnan(got)], alone.view(np.uint32)[~np.isnan(got)])
    assert np.array_equal(np.isnan(got), np.isnan(alone))


@pytest.mark.parametrize("pad", [0, 3])
@pytest.mark.parametrize("tokens", [960, 965, 1025])  # 15, 16 and 17 chunks
def test_gdn_chunked_tiles_long_bf16(torch_gpu, tokens, pad):
    """Two and six bf16 sequences take two column tiles from 16 chunks on, one below."""
    case_note(f"column tiles long T {tokens} pad {pad}")
    case = make_gdn_case(tokens, 1, B=6, bf16=True, pad=pad)
    alone = np.concatenate([_run(case, 1, b) for b in range(6)])
    for n in (2, 6):
        assert np.array_equal(_run(case, n), alone[:n]), f"{n} sequences"
