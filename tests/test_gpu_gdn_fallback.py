"""Column blocks of the chunked prefill that run token by token: they read the
entering state before anything is written over it, and the blocks that share a
workgroup with them keep their bits."""
import numpy as np
import pytest
import torch

import xqattn
from conftest import case_note
from gdn_cases import make_gdn_case
from test_gpu_gdn_tiles import _run
from xqattn import workloads as wl

pytestmark = pytest.mark.gpu


def _same(a, b):
    return np.array_equal(np.isnan(a), np.isnan(b)) and \
        np.array_equal(a.view(np.uint32)[~np.isnan(a)], b.view(np.uint32)[~np.isnan(b)])


@pytest.mark.parametrize("bf16", [True, False])
@pytest.mark.parametrize("tokens", [65, 130])
def test_gdn_chunked_nonfinite_block_in_place(torch_gpu, tokens, bf16):
    """The entering state in the place where the final state goes (a program that
    keeps one buffer per sequence and length)."""
    def edit(v, st):
        v[0, 40, 3, 40] = np.inf
        st[0, 31, 100, 7] = np.nan
    case_note(f"in place, non-finite blocks T {tokens} bf16 {bf16}")
    case = make_gdn_case(tokens, 1, bf16=bf16, vs_edit=edit)
    want = _run(case, 1)
    assert np.isnan(want).any() and np.isfinite(want[:, :40]).any()
    dev = [xqattn.DevTensor.from_host(t) for t in (case.q, case.k, case.v, case.g, case.beta, case.state)]
    dst = xqattn.DevTensor.from_host(case.dst)
    at = dst.t[tokens * 16384:]
    at[:] = dev[5].t
    dev[5].t = at
    size = xqattn.gated_delta_net_workspace(dev[0], dev[2], 1, xqattn.GDN_CHUNKED)
    ws = torch.empty(size + 512, dtype=torch.uint8, device="cuda")
    xqattn.gated_delta_net(*dev, dst, 1, mode=xqattn.GDN_CHUNKED, workspace=ws)
    torch.cuda.synchronize()
    got = np.frombuffer(dst.to_host_bytes(), np.float32).reshape(want.shape)
    assert _same(got, want)


@pytest.mark.parametrize("bf16,seqs,tokens", [(True, 2, 131), (True, 2, 965), (True, 8, 131), (False, 2, 131)])
def test_gdn_chunked_several_nonfinite_blocks(torch_gpu, bf16, seqs, tokens):
    """Two blocks of one workgroup, all blocks of one, and none (two bf16 sequences take
    two column tiles from 16 chunks on)."""
    def edit(v, st):
        v[1, 70, 3, 5] = np.nan
        v[1, 3, 3, 55] = np.inf
        st[0, 9, ::16, 1] = -np.inf
    case_note(f"several non-finite blocks bf16 {bf16} B {seqs} T {tokens}")
    case = make_gdn_case(tokens, 1, B=seqs, bf16=bf16, vs_edit=edit)
    alone = np.concatenate([_run(case, 1, b) for b in range(seqs)])
    assert np.isnan(alone).any()
    assert _same(_run(case, seqs), alone)
