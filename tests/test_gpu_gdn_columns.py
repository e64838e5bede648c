"""The step kernel's columns per row (1, 2, 4 or 8, by tokens and sequences): a
sequence's bits do not depend on how many share the call, and the first lies
within the selftest's bar of float64."""
import numpy as np
import pytest
import torch

import xqattn
from conftest import case_note
from gdn_cases import make_gdn_case, out_array
from xqattn import workloads as wl

pytestmark = pytest.mark.gpu


def _run(case):
    dev = [xqattn.DevTensor.from_host(t) for t in (case.q, case.k, case.v, case.g, case.beta, case.state)]
    dst = xqattn.DevTensor.from_host(case.dst)
    xqattn.gated_delta_net(*dev, dst, case.slots, mode=xqattn.GDN_STEP)
    torch.cuda.synchronize()
    return out_array(case, dst.to_host_bytes())


def _first(case, n):
    """The first n sequences of a case."""
    def cut(t, d):
        ne = list(t.ne)
        ne[d] = n
        return wl.HostTensor(t.type, tuple(ne), t.nb, np.ascontiguousarray(t.buf[:t.nbytes * n // case.B]))
    ts = [cut(t, 3) for t in (case.q, case.k, case.v, case.g, case.beta, case.state)]
    return type(case)(case.T, case.slots, n, *ts, cut(case.dst, 2))


@pytest.mark.parametrize("bf16,pad", [(False, 0), (True, 0), (False, 3)])
@pytest.mark.parametrize("tokens,slots", [(1, 1), (2, 2), (8, 3), (9, 9), (21, 1)])
def test_gdn_step_columns(torch_gpu, tokens, slots, bf16, pad):
    case_note(f"step columns T {tokens} slots {slots} bf16 {bf16} pad {pad}")
    case = make_gdn_case(tokens, slots, B=13, bf16=bf16, pad=pad)
    full = _run(case)
    one = _first(case, 1)
    ref = one.oracle_f64()
    assert np.abs(_run(one) - ref)[np.isfinite(ref)].max() <= 1e-4 * np.abs(ref[np.abs(ref) < 1e20]).max()
    for n in (1, 3, 4, 6, 8, 12):  # every column count of both token ranges
        assert np.array_equal(_run(_first(case, n)), full[:n]), f"{n} sequences"
