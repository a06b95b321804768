"""The affine form's output correction at the edges of its split.

A workgroup corrects two chunks of a later segment while all workgroups are
resident at once (two per CU), four beyond, eight waves on two chunks at a
time. The lengths lie on both sides of that line, with segments that leave one
chunk over for the last workgroup and a partial last chunk. The decay is weak,
so every later output depends on its segment's start state. Against the fp32
recurrence on the GPU (itself within 1e-5 of the oracle), at the contract's
tolerances.
"""

import dataclasses

import pytest
import torch

from tests import kda_cases as C

pytestmark = pytest.mark.gpu

DEV = "cuda"

# heads, sequence bounds, tokens: (P - 1) ceil(W / 2) H workgroups of 512 resident on 256 CUs
CASES = {
    "two_chunks_fill_the_line": (8, (0, 16384 - 20), 16384),  # P=2, W=128: 512
    "four_chunks_one_left_over": (8, (3, 16512 - 7), 16512),  # P=2, W=129: 520
    "two_chunks_odd_segment": (6, (0, 6208 - 63), 6208),  # P=3, W=33
    "four_chunks_many_segments": (4, (64, 22000), 22016),  # P=4, W=86: 516
}


@pytest.mark.parametrize("name", list(CASES))
def test_correction_split(gpu_ops, name):
    heads, bounds, T = CASES[name]
    case = C.raw_case(heads, (T,), indices=[1], slots=3, seed=41, lower_bound=-2e-4)
    case = dataclasses.replace(case, cu_seqlens=torch.tensor(bounds, dtype=torch.int32))
    got, want = C.to_dev(case.pool, DEV), C.to_dev(case.pool, DEV)
    out = gpu_ops.kda_varlen_chunk(prefill=True, **case.kwargs(DEV, pool=got))
    ref = gpu_ops.kda_varlen_recurrent(prefill=False, **case.kwargs(DEV, pool=want))
    torch.cuda.synchronize()
    # both are rounded to bf16: half an ulp (2^-9 of a value) each
    assert C.max_rel_err(out.cpu(), ref.cpu().float()) <= C.OUT_TOL + 2.0 ** -8
    C.assert_rel(got.cpu(), want.cpu(), C.STATE_TOL, name)
    assert torch.all(out[:, :bounds[0]] == 0) and torch.all(out[:, bounds[1]:] == 0)
