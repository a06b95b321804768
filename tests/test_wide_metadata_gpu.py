"""int64 metadata read in place gives exactly what its int32 conversion gives.

The kernels read the low words of int64 arrays. Each of the four metadata
tensors is passed as int64 alone and all together, on every kernel family that
reads them (one-token decode, token blocks, the chunk index and persistent
scan, the one-pass scan, the affine form), with entries outside the pool and
one that only its low word brings inside: outputs and pools equal bit for bit.
"""

import pytest
import torch

from tests import kda_cases as C

pytestmark = pytest.mark.gpu

DEV = "cuda"
META = ("initial_state_indices", "cu_seqlens", "track_state_indices", "track_state_lens")

# op, prefill, heads, lengths, tracked
CASES = {
    "decode": ("kda_varlen_recurrent", False, 16, (1,) * 9, False),
    "blocks": ("kda_varlen_recurrent", True, 4, (3, 0, 17, 40, 5), True),
    "persistent": ("kda_varlen_chunk", True, 9, (70, 1, 64, 130, 0, 65, 200, 5, 63), True),
    "one_pass": ("kda_varlen_chunk", True, 8, (300,), True),
    "affine": ("kda_varlen_chunk", True, 1, (6200,), True),
}


@pytest.mark.parametrize("name", list(CASES))
def test_int64_metadata_is_its_low_words(gpu_ops, name):
    op, prefill, heads, lengths, tracked = CASES[name]
    n = len(lengths)
    track = ([n + 1 + i for i in range(n)], [x // 2 + (x > 64) for x in lengths]) if tracked else None
    case = C.raw_case(heads, lengths, slots=2 * n + 2, seed=3, track=track)
    if n > 3:
        case.indices[1] = -4  # outside the pool: the padding slot

    def call(wide):
        kw = case.kwargs(DEV, pool=C.to_dev(case.pool, DEV))
        for m in META:
            if m in kw and m in wide:
                kw[m] = kw[m].long()
        if "initial_state_indices" in wide:
            kw["initial_state_indices"][0] += 1 << 32  # int32 keeps the low word
        out = getattr(gpu_ops, op)(prefill=prefill, **kw)
        return out, kw["initial_state_source"]

    out, pool = call(())
    for wide in [(m,) for m in META] + [META]:
        out64, pool64 = call(wide)
        assert torch.equal(out64, out), wide
        assert torch.equal(pool64, pool), wide
