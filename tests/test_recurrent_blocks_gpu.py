"""The recurrent kernel's token blocks against the oracle, at their edges.

Several tokens per sequence run in blocks (16 tokens shared by a workgroup, or
four by a wave); the launcher picks the tile by gate form, pairs (requests x
heads), tokens per request, head dimension and, for decay gates, pool layout.
Each case sits in one branch of that choice, with lengths on both sides of a block's end, empty requests, a padding
request, uncovered tokens and tracked prefixes; v is also passed from an
address that no vector load may use. Tolerance: fp32 arithmetic on both sides
(sums of 128 products, at most 40 steps of a decaying recurrence), 1e-5 of the
largest value as for the other recurrent tests, output rounding aside.
"""

import pytest
import torch

from oracle import kda_ref as R
from tests import kda_cases as C

pytestmark = pytest.mark.gpu

DEV = "cuda"
TOL = 1e-5

# (heads, lengths, D): the branch that takes it
BLOCK_CASES = {
    "tile16": (3, (0, 1, 2, 15, 16, 17, 33), 128),
    "tile16_long": (8, (0, 1, 16, 40, 17, 33), 128),
    "tile32": (16, (1, 3, 4, 5, 15, 16, 17, 0, 31, 32, 33, 2), 128),
    "tile64": (32, (1, 3, 4, 5, 15, 16, 17, 0, 31, 32, 33, 2), 128),
    "tile128": (16, tuple([0, 1, 4, 5, 16, 17, 2, 3] * 5), 128),
    "tile64_many_long": (16, tuple([33, 16, 17, 40] * 9), 128),
    "wave": (64, tuple([0, 1, 2, 3, 4, 5, 8, 9] * 4), 128),
    "wave64": (64, tuple([0, 1, 2, 3, 4, 2, 1] * 4), 128),
    "tile128_many_short": (64, tuple([4, 5, 6, 7, 3, 5, 4, 6] * 4), 128),
    "tile128_many": (64, tuple([0, 5, 8, 9, 16, 4, 17, 1] * 4), 128),
    "d64_tile16": (2, (1, 16, 17, 5, 0), 64),
    "d64_tile64": (16, tuple([1, 4, 16, 17] * 4), 64),
}


def _track(lengths):
    n = len(lengths)
    return [n + 1 + i if i % 2 else 0 for i in range(n)], [min(x, 1 + 4 * (i % 5)) for i, x in enumerate(lengths)]


@pytest.mark.parametrize("aligned", [True, False])
@pytest.mark.parametrize("name", list(BLOCK_CASES))
def test_raw_blocks(gpu_ops, name, aligned):
    heads, lengths, D = BLOCK_CASES[name]
    n = len(lengths)
    indices = [i + 1 for i in range(n)]
    indices[1] = 0  # a padding request
    case = C.raw_case(heads, lengths, D=D, slots=2 * n + 2, indices=indices, seed=7, track=_track(lengths))
    kw = case.kwargs(DEV, pool=C.to_dev(case.pool, DEV))
    if not aligned:
        buf = torch.empty(case.v.numel() + 1, dtype=torch.bfloat16, device=DEV)
        kw["v"] = buf[1:].copy_(case.v.flatten()).view(case.v.shape)
    # the chunked form would take long prefills at D = 128; these stay below its 128 tokens a request
    out = gpu_ops.kda_varlen_recurrent(prefill=True, **kw)
    ref_pool = C.clone_pool(case.pool)
    q, k, g, beta = R.kda_prepare(case.A_log, case.a, case.dt_bias, case.q, case.k, case.b, case.lower_bound,
                                  case.scale)
    ref = R.kda_recurrent(q, k, case.v, g, beta, state_pool=ref_pool, state_indices=case.indices,
                          cu_seqlens=case.cu_seqlens, out_dtype=torch.float32, track_state_indices=case.track_indices,
                          track_state_lens=case.track_lens)
    C.assert_out(out.cpu(), ref, TOL, f"{name} output")
    C.assert_rel(kw["initial_state_source"].cpu(), ref_pool, TOL, f"{name} states")


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("heads,n,steps", [(4, 3, 4), (16, 16, 5), (16, 20, 3), (16, 30, 3), (16, 40, 4),
                                           (16, 40, 17), (16, 64, 12), (64, 32, 4), (64, 32, 6)])
def test_prepared_blocks_with_checkpoints(gpu_ops, heads, n, steps, dtype):
    lengths = [steps - (i % 3 if i % 4 == 1 else 0) for i in range(n)]
    D = 128
    case = C.prepared_case(heads, lengths, dtype=dtype, slots=n + 2, seed=9)
    # a row of uncovered tokens behind the last request
    pad = {x: torch.cat([getattr(case, x), getattr(case, x)[:, :2]], 1).to(DEV) for x in ("q", "k", "v", "g", "beta")}
    pool = C.to_dev(case.pool, DEV)
    mid = torch.full((n, steps, heads, D, D), 7.0, device=DEV).transpose(-1, -2)
    args = dict(initial_state_source=pool, initial_state_indices=case.indices.to(DEV),
                cu_seqlens=case.cu_seqlens.to(DEV), scale=case.scale)
    out = gpu_ops.kda_prepared_varlen_recurrent(*pad.values(), intermediate_state=mid, **args)
    assert torch.equal(pool.cpu(), case.pool), "checkpoints leave the pool as it is"
    assert not out[:, case.q.shape[1]:].any(), "uncovered tokens are zero"
    final = gpu_ops.kda_prepared_varlen_recurrent(*pad.values(), **args)
    assert torch.equal(final, out)
    ref_pool = C.clone_pool(case.pool)
    ref = R.kda_recurrent(case.q.float() * case.scale, case.k.float(),
                          case.v.float(), case.g, case.beta, state_pool=ref_pool, state_indices=case.indices,
                          cu_seqlens=case.cu_seqlens, out_dtype=torch.float32)
    C.assert_out(out[:, :case.q.shape[1]].cpu(), ref, TOL, "output")
    C.assert_rel(pool.cpu(), ref_pool, TOL, "states")
    for i, length in enumerate(lengths):
        assert torch.equal(mid[i, length - 1], pool[int(case.indices[i])]), "the last checkpoint is the final state"
        assert (mid[i, length:] == 7.0).all(), "steps beyond the request stay"


@pytest.mark.parametrize("k_contiguous", [True, False])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("n,steps", [(11, 1), (12, 1), (20, 1), (40, 1), (32, 3), (64, 5), (75, 4), (100, 3), (160, 3),
                                     (300, 9), (512, 4)])
def test_decay_blocks(gpu_ops, n, steps, dtype, k_contiguous):
    """``prepared_recurrent`` (four heads) over its tiles and one-token shapes, on
    both pool layouts, with ragged lengths, a padding request, uncovered tokens and tracked prefixes."""
    H, D = 4, 128
    lengths = [max(0, steps - (i % 3 if i % 4 == 1 else 0)) for i in range(n)]
    case = C.prepared_case(H, lengths, dtype=torch.float32, slots=2 * n + 1, seed=19)
    indices = case.indices.clone()
    indices[2] = 0
    track = _track(lengths)
    track = [torch.tensor(x, dtype=torch.int32) for x in track]
    pool = C.to_dev(case.pool, DEV) if k_contiguous else case.pool.contiguous().to(DEV)
    T = case.q.shape[1]
    pad = lambda x: torch.cat([x, x[:, :2]], 1).to(DEV)  # noqa: E731  two tokens no request covers
    v = case.v.to(dtype)
    out = torch.full((1, T + 2, H, D), 3.0, dtype=dtype, device=DEV)
    gpu_ops.prepared_recurrent(pad(case.q * case.scale), pad(case.k), pad(v), pad(case.g.exp()), pad(case.beta), out, pool,
                               indices.to(DEV), case.cu_seqlens.to(DEV), track[0].to(DEV), track[1].to(DEV), True, 0)
    ref_pool = C.clone_pool(case.pool)
    ref = R.kda_recurrent(case.q * case.scale, case.k, v.float(), case.g, case.beta, state_pool=ref_pool,
                          state_indices=indices, cu_seqlens=case.cu_seqlens, out_dtype=torch.float32,
                          track_state_indices=track[0], track_state_lens=track[1])
    assert (out[:, T:] == 3.0).all(), "uncovered rows stay"
    check = C.assert_out if dtype == torch.bfloat16 else C.assert_rel
    check(out[:, :T].cpu(), ref, TOL, "output")
    C.assert_rel(pool.cpu(), ref_pool, TOL, "states")
