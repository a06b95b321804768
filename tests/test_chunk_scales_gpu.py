"""The chunk kernels' fp16 operands where magnitudes differ within one chunk.

e^G k and q e^G carry one power-of-two scale per 16-row tile and channel half,
kd one per 16 channels, Aqk one per 16-row tile, and y the bound that max |v|,
max |S| and the rows' sums of |e^G k| give. Here a chunk mixes magnitudes that
one scale for all of it could not hold (fp16 keeps its bits down to 2^-28 of
the scaled value's bound and is zero below 2^-38), and takes log decays above
zero, which make the factors grow instead of shrink. Each tile (each channel
group of a state) is compared on its own with the 64-bit oracle at the
tolerance contract, whose budget is relative to the largest value compared.
"""

import dataclasses

import pytest
import torch

from oracle import kda_ref as R
from tests import kda_cases as C

pytestmark = pytest.mark.gpu

DEV = "cuda"
LENGTHS = (128, 37, 64)


def _case(**more):
    case = C.prepared_case(2, LENGTHS, slots=8, indices=[1, 3, 2], seed=61)
    return dataclasses.replace(case, **{k: f(getattr(case, k)) for k, f in more.items()})


def _run(gpu_ops, case, l2norm=False):
    """Output, pool and their 64-bit references; every request's prefix of 21 tokens tracked."""
    track = (torch.tensor([4, 5, 6], dtype=torch.int32), torch.full((3,), 21, dtype=torch.int32))
    pool = C.to_dev(case.pool, DEV)
    out = gpu_ops.kda_prepared_varlen_chunk(
        case.q.to(DEV), case.k.to(DEV), case.v.to(DEV), case.g.to(DEV), case.beta.to(DEV),
        initial_state_source=pool, initial_state_indices=case.indices.to(DEV), cu_seqlens=case.cu_seqlens.to(DEV),
        scale=case.scale, use_qk_l2norm=l2norm, track_state_indices=track[0].to(DEV), track_state_lens=track[1].to(DEV))
    q, k = case.q.double(), case.k.double()
    if l2norm:
        q, k = (x / torch.sqrt((x * x).sum(-1, keepdim=True) + 1e-6) for x in (q, k))
    ref_pool = C.clone_pool(case.pool).double()
    ref = R.kda_recurrent(q * case.scale, k, case.v.double(), case.g.double(), case.beta.double(),
                          state_pool=ref_pool, state_indices=case.indices, cu_seqlens=case.cu_seqlens,
                          track_state_indices=track[0], track_state_lens=track[1], dtype=torch.float64,
                          out_dtype=torch.float64)
    assert torch.isfinite(out).all() and torch.isfinite(pool).all()
    return out.cpu(), pool.cpu(), ref, ref_pool


def _tiles(out, ref, what):
    for bos, eos in zip((0,) + tuple(torch.tensor(LENGTHS).cumsum(0).tolist()), torch.tensor(LENGTHS).cumsum(0).tolist()):
        for t in range(bos, eos, 16):
            rows = slice(t, min(t + 16, eos))
            C.assert_out(out[:, rows], ref[:, rows], C.OUT_TOL, f"{what}, rows {t - bos} of a request")


def _spread_rows(x):
    """Rows scaled by 2^0, 2^-20, 2^-45, 2^0 in turn, sixteen rows each."""
    t = torch.cat([torch.arange(n) for n in LENGTHS])
    return (x.float() * torch.tensor([1.0, 2.0 ** -20, 2.0 ** -45, 1.0])[t // 16 % 4][None, :, None, None]).to(x.dtype)


@pytest.mark.parametrize("pool_scale", [0.0, 1.0])
def test_q_rows_of_unlike_magnitude(gpu_ops, pool_scale):
    """q e^G and Aqk: a tile of small q rows beside large ones keeps its outputs."""
    case = _case(q=_spread_rows, pool=lambda p: C.clone_pool(p * pool_scale))
    out, pool, ref, ref_pool = _run(gpu_ops, case)
    _tiles(out, ref, "q rows")
    C.assert_rel(pool, ref_pool, C.STATE_TOL, "pool")


def test_k_channels_of_unlike_magnitude(gpu_ops):
    """kd and the tracked prefix's kd: the state's rows of a small channel group beside large ones."""
    factor = torch.tensor([1.0, 2.0 ** -15, 2.0 ** -30, 2.0 ** -45] * 2).repeat_interleave(16)
    case = _case(k=lambda k: (k.float() * factor).to(k.dtype), pool=lambda p: C.clone_pool(p * 0.0))
    out, pool, ref, ref_pool = _run(gpu_ops, case)
    _tiles(out, ref, "k channels")
    for slot in range(1, 7):
        for k in range(0, 128, 16):
            C.assert_rel(pool[slot, :, k:k + 16], ref_pool[slot, :, k:k + 16], C.STATE_TOL, f"slot {slot}, rows {k}")


def test_readout_far_below_the_chunks_start(gpu_ops):
    """q e^G decaying by 2^-46 over a chunk (beta = 0: the outputs are the initial state's alone)."""
    case = _case(g=lambda g: torch.full_like(g, -0.5), beta=torch.zeros_like)
    out, pool, ref, ref_pool = _run(gpu_ops, case)
    _tiles(out, ref, "decay")
    C.assert_rel(pool, ref_pool, C.STATE_TOL, "pool")


def test_small_values_after_a_reset(gpu_ops):
    """y's scale: a first token that forgets a large state leaves the small values their bits."""
    def reset(g):
        g = g.clone()
        g[:, [0, 128, 165]] = -40.0
        return g

    case = _case(g=reset, v=lambda v: (v.float() * 1e-3).to(v.dtype), pool=lambda p: C.clone_pool(p * 1e7))
    out, pool, ref, ref_pool = _run(gpu_ops, case)
    _tiles(out, ref, "after a reset")
    for slot in range(1, 7):
        C.assert_rel(pool[slot], ref_pool[slot], C.STATE_TOL, f"slot {slot}")


@pytest.mark.parametrize("l2norm", [False, True])
@pytest.mark.parametrize("g_up", [0.05, 0.3, 0.6, 2.0])
def test_some_log_decays_above_zero(gpu_ops, g_up, l2norm):
    """A few tokens' channels grow: the scales follow the operands, not the largest step."""
    def grow(g):
        g = g.clone()
        g[:, 3::40, :, ::7] = g_up
        return g

    case = _case(g=grow)
    out, pool, ref, ref_pool = _run(gpu_ops, case, l2norm)
    _tiles(out, ref, f"g {g_up}")
    C.assert_rel(pool, ref_pool, C.STATE_TOL, "pool")
