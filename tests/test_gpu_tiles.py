"""The tile kernel (k_tile_fwd) at the sizes where it can go wrong: every count
of 32-row subtiles, step counts around its register and LDS rings (K / 64 from
1), output widths that end inside a tile, a store chunk or a wave, tiles that
follow one another in a workgroup with the rings running on or starting anew.

Against float64 of the decoded weights: a bf16 weight and a bf16 output round
by 2^-9 each at most, so 1e-2 relative Frobenius error is above what any
correct tile shows (about 2.3e-3), and far below one wrong 64-wide step. Rows
are computed alone, so the same rows in tiles of another height (block_m) must
come out bit for bit."""
import pytest
import torch

from _fixtures import fp64_ref, rand_acts, rel_err
from test_gpu_forward import _ops, _stack

pytestmark = pytest.mark.gpu


def _check(fmt, W, S, sizes, ids, K, heights=(64,), seed=5):
    a = rand_acts(sum(sizes), K, seed=seed)
    op = _ops()[fmt]
    out = op(a, W, S, sizes, ids, block_m=256)
    assert rel_err(out, fp64_ref(fmt, a, W, S, sizes, ids)) <= 1e-2
    for bm in heights:
        assert torch.equal(out, op(a, W, S, sizes, ids, block_m=bm))
    assert torch.equal(out, op(a, W, S, sizes, ids, block_m=256))


@pytest.mark.parametrize("fmt", ["nf4", "mxfp4"])
@pytest.mark.parametrize("steps", [1, 2, 3, 4, 5, 7, 8, 9, 11, 12, 16, 17, 24, 31])
def test_step_counts(fmt, steps):
    """Every subtile count at step counts around the rings' lengths."""
    K = 64 * steps
    sizes = [17, 40, 70, 100, 0, 130, 165, 200, 256, 33, 250]
    W, S = _stack(fmt, len(sizes), 260, K, seed=steps)
    _check(fmt, W, S, sizes, list(range(len(sizes)))[::-1], K, heights=(32, 64, 128))


@pytest.mark.parametrize("fmt", ["nf4", "mxfp4"])
@pytest.mark.parametrize("N", [4, 28, 36, 252, 256, 260, 516, 764])
def test_output_widths(fmt, N):
    K = 320
    sizes = [60, 290, 1, 129]
    W, S = _stack(fmt, 4, N, K, seed=N)
    _check(fmt, W, S, sizes, [2, 0, 3, 1], K)


@pytest.mark.parametrize("fmt", ["nf4", "mxfp4"])
@pytest.mark.parametrize("K", [512, 704, 768])
@pytest.mark.parametrize("mix", ["short", "tall", "all"])
def test_many_tiles_per_workgroup(fmt, K, mix):
    """More tiles than CUs: a workgroup's tiles follow one another, of one
    ring class or of several, over step counts that do and do not come out
    even in the weight ring."""
    lo, hi = {"short": (17, 64), "tall": (130, 256), "all": (17, 256)}[mix]
    E = 96
    g = torch.Generator().manual_seed(K)
    sizes = torch.randint(lo, hi + 1, (E,), generator=g).tolist()
    W, S = _stack(fmt, E, 1540, K, seed=K + 1)
    _check(fmt, W, S, sizes, torch.randperm(E, generator=g).tolist(), K, heights=(128,))
