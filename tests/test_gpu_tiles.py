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

from _fixtures import dequant, fp64_ref, rand_acts, rel_err
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


@pytest.mark.parametrize("fmt", ["nf4", "mxfp4"])
@pytest.mark.parametrize("kind,bm,K", [("fwd", 256, 320), ("dgrad", 256, 576), ("dgrad", 128, 1024)])
@pytest.mark.parametrize("empty", ["some", "first_and_last", "all"])
def test_empty_tiles_in_a_device_table(fmt, kind, bm, K, empty):
    """A table of fixed capacity has entries of no rows, anywhere: nothing is
    computed for them, and every other tile is written with the bits of the
    table without them. 384 entries, several per workgroup; on 256 CUs the
    dgrad calls reach both the 256-row and the 512-column kernel (K = 1024: 3
    rounds of tiles against 6)."""
    import _hiplib
    n, N = 384, 128
    g = torch.Generator().manual_seed(bm + K)
    rows = torch.randint(1, min(bm, 160) + 1, (n,), generator=g)
    if empty == "some":
        rows[torch.rand(n, generator=g) < 0.4] = 0
    elif empty == "first_and_last":
        rows[:40] = 0
        rows[-40:] = 0
    else:
        rows[:] = 0
    W, S = _stack(fmt, 4, N, K, seed=7)
    T = max(int(rows.sum()), 1)
    x = rand_acts(T, K if kind == "fwd" else N, seed=8)
    width = N if kind == "fwd" else K
    row0 = torch.cumsum(rows, 0) - rows
    call = getattr(_hiplib.load(), "gnf4_hip_grouped_" + kind)

    def run(keep):
        dev = lambda v: v.to(torch.int32).cuda()  # noqa: E731
        eids, t0, tr = dev(torch.arange(n) % 4), dev(row0[keep]), dev(rows[keep])
        tg = dev(torch.arange(n)[keep])
        out = torch.full((T, width), 7.0, dtype=torch.bfloat16, device="cuda")
        head = (0 if fmt == "nf4" else 1, x.data_ptr(), _hiplib.DTYPE_BF16, x.stride(0),
                W.data_ptr(), W.stride(0), W.stride(1), S.data_ptr(), S.stride(0), S.stride(1),
                eids.data_ptr())
        mid = (None, n) if kind == "fwd" else ()
        _hiplib.check(call(*head, *mid, t0.data_ptr(), tr.data_ptr(), tg.data_ptr(), t0.numel(),
                           bm, N, K, out.data_ptr(), out.stride(0),
                           torch.cuda.current_stream().cuda_stream), kind)
        return out

    got = run(torch.ones(n, dtype=torch.bool))
    if empty == "all":
        assert bool((got == 7).all())
        return
    assert torch.equal(got, run(rows > 0))
    w = [dequant(fmt, W[e], S[e]).double() for e in range(4)]
    ref = torch.cat([x[r0:r0 + m].double() @ (w[i % 4].t() if kind == "fwd" else w[i % 4])
                     for i, (r0, m) in enumerate(zip(row0.tolist(), rows.tolist())) if m])
    assert rel_err(got, ref) <= 1e-2


def _spread(t, stride):
    """``t [T, C]`` in rows ``stride`` elements apart."""
    T, C = t.shape
    buf = torch.empty((T - 1) * stride + C, dtype=t.dtype, device="cuda")
    return buf.as_strided((T, C), (stride, 1)).copy_(t)


@pytest.mark.parametrize("fmt", ["nf4", "mxfp4"])
@pytest.mark.parametrize("kind", ["fwd", "dgrad"])
@pytest.mark.parametrize("which", ["rows", "weights"])
def test_strides_past_the_tile_kernels_offsets(fmt, kind, which):
    """Rows so far apart that 256 of them (of an expert's packed rows, in the
    dgrad) span 2 GiB: the tile kernels' 32-bit offsets do not reach them and
    the general kernels run. Host and device ids."""
    from test_gpu_dgrad import _ops as dgrad_ops
    N, K, sizes, ids = 64, 128, [20, 3, 17], [0, 1, 0]
    W, S = _stack(fmt, 2, N, K, seed=3)
    x = rand_acts(sum(sizes), K if kind == "fwd" else N, seed=4)
    op = (_ops() if kind == "fwd" else dgrad_ops())[fmt]
    want = op(x, W, S, sizes, ids)
    xs, Ws = x, W
    if which == "rows":
        xs = _spread(x, 1 << 22)
    else:
        # one row of both experts in turn, 2^31 / 256 (forward) or / 64 apart
        step = 1 << (23 if kind == "fwd" else 25)
        buf = torch.empty((N - 1) * step + 2 * K, dtype=torch.uint8, device="cuda")
        Ws = buf.as_strided(W.shape, (K, step, 1)).copy_(W)
    for arg in (ids, torch.tensor(ids, device="cuda")):
        got = op(xs, Ws, S, sizes, arg)
        assert rel_err(got, want.double()) <= 1e-3   # another order of fp32 sums


@pytest.mark.parametrize("fmt", [0, 1])
@pytest.mark.parametrize("K", [256, 1024])
def test_planned_launch_into_an_output_off_the_tile_kernels_alignment(fmt, K):
    """A plan's launch may write into columns of a wider buffer: an odd row
    stride or offset, which the tile kernel's 8-byte stores do not take, runs
    the general kernel, with and without tables built for the shape."""
    import nf4_grouped
    name, N, sizes, ids = ("nf4", "mxfp4")[fmt], 72, [40, 128, 5], [2, 0, 1]
    W, S = _stack(name, 3, N, K, seed=5)
    a = rand_acts(sum(sizes), K, seed=6)
    want = _ops()[name](a, W, S, sizes, ids)
    for shape in (None, (N, K)):
        plan = nf4_grouped.GroupPlan(sizes, ids, "cuda", shape=shape)
        for off, width in ((1, N + 3), (2, N + 4), (0, N + 2)):
            buf = torch.full((sum(sizes), width), 7.0, dtype=torch.bfloat16, device="cuda")
            out = buf[:, off:off + N]
            nf4_grouped.launch_planned(fmt, a, W, S, plan, out=out)
            assert rel_err(out, want.double()) <= 1e-3
            out.fill_(7)
            assert bool((buf == 7).all())
        assert torch.equal(nf4_grouped.launch_planned(fmt, a, W, S, plan), want)
