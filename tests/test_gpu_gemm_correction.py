"""GPU parity of the correction inside the GEMM on the tiled weights (the steps over the rank behind the K loop): ranks around its 128-column
steps and 64-column blocks, K groups of unequal depth, slices of K, ragged rows, and rows that are not finite beside rows that are."""
import pytest
import torch

from glowq_amd.kernels import PreparedGroup
from glowq_amd.linear import CudaW4A16Linear

pytestmark = pytest.mark.gpu


def make(seed, M, K, Ns, rank):
    g = torch.Generator(device="cuda").manual_seed(seed)
    x = torch.randn(M, K, device="cuda", generator=g).half()
    R = (torch.randn(rank, K, device="cuda", generator=g) * K ** -0.5).half()
    members, weights = [], []
    for N in Ns:
        lin = torch.nn.Linear(K, N, bias=False, device="cuda", dtype=torch.float16)
        with torch.no_grad():
            lin.weight.normal_(0.0, 0.02, generator=g)
        mod = CudaW4A16Linear.from_float(lin, 128)
        weights.append(mod.dequantize())
        members.append({"qweight": mod.qweight_i32, "scales": mod.scales_f16, "qzeros": mod.qzeros_i32, "bias": None,
                        "L": (torch.randn(N, rank, device="cuda", generator=g) * 0.05).half()})
    return x, R, members, weights


def check(y, x, r, weights, members, alpha, what):
    for got, w, m in zip(y, weights, members):
        want = x.double() @ w.double().t() + alpha * (r.double() @ m["L"].double().t())
        # |deq(W)| < 0.1, |r| and |x| around 1: the fp16 rounding of the output (2^-11) and, far below it, fp32 sums
        assert ((got.double() - want).abs() <= 2.0 ** -11 * want.abs() + 2e-4).all(), what


# (row tiles, column tiles, K groups) by the sizes: one row block and several, K of an odd number of 256-column blocks (the second
# K group has fewer), K in slices (the last one carries the correction)
@pytest.mark.parametrize("M,K,Ns", [(65, 768, [200]), (100, 3328, [4096, 300]), (333, 3584, [3584, 512, 500]), (130, 14336, [1000]), (2000, 2304, [2050])])
@pytest.mark.parametrize("rank", [8, 64, 120, 136, 256, 264, 392])
def test_ranks_around_the_steps(ext, M, K, Ns, rank):
    x, R, members, weights = make(M + rank, M, K, Ns, rank)
    for alpha in (1.0, -0.375):
        pg = PreparedGroup(ext, members, K, 128, alpha, R=R)
        y = pg.run(x)
        r = pg.last_r
        assert ((r.double() - x.double() @ R.double().t()).abs() <= 2.0 ** -11 * r.double().abs() + 1e-4).all()
        check(y, x, r, weights, members, alpha, f"M={M} K={K} rank={rank} alpha={alpha}")


@pytest.mark.parametrize("bad", [float("inf"), float("nan")])
@pytest.mark.parametrize("M,K,Ns,rank", [(100, 3328, [4096, 300], 72), (333, 3584, [3584, 512, 500], 128), (129, 14336, [1000], 40)])
def test_rows_that_are_not_finite_stay_by_themselves(ext, M, K, Ns, rank, bad):
    """Neither a row of activations nor its r reaches another row through what a tile reads past its end."""
    x, R, members, weights = make(M, M, K, Ns, rank)
    rows = torch.tensor([1, 32, M - 2], device="cuda")
    x[rows] = bad
    fine = torch.ones(M, dtype=torch.bool, device="cuda")
    fine[rows] = False
    pg = PreparedGroup(ext, members, K, 128, 1.0, R=R)
    y = pg.run(x)
    check([v[fine] for v in y], x[fine], pg.last_r[fine], weights, members, 1.0, f"M={M} K={K}")
    assert not any(torch.isfinite(v[rows]).any() for v in y)
