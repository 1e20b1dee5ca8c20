"""GPU parity of the correction inside the GEMM on the tiled weights (the steps over the rank behind the K loop): ranks around its 128-column
steps and 64-column blocks, K groups of unequal depth, slices of K, ragged rows, and rows that are not finite beside rows that are."""
import pytest
import torch

from glowq_amd.kernels import PreparedGroup
from glowq_amd.linear import CudaW4A16Linear
from helpers import tuning

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


# ---- launches that compute r = x R^T themselves (workgroups in front of the grid, words in the workspace) ----------------------------
@pytest.fixture
def wherever_they_can(ext):
    with tuning(ext, proj_any_cost=1):
        yield


def computed_r(ext, run):
    """Whether `run` raised a word of its own at the head of the workspace: a tag of 48 bits, its top bit set (sums left there by other
    launches have sixteen more bits)."""
    dev = torch.device("cuda", torch.cuda.current_device())
    ext._workspace(dev, 65)
    head = ext._workspaces[(dev.index, ext._stream(dev), False)][:8]
    head.zero_()
    run()
    torch.cuda.synchronize()
    return int(head.view(torch.int64).item()) >> 47 == 1


# 32 x 32 tiles of r with K in one slice and in many, 64 x 64 tiles (more than 256 small ones), both on four and on eight waves, fronts filled
# up to one workgroup a compute unit, ragged rows and ranks, ranks of several steps, launches of one and of several rounds, tails and slices
FRONT_CASES = [(65, 256, [130], 8), (65, 768, [200], 40), (100, 3328, [4096, 300], 136), (333, 3584, [3584, 512, 500], 128), (130, 14336, [1000], 64),
               (333, 14336, [4096], 120), (1500, 2304, [2050], 256), (300, 1024, [20000], 392), (1500, 5120, [5120], 264), (1030, 17408, [5120], 200)]


@pytest.mark.parametrize("M,K,Ns,rank", FRONT_CASES)
def test_launch_computes_r_itself(ext, wherever_they_can, M, K, Ns, rank):
    print(f"case M={M} K={K} Ns={Ns} rank={rank}", flush=True)
    x, R, members, weights = make(M + rank, M, K, Ns, rank)
    if len(Ns) > 1:
        members[1]["L"] = None if M % 2 else members[1]["L"]  # (a member without correction)
    pg = PreparedGroup(ext, members, K, 128, 0.75, R=R)
    pg.run(x)  # (makes the copies)
    want_r = x.double() @ R.double().t()
    for _ in range(2):
        got = []
        assert computed_r(ext, lambda: got.extend(pg.run(x)))
        r = pg.last_r
        # one rounding to fp16 (2^-11), fp32 sums of K terms around K^-1/2
        assert ((r.double() - want_r).abs() <= 2.0 ** -11 * want_r.abs() + 1e-4).all()
        for y, w, m in zip(got, weights, members):
            if m["L"] is None:
                want = x.double() @ w.double().t()
                assert ((y.double() - want).abs() <= 2.0 ** -11 * want.abs() + 2e-4).all()
            else:
                check([y], x, r, [w], [m], 0.75, f"M={M} K={K} rank={rank}")
    with tuning(ext, proj_in_launch=0):
        apart = []
        assert not computed_r(ext, lambda: apart.extend(pg.run(x)))
    for a, b in zip(got, apart):
        assert ((a.double() - b.double()).abs() <= 2.0 ** -10 * b.double().abs() + 4e-4).all()


@pytest.mark.parametrize("M,K,Ns,rank", [(65, 768, [200], 40), (333, 3584, [3584, 512, 500], 128), (130, 14336, [1000], 64)])
def test_readers_that_never_hear_from_the_front(ext, wherever_they_can, M, K, Ns, rank):
    """Words that never go up: the first slice of a tile walks all of K, and every reader computes its r."""
    x, R, members, weights = make(M + rank, M, K, Ns, rank)
    pg = PreparedGroup(ext, members, K, 128, 1.0, R=R)
    with tuning(ext, proj_in_launch=2, proj_spin_limit=3):
        y = pg.run(x)
        torch.cuda.synchronize()
    want_r = x.double() @ R.double().t()
    assert ((pg.last_r.double() - want_r).abs() <= 2.0 ** -11 * want_r.abs() + 1e-4).all()
    for got, w, m in zip(y, weights, members):
        want = x.double() @ w.double().t() + want_r @ m["L"].double().t()
        # r of a reader and r_out may round apart: half an ulp of r (2^-11 of a few units) through 8 to 128 entries of L (0.05)
        assert ((got.double() - want).abs() <= 2.0 ** -11 * want.abs() + 2e-3).all()


def test_replays_and_launches_see_their_own_r(ext, wherever_they_can):
    """Eager launches and replays in turn through the same words, new activations each time, another group with other tiles between."""
    M, K, Ns, rank = 100, 3328, [4096, 300], 136
    x, R, members, weights = make(3, M, K, Ns, rank)
    x2, R2, members2, weights2 = make(4, 333, 2304, [2050], 64)
    pg, pg2 = PreparedGroup(ext, members, K, 128, 1.0, R=R), PreparedGroup(ext, members2, 2304, 128, 1.0, R=R2)
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        pg.run(x), pg2.run(x2)
        side.synchronize()
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph, stream=side):
            y = pg.run(x)
            r = pg.last_r
        g = torch.Generator(device="cuda").manual_seed(9)
        for it in range(6):
            x.copy_(torch.randn(M, K, device="cuda", generator=g))
            graph.replay()
            side.synchronize()
            check(y, x, r, weights, members, 1.0, f"replay {it}")
            want_r = x.double() @ R.double().t()
            assert ((r.double() - want_r).abs() <= 2.0 ** -11 * want_r.abs() + 1e-4).all(), it
            x2.copy_(torch.randn(333, 2304, device="cuda", generator=g))
            y2 = pg2.run(x2)
            check(y2, x2, pg2.last_r, weights2, members2, 1.0, f"eager {it}")
    torch.cuda.current_stream().wait_stream(side)


def test_calls_without_room_for_the_words_keep_the_projection_launch(ext, wherever_they_can):
    M, K, Ns, rank = 100, 3328, [4096, 300], 136
    x, R, members, weights = make(5, M, K, Ns, rank)
    pg = PreparedGroup(ext, members, K, 128, 1.0, R=R)
    saved = ext.WORKSPACE_BYTES
    try:
        for nbytes in (16, 4096, 1 << 20):
            ext.WORKSPACE_BYTES = nbytes
            ext._workspaces.clear()
            y = pg.run(x)
            check(y, x, pg.last_r, weights, members, 1.0, f"workspace {nbytes}")
    finally:
        ext.WORKSPACE_BYTES = saved
        ext._workspaces.clear()


# ---- up to 64 rows: the unrounded form ---------------------------------------------------------------------------------------
@pytest.mark.parametrize("in_front", [False, True])
@pytest.mark.parametrize("M,K,Ns,rank,gs", [(33, 256, [32], 8, 128), (64, 512, [130, 40], 40, 256), (57, 5120, [5120, 1024, 1024], 256, 128), (40, 17408, [5120], 264, 128),
                                            (64, 1280, [34816], 64, 512), (17, 2048, [16600, 9000], 72, 128), (32, 2304, [30000], 128, 128), (49, 3328, [300], 136, 128)])
def test_unrounded_form(ext, M, K, Ns, rank, gs, in_front):
    """Weights that are never rounded, to the accuracy of the outputs' rounding: with activations in the hundreds of which rounded weights
    would be off by more."""
    print(f"case M={M} K={K} Ns={Ns} rank={rank} gs={gs} {in_front}", flush=True)
    g = torch.Generator(device="cuda").manual_seed(M + K)
    x = (torch.randn(M, K, device="cuda", generator=g) * 64).half()
    R = (torch.randn(rank, K, device="cuda", generator=g) * K ** -0.5).half()
    members, exact = [], []
    for N in Ns:
        codes = torch.randint(0, 16, (N, K), device="cuda", generator=g)
        zeros = torch.randint(0, 16, (N, (K + gs - 1) // gs), device="cuda", generator=g)
        scales = (torch.rand(N, zeros.size(1), device="cuda", generator=g) * 0.01 + 0.001).half()
        qw = sum(codes.view(N, K // 8, 8)[:, :, i] << (4 * i) for i in range(8))
        zp = torch.nn.functional.pad(zeros, (0, -zeros.size(1) % 8))
        qz = sum(zp.view(N, -1, 8)[:, :, i] << (4 * i) for i in range(8))
        members.append({"qweight": qw.to(torch.int32), "qzeros": qz.to(torch.int32), "scales": scales, "bias": None,
                        "L": (torch.randn(N, rank, device="cuda", generator=g) * 0.05).half()})
        exact.append((codes - zeros.repeat_interleave(gs, 1)[:, :K]).double() * scales.repeat_interleave(gs, 1)[:, :K].double())
    pg = PreparedGroup(ext, members, K, gs, 1.0, R=R)
    with tuning(ext, tiled_shape_rule=0, proj_any_cost=1, proj_in_launch=1 if in_front else 0):
        for _ in range(2):
            y = pg.run(x)
            assert ext.last_launch()["kernel"].startswith("gemm_tiled_kernel") and "exact" in ext.last_launch()["kernel"]
            r = pg.last_r
            want_r = x.double() @ R.double().t()
            assert ((r.double() - want_r).abs() <= 2.0 ** -11 * want_r.abs() + 6e-3).all()
            for got, w, m in zip(y, exact, members):
                want = x.double() @ w.t() + r.double() @ m["L"].double().t()
                # outputs in the hundreds: their own rounding, and fp32 sums of terms up to 64 x 4 x 0.15
                assert ((got.double() - want).abs() <= 2.0 ** -11 * want.abs() + 2e-2).all()
                assert (got.double() - want).norm() <= 3.2e-4 * want.norm()
