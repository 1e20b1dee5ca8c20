"""GPU parity of the 16 x 16 tiles for up to sixteen token rows, on the tiled copy of the weights and on the canonical buffers: both staged row
counts, ragged row blocks and members, K groups and slices of unequal depth, ranks around the blocks and past a pass, r inside the launch
and ahead of it, strided buffers, rows that are not finite, and replays of a graph."""
import pytest
import torch

from glowq_amd.kernels import PreparedGroup
from helpers import tuning

pytestmark = pytest.mark.gpu


def make(seed, M, K, Ns, rank, gs=128):
    """Activations in the hundreds (rounded weights would be off by more than the outputs are), weights as stored and in fp64."""
    g = torch.Generator(device="cuda").manual_seed(seed)
    x = (torch.randn(M, K, device="cuda", generator=g) * 64).half()
    R = (torch.randn(rank, K, device="cuda", generator=g) * K ** -0.5).half() if rank else None
    members, exact = [], []
    for N in Ns:
        codes = torch.randint(0, 16, (N, K), device="cuda", generator=g)
        zeros = torch.randint(0, 16, (N, K // gs), device="cuda", generator=g)
        scales = (torch.rand(N, K // gs, device="cuda", generator=g) * 0.01 + 0.001).half()
        qw = sum(codes.view(N, K // 8, 8)[:, :, i] << (4 * i) for i in range(8))
        zp = torch.nn.functional.pad(zeros, (0, -zeros.size(1) % 8))
        qz = sum(zp.view(N, -1, 8)[:, :, i] << (4 * i) for i in range(8))
        members.append({"qweight": qw.to(torch.int32), "qzeros": qz.to(torch.int32), "scales": scales, "bias": None,
                        "L": (torch.randn(N, rank, device="cuda", generator=g) * 0.05).half() if rank else None})
        exact.append((codes - zeros.repeat_interleave(gs, 1)).double() * scales.repeat_interleave(gs, 1).double())
    return x, R, members, exact


def check(y, x, r, exact, members, rows=slice(None)):
    for got, w, m in zip(y, exact, members):
        want = x.double() @ w.t()
        if m["L"] is not None:
            want = want + r.double() @ m["L"].double().t()
        got, want = got.double()[rows], want[rows]
        # outputs in the hundreds: their own rounding, and fp32 sums of terms up to 64 x 4 x 0.15
        assert ((got - want).abs() <= 2.0 ** -11 * want.abs() + 2e-2).all()
        assert (got - want).norm() <= 3.2e-4 * want.norm()


@pytest.fixture(params=["tiled", "words"])
def form(request, ext):
    limits = {"tiled_shape_rule": 0} if request.param == "tiled" else {"tiled_max_m": 0}
    with tuning(ext, **limits):
        yield request.param


def launched(ext, form):
    return ext.last_launch()["kernel"].startswith(f"skinny_{form}_kernel")


SHAPES = [(256, [4000], 8), (512, [130, 2040], 40), (1024, [4100, 3000], 40), (1280, [2600, 33], 72), (2304, [2336], 256), (5120, [5120, 1024, 1024], 256),
          (17408, [5120], 264), (768, [34000], 136), (4096, [28672], 64), (1024, [1], 0), (3328, [40, 7], 0), (14336, [4096], 0), (2816, [9472, 9472], 0)]
# K of those with a correction that have r inside their launch, where the call allows it, on the tiled copy and on the canonical buffers (the canonical
# form leaves all other corrected ones, and those with K below 1024, to the skinny kernel)
INSIDE = {"tiled": {768, 1024, 1280, 2304, 4096, 5120}, "words": {1024, 1280, 2304, 4096}}


@pytest.mark.parametrize("K,Ns,rank", SHAPES)
@pytest.mark.parametrize("M", [5, 8, 9, 16])
def test_against_fp64(ext, form, M, K, Ns, rank):
    print(f"case M={M} K={K} Ns={Ns} rank={rank} {form}", flush=True)
    x, R, members, exact = make(M + K, M, K, Ns, rank)
    pg = PreparedGroup(ext, members, K, 128, 1.0 if rank else 0.0, R=R)
    for in_front in (0, 1):
        with tuning(ext, proj_in_launch=in_front):
            y = pg.run(x)
        if form == "words" and rank and K not in INSIDE[form]:
            assert ext.last_launch()["kernel"].startswith(("skinny_codes_mfma", "skinny_mfma", "skinny_group_kernel<"))
            continue  # a group that the skinny kernel keeps
        assert launched(ext, form), ext.last_launch()
        inside = ext.last_launch()["kernel"].split(">")[0].count(",") == 3  # rows, K groups, producer waves and, with r inside, a 1
        assert inside == bool(in_front and rank and K in INSIDE[form]), ext.last_launch()
        r = pg.last_r
        if rank:
            want_r = x.double() @ R.double().t()
            assert ((r.double() - want_r).abs() <= 2.0 ** -11 * want_r.abs() + 6e-3).all()
        check(y, x, r, exact, members)


@pytest.mark.parametrize("bad", [float("inf"), float("nan")])
@pytest.mark.parametrize("K,Ns,rank", [(2304, [2336], 40), (14336, [4096], 0), (2816, [9472, 9472], 256)])
def test_rows_that_are_not_finite_stay_by_themselves(ext, form, K, Ns, rank, bad):
    M = 13
    x, R, members, exact = make(K, M, K, Ns, rank)
    x[[1, 11]] = bad
    fine = [m for m in range(M) if m not in (1, 11)]
    pg = PreparedGroup(ext, members, K, 128, 1.0 if rank else 0.0, R=R)
    y = pg.run(x)
    assert launched(ext, form)
    for out in y:
        assert not torch.isfinite(out[[1, 11]]).any()
        assert torch.isfinite(out[fine]).all()
    xs, r = x[fine], pg.last_r[fine] if rank else None
    check([o[fine] for o in y], xs, r, exact, members)


@pytest.mark.parametrize("at_end", [False, True])
@pytest.mark.parametrize("M", [5, 11])
def test_strided_buffers_and_bias(ext, M, at_end):
    """Members inside wider buffers (row strides above the shape's) on the canonical form, with a bias: the first columns of a buffer, and the
    last ones, so that nothing lies behind the last row."""
    K, N = 1280, 2600
    x, _, (m,), exact = make(3, M, K, [N], 0)
    wide = {}
    for k, pad in (("qweight", 4), ("scales", 2), ("qzeros", 1)):
        whole = torch.full((N, m[k].size(1) + pad), 7, dtype=m[k].dtype, device="cuda")
        wide[k] = whole[:, pad:] if at_end else whole[:, :m[k].size(1)]
        wide[k].copy_(m[k])
    bias = (torch.randn(N, device="cuda") * 100).half()
    with tuning(ext, tiled_max_m=0):
        pg = PreparedGroup(ext, [{**m, "bias": bias}], K, 128, 0.0)
        e = pg.arr[0]
        for k, (ptr, ld) in {"qweight": ("qweight", "ldw_i32"), "scales": ("scales", "lds"), "qzeros": ("qzeros", "ldz_i32")}.items():
            setattr(e, ptr, wide[k].data_ptr())
            setattr(e, ld, wide[k].stride(0))
        (y,) = pg.run(x)
        assert launched(ext, "words")
    want = x.double() @ exact[0].t() + bias.double()
    assert ((y.double() - want).abs() <= 2.0 ** -11 * want.abs() + 2e-2).all()


def test_replays_follow_rows_and_weights(ext):
    """A recorded call on the canonical buffers: replays with new activations and after writes to the weights."""
    M, K, Ns, rank = 12, 2048, [2048, 2048, 2048], 64
    x, R, members, exact = make(5, M, K, Ns, rank)
    pg = PreparedGroup(ext, members, K, 128, 1.0, R=R)
    pg.run(x)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        y = pg.run(x)
        r = pg.last_r
    assert launched(ext, "words")
    for seed in (6, 7, 8):
        x2, R2, members2, exact2 = make(seed, M, K, Ns, rank)
        x.copy_(x2), R.copy_(R2)
        for a, b in zip(members, members2):
            for k in ("qweight", "qzeros", "scales", "L"):
                a[k].copy_(b[k])
        graph.replay()
        torch.cuda.synchronize()
        check(y, x, r, exact2, members)


@pytest.mark.parametrize("K,Ns,given,workspace,words", [
    (4096, [2048, 512], False, False, True), (4096, [2048, 512], True, True, False), (1024, [2048, 512], True, False, True),
    (4096, [8000, 400], True, False, True), (14336, [4096], False, False, False), (14336, [4096], False, True, True), (14336, [4096], True, True, True),
    (8192, [2048], True, False, False), (8192, [2048], True, True, True)])
@pytest.mark.parametrize("M", [5, 16])
def test_short_groups_with_r_given_and_long_k_without_slices(ext, M, K, Ns, given, workspace, words):
    """Which calls without an r to compute take the canonical form; the others stay on the skinny kernel, and both are right."""
    rank = 40 if given else 0
    words = words and not (given and M <= 8 and K >= 12288)  # (the skinny kernel cuts that K itself)
    x, R, members, exact = make(M + K, M, K, Ns, rank)
    r = (torch.randn(M, rank, device="cuda") * 64).half() if given else None
    pg = PreparedGroup(ext, members, K, 128, 1.0 if given else 0.0)
    outs = [torch.empty(M, N, dtype=torch.float16, device="cuda") for N in Ns]
    for e, y in zip(pg.arr, outs):
        e.y, e.ldy = y.data_ptr(), y.stride(0)
    ws = torch.empty((8 << 20) if workspace else 16, dtype=torch.uint8, device="cuda")
    with tuning(ext, tiled_max_m=0):
        assert ext.lib.glowq_w4a16_group_forward_ws(x.data_ptr(), r.data_ptr() if given else None, pg.arr, len(Ns), M, K, 128, rank, 1.0,
                                                    ws.data_ptr(), ws.numel() if workspace else 0, torch.cuda.current_stream().cuda_stream) == 0
    assert launched(ext, "words") == words, ext.last_launch()
    if words or M <= 8:
        check(outs, x, r, exact, members)
    else:  # rounded weights
        check(outs, x, r, [w.half().double() for w in exact], members)


@pytest.mark.parametrize("limit", ["words_max_m", "skinny_codes_max_m"])
def test_switched_off_the_weights_are_rounded(ext, limit):
    """Without the narrow tiles, or without raw codes at all, sixteen rows take the kernel that rounds the weights: further from fp64 than they are
    with unrounded ones (here 2e-4), as near as half an ulp of a weight allows."""
    M, K, N = 16, 2048, 3000
    x, _, members, (w,) = make(9, M, K, [N], 0)
    pg = PreparedGroup(ext, members, K, 128, 0.0)
    want = x.double() @ w.t()
    with tuning(ext, tiled_max_m=0, **{limit: 0}):
        (y,) = pg.run(x)
        assert ext.last_launch()["kernel"] == "skinny_mfma"
    rounded = x.double() @ w.half().double().t()
    near = (y.double() - rounded).norm() / want.norm()
    assert near <= 3.2e-4 and (y.double() - want).norm() / want.norm() > near


@pytest.mark.parametrize("std", [1e-4, 3e-5])
@pytest.mark.parametrize("K,Ns,rank", [(4096, [300], 0), (2816, [3000, 40], 40)])
@pytest.mark.parametrize("M", [5, 8, 9, 16])
def test_small_activations(ext, form, M, K, Ns, rank, std):
    """Activations far below 2^-10 keep their bits on the canonical buffers from 9 rows on, where the rounding kernel has the other groups.  The tiled
    copy and fewer rows take half of the columns as x / 16, in fp16 multiples of 2^-24: an error of at most 2^-21 in x, evenly spread."""
    x, R, members, exact = make(M + K, M, K, Ns, rank)
    x = (x.float() * (std / 64)).half()
    for m in members:  # outputs of order one
        m["scales"] *= 2048
    exact = [2048 * w for w in exact]
    if rank:
        R *= 2048
    pg = PreparedGroup(ext, members, K, 128, 1.0 if rank else 0.0, R=R)
    y = pg.run(x)
    assert launched(ext, form), ext.last_launch()
    of_x = 2.0 ** -20 / 24 ** 0.5 / std if form == "tiled" or M <= 8 else 0.0
    for got, w, m in zip(y, exact, members):
        want = x.double() @ w.t()
        if m["L"] is not None:
            want = want + pg.last_r.double() @ m["L"].double().t()
        # the output's own rounding: at most 2^-11 of a value and 0.29 / 0.5 of that in the mean.  Both norms of the rest hang on the sums of the
        # K / 128 groups of a row (a weight's mean over its group is as large as its spread): 110 of them in the smallest case, 7 % of
        # deviation each, 10 % of the ratio; four deviations
        assert (got.double() - want).norm() <= (3.2e-4 ** 2 + (1.4 * of_x) ** 2) ** 0.5 * want.norm()


@pytest.mark.parametrize("K,Ns,rank", [(4096, [300], 0), (2816, [3000, 40], 40)])
@pytest.mark.parametrize("M", [9, 16])
def test_an_infinite_activation_keeps_its_sign(ext, M, K, Ns, rank):
    """On the canonical buffers from 9 rows on an infinite activation makes outputs of the sign of its weight, and no number where that is zero."""
    x, R, members, exact = make(M + K, M, K, Ns, rank)
    x[1, 5], x[M - 1, K - 3] = float("inf"), float("-inf")
    with tuning(ext, tiled_max_m=0):
        for m in members:
            m["L"] = None  # (r of these rows is infinite or no number, whatever the weights are)
        pg = PreparedGroup(ext, members, K, 128, 0.0)
        y = pg.run(x)
        assert launched(ext, "words"), ext.last_launch()
    for got, w in zip(y, exact):
        want = torch.where(torch.isfinite(x), x, 0).double() @ w.t()
        for row, col in ((1, 5), (M - 1, K - 3)):
            want[row] = x[row, col].double() * w[:, col]
        finite = torch.isfinite(want)
        assert torch.equal(got.double()[~finite].nan_to_num(nan=1.0), want[~finite].nan_to_num(nan=1.0))
        assert ((got.double() - want)[finite].abs() <= 2.0 ** -11 * want[finite].abs() + 2e-2).all()
