"""The fp32 precision mode (DAV2_CREATE_FORCE_FP32): the fp32 MFMA GEMM and
im2col kernels against float64 products and torch's unfold, the fp32
operators (src/operators.cpp:882-955, :1211-1452, :1528-1676, :1807-1861)
against the oracle, and whole models against the oracle's fp32 graph.

fp32 sums in a different order than the oracle's: the gate is the depth
tolerance, max|gpu - cpu| <= 1e-3 of the depth range; the operators are held
to 1e-5 of their output's magnitude."""

import ctypes as C

import numpy as np
import pytest
import torch.nn.functional as F

from gpu_util import db, dev, empty, host, ok, ptr, stream

pytestmark = pytest.mark.gpu

SEED = 0xDA20000
ENC = {"vits": 0, "vitb": 1, "vitl": 2}
EPI = {"row": 1, "gelu": 2, "layerscale": 3, "transposed": 4, "convt": 5}


def _announce(*args):
    print("case:", *args, flush=True)


def _rel(got, want):
    return float(np.abs(got.astype(np.float64) - want).max() / max(np.abs(want).max(), 1e-30))


@pytest.fixture(scope="module")
def ops(gpu, lib):
    h = lib.dav2_ops_create(0)
    assert h, lib.dav2_ops_last_error()
    yield h
    lib.dav2_ops_destroy(h)


def _resident(torch, *arrays):
    """Device copies, complete before the operator set's own stream reads them
    (the copies run on torch's stream) and held until the caller drops them."""
    out = [dev(torch, a) for a in arrays]
    torch.cuda.synchronize()
    return out


def run(lib, rc):
    assert rc == 0, f"status {rc}: {lib.dav2_ops_last_error().decode()}"


@pytest.mark.parametrize("m,n,k", [(37, 80, 96), (1370, 1024, 1024), (200, 33, 588), (1, 5, 4)])
@pytest.mark.parametrize("epi", ["row", "gelu", "layerscale", "transposed"])
def test_gemm_f32_epilogues(gpu, pkg, lib, oracle, m, n, k, epi):
    torch = gpu
    _announce("gemm_f32", m, n, k, epi)
    rng = np.random.default_rng(m * 7 + n + k)
    a = rng.standard_normal((m, k)).astype(np.float32)
    b = (rng.standard_normal((n, k)) * 0.05).astype(np.float32)
    bias = rng.standard_normal(n).astype(np.float32)
    gamma = rng.standard_normal(n).astype(np.float32)
    v = a.astype(np.float64) @ b.astype(np.float64).T + bias
    ad, bd, biasd, gd = dev(torch, a), dev(torch, b), dev(torch, bias), dev(torch, gamma)
    args = pkg.GemmF32Args()
    args.a, args.lda, args.b, args.ldb = ptr(ad), k, ptr(bd), k
    args.m, args.n, args.k, args.epilogue, args.bias = m, n, k, EPI[epi], ptr(biasd)
    if epi == "transposed":
        res = rng.standard_normal((n, m + 3)).astype(np.float32)
        out = dev(torch, res.copy())
        args.out, args.out_row_stride, args.out_row_offset = ptr(out), m + 3, 2
        resd = dev(torch, res)
        args.residual, args.relu_output = ptr(resd), 1
        want = res.astype(np.float64).copy()
        want[:, 2:2 + m] = np.maximum(v.T + res[:, 2:2 + m], 0.0)
    else:
        res = rng.standard_normal((m + 1, n)).astype(np.float32)
        out = dev(torch, res)
        args.out, args.out_row_offset = ptr(out), 1
        want = res.astype(np.float64).copy()
        if epi == "row":
            want[1:] = v
        elif epi == "gelu":
            want[1:] = oracle.gelu(v.astype(np.float32))
        else:
            args.residual, args.gamma = ptr(out), ptr(gd)
            want[1:] = res[1:] + v * gamma
    ok(lib, lib.dav2_hip_gemm_f32(C.byref(args), stream(torch)))
    got = host(torch, out)
    assert _rel(got, want) < 1e-5


@pytest.mark.parametrize("half", [0, 1])
@pytest.mark.parametrize("m,n,k", [(33, 65, 36), (31, 32, 4), (1297, 2307, 44), (1373, 772, 100), (2443, 3076, 36)])
def test_gemm_f32_tiles(gpu, pkg, lib, m, n, k, half):
    """Every tile of both operand forms, ragged in rows, columns and K: within
    the fp32 sum bound of k terms, binary16 subnormals and overflow included."""
    torch = gpu
    _announce("gemm_f32 tiles", m, n, k, half)
    g = torch.Generator().manual_seed(m + n + k)
    a, b = torch.randn((m, k), generator=g), torch.randn((n, k), generator=g)
    a[::7] *= 2.0 ** -20  # binary16 subnormals
    a[5, 3] = 1.0e5  # past binary16: infinite there, a finite product in fp32
    ad, bd = a.cuda(), b.cuda()
    out = torch.full((m, n), float("nan"), device="cuda")
    args = pkg.GemmF32Args()
    args.a, args.lda, args.b, args.ldb = ptr(ad), k, ptr(bd), k
    args.m, args.n, args.k, args.epilogue, args.out, args.half_operands = m, n, k, 1, ptr(out), half
    ok(lib, lib.dav2_hip_gemm_f32(C.byref(args), stream(torch)))
    if half:
        ad, bd = ad.half(), bd.half()
    want = ad.double() @ bd.double().T
    mag = ad.double().abs() @ bd.double().abs().T
    finite = torch.isfinite(want)
    assert bool((finite[5] == (half == 0)).all())
    assert torch.equal(out.double()[~finite], want[~finite])
    # k products (exact for binary16 operands) and k - 1 sums, each within
    # 2^-24 of its magnitude; 2 k covers both
    assert bool(((out.double() - want).abs()[finite] <= 2 * k * 2.0 ** -24 * mag[finite]).all())


@pytest.mark.parametrize("m,n,k", [(2000, 2100, 4), (2017, 2049, 32), (1985, 2177, 68), (2500, 2052, 100)])
def test_gemm_f32_split(gpu, pkg, lib, m, n, k):
    """Grids that take the bfloat16 split (from K = 64 on): magnitudes over 40
    binades within the bound of test_gemm_f32_tiles (the three parts are exact
    and the products left out below 1.001 x 2^-24 of their magnitude),
    infinities and NaN as in fp32."""
    torch = gpu
    _announce("gemm_f32 split", m, n, k)
    g = torch.Generator().manual_seed(m + n + k)
    a, b = torch.randn((m, k), generator=g), torch.randn((n, k), generator=g)
    a[::7] *= 2.0 ** -20
    b[::5] *= 2.0 ** 20
    a[5, 3], a[70, 2], b[9, 3], a[131, 1] = float("inf"), float("nan"), 0.0, -float("inf")
    ad, bd = a.cuda(), b.cuda()
    out = torch.full((m, n), 7.0, device="cuda")
    args = pkg.GemmF32Args()
    args.a, args.lda, args.b, args.ldb = ptr(ad), k, ptr(bd), k
    args.m, args.n, args.k, args.epilogue, args.out = m, n, k, 1, ptr(out)
    ok(lib, lib.dav2_hip_gemm_f32(C.byref(args), stream(torch)))
    want = ad.double() @ bd.double().T
    finite = torch.isfinite(want)
    assert not bool(finite[5].any()) and not bool(finite[70].any()) and int((~finite).sum()) == 3 * n
    assert torch.equal(out[~finite].nan_to_num(1.0, 2.0, 3.0).double(), want[~finite].nan_to_num(1.0, 2.0, 3.0))
    mag = ad.double().abs() @ bd.double().abs().T
    assert bool(((out.double() - want).abs()[finite] <= (2 * k + 3) * 2.0 ** -24 * mag[finite]).all())


@pytest.mark.parametrize("family,k", [("one product", 64), ("one product", 1024), ("normal", 64), ("normal", 1028),
                                      ("positive", 384), ("positive", 4096), ("tiny", 64), ("subnormal", 128)])
def test_gemm_f32_split_precision(gpu, pkg, lib, family, k):
    """The bfloat16 split against float64, in units of 2^-24 of the sum of
    magnitudes: the products left out 1.001, the last addition 1, the small sums
    2^-6, and every MFMA (32 k) up to 2 of the sum it ends with, a truncation.
    Sums of positive products grow in proportion, so theirs average half the last
    one; a sum of one product is exact up to the last addition."""
    torch = gpu
    _announce("gemm_f32 split precision", family, k)
    m, n = 2001, 2100
    g = torch.Generator().manual_seed(k)
    a, b = torch.randn((m, k), generator=g), torch.randn((n, k), generator=g)
    steps = (k + 31) // 32
    bound = 2.02 + 2 * steps
    if family == "one product":  # of mantissas whose left-out parts are largest, cut off or rounded
        one = torch.zeros((m, k))
        worst = torch.tensor([1 + 2.0 ** -7 - 2.0 ** -23, 1 + 2.0 ** -8 - 2.0 ** -17 - 2.0 ** -23])
        row, col = torch.arange(m), torch.arange(n)
        one[row, row % k] = torch.where(row % 3 == 2, a[:, 0], worst[row % 2])
        a, b, bound = one, torch.where(col[:, None] % 3 == 2, b, worst[col % 2][:, None]), 2.02
    elif family == "positive":
        a, b, bound = a.abs(), b.abs(), 4.0 + steps
    elif family in ("tiny", "subnormal"):
        a, b = a * 2.0 ** (-120 if family == "tiny" else -130), b * 2.0 ** 100
    ad, bd = a.cuda(), b.cuda()
    out = torch.full((m, n), float("nan"), device="cuda")
    args = pkg.GemmF32Args()
    args.a, args.lda, args.b, args.ldb = ptr(ad), k, ptr(bd), k
    args.m, args.n, args.k, args.epilogue, args.out = m, n, k, 1, ptr(out)
    ok(lib, lib.dav2_hip_gemm_f32(C.byref(args), stream(torch)))
    want = ad.double() @ bd.double().T
    mag = ad.double().abs() @ bd.double().abs().T
    assert bool(((out.double() - want).abs() <= bound * 2.0 ** -24 * mag).all())


def test_gemm_f32_split_range(gpu, pkg, lib):
    """Operands and sums past the split's range are summed in fp32, and only
    those: the other sums keep their bits."""
    torch = gpu
    m, n, k = 2048, 2112, 96
    g = torch.Generator().manual_seed(3)
    ad, bd = torch.randn((m, k), generator=g).cuda(), torch.randn((n, k), generator=g).cuda()
    args = pkg.GemmF32Args()
    out = torch.full((2, m, n), float("nan"), device="cuda")
    args.lda, args.b, args.ldb = k, ptr(bd), k
    args.m, args.n, args.k, args.epilogue = m, n, k, 1
    large = ad.clone()
    large[::5] *= 2.0 ** 104  # past bfloat16 parts
    large[1::5] *= 2.0 ** 90  # sums past the largest float once scaled
    for i, x in enumerate((ad, large)):
        args.a, args.out = ptr(x), ptr(out[i])
        ok(lib, lib.dav2_hip_gemm_f32(C.byref(args), stream(torch)))
    want = large.double() @ bd.double().T
    mag = large.double().abs() @ bd.double().abs().T
    assert bool(((out[1].double() - want).abs() <= 2 * k * 2.0 ** -24 * mag).all())
    rest = torch.ones(m, dtype=torch.bool, device="cuda")
    rest[::5] = rest[1::5] = False
    assert torch.equal(out[0][rest], out[1][rest])


@pytest.mark.parametrize("w,h,n,k", [(31, 1, 63, 68), (109, 5, 1017, 132), (137, 10, 765, 64), (2081, 1, 2052, 100)])
@pytest.mark.parametrize("epi", ["row", "gelu", "layerscale", "transposed", "convt"])
def test_gemm_f32_split_epilogues(gpu, pkg, lib, oracle, w, h, n, k, epi):
    """Every tile of the split with every epilogue, ragged: LayerScale in place,
    an output offset, and an infinite row whose block is summed again."""
    torch = gpu
    _announce("gemm_f32 split epilogues", w, h, n, k, epi)
    m = w * h
    rng = np.random.default_rng(m + n + k)
    a = rng.standard_normal((m, k)).astype(np.float32)
    b = (rng.standard_normal((n, k)) * 0.05).astype(np.float32)
    bias, gamma = rng.standard_normal(n).astype(np.float32), rng.standard_normal(n).astype(np.float32)
    v = a.astype(np.float64) @ b.astype(np.float64).T
    a[7, 2] = np.inf
    ad, bd, biasd, gd = dev(torch, a), dev(torch, b), dev(torch, bias), dev(torch, gamma)
    args = pkg.GemmF32Args()
    args.a, args.lda, args.b, args.ldb = ptr(ad), k, ptr(bd), k
    args.m, args.n, args.k, args.epilogue, args.bias = m, n, k, EPI[epi], ptr(biasd)
    if epi == "convt":
        c = n // 9
        out = empty(torch, (c, 3 * h, 3 * w), torch.float32)
        args.convt_kernel, args.convt_width, args.convt_height, args.convt_channels = 3, w, h, c
        want = v.reshape(h, w, 3, 3, c).transpose(4, 0, 2, 1, 3).reshape(c, 3 * h, 3 * w) + bias[:c, None, None]
        row7 = np.zeros((h, w), bool)
        row7.reshape(-1)[7] = True
        row7 = np.broadcast_to(np.kron(row7, np.ones((3, 3), bool)), want.shape)
    elif epi == "transposed":
        res = rng.standard_normal((n, m + 5)).astype(np.float32)
        out, resd = dev(torch, res), dev(torch, res)
        args.out, args.out_row_stride, args.out_row_offset, args.residual = ptr(out), m + 5, 3, ptr(resd)
        args.relu_output = 1
        want = res.astype(np.float64)
        want[:, 3:3 + m] = np.maximum(v.T + bias[:, None] + want[:, 3:3 + m], 0.0)
        row7 = np.zeros(want.shape, bool)
        row7[:, 10] = True
    else:
        res = rng.standard_normal((m + 1, n)).astype(np.float32)
        out = dev(torch, res)
        args.out_row_offset = 1
        want = res.astype(np.float64)
        if epi == "layerscale":
            args.residual, args.gamma = ptr(out), ptr(gd)
            want[1:] += (v + bias) * gamma
        else:
            want[1:] = oracle.gelu((v + bias).astype(np.float32)) if epi == "gelu" else v + bias
        row7 = np.zeros(want.shape, bool)
        row7[8] = True
    args.out = ptr(out)
    ok(lib, lib.dav2_hip_gemm_f32(C.byref(args), stream(torch)))
    got = host(torch, out)
    assert _rel(got[~row7], want[~row7]) < 1e-5
    # the infinite row: +-inf by the weight's sign (GELU of -inf is NaN, ReLU of it 0)
    sign = np.sign(b[:, 2])
    if epi == "convt":
        seven = got.reshape(c, h, 3, w, 3)[:, 7 // w, :, 7 % w, :].transpose(1, 2, 0).reshape(-1)
        assert np.array_equal(seven, np.inf * sign)
    elif epi == "transposed":
        assert np.array_equal(got[:, 10], np.where(sign > 0, np.inf, 0.0))
    elif epi == "layerscale":
        assert np.array_equal(got[8], np.inf * sign * np.sign(gamma))
    elif epi == "gelu":
        assert np.all(got[8][sign > 0] == np.inf) and not np.any(np.isposinf(got[8][sign < 0]))
    else:
        assert np.array_equal(got[8], np.inf * sign)


@pytest.mark.parametrize("half", [0, 1])
@pytest.mark.parametrize("n,k", [(384, 384), (772, 1028), (4096, 128), (1155, 44), (768, 64), (31, 60)])
def test_gemm_f32_rows_alone(gpu, pkg, lib, n, k, half):
    """A row's bits do not depend on the rows that come with it, whatever tile
    or arithmetic the sizes choose; an infinite row leaves the others alone."""
    torch = gpu
    _announce("gemm_f32 rows", n, k, half)
    g = torch.Generator().manual_seed(n + k)
    m = 5481
    ad, bd = torch.randn((m, k), generator=g).cuda(), torch.randn((n, k), generator=g).cuda()
    ad[70, 1] = float("inf")
    args = pkg.GemmF32Args()
    args.a, args.lda, args.b, args.ldb = ptr(ad), k, ptr(bd), k
    args.n, args.k, args.epilogue, args.half_operands = n, k, 1, half
    whole = torch.full((m, n), float("nan"), device="cuda")
    args.m, args.out = m, ptr(whole)
    ok(lib, lib.dav2_hip_gemm_f32(C.byref(args), stream(torch)))
    for rows in (1, 33, 70, 253, 545, 1370, 1814, 2740):
        out = torch.full((rows, n), float("nan"), device="cuda")
        args.m, args.out = rows, ptr(out)
        ok(lib, lib.dav2_hip_gemm_f32(C.byref(args), stream(torch)))
        assert torch.equal(out.view(torch.int32), whole[:rows].view(torch.int32)), rows


@pytest.mark.parametrize("k,rows", [(4, 2 ** 29 + 33), (64, 2 ** 27 + 33)])
def test_gemm_f32_many_rows(gpu, pkg, lib, k, rows):
    """More row tiles than grid x holds (k = 4: 2^32 threads of 32-row tiles), small
    whole numbers, exact."""
    torch = gpu
    _announce("gemm_f32 many rows", k, rows)
    small = torch.randint(-8, 9, (rows, 4), dtype=torch.int8, device="cuda")
    ad = torch.zeros((rows, k), device="cuda")
    ad[:, k - 4:] = small
    bd = torch.zeros((1, k), device="cuda")
    bd[0, k - 4:] = torch.tensor([1.0, -2.0, 3.0, 5.0], device="cuda")
    out = torch.full((rows,), 7.5, device="cuda")
    args = pkg.GemmF32Args()
    args.a, args.lda, args.b, args.ldb = ptr(ad), k, ptr(bd), k
    args.m, args.n, args.k, args.epilogue, args.out = rows, 1, k, 1, ptr(out)
    ok(lib, lib.dav2_hip_gemm_f32(C.byref(args), stream(torch)))
    want = small[:, 0].short() - 2 * small[:, 1].short() + 3 * small[:, 2].short() + 5 * small[:, 3].short()
    assert torch.equal(out, want.float())


def test_gemm_f32_rejects(gpu, pkg, lib):
    torch = gpu
    a = empty(torch, (8, 8), torch.float32)
    args = pkg.GemmF32Args()
    args.a, args.lda, args.b, args.ldb, args.m, args.n, args.k = ptr(a), 8, ptr(a), 8, 8, 8, 6  # k % 4
    args.epilogue, args.out = 1, ptr(a)
    assert lib.dav2_hip_gemm_f32(C.byref(args), stream(torch)) != 0
    args.k, args.epilogue = 8, 6  # ROW_COLMAX is int8 only
    assert lib.dav2_hip_gemm_f32(C.byref(args), stream(torch)) != 0


@pytest.mark.parametrize("c,h,w,k,s,p,relu", [(8, 11, 9, 3, 1, 1, False), (16, 13, 10, 3, 2, 1, True),
                                              (3, 28, 42, 14, 14, 0, False), (4, 5, 7, 1, 1, 0, True)])
def test_im2col_f32_matches_unfold(gpu, lib, c, h, w, k, s, p, relu):
    torch = gpu
    _announce("im2col_f32", c, h, w, k, s, p, relu)
    x = np.random.default_rng(c + h).standard_normal((c, h, w)).astype(np.float32)
    ow, oh = (w + 2 * p - k) // s + 1, (h + 2 * p - k) // s + 1
    ld = (c * k * k + 3) // 4 * 4 + 4
    xd = dev(torch, x)
    out = empty(torch, (ow * oh, ld), torch.float32)
    ok(lib, lib.dav2_hip_im2col_f32(ptr(xd), w, h, c, ow, oh, k, s, p, int(relu), ptr(out), ld, stream(torch)))
    src = torch.from_numpy(np.maximum(x, 0) if relu else x)[None]
    want = F.unfold(src, k, padding=p, stride=s)[0].T.numpy()
    got = host(torch, out)
    assert np.array_equal(got[:, : c * k * k], want)
    assert not got[:, c * k * k:].any()


def test_ops_linear(gpu, pkg, lib, oracle, ops):
    torch = gpu
    rng = np.random.default_rng(3)
    rows, ic, oc = 333, 384, 1536
    x = rng.standard_normal((rows, ic)).astype(np.float32)
    w = (rng.standard_normal((oc, ic)) * 0.05).astype(np.float32)
    b = rng.standard_normal(oc).astype(np.float32)
    xd, wd, bd = _resident(torch, x, w, b)
    for gelu in (False, True):
        out = empty(torch, (rows, oc), torch.float32)
        run(lib, lib.dav2_ops_linear(ops, db(pkg, out), db(pkg, xd), db(pkg, wd), db(pkg, bd), rows, ic, oc,
                                     int(gelu)))
        run(lib, lib.dav2_ops_synchronize(ops))
        assert _rel(host(torch, out), oracle.linear_f32(x, w, b, gelu=gelu)) < 1e-5
    bad = empty(torch, (rows, oc - 1), torch.float32)
    assert lib.dav2_ops_linear(ops, db(pkg, bad), db(pkg, xd), db(pkg, wd), db(pkg, bd), rows, ic, oc, 0) == 1


@pytest.mark.parametrize("c,oc,h,w,k,s,p", [(64, 64, 37, 37, 3, 1, 1), (32, 16, 20, 24, 3, 2, 1),
                                            (64, 32, 9, 11, 1, 1, 0)])
def test_ops_conv2d(gpu, pkg, lib, oracle, ops, c, oc, h, w, k, s, p):
    torch = gpu
    _announce("conv2d fp32", c, oc, h, w, k, s, p)
    rng = np.random.default_rng(c + oc + h)
    x = rng.standard_normal((c, h, w)).astype(np.float32)
    wt = (rng.standard_normal((oc, c, k, k)) * 0.05).astype(np.float32)
    b = rng.standard_normal(oc).astype(np.float32)
    ow, oh = (w + 2 * p - k) // s + 1, (h + 2 * p - k) // s + 1
    out = empty(torch, (oc, oh, ow), torch.float32)
    xd, wd, bd = _resident(torch, x, wt, b)
    run(lib, lib.dav2_ops_conv2d(ops, db(pkg, out), db(pkg, xd), db(pkg, wd), db(pkg, bd), w, h, c, oc, k, s, p, 1))
    run(lib, lib.dav2_ops_synchronize(ops))
    assert _rel(host(torch, out), oracle.conv2d_f32(x, wt, b, s, p)) < 1e-5


@pytest.mark.parametrize("c,oc,h,w,k", [(4, 1, 1, 1, 3), (8, 33, 3, 70, 3), (128, 40, 41, 37, 3), (12, 70, 149, 131, 3),
                                        (4, 32, 301, 290, 3), (16, 5, 6, 11, 1), (48, 66, 150, 149, 1)])
@pytest.mark.parametrize("fused", [False, True])
def test_conv2d_f32_implicit(gpu, pkg, lib, c, oc, h, w, k, fused):
    """Every tile, ragged in pixels and channels, one-pixel to 301-row maps: the
    same as float64 within the fp32 sum bound; residual in place, both ReLUs."""
    torch = gpu
    _announce("conv2d fp32 implicit", c, oc, h, w, k, fused)
    g = torch.Generator().manual_seed(c + oc + h)
    x, wt = torch.randn((c, h, w), generator=g).cuda(), torch.randn((oc, c, k, k), generator=g).cuda()
    b, res = torch.randn(oc, generator=g).cuda(), torch.randn((oc, h, w), generator=g).cuda()
    args = pkg.ConvF32Args()
    args.input, args.width, args.height, args.channels, args.kernel = ptr(x), w, h, c, k
    args.weight, args.bias, args.out_channels = ptr(wt), ptr(b), oc
    out = res.clone() if fused else torch.full_like(res, float("nan"))
    args.out, args.residual, args.flags = ptr(out), ptr(out) if fused else None, 3 if fused else 0
    ok(lib, lib.dav2_hip_conv2d_f32(C.byref(args), stream(torch)))
    xin = x.double().relu() if fused else x.double()
    want = F.conv2d(xin[None].cpu(), wt.double().cpu(), b.double().cpu(), padding=k // 2)[0]
    mag = F.conv2d(xin.abs()[None].cpu(), wt.double().abs().cpu(), b.double().abs().cpu(), padding=k // 2)[0]
    if fused:
        want, mag = (want + res.double().cpu()).relu(), mag + res.double().abs().cpu()
    # c k k products and as many sums, bias and residual, each within 2^-24 of its magnitude
    assert bool(((out.double().cpu() - want).abs() <= (2 * c * k * k + 2) * 2.0 ** -24 * mag).all())


@pytest.mark.parametrize("c,h,w", [(384, 7, 9), (400, 7, 9), (400, 32, 32)])
def test_ops_conv2d_routes(gpu, pkg, lib, oracle, ops, c, h, w):
    """Both sides of the line between the implicit GEMM and im2col, 1024 pixels and 384 channels."""
    test_ops_conv2d(gpu, pkg, lib, oracle, ops, c, 40, h, w, 3, 1, 1)


def test_ops_conv2d_in_place(gpu, pkg, lib, ops):
    """The output may be the input's buffer (im2col has read it before the GEMM writes)."""
    torch = gpu
    g = torch.Generator().manual_seed(1)
    x, wt, b = torch.randn((16, 9, 70), generator=g), torch.randn((16, 16, 3, 3), generator=g), torch.randn(16)
    xd, wd, bd = _resident(torch, x.numpy(), wt.numpy(), b.numpy())
    run(lib, lib.dav2_ops_conv2d(ops, db(pkg, xd), db(pkg, xd), db(pkg, wd), db(pkg, bd), 70, 9, 16, 16, 3, 1, 1, 1))
    run(lib, lib.dav2_ops_synchronize(ops))
    want = F.conv2d(x.double()[None], wt.double(), b.double(), padding=1)[0].numpy()
    assert _rel(host(torch, xd), want) < 1e-5


@pytest.mark.parametrize("k", [2, 4])
def test_ops_conv_transpose(gpu, pkg, lib, oracle, ops, k):
    torch = gpu
    rng = np.random.default_rng(k)
    ic, oc, h, w = 32, 24, 7, 9
    x = rng.standard_normal((ic, h, w)).astype(np.float32)
    wt = (rng.standard_normal((ic, oc, k, k)) * 0.1).astype(np.float32)
    b = rng.standard_normal(oc).astype(np.float32)
    rows = wt.transpose(2, 3, 1, 0).reshape(k * k * oc, ic)  # row (ky k + kx) OC + oc, column ic
    out = empty(torch, (oc, h * k, w * k), torch.float32)
    xd, rd, bd = _resident(torch, x, np.ascontiguousarray(rows), b)
    run(lib, lib.dav2_ops_conv_transpose_nonoverlap(ops, db(pkg, out), db(pkg, xd), db(pkg, rd), db(pkg, bd), w, h,
                                                    ic, oc, k))
    run(lib, lib.dav2_ops_synchronize(ops))
    assert _rel(host(torch, out), oracle.conv_transpose_f32(x, wt, b)) < 1e-5


def test_ops_project_tokens(gpu, pkg, lib, oracle, ops):
    torch = gpu
    rng = np.random.default_rng(8)
    pw, ph, d, c = 19, 11, 64, 48
    tokens = rng.standard_normal((pw * ph + 1, d)).astype(np.float32)
    w = rng.standard_normal((c, d)).astype(np.float32)
    b = rng.standard_normal(c).astype(np.float32)
    out = empty(torch, (c, ph, pw), torch.float32)
    td, wd, bd = _resident(torch, tokens, w, b)
    run(lib, lib.dav2_ops_project_tokens(ops, db(pkg, out), db(pkg, td), db(pkg, wd), db(pkg, bd), pw, ph, d, c))
    run(lib, lib.dav2_ops_synchronize(ops))
    assert _rel(host(torch, out), oracle.project_tokens_f32(tokens, w, b, pw, ph)) < 1e-5


def test_ops_prepare_tokens_f32(gpu, pkg, lib, oracle, ops):
    torch = gpu
    rng = np.random.default_rng(9)
    pw, ph, d = 9, 6, 32
    width, height = 14 * pw, 14 * ph
    image = rng.standard_normal((3, height, width)).astype(np.float32)
    w = (rng.standard_normal((d, 3, 14, 14)) * 0.05).astype(np.float32)
    b = rng.standard_normal(d).astype(np.float32)
    cls = rng.standard_normal(d).astype(np.float32)
    pos = rng.standard_normal((1370, d)).astype(np.float32)
    toks = empty(torch, (pw * ph + 1, d), torch.float32)
    imd, wd, bd, cd, pd = _resident(torch, image, w, b, cls, pos)
    run(lib, lib.dav2_ops_prepare_tokens_f32(ops, db(pkg, toks), db(pkg, imd), db(pkg, wd), db(pkg, bd), db(pkg, cd),
                                             db(pkg, pd), width, height, d))
    run(lib, lib.dav2_ops_synchronize(ops))
    want = oracle.prepare_tokens_f32(image, w, b, cls, pos, width, height)
    assert _rel(host(torch, toks), want) < 1e-5


@pytest.fixture(scope="module")
def models(pkg, tmp_path_factory):
    root = tmp_path_factory.mktemp("fp32_models")
    paths = {}
    for enc in ("vits", "vitb"):
        p = root / f"{enc}.dav2"
        pkg.dav2_format.write_synthetic_model(p, enc, seed=SEED + ENC[enc] + 1)
        paths[enc] = p
    return paths


def _span_err(got, ref):
    span = float(ref.max() - ref.min())
    return float(np.abs(got - ref).max()) / (span if span > 0 else 1.0)


@pytest.mark.parametrize("enc,width,height", [("vits", 266, 266), ("vits", 350, 266), ("vitb", 196, 252)])
def test_fp32_mode_depth_parity(gpu, pkg, lib, oracle, models, enc, width, height):
    torch = gpu
    _announce("fp32 model", enc, width, height)
    x = pkg.dav2_format.imagenet_input(width, height, seed=SEED + width + 1)[0]
    with pkg.Context(str(models[enc]), enc, pkg.FORCE_FP32) as ctx:
        depth = ctx.infer(x, width, height)
        xd = dev(torch, x)
        d2 = empty(torch, (height, width), torch.float32)
        logits = empty(torch, (height, width), torch.float32)
        assert lib.dav2_infer_tensor_f32_device_logits(ctx.handle, xd.data_ptr(), width, height, d2.data_ptr(),
                                                       logits.data_ptr(), stream(torch)) == 0
        d2, logits = host(torch, d2), host(torch, logits)
    h = oracle.load_model(models[enc], ENC[enc])
    try:
        ref_depth, ref_logits = oracle.infer_fp32(h, x, width, height)
    finally:
        oracle.free_model(h)
    assert np.isfinite(depth).all() and np.array_equal(depth, d2)
    e_depth, e_logits = _span_err(depth, ref_depth), _span_err(logits, ref_logits)
    print(f"fp32 parity {enc} {width}x{height}: depth {e_depth:.3g}, logits {e_logits:.3g}", flush=True)
    assert e_depth <= 1e-3 and e_logits <= 1e-3


def _live_model(pkg, path, encoder, seed):
    """A model whose blocks reach its output: LayerScale 0.1 and a head whose depth varies."""
    state = pkg.dav2_format.synthetic_state(encoder, seed)
    state = {k: v + 0.1 if k.endswith("gamma") else v for k, v in state.items()}
    state["depth_head.scratch.output_conv2.2.weight"] = state["depth_head.scratch.output_conv2.2.weight"] * 8.0
    state["depth_head.scratch.output_conv2.2.bias"] = state["depth_head.scratch.output_conv2.2.bias"] + 0.25
    pkg.dav2_format.write_model(path, encoder, state)
    return path


@pytest.mark.parametrize("enc,width,height", [("vits", 266, 182), ("vitb", 126, 154), ("vitl", 112, 98)])
def test_fp32_mode_live_blocks_parity(gpu, pkg, lib, oracle, tmp_path, enc, width, height):
    _announce("fp32 model, live blocks", enc, width, height)
    path = _live_model(pkg, tmp_path / "model.dav2", enc, SEED + 9)
    x = pkg.dav2_format.imagenet_input(width, height, seed=SEED + 2)[0]
    with pkg.Context(str(path), enc, pkg.FORCE_FP32) as ctx:
        depth = ctx.infer(x, width, height)
    h = oracle.load_model(path, ENC[enc])
    try:
        ref, _ = oracle.infer_fp32(h, x, width, height)
    finally:
        oracle.free_model(h)
    span, err = float(ref.max() - ref.min()), _span_err(depth, ref)
    print(f"fp32 parity {enc} {width}x{height}: depth {err:.3g} of {span:.3g}", flush=True)
    assert span > 1e-3 and err <= 1e-3


@pytest.mark.parametrize("mode", ["FORCE_FP32", "FORCE_FP16"])
def test_float_modes_batch_equals_singles(gpu, pkg, lib, tmp_path, mode):
    """An image's depth has the same bits alone and in a batch of eight (3808 token
    rows); LayerScale large enough for the blocks to reach the output, a head
    whose depth varies."""
    torch = gpu
    _announce("float mode batch", mode)
    width, height, batch = 350, 266, 8
    path = _live_model(pkg, tmp_path / "vits.dav2", "vits", SEED + 9)
    xd = dev(torch, pkg.dav2_format.imagenet_input(width, height, seed=SEED + 5, batch=batch))
    out, single = empty(torch, (batch, height, width), torch.float32), empty(torch, (height, width), torch.float32)
    s = torch.cuda.current_stream().cuda_stream
    with pkg.Context(str(path), "vits", getattr(pkg, mode)) as ctx:
        ctx.infer_device(xd.data_ptr(), batch, width, height, out.data_ptr(), out.numel(), s)
        together = host(torch, out)
        assert together.std() > 1e-3
        for b in range(batch):
            ctx.infer_device(xd[b].data_ptr(), 1, width, height, single.data_ptr(), single.numel(), s)
            assert np.array_equal(host(torch, single).view(np.uint32), together[b].view(np.uint32)), b
