"""
The network's large kernels against float64 products of the same bf16 operands: panel GEMM,
weight gradients over blocks of rows, 16-lane neighbour sums, ReLU backward and head, at the
edges of their tiles and of their dispatch.  fp32 sums of n terms: n * 2^-24 of the sum of
absolute terms bounds the error; bf16 outputs add 2^-8 of the value.
"""

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _bf(rng, *shape):
    import torch

    return torch.from_numpy(rng.standard_normal(shape).astype(np.float32)).to(torch.bfloat16).cuda()


def _close(got, ref, mag, terms, bf16=False):
    err = np.abs(got.double().cpu().numpy() - ref)
    bound = terms * 2.0**-24 * mag + (2.0**-8 * np.abs(ref) if bf16 else 0) + 1e-30
    assert (err <= bound).all(), (err / bound).max()


@pytest.mark.parametrize("M", [1023, 1024, 1037, 20000])
@pytest.mark.parametrize("K,N,kfast", [(32, 128, 0), (128, 128, 1), (128, 256, 1), (256, 128, 0), (384, 128, 0)])
def test_panel_products(M, K, N, kfast):
    import torch

    from tensorsat_amd import _native as N_

    rng = np.random.default_rng([M, K, N])
    a, b = _bf(rng, M, K), _bf(rng, N, K) if kfast else _bf(rng, K, N)
    bias = torch.from_numpy(rng.standard_normal(N).astype(np.float32)).cuda()
    a64, b64 = a.double().cpu().numpy(), (b.T if kfast else b).double().cpu().numpy()
    ref, mag = a64 @ b64, np.abs(a64) @ np.abs(b64)
    sb = (1, K) if kfast else (N, 1)
    for out_bf16, acc, relu in ((0, 0, 0), (1, 0, 1), (0, 1, 0), (1, 1, 0)):
        ldc = N + 8
        c = torch.full((M, ldc), 2.0, dtype=torch.bfloat16 if out_bf16 else torch.float32, device="cuda")
        print(f"M {M} K {K} N {N} kfast {kfast} bf16 {out_bf16} acc {acc}", flush=True)
        N_.check(N_.lib().ts_gnn_gemm(N_.dptr(a), K, 1, N_.dptr(b), *sb, N_.dptr(c), ldc, M, N, K,
                                      bias.data_ptr() if relu else None, relu, out_bf16, acc, N_.stream_ptr()), "gemm")
        want = ref + (bias.double().cpu().numpy() if relu else 0) + (2.0 if acc else 0)
        _close(c[:, :N], np.maximum(want, 0) if relu else want, mag + 4, K + 2, out_bf16)
        assert (c[:, N:] == 2.0).all()


@pytest.mark.parametrize("rows", [1, 63, 65, 300, 5000])
@pytest.mark.parametrize("M,N,off", [(32, 128, 0), (128, 128, 0), (384, 128, 0), (132, 128, 0), (36, 64, 0), (128, 128, 1)])
def test_weight_gradients(rows, M, N, off):
    import torch

    from tensorsat_amd import _native as N_

    rng = np.random.default_rng([rows, M, N])
    x, z = _bf(rng, rows, M + 4)[:, off : off + M], _bf(rng, rows, N)
    dw = torch.full((M, N), 0.5, device="cuda")
    need = N_.i64(0)
    N_.check(N_.lib().ts_gnn_wgrad_scratch(M, rows, N_.ctypes.byref(need)), "scratch")
    scratch = torch.full((need.value,), 255, dtype=torch.uint8, device="cuda")
    print(f"rows {rows} M {M} N {N} off {off}", flush=True)
    N_.check(N_.lib().ts_gnn_wgrad(x.data_ptr(), M + 4, N_.dptr(z), N, M, N, rows, N_.dptr(dw), N, N_.dptr(scratch),
                                   need.value, N_.stream_ptr()), "wgrad")
    x64, z64 = x.double().cpu().numpy(), z.double().cpu().numpy()
    _close(dw, x64.T @ z64 + 0.5, np.abs(x64).T @ np.abs(z64) + 1, rows + 2)


@pytest.mark.parametrize("nrows", [1, 7, 16383, 16385])
@pytest.mark.parametrize("x_f32,acc", [(0, 0), (1, 1), (1, 0), (0, 1)])
def test_neighbour_sums(nrows, x_f32, acc):
    import torch

    from tensorsat_amd import _native as N_

    rng = np.random.default_rng(nrows)
    deg = rng.choice([0, 1, 3, 4, 5, 17, 130], size=nrows, p=[0.1, 0.1, 0.4, 0.1, 0.2, 0.07, 0.03])
    rowptr = np.concatenate([[0], np.cumsum(deg)]).astype(np.int32)
    nx, e = 500, int(rowptr[-1])
    col = rng.integers(0, nx, size=max(e, 1)).astype(np.int32)
    w = rng.standard_normal(max(e, 1)).astype(np.float32)
    x = _bf(rng, nx, 256)
    dev = [torch.from_numpy(t).cuda() for t in (rowptr, col, w)]
    xin = x.float() if x_f32 else x
    out = torch.full((nrows, 384), 3.0, dtype=torch.float32 if acc else torch.bfloat16, device="cuda")
    N_.check(N_.lib().ts_gnn_segsum(*(N_.dptr(t) for t in dev), nrows, N_.dptr(xin), 256, 0, 128, x_f32, N_.dptr(out),
                                    384, 128, 256, 128, acc, N_.stream_ptr()), "segsum")
    x64 = x.double().cpu().numpy()
    row = np.repeat(np.arange(nrows), deg)
    sums = {}
    for sign, part, off in ((1, w[:e] > 0, 0), (-1, ~(w[:e] > 0), 128)):
        for absolute in (0, 1):
            t = np.abs(w[:e][part].astype(np.float64))[:, None] * x64[col[:e][part], off : off + 128]
            s = np.zeros((nrows, 128))
            np.add.at(s, row[part], np.abs(t) if absolute else t)
            sums[sign, absolute] = s
    if acc:
        _close(out[:, 128:256], sums[1, 0] + sums[-1, 0] + 3.0, sums[1, 1] + sums[-1, 1] + 3, 140)
    else:
        _close(out[:, 128:256], sums[1, 0], sums[1, 1], 140, True)
        _close(out[:, 256:], sums[-1, 0], sums[-1, 1], 140, True)
    assert (out[:, :128] == 3.0).all()


@pytest.mark.parametrize("rows", [1, 31, 33, 9000])
def test_relu_backward(rows):
    import torch

    from tensorsat_amd import _native as N_

    rng = np.random.default_rng(rows)
    dh = torch.from_numpy(rng.standard_normal((rows, 128)).astype(np.float32)).cuda()
    h = torch.relu(_bf(rng, rows, 384))
    dz, db = torch.zeros((rows, 128), dtype=torch.bfloat16, device="cuda"), torch.full((128,), 0.25, device="cuda")
    N_.check(N_.lib().ts_gnn_relu_back(N_.dptr(dh), 128, N_.dptr(h), 384, rows, 128, N_.dptr(dz), 128, N_.dptr(db),
                                       N_.stream_ptr()), "relu_back")
    want = np.where(h[:, :128].float().cpu().numpy() > 0, dh.cpu().numpy(), 0).astype(np.float64)
    np.testing.assert_array_equal(dz.float().cpu().numpy(),
                                  torch.from_numpy(want.astype(np.float32)).to(torch.bfloat16).float().numpy())
    _close(db, want.sum(0) + 0.25, np.abs(want).sum(0) + 1, rows + 2)


@pytest.mark.parametrize("masked", [False, True])
@pytest.mark.parametrize("F", [1, 64, 65, 100, 128])
@pytest.mark.parametrize("rows", [1, 3, 4, 5, 2049])
def test_head(rows, F, masked):
    """Outputs, loss and gradients of the scalar head: u = 2^-24 per operation, carried through
    y -> d = y - t -> g = 2 m d / n to the sums."""
    import torch

    from tensorsat_amd import _native as N_

    rng = np.random.default_rng([rows, F, masked])
    ldh = F + 5
    h = torch.relu(_bf(rng, rows, ldh))
    w, b, t = (torch.from_numpy(rng.standard_normal(n).astype(np.float32)).cuda() for n in (F, 1, rows))
    m = torch.from_numpy((rng.random(rows) < 0.7).astype(np.float32)).cuda() if masked else None
    inv = float(np.float32(1.0 / rows))
    y, dh = torch.full((rows + 1,), 9.0, device="cuda"), torch.full((rows * F + 1,), 9.0, device="cuda")
    dw, db, loss = (torch.full((n,), 0.5, device="cuda") for n in (F, 1, 1))
    print(f"rows {rows} F {F} mask {masked}", flush=True)
    base = (N_.dptr(h), ldh, rows, N_.dptr(w), N_.dptr(b))
    N_.check(N_.lib().ts_gnn_head(*base, None, None, 0.0, N_.dptr(y), None, None, None, None, F, 0, N_.stream_ptr()), "head")
    infer = y.clone()
    N_.check(N_.lib().ts_gnn_head(*base, N_.dptr(t), N_.dptr(m) if masked else None, inv, N_.dptr(y), N_.dptr(loss),
                                  N_.dptr(dh), N_.dptr(dw), N_.dptr(db), F, 1, N_.stream_ptr()), "head")
    assert torch.equal(y, infer) and float(y[rows]) == 9.0 and float(dh[rows * F]) == 9.0
    h64, w64, b64, t64 = (x.double().cpu().numpy() for x in (h[:, :F], w, b, t))
    m64 = m.double().cpu().numpy() if masked else np.ones(rows)
    u = 2.0**-24

    def close(got, want, bound):
        err = np.abs(got.double().cpu().numpy().reshape(want.shape) - want)
        assert (err <= bound + 1e-30).all(), (err / (bound + 1e-30)).max()

    y64 = h64 @ w64 + b64
    ey = (F + 1) * u * (np.abs(h64) @ np.abs(w64) + np.abs(b64))
    close(y[:rows], y64, ey)
    d = y64 - t64
    ed = ey + u * np.abs(d)
    g, eg = 2 * m64 * d * inv, 2 * m64 * inv * (ed + 4 * u * np.abs(d))
    close(dh[: rows * F], g[:, None] * w64, eg[:, None] * np.abs(w64) + u * np.abs(g[:, None] * w64))
    many = (rows + 4) * u  # the rows' sums, in any order, and the value they are added to
    close(dw, g @ h64 + 0.5, eg @ np.abs(h64) + many * (np.abs(g) @ np.abs(h64) + 0.5))
    close(db, np.array([g.sum() + 0.5]), eg.sum() + many * (np.abs(g).sum() + 0.5))
    sq = m64 * d * d * inv
    close(loss, np.array([sq.sum() + 0.5]), (2 * m64 * np.abs(d) * inv * ed).sum() + many * (sq.sum() + 0.5) + 4 * u * sq.sum())
