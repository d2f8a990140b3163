"""GPU parity of the LayerNorm kernels against the CPU oracle (restatement of
FC/tests/test_layernorm.cu:8-24 and FC/src/kernels/layernorm.cu:187-269),
through the C ABI.  Tolerances: tests/tol.py."""
import numpy as np
import pytest
import torch

import cme213_amd as M
import oracle as O
from gpu_util import dev_t, host, ln_inputs, note
from tol import assert_bwd, assert_colsum, assert_exact, assert_fwd, colsum_relative

pytestmark = pytest.mark.gpu

# (rows, cols, seed): config 0, the metric's LN, config 4 (C=1600 tail and
# the wide sweep), the reference test shape, scalar / odd widths, widths past
# the register-resident templates.  Tensors of 6M-16M elements with at least
# 6144 rows take the two-rows-per-wave forward; (6161, 1022) covers it with
# scalar loads and an odd row count (the last wave has one row); (12289, 512)
# and (24700, 255) cover its gamma/beta-once form (at most 4 vectors per
# lane), with 16-byte and scalar loads, the first with an odd row count.
SHAPES = [
    (12289, 512, 20266),
    (24700, 255, 20267),
    (4096, 768, 20260),
    (8192, 768, 20261),
    (4096, 1600, 20264),
    (6161, 1022, 20265),
    (2048, 128, 42),
    (37, 33, 1),
    (1, 768, 2),
    (3, 1, 3),
    (300, 4096, 4),
    (5, 5000, 5),
    (3, 20000, 6),
    (130, 1026, 7),
]


def _colterms(g, x, mean, rstd):
    xh = (x.astype(np.float64) - mean[:, None]) * rstd[:, None]
    return g.astype(np.float64) * xh, g


@pytest.mark.parametrize("rows,cols,seed", SHAPES)
def test_layernorm_forward_backward(dev, rows, cols, seed):
    note(f"layernorm rows={rows} cols={cols} seed={seed}")
    x, gamma, beta, g = ln_inputs(rows, cols, seed)
    y_o, m_o, s_o = O.layernorm_forward(x, gamma, beta)
    dx_o, dg_o, db_o = O.layernorm_backward(g, x, m_o, s_o, gamma, dgamma=np.full(cols, 0.5, np.float32),
                                            dbeta=np.full(cols, -0.25, np.float32))

    X, G, B, Gr = dev_t(x), dev_t(gamma), dev_t(beta), dev_t(g)
    Y = torch.empty_like(X)
    Mn = torch.empty(rows, device=dev)
    Rs = torch.empty(rows, device=dev)
    M.layernorm_forward_save(X, G, B, Y, Mn, Rs, rows, cols, 1e-5)
    assert_fwd("y", host(Y), y_o)
    assert_fwd("mean", host(Mn), m_o)
    assert_fwd("rstd", host(Rs), s_o)

    Y2 = torch.empty_like(X)
    M.layernorm_forward(X, G, B, Y2, rows, cols, 1e-5)
    assert_exact("layernorm_forward == layernorm_forward_save.y", host(Y2), host(Y))

    # backward from the oracle's statistics, so dx isolates the backward
    DX = torch.empty_like(X)
    DG = torch.full((cols,), 0.5, device=dev)
    DB = torch.full((cols,), -0.25, device=dev)
    M.layernorm_backward(Gr, X, dev_t(m_o), dev_t(s_o), G, DX, DG, DB, rows, cols)
    assert_bwd("dx", host(DX), dx_o)
    tg, tb = _colterms(g, x, m_o, s_o)
    assert_colsum("dgamma", host(DG), dg_o, tg)
    assert_colsum("dbeta", host(DB), db_o, tb)


@pytest.mark.parametrize("rows,cols,seed", [(4096, 768, 11), (1024, 1600, 12), (33, 65, 13),
                                            (64, 4096, 14), (6145, 1600, 15),
                                            # partial last workgroups: waves past the last
                                            # row still reach the gamma/beta staging barrier
                                            (4097, 768, 16), (2, 768, 17)])
def test_residual_layernorm_and_backward_residual(dev, rows, cols, seed):
    note(f"residual layernorm rows={rows} cols={cols}")
    x, gamma, beta, g = ln_inputs(rows, cols, seed)
    r = np.random.default_rng(seed + 100)
    b = r.standard_normal((rows, cols), dtype=np.float32)
    res0 = r.standard_normal((rows, cols), dtype=np.float32)
    ro, yo, mo, so = O.residual_layernorm_forward(x, b, gamma, beta)

    A, Bt, G, Be = dev_t(x), dev_t(b), dev_t(gamma), dev_t(beta)
    R = torch.empty_like(A)
    Y = torch.empty_like(A)
    Mn = torch.empty(rows, device=dev)
    Rs = torch.empty(rows, device=dev)
    M.residual_layernorm_forward_save(A, Bt, G, Be, R, Y, Mn, Rs, rows, cols, 1e-5)
    assert_exact("residual_out", host(R), ro)
    assert_fwd("y", host(Y), yo)
    assert_fwd("mean", host(Mn), mo)
    assert_fwd("rstd", host(Rs), so)

    gx_o, dg_o, db_o = O.layernorm_backward(g, ro, mo, so, gamma, grad_x=res0, add_to_grad=True)
    GR = dev_t(res0)
    DG = torch.zeros(cols, device=dev)
    DB = torch.zeros(cols, device=dev)
    M.layernorm_backward_residual(dev_t(g), R, dev_t(mo), dev_t(so), G, GR, DG, DB, rows, cols)
    assert_bwd("grad_residual", host(GR), gx_o)
    tg, tb = _colterms(g, ro, mo, so)
    assert_colsum("dgamma", host(DG), dg_o, tg)
    assert_colsum("dbeta", host(DB), db_o, tb)


def test_reference_layernorm_test_case(dev):
    # FC/tests/test_layernorm.cu:29-56: 2048x128, srand(42) inputs, gamma=1,
    # beta=0; the reference accepts max-abs error < 1e-3 and logged 7.15e-7
    # for its own GPU kernel (FC/results/correctness_matrix_85267.md:23).
    rows, cols = 2048, 128
    (x,) = O.rand_unit_sequence(42, [rows * cols])
    x = x.reshape(rows, cols)
    gamma, beta = np.ones(cols, np.float32), np.zeros(cols, np.float32)
    y_o, _, _ = O.layernorm_forward(x, gamma, beta)
    Y = torch.empty(rows, cols, device=dev)
    M.layernorm_forward(dev_t(x), dev_t(gamma), dev_t(beta), Y, rows, cols, 1e-5)
    y = host(Y)
    err = float(np.abs(y - y_o).max())
    note(f"reference LN test: max abs error {err:.3e}")
    assert err < 1e-5
    assert_fwd("y", y, y_o)


def test_unaligned_pointers_take_scalar_path(dev):
    rows, cols = 64, 768
    x, gamma, beta, g = ln_inputs(rows, cols, 21)
    y_o, m_o, s_o = O.layernorm_forward(x, gamma, beta)
    dx_o, dg_o, db_o = O.layernorm_backward(g, x, m_o, s_o, gamma)
    # views that start one float past a 16-byte boundary
    buf = torch.zeros(rows * cols + 1, device=dev)
    X = buf[1:].view(rows, cols)
    X.copy_(dev_t(x))
    Y = torch.zeros(rows * cols + 1, device=dev)[1:].view(rows, cols)
    Mn = torch.empty(rows, device=dev)
    Rs = torch.empty(rows, device=dev)
    M.layernorm_forward_save(X, dev_t(gamma), dev_t(beta), Y, Mn, Rs, rows, cols, 1e-5)
    assert_fwd("y", host(Y), y_o)
    DX = torch.zeros(rows * cols + 1, device=dev)[1:].view(rows, cols)
    DG = torch.zeros(cols, device=dev)
    DB = torch.zeros(cols, device=dev)
    M.layernorm_backward(dev_t(g), X, dev_t(m_o), dev_t(s_o), dev_t(gamma), DX, DG, DB, rows, cols)
    assert_bwd("dx", host(DX), dx_o)
    tg, tb = _colterms(g, x, m_o, s_o)
    assert_colsum("dgamma", host(DG), dg_o, tg)
    assert_colsum("dbeta", host(DB), db_o, tb)


def test_backward_is_deterministic_and_constant_rows(dev):
    rows, cols = 8192, 768
    x, gamma, beta, g = ln_inputs(rows, cols, 31)
    x[::97] = 1.5  # constant rows: y must be beta exactly
    X, G, Be, Gr = dev_t(x), dev_t(gamma), dev_t(beta), dev_t(g)
    Y = torch.empty_like(X)
    Mn = torch.empty(rows, device=dev)
    Rs = torch.empty(rows, device=dev)
    M.layernorm_forward_save(X, G, Be, Y, Mn, Rs, rows, cols, 1e-5)
    y = host(Y)
    assert np.array_equal(y[::97], np.broadcast_to(beta, y[::97].shape))
    outs = []
    for _ in range(3):
        DX = torch.empty_like(X)
        DG = torch.zeros(cols, device=dev)
        DB = torch.zeros(cols, device=dev)
        M.layernorm_backward(Gr, X, Mn, Rs, G, DX, DG, DB, rows, cols)
        outs.append((host(DX), host(DG), host(DB)))
    for o in outs[1:]:
        for a, b in zip(o, outs[0]):
            assert_exact("repeat", a, b)
    # size-independent invariant: sum_c dx = 0 per row (up to fp32 rounding)
    dx = outs[0][0].astype(np.float64)
    assert np.all(np.abs(dx.sum(axis=1)) <= 1e-4 * np.abs(dx).sum(axis=1) + 1e-6)


def test_wide_sweep_config4(dev):
    # BASELINE config 4 wide sweep: LN fwd/bwd at C=4096 with 32768 rows.
    # Rows are independent, so y/mean/rstd/dx are compared with the oracle on
    # every 16th row; dgamma/dbeta (sums over all rows) are compared with a
    # float64 brute-force sum over all rows.
    rows, cols = 32768, 4096
    note(f"wide LN rows={rows} cols={cols}")
    gen = torch.Generator(device="cuda")
    gen.manual_seed(20265)
    X = torch.randn(rows, cols, device=dev, generator=gen)
    Gr = torch.randn(rows, cols, device=dev, generator=gen)
    G = 1 + 0.02 * torch.randn(cols, device=dev, generator=gen)
    Be = 0.02 * torch.randn(cols, device=dev, generator=gen)
    Y = torch.empty_like(X)
    Mn = torch.empty(rows, device=dev)
    Rs = torch.empty(rows, device=dev)
    M.layernorm_forward_save(X, G, Be, Y, Mn, Rs, rows, cols, 1e-5)
    DX = torch.empty_like(X)
    DG = torch.zeros(cols, device=dev)
    DB = torch.zeros(cols, device=dev)
    M.layernorm_backward(Gr, X, Mn, Rs, G, DX, DG, DB, rows, cols)
    torch.cuda.synchronize()

    sel = slice(0, rows, 16)
    x, g, gamma, beta = host(X[sel]), host(Gr[sel]), host(G), host(Be)
    y_o, m_o, s_o = O.layernorm_forward(x, gamma, beta)
    assert_fwd("y", host(Y[sel]), y_o)
    assert_fwd("mean", host(Mn[sel]), m_o)
    assert_fwd("rstd", host(Rs[sel]), s_o)
    dx_o, _, _ = O.layernorm_backward(g, x, host(Mn[sel]), host(Rs[sel]), gamma)
    assert_bwd("dx", host(DX[sel]), dx_o)

    x64 = X.double()
    xh = (x64 - Mn.double()[:, None]) * Rs.double()[:, None]
    g64 = Gr.double()
    tg = g64 * xh
    dg_ref = tg.sum(0)
    l2g = tg.square().sum(0).sqrt()
    db_ref = g64.sum(0)
    l2b = g64.square().sum(0).sqrt()
    del x64, xh, tg
    for name, got, ref, l2 in (("dgamma", DG, dg_ref, l2g), ("dbeta", DB, db_ref, l2b)):
        err = (got.double() - ref).abs()
        bound = 1e-4 * (ref.abs() + l2)
        assert bool((err <= bound).all()), f"{name}: max err/bound {float((err / bound).max()):.3f}"
        worst = colsum_relative(name, host(got), host(ref), host(l2))
        note(f"  {name}: max relative error {worst:.2e} on non-cancelling columns")


# Edges of the narrow-row kernels (16 and 32 lanes a row, up to 128 columns),
# of the rows spread over 4 and 16 waves (forward: 16-byte vectors from 4100 columns,
# scalars from 1025; past 49152 and 12288 the block kernel) and of the scalar
# backward's vectors per lane, with row counts that leave partial workgroups, and
# of up to 1024 rows over 4 waves each (forward, past one vector per lane).
@pytest.mark.parametrize("rows,cols", [
    (1, 4), (17, 60), (1025, 64), (16385, 64), (9, 68), (33, 124), (2049, 128), (40000, 96),
    (65, 132), (19, 1025), (7, 1281), (300, 1538), (5, 4095), (4, 4097), (3, 8191), (2, 8195),
    (1024, 260), (1025, 260), (2, 1024), (1024, 516), (33, 257), (16, 1600), (1000, 70),
    (3, 12289), (6, 4100), (300, 5120), (3, 12292), (2, 16388), (2, 49156), (700, 640 + 255),
    (9, 1279), (259, 1280), (260, 1281),
])
def test_layernorm_width_edges(dev, rows, cols):
    test_layernorm_forward_backward(dev, rows, cols, rows + cols)
    test_residual_layernorm_and_backward_residual(dev, rows, cols, rows + cols)


# Rows with a NaN, an infinity or the lowest float among rows that share their
# wave or workgroup: those others keep their bits, forward and backward, and
# the affected rows and the column sums that they reach are not finite.
@pytest.mark.parametrize("rows,cols", [(70, 60), (70, 96), (2100, 128), (30, 516), (9, 1026), (7, 5120)])
def test_non_finite_rows_stay_alone(dev, rows, cols):
    x, gamma, beta, g = ln_inputs(rows, cols, rows + cols)
    bad = {1: np.nan, 4: np.inf, rows - 1: np.finfo(np.float32).min}
    xb = x.copy()
    for r, v in bad.items():
        xb[r, r % cols] = v
    out = []
    for a in (x, xb):
        X, G, Gm = dev_t(a), dev_t(g), dev_t(gamma)
        y, dx = torch.empty(rows, cols, device=dev), torch.empty(rows, cols, device=dev)
        mean, rstd = torch.empty(rows, device=dev), torch.empty(rows, device=dev)
        dg, db = torch.zeros(cols, device=dev), torch.zeros(cols, device=dev)
        M.layernorm_forward_save(X, Gm, dev_t(beta), y, mean, rstd, rows, cols, 1e-5)
        M.layernorm_backward(G, X, mean, rstd, Gm, dx, dg, db, rows, cols)
        out.append([host(t) for t in (y, mean, rstd, dx, dg, db)])
    keep = np.array([r not in bad for r in range(rows)])
    for name, want, got in zip(("y", "mean", "rstd", "dx"), out[0], out[1]):
        assert_exact(name, got[keep], want[keep])
    assert not np.isfinite(out[1][0][[1, 4]]).any() and not np.isfinite(out[1][3][[1, 4]]).any()
    assert np.isnan(out[1][4]).all()            # dgamma: NaN normalised values reach every column
    assert_exact("dbeta", out[1][5], out[0][5])  # sums of grad_out alone
