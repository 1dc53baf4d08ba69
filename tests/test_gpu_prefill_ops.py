"""GPU parity for the fp32 products and row moves of a prefill pass
(csrc/prefill_ops.hip) through the C ABI:

  * gemm_nt / gemm_nn (the reference's cuBLAS SGEMMs, src/backend/cuda/
    ops.cu:289-309) against float64 products of the same fp32 operands, at
    1e-5 of the largest |c| (fp32 accumulation), over ragged shapes, leading
    dimensions wider than the rows, and strided batches shaped as the
    prefill attention uses them (per-head slices of q, K and V);
  * gather_rows exactly; scatter_add_rows bitwise against the same fp32
    steps in order (dst + fp32(weight * src), row by row, repeats included).
"""

import numpy as np
import pytest

from parity import assert_f32_close, dev_f32, dev_i64, host_f32, normal

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


@pytest.fixture(scope="module", autouse=True)
def device(backend):
    if not torch.cuda.is_available() or backend.device_count() == 0:
        pytest.skip("no HIP device")
    torch.cuda.set_device(0)
    yield
    torch.cuda.synchronize()


@pytest.mark.parametrize("m,n,k", [(1, 1, 1), (7, 5, 3), (64, 64, 16), (65, 130, 33), (300, 200, 128), (37, 4096, 16)])
def test_gemm_nt_and_nn(backend, m, n, k):
    a, b_nt, b_nn = normal(500 + m, (m, k)), normal(501 + n, (n, k)), normal(502 + k, (k, n))
    c = torch.full((m, n), float("nan"), device="cuda")
    backend.gemm_nt(m, n, k, 0.37, dev_f32(a), k, 0, dev_f32(b_nt), k, 0, c, n, 0)
    assert_f32_close(host_f32(c), (0.37 * (a.astype(np.float64) @ b_nt.T.astype(np.float64))).astype(np.float32),
                     1e-5, f"gemm_nt {m}x{n}x{k}")
    backend.gemm_nn(m, n, k, dev_f32(a), k, 0, dev_f32(b_nn), n, 0, c, n, 0)
    assert_f32_close(host_f32(c), (a.astype(np.float64) @ b_nn.astype(np.float64)).astype(np.float32), 1e-5,
                     f"gemm_nn {m}x{n}x{k}")


def test_gemm_attention_shapes(backend):
    """The prefill attention's calls: per head h, S_h = scale q_h K_h^T over
    rows x keys and O_h = P_h V_h, q/K/V rows [*, heads * hd] with head h at
    column h * hd, S/P [heads, rows, keys]."""
    heads, hd, rows, keys = 4, 32, 50, 90
    width = heads * hd
    q, kc, vc = normal(510, (rows, width)), normal(511, (keys, width)), normal(512, (keys, width))
    s = torch.empty(heads, rows, keys, device="cuda")
    scale = float(1 / np.sqrt(hd))
    backend.gemm_nt(rows, keys, hd, scale, dev_f32(q), width, hd, dev_f32(kc), width, hd, s, keys, rows * keys, heads)
    p = normal(513, (heads, rows, keys))
    o = torch.full((rows, width), float("nan"), device="cuda")
    backend.gemm_nn(rows, hd, keys, dev_f32(p), keys, rows * keys, dev_f32(vc), width, hd, o, width, hd, heads)
    q64, k64, v64 = q.astype(np.float64), kc.astype(np.float64), vc.astype(np.float64)
    for h in range(heads):
        cols = slice(h * hd, (h + 1) * hd)
        assert_f32_close(host_f32(s)[h], (scale * q64[:, cols] @ k64[:, cols].T).astype(np.float32), 1e-5,
                         f"scores head {h}")
        assert_f32_close(host_f32(o)[:, cols], (p[h].astype(np.float64) @ v64[:, cols]).astype(np.float32), 1e-5,
                         f"values head {h}")


def test_gemm_rejects_bad_leading_dimension(backend):
    a = torch.zeros(4, 8, device="cuda")
    c = torch.zeros(4, 4, device="cuda")
    with pytest.raises(ValueError):
        backend.gemm_nt(4, 4, 8, 1.0, a, 4, 0, a, 8, 0, c, 4, 0)


def test_gather_and_scatter_add_rows(backend):
    rows, cols, n = 40, 77, 25
    src = normal(520, (rows, cols))
    idx = np.random.default_rng(521).integers(0, rows, n).astype(np.int64)
    idx[3] = idx[4] = 9  # a repeated index
    out = torch.empty(n, cols, device="cuda")
    backend.gather_rows(dev_f32(src), dev_i64(idx), out)
    assert np.array_equal(host_f32(out), src[idx])
    dst0 = normal(522, (rows, cols))
    w = normal(523, n)
    part = normal(524, (n, cols))
    dst = dev_f32(dst0)
    backend.scatter_add_rows(dst, dev_i64(idx), dev_f32(w), dev_f32(part))
    want = dst0.copy()
    for i in range(n):
        want[idx[i]] = want[idx[i]] + (np.float32(w[i]) * part[i]).astype(np.float32)
    assert np.array_equal(host_f32(dst).view(np.uint32), want.view(np.uint32))


@pytest.mark.parametrize("rows,cols", [(1, 4), (2, 513), (64, 512), (65, 516), (256, 1), (257, 1280), (1000, 77),
                                       (1281, 132)])
@pytest.mark.parametrize("pick", ["distinct", "repeats", "one"])
def test_scatter_add_rows_in_order(backend, rows, cols, pick):
    """Bitwise the rows added one by one: distinct indices (an expert's rows),
    indices repeated across the scan's steps, and every row onto one."""
    g = np.random.default_rng(rows * cols)
    count = rows + 3
    idx = {"distinct": g.permutation(count)[:rows], "repeats": g.integers(0, max(1, rows // 3), rows),
           "one": np.full(rows, 2)}[pick].astype(np.int64)
    dst0, w, part = normal(530, (count, cols)), normal(531, rows), normal(532, (rows, cols))
    # one element past the start: a base that allows no 16-byte access
    for shift in (0, 1):
        buf = torch.zeros(count * cols + 4, device="cuda")
        dst = buf[shift:shift + count * cols].view(count, cols)
        dst.copy_(dev_f32(dst0))
        backend.scatter_add_rows(dst, dev_i64(idx), dev_f32(w), dev_f32(part))
        want = dst0.copy()
        for i in range(rows):
            want[idx[i]] = want[idx[i]] + (np.float32(w[i]) * part[i]).astype(np.float32)
        assert np.array_equal(host_f32(dst).view(np.uint32), want.view(np.uint32)), f"shift {shift}"
        assert torch.count_nonzero(buf[:shift]) == 0 and torch.count_nonzero(buf[shift + count * cols:]) == 0


# (m, n, k, batch): each form (wide tiles with short k, k over the waves with
# 64- and 32-row tiles) at its tile edges and at k of less than a run, whole
# spans and remainders; pad: extra columns in every leading dimension and
# between slices (odd: no 16-byte reads).
@pytest.mark.parametrize("m,n,k,batch", [(2049, 2047, 33, 1), (193, 130, 160, 90), (64, 64, 8, 1100), (257, 257, 96, 16),
                                         (1003, 96, 517, 3), (33, 31, 7, 2), (65, 64, 1283, 1), (1, 1, 129, 5),
                                         (4096, 64, 1280, 1)])
@pytest.mark.parametrize("pad", [0, 1, 4])
def test_gemm_forms(backend, m, n, k, batch, pad):
    def operand(seed, r, c):
        ld, st = c + pad, r * (c + pad) + pad
        flat = dev_f32(normal(seed, batch * st))
        return flat, ld, st, torch.as_strided(flat, (batch, r, c), (st, ld, 1))

    a, lda, sa, av = operand(540, m, k)
    c_flat = torch.full((batch * (m * (n + pad) + pad),), float("nan"), device="cuda")
    ldc, sc = n + pad, m * (n + pad) + pad
    cv = torch.as_strided(c_flat, (batch, m, n), (sc, ldc, 1))
    for nt in (True, False):
        b, ldb, sb, bv = operand(541, n, k) if nt else operand(542, k, n)
        if nt:
            backend.gemm_nt(m, n, k, 0.5, a, lda, sa, b, ldb, sb, c_flat, ldc, sc, batch)
        else:
            backend.gemm_nn(m, n, k, a, lda, sa, b, ldb, sb, c_flat, ldc, sc, batch)
        alpha = 0.5 if nt else 1.0
        for s in range(0, batch, max(1, batch // 3)):
            x, y = av[s].double(), (bv[s].t() if nt else bv[s]).double().contiguous()
            want, bound = alpha * (x @ y), alpha * (x.abs() @ y.abs()) * (k + 2) * 2.0 ** -24
            assert torch.all((cv[s].double() - want).abs() <= bound + 1e-37), f"nt {nt} slice {s}"
        c_flat.fill_(float("nan"))


def test_gemm_special_values(backend):
    """Infinities and NaN reach exactly the outputs they meet; products and
    sums below the normal range are kept; k = 0 gives zeros."""
    m, n, k = 70, 40, 140
    a, b = normal(550, (m, k)), normal(551, (n, k))
    a[3, 139], a[5, 0], b[7, 64], a[9, 3], b[9, 3] = np.inf, np.nan, -np.inf, np.inf, 0.0
    a[11], b[11] = 0.0, 0.0
    a[11, 5], b[11, 5] = 2.0 ** -100, 2.0 ** -40
    with np.errstate(invalid="ignore"):
        want = (a.astype(np.float64) @ b.T.astype(np.float64)).astype(np.float32)
    c = torch.empty(m, n, device="cuda")
    for nt in (True, False):
        if nt:
            backend.gemm_nt(m, n, k, 1.0, dev_f32(a), k, 0, dev_f32(b), k, 0, c, n, 0)
        else:
            backend.gemm_nn(m, n, k, dev_f32(a), k, 0, dev_f32(np.ascontiguousarray(b.T)), n, 0, c, n, 0)
        got = host_f32(c)
        finite = np.isfinite(want)
        assert np.array_equal(np.isnan(got), np.isnan(want)) and np.array_equal(got[np.isinf(want)], want[np.isinf(want)])
        assert np.max(np.abs(got[finite] - want[finite])) <= 1e-5 * np.max(np.abs(want[finite]))
        assert got[11, 11] == np.float32(2.0 ** -140)
    backend.gemm_nt(m, n, 0, 1.0, dev_f32(a), k, 0, dev_f32(b), k, 0, c, n, 0)
    assert torch.count_nonzero(c) == 0
