"""GPU kernels at the edges of their tiles, chunks and dispatch rules, against
64-bit references."""
import numpy as np
import pytest

from tests.gpu_util import dev, empty, host, ptr, torch_cuda

pytestmark = pytest.mark.gpu


def _L():
    from openmxp_amd import _lib
    return _lib.lib()


# one sample, the 16-sample passes, the 41-sample chunks (one, two, the most
# kept: 256) and a ragged last pass of each
@pytest.mark.parametrize("B", [1, 4, 5, 16, 17, 81, 82, 83, 123, 700, 10496, 10497])
def test_mlp_step_chunks(B):
    torch = torch_cuda()
    from openmxp_amd import scheduler
    L = _L()
    rng = np.random.default_rng(B)
    P = dev(scheduler.init_params(B))
    X = dev(rng.standard_normal((B, 16)).astype(np.float32))
    y = dev((rng.random(B) < 0.5).astype(np.int32))
    t, m = dev(rng.random(B).astype(np.float32)), dev((rng.random(B) < 0.5).astype(np.float32))
    H1, H2, Z = (empty(B * k, torch.float32).fill_(float("nan")) for k in (64, 64, 3))
    G, loss = empty(P.numel(), torch.float32).fill_(float("nan")), empty(1, torch.float32)
    wb = L.omx_mlp_backward_workspace_bytes(B)
    W = empty(wb, torch.uint8).fill_(255)
    guard = empty(B * 64 + 64, torch.float32).fill_(7.0)
    assert L.omx_mlp_forward_f32(B, ptr(P), ptr(X), ptr(guard), ptr(H2), ptr(Z), None) == 0
    assert bool((guard[B * 64:] == 7.0).all())
    assert L.omx_mlp_forward_f32(B, ptr(P), ptr(X), ptr(H1), ptr(H2), ptr(Z), None) == 0
    assert L.omx_mlp_backward_f32(B, ptr(P), ptr(X), ptr(H1), ptr(H2), ptr(Z), ptr(y), ptr(t), ptr(m), ptr(G),
                                  ptr(loss), ptr(W), wb, None) == 0
    Pd = P.double().cpu().requires_grad_()
    W1, b1, W2, b2, W3, b3 = torch.split(Pd, [1024, 64, 4096, 64, 192, 3])
    h1 = torch.relu(X.double().cpu() @ W1.view(16, 64) + b1)
    h2 = torch.relu(h1 @ W2.view(64, 64) + b2)
    z = h2 @ W3.view(64, 3) + b3
    want = torch.nn.functional.cross_entropy(z[:, :2], y.long().cpu()) + \
        (0.5 * m.cpu() * (z[:, 2] - t.cpu()) ** 2).mean()
    want.backward()
    # FP32 sums of at most max(82, B / 256) + 256 terms after three layers of
    # 64-term sums: (64 * 4 + terms) units of 2^-24 of the largest gradient,
    # with a factor 4 for terms larger than their sum
    tol = 4 * (64 * 4 + max(82, B / 256) + 256) * 2.0 ** -24
    g = Pd.grad.numpy()
    assert np.max(np.abs(host(G) - g)) <= tol * np.abs(g).max()
    assert abs(float(host(loss)[0]) - want.item()) <= tol * max(1.0, abs(want.item()))


def _dominant(n, seed):
    rng = np.random.default_rng(seed)
    A = rng.uniform(-0.5, 0.5, (n, n))
    A[np.arange(n), np.arange(n)] = n / 4 * (1 + 0.1 * rng.uniform(size=n))
    return A.astype(np.float32)


def _getrf(A, lda):
    """Factors of A by omx_getrf_nopiv_f32 in a buffer of leading dimension lda whose padding must stay."""
    torch = torch_cuda()
    n = A.shape[0]
    buf = np.full((n, lda), 7.0, np.float32)  # buf[j]: column j
    buf[:, :n] = A.T
    d, info = dev(buf), empty(1, torch.int32)
    assert _L().omx_getrf_nopiv_f32(n, ptr(d), lda, ptr(info), None) == 0
    out = host(d)
    assert np.all(out[:, n:] == 7.0)
    return out[:, :n].T.copy(), int(host(info)[0])


# one step, half-empty 128-wide tiles, the order of the update's sums changing
# at 512 rows, aligned and unaligned leading dimensions
@pytest.mark.parametrize("pad", [0, 4, 1])
@pytest.mark.parametrize("n", [64, 128, 192, 256, 448, 512, 576, 640, 1088])
def test_getrf_steps(n, pad):
    A = _dominant(n, n + pad)
    F, info = _getrf(A, n + pad)
    assert info == 0x7fffffff
    L, U = np.tril(F.astype(np.float64), -1) + np.eye(n), np.triu(F.astype(np.float64))
    # each entry: n products summed in FP32, one reciprocal and its product
    bound = (n + 4) * 2.0 ** -24 * (np.abs(L) @ np.abs(U))
    assert np.all(np.abs(L @ U - A) <= bound)


# pivots outside [2^-123, 2^124) take divisions instead of the refined
# hardware reciprocal: a power-of-two scaling leaves L as it is, bit for bit,
# and scales U exactly
@pytest.mark.parametrize("n", [64, 192, 576])
def test_getrf_extreme_pivots(n):
    A = _dominant(n, n)
    F, _ = _getrf(A, n)
    e = 126 - int(np.ceil(np.log2(np.abs(np.triu(F)).max())))
    G, info = _getrf((A * np.float32(2.0) ** e).astype(np.float32), n)
    assert info == 0x7fffffff and np.abs(np.diag(G)).max() >= 2.0 ** 124
    low = np.tril(np.ones((n, n), bool), -1)
    assert np.array_equal(F[low], G[low])
    assert np.array_equal(F[~low].astype(np.float64) * 2.0 ** e, G[~low].astype(np.float64))


@pytest.mark.parametrize("n,k", [(64, 0), (64, 63), (192, 70), (576, 511), (576, 575)])
def test_getrf_reports_the_first_zero_pivot(n, k):
    # a block-triangular matrix whose column k is zero from row k on
    A = np.triu(_dominant(n, k))
    A[k, k] = 0.0
    assert _getrf(A, n)[1] == k + 1


# a pivot whose reciprocal is infinite or NaN: the rows of U up to and with
# its own are finished, so they are those of the matrix with a healthy pivot in
# its place, bit for bit (first, inner and last column of a wave's eight)
@pytest.mark.parametrize("pivot", [0.0, -0.0, 1e-40, np.nan])
@pytest.mark.parametrize("n,k", [(64, 0), (64, 5), (64, 62), (64, 63), (192, 70), (576, 515)])
def test_getrf_keeps_finished_rows(n, k, pivot):
    A = _dominant(n, n + k)
    A[k:, :k] = 0.0  # row k reaches its pivot as it is
    F, _ = _getrf(A, n)
    A[k, k] = pivot
    G, info = _getrf(A, n)
    assert info == (k + 1 if pivot == 0.0 else 0x7fffffff) or np.isnan(pivot)
    assert np.array_equal(G[k, k], np.float32(pivot), equal_nan=True)
    F[k, k] = G[k, k] = 1.0
    assert np.array_equal(G[:k + 1], F[:k + 1])


# The pivots' reciprocals (hardware reciprocal and one Newton step) are the
# rounded quotients 1 / u: every mantissa, and a sample of exponents and signs.
# A diagonal matrix with ones in its last row leaves 63 of them there.
def test_getrf_reciprocals_are_rounded_quotients():
    torch = torch_cuda()
    L = _L()
    rng = np.random.default_rng(0)
    u = np.arange(0x3f800000, 0x40000000, dtype=np.uint32)
    v = rng.integers(0, 1 << 32, 1 << 18, dtype=np.uint32) & 0x807fffff | \
        (rng.integers(4, 251, 1 << 18, dtype=np.uint32) << 23)
    u = np.concatenate([u, v])
    nm = -(-len(u) // 63)
    u = np.concatenate([u, np.full(nm * 63 - len(u), u[0])]).view(np.float32).reshape(nm, 63)
    A = torch.zeros((nm, 64, 64), dtype=torch.float32, device="cuda")  # [matrix][column][row]
    i = torch.arange(63, device="cuda")
    A[:, i, i] = dev(u)
    A[:, :, 63] = 1.0
    base = ptr(A)
    torch.cuda.synchronize()
    for q in range(nm):
        assert L.omx_getrf_nopiv_f32(64, base + q * 64 * 64 * 4, 64, None, None) == 0
    got = host(A[:, :63, 63].contiguous())
    assert np.array_equal(got, np.float32(1.0) / u)


# ranges that pair up evenly, leave an odd one, and pair unequal sizes; merges
# in LDS (to 256 rows a side) and beyond; aligned and unaligned
@pytest.mark.parametrize("pad", [0, 1])
@pytest.mark.parametrize("n", [64, 128, 192, 256, 320, 448, 576, 640, 704, 1088])
def test_triangular_inverses(n, pad):
    torch = torch_cuda()
    F, _ = _getrf(_dominant(n, n), n)
    ld = n + pad
    buf = np.zeros((n, ld), np.float32)
    buf[:, :n] = F.T
    D = dev(buf)
    Xu, Xl = (empty(n * ld, torch.float32).fill_(float("nan")) for _ in range(2))
    W = empty(n * n, torch.float32).fill_(float("nan"))
    assert _L().omx_trtri_lu_f32(n, ptr(D), ld, ptr(Xu), ptr(Xl), ld, ptr(W), None) == 0
    L, U = np.tril(F.astype(np.float64), -1) + np.eye(n), np.triu(F.astype(np.float64))
    for X, T, tri in ((Xu, U, np.triu), (Xl, L, np.tril)):
        got = host(X).reshape(n, ld)[:, :n].T.astype(np.float64)
        assert np.array_equal(got, tri(got))
        want = np.linalg.inv(T)
        # products of at most n terms at every one of log2(n / 64) + 1 levels
        tol = 2 * n * 2.0 ** -24 * (np.log2(n / 64) + 1)
        assert np.all(np.abs(got - want) <= tol * (np.abs(want) @ np.abs(T) @ np.abs(want)))


# with the workspace (one launch above 512, one per block up to it): exact
# blocks, ragged last blocks, more blocks than workgroups (n > 65536 is left to the solver's
# tests), against LAPACK; x and the workspace are not written beyond n
@pytest.mark.parametrize("n,lda", [(257, 260), (300, 300), (512, 512), (575, 576), (777, 780), (1024, 1028),
                                   (2303, 2304), (4096, 4096)])
def test_trsv_with_workspace(n, lda):
    import scipy.linalg as sla
    torch = torch_cuda()
    L = _L()
    rng = np.random.default_rng(n)
    F = (np.tril(rng.uniform(-1, 1, (n, n)) / n, -1) + np.triu(rng.uniform(-1, 1, (n, n)) / n, 1)
         + np.diag(rng.uniform(1, 2, n))).astype(np.float32)
    store = np.full((n, lda), np.nan, np.float32)
    store[:, :n] = F.T
    Ad = dev(store)
    r = rng.uniform(-1, 1, n)
    wb = L.omx_trsv_workspace_bytes(n)
    W = empty(wb + 64, torch.uint8).fill_(255)
    xd = dev(np.concatenate([r, np.full(8, 3.0)]))
    F64 = F.astype(np.float64)
    y = sla.solve_triangular(np.tril(F64, -1) + np.eye(n), r, lower=True, unit_diagonal=True)
    z = sla.solve_triangular(np.triu(F64), y, lower=False)
    for rep in range(3):  # the workspace as the last call left it
        xd[:n] = dev(r)
        assert L.omx_trsv_lower_unit_f32f64(n, n, ptr(Ad), lda, ptr(xd), ptr(W), wb, None) == 0
        yg = host(xd)
        assert np.max(np.abs(yg[:n] - y)) <= 1e-13 * np.max(np.abs(y)) and np.all(yg[n:] == 3.0)
        assert L.omx_trsv_upper_f32f64(n, n, ptr(Ad), lda, ptr(xd), ptr(W), wb, None) == 0
        zg = host(xd)
        assert np.max(np.abs(zg[:n] - z)) <= 1e-13 * np.max(np.abs(z)) and np.all(zg[n:] == 3.0)
    assert bool((W[wb:] == 255).all())
    if n <= 512:  # (launch per block: a NaN reaches its whole 64-entry chain there)
        return
    # a NaN spreads as in a substitution: to every later entry, to none before
    k = 300 % n
    r[k] = np.nan
    for solve, before, after in ((L.omx_trsv_lower_unit_f32f64, slice(0, k), slice(k, n)),
                                 (L.omx_trsv_upper_f32f64, slice(k + 1, n), slice(0, k + 1))):
        xd[:n] = dev(r)
        assert solve(n, n, ptr(Ad), lda, ptr(xd), ptr(W), wb, None) == 0
        g = host(xd)[:n]
        assert np.all(np.isfinite(g[before])) and np.all(np.isnan(g[after]))


def _lu_nopiv_f32(A):
    F = A.astype(np.float32)
    for k in range(F.shape[0] - 1):
        F[k + 1:, k] /= F[k, k]
        F[k + 1:, k + 1:] -= np.outer(F[k + 1:, k], F[k, k + 1:])
    return F


def _trsv_factor(kind, n, rng):
    """LU factors whose 64 x 64 diagonal sub-blocks are ill-conditioned."""
    if kind == "randsvd":  # condition 1e6, no pivoting
        Q = [np.linalg.qr(rng.standard_normal((n, n)))[0] for _ in range(2)]
        return _lu_nopiv_f32((Q[0] * np.logspace(0, -6, n)) @ Q[1])
    F = rng.uniform(-1, 1, (n, n)) / n
    for o in range(0, n, 64):
        F[o:o + 64, o:o + 64] *= n / 4
    F[np.arange(n), np.arange(n)] = rng.uniform(1, 2, n)
    for k in (20, n // 2 + 5, n - 30):  # a small pivot and the multipliers that it leaves
        F[k, k] = kind
        F[k + 1:k // 64 * 64 + 64, k] /= kind
    return F.astype(np.float32)


# the one-launch solves and the launch per block on ill-conditioned diagonal
# sub-blocks: the backward error of each row is that of a substitution.  A
# term of a row meets at most 118 roundings (its sub-block's substitution 63 or
# 64, the sums of the columns before it 48 + 4, or 16 a tile and the tiles' sums)
@pytest.mark.parametrize("workspace", [True, False])
@pytest.mark.parametrize("n", [768, 1036])
@pytest.mark.parametrize("kind", [1e-3, 1e-6, 1e-12, "randsvd"])
def test_trsv_backward_error(kind, n, workspace):
    torch = torch_cuda()
    L = _L()
    rng = np.random.default_rng(n)
    F = _trsv_factor(kind, n, rng)
    Ad = dev(F.T.copy())
    wb = L.omx_trsv_workspace_bytes(n) if workspace else 0
    W = empty(max(wb, 8), torch.uint8).fill_(255)
    F64 = F.astype(np.float64)
    for solve, T in ((L.omx_trsv_lower_unit_f32f64, np.tril(F64, -1) + np.eye(n)),
                     (L.omx_trsv_upper_f32f64, np.triu(F64))):
        r = T @ rng.uniform(-1, 1, n)
        xd = dev(r)
        assert solve(n, n, ptr(Ad), n, ptr(xd), ptr(W) if workspace else None, wb, None) == 0
        x, T = host(xd).astype(np.longdouble), T.astype(np.longdouble)
        err = np.abs(r - T @ x) / (np.abs(r) + np.abs(T) @ np.abs(x))
        print(f"trsv {kind} n={n} workspace={workspace}: backward error {float(err.max()):.2e}", flush=True)
        assert err.max() <= 128 * 2.0 ** -53


# a zero u_kk makes x_k infinite; what was solved before it stays a solution
@pytest.mark.parametrize("k", [0, 13, 16, 63, 300, 575])
def test_trsv_zero_pivot_leaves_the_solved_entries(k):
    torch = torch_cuda()
    L, n = _L(), 576
    rng = np.random.default_rng(k)
    F = (np.triu(rng.uniform(-1, 1, (n, n)) / n, 1) + np.diag(rng.uniform(1, 2, n))).astype(np.float32)
    F[k, k] = 0.0
    r = rng.uniform(-1, 1, n)
    wb = L.omx_trsv_workspace_bytes(n)
    Ad, xd, W = dev(F.T.copy()), dev(r), empty(wb, torch.uint8).fill_(255)
    assert L.omx_trsv_upper_f32f64(n, n, ptr(Ad), n, ptr(xd), ptr(W), wb, None) == 0
    x = host(xd)
    assert not np.any(np.isfinite(x[:k + 1])) and np.isinf(x[k])
    T, x, r = F[k + 1:, k + 1:].astype(np.longdouble), x[k + 1:].astype(np.longdouble), r[k + 1:]
    assert np.all(np.abs(r - T @ x) <= 128 * 2.0 ** -53 * (np.abs(r) + np.abs(T) @ np.abs(x)))


# more blocks than workgroups (a workgroup solves several): a factor with a
# few bands, within and across blocks, solved on the host band by band
@pytest.mark.parametrize("n", [65792, 66052])
def test_trsv_more_blocks_than_workgroups(n):
    torch = torch_cuda()
    L = _L()
    rng = np.random.default_rng(n)
    bands = [1, 17, 64, 255, 256, 300, 5000, 65536]
    A = torch.zeros(n * n, dtype=torch.float32, device="cuda")  # column-major
    d = rng.uniform(1, 2, n).astype(np.float32)
    A[::n + 1] = dev(d)
    lo, up = {}, {}
    for o in bands:
        lo[o], up[o] = (rng.uniform(-0.2, 0.2, n - o).astype(np.float32) for _ in range(2))
        A[o::n + 1][:n - o] = dev(lo[o])            # (i + o, i)
        A[o * n::n + 1][:n - o] = dev(up[o])        # (i, i + o)
    wb = L.omx_trsv_workspace_bytes(n)
    W = empty(wb, torch.uint8).fill_(255)
    for solve, coef, upper in ((L.omx_trsv_lower_unit_f32f64, lo, False), (L.omx_trsv_upper_f32f64, up, True)):
        r = rng.uniform(-1, 1, n)
        xd = dev(r)
        print(f"trsv n={n} upper={upper}", flush=True)
        assert solve(n, n, ptr(A), n, ptr(xd), ptr(W), wb, None) == 0
        x = host(xd)
        res, mag = r - x * (d.astype(np.float64) if upper else 1.0), np.abs(r) + np.abs(x) * 2
        for o in bands:
            t = coef[o].astype(np.float64) * (x[o:] if upper else x[:-o])
            (res[:-o] if upper else res[o:])[:] -= t
            (mag[:-o] if upper else mag[o:])[:] += np.abs(t)
        # 118 roundings a term (above), and those of this check
        assert np.all(np.abs(res) <= 160 * 2.0 ** -53 * mag)
    del A


# the smallest buffer a factor may lie in: it ends with the last column's row n,
# and nothing beyond is read (the bytes after it are another tensor's)
@pytest.mark.parametrize("n", [513, 770, 1023])
def test_trsv_smallest_buffer(n):
    torch = torch_cuda()
    L = _L()
    rng = np.random.default_rng(n)
    lda = (n + 3) // 4 * 4
    F = (rng.uniform(-1, 1, (n, n)) / n + np.diag(rng.uniform(1, 2, n))).astype(np.float32)
    store = np.full((n, lda), np.nan, np.float32)
    store[:, :n] = F.T
    Ad = dev(store.reshape(-1)[:(n - 1) * lda + n])
    wb = L.omx_trsv_workspace_bytes(n)
    W = empty(wb, torch.uint8)
    r = rng.uniform(-1, 1, n)
    F64 = F.astype(np.float64)
    for solve, T in ((L.omx_trsv_lower_unit_f32f64, np.tril(F64, -1) + np.eye(n)),
                     (L.omx_trsv_upper_f32f64, np.triu(F64))):
        xd = dev(r)
        assert solve(n, n, ptr(Ad), lda, ptr(xd), ptr(W), wb, None) == 0
        want = np.linalg.solve(T, r)
        assert np.max(np.abs(host(xd) - want)) <= 1e-13 * np.max(np.abs(want))


# one workgroup's rows, one more, ragged ends; the largest entries at either
# end of the sums
@pytest.mark.parametrize("n", [2, 63, 64, 1023, 1024, 1025, 2048, 5000])
def test_higham_gemv_running_sums(n):
    torch = torch_cuda()
    rng = np.random.default_rng(n)
    a, b = -0.5 / n, 1.0 / n
    i = np.arange(n, dtype=np.float64)
    A = np.where(i[:, None] < i[None, :], -b + a * b * i[:, None], -a + a * b * i[None, :])
    A[np.arange(n), np.arange(n)] = 1.0 + a * b * i
    for x in (rng.uniform(-1, 1, n), np.exp(-20 * i / n), np.exp(20 * (i / n - 1))):
        y0 = rng.uniform(-1, 1, n)
        xd, yd = dev(x), dev(np.concatenate([y0, [5.0]]))
        assert _L().omx_higham_gemv_f64(n, a, b, 1.5, ptr(xd), ptr(yd), None) == 0
        got = host(yd)
        assert got[n] == 5.0
        want = y0 + 1.5 * (A @ x)
        # |u_i| sum_{j>i} |x_j| and the like: n terms, each rounded a few times
        assert np.all(np.abs(got[:n] - want) <= 4 * n * 2.0 ** -53 * (np.abs(A) @ np.abs(x) * 1.5 + np.abs(y0)))


# blocks of one to four pieces and a ragged last one, one line, full and
# ragged workgroups, both orders of sums (2^18 entries), unaligned operands
@pytest.mark.parametrize("pad", [0, 1])
@pytest.mark.parametrize("w,lines", [(64, 1), (128, 63), (192, 64), (256, 65), (320, 200), (448, 1500), (576, 4097)])
@pytest.mark.parametrize("variant", [0, 1])
def test_trsm_blocks(variant, w, lines, pad):
    import scipy.linalg as sla
    torch = torch_cuda()
    rng = np.random.default_rng(w + lines)
    T = np.triu(rng.uniform(-0.5, 0.5, (w, w)), 1) + np.tril(rng.uniform(-0.5, 0.5, (w, w)) * 4 / w, -1) \
        + np.diag(w / 4 * (1 + 0.1 * rng.uniform(size=w)))
    T = T.astype(np.float32)
    m, n = (lines, w) if variant == 0 else (w, lines)
    B = rng.uniform(-0.5, 0.5, (m, n)).astype(np.float32)
    ldt, ldb = w + pad, (m + 3) // 4 * 4 + pad
    tb, bb = np.zeros((w, ldt), np.float32), np.full((n, ldb), 7.0, np.float32)
    tb[:, :w], bb[:, :m] = T.T, B.T
    Td, Bd = dev(tb), dev(bb)
    assert _L().omx_trsm_f32(variant, m, n, ptr(Td), ldt, ptr(Bd), ldb, None) == 0
    out = host(Bd)
    assert np.all(out[:, m:] == 7.0)
    X = out[:, :m].T.astype(np.float64)
    T64 = T.astype(np.float64)
    # residual of substitution: w products a entry, rounded one by one
    if variant == 0:
        U = np.triu(T64)
        assert np.all(np.abs(X @ U - B) <= (w + 4) * 2.0 ** -24 * (np.abs(X) @ np.abs(U) + np.abs(B)))
    else:
        L = np.tril(T64, -1) + np.eye(w)
        assert np.all(np.abs(L @ X - B) <= (w + 4) * 2.0 ** -24 * (np.abs(L) @ np.abs(X) + np.abs(B)))


def _lu(n, b, alt, flags, sched, seed=3):
    """Factors of the generated system; flags of omx_solver_create."""
    import ctypes as C
    torch = torch_cuda()
    L = _L()
    A, d = empty(n * n, torch.float32), empty(n, torch.float64)
    assert L.omx_matgen_f32(n, seed, ptr(A), n, ptr(d), None) == 0
    h = C.c_void_p()
    assert L.omx_solver_create(n, b, alt, flags, C.byref(h)) == 0
    s = np.ascontiguousarray(sched, np.int32)
    assert L.omx_lu_factor(h, ptr(A), n, s.ctypes.data, None) == 0
    L.omx_solver_destroy(h)
    return host(A)


# the solver with phase timers (flag 8) runs every pack and product of a step
# as a launch of its own; without them a step's are merged: same factors, bit
# for bit, for every panel method, precision and grouping
@pytest.mark.parametrize("n,b,alt,flags,prec", [
    (256, 256, 1, 0, 0), (512, 256, 1, 0, 0), (1536, 256, 1, 0, 0), (2560, 512, 2, 0, 0), (1280, 256, 0, 0, 0),
    (1536, 256, 1, 1, 1), (2304, 256, 2, 5, 2), (3072, 768, 1, 5, 1), (2048, 256, 1, 2, 0), (1536, 256, 1, 0, -1),
    (2560, 256, 1, 5, None)])
def test_merged_launches_leave_the_factors_alone(n, b, alt, flags, prec):
    nb = n // b
    sched = [0, 1, -1, 2][:4] * nb if prec is None else [prec] * nb
    assert np.array_equal(_lu(n, b, alt, flags, sched[:nb]), _lu(n, b, alt, flags | 8, sched[:nb]))


# device memory of a solver: the group buffers, one packed panel for the
# inverse products, and what is small beside them (GMRES's basis, the inverses
# and a page an allocation within 128 MiB; a second panel would be 288 MiB)
def test_solver_memory():
    import ctypes as C
    torch = torch_cuda()
    L = _L()
    n, b = 40960, 4096
    h = C.c_void_p()
    torch.cuda.empty_cache()
    free = torch.cuda.mem_get_info()[0]
    assert L.omx_solver_create(n, b, 1, 0, C.byref(h)) == 0
    used = free - torch.cuda.mem_get_info()[0]
    L.omx_solver_destroy(h)
    panels = 4 * L.omx_panel_bytes(n - b, 2 * b, 0) + L.omx_panel_bytes(n - b, b, 0)
    inverses = 3 * 4 * b * b + 2 * L.omx_panel_bytes(b, b, 0)
    assert used <= panels + inverses + (128 << 20), (used, panels, inverses)


# FP32 product on the matrix cores: with whole groups of 64 in k and whole
# float4s of rows (or none, in the last row tile) and without either; one,
# two and many groups; last columns and rows of a tile (of 128 rows in the last
# three); nothing else written
@pytest.mark.parametrize("m,n,k,beta", [(1024, 257, 64, 1.0), (1023, 320, 128, 1.0), (513, 513, 192, 0.5),
                                        (4097, 65, 256, 0.0), (516, 1027, 48, 1.0), (1025, 256, 80, 1.0),
                                        (524288, 1, 64, 1.0), (2, 131072, 64, 1.0), (2048, 129, 1040, 0.0),
                                        (4100, 4033, 576, 1.0), (4099, 4000, 528, 0.5), (4224, 3970, 512, 0.0)])
def test_sgemm_stage_and_tile_edges(m, n, k, beta):
    torch = torch_cuda()
    print(f"sgemm edges m={m} n={n} k={k} beta={beta}", flush=True)
    L = _L()
    rng = np.random.default_rng(m + n + k)
    lda, ldb, ldc = (m + 3) // 4 * 4 + 4, k + 4, m + 3
    A = rng.uniform(-1, 1, (k, lda)).astype(np.float32)
    B = rng.uniform(-1, 1, (n, ldb)).astype(np.float32)
    C = np.full((n + 1, ldc), 7.0, np.float32)
    C[:n, :m] = rng.uniform(-1, 1, (n, m)) if beta else np.nan
    Ad, Bd, Cd = dev(A.ravel()), dev(B.ravel()), dev(C.ravel())
    assert L.omx_sgemm_f32(m, n, k, -1.0, ptr(Ad), lda, ptr(Bd), ldb, beta, ptr(Cd), ldc, None) == 0
    out = host(Cd).reshape(n + 1, ldc)
    assert np.all(out[n] == 7.0) and np.all(out[:n, m:] == 7.0)
    A64, B64 = A[:, :m].astype(np.float64), B[:, :k].astype(np.float64)
    c0 = beta * C[:n, :m].astype(np.float64) if beta else np.zeros((n, m))
    bound = (k + 2) * 2.0 ** -24 * (np.abs(c0) + np.abs(B64) @ np.abs(A64))
    assert np.all(np.abs(out[:n, :m] - (c0 - B64 @ A64)) <= bound)


# residual GEMV at the edges of its row blocks (256), column segments (64 and
# up, 4 columns a trip) and of the segments that hold a row block's diagonal
@pytest.mark.parametrize("n", [1, 63, 65, 129, 255, 257, 515, 1151, 4097, 4161])
def test_otf_gemv_segment_edges(orc, n):
    torch_cuda()
    L = _L()
    rng = np.random.default_rng(n)
    d, x, y0 = rng.uniform(n, 2 * n, n), rng.standard_normal(n), rng.standard_normal(n)
    wb = L.omx_otf_gemv_workspace_bytes(n)
    D, X, Y, W = dev(d), dev(x), dev(y0), dev(np.full(wb // 8 + 8, np.nan))
    assert L.omx_otf_gemv_f64(n, 42, ptr(D), -1.0, ptr(X), ptr(Y), ptr(W), wb, None) == 0
    assert np.all(np.isnan(host(W)[wb // 8:]))
    ref = orc.otf_gemv(n, 42, d, -1.0, x, y0)
    # both sides: n rounded additions of terms of at most |x| / 2, and d x
    bound = (2 * n + 8) * 2.0 ** -53 * (np.abs(y0) + d * np.abs(x) + 0.5 * np.abs(x).sum())
    assert np.all(np.abs(host(Y) - ref) <= bound)


# a workspace for segments of 256 columns (none up to n = 256) is taken, with
# fewer segments; one byte less is refused
@pytest.mark.parametrize("n", [1, 100, 256, 257, 1024, 5000, 16000])
def test_otf_gemv_smaller_workspace(orc, n):
    torch_cuda()
    L = _L()
    rng = np.random.default_rng(n)
    d, x, y0 = rng.uniform(n, 2 * n, n), rng.standard_normal(n), rng.standard_normal(n)
    segs = min(64, -(-n // 256))
    wb = segs * n * 8 if segs > 1 else 0
    D, X, Y, W = dev(d), dev(x), dev(y0), dev(np.full(wb // 8 + 8, np.nan))
    if wb:
        assert L.omx_otf_gemv_f64(n, 42, ptr(D), -1.0, ptr(X), ptr(Y), ptr(W), wb - 1, None) == -3
        assert L.omx_otf_gemv_f64(n, 42, ptr(D), -1.0, ptr(X), ptr(Y), None, wb, None) == -3
    assert L.omx_otf_gemv_f64(n, 42, ptr(D), -1.0, ptr(X), ptr(Y), ptr(W) if wb else None, wb, None) == 0
    assert np.all(np.isnan(host(W)[wb // 8:]))
    ref = orc.otf_gemv(n, 42, d, -1.0, x, y0)
    bound = (2 * n + 8) * 2.0 ** -53 * (np.abs(y0) + d * np.abs(x) + 0.5 * np.abs(x).sum())
    assert np.all(np.abs(host(Y) - ref) <= bound)


# x at either end of the FP64 range: a power of two times x gives that times y,
# bit for bit (no product or sum leaves the range)
@pytest.mark.parametrize("e", [1005, -900])
def test_otf_gemv_range(e):
    torch = torch_cuda()
    L, n = _L(), 1000
    rng = np.random.default_rng(5)
    D, wb = dev(rng.uniform(n, 2 * n, n)), L.omx_otf_gemv_workspace_bytes(n)
    W, x, y = empty(wb, torch.uint8), rng.uniform(-1, 1, n), []
    for s in (0, e):
        X, Y = dev(np.ldexp(x, s)), dev(np.zeros(n))
        assert L.omx_otf_gemv_f64(n, 42, ptr(D), -1.0, ptr(X), ptr(Y), ptr(W), wb, None) == 0
        y.append(host(Y))
    assert np.array_equal(np.ldexp(y[0], e), y[1])


# FP16 and FP8 products whose last tiles are cut at any row and column, with C
# on whole lines, on 16 bytes and on neither: the entries that exist are those
# of the product of whole tiles, bit for bit, and no other is written
@pytest.mark.parametrize("fp8", [False, True])
@pytest.mark.parametrize("m,n", [(1, 1), (31, 300), (300, 33), (127, 129), (257, 256), (256, 480), (512, 511),
                                 (481, 512), (385, 4)])
def test_product_tiles_cut_anywhere(fp8, m, n):
    torch = torch_cuda()
    print(f"cut tiles fp8={fp8} m={m} n={n}", flush=True)
    L = _L()
    S, k = 512, 256
    rng = np.random.default_rng(m * 1000 + n)
    col, row = dev(rng.uniform(-1, 1, S * k).astype(np.float32)), dev(rng.uniform(-1, 1, S * k).astype(np.float32))
    X, Y = (empty(L.omx_panel_bytes(S, k, int(fp8)), torch.uint8) for _ in range(2))
    if fp8:
        ne = L.omx_panel_exps_count(S, k)
        Xe, Ye, tm = empty(ne, torch.int32), empty(ne, torch.int32), empty(ne, torch.float32)
        assert L.omx_pack_f8(S, k, ptr(col), 1, S, ptr(X), ptr(Xe), ptr(tm), None) == 0
        assert L.omx_pack_f8(S, k, ptr(row), k, 1, ptr(Y), ptr(Ye), ptr(tm), None) == 0
    else:
        assert L.omx_pack_f16(S, k, ptr(col), 1, S, 0, ptr(X), None, None) == 0
        assert L.omx_pack_f16(S, k, ptr(row), k, 1, 0, ptr(Y), None, None) == 0
    c0 = rng.uniform(-1, 1, (S, S)).astype(np.float32)  # c0[column][row]

    def product(mm, nn, beta, ldc, skip):
        buf = np.full(skip + (nn + 1) * ldc, 7.0, np.float32)
        view = buf[skip:skip + nn * ldc].reshape(nn, ldc)
        view[:, :mm] = c0[:nn, :mm] if beta else np.nan
        B = dev(buf)
        p = ptr(B) + 4 * skip
        if fp8:
            rc = L.omx_gemm_f8_packed(mm, nn, k, -1.0, ptr(X), ptr(Xe), 0, ptr(Y), ptr(Ye), 0, beta, p, ldc, None)
        else:
            rc = L.omx_gemm_f16_packed(mm, nn, k, -1.0, ptr(X), 0, ptr(Y), 0, beta, p, ldc, None)
        assert rc == 0
        out = host(B)
        body = out[skip:skip + nn * ldc].reshape(nn, ldc)
        assert np.all(out[:skip] == 7.0) and np.all(out[skip + nn * ldc:] == 7.0) and np.all(body[:, mm:] == 7.0)
        return body[:, :mm]

    for beta in (1.0, 0.0):
        whole = product(S, S, beta, S, 0)
        for ldc, skip in ((544, 0), (548, 0), (513, 0), (512, 1)):
            assert np.array_equal(product(m, n, beta, ldc, skip), whole[:n, :m]), (beta, ldc, skip)
