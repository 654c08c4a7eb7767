"""Kernels and branches of a dispatch at the sizes where they can go wrong, against plain float64 or the oracle."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def X():
    import qtensor.functional as F
    from qtensor import fused
    assert torch.cuda.is_available() and F.lib is not None
    return fused


def rel(a, b):
    a, b = torch.as_tensor(a).double().cpu(), torch.as_tensor(b).double().cpu()
    return float((a - b).norm() / b.norm().clamp_min(1e-300))


@pytest.mark.parametrize("column", [1, 15, 16, 17, 31, 32, 47, 48, 63])
def test_64_column_factor_with_a_dependent_column_at_the_edges_of_its_blocks_of_sixteen(X, column):
    g = torch.Generator().manual_seed(column)
    A = torch.randn(256, 64, generator=g, dtype=torch.float64)
    A[:, column] = A[:, :column] @ torch.randn(column, generator=g, dtype=torch.float64)
    A = A / A.norm(dim=0, keepdim=True)
    gram = (A.T @ A).float().cuda().repeat(3, 1, 1).contiguous()
    gram[2, column, column:] = float("nan")                                # a third matrix that fails there
    U, inv = torch.zeros(3, 64, 64, device="cuda"), torch.zeros(3, 64, 64, device="cuda")
    info = torch.zeros(3, dtype=torch.int32, device="cuda")
    X.cholesky_upper(gram, U, inv, info, pivot_floor=2e-4)
    assert info.tolist()[:2] == [2, 2] and info[2].item() & 1
    assert torch.equal(U[0], U[1]) and torch.equal(inv[0], inv[1])
    upper = torch.triu(U[0]).cpu()
    assert abs(float(upper[column, column]) - 2e-4 ** 0.5) < 1e-6
    assert column == 63 or float(upper[column, column + 1:].abs().max()) == 0.0
    keep = [j for j in range(64) if j != column]
    assert rel(upper[keep][:, keep], torch.linalg.cholesky(A[:, keep].T @ A[:, keep], upper=True)) <= 1e-5   # (fp32 Gram matrix, condition below 100)
    # U U^-1 = I: forward error n * 2^-24 * condition of U (1 / sqrt(floor) = 70 at most)
    assert float((upper.double() @ inv[0].double().cpu() - torch.eye(64)).abs().max()) <= 64 * 2 ** -24 * 70
    assert float(torch.tril(inv[0], -1).abs().max()) == 0.0


def fma32(a, b, c):
    """a b + c of float32 arrays, rounded once: the float64 sum is made odd where it is inexact, so that its own rounding
    decides no tie of the second one."""
    import numpy as np
    p, c = a.astype(np.float64) * b.astype(np.float64), c.astype(np.float64)               # (the product is exact)
    s = p + c
    t = s - p
    low = (p - (s - t)) + (c - t)                                                          # what the sum lost, exactly
    odd = np.where(low > 0, np.nextafter(s, np.inf), np.nextafter(s, -np.inf))
    return np.where((low != 0) & (s.view(np.int64) % 2 == 0), odd, s).astype(np.float32)


@pytest.mark.parametrize("condition", [1.0, 30.0, 1000.0])
@pytest.mark.parametrize("dependent", [None, 1, 16, 31, 47, 63])
def test_64_column_factor_and_inverse_are_the_column_by_column_recurrences(X, condition, dependent):
    """U and U^-1 bit for bit: L[i][k] = a[i][k] r_k, a[i][j] -= L[i][k] L[j][k], x[k] = s[k] r_k, s[j] -= L[j][k] x[k], one
    rounding each, k ascending (r_k = 1 / sqrt(pivot) is the diagonal of the inverse)."""
    import numpy as np
    floor = 2e-4
    g = torch.Generator().manual_seed(int(condition) + (dependent or 0))
    A = torch.linalg.qr(torch.randn(256, 64, generator=g, dtype=torch.float64))[0]
    A = A * torch.logspace(0, -float(np.log10(condition)), 64, dtype=torch.float64)
    A = A @ torch.linalg.qr(torch.randn(64, 64, generator=g, dtype=torch.float64))[0]
    if dependent is not None:
        A[:, dependent] = A[:, :dependent] @ torch.randn(dependent, generator=g, dtype=torch.float64)
    A = A / A.norm(dim=0, keepdim=True)
    gram = (A.T @ A).float()
    U, inv = torch.zeros(1, 64, 64, device="cuda"), torch.zeros(1, 64, 64, device="cuda")
    X.cholesky_upper(gram[None].cuda().contiguous(), U, inv, torch.zeros(1, dtype=torch.int32, device="cuda"), pivot_floor=floor)
    U, inv = torch.triu(U[0]).cpu().numpy(), inv[0].cpu().numpy()
    a, s = gram.numpy().T.copy(), np.eye(64, dtype=np.float32)               # (the upper triangle is what is read)
    L = np.zeros((64, 64), np.float32)
    for k in range(64):
        d, r = a[k, k], inv[k, k]
        dropped = not d > floor
        d = np.float32(floor) if dropped else d
        assert abs(float(r) ** 2 * float(d) - 1.0) <= 8 * 2.0 ** -24          # a reciprocal root off by two roundings at most, squared
        L[k:, k] = a[k:, k] * r
        if dropped:
            L[k:, k] = 0.0
            L[k, k] = d * r
        s[k] *= r
        for j in range(k + 1, 64):
            v = np.full(64, L[j, k])
            a[j:, j] = fma32(-L[j:, k], v[j:], a[j:, j])
            s[j] = fma32(-v, s[k], s[j])
    assert np.array_equal(U, L.T)
    assert np.array_equal(inv, s.T)


@pytest.mark.parametrize("column", [0, 15, 16, 40, 63])
def test_64_column_factor_keeps_the_column_of_a_pivot_that_fails(X, column):
    """A NaN shows in the factor (not only in info), and without a floor a pivot that is not positive counts as 1."""
    gram = torch.eye(64).repeat(2, 1, 1) + 2.0 ** -8 * torch.triu(torch.ones(64, 64), 1)
    gram[0, column, column] = float("nan")
    gram[1, column, column] = -4.0
    U, inv = torch.zeros(2, 64, 64, device="cuda"), torch.zeros(2, 64, 64, device="cuda")
    for floor in (2e-4, 0.0):
        info = torch.zeros(2, dtype=torch.int32, device="cuda")
        X.cholesky_upper(gram.cuda(), U, inv, info, pivot_floor=floor)
        assert info[0].item() & 1 and info[1].item() == (2 if floor else 1)
        assert bool(torch.isnan(U[0, column, column])) and bool(torch.isfinite(U[0, :column]).all())
    row = U[1].cpu()[column]                                                 # floor 0: L[i][column] = a[i][column] / 1
    assert row[column] < -3.9
    assert column == 63 or bool((row[column + 1:] > 0).all())


@pytest.mark.parametrize("row,column", [(0, 1), (3, 12), (3, 20), (21, 32), (21, 60), (33, 40), (50, 63), (62, 63)])
@pytest.mark.parametrize("entry", [float("nan"), float("inf")])
def test_64_column_inverse_of_a_factor_that_is_not_finite_is_the_column_by_column_recurrence(X, entry, row, column):
    """Where the forward substitution meets a NaN (zero times a number that is not finite is one) the inverse has it."""
    import numpy as np
    gram = (torch.eye(64) + 2.0 ** -8 * torch.triu(torch.ones(64, 64), 1)).repeat(2, 1, 1)
    gram[0, row, column] = entry
    for floor in (2e-4, 0.0):
        U, inv, info = torch.zeros(2, 64, 64, device="cuda"), torch.zeros(2, 64, 64, device="cuda"), torch.zeros(2, dtype=torch.int32, device="cuda")
        X.cholesky_upper(gram.cuda(), U, inv, info, pivot_floor=floor)
        assert info[0].item() != 0 and info[1].item() == 0 and bool(torch.isfinite(inv[1]).all())   # (an infinite entry makes a pivot of minus infinity: dropped with a floor)
        a, s = gram[0].numpy().T.copy(), np.eye(64, dtype=np.float32)
        with np.errstate(invalid="ignore"):
            for k in range(64):
                d = a[k, k]
                dropped = bool(d <= floor) and floor > 0
                d = np.float32(floor) if dropped else d if d > floor else np.float32(1.0)
                r = np.float32(1.0) / np.sqrt(d)
                L = np.where(np.arange(64) > k, 0.0, d * r).astype(np.float32) if dropped else a[:, k] * r
                s[k] *= r
                for j in range(k + 1, 64):
                    a[j:, j] -= L[j:] * L[j]
                    s[j] -= L[j] * s[k]
        assert np.isnan(s).any() and np.array_equal(np.isnan(inv[0].cpu().numpy()), np.isnan(s.T))


@pytest.mark.parametrize("order,blocksize", [(1, 64), (3, 64), (27, 64), (66, 64), (100, 64), (129, 128), (255, 256), (260, 2048),
                                             (1200, 64), (1201, 64), (1202, 512), (2049, 2048), (4099, 2048)])
@pytest.mark.parametrize("bits", [4, 8])
def test_general_quantizer_over_ragged_segments_shared_bytes_and_odd_addresses(X, order, blocksize, bits):
    import numpy as np
    import qtensor.functional as F
    from oracle import quant_np as Q
    code = F.create_linear_map(True, 4, 2) if bits == 4 else F.create_dynamic_map(True, 8, 1)
    g = torch.Generator().manual_seed(order)
    for diagonal, dtype, skew in ((True, torch.float32, 0), (False, torch.float32, 1), (True, torch.bfloat16, 1)):
        A = torch.randn(order, order, generator=g).to(dtype)
        A[order // 2] = 0.0                                                # zero segments, and one NaN segment
        A[order - 1, order - 1 if order < 3 else 1] = float("nan")
        dev = torch.empty(order * order + skew, dtype=dtype, device="cuda")[skew:].view(order, order).copy_(A)
        n_bytes = -(-order * order * bits // 8)
        room = torch.full((n_bytes + 8,), 0xA5, dtype=torch.uint8, device="cuda")
        out = room[4 + skew:4 + skew + n_bytes]
        o = Q.quantize_c(A.float().numpy(), code.numpy(), order, blocksize, bits, diagonal)
        if diagonal:
            got = F.quantize_blockwise_diagreal(dev, code.cuda(), order, blocksize=blocksize, bits=bits, out=out)
            assert np.array_equal(got[2].cpu().numpy(), o[2], equal_nan=True)
            back = F.dequantize_blockwise_diagreal(out, code.cuda(), order, got[1], got[2], blocksize=blocksize, bits=bits, outdtype=dtype)
        else:
            got = F.quantize_blockwise(dev, code.cuda(), order, blocksize=blocksize, bits=bits, out=out)
            land = torch.empty(order * order + 1, device="cuda")[1:].view(order, order)
            back = F.dequantize_blockwise(out, code.cuda(), order, got[1], blocksize=blocksize, bits=bits, out=land)
        assert np.array_equal(out.cpu().numpy(), o[0])
        assert np.array_equal(got[1].cpu().numpy(), o[1], equal_nan=True)
        assert (room[:4 + skew] == 0xA5).all() and (room[4 + skew + n_bytes:] == 0xA5).all()
        want = Q.dequantize_c(o[0], code.numpy(), order, o[1], blocksize, bits, diag=o[2] if diagonal else None,
                              to_bf16=dtype == torch.bfloat16)
        assert np.array_equal(back.float().cpu().numpy().reshape(-1), np.asarray(want).reshape(-1), equal_nan=True)


@pytest.mark.parametrize("order", [27, 100, 257])
def test_general_quantizer_over_a_stack_is_the_single_matrix_one(X, order):
    import qtensor.functional as F
    code = F.create_linear_map(True, 4, 2).cuda()
    mats = torch.randn(5, order, order, device="cuda", generator=torch.Generator(device="cuda").manual_seed(order))
    q = X.quantize_stack(mats, X.empty_quantized(5, order, 64, 4, code, True))
    back = X.dequantize_stack(q)
    for b in range(5):
        codes, absmax, diag = F.quantize_blockwise_diagreal(mats[b], code, order, blocksize=64, bits=4)
        assert torch.equal(q.codes[b], codes) and torch.equal(q.absmax[b], absmax) and torch.equal(q.diag[b], diag)
        assert torch.equal(back[b], F.dequantize_blockwise_diagreal(codes, code, order, absmax, diag, blocksize=64, bits=4))


@pytest.mark.parametrize("order,blocksize", [(1, 2048), (27, 512), (32, 64), (33, 128), (64, 2048), (65, 2048), (100, 2048), (128, 256), (129, 512),
                                             (256, 512), (300, 2048), (511, 1024), (513, 2048), (1025, 2048), (1090, 1024), (1600, 512)])
@pytest.mark.parametrize("bits", [4, 8])
def test_general_quantizer_with_segments_longer_than_the_row(X, order, blocksize, bits):
    """Stacks whose rows are one segment, shorter than the blocksize by less or more than a factor of two, and rows with a short
    last segment: every matrix against the oracle, bit for bit."""
    import numpy as np
    from oracle import quant_np as Q
    import qtensor.functional as F
    code = F.create_linear_map(True, 4, 2) if bits == 4 else F.create_dynamic_map(True, 8, 1)
    for diagonal, dtype in ((True, torch.float32), (False, torch.bfloat16)):
        mats = torch.randn(3, order, order, generator=torch.Generator().manual_seed(order)).to(dtype)
        mats[1, order // 2] = 0.0
        q = X.quantize_stack(mats.cuda(), X.empty_quantized(3, order, blocksize, bits, code.cuda(), diagonal))
        for b in range(3):
            want = Q.quantize_c(mats[b].float().numpy(), code.numpy(), order, blocksize, bits, diagonal)
            assert np.array_equal(q.codes[b].cpu().numpy(), want[0]) and np.array_equal(q.absmax[b].cpu().numpy(), want[1])
            assert not diagonal or np.array_equal(q.diag[b].cpu().numpy(), want[2])


@pytest.mark.parametrize("order,batch", [(5, 39999), (5, 40001), (27, 1371), (27, 1372), (101, 99), (999, 1), (1001, 1), (60, 36), (60, 37)])
@pytest.mark.parametrize("bits", [4, 8])
def test_general_dequantizer_on_either_side_of_the_size_at_which_a_thread_takes_more_than_a_byte(X, order, batch, bits):
    """(odd orders: a million elements in the stack; multiples of four: 2^17 in 8 bits).  The first, the middle and the last
    matrix against the oracle, bit for bit, the others against the single-matrix entry point's arithmetic."""
    import numpy as np
    import qtensor.functional as F
    from oracle import quant_np as Q
    code = F.create_linear_map(True, 4, 2) if bits == 4 else F.create_dynamic_map(True, 8, 1)
    mats = torch.randn(batch, order, order, device="cuda", generator=torch.Generator(device="cuda").manual_seed(order))
    mats[batch // 2, order // 2] = 0.0                                     # zero segments
    for diagonal, dtype in ((True, torch.float32), (False, torch.bfloat16)):
        q = X.quantize_stack(mats, X.empty_quantized(batch, order, 64, bits, code.cuda(), diagonal))
        room = torch.full((2 + batch * order * order + 2,), -7.0, dtype=dtype, device="cuda")
        back = X.dequantize_stack(q, out=room[2:-2].view(batch, order, order), outdtype=dtype)
        assert bool((room[:2] == -7.0).all()) and bool((room[-2:] == -7.0).all())
        for b in {0, batch // 2, batch - 1}:
            want = Q.dequantize_c(q.codes[b].cpu().numpy(), code.numpy(), order, q.absmax[b].cpu().numpy(), 64, bits,
                                  diag=q.diag[b].cpu().numpy() if diagonal else None, to_bf16=dtype == torch.bfloat16)
            assert np.array_equal(back[b].float().cpu().numpy().reshape(-1), np.asarray(want).reshape(-1))
        # every other element: code[id] * maximum in fp32, by torch
        ids = q.codes.long() if bits == 8 else torch.stack([q.codes.long() >> 4, q.codes.long() & 15], 2).flatten(1)
        ids = ids[:, :order * order].view(batch, order, order)
        a = q.absmax.view(batch, order, -1).repeat_interleave(64, 2)[:, :, :order]
        full = torch.where(a == 0, torch.zeros_like(a), code.cuda()[ids] * a)
        if diagonal:
            full.diagonal(dim1=1, dim2=2).copy_(q.diag)
        assert torch.equal(back, full.to(dtype))


def table_of(kind, bits):
    import qtensor.functional as F
    n = 1 << bits
    code = F.create_linear_map(True, 4, 2) if bits == 4 else F.create_dynamic_map(True, 8, 1)
    if kind == "descending":
        return code.flip(0).contiguous()
    if kind == "shuffled":
        return code[torch.randperm(n, generator=torch.Generator().manual_seed(n))].contiguous()
    if kind == "repeated":
        code = code.clone()
        code[n // 4:n // 2] = code[n // 4]
    elif kind == "neighbours":                                             # gaps of one, two, ... values of fp32 around a half
        code = (0.5 + torch.cumsum(torch.arange(n), 0).double() * 2.0 ** -24).float()
    elif kind == "tiny":                                                   # thresholds too near zero for the fast quotient
        code = code * 2.0 ** -60
    elif kind == "lopsided":                                               # one gap over many binades on either side of zero
        code = torch.cat([torch.tensor([-1.0, -2.0 ** -40, 0.0]), torch.linspace(2.0 ** -20, 1.0, n - 3)])
    return code


def around_the_thresholds(code):
    """(values, below, above): every entry, and up to six values of fp32 on either side of every gap's middle and of the value at
    which |v - lo| > |hi - v| (each difference rounded to fp32) turns true; below, above: the two values at that turn, per gap."""
    import numpy as np

    def key(x):
        b = x.view(np.int32).astype(np.int64)
        return np.where(b >= 0, b, -(b & 0x7fffffff))

    def value(k):
        return np.where(k >= 0, k, (-k) | 0x80000000).astype(np.uint32).view(np.float32)

    c = np.unique(code.numpy() + np.float32(0.0))                          # (no -0)
    lo, hi = c[:-1], c[1:]
    low, high = key(lo), key(hi)
    for _ in range(33):
        mid = (low + high) // 2
        upper = np.abs(value(mid) - lo) > np.abs(hi - value(mid))
        inside = high - low > 1
        low, high = np.where(inside & ~upper, mid, low), np.where(inside & upper, mid, high)
    middle = key((np.float32(0.5) * lo + np.float32(0.5) * hi).astype(np.float32))
    steps = np.arange(-6, 7)[:, None]
    values = np.concatenate([c, value(middle + steps).ravel(), value(high + steps).ravel()])
    return np.clip(values, -1.0, 1.0), value(high - 1), value(high)


@pytest.mark.parametrize("table", ["as it ships", "descending", "shuffled", "repeated", "neighbours", "tiny", "lopsided"])
@pytest.mark.parametrize("order", [64, 66, 1024])
@pytest.mark.parametrize("bits", [4, 8])
def test_threshold_tables_of_unusual_code_tables(X, bits, order, table):
    """Thresholds bracketed around the middle of a gap, the table taken as it stands where it ascends: codes, maxima and
    the dequantized matrix are the oracle's, bit for bit, on either side of every threshold and of the bracket's ends (small
    matrices search, ragged ones in chunks, large ones use the bucket table)."""
    import numpy as np
    import qtensor.functional as F
    from oracle import quant_np as Q
    code = table_of(table, bits)
    values, below, above = around_the_thresholds(code)
    # segments of 64 with a 1 in each, so that the quotients are the values themselves (a row of 66 has a short one as well)
    g = torch.Generator().manual_seed(order)
    per = order * (order - -(-order // 64))
    count = -(-len(values) // per)
    rows = torch.ones(count * order, order)
    free = torch.arange(order) % 64 != 0
    fill = torch.from_numpy(np.resize(values, count * per).copy())[torch.randperm(count * per, generator=g)]
    rows[:, free] = fill.view(count * order, -1)
    seen, want_code = [], []
    for A in rows.view(count, order, order):
        want, want_absmax = Q.quantize_c(A.numpy(), code.numpy(), order, 64, bits, False)
        assert (want_absmax == 1.0).all()
        out, absmax = F.quantize_blockwise(A.cuda(), code.cuda(), order, blocksize=64, bits=bits)
        back = F.dequantize_blockwise(out, code.cuda(), order, absmax, blocksize=64, bits=bits)
        assert np.array_equal(out.cpu().numpy(), want) and np.array_equal(absmax.cpu().numpy(), want_absmax)
        assert np.array_equal(back.cpu().numpy(), Q.dequantize_c(want, code.numpy(), order, want_absmax, bits=bits, blocksize=64))
        seen.append(A.numpy().ravel())
        ids = want if bits == 8 else np.stack([want >> 4, want & 15], 1).ravel()
        want_code.append(code.numpy()[ids[:order * order]])
    # the matrices held both sides of every gap's threshold, and the oracle put them on different entries
    seen, want_code = np.concatenate(seen), np.concatenate(want_code)
    entry_of = dict(zip(seen.tolist(), want_code.tolist()))
    assert all(entry_of[b] < entry_of[a] for b, a in zip(below.tolist(), above.tolist()))


@pytest.mark.parametrize("bits,order,table", [(b, n, t) for b, lines in ((4, (2688, 2752)), (8, (1216, 1280))) for n in lines
                                              for t in ("as it ships", "shuffled", "neighbours", "tiny", "lopsided")] +
                         [(b, n, "as it ships") for b in (4, 8) for n in (1408, 1472, 1728, 1792)])
def test_whole_segments_on_either_side_of_the_lines_between_the_kernels(X, bits, order, table):
    """Orders that the blocksize divides take the general kernels when small and the flat ones, with their bucket table, from some
    size on (quantizer: 7 x 2^20 elements in 4 bits, 3 x 2^19 in 8; dequantizer: 2^21, with a diagonal and for bf16 3 x 2^20):
    codes, maxima, diagonal and the dequantized matrix are the oracle's, bit for bit, around every threshold of the table."""
    import numpy as np
    import qtensor.functional as F
    from oracle import quant_np as Q
    code = table_of(table, bits)
    values, _, _ = around_the_thresholds(code)
    A = torch.from_numpy(np.resize(values, order * order).copy()).view(order, order)
    A[:, ::64] = 1.0                                   # segments of 64 with a 1 in each: the quotients are the values themselves
    A[order // 2] = 0.0
    for diag, dtype in ((False, torch.float32), (True, torch.bfloat16), (True, torch.float32)):
        if diag and table != "as it ships":
            continue
        given = A.to(dtype)
        want = Q.quantize_c(given.float().numpy(), code.numpy(), order, 64, bits, diag)
        quantize, dequantize = ((F.quantize_blockwise_diagreal, F.dequantize_blockwise_diagreal) if diag else
                                (F.quantize_blockwise, F.dequantize_blockwise))
        got = quantize(given.cuda(), code.cuda(), order, blocksize=64, bits=bits)
        back = dequantize(got[0], code.cuda(), order, *got[1:], outdtype=dtype, blocksize=64, bits=bits)
        assert all(np.array_equal(a.cpu().numpy(), b) for a, b in zip(got, want))
        full = Q.dequantize_c(want[0], code.numpy(), order, want[1], bits=bits, blocksize=64, diag=want[2] if diag else None,
                              to_bf16=dtype == torch.bfloat16)
        assert np.array_equal(back.float().cpu().numpy(), full.reshape(order, order))


@pytest.mark.parametrize("trans", ["", "a", "b"])
@pytest.mark.parametrize("k", [32, 48, 64, 80, 96, 112, 144, 1216])
@pytest.mark.parametrize("m,n", [(64, 64), (65, 128), (2, 3), (200, 70)])
def test_products_of_a_few_tiles_equal_the_same_products_in_a_large_stack(X, m, n, k, trans):
    """Loads several k tiles ahead (from k = 64 on; k ranges around the number of register sets, ragged tiles): the bits of the
    large stack's kernels, and fp32 accuracy against float64; beta E + alpha A B over it as well."""
    g = torch.Generator().manual_seed(m + n + k)
    A, B = torch.randn(m, k, generator=g), torch.randn(k, n, generator=g)
    a = (A.T if trans == "a" else A).contiguous().cuda()
    b = (B.T if trans == "b" else B).contiguous().cuda()
    E = torch.randn(m, n, generator=g).cuda()
    kw = dict(trans_a=trans == "a", trans_b=trans == "b")
    few = X.gemm(a.unsqueeze(0), b.unsqueeze(0), addend=E.unsqueeze(0), alpha=-1.0, beta=1.0, **kw)[0]
    many = X.gemm(a.repeat(400, 1, 1), b.repeat(400, 1, 1), addend=E.repeat(400, 1, 1), alpha=-1.0, beta=1.0, **kw)
    assert torch.equal(few, many[0]) and torch.equal(few, many[399])
    want = E.cpu().double() - A.double() @ B.double()
    # dropped pieces 2^-24 |a b| each and k fp32 additions: (k + 2) 2^-24 sum |a b|, plus the last sum's rounding
    bound = (k + 2) * 2 ** -24 * (A.abs().double() @ B.abs().double()) + 2 ** -23 * want.abs() + 1e-30
    assert bool(((few.cpu().double() - want).abs() <= bound).all())
    plain = X.gemm(a.unsqueeze(0), b.unsqueeze(0), **kw)[0].cpu().double()
    assert bool(((plain - A.double() @ B.double()).abs() <= bound + 2 ** -23 * (A.double() @ B.double()).abs()).all())


@pytest.mark.parametrize("form", ["plain", "addend", "symmetric", "symmetric addend", "upper a", "upper b", "skip", "word rows"])
@pytest.mark.parametrize("k", [48, 64, 80, 96, 112, 128, 144, 208])
@pytest.mark.parametrize("m", [64, 130, 208])
def test_launches_on_either_side_of_the_lines_of_the_loads_far_ahead_have_the_same_bits(X, m, k, form):
    """Dense products of at most half as many 64 x 64 tiles as units, on four k tiles or more, load several tiles ahead: a stack
    at that line against one beyond it, entry by entry, in every form that reaches the variant.  (Below k = 256 no product is
    cut along k, and up to as many tiles as units the tiles are 64 x 64 ones.)"""
    if form.startswith("upper"):
        m = k
    tiles_1 = -(-m // 64)
    tiles = tiles_1 * (tiles_1 + 1) // 2 if form.startswith("symmetric") else tiles_1 * tiles_1
    half = torch.cuda.get_device_properties(0).multi_processor_count // 2
    few, many = half // tiles, half // tiles + 1
    assert few >= 1 and few * tiles <= half < many * tiles <= 2 * half
    g = torch.Generator(device="cuda").manual_seed(m + k)
    A = torch.randn(many, m, k, device="cuda", generator=g)
    B = torch.randn(many, k, m, device="cuda", generator=g)
    kw = {}
    if form == "word rows":                                                # rows that are not 16-byte aligned: the other loads of the loaders
        A = torch.randn(many, m, k + 1, device="cuda", generator=g)[:, :, 1:]
        B = torch.randn(many, m, k + 3, device="cuda", generator=g)[:, :, 3:]
        kw = dict(trans_b=True)
    elif form.startswith("symmetric"):
        B, kw = A, dict(trans_b=True, symmetric=True)
    elif form == "upper a":
        A, kw = A.triu(), dict(upper_a=True)
    elif form == "upper b":
        B, kw = B.triu(), dict(upper_b=True)
    E = torch.randn(many, m, m, device="cuda", generator=g)
    E = E + E.transpose(1, 2)
    flags = (torch.arange(many, device="cuda") % 3 == 0).int()

    def product(count):
        more = dict(kw)
        if form.endswith("addend"):
            more.update(addend=E[:count], alpha=-1.0, beta=1.0)
        if form == "skip":
            more.update(skip=flags[:count].contiguous())
        out = torch.full((count, m, m), -7.0, device="cuda")
        return X.gemm(A[:count], B[:count], out=out, **more)

    a, b = product(few), product(many)
    assert torch.equal(a, b[:few])
    want = A.double().cpu() @ (B.transpose(1, 2) if kw.get("trans_b") else B).double().cpu()
    size = A.abs().double().cpu() @ (B.transpose(1, 2) if kw.get("trans_b") else B).abs().double().cpu()
    if form.endswith("addend"):
        want, size = E.double().cpu() - want, size + E.abs().double().cpu()
    if form == "skip":
        want[flags.bool().cpu()] = -7.0
    # dropped pieces 2^-24 |a b| each and k fp32 additions, plus the last sum's rounding
    assert bool(((b.cpu().double() - want).abs() <= (k + 4) * 2 ** -24 * size + 1e-30).all())


@pytest.mark.parametrize("order,batch,blocksize", [(2896, 1, 512), (2900, 1, 64), (2897, 1, 128), (102, 807, 64), (4100, 1, 2048)])
def test_general_quantizer_on_either_side_of_the_size_from_which_it_has_a_bucket_table(order, batch, blocksize):
    """8-bit codes, 2^23 elements: the first and the last matrix against the oracle, bit for bit."""
    import numpy as np
    import qtensor.functional as F
    from oracle import quant_np as Q
    from qtensor import fused
    code = F.create_dynamic_map(True, 8, 1)
    mats = torch.randn(batch, order, order, generator=torch.Generator().manual_seed(order))
    mats[0, order // 2] = 0.0
    mats[0, 3, 5] = float("nan")
    mats[batch - 1, order - 1] *= 1e-30                                    # maxima outside the fast division's range
    q = fused.quantize_stack(mats.cuda(), fused.empty_quantized(batch, order, blocksize, 8, code.cuda(), True))
    for b in {0, batch - 1}:
        want = Q.quantize_c(mats[b].numpy(), code.numpy(), order, blocksize, 8, True)
        assert np.array_equal(q.codes[b].cpu().numpy(), want[0])
        assert np.array_equal(q.absmax[b].cpu().numpy(), want[1], equal_nan=True) and np.array_equal(q.diag[b].cpu().numpy(), want[2], equal_nan=True)


@pytest.mark.parametrize("order,batch,bits,blocksize", [(1984, 1, 4, 64), (2048, 3, 4, 64), (2048, 1, 8, 2048), (2112, 2, 8, 64), (4096, 1, 4, 256), (5888, 1, 8, 256),
                                                       (5824, 1, 4, 64), (2112, 8, 4, 64)])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_flat_dequantizer_puts_the_diagonal_where_it_belongs_in_wide_matrices(order, batch, bits, blocksize, dtype):
    """Orders on either side of the step's 2048 elements, launches on either side of the streaming one, segments that are zero
    or not finite and NaN on the diagonal (bf16: the same NaN): against the oracle's dequantizer, bit for bit."""
    import numpy as np
    import qtensor.functional as F
    from oracle import quant_np as Q
    from qtensor import fused
    code = F.create_linear_map(True, 4, 2) if bits == 4 else F.create_dynamic_map(True, 8, 1)
    g = torch.Generator().manual_seed(order)
    q = fused.empty_quantized(batch, order, blocksize, bits, code.cuda(), True)
    q.codes.copy_(torch.randint(0, 256, q.codes.shape, generator=g, dtype=torch.uint8))
    q.absmax.copy_(torch.rand(q.absmax.shape, generator=g))
    q.diag.copy_(torch.randn(q.diag.shape, generator=g))
    q.absmax[0, 5], q.absmax[0, 6], q.absmax[0, 7] = 0.0, float("inf"), float("nan")
    q.diag[0, 9], q.diag[batch - 1, order - 1] = float("nan"), -float("nan")
    got = fused.dequantize_stack(q, outdtype=dtype)
    for b in range(batch):
        want = Q.dequantize_c(q.codes[b].cpu().numpy(), code.numpy(), order, q.absmax[b].cpu().numpy(), blocksize, bits,
                              diag=q.diag[b].cpu().numpy(), to_bf16=dtype == torch.bfloat16)
        assert np.array_equal(got[b].float().cpu().numpy(), np.asarray(want).reshape(order, order), equal_nan=True)
        if dtype == torch.bfloat16:
            bad = got[b].isnan()
            assert bool((got[b].view(torch.int16)[bad] == 0x7FC0).all())


@pytest.mark.parametrize("bits,n,k,batch", [(4, 64, 48, 1), (4, 64, 64, 1), (8, 192, 80, 3), (4, 448, 1024, 2), (4, 1216, 2400, 1),
                                            (4, 768, 128, 40), (8, 256, 64, 400)])
@pytest.mark.parametrize("left,symmetric", [(True, True), (False, True), (True, False)])
def test_reencoding_products_with_tiles_of_either_size_equal_update_then_quantize(bits, n, k, batch, left, symmetric):
    """Few workgroups of 64 x 64 tiles (loads far ahead from four k tiles on), more of them, and stacks that keep 128 x 128:
    codes, maxima and diagonal are those of the fused product to fp32 and the stack quantizer after it, bit for bit."""
    import qtensor.functional as F
    from qtensor import fused
    code = (F.create_linear_map(True, 4, 2) if bits == 4 else F.create_dynamic_map(True, 8, 1)).cuda()
    g = torch.Generator().manual_seed(n + k)
    G = 0.1 * torch.randn(batch, *((n, k) if left else (k, n)), generator=g)
    G[batch - 1, 3] = 0.0
    G[0, n - 1 if left else 0, 1] = float("nan")
    G = G.cuda()
    start = torch.randn(batch, n, n, generator=g).cuda()
    start = start + start.transpose(1, 2)
    one = fused.quantize_stack(start, fused.empty_quantized(batch, n, 64, bits, code, True))
    two = fused.quantize_stack(start, fused.empty_quantized(batch, n, 64, bits, code, True))
    kw = dict(alpha=0.05, beta=0.95, symmetric=symmetric, trans_a=not left, trans_b=left)
    fused.quantize_stack(fused.gemm(G, G, addend=two, **kw), two)
    fused.gemm(G, G, addend=one, requantize=True, **kw)
    assert torch.equal(one.codes, two.codes)
    assert torch.equal(one.absmax.view(torch.int32), two.absmax.view(torch.int32))
    assert torch.equal(one.diag.nan_to_num(7.0), two.diag.nan_to_num(7.0))


@pytest.mark.parametrize("order,blocksize,count,batch", [(4, 64, 2, 3), (64, 64, 1, 5), (68, 64, 34, 3), (256, 256, 256, 2), (1200, 64, 600, 2),
                                                         (1024, 128, 512, 3), (65, 64, 32, 2)])
@pytest.mark.parametrize("bits", [4, 8, 32])
def test_chosen_rows_of_a_stack_equal_dequantize_index_and_multiply(order, blocksize, count, batch, bits):
    """Whole matrices and views of a stack that begin anywhere, an order whose rows do not begin with whole fours (the general
    way), repeated rows, segments that are zero, infinite or NaN: bit for bit."""
    import qtensor.functional as F
    from qtensor import fused
    g = torch.Generator().manual_seed(order + bits)
    if bits == 32:
        stack = fused.DenseStack(torch.randn(batch, order, order, generator=g).cuda())
    else:
        code = (F.create_linear_map(True, 4, 2) if bits == 4 else F.create_dynamic_map(True, 8, 1)).cuda()
        stack = fused.quantize_stack(torch.randn(batch, order, order, generator=g).cuda(),
                                     fused.empty_quantized(batch, order, blocksize, bits, code, False))
        stack.absmax[0, 0], stack.absmax[-1, 1], stack.absmax[-1, -1] = 0.0, float("inf"), float("nan")
    rows = torch.randint(0, order, (batch, count), generator=g).cuda()
    rows[:, -1] = order - 1
    weights = torch.randn(batch, count, generator=g).cuda()
    full = fused.load_stack(stack)
    for first in (0, 1):
        part = stack.rows(first, batch - first)
        want = full[first:].gather(1, rows[first:].unsqueeze(2).expand(-1, -1, order))
        kept, weighted = fused.rows_of(part, rows[first:], weights[first:])
        for got, w in ((kept, want), (weighted, want * weights[first:].unsqueeze(2)), (fused.rows_of(part, rows[first:]), want),
                       (fused.rows_of(full[first:], rows[first:]), want)):
            assert torch.equal(got.nan_to_num(7.0), w.nan_to_num(7.0)) and torch.equal(got.isnan(), w.isnan())


@pytest.mark.parametrize("n,k,batch", [(4, 16, 3), (68, 32, 2), (132, 64, 3), (260, 256, 2), (1028, 288, 1)])
@pytest.mark.parametrize("symmetric,known", [(True, False), (False, False), (True, True)])
def test_products_added_to_their_own_result_buffer(X, n, k, batch, symmetric, known):
    """The addend's elements are read ahead of the stores of the same block, at the mirrored places too: an addend that is not symmetric
    and is the result as well, rows and columns that end inside a block.  fp32 sums of k terms: k 2^-24 |G| |G|^T bounds the
    products' error, two roundings the rest."""
    g = torch.Generator().manual_seed(n + k)
    G = torch.randn(batch, n, k, generator=g).cuda()
    E = torch.randn(batch, n, n, generator=g).cuda()
    G64, E64 = G.double(), E.double()
    want = 0.75 * E64 + 0.5 * (G64 @ G64.transpose(1, 2))
    size = X.measure(G) if known else None
    out = X.gemm(G, G, trans_b=True, addend=E, out=E, alpha=0.5, beta=0.75, symmetric=symmetric, amax=(size, size) if known else None)
    assert out.data_ptr() == E.data_ptr()
    bound = 2 ** -24 * (0.5 * k * (G64.abs() @ G64.abs().transpose(1, 2)) + 2 * want.abs() + 2 * E64.abs())
    assert float(((E.double() - want).abs() - bound).max()) <= 0.0


def test_rows_of_a_stack_that_is_not_one_of_fp32_matrices_are_refused():
    """Before anything is launched: the kernel reads four bytes an element and takes every address for one of the GPU."""
    from qtensor import fused
    stack, rows = torch.randn(2, 64, 64, device="cuda"), torch.zeros(2, 3, dtype=torch.int64, device="cuda")
    weights = torch.ones(2, 3, device="cuda")
    assert torch.equal(fused.rows_of(stack, rows), stack[:, :1].expand(-1, 3, -1))
    for bad, r, w in ((stack.bfloat16(), rows, None), (stack.double(), rows, None), (stack[:, :32].contiguous(), rows, None),
                      (stack.cpu(), rows, None), (stack, rows.cpu(), None), (stack, rows.int(), None), (stack, rows, weights.cpu()),
                      (stack, rows, weights.double()), (stack, rows[:1], None)):
        with pytest.raises(ValueError):
            fused.rows_of(bad, r, w)
