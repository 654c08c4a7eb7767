"""Products with known operand sizes (qtensor.fused.gemm(amax=...) -> qtensor_hip_gemm_ranged): the half pipe, where it
hands a tile back to the bf16 split, and the largest elements it reports.  Compared with float64 products of the same
operands.

Bound of an element's error, relative to (|A| |B|)[i][j]: an operand is kept to 2^-23 (22 bits and the sign of the rest),
the product of the rests (2^-24) is left out, and 3 k / 16 + 2 additions round to 2^-24 of sums that stay below (|A| |B|),
in blocks of 16 whose own order is the matrix instruction's: twice that is allowed for."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def X():
    import qtensor.functional as F
    import qtensor.fused as X
    assert torch.cuda.is_available() and F.lib is not None
    return X


def check(got, A, B, k):
    bound = (2 * 2.0 ** -23 + 2.0 ** -24) + 2 * (3 * k / 16 + 2) * 2.0 ** -24
    err = (got.double() - A.double() @ B.double()).abs()
    assert bool((err <= bound * (A.double().abs() @ B.double().abs()) + 1e-300).all())


@pytest.mark.parametrize("m,n,k,batch", [(64, 64, 256, 1), (2, 3, 256, 3), (129, 127, 288, 2), (128, 256, 256, 2), (257, 64, 512, 1),
                                         (100, 300, 576, 5), (1030, 520, 512, 1), (256, 256, 2048, 1), (384, 384, 544, 60)])
def test_half_pipe_against_float64_all_layouts(X, m, n, k, batch):
    g = torch.Generator(device="cuda").manual_seed(m + n + k)
    A = torch.randn(batch, m, k, device="cuda", generator=g)
    B = torch.randn(batch, k, n, device="cuda", generator=g) * 1e-6
    top = (X.amax(A), X.amax(B))
    none = torch.zeros(batch, dtype=torch.int32, device="cuda")         # (skip flags: keeps the products from being cut along k)
    assert torch.equal(top[0], A.abs().amax((1, 2))) and torch.equal(top[1], B.abs().amax((1, 2)))
    for kw, a, b in ((dict(), A, B), (dict(trans_a=True), A.transpose(1, 2).contiguous(), B), (dict(trans_b=True), A, B.transpose(1, 2).contiguous())):
        tops = torch.zeros(batch, device="cuda")
        got = X.gemm(a, b, amax=top, amax_out=tops, **kw)
        check(got, A, B, k)
        assert torch.equal(tops, got.abs().amax((1, 2)))
        # rows that are not aligned take the bf16 split: the very same bits as without amax
        if kw.get("trans_a"):
            continue
        wide = torch.zeros(batch, m, k + 5, device="cuda")
        wide[:, :, 1:k + 1] = A
        assert torch.equal(X.gemm(wide[:, :, 1:k + 1], b, amax=top, skip=none, **kw), X.gemm(A, b, skip=none, **kw))
    for short in (224, 240):                             # below the least k, and not whole lines
        assert torch.equal(X.gemm(A[:, :, :short], B[:, :short], amax=top, skip=none), X.gemm(A[:, :, :short], B[:, :short], skip=none))


@pytest.mark.parametrize("n", [128, 192])
def test_tiles_the_half_pipe_hands_back_have_the_bits_of_the_split(X, n):
    g = torch.Generator(device="cuda").manual_seed(n)
    A = torch.randn(2, n, 544, device="cuda", generator=g)
    B = torch.randn(2, 544, n, device="cuda", generator=g)
    ones = torch.ones(2, device="cuda")
    none = torch.zeros(2, dtype=torch.int32, device="cuda")             # (skip flags: keeps the products from being cut along k)
    product = lambda *args, **kw: X.gemm(*args, skip=none, **kw)           # noqa: E731
    split = product(A, B)
    top = (X.amax(A), X.amax(B))
    assert not torch.equal(product(A, B, amax=top), split)
    # bounds that are far too small or of no use: the whole product
    for bad in (1e-3, 0.0, float("inf"), float("nan"), 1e25, 1e-25):
        assert torch.equal(product(A, B, amax=(bad * ones, top[1])), split)
        assert torch.equal(product(A, B, amax=(top[0], bad * ones)), split)
    # a bound that is too large by 2^10 is still near enough
    check(product(A, B, amax=(1024 * top[0], top[1])), A, B, 544)
    # a row of an operand that is tiny, not finite, or above the bound: its tile; elsewhere, and for zero rows, the half pipe.
    # 64 covers every tile shape's rows
    for value in (1e-12, float("inf"), 1e6):
        C = A.clone()
        C[1, 3, :] = value
        C[0, 5, :] = 0.0
        got, want = product(C, B, amax=top), product(C, B)
        assert np.array_equal(got[1, :64].cpu().numpy(), want[1, :64].cpu().numpy(), equal_nan=True)
        check(got[0], C[0], B[0], 544)
        D = B.clone()
        D[1, :, n - 2] = value
        got, want = product(A, D, amax=top), product(A, D)
        assert np.array_equal(got[1, :, n - 64:].cpu().numpy(), want[1, :, n - 64:].cpu().numpy(), equal_nan=True)
        check(got[0], A[0], B[0], 544)
    # NaN makes its row NaN, as on the other pipes, and leaves the others alone
    C = A.clone()
    C[1, 3, 7] = float("nan")
    got = product(C, B, amax=top)
    assert bool(got[1, 3].isnan().all())
    got[1, 3], C[1, 3] = 0.0, 0.0
    check(got, C, B, 544)


def test_half_pipe_epilogues_skip_flags_and_pointer_lists(X):
    g = torch.Generator(device="cuda").manual_seed(5)
    n, batch = 576, 3
    A = torch.randn(batch, n, n, device="cuda", generator=g) / n ** 0.5
    E = torch.randn(batch, n, n, device="cuda", generator=g)
    top, ones = X.amax(A), torch.ones(batch, device="cuda")
    P = A.double() @ A.double()
    # addend, in place, an odd width
    got = E[:, :, :575].clone()
    tops = torch.zeros(batch, device="cuda")
    X.gemm(A, A[:, :, :575], addend=got, out=got, alpha=-0.5, beta=1.5, amax=(top, top), amax_out=tops)
    assert float((got.double() - (1.5 * E.double() - 0.5 * P)[:, :, :575]).abs().max()) <= 1e-5
    assert torch.equal(tops, got.abs().amax((1, 2)))
    # Newton epilogue with a skipped entry, operands through lists of which one entry is not aligned
    flat = torch.zeros(n * n + 4, device="cuda")
    shifted = flat[1:1 + n * n].view(n, n)
    shifted.copy_(A[2])
    ptrs = torch.tensor([A[0].data_ptr(), A[1].data_ptr(), shifted.data_ptr()], dtype=torch.int64, device="cuda")
    C, T = torch.full_like(A, 7.0), torch.full_like(A, 7.0)
    err, tops = torch.zeros(batch, device="cuda"), torch.zeros(batch, device="cuda")
    skip = torch.tensor([0, 1, 0], dtype=torch.int32, device="cuda")
    X.gemm(X.PtrList(ptrs, (batch, n, n)), A, out=C, newton=(T, -0.25, err), skip=skip, amax=(top, top), amax_out=tops)
    eye = torch.eye(n, device="cuda", dtype=torch.float64)
    for b in (0, 2):
        check(C[b], A[b], A[b], n)
        assert float((T[b].double() - (1.25 * eye - 0.25 * P[b])).abs().max()) <= 1e-5
        assert abs(float(err[b]) - float((P[b] - eye).abs().max())) <= 1e-5 and float(tops[b]) == float(C[b].abs().max())
    assert torch.equal(C[2], X.gemm(A, A, skip=skip)[2]) and bool((C[1] == 7.0).all()) and float(err[1]) == float(tops[1]) == 0.0
    # symmetric: exactly mirrored
    S = X.gemm(A, A, trans_b=True, symmetric=True, amax=(top, top))
    assert torch.equal(S, S.transpose(1, 2))
    check(S[0], A[0], A[0].T, n)
    # few tiles, long k: cut along k, with and without an upper triangular factor
    L = torch.randn(1, 64, 4096, device="cuda", generator=g)
    R = torch.randn(1, 4096, 64, device="cuda", generator=g)
    tops = torch.zeros(1, device="cuda")
    got = X.gemm(L, R, amax=(X.amax(L), X.amax(R)), amax_out=tops)
    check(got, L, R, 4096)
    assert float(tops) == float(got.abs().max())
    U = torch.triu(A)
    check(X.gemm(E, U, upper_b=True, amax=(X.amax(E), top)), E, U, n)
    with pytest.raises(ValueError):
        X.gemm(A, A, amax=(top, ones[:2]))
    assert float(X.amax(torch.full((3, 5), -2.0, device="cuda"))) == 2.0


def test_half_pipe_errors_against_those_of_the_split(X):
    """2-norm against float64 over kinds of operands that the optimizers multiply: no larger than the bf16 split's, but for
    near-identities (1.6e-7 against 1.5e-7 at k = 256): there one pair of elements makes most of a sum and shows the bit
    that is not kept, 2^-23 of either at most."""
    g = torch.Generator(device="cuda").manual_seed(7)
    for k in (256, 512, 768, 1024):
        graded = torch.exp(0.25 * torch.randn(k, 1, device="cuda", generator=g))
        kinds = [torch.randn(k, k, device="cuda", generator=g), graded * torch.randn(k, k, device="cuda", generator=g) * graded.T,
                 torch.rand(k, k, device="cuda", generator=g), torch.eye(k, device="cuda") + 1e-3 * torch.randn(k, k, device="cuda", generator=g)]
        for kind, A in enumerate(kinds):
            B = A.T.contiguous()
            want, top = A.double() @ B.double(), (X.amax(A), X.amax(B))
            half = float((X.gemm(A, B, amax=top).double() - want).norm())
            split = float((X.gemm(A, B).double() - want).norm())
            assert half <= split + (2.0 ** -22 * float(want.norm()) if kind == 3 else 0.0), (k, kind, half, split)


def test_inverse_roots_on_the_half_pipe_are_no_further_from_float64(X, monkeypatch):
    """The iteration on the half pipe against the same iteration on the bf16 split (whose products take no amax)."""
    import optimizers.matrix_functions as MF
    monkeypatch.setattr(X, "MEASURE_FROM", 0)                              # (these stacks are below the size that is measured)
    for n in (256, 320, 768):
        errors = {"half": 0.0, "split": 0.0}
        for seed in range(4):
            g = torch.Generator().manual_seed(n + seed)
            q, _ = torch.linalg.qr(torch.randn(n, n, generator=g, dtype=torch.float64))
            lam = torch.logspace(0, -1.3, n, dtype=torch.float64)
            A = ((q * lam) @ q.T).float()
            A = (A + A.T) / 2
            value, vectors = torch.linalg.eigh(A.double())
            want = (vectors * (value + 1e-6 * float(value[-1])) ** -0.25) @ vectors.T
            plain = X.gemm
            for name in errors:
                if name == "split":
                    X.gemm = lambda *a, amax=None, amax_out=None, **kw: plain(*a, **kw)
                try:
                    root = MF.ComputePowerBatched(A[None].cuda(), 4, v0=torch.ones(1, n, device="cuda"))[0].cpu().double()
                finally:
                    X.gemm = plain
                errors[name] += float((root - want).norm() / want.norm()) / 4
        assert errors["half"] <= errors["split"], (n, errors)


@pytest.mark.parametrize("bits,bs,name", [(4, 64, "linear-2"), (8, 256, "dynamic"), (8, 64, "linear-2"), (4, 128, "dynamic")])
@pytest.mark.parametrize("diag", [False, True])
def test_half_pipe_with_a_quantized_factor(X, code_maps, bits, bs, name, diag):
    """Either factor, sizes that take every tile shape, the cut along k and partners that end inside a tile; the operand is
    what the stack dequantizer (pinned to the oracle elsewhere) writes."""
    code = torch.from_numpy(code_maps[(name, bits)]).cuda()
    g = torch.Generator(device="cuda").manual_seed(bits + bs)
    for n, other, batch in ((256, 100, 2), (768, 320, 1), (1024, 64, 1), (256, 200, 40), (512, 132, 24), (320, 96, 60), (1536, 256, 1), (2304, 768, 1)):
        if n % bs:
            continue
        mats = torch.randn(batch, n, n, device="cuda", generator=g)
        mats[:, 3, :64] = 0.0                                  # a segment of zeros
        mats[0, n - 1] *= 1e-3
        q = X.quantize_stack(mats, X.empty_quantized(batch, n, bs, bits, code, diag))
        if diag:
            q.diag[0, 5] = 0.0
        deq = X.dequantize_stack(q)
        left, right = torch.randn(batch, n, other, device="cuda", generator=g), torch.randn(batch, other, n, device="cuda", generator=g)
        top = X.amax(q)
        assert bool((top >= deq.abs().amax((1, 2))).all())
        tops = torch.zeros(batch, device="cuda")
        got = X.gemm(q, left, amax=(top, X.amax(left)), amax_out=tops)
        check(got, deq, left, n)
        assert torch.equal(tops, got.abs().amax((1, 2)))
        tops.zero_()
        got = X.gemm(right, q, amax=(X.amax(right), top), amax_out=tops)
        check(got, right, deq, n)
        assert torch.equal(tops, got.abs().amax((1, 2)))
        if n > 1024:
            continue
        none = torch.zeros(batch, dtype=torch.int32, device="cuda")
        zero = torch.zeros(batch, device="cuda")               # a bound of no use: the bf16 split
        assert torch.equal(X.gemm(q, left, amax=(zero, top), skip=none), X.gemm(q, left, skip=none))
        assert torch.equal(X.gemm(right, q, amax=(top, zero), skip=none), X.gemm(right, q, skip=none))
        # maxima that are not finite or beyond the bound make their tile the split's
        q.absmax[0, 2 * (n // bs)] = float("inf")
        for product in (lambda **kw: X.gemm(q, left, **kw)[0, :64], lambda **kw: X.gemm(right, q, **kw)[0, :, :64]):
            a, b = product(amax=(top, top), skip=none), product(skip=none)
            assert np.array_equal(a.cpu().numpy(), b.cpu().numpy(), equal_nan=True)


def test_preconditioned_gradients_look_their_operands_up_where_it_pays(X, code_maps):
    """Whole products on either side of the line, which is a higher one for a call by itself than inside a bank."""
    code = torch.from_numpy(code_maps[("linear-2", 4)]).cuda()
    g = torch.Generator(device="cuda").manual_seed(1)
    for m, n, batch in ((1536, 3072, 1), (768, 3072, 1), (256, 256, 3)):
        made = [torch.randn(batch, k, k, device="cuda", generator=g) * 0.02 + torch.eye(k, device="cuda") for k in (m, n)]
        left, right = (X.quantize_stack(t, X.empty_quantized(batch, t.shape[1], 64, 4, code, True)) for t in made)
        G = torch.randn(batch, m, n, device="cuda", generator=g)
        assert X.worth_measuring(left, G, right) == (m >= 768) and X.worth_measuring(left, G, right, X.LONE_CALL) == (m == 1536)
        if m == 768:                                     # not looked up: the very bits of the products without amax
            assert torch.equal(X.precondition(G, left, right), X.gemm(X.gemm(left, G), right))
        want = X.dequantize_stack(left).double() @ G.double() @ X.dequantize_stack(right).double()
        assert float((X.precondition(G, left, right).double() - want).norm() / want.norm()) <= 1e-6
    left = X.quantize_stack(made[0], X.empty_quantized(batch, 256, 64, 4, code, True))
    flat = X.precondition(G[0], X.Quantized(left.codes[:1], left.absmax[:1], left.diag[:1], 256, 64, 4, code), right.rows(0, 1))
    assert flat.shape == (256, 256)


def test_short_sums_are_not_looked_up(X, code_maps, monkeypatch):
    """Products over short sums gain less than the look-up takes, whatever the number of matrices: preconditioned gradients
    up to 512 x 512, statistics below order 768 (re-encoded) and 512 (added to in fp32)."""
    import qtensor.functional as F
    from optimizers.engine import ShampooBank
    from optimizers.engine2 import ShampooBank2
    monkeypatch.setattr(X, "MEASURE_FROM", 0)
    code = torch.from_numpy(code_maps[("linear-2", 4)]).cuda()
    looked = []
    into = X.amax_into
    monkeypatch.setattr(X, "amax_into", lambda *a, **kw: (looked.append(a), into(*a, **kw)))
    for m, n, expect in ((256, 256, False), (512, 512, False), (384, 1024, False), (512, 576, True)):
        left, right = (X.quantize_stack(torch.eye(k, device="cuda")[None], X.empty_quantized(1, k, 64, 4, code, True)) for k in (m, n))
        del looked[:]
        X.precondition(torch.randn(1, m, n, device="cuda"), left, right)
        assert bool(looked) == expect
    for kind, order, expect in ((ShampooBank, 512, False), (ShampooBank, 768, True), (ShampooBank2, 448, False), (ShampooBank2, 512, True)):
        bank = kind([torch.nn.Parameter(torch.randn(order, order, device="cuda"))], {"linear-2": F.create_linear_map(True, 4, 2)}, "linear-2",
                    prec_maxorder=1024)
        del looked[:]
        bank.add_statistics([torch.randn(order, order, device="cuda")])
        assert any(isinstance(t, X.PtrList) for call in looked for t, _ in call) == expect


def test_matrices_that_are_left_out_are_not_looked_at(X, monkeypatch):
    """Skip flags of the look-up itself, and a bank with a parameter whose gradient is missing: its storage (here 768 floats
    for a 768 x 768 matrix) stands in the address tables and must not be read."""
    import qtensor.functional as F
    from optimizers.engine import ShampooBank
    from optimizers.engine2 import ShampooBank2
    skip = torch.tensor([0, 1, 0], dtype=torch.int32, device="cuda")
    A = torch.randn(3, 64, 96, device="cuda")
    assert torch.equal(X.amax(A, skip=skip), A.abs().amax((1, 2)) * (1 - skip))
    nowhere = torch.tensor([A[0].data_ptr(), 0, A[2].data_ptr()], dtype=torch.int64, device="cuda")
    assert torch.equal(X.amax(X.PtrList(nowhere, (3, 64, 96)), skip=skip), A.abs().amax((1, 2)) * (1 - skip))
    monkeypatch.setattr(X, "MEASURE_FROM", 0)
    code = F.create_linear_map(True, 4, 2)
    g = torch.Generator(device="cuda").manual_seed(3)
    present = torch.randn(768, 768, device="cuda", generator=g)
    absent = torch.nn.Parameter(torch.randn(1, 768, device="cuda", generator=g).expand(768, 768))
    assert absent.untyped_storage().nbytes() == 4 * 768
    grad = torch.randn(768, 768, device="cuda", generator=g)
    for kind in (ShampooBank, ShampooBank2):
        banks = [kind(params, {"linear-2": code}, "linear-2", prec_maxorder=1024)
                 for params in ([torch.nn.Parameter(present), absent], [torch.nn.Parameter(present)])]
        for bank, grads in zip(banks, ([grad, None], [grad])):
            bank.add_statistics(grads, only=[0])
        if kind is ShampooBank:                          # the statistics of the parameter that is there: rows 0, 2 and 0, 1
            for part in ("codes", "absmax", "diag"):
                both, alone = (getattr(bank.stats[768], part) for bank in banks)
                assert torch.equal(both[[0, 2]], alone)
        # both with the same roots, so that the directions can be compared (products without skip flags are cut along k)
        for bank in banks:
            for at in range(0, bank.precs[768].batch, bank.precs[768].batch // 2):
                X.quantize_stack(torch.eye(768, device="cuda")[None] + 0.01 * present[None], bank.precs[768].rows(at, 1))
        got, want = (bank.preconditioned_grads(grads, only=[0]) for bank, grads in zip(banks, ([grad, None], [grad])))
        assert got[1] is None and float((got[0] - want[0]).norm() / want[0].norm()) <= 1e-6


def two_products_bound(L, G, R):
    """Elementwise bound of deq(L) G deq(R) by the rule above for either product, and for what the first one's error becomes."""
    one = lambda k: (2 * 2.0 ** -23 + 2.0 ** -24) + 2 * (3 * k / 16 + 2) * 2.0 ** -24        # noqa: E731
    return 1.01 * (one(L.shape[-1]) + one(R.shape[-1])) * (L.double().abs() @ G.double().abs() @ R.double().abs())


@pytest.mark.parametrize("down", [20, 28, 32, 36, 40, 44, 52, 60, 100])
@pytest.mark.parametrize("factors", ["diagonal", "roots"])
def test_preconditioned_gradients_keep_small_rows_and_columns(X, code_maps, monkeypatch, down, factors):
    """Rows and columns of a gradient that are 2^-down of the others (units that hardly learn), with factors that keep them
    apart: element by element against float64.  Small rows are lines of the first product's k, small columns of the second's."""
    monkeypatch.setattr(X, "MEASURE_FROM", 0)
    code = torch.from_numpy(code_maps[("linear-2", 4)]).cuda()
    g = torch.Generator(device="cuda").manual_seed(down)
    m, n = 512, 768
    for bits in (4, 8):
        code = torch.from_numpy(code_maps[("linear-2", 4) if bits == 4 else ("dynamic", 8)]).cuda()
        made = []
        for k in (m, n):
            mats = torch.diag_embed(1 + torch.rand(2, k, device="cuda", generator=g))
            if factors == "roots":
                half = torch.arange(k, device="cuda") % 2                # units of two kinds that have nothing to do with each other
                mats = mats + 0.02 * torch.randn(2, k, k, device="cuda", generator=g) * (half[:, None] == half[None, :])
            made.append(X.quantize_stack(mats.contiguous(), X.empty_quantized(2, k, 64, bits, code, True)))
        L, R = (X.dequantize_stack(q) for q in made)
        for which in ("row", "column", "rows and columns"):
            G = torch.randn(2, m, n, device="cuda", generator=g)
            small = 2.0 ** -down
            if which == "row":
                G[0, 3] *= small
            elif which == "column":
                G[1, :, 5] *= small
            else:
                G[:, 1::2] *= small
                G[:, :, 1::2] *= small
            want = L.double() @ G.double() @ R.double()
            err = (X.precondition(G, *made).double() - want).abs()
            # (2^-120: below 2^-110 the pieces of the bf16 split reach the end of the exponents)
            assert bool((err <= two_products_bound(L, G, R) + 2.0 ** -120).all()), (bits, which)


@pytest.mark.parametrize("k,m,n", [(512, 130, 200), (768, 384, 256), (4096, 64, 64)])
def test_products_of_measured_operands_keep_small_pieces(X, k, m, n):
    """Either operand with one small line of k, small lines all along one half of k, or small elements everywhere beside one
    large row and one large column (all layouts, the cut along k): element by element against float64."""
    g = torch.Generator(device="cuda").manual_seed(k)
    for down in (30, 45, 70):
        small = 2.0 ** -down
        for kind in ("line", "half", "cross"):
            A, B = torch.randn(2, m, k, device="cuda", generator=g), torch.randn(2, k, n, device="cuda", generator=g)
            for side in (0, 1):
                a, b = A.clone(), B.clone()
                t = a if side == 0 else b.transpose(1, 2)               # [batch, rows, k]
                if kind == "line":
                    t[0, :, 7] *= small
                    (b[0, 8:] if side == 0 else a[0, :, 8:]).zero_()     # so that the line makes a part of every sum ...
                    (b[0, :7] if side == 0 else a[0, :, :7]).zero_()     # ... which nothing else does
                elif kind == "half":
                    t[:, :, 1::2] *= small
                    (b[:, ::2, ::2] if side == 0 else a[:, ::2, ::2]).zero_()
                else:
                    t[:, 1:, 1:] *= small
                    (b[:, 0, 1:] if side == 0 else a[:, 1:, 0]).zero_()
                for kw, x, y in ((dict(), a, b), (dict(trans_a=True), a.transpose(1, 2).contiguous(), b),
                                 (dict(trans_b=True), a, b.transpose(1, 2).contiguous())):
                    check(X.gemm(x, y, amax=(X.measure(x), X.measure(y)), **kw), a, b, k)


def test_measures_of_matrices_and_results(X):
    """The largest element and the fineness (1 / the smallest piece) against those counted piece by piece, of matrices of
    whole and ragged sizes and of results on every route; ordinary operands stay on the half pipe."""
    def fineness(t, rows):                                               # t [n, n]; column pieces of `rows` at these places
        a = t.abs()
        c = torch.nn.functional.pad(a, (0, -a.shape[1] % 4, 0, -a.shape[0] % rows))
        tops = torch.cat([c.reshape(c.shape[0], -1, 4).amax(2).flatten(), c.reshape(-1, rows, c.shape[1]).amax(1).flatten()])
        return 1 / tops[tops > 0].min()
    g = torch.Generator(device="cuda").manual_seed(2)
    for rows, cols in ((64, 64), (9, 4), (1, 7), (130, 33), (1000, 516)):
        t = torch.randn(3, rows, cols, device="cuda", generator=g)
        t[1] *= (torch.rand(rows, cols, device="cuda", generator=g) < 0.3)
        t[2] = 0.0
        size = X.measure(t)
        assert torch.equal(size[0], t.abs().amax((1, 2))) and float(size[1, 2]) == 0.0
        if cols % 4 == 0 or cols < 4:
            for b in (0, 1):
                assert float(size[1, b]) == float(fineness(t[b], 8))
    t[0, 3, 5] = float("nan")
    assert bool(X.measure(t)[0, 0].isnan())
    code = torch.linspace(-1, 1, 16, device="cuda")
    q = X.quantize_stack(torch.randn(2, 128, 128, device="cuda", generator=g), X.empty_quantized(2, 128, 64, 4, code, True))
    q.absmax[0, 3], q.absmax[0, 4], q.diag[1, 7] = 1e-5, 0.0, 1e-7
    assert torch.allclose(X.measure(q)[1], torch.tensor([1e5 * 15, 1e7], device="cuda"), rtol=1e-6)        # (codes of 1/15 and up)
    A = torch.randn(2, 544, 544, device="cuda", generator=g)
    A[0, 1::2, 1::2] *= 1e-3
    size = X.measure(A)
    none = torch.zeros(2, dtype=torch.int32, device="cuda")
    split, half = X.gemm(A, A, skip=none), X.gemm(A, A, amax=(size[0], size[0]), skip=none)
    assert not torch.equal(split, half)
    for kw, want in ((dict(amax=(size, size), skip=none), half), (dict(amax=(size, 1e6 * size), skip=none), split),
                     (dict(amax=(size, size), pipe="f32", skip=none), X.gemm(A, A, pipe="f32", skip=none))):
        found = torch.zeros(2, 2, device="cuda")
        got = X.gemm(A, A, amax_out=found, **kw)
        assert torch.equal(got, want) and torch.equal(found[0], got.abs().amax((1, 2)))
        for b in (0, 1):                                                 # pieces of four or eight rows: between the smallest elements ...
            assert float(1 / got[b].abs()[got[b] != 0].min()) >= float(found[1, b]) >= float(fineness(got[b], 32))     # ... and rows
    # second outputs are looked at as well
    found, T, err = torch.zeros(2, 2, device="cuda"), torch.empty_like(A), torch.zeros(2, device="cuda")
    C = torch.empty_like(A)
    X.gemm(A, A, addend=A, out=C, deviation=(T, err), amax=(size, size), amax_out=found)
    assert torch.equal(found[0], C.abs().amax((1, 2))) and torch.equal(T, C - torch.eye(544, device="cuda"))


def test_inverse_roots_keep_units_that_hardly_learn(X, monkeypatch):
    """A statistic with 64 units at 2^-40 of the others' gradients (their diagonal is the ridge's): the blocks of the root
    that tie them to the others, against the same iteration in float64.  Every round rounds them like the rest."""
    import optimizers.matrix_functions as MF
    monkeypatch.setattr(X, "MEASURE_FROM", 0)
    n = 512
    g = torch.Generator(device="cuda").manual_seed(1)
    q, _ = torch.linalg.qr(torch.randn(n, n, device="cuda", generator=g, dtype=torch.float64))
    d = torch.ones(n, device="cuda", dtype=torch.float64)
    d[-64:] = 2.0 ** -40
    mat = (d[:, None] * (q * torch.exp(-3 * torch.rand(n, device="cuda", generator=g, dtype=torch.float64))) @ q.T * d).float()
    mat = ((mat + mat.T) / 2)[None].contiguous()
    v0 = torch.ones(1, n, device="cuda")
    got = MF.ComputePowerBatched(mat.clone(), 4, v0=v0)[0].double()
    A, eye = mat[0].double(), torch.eye(n, device="cuda", dtype=torch.float64)
    A = A + 1e-6 * MF.PowerIterBatched(mat, v0=v0).double() * eye
    z = 5 / (2 * A.norm())
    M, R = A * z, eye * z ** 0.25
    for _ in range(int(MF._LAST_ROUNDS[n])):
        T = 1.25 * eye - 0.25 * M
        R, M = R @ T, (T @ T) @ (T @ T) @ M
    for block in (got[:-64, -64:] - R[:-64, -64:], got[-64:, :-64] - R[-64:, :-64]):
        assert float(block.norm() / R[:-64, -64:].norm()) <= 3e-6
    assert float((got - R).norm() / R.norm()) <= 3.3e-7


def test_preconditioned_gradients_take_every_form_of_their_factors_where_they_are_measured(X, code_maps, monkeypatch):
    """One matrix in vectors, as quantize_blockwise_diagreal returns it, with and without a diagonal, and factors given by
    addresses: the same bits as stacks and tensors."""
    import qtensor.functional as F
    monkeypatch.setattr(X, "MEASURE_FROM", 0)
    code = torch.from_numpy(code_maps[("linear-2", 4)]).cuda()
    g = torch.Generator(device="cuda").manual_seed(8)
    G, left, right = (torch.randn(*s, device="cuda", generator=g) for s in ((512, 768), (512, 512), (768, 768)))
    for diag in (True, False):
        flat, stacked = [], []
        for mat in (left, right):
            made = (F.quantize_blockwise_diagreal if diag else F.quantize_blockwise)(mat, code, mat.shape[0], blocksize=64, bits=4)
            codes, absmax, d = made if diag else made + (None,)
            assert absmax.dim() == 1
            flat.append(X.Quantized(codes, absmax, d, mat.shape[0], 64, 4, code))
            stacked.append(X.Quantized(codes[None], absmax[None], None if d is None else d[None], mat.shape[0], 64, 4, code))
        want = X.precondition(G, *stacked)
        assert torch.equal(X.precondition(G, *flat), want) and torch.equal(X.measure(flat[0]), X.measure(stacked[0]))
        half = X.Quantized(flat[0].codes[None], flat[0].absmax, flat[0].diag, 512, 64, 4, code)          # (codes stacked, the rest not)
        assert torch.equal(X.precondition(G, half, flat[1]), want)
    listed = [X.PtrList(torch.tensor([t.data_ptr()], dtype=torch.int64, device="cuda"), (1,) + tuple(t.shape)) for t in (G, left, right)]
    want = X.precondition(G[None], left[None], right[None])
    assert torch.equal(X.precondition(*listed), want) and torch.equal(X.precondition(G[None], listed[1], right[None]), want)


@pytest.mark.parametrize("variant", [1, 2])
def test_inverse_roots_of_a_part_have_the_bits_of_the_whole_stack(X, monkeypatch, variant):
    """Ten matrices of order 512, measured as a stack and not in parts of four, or of the two of one parameter."""
    import qtensor.functional as F
    from optimizers.engine import ShampooBank
    from optimizers.engine2 import ShampooBank2
    monkeypatch.setattr(X, "MEASURE_FROM", 6 * 512 ** 3)
    g = torch.Generator(device="cuda").manual_seed(4)
    grads = [torch.randn(512, 512, device="cuda", generator=g) for _ in range(5)]
    v0 = {512: torch.rand(10, 512, device="cuda", generator=g) * 2 - 1}
    make = ShampooBank if variant == 1 else lambda *a, **kw: ShampooBank2(*a, inv_root_mode=1, **kw)
    code = F.create_linear_map(True, 4, 2)
    roots = {}
    for name, part, only in (("whole", 10, None), ("parts", 4, None), ("chosen", 10, [1])):
        bank = make([torch.nn.Parameter(p) for p in grads], {"linear-2": code}, "linear-2", prec_maxorder=1024)
        bank.NEWTON_PART_BYTES = part * 4 * 512 * 512
        bank.add_statistics(grads)
        bank.compute_preconditioners(v0=v0, only=only)
        roots[name] = X.load_stack(bank.precs[512])
    assert torch.equal(roots["parts"], roots["whole"])
    assert torch.equal(roots["chosen"][[1, 6]], roots["whole"][[1, 6]])
