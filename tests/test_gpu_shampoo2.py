"""The batched eigenbasis engine (optimizers.engine2.ShampooBank2) against the per-parameter
Preconditioner of optimizers.shampoo2 on the GPU, and its Cholesky QR against Householder QR.

What can agree how closely.  The Q factor of a QR factorisation is unique up to the signs of its
columns; the vendor's Householder routine and the Cholesky QR pick different signs, and the 4-bit
table is not symmetric around zero, so the stored bases differ in a few codes even when both Q
agree to rounding.  The strict comparison therefore runs the per-parameter path with the same
orthonormalisation, its default on a GPU (everything else -- quantizer, Bjorck steps, Rayleigh quotients, sorting,
inverse roots -- is then the reference flow per matrix against the batched flow per stack); the
comparison with the per-parameter path on Householder QR uses the tolerance of one 4-bit re-encoding."""
import pytest
import torch

pytestmark = pytest.mark.gpu
SHAPES = [(128, 192), (256, 128), (128, 1, 256)]      # only the first has a block (128 x 64) with a rank-deficient statistic
KW = dict(stat_decay=0.95, matrix_eps=1e-6, prec_maxorder=128, prec_bits=4, min_lowbit_size=4096, quan_blocksize=64)


def rel(a, b):
    a, b = torch.as_tensor(a).double().cpu(), torch.as_tensor(b).double().cpu()
    return float((a - b).norm() / b.norm().clamp_min(1e-300))


@pytest.fixture(scope="module")
def mods():
    import qtensor.functional as F
    from optimizers import shampoo2 as S2
    from optimizers import engine2 as E2
    assert torch.cuda.is_available() and F.lib is not None
    return S2, E2


@pytest.mark.parametrize("n,batch,rows", [(64, 3, 64), (256, 4, 256), (768, 2, 100), (320, 3, 320), (1024, 2, 130), (576, 1, 64)])
def test_blocked_cholesky_and_right_solve_against_float64(mods, n, batch, rows):
    import qtensor.fused as X
    g = torch.Generator().manual_seed(n)
    A = torch.randn(batch, n, n, generator=g)
    G = (A.transpose(1, 2) @ A / n + 0.1 * torch.eye(n)).cuda()
    gram, U = G.clone(), torch.full((batch, n, n), 7.0, device="cuda")
    inv = torch.zeros(batch, n, n, device="cuda")               # diagonal blocks: inverses of U's; below them: stays zero
    info = torch.zeros(batch, dtype=torch.int32, device="cuda")
    X.cholesky_upper(gram, U, inv, info)
    assert info.tolist() == [0] * batch
    blocks = torch.arange(n) // 64
    keep = (blocks[:, None] <= blocks[None, :]).cuda()            # block rows on and above the diagonal are written
    Ut = torch.where(keep, U, torch.zeros_like(U)).double()
    assert bool((torch.tril(Ut, -1) == 0).all())
    want = torch.linalg.cholesky(G.double().cpu(), upper=True)
    assert rel(Ut, want) <= 1e-5
    for j in range(n // 64):
        blk = want[:, 64 * j:64 * j + 64, 64 * j:64 * j + 64]
        assert rel(inv[:, 64 * j:64 * j + 64, 64 * j:64 * j + 64], torch.linalg.inv(blk)) <= 1e-4
    off = (blocks[:, None] != blocks[None, :]).cuda()
    assert bool((torch.where(off, inv, torch.zeros_like(inv)) == 0).all())       # nothing but the diagonal blocks written
    Q = torch.randn(batch, rows, n, generator=g).cuda()
    out = torch.empty_like(Q)
    X.solve_upper_right(Q, U, inv, gram, out)                  # doubles the inverted diagonal blocks up to 256 x 256
    for j0 in range(0, n, 256):
        j1 = min(j0 + 256, n)
        assert rel(inv[:, j0:j1, j0:j1], torch.linalg.inv(want[:, j0:j1, j0:j1])) <= 1e-4
    wide = torch.arange(n) // 256
    assert bool((torch.where((wide[:, None] != wide[None, :]).cuda(), inv, torch.zeros_like(inv)) == 0).all())
    assert bool((torch.tril(inv, -1) == 0).all())
    assert rel(out, torch.linalg.solve_triangular(want, Q.double().cpu(), upper=True, left=False)) <= 1e-4
    # a non-positive pivot is flagged, and only for its matrix
    bad = G.clone()
    bad[0, 5, 5] = -1.0
    info.zero_()
    X.cholesky_upper(bad, U, inv, info)
    assert info.tolist() == [1] + [0] * (batch - 1)
    assert rel(torch.where(keep, U, torch.zeros_like(U))[1:], want[1:]) <= 1e-5          # the others are unaffected
    with pytest.raises((RuntimeError, ValueError)):
        X.cholesky_upper(torch.zeros(1, 100, 100, device="cuda"), torch.zeros(1, 100, 100, device="cuda"),
                         torch.zeros(1, 100, 100, device="cuda"), torch.zeros(1, dtype=torch.int32, device="cuda"))


@pytest.mark.parametrize("n,batch", [(64, 5), (320, 3), (1024, 2)])
def test_distance_of_gram_matrices_from_the_identity_in_one_pass(mods, n, batch):
    import qtensor.fused as X
    g = torch.Generator().manual_seed(n)
    G = torch.eye(n) + 0.01 * torch.randn(batch, n, n, generator=g)
    G[0, 3, n - 1] = -0.75                                     # the largest deviation is negative and off the diagonal
    out = X.gram_deviation(G.cuda()).cpu()
    E = G.double() - torch.eye(n, dtype=torch.float64)
    assert torch.allclose(out[:, 0].double(), E.abs().amax(dim=(1, 2)), rtol=1e-6, atol=0)
    assert torch.allclose(out[:, 1].double(), (E * E).sum(dim=(1, 2)), rtol=1e-5, atol=0)
    assert torch.equal(out, X.gram_deviation(G.cuda()).cpu())                  # fixed summation order
    G[batch - 1, 7, 9] = float("nan")
    out = X.gram_deviation(G.cuda()).cpu()
    assert bool(out[batch - 1].isnan().all()) and not bool(out[:batch - 1].isnan().any())


def test_flagged_matrices_are_put_back_and_only_those(mods):
    import qtensor.fused as X
    g = torch.Generator().manual_seed(5)
    src, dst = torch.randn(5, 128, 128, generator=g).cuda(), torch.randn(5, 128, 128, generator=g).cuda()
    before = dst.clone()
    flags = torch.tensor([0, 1, 0, 0, 7], dtype=torch.int32, device="cuda")
    X.copy_flagged(dst, src, flags)
    assert torch.equal(dst[[1, 4]], src[[1, 4]]) and torch.equal(dst[[0, 2, 3]], before[[0, 2, 3]])


def test_cholesky_qr_gives_the_householder_factor_up_to_signs(mods):
    _, E2 = mods
    g = torch.Generator().manual_seed(3)
    n, B = 256, 6
    U, _ = torch.linalg.qr(torch.randn(B, n, n, generator=g))
    for cond in (1e1, 1e3, 1e5):
        lam = torch.logspace(0, -torch.log10(torch.tensor(cond)).item(), n)
        L = ((U * lam) @ U.transpose(1, 2)).cuda()
        V, _ = torch.linalg.qr(U + 0.05 * torch.randn(B, n, n, generator=g) / n ** 0.5)
        for basis in (torch.eye(n).expand(B, n, n).cuda(), V.cuda()):
            Y = (L @ basis).contiguous()
            Q, redone = E2.cholesky_qr(Y)
            assert redone == 0
            eye = torch.eye(n, device="cuda")
            assert float((Q.transpose(1, 2) @ Q - eye).abs().max()) < 1e-4
            R = Q.transpose(1, 2) @ Y                                  # upper triangular, positive diagonal
            assert float(torch.tril(R, -1).abs().max() / R.abs().max()) < 1e-4
            assert bool((torch.diagonal(R, dim1=1, dim2=2) > 0).all())
            Qh, Rh = torch.linalg.qr(Y.double().cpu())                 # the reference factor on the host
            Qh = Qh * torch.sign(torch.diagonal(Rh, dim1=1, dim2=2)).unsqueeze(1)
            # columns belonging to tiny pivots are determined to (rounding / pivot) only
            assert float(((Q.double().cpu() - Qh).abs() * torch.diagonal(Rh, dim1=1, dim2=2).abs().unsqueeze(1)).max()
                         / Rh.abs().max()) < 1e-5
    # an order that is not a multiple of 64 is padded with an identity block
    Y = torch.randn(3, 100, 100, generator=g).cuda()
    Q, redone = E2.cholesky_qr(Y)
    Qh, Rh = torch.linalg.qr(Y.double().cpu())
    Qh = Qh * torch.sign(torch.diagonal(Rh, dim1=1, dim2=2)).unsqueeze(1)
    assert redone == 0 and Q.shape == (3, 100, 100) and rel(Q, Qh) <= 1e-4
    # a zero column depends on the columns before it in the plainest way: it gets a stand-in, the columns
    # before it are what Householder reflections give, and the whole is orthonormal
    Y = torch.randn(2, n, n, generator=g).cuda()
    Y[1, :, 5] = 0.0
    Q, redone = E2.cholesky_qr(Y)
    assert redone == 0 and float((Q.transpose(1, 2) @ Q - torch.eye(n, device="cuda")).abs().max()) < 1e-4
    Qh, Rh = torch.linalg.qr(Y[1].double().cpu())
    Qh = Qh * torch.sign(torch.diagonal(Rh)).unsqueeze(0)
    assert rel(Q[1][:, :5], Qh[:, :5]) <= 1e-5


@pytest.mark.parametrize("n,batch,cond", [(64, 3, 1e2), (192, 4, 1e4), (320, 2, 1e1), (768, 3, 1e5), (1024, 2, 1e3)])
def test_block_gram_schmidt_sweep_against_float64_householder(mods, n, batch, cond):
    """One sweep of qtensor_hip_block_gram_schmidt_batched: orthonormal to fp32 rounding whatever the conditioning,
    nested spans kept (R = Q^T Y upper triangular with a positive diagonal), the Householder factor up to what
    the pivots allow."""
    import qtensor.fused as X
    g = torch.Generator().manual_seed(n)
    U, _ = torch.linalg.qr(torch.randn(batch, n, n, generator=g))
    V, _ = torch.linalg.qr(torch.randn(batch, n, n, generator=g))
    lam = torch.logspace(0, -torch.log10(torch.tensor(cond)).item(), n)
    Y = ((U * lam) @ V.transpose(1, 2))
    Y = (Y / torch.linalg.vector_norm(Y, dim=1, keepdim=True)).cuda().contiguous()      # unit columns, as the caller provides
    Q = Y.clone()
    info = torch.zeros(batch, dtype=torch.int32, device="cuda")
    X.block_gram_schmidt(Q, info)
    assert info.tolist() == [0] * batch                        # no pivot near the floor, nothing replaced
    eye = torch.eye(n, device="cuda")
    assert float((Q.transpose(1, 2) @ Q - eye).abs().max()) < 2e-5
    R = (Q.transpose(1, 2).double() @ Y.double()).cpu()
    assert float(torch.tril(R, -1).abs().max()) < 2e-5 and bool((torch.diagonal(R, dim1=1, dim2=2) > 0).all())
    Qh, Rh = torch.linalg.qr(Y.double().cpu())
    Qh = Qh * torch.sign(torch.diagonal(Rh, dim1=1, dim2=2)).unsqueeze(1)
    # a column is determined to (fp32 rounding / its pivot): Gram-Schmidt with reorthogonalisation reaches that,
    # where repeated Cholesky QR of the whole matrix only reached (rounding of the Gram matrix / pivot)
    weighted = (Q.double().cpu() - Qh).norm(dim=1) * torch.diagonal(Rh, dim1=1, dim2=2).abs()
    assert float(weighted.max()) < 5e-6, float(weighted.max())


def test_rank_deficient_stacks_get_a_completed_basis(mods):
    import qtensor.fused as X
    g = torch.Generator().manual_seed(17)
    n, r = 256, 96
    A = torch.randn(2, n, r, generator=g)
    Y = (A @ torch.randn(2, r, n, generator=g))                 # rank 96: columns 96.. depend on the first 96
    Y[1] = torch.randn(n, n, generator=g)                       # the second matrix is regular
    Y = (Y / torch.linalg.vector_norm(Y, dim=1, keepdim=True)).cuda().contiguous()
    Q, redone = X.cholesky_qr(Y)
    assert redone == 0
    assert float((Q.transpose(1, 2) @ Q - torch.eye(n, device="cuda")).abs().max()) < 1e-4
    Qh, Rh = torch.linalg.qr(Y.double().cpu())
    Qh = Qh * torch.sign(torch.diagonal(Rh, dim1=1, dim2=2)).unsqueeze(1)
    assert rel(Q[0][:, :r - 8], Qh[0][:, :r - 8]) <= 1e-4       # (the last few independent columns have small pivots)
    assert rel(Q[1], Qh[1]) <= 1e-3
    # the first 96 columns span the range of Y[0]: every column of Y[0] lies in it
    lead = Q[0][:, :r].double().cpu()
    resid = Y[0].double().cpu() - lead @ (lead.T @ Y[0].double().cpu())
    assert float(resid.norm(dim=0).max()) < 1e-5
    # the sweep alone: bit 2 of info marks the matrix whose noise columns were replaced, and only that one
    Q2 = Y.clone()
    info = torch.zeros(2, dtype=torch.int32, device="cuda")
    X.block_gram_schmidt(Q2, info)
    assert (info[0].item() & 4) != 0 and (info[1].item() & 4) == 0
    # without stand-ins the noise columns stay noise: the sweep then leaves the matrix far from orthonormal
    Q3 = Y.clone()
    info.zero_()
    X.block_gram_schmidt(Q3, info, complete=False)
    assert (info[0].item() & 4) == 0
    assert float((Q3[1].T @ Q3[1] - torch.eye(n, device="cuda")).abs().max()) < 2e-5


@pytest.mark.parametrize("cond", [1e12, 1e16])
def test_stacks_of_low_numerical_rank_are_swept_again_with_replacement(mods, cond):
    """Singular values that fall through the whole fp32 range: what the first pass of a plain sweep leaves of the
    later columns is rounding noise that depends on the earlier columns again in the second pass, so it ends with
    columns that are not orthogonal, and Cholesky QR rounds on such a matrix diverge.  The state machine sweeps these
    matrices again with every dependent column replaced by a stand-in: orthonormal to rounding, the leading columns
    span what Householder's span, nothing goes to the library routine."""
    import numpy as np
    import qtensor.fused as X
    n, batch = 256, 16
    g = torch.Generator().manual_seed(n + int(np.log10(cond)))
    U, _ = torch.linalg.qr(torch.randn(batch, n, n, generator=g, dtype=torch.float64))
    V, _ = torch.linalg.qr(torch.randn(batch, n, n, generator=g, dtype=torch.float64))
    lam = torch.logspace(0, -float(np.log10(cond)), n, dtype=torch.float64)
    Y = ((U * lam) @ V.transpose(1, 2)).float()
    Y = (Y / torch.linalg.vector_norm(Y, dim=1, keepdim=True)).cuda().contiguous()
    eye = torch.eye(n, device="cuda")
    plain = Y.clone()
    info = torch.zeros(batch, dtype=torch.int32, device="cuda")
    X.block_gram_schmidt(plain, info)
    far = (plain.transpose(1, 2) @ plain - eye).abs().amax(dim=(1, 2)) > 0.3
    assert int(far.sum()) >= batch // 2 and bool((info != 0).all())         # the case this test is about
    state = X.CholeskyQR(Y)
    while not state.finished:
        state.check()
        if not state.poll():
            state.advance()
    Q, redone = state.result()
    assert redone == 0 and state.repairs >= int(far.sum()) and state.rounds <= 3
    assert float((Q.transpose(1, 2) @ Q - eye).abs().max()) < 5e-5
    Qh, _ = torch.linalg.qr(Y.double().cpu())
    k = n // 8                                                               # singular values down to cond^(-1/8)
    lead = Q[:, :, :k].double().cpu()
    resid = Qh[:, :, :k] - lead @ (lead.transpose(1, 2) @ Qh[:, :, :k])
    assert float(resid.norm(dim=1).max()) < 2e-5
    # the replacing sweep on its own: three passes, stand-ins flagged; what it leaves far (a stand-in for one of the
    # last columns with next to nothing of it outside the span of the others) is few and within reach of a round
    again = Y.clone()
    info.zero_()
    X.block_gram_schmidt(again, info, replace_dependent=True)
    assert bool(((info & 4) != 0).all()) and bool(((info & 1) == 0).all())
    still = (again.transpose(1, 2) @ again - eye).abs().amax(dim=(1, 2)) > 0.3
    assert int(still.sum()) <= batch // 4 and int(still.sum()) < int(far.sum())
    with pytest.raises(ValueError):
        X.block_gram_schmidt(again, info, complete=False, replace_dependent=True)
    # a caller that knows the stack goes to the replacing sweep directly: same outcome, no second sweep
    direct = X.CholeskyQR(Y, replace_first=True)
    while not direct.finished:
        direct.check()
        if not direct.poll():
            direct.advance()
    Qd, redone = direct.result()
    assert redone == 0 and direct.repairs == 0 and direct.rounds <= 3
    assert float((Qd.transpose(1, 2) @ Qd - eye).abs().max()) < 5e-5
    lead = Qd[:, :, :k].double().cpu()
    resid = Qh[:, :, :k] - lead @ (lead.transpose(1, 2) @ Qh[:, :, :k])
    assert float(resid.norm(dim=1).max()) < 2e-5


def test_low_rank_gradients_do_not_reach_the_library_qr(mods, tmp_path, monkeypatch):
    """Gradients of rank two plus a little noise (a small batch): every statistic has a few large directions and a
    floor, the regime in which the plain sweep is not enough.  The bank must get through on its own kernels."""
    monkeypatch.chdir(tmp_path)
    S2, E2 = mods
    from optimizers.shampoo_common import build_code_maps
    import qtensor.fused as X
    g = torch.Generator(device="cuda").manual_seed(5)
    params = [torch.zeros(512, 384, device="cuda"), torch.zeros(256, 640, device="cuda")]
    bank = E2.ShampooBank2(params, build_code_maps(4), "linear-2", inv_root_mode=1, **KW)
    for _ in range(6):
        grads = []
        for p in params:
            a = torch.randn(p.shape[0], 2, device="cuda", generator=g)
            b = torch.randn(2, p.shape[1], device="cuda", generator=g)
            grads.append(0.02 * (a @ b) + 1e-4 * torch.randn(p.shape, device="cuda", generator=g))
        bank.add_statistics(grads)
    assert bank.qr_fallbacks == 0
    for order in bank.per_order:
        vt = X.dequantize_stack(bank.basis[order])
        gram = vt @ vt.transpose(1, 2)
        assert bool(torch.isfinite(vt).all())
        # rows of a 4-bit basis are orthonormal up to the quantization error
        assert float((gram - torch.eye(order, device="cuda")).abs().max()) < 0.35
    bank.compute_preconditioners()
    out = bank.preconditioned_grads(grads)
    assert all(bool(torch.isfinite(o).all()) for o in out)
    print("matrices swept again:", bank.qr_repairs, "rounds:", bank.qr_rounds)
    # A stack that needed the replacing sweep for most of its matrices starts there for the next updates and looks
    # again after LOOK_AGAIN of them; with gradients of full rank the plain sweep is then enough and stays.
    order = max(bank.per_order, key=bank.per_order.get)
    bank.low_rank[order] = [True, 0]
    fallbacks = bank.qr_fallbacks
    for i in range(bank.LOOK_AGAIN):
        full = [0.02 * torch.randn(p.shape, device="cuda", generator=g) for p in params]
        bank.add_statistics(full)
        assert bank.low_rank[order] == ([True, i + 1] if i + 1 < bank.LOOK_AGAIN else [False, 0])
    assert bank.qr_fallbacks == fallbacks
    vt = X.dequantize_stack(bank.basis[order])
    assert float((vt @ vt.transpose(1, 2) - torch.eye(order, device="cuda")).abs().max()) < 0.35


def test_pivot_floor_takes_a_dependent_column_out_of_the_factorisation(mods):
    import qtensor.fused as X
    g = torch.Generator().manual_seed(23)
    n = 128
    A = torch.randn(n, n, generator=g, dtype=torch.float64)
    A[:, 70] = A[:, :70] @ torch.randn(70, generator=g, dtype=torch.float64)           # column 70 depends on the ones before
    A = A / A.norm(dim=0, keepdim=True)
    G = (A.T @ A).float().cuda().unsqueeze(0).contiguous()
    U, inv = torch.zeros(1, n, n, device="cuda"), torch.zeros(1, n, n, device="cuda")
    info = torch.zeros(1, dtype=torch.int32, device="cuda")
    X.cholesky_upper(G.clone(), U, inv, info, pivot_floor=2e-4)
    assert info.item() == 2
    Ut = torch.triu(U[0]).cpu()
    assert abs(float(Ut[70, 70]) - 2e-4 ** 0.5) < 1e-6 and float(Ut[70, 71:].abs().max()) == 0.0
    keep = [j for j in range(n) if j != 70]
    want = torch.linalg.cholesky((A[:, keep].T @ A[:, keep]), upper=True)              # the factor without that column
    assert rel(Ut[keep][:, keep], want) <= 1e-4
    info.zero_()
    X.cholesky_upper(G.clone(), U, inv, info)                                          # no floor: flagged as failed (or barely positive)
    assert info.item() in (0, 1)


def run_both(S2, E2, code_maps, mode, same_qr, monkeypatch, steps=3):
    import qtensor.utils as U
    if not same_qr:                      # the per-parameter path with the vendor's Householder QR, as in the reference
        def householder(Y):              # (fenced: this build's batched linalg calls are not reliably stream-ordered)
            torch.cuda.synchronize()
            Q = torch.linalg.qr(Y)[0]
            torch.cuda.synchronize()
            return Q
        monkeypatch.setattr(U, "_orthonormal_basis", householder)
    g = torch.Generator().manual_seed(21)
    grads = [[0.02 * torch.randn(s, generator=g).cuda() for s in SHAPES] for _ in range(steps)]
    qmap = {"linear-2": torch.from_numpy(code_maps[("linear-2", 4)])}
    params = [torch.zeros(s, device="cuda") for s in SHAPES]
    pres = [S2.Preconditioner(p, qmap, inv_root_mode=mode, **KW) for p in params]
    bank = E2.ShampooBank2(params, qmap, "linear-2", inv_root_mode=mode, **KW)
    for st in range(steps):
        if same_qr and st:
            # 4-bit re-encoding is a discontinuous map, so two flows that differ by rounding drift apart
            # at the quantization-noise level within a few updates: every update is therefore compared
            # from the same stored state (the bank's)
            for (pi, j, side, order, row) in bank.block_table():
                h = pres[pi].statistics[2 * j + side]
                h.var.copy_(bank.basis[order].codes[row])
                h.absmax.copy_(bank.basis[order].absmax[row])
                h.Svalue, h.keep_indices = bank.svalue[order][row].clone(), bank.keep[order][row].clone()
                h.max_eigenvalue = bank.max_eig[order][row].clone()
        for pre, gr in zip(pres, grads[st]):
            pre.add_statistics(gr)
        bank.add_statistics([gr.contiguous() for gr in grads[st]])
    starts = {}
    for (pi, j, side, order, row) in bank.block_table():
        starts.setdefault(order, {})[row] = (pi, j, side)
    gen = torch.Generator().manual_seed(5)
    v0 = {o: torch.rand(len(rows), o, generator=gen).cuda() * 2 - 1 for o, rows in starts.items()}
    for pi, pre in enumerate(pres):
        per = [None] * len(pre.statistics)
        for (qi, j, side, order, row) in bank.block_table():
            if qi == pi:
                per[2 * j + side] = v0[order][row]
        pre.compute_preconditioners(v0=per)
    bank.compute_preconditioners(v0=v0)
    outs_ref = [pre.preconditioned_grad(gr) for pre, gr in zip(pres, grads[-1])]
    outs = bank.preconditioned_grads([gr.contiguous() for gr in grads[-1]])
    return pres, bank, outs_ref, outs


@pytest.mark.parametrize("mode", [0, 1])
def test_bank_equals_per_parameter_flow_with_the_same_orthonormalisation(mods, code_maps, mode, monkeypatch, tmp_path):
    S2, E2 = mods
    import qtensor.fused as X
    monkeypatch.chdir(tmp_path)
    pres, bank, outs_ref, outs = run_both(S2, E2, code_maps, mode, True, monkeypatch)
    assert bank.qr_fallbacks == 0
    checked_codes = 0
    for (pi, j, side, order, row) in bank.block_table():
        h = pres[pi].statistics[2 * j + side]
        assert h.bits == 4
        # a statistic with a null space (a 128 x 64 gradient block gives a rank-64 term, and only half of
        # the quotients are kept) has basis vectors fixed by rounding noise alone: codes are compared
        # where the statistic is regular, everything derived from it everywhere
        regular = float(bank.svalue[order][row].min()) > 1e-3 * float(bank.max_eig[order][row])
        if regular:
            # the leading basis vectors are well determined (the trailing ones to rounding / pivot
            # only: a square Gaussian block has a condition number around its order squared)
            lead = slice(0, order // 4)
            mine = X.dequantize_stack(bank.basis[order])[row][lead]
            assert rel(mine, h._basis()[lead]) <= 0.05, (pi, j, side)
            checked_codes += 1
        top = float(h.max_eigenvalue)
        # (the noise-determined vectors are stored in 4 bits too, so a null space costs about one
        # re-encoding of accuracy in everything that follows)
        assert rel(bank.max_eig[order][row], h.max_eigenvalue) <= (1e-4 if regular else 2e-2)
        assert float((bank.svalue[order][row] - h.Svalue).abs().max()) <= (1e-4 if regular else 2e-2) * top
        want = h.dequantize()[0]
        got = bank._statistic(order, bank._rectified_basis(order))[row]
        assert float((got - want).norm()) <= (2e-2 if regular else 1e-1) * max(float(want.norm()), top)
    assert checked_codes >= 2
    # where a statistic has a null space the inverse root weighs rounding-noise directions by
    # (tiny quotient)^(-1/4): those blocks are not comparable, here or in the reference
    pairs = [(outs[0][:, :128], outs_ref[0][:, :128])] + list(zip(outs[1:], outs_ref[1:]))
    print("preconditioned gradients", [rel(a, b) for a, b in pairs])
    for a, b in pairs:
        assert rel(a.reshape(b.shape), b) <= 0.05


@pytest.mark.parametrize("mode", [0, 1])
def test_bank_against_unmodified_per_parameter_path(mods, code_maps, mode, monkeypatch, tmp_path):
    """One update from the common start (identity basis) against the per-parameter path with the
    vendor's Householder QR: the two Q differ in column signs, the stored 4-bit bases therefore in a
    few codes (the table is not symmetric around zero), everything derived from them by about one
    re-encoding."""
    S2, E2 = mods
    monkeypatch.chdir(tmp_path)
    pres, bank, outs_ref, outs = run_both(S2, E2, code_maps, mode, False, monkeypatch, steps=1)
    for (pi, j, side, order, row) in bank.block_table():
        h = pres[pi].statistics[2 * j + side]
        top = float(h.max_eigenvalue)
        assert rel(bank.max_eig[order][row], h.max_eigenvalue) <= 1e-3
        assert float((bank.svalue[order][row] - h.Svalue).abs().max()) <= 1e-3 * top
        want = h.dequantize()[0]
        got = bank._statistic(order, bank._rectified_basis(order))[row]
        assert float((got - want).norm()) <= 0.1 * max(float(want.norm()), top)


def test_steps_issued_from_another_stream_give_the_same_parameters(mods, tmp_path, monkeypatch):
    """The engines run on side streams of their own and join the stream that is current when step() is called:
    steps issued from a stream of the application, next to other streams of the application that are busy, end in
    the same bits as steps issued from the default stream."""
    S2, _ = mods
    import optimizers.matrix_functions as MF
    monkeypatch.chdir(tmp_path)
    real_rand = torch.rand
    monkeypatch.setattr(MF.torch, "rand", lambda *size, **kw: torch.full(size, 0.75, **kw))
    g = torch.Generator().manual_seed(12)
    shapes = SHAPES + [(64,), (128, 100)]
    init = [real_rand(s, generator=g) for s in shapes]
    gs = [[0.02 * torch.randn(s, generator=g) for s in shapes] for _ in range(4)]

    def run(stream):
        params = [torch.nn.Parameter(t.clone().cuda()) for t in init]
        opt = S2.ShampooAdamW(params, lr=1e-2, weight_decay=0.05, start_prec_step=2, stat_compute_steps=1, prec_compute_steps=2,
                              fused=True, inv_root_mode=1, **KW)
        grads = [[gr.cuda() for gr in step] for step in gs]
        torch.cuda.synchronize()
        busy = [torch.cuda.Stream() for _ in range(3)]
        noise = torch.zeros(1 << 20, device="cuda")
        with torch.cuda.stream(stream) if stream is not None else torch.cuda.stream(torch.cuda.current_stream()):
            for step in grads:
                for other in busy:                                   # the application keeps its own streams busy
                    with torch.cuda.stream(other):
                        noise.add_(1.0)
                for p_, gr in zip(params, step):
                    p_.grad = gr.clone()
                opt.step()
        torch.cuda.synchronize()
        return [p_.detach().clone() for p_ in params]

    plain = run(None)
    other = run(torch.cuda.Stream())
    assert all(bool(torch.isfinite(p_).all()) for p_ in plain)
    for a, b in zip(plain, other):
        assert torch.equal(a, b)


@pytest.mark.parametrize("which,mode", [("adamw", 1), ("sgd", 0)])
def test_fused_shampoo2_optimizer_runs_and_resumes_from_a_checkpoint(mods, which, mode, tmp_path, monkeypatch):
    import io
    S2, _ = mods
    import optimizers.matrix_functions as MF
    monkeypatch.chdir(tmp_path)
    real_rand = torch.rand
    monkeypatch.setattr(MF.torch, "rand", lambda *size, **kw: torch.full(size, 0.75, **kw))
    g = torch.Generator().manual_seed(8)
    shapes = SHAPES + [(64,), (128, 100), (96, 40)]        # a vector, an order the blocksize does not divide, one kept in fp32
    init = [real_rand(s, generator=g) for s in shapes]
    gs = [[0.02 * torch.randn(s, generator=g) for s in shapes] for _ in range(5)]

    def make(params):
        common = dict(start_prec_step=2, stat_compute_steps=1, prec_compute_steps=2, fused=True, inv_root_mode=mode, **KW)
        return (S2.ShampooAdamW(params, lr=1e-2, weight_decay=0.05, **common) if which == "adamw"
                else S2.ShampooSGD(params, lr=1e-2, momentum=0.9, **common))

    def run(opt, params, steps):
        for st in steps:
            for p, gr in zip(params, gs[st]):
                p.grad = gr.clone().cuda()
            opt.step()

    straight = [torch.nn.Parameter(t.clone().cuda()) for t in init]
    run(make(straight), straight, range(5))
    assert all(bool(torch.isfinite(p).all()) for p in straight)
    assert all(not torch.equal(p.detach().cpu(), t) for p, t in zip(straight, init))

    first = [torch.nn.Parameter(t.clone().cuda()) for t in init]
    opt = make(first)
    run(opt, first, range(3))
    sd = opt.state_dict()
    bank = sd["shampoo_bank"]
    assert any(k.startswith("basis.128.") for k in bank[0]) and any(k.startswith("basis.100.") for k in bank[0])
    assert all(opt.state[p]["step"] == 3 for p in first)
    assert not any("preconditioner" in opt.state[p] for p in first if p.dim() > 1)      # every matrix lives in the bank
    buf = io.BytesIO()
    torch.save(sd, buf)                                   # the WHOLE state: nothing in it is a pickled object
    buf.seek(0)
    sd = torch.load(buf, weights_only=True, map_location="cpu")
    resumed = [torch.nn.Parameter(p.detach().clone()) for p in first]
    opt2 = make(resumed)
    opt2.load_state_dict(sd)
    run(opt2, resumed, range(3, 5))
    for a, b in zip(straight, resumed):
        assert torch.equal(a.detach(), b.detach())


@pytest.mark.parametrize("mode", [0, 1])
def test_fused_shampoo2_step_skips_and_counts_per_parameter_like_the_reference(mods, mode, tmp_path, monkeypatch):
    """A parameter without a gradient is skipped and every parameter counts its own steps (reference:
    optimizers/shampoo2.py:415, 335-342): the fused step with gradients missing on some steps against the
    per-parameter optimizer on the same gradients.  The gradients are well conditioned, so that the two paths'
    re-encoded bases differ in few codes (see test_gpu_shampoo2_oracle.py) and the parameters stay comparable."""
    S2, _ = mods
    import optimizers.matrix_functions as MF
    from test_gpu_shampoo2_oracle import conditioned
    monkeypatch.chdir(tmp_path)
    shapes = [(128, 128), (256, 128), (128, 256), (64,)]
    g = torch.Generator().manual_seed(21)
    init = [torch.rand(s, generator=g) for s in shapes]
    gs = [[conditioned(s, 128, g) if len(s) == 2 else 0.02 * torch.randn(s, generator=g) for s in shapes] for _ in range(6)]
    monkeypatch.setattr(MF.torch, "rand", lambda *size, **kw: torch.full(size, 0.75, **kw))
    present = [[st not in (2, 3), st >= 1, True, st != 4] for st in range(6)]
    finals, counts = [], []
    for fused in (False, True):
        params = [torch.nn.Parameter(t.clone().cuda()) for t in init]
        opt = S2.ShampooSGD(params, lr=1e-2, momentum=0.9, start_prec_step=2, stat_compute_steps=1, prec_compute_steps=2,
                            fused=fused, inv_root_mode=mode, **KW)
        for st in range(6):
            for p, gr, there in zip(params, gs[st], present[st]):
                p.grad = gr.clone().cuda() if there else None
            opt.step()
        finals.append([p.detach().cpu() for p in params])
        counts.append([opt.state[p]["step"] for p in params])
    assert counts[0] == counts[1] == [sum(row[k] for row in present) for k in range(len(shapes))]
    worst = max(rel(a, b) for a, b in zip(*finals))
    print("fused against per-parameter step with gradients missing, mode", mode, ":", worst)
    assert worst <= 2e-3


def test_roots_applied_next_to_the_factorisations_change_nothing(mods, tmp_path, monkeypatch):
    """On steps that keep the inverse roots the bank applies them to the gradients on a thread and stream of its own
    while the statistics update factorises; parameters and stored bases must be bit-identical to the run in line."""
    S2, _ = mods
    import optimizers.matrix_functions as MF
    monkeypatch.chdir(tmp_path)
    real_rand = torch.rand
    monkeypatch.setattr(MF.torch, "rand", lambda *size, **kw: torch.full(size, 0.75, **kw))
    g = torch.Generator().manual_seed(12)
    init = [real_rand(s, generator=g) for s in SHAPES]
    gs = [[0.02 * torch.randn(s, generator=g) for s in SHAPES] for _ in range(7)]
    overlapped = []

    def run(overlap):
        monkeypatch.setattr(S2.ShampooAdamW, "overlap_precondition", overlap)
        params = [torch.nn.Parameter(x.clone().cuda()) for x in init]
        opt = S2.ShampooAdamW(params, lr=1e-2, weight_decay=0.05, start_prec_step=2, stat_compute_steps=1,
                              prec_compute_steps=3, fused=True, inv_root_mode=1, **KW)
        bank = None
        for grads in gs:
            for p, gr in zip(params, grads):
                p.grad = gr.clone().cuda()
            if bank is not None and overlap and not hasattr(bank, "wrapped"):
                real, bank.wrapped = bank.preconditioned_grads, True
                monkeypatch.setattr(bank, "preconditioned_grads",
                                    lambda gr, inline=False, real=real, **kw: (overlapped.append(inline), real(gr, inline=inline, **kw))[1])
            opt.step()
            bank = next(iter(opt._fused_cache.values()))["bank"]
        torch.cuda.synchronize()
        return [p.detach().cpu() for p in params], [t.cpu() for t in bank.state_dict().values() if torch.is_tensor(t)]

    beside, inline = run(True), run(False)
    assert overlapped.count(True) >= 3                      # steps 4, 5 and 7 keep their roots
    for a, b in zip(beside[0] + beside[1], inline[0] + inline[1]):
        assert torch.equal(a, b)


@pytest.mark.parametrize("variant,fused", [("shampoo1", True), ("shampoo1", False), ("shampoo2", True)])
def test_optimizers_reduce_a_small_regression_loss(variant, fused, tmp_path, monkeypatch):
    """End-to-end sanity: a two-layer network fitted to a random teacher with 4-bit Shampoo + AdamW."""
    import importlib
    monkeypatch.chdir(tmp_path)
    S = importlib.import_module("optimizers." + variant)
    torch.manual_seed(0)
    dev = "cuda"
    X_ = torch.randn(512, 128, device=dev)
    teacher = torch.randn(128, 64, device=dev) / 128 ** 0.5
    Y = torch.tanh(X_ @ teacher)
    model = torch.nn.Sequential(torch.nn.Linear(128, 128), torch.nn.Tanh(), torch.nn.Linear(128, 64)).to(dev)
    opt = S.ShampooAdamW(model.parameters(), lr=3e-3, weight_decay=0.0, start_prec_step=5, stat_compute_steps=1,
                         prec_compute_steps=5, prec_bits=4, prec_maxorder=128, quan_blocksize=64, min_lowbit_size=4096,
                         fused=fused)
    losses = []
    for _ in range(60):
        opt.zero_grad(set_to_none=True)
        loss = torch.nn.functional.mse_loss(model(X_), Y)
        loss.backward()
        opt.step()
        losses.append(float(loss.detach()))
    # (shampoo2 with inv_root_mode=0 preconditions with the kept half of the eigenpairs only: slower progress)
    bound = 0.3 if variant == "shampoo1" else 0.6
    assert all(l == l for l in losses) and losses[-1] < bound * losses[0], (losses[0], losses[-1])


@pytest.mark.parametrize("n,batch", [(64, 3), (320, 4), (1024, 2)])
def test_column_dots_is_the_diagonal_of_the_product(mods, n, batch):
    import qtensor.fused as X
    g = torch.Generator().manual_seed(n)
    A, B = torch.randn(batch, n, n, generator=g), torch.randn(batch, n, n, generator=g)
    got = X.column_dots(A.cuda(), B.cuda())
    want = (A.double() * B.double()).sum(dim=1)
    scale = (A.double().abs() * B.double().abs()).sum(dim=1)
    assert got.shape == (batch, n)
    assert float(((got.cpu().double() - want).abs() / scale).max()) <= 1e-6
    assert torch.equal(got, X.column_dots(A.cuda(), B.cuda()))                 # fixed summation order
    with pytest.raises(ValueError):
        X.column_dots(A.cuda(), B[:, :, :32].contiguous().cuda())


def test_a_clean_sweep_means_an_orthonormal_result(mods):
    """CholeskyQR takes a swept matrix whose flags are all clear as final without testing it.  That rests on the sweep:
    whenever it reports nothing (no pivot at the floor, no column replaced, no NaN) the result must be orthonormal to
    fp32 rounding -- checked here over well and ill conditioned matrices, graded column scales, numerically dependent
    columns and low rank, where the sweep has to raise a flag for whatever it cannot finish."""
    _, E2 = mods
    import qtensor.fused as X
    g = torch.Generator().manual_seed(99)
    n = 256
    mats, kinds = [], []
    for cond in (0.0, 2.0, 4.0, 6.0, 8.0):                                      # singular values 1 .. 10^-cond
        u, _ = torch.linalg.qr(torch.randn(n, n, generator=g, dtype=torch.float64))
        v, _ = torch.linalg.qr(torch.randn(n, n, generator=g, dtype=torch.float64))
        mats.append(((u * torch.logspace(0, -cond, n, dtype=torch.float64)) @ v.T).float())
        kinds.append("cond 1e%d" % cond)
    graded = torch.randn(n, n, generator=g) * torch.logspace(0, -12, n)             # column scales over twelve decades
    mats.append(graded); kinds.append("graded columns")
    twin = torch.randn(n, n, generator=g)
    twin[:, 100] = twin[:, 7] * (1 + 1e-7) + 1e-9 * torch.randn(n, generator=g)     # a column that repeats an earlier one
    mats.append(twin); kinds.append("repeated column")
    for rank in (n // 2, 8):
        low = torch.randn(n, rank, generator=g) @ torch.randn(rank, n, generator=g)
        mats.append(low + 1e-7 * torch.randn(n, n, generator=g)); kinds.append("rank %d plus noise" % rank)
        mats.append(low); kinds.append("rank %d exactly" % rank)
    Y = torch.stack(mats).cuda()
    Q = (Y / torch.linalg.vector_norm(Y, dim=1, keepdim=True).clamp_min(1e-30)).contiguous()
    info = torch.zeros(len(mats), dtype=torch.int32, device="cuda")
    X.block_gram_schmidt(Q, info)
    gram = Q.double().transpose(1, 2) @ Q.double()
    off = (gram - torch.eye(n, dtype=torch.float64, device="cuda")).abs().amax(dim=(1, 2)).cpu()
    flags = info.cpu().tolist()
    for kind, flag, worst in zip(kinds, flags, off.tolist()):
        print("%-22s flags %d  max |Q^T Q - I| %.2e" % (kind, flag, worst))
        if flag == 0:
            assert worst <= 2e-5, (kind, worst)
    assert flags[0] == 0 and flags[1] == 0                                         # the easy ones are clean
    assert all(f != 0 for f, k in zip(flags, kinds) if k.startswith("rank") or k == "repeated column")
    # and the whole solver ends orthonormal for every one of them
    final, redone = X.cholesky_qr(Y)
    gram = final.double().transpose(1, 2) @ final.double()
    assert float((gram - torch.eye(n, dtype=torch.float64, device="cuda")).abs().max()) <= 5e-5


def test_matrices_left_to_the_caller_are_neither_tested_nor_polished(mods):
    """CholeskyQR(leave=...): the matrices a caller orthonormalises some other way (the eigenbasis bank sweeps its few
    known low-rank matrices apart from their stack) cost the stack no test, no polishing round and no second sweep,
    and the other matrices come out with the same bits as without them."""
    _, E2 = mods
    import qtensor.fused as X
    g = torch.Generator().manual_seed(5)
    n = 256
    good = [torch.randn(n, n, generator=g) for _ in range(5)]
    low = torch.randn(n, 24, generator=g) @ torch.randn(24, n, generator=g)                # rank 24: the plain sweep cannot finish it
    Y = torch.stack(good[:2] + [low] + good[2:]).cuda()
    with_it = X.CholeskyQR(Y.clone())
    while not with_it.finished:
        with_it.check()
        if not with_it.poll():
            with_it.advance()
    q_all, _ = with_it.result()
    assert with_it.rounds + with_it.repairs >= 1                                            # the low-rank matrix cost extra work
    left = X.CholeskyQR(Y.clone(), leave=[2])
    left.check()
    assert left.finished and left.rounds == 0 and left.repairs == 0                         # nothing to test: the other sweeps are clean
    q_left, redone = left.result()
    keep = [0, 1, 3, 4, 5]
    assert redone == 0 and torch.equal(q_left[keep], q_all[keep])
    # and the matrix itself, as a stack of its own that starts with the replacing sweep, ends orthonormal
    own = X.CholeskyQR(Y[2:3].clone(), replace_first=True)
    while not own.finished:
        own.check()
        if not own.poll():
            own.advance()
    q_own, redone = own.result()
    gram = q_own[0].double().T @ q_own[0].double()
    assert redone == 0 and float((gram - torch.eye(n, dtype=torch.float64, device="cuda")).abs().max()) <= 5e-5
    # its leading columns span what the matrix's leading columns span
    lead = Y[2, :, :16].double()
    proj = q_own[0, :, :16].double() @ (q_own[0, :, :16].double().T @ lead)
    assert float((proj - lead).norm() / lead.norm()) <= 1e-4


@pytest.mark.parametrize("n", [100, 200, 832])
def test_stand_in_columns_of_a_padded_order_stay_inside_the_matrix(mods, n):
    """Orders that are not a multiple of 64 are factored as diag(Y, I).  A stand-in column for a dependent column of Y
    must have nothing in the padding rows, or the leading n x n block that is handed back is not orthonormal (a
    stand-in in general position of the padded space loses n / n_padded of its length there)."""
    _, E2 = mods
    import qtensor.fused as X
    g = torch.Generator().manual_seed(n)
    dep = torch.randn(2, n, n, generator=g)
    dep[:, :, n // 2] = dep[:, :, 1] * 2.0                                     # one column repeats an earlier one
    low = torch.randn(2, n, n // 4, generator=g) @ torch.randn(2, n // 4, n, generator=g)   # and a stack of rank n / 4
    for Y in (dep.cuda(), low.cuda()):
        Q, redone = X.cholesky_qr(Y)
        gram = Q.double().transpose(1, 2) @ Q.double()
        assert float((gram - torch.eye(n, dtype=torch.float64, device="cuda")).abs().max()) <= 5e-5
        k = n // 8                                                             # the leading columns still span what Y's span
        lead = Y[:, :, :k].double()
        proj = Q[:, :, :k].double() @ (Q[:, :, :k].double().transpose(1, 2) @ lead)
        assert float((proj - lead).norm() / lead.norm()) <= 1e-4


def test_a_dependent_column_next_to_an_ill_conditioned_panel_is_flagged(mods):
    """A column that depends on the 64 columns before it sits in the second 64-column panel of its 128-column outer
    panel.  In the first pass that first panel has had one Cholesky QR round only (orthonormal to rounding times its
    squared conditioning), so what the projection leaves of the column is far above rounding noise and nobody can
    tell that it is dependent; the last pass then finds next to nothing left of it, lifts that back to unit length,
    and the result is off by rounding over what was left.  The sweep must flag such a matrix (so that it is tested
    and polished): whatever it reports clean is orthonormal, and the solver's result always is."""
    _, E2 = mods
    import qtensor.fused as X
    g = torch.Generator().manual_seed(64)
    mats = []
    for n, r in ((65, 64), (65, 64), (128, 64), (100, 70), (130, 64)):
        for _ in range(6):
            mats.append((n, torch.randn(n, r, generator=g) @ torch.randn(r, n, generator=g)))
    flagged = 0
    for n, Y in mats:
        Y = Y.unsqueeze(0).cuda()
        s = X.CholeskyQR(Y)
        info = int(s.info.cpu()[0])
        swept = s.Q[0].double()
        off = float((swept.T @ swept - torch.eye(swept.shape[0], dtype=torch.float64, device="cuda")).abs().max())
        if info == 0:
            assert off <= 2e-5, (n, off)
        flagged += info != 0
        while not s.finished:
            s.check()
            if not s.poll():
                s.advance()
        Q, redone = s.result()
        gram = Q[0].double().T @ Q[0].double()
        assert float((gram - torch.eye(n, dtype=torch.float64, device="cuda")).abs().max()) <= 5e-5
    assert flagged >= len(mats) // 2                                        # these matrices are rank deficient: most must be flagged


@pytest.mark.parametrize("stack_bytes,lanes", [(256 << 20, 3), (1, 2), (4 * 96 * 96, 1)])
def test_statistics_taken_together_are_those_taken_one_by_one(monkeypatch, stack_bytes, lanes):
    """fused=False: the statistics of all parameters in stacks on a few streams, or parameter by parameter: quotients, maxima and
    parameters over five steps, every second of which takes statistics, with a parameter that has no gradient at times.  (Square
    gradients with singular values between 1/2 and 2: statistics whose eigenvectors rounding does not choose.)  A stack's products may be cut along k in another way than
    a single matrix's, which rounds sums of up to 130 fp32 products differently: 130 x 2^-24 = 8e-6 of a quotient, and where
    a maximum or a code sits on an edge the element moves a level, in few places."""
    from optimizers import shampoo2, shampoo_common
    monkeypatch.setattr(shampoo_common._ShampooOptimizer, "STACK_BYTES", stack_bytes)
    monkeypatch.setattr(shampoo_common._ShampooOptimizer, "LANES", lanes)
    shapes = [(96, 96), (128, 128), (64, 64), (100, 100), (130, 130), (45, 5, 3, 3), (17,), (96, 96)]
    gen = torch.Generator().manual_seed(5)
    start = [0.1 * torch.randn(s, generator=gen) for s in shapes]

    def gradient(shape):
        n = shape[0]
        if len(shape) == 1:
            return torch.randn(n, generator=gen)
        (u, _), (v, _) = [torch.linalg.qr(torch.randn(n, n, generator=gen)) for _ in range(2)]
        return ((u * torch.logspace(-1, 1, n, base=2.0)) @ v).reshape(shape)

    grads = [[gradient(s) for s in shapes] for _ in range(5)]
    made, taken = [], []
    together = shampoo_common._ShampooOptimizer._statistics_together
    for alone in (False, True):
        def spy(self, group):
            done = () if alone else together(self, group)
            taken.append(len(done))
            return done
        monkeypatch.setattr(shampoo_common._ShampooOptimizer, "_statistics_together", spy)
        params = [torch.nn.Parameter(t.cuda()) for t in start]
        opt = shampoo2.ShampooAdamW(params, lr=1e-2, start_prec_step=1, stat_compute_steps=2, prec_compute_steps=4, prec_maxorder=1200,
                                    prec_bits=4, quan_blocksize=64, min_lowbit_size=4096)
        for step, gs in enumerate(grads):
            for i, (p, g) in enumerate(zip(params, gs)):
                p.grad = None if (i == 2 and step in (1, 2)) or (i == 7 and step == 0) else g.cuda()
            opt.step()
        made.append((params, opt))
    # the first step finds no state; then parameters at an even count: (step, counts of parameters 2 and 7)
    assert taken[:5] == [0, 5, 1, 6, 1] and taken[5:] == [0] * 5
    for pa, pb in zip(made[0][0], made[1][0]):
        a, b = pa.detach(), pb.detach()
        stats = [opt.state[p]["preconditioner"].statistics for (_, opt), p in zip(made, (pa, pb))]
        for x, y in zip(*stats):
            assert float((x.Svalue - y.Svalue).norm() / y.Svalue.norm()) <= 1e-5 * 4
            assert torch.equal(x.keep_indices, y.keep_indices)
            if x.bits < 16:
                assert float((x.absmax - y.absmax).norm() / y.absmax.norm()) <= 1e-3
        assert float((a - b).abs().max()) <= 1e-4 * 5e-2                       # five steps of 1e-2


@pytest.mark.parametrize("stack_bytes", [256 << 20, 4 * 4 * 130 * 130])
def test_statistics_of_a_parameter_do_not_depend_on_its_neighbours(monkeypatch, stack_bytes):
    """fused=False: ten statistics of order 130 and three of order 288 and of low rank, for which the orthonormalisation has to decide (stand-in
    columns, another sweep), beside others of full rank: in stacks, whole or cut small, the bits of the state and of the
    parameters are those of the parameters taken one by one, also where neighbours have no gradient."""
    from optimizers import shampoo2, shampoo_common
    monkeypatch.setattr(shampoo_common._ShampooOptimizer, "STACK_BYTES", stack_bytes)
    shapes = [(130, 30)] * 10 + [(288, 72)] * 3 + [(130, 130), (64, 288), (200, 64)]
    gen = torch.Generator().manual_seed(7)
    start = [0.1 * torch.randn(s, generator=gen) for s in shapes]
    grads = [[torch.randn(s, generator=gen) for s in shapes] for _ in range(5)]
    together = shampoo_common._ShampooOptimizer._statistics_together
    made = []
    for alone in (False, True):
        monkeypatch.setattr(shampoo_common._ShampooOptimizer, "_statistics_together", (lambda self, group: ()) if alone else together)
        torch.manual_seed(3)                                                  # the roots' start vectors
        params = [torch.nn.Parameter(t.cuda()) for t in start]
        opt = shampoo2.ShampooAdamW(params, lr=1e-2, start_prec_step=1, stat_compute_steps=1, prec_compute_steps=2, prec_maxorder=1200,
                                    prec_bits=4, quan_blocksize=64, min_lowbit_size=4096)
        for step, gs in enumerate(grads):
            for i, (p, g) in enumerate(zip(params, gs)):
                p.grad = None if i in (0, 3, 4, 11)[:step] else g.cuda()
            opt.step()
        made.append((params, opt))
    for pa, pb in zip(made[0][0], made[1][0]):
        assert torch.equal(pa, pb)
        for x, y in zip(*[opt.state[p]["preconditioner"].statistics for (_, opt), p in zip(made, (pa, pb))]):
            for name in ("Svalue", "keep_indices", "max_eigenvalue", "var") + (("absmax",) if x.bits < 16 else ()):
                assert torch.equal(getattr(x, name), getattr(y, name)), (tuple(pa.shape), name)


def test_state_made_on_a_side_stream_outlives_what_the_callers_stream_reads():
    """fused=False: an optimizer that is let go while its stream still has work to do.  Its statistics were made on the shared
    side streams, and another optimizer's step must not be handed their memory there before that work is through."""
    import bisect
    import gc
    from optimizers import shampoo2
    from optimizers.engine import shared_stream
    device = torch.device("cuda", torch.cuda.current_device())
    gen = torch.Generator(device="cuda").manual_seed(11)
    params = [torch.nn.Parameter(torch.randn(96, 96, device="cuda", generator=gen)) for _ in range(6)]
    opt = shampoo2.ShampooSGD(params, lr=1e-3, start_prec_step=1, stat_compute_steps=1, prec_compute_steps=10 ** 6, prec_bits=4,
                              quan_blocksize=64, min_lowbit_size=4096)
    for _ in range(3):
        for p in params:
            p.grad = torch.randn(96, 96, device="cuda", generator=gen)
        opt.step()
    held = []
    for p in params:
        for holder in opt.state[p]["preconditioner"].statistics:
            held += [(t.data_ptr(), t.data_ptr() + t.numel() * t.element_size()) for t in
                     (holder.var, holder.absmax, holder.Svalue, holder.keep_indices, holder.max_eigenvalue)]
    del holder
    a = torch.randn(8192, 8192, device="cuda", generator=gen)
    b, done = torch.empty_like(a), torch.cuda.Event()
    torch.cuda.synchronize()
    for _ in range(100):
        torch.mm(a, a, out=b)
    done.record()
    del opt, params, p
    gc.collect()                                         # (an optimizer is in a cycle with its hooks)
    reused, made = 0, []
    for lane in range(3):
        with torch.cuda.stream(shared_stream(device, lane)):
            reserved = torch.cuda.memory_reserved()
            while torch.cuda.memory_reserved() == reserved:          # everything that the lane's pool has to give
                made += [torch.empty(512, dtype=torch.uint8, device="cuda") for _ in range(1000)]
    still_busy = not done.query()
    at = sorted(t.data_ptr() for t in made)
    for low, high in held:
        i = bisect.bisect_left(at, low - 511)
        reused += i < len(at) and at[i] < high
    assert still_busy and reused == 0


@pytest.mark.parametrize("what", ["accumulate", "add_statistics", "holder", "wrapped", "none"])
def test_an_own_way_of_taking_statistics_is_taken(what, monkeypatch):
    """fused=False: a preconditioner class with its own _accumulate or add_statistics, one with holders of its own, an object whose
    method has been wrapped: each is called for every statistic (two parameters of two sides, three steps); "none": the stacks are."""
    from optimizers import shampoo2
    from qtensor.utils import QTensorSVDFast
    calls = []

    class Holder(QTensorSVDFast):
        def quantize(self, var, Vt=None):
            calls.append("holder")
            super().quantize(var, Vt)

    class Prec(shampoo2.Preconditioner):
        if what == "accumulate":
            def _accumulate(self, *args):
                calls.append(what)
                super()._accumulate(*args)
        if what == "add_statistics":
            def add_statistics(self, grad):
                calls.extend([what] * 2)
                super().add_statistics(grad)
        if what == "holder":
            def _new_statistic(self, order, device, index, rank, quant_args, extra):
                return Holder(self.matrix_eps * torch.eye(order, device=device), rect_t1=extra["rect_t1"], rect_t2=extra["rect_t2"], **quant_args)

    class Optimizer(shampoo2.ShampooSGD):
        preconditioner_class = Prec

    params = [torch.nn.Parameter(torch.randn(96, 96, device="cuda")) for _ in range(2)]
    opt = Optimizer(params, lr=1e-3, start_prec_step=1, stat_compute_steps=1, prec_compute_steps=10 ** 6, prec_bits=4, quan_blocksize=64,
                    min_lowbit_size=4096)
    for step in range(3):
        for p in params:
            p.grad = torch.randn(96, 96, device="cuda")
        opt.step()
        if what == "wrapped" and step == 0:
            calls.extend([what] * 4)
            for p in params:
                prec = opt.state[p]["preconditioner"]
                plain = prec._accumulate
                prec._accumulate = lambda *args, plain=plain: (calls.append(what), plain(*args))
    assert calls == ([] if what == "none" else [what] * 12)
    taken = [s for p in params for s in [opt.state[p]["preconditioner"].statistics_in_stacks()]]
    assert taken == [what == "none"] * 2


@pytest.mark.parametrize("row", [-1, 96])
def test_a_checkpoint_with_rows_that_no_basis_has_is_refused(row):
    """Kept rows outside their basis: refused when the checkpoint is loaded, and nothing of it is taken."""
    from optimizers import shampoo2
    params = [torch.nn.Parameter(torch.randn(96, 64, device="cuda")) for _ in range(2)]
    opt = shampoo2.ShampooSGD(params, lr=1e-3, start_prec_step=1, stat_compute_steps=1, prec_compute_steps=1, prec_bits=4, quan_blocksize=64,
                              min_lowbit_size=4096, fused=True)
    for p in params:
        p.grad = torch.randn(96, 64, device="cuda")
    opt.step()
    saved = opt.state_dict()
    bank = {k: v.clone() if torch.is_tensor(v) else v for k, v in saved["shampoo_bank"][0].items()}
    held = {k: v.clone() for k, v in opt.state_dict()["shampoo_bank"][0].items() if torch.is_tensor(v)}
    bank["basis.96.keep"][1, 5] = row
    bank["basis.96.absmax"] += 1.0
    with pytest.raises(ValueError):
        opt.load_state_dict({**saved, "shampoo_bank": [bank]})
    assert all(torch.equal(v, held[k]) for k, v in opt.state_dict()["shampoo_bank"][0].items() if torch.is_tensor(v))
