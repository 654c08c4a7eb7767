"""Inverse p-th roots of PSD matrices by the coupled Newton iteration.

Same three entry points, argument meaning and return values as the reference's
optimizers/matrix_functions.py (PowerIter :21-48, MatPower :51-76, ComputePower :79-141); they
accept CPU or GPU tensors and then behave like the reference, sync for sync.

ComputePowerBatched is the MI355X form of ComputePower for a whole stack of equally sized
matrices: every product runs on the matrix cores through qtensor.fused.gemm (4 launches per
iteration for the whole stack), max|M - I| and M - I come out of the last product's epilogue, and
the per-matrix stopping rules are evaluated on the device, so the host never waits inside the
iteration.  Beside M it keeps E = M - I, and it multiplies deviations from the identity out:

    T = I + w E (w = -1/p),  R T = R + w R E,  F = T^2 - I = 2 w E + w^2 E E,  F <- 2 F + F F for
    every further squaring,  T^p M = M + F M

-- in exact arithmetic the reference's iteration.  Products of M and T themselves are products of
near-identities: one pair of elements makes most of every sum, and what its operands lose when
they are split, and the sum when it is rounded, is a part of the identity.  Relative error of the
root against the same iteration in float64 (4-bit statistics of condition 20, half pipe; the bf16
split for order 128): order 128 3.6e-7 -> 1.2e-7, 256 6.9e-7 -> 1.5e-7, 768 9.1e-7 -> 2.3e-7,
1024 1.1e-6 -> 2.8e-7; on the bf16 split the same but for 4 % (from 4.8e-7 at 256, 9.5e-7 at 1024).
"""
import ctypes as ct
from typing import Optional

import torch


@torch.no_grad()
def PowerIter(mat_g, error_tolerance=1e-6, num_iters=10, v0=None):
    """Largest eigenvalue of a symmetric PSD matrix by at most num_iters normalised
    matrix-vector products, starting from v0 (default: uniform in (-1, 1), drawn on mat_g's
    device from the global generator).  Stops once the Rayleigh quotient moves by no more than
    error_tolerance.  Returns (eigenvalue, unit vector, iterations used)."""
    n = mat_g.shape[0]
    v = torch.rand(n, device=mat_g.device) * 2 - 1 if v0 is None else v0.to(mat_g.device)
    change, used, value = 1, 0, 0
    while change > error_tolerance and used < num_iters:
        v = v / torch.norm(v)
        w = torch.mv(mat_g, v)
        quotient = torch.dot(v, w)
        change = torch.abs(quotient - value)
        v, value = w, quotient
        used += 1
    return value, v / torch.norm(v), used


@torch.no_grad()
def MatPower(mat_m, p):
    """mat_m ** p for a positive integer p: repeated squaring for powers of two up to 32,
    square-and-multiply otherwise."""
    if p in (1, 2, 4, 8, 16, 32):
        out, done = mat_m, 1
        while done < p:
            out = torch.matmul(out, out)
            done *= 2
        return out
    result, base = None, mat_m
    while p > 0:
        if p & 1:
            result = base if result is None else torch.matmul(base, result)
        p >>= 1
        base = torch.matmul(base, base)
    return result


@torch.no_grad()
def ComputePower(mat_g, p, iter_count=10, error_tolerance=1e-6, ridge_epsilon=1e-6, v0=None):
    """(mat_g + r I)^(-1/p), r = ridge_epsilon * (largest eigenvalue estimate), by the coupled
    Newton iteration of Guo & Higham (SIAM J. Matrix Anal. Appl. 28(3), 2006, eq. 3.2).

    A vector argument is treated as a diagonal: (mat_g + ridge_epsilon)^(-1/p) elementwise.
    A 1 x 1 matrix returns the identity.  Like the reference, the ridge is added to mat_g IN
    PLACE.  The iteration stops when max|M - I| <= error_tolerance, after iter_count rounds, or
    when that error grows by more than 20 % (the previous iterate is then returned)."""
    if mat_g.dim() == 1:
        return torch.pow(mat_g + ridge_epsilon, -1 / p)
    n = mat_g.shape[0]
    eye = torch.eye(n, device=mat_g.device)
    if n == 1:
        return eye
    w = -1.0 / p
    top, _, _ = PowerIter(mat_g, v0=v0)
    mat_g += (ridge_epsilon * top) * eye
    z = (1 + p) / (2 * torch.norm(mat_g))
    root = eye * torch.pow(z, 1.0 / p)
    m = mat_g * z
    err = torch.max(torch.abs(m - eye))
    rounds = 0
    while err > error_tolerance and rounds < iter_count:
        t = (1 - w) * eye + w * m
        candidate = torch.matmul(root, t)
        m = torch.matmul(MatPower(t, p), m)
        new_err = torch.max(torch.abs(m - eye))
        if new_err > err * 1.2:
            break
        root, err = candidate, new_err
        rounds += 1
    return root


_LAST_ROUNDS = {}                                  # order -> int32 [B], for diagnostics


@torch.no_grad()
def PowerIterBatched(mats, error_tolerance=1e-6, num_iters=10, v0=None):
    """PowerIter for a stack [B, n, n]; every matrix follows its own stopping rule (entries that
    have converged are frozen).  v0: optional [B, n] or [n] start vectors.  Returns the [B]
    eigenvalue estimates.  No host synchronisation.
    Sums are taken in float64 and rounded, so that they do not depend on the number of matrices."""
    from qtensor import fused as X
    B, n, _ = mats.shape
    if v0 is None:
        v = torch.rand(B, n, device=mats.device) * 2 - 1
    else:
        v = v0.to(mats.device).expand(B, n).clone()
        if v.dtype in (torch.bfloat16, torch.float16):
            v = v.float()
    if X.on_matrix_cores(mats) and mats.is_contiguous():            # the library's kernels: two launches a round
        return X.power_iteration(mats, v.contiguous(), error_tolerance, num_iters)
    value = torch.zeros(B, device=mats.device)
    change = torch.ones(B, device=mats.device)
    for _ in range(num_iters):
        active = change > error_tolerance
        u = v / torch.linalg.vector_norm(v, dim=1, keepdim=True, dtype=torch.float64).float()
        w = torch.bmm(mats, u.unsqueeze(2)).squeeze(2)
        quotient = (u * w).sum(dim=1, dtype=torch.float64).float()
        change = torch.where(active, (quotient - value).abs(), change)
        value = torch.where(active, quotient, value)
        v = torch.where(active.unsqueeze(1), w, v)
    return value


@torch.no_grad()
def ComputePowerBatched(mats, p=4, iter_count=10, error_tolerance=1e-6, ridge_epsilon=1e-6, v0=None,
                        out: Optional[torch.Tensor] = None, symmetric: bool = False, stack: Optional[int] = None):
    """ComputePower for a GPU stack mats [B, n, n] (fp32, overwritten with mats + ridge like the
    reference does for its argument).  Returns [B, n, n].

    symmetric: the caller guarantees mats[b] == mats[b].T bit for bit.  All iterates are then
    symmetric in exact arithmetic and only their upper halves are multiplied out (half the work).
    A dequantized low-bit statistic is NOT symmetric (every row segment has its own scale), and
    the reference iterates on it as it is: leave the flag off for those.

    stack: of how many matrices mats is a part (default: all).  Which matrix pipe multiplies is decided for the whole stack,
    so that the bits of a root do not depend on the part that its matrix is in."""
    from qtensor import fused as X

    if not mats.is_cuda or mats.dtype != torch.float32 or mats.dim() != 3:
        raise ValueError("ComputePowerBatched takes an fp32 GPU stack [B, n, n]")
    if p not in (1, 2, 4, 8, 16, 32):
        raise ValueError("ComputePowerBatched supports p in 1, 2, 4, ..., 32")
    B, n, _ = mats.shape
    dev = mats.device
    if n == 1:
        res = torch.ones(B, 1, 1, device=dev)
        return res if out is None else out.copy_(res)
    w = -1.0 / p
    work = mats if mats.is_contiguous() else mats.contiguous()
    top = PowerIterBatched(work, v0=v0)
    R, M, E, F = [[torch.empty(B, n, n, device=dev) for _ in range(2)] for _ in range(4)]     # F: T^2 - I, T^4 - I, ... in turn
    # How large the iterates' elements are, for the pipe that wants to know: the bounds of E and M follow from err = max |E|,
    # the rest is looked at by the launches that write them (both of E and M by one).
    measured = X.worth_measuring_for((B if stack is None else stack) * n ** 3, n)
    squarings = p.bit_length() - 1
    # errors before the first round and after each; what the rounds' products find (root, powers, E with M)
    zeros = torch.zeros((iter_count + 2) * B + (2 * iter_count * (2 + squarings) * B if measured else 0), device=dev)
    errors, first_fine = zeros[:(iter_count + 1) * B].view(-1, B), zeros[(iter_count + 1) * B:(iter_count + 2) * B]
    found = zeros[(iter_count + 2) * B:].view(iter_count, 2 + squarings, 2, B) if measured else None
    floats = torch.empty(5, B, device=dev)
    first_root, err, top_m, root_bound, root_fine = floats
    flags = torch.empty(3, B, dtype=torch.int32, device=dev)
    done, side, rounds = flags
    tables = torch.empty(6, B, dtype=torch.int64, device=dev)
    X.newton_first(work, top, ridge_epsilon, p, M[0], E[0], R[1], first_root, errors[0], first_fine if measured else None)
    if work is not mats:
        mats.copy_(work)
    err.copy_(errors[0])
    state = X.NewtonState(B, iter_count, error_tolerance, w, err.data_ptr(), done.data_ptr(), side.data_ptr(), rounds.data_ptr(),
                          first_root.data_ptr(), first_fine.data_ptr(), root_bound.data_ptr() if measured else None,
                          root_fine.data_ptr(), tables.data_ptr(),
                          (ct.c_longlong * 6)(*[t.data_ptr() for pair in (R, M, E) for t in pair]), 4 * n * n)

    def decide(new_err):
        X.F._call(X.F.lib.qtensor_hip_newton_decide, dev, ct.byref(state), None if new_err is None else new_err.data_ptr(),
                  top_m.data_ptr())

    # the buffer that holds matrix b's accepted R / M / E, and the other one: rewritten on the device after every round
    Rc, Ro, Mc, Mo, Ec, Eo = [X.PtrList(table, (B, n, n)) for table in tables]
    decide(None)
    fine, top_r = first_fine, (root_bound, root_fine)
    for round_number in range(iter_count):
        top_e = (errors[round_number], fine)
        if round_number > 0:                       # (the first round's candidate root is there already)
            X.gemm(Rc, Ec, addend=Rc, alpha=w, beta=1.0, out=Ro, skip=done, symmetric=symmetric,        # candidate root
                   **(dict(amax=(top_r, top_e), amax_out=found[round_number, 0]) if measured else {}))
            if measured:
                top_r = found[round_number, 0]                               # (a rejected candidate ends its matrix's iteration)
        power, scale = Ec, w                                                 # T^p = I + scale * power by repeated squaring
        top = top_e if measured else None
        for square in range(1, 1 + squarings):
            dst = F[square % 2]
            after = found[round_number, square] if measured else None
            X.gemm(power, power, addend=power, alpha=scale * scale, beta=2 * scale, out=dst, skip=done, symmetric=symmetric,
                   amax=(top, top) if measured else None, amax_out=after)
            power, scale, top = dst, 1.0, after
        new_err = errors[round_number + 1]
        X.gemm(power, Mc, addend=Mc, alpha=scale, beta=1.0, out=Mo, deviation=(Eo, new_err), skip=done, symmetric=symmetric,
               amax=(top, (top_m, fine)) if measured else None, amax_out=found[round_number, 1 + squarings] if measured else None)
        if measured:
            fine = found[round_number, 1 + squarings, 1]
        decide(new_err)
    _LAST_ROUNDS[n] = rounds                       # accepted rounds per matrix of the last stack of this order
    res = R[0]
    if out is not None and out.is_contiguous() and out.dtype == torch.float32 and out.device == dev and out.shape == R[0].shape:
        res = out
    X.F._call(X.F.lib.qtensor_hip_newton_result_batched, dev, R[0].data_ptr(), R[1].data_ptr(), side.data_ptr(), rounds.data_ptr(),
              first_root.data_ptr(), res.data_ptr(), n, B)
    return res if out is None or res is out else out.copy_(res)
