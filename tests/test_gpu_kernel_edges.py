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
