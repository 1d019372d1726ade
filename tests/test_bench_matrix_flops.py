"""bench.py's count of the matrix form's work: real products over the nonzero real and imaginary parts of 16 x 16 operator
blocks, against a count block by block."""
import numpy as np
import pytest


def _count(Heff, c_ops):
    d = Heff.shape[0]
    nt = -(-d // 16)
    total = 0
    # (operator, multiplies from the left): H X, X H^dagger, X c^dagger, c T
    ops = [(Heff, True), (Heff.conj().T, False)] + [(c.conj().T, False) for c in c_ops] + [(c, True) for c in c_ops]
    for op, left in ops:
        for i in range(nt):
            for j in range(nt):          # output tile
                for k in range(nt):
                    r, c = (i, k) if left else (k, j)
                    blk = op[16 * r:16 * r + 16, 16 * c:16 * c + 16]
                    for part in (blk.real, blk.imag):
                        if part.any():   # times the real and the imaginary part of the other factor
                            total += 2 * 2 * 16 ** 3
    return 4 * total


@pytest.mark.parametrize("d", [16, 40, 64])
def test_matrix_form_flops(d):
    from bench import cavity_problem, matrix_form_flops
    H, c_ops, _, _ = cavity_problem(d, 1)
    Heff = H - 0.5j * sum(c.conj().T @ c for c in c_ops)
    assert matrix_form_flops(Heff, c_ops) == _count(Heff, c_ops)
    rng = np.random.default_rng(d)
    M = rng.normal(size=(d, d)) + 1j * rng.normal(size=(d, d))
    nt = -(-d // 16)
    assert matrix_form_flops(M, [M]) == 4 * 4 * 8 * 16 ** 3 * nt ** 3 == _count(M, [M])

