"""Kernel variants at the sizes where their dispatch changes or their tiles
end: each against the oracle or a sparse LU solve of the same system."""
import numpy as np
import pytest

from test_gpu_mg import _reference

pytestmark = pytest.mark.gpu

# The one-workgroup coarse end: whole requests of up to 2048 rows (P1 44 / 45,
# P2 22 / 23, elasticity 31 / 32), level sets that do and do not fit LDS (P2 16
# / 17, elasticity 21 / 31), odd and even coarsening, one level only.
COARSE = [(1, 1, 2), (1, 1, 44), (1, 1, 45), (1, 1, 63), (1, 2, 16), (1, 2, 17), (1, 2, 22), (1, 2, 23), (2, 1, 4),
          (2, 1, 21), (2, 1, 31), (2, 1, 32), (2, 1, 48), (2, 1, 49)]


@pytest.mark.parametrize("batch", [0, 16])
def test_coarse_end_matches_lu(grmp, O, batch):
    """1e-8: the residual is 1e-12 and these systems' condition below 1e4"""
    print(f"[case] one-workgroup coarse end, batch {batch}", flush=True)
    with grmp.Server("mg", mg_batch=batch) as S:
        ts = [S.submit(*spec, 40 + k, rtol=1e-12) for k, spec in enumerate(COARSE)]
        for k, (spec, t) in enumerate(zip(COARSE, ts)):
            r = S.wait(t)
            x = _reference(grmp, O, *spec, 40 + k)
            err = np.linalg.norm(S.solution(t) - x) / max(np.linalg.norm(x), 1e-300)
            assert r.status == 0 and r.iterations <= 40 and err <= 1e-8, (spec, r.status, r.iterations, err)
