"""The class walk's workgroup errors as the sampled error measurement takes
them: independent from one workgroup to the next, although all of them read
the same rounded offsets of the class and walk columns."""
import numpy as np
import pytest

import permanent_amd as P

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,density", [(24, 0.2), (24, 0.5), (25, 0.7), (26, 0.35)])
def test_workgroup_errors_add_up_as_independent_ones(n, density):
    """E_b: a workgroup's FP64 sum minus its double-double X sum.  (sum of
    E_b)^2 / sum of E_b^2 has mean 1 for independent errors, and over eight
    matrices of each kind a mean above 1 + 3 sqrt(2 / 8) in one of a thousand
    draws."""
    ratios = []
    for seed in range(8):
        a = P.synthetic_matrix(n, density, 900 + 10 * n + seed, full_support=True)
        plan = P.Plan(a)
        assert plan.run(mode=0).clock_ghz > 0.0
        _, _, blocks = plan.geometry()
        e = np.empty(blocks)
        for b in range(blocks):
            f, d = plan.run_blocks(b, b + 1, mode=0), plan.run_blocks(b, b + 1, mode=2)
            e[b] = (f.sum_hi - d.sum_hi) + (f.sum_lo - d.sum_lo)
        plan.close()
        ratios.append(float(e.sum() ** 2 / (e ** 2).sum()))
    print(f"n={n} density {density}: {blocks} workgroups, mean {np.mean(ratios):.2f} "
          f"of {[round(r, 2) for r in ratios]}")
    assert np.mean(ratios) <= 1.0 + 3.0 * np.sqrt(2.0 / 8.0)
