"""A batch whose meshes' subtrees fall into every LDS class (budgets 0 to 1024, the smallest class with
more than 1,024 subtrees, meshes without subtrees, a merged whole system) iterates each mesh bitwise as
it iterates alone, in both precisions."""
import numpy as np
import pytest

import meshgen
import mdarap

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("precision", [mdarap.PREC_FP64, mdarap.PREC_FP32_REFINE])
@pytest.mark.parametrize("budgets", [(64, 512, 1024, 0), (1024, 1024, 64, 512), (128, 128, 128, 128)])
def test_mixed_layouts_match_alone(precision, budgets):
    if mdarap.device_count() == 0:
        pytest.fail("no GPU visible: the HIP path cannot run")
    ctx = mdarap.Context(0)
    probs = [meshgen.noisy_icosphere_problem(6), meshgen.noisy_icosphere_problem(5), meshgen.bar_problem(40, 8, 8),
             meshgen.noisy_icosphere_problem(2)]
    out = []
    for together in (False, True):
        ms = []
        for pr, budget in zip(probs, budgets):
            print("case: budgets=%s precision=%d n=%d together=%s" % (budgets, precision, pr.n, together), flush=True)
            m = mdarap.Mesh(ctx, pr.xyz, pr.tri, mdarap.config(precision=precision, subtree_budget=budget))
            m.set_constraints(*pr.constraints())
            m.prepare()
            ms.append(m)
        if together:
            b = mdarap.Batch(ctx, ms)
            b.iterate(3)
            b.close()
        else:
            for m in ms:
                m.iterate(3)
        out.append([m.download() for m in ms])
        for m in ms:
            m.close()
    for a, b in zip(*out):
        assert np.all(np.isfinite(a)) and np.array_equal(a, b)
    ctx.close()
