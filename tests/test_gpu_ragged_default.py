"""One default for untuned and tuned ragged plans: a class that the cost model expects
no gain for runs the plan of an untuned batch, bit for bit, and both report it."""
import numpy as np
import pytest

import kfft_amd as K
from kfft_amd.workloads import ragged_batch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("count", [200, 3000])  # (below and above the model's 2^22 points)
def test_tuned_without_a_gain_is_the_untuned_plan(count):
    import torch

    lengths, kinds = ragged_batch(count, seed=5, hi=20000)
    assert (int(lengths.sum()) >= 1 << 22) == (count == 3000)
    m = K.Mlp(len(K.cost_features(16, 0, 1, (16, 0, 0))), 64)
    m.set_params(np.zeros_like(m.get_params()))  # every choice predicted alike
    m.use_as_cost_model()
    try:
        tuned = K.RaggedPlan(lengths, kinds, flags=K.FLAG_GPU_TUNED, half=True)
    finally:
        K.clear_cost_model()
    base = K.RaggedPlan(lengths, kinds, half=True)
    g = torch.Generator(device="cuda").manual_seed(3)
    x = torch.rand(base.in_bytes // 4 + 1, generator=g, device="cuda") * 2 - 1
    out = [torch.zeros(base.out_bytes // 4 + 1, device="cuda") for _ in range(2)]
    base(x, out[0])
    tuned(x, out[1])
    assert torch.equal(out[0], out[1])
    assert tuned.classes() == base.classes()
    cands = [tuple(c) for c in K.tune_candidates()]
    shapes = {tuple(c[3:]) for c in base.classes()}
    assert shapes <= set(cands)
    assert any(ff & 2 for _, ff, _ in shapes)  # Bluestein classes: power-of-two lengths
