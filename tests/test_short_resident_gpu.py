"""Short K-quant prompts do not depend on which copies of the weights are resident: the repack is read wherever it is there."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("mix", ["Q4_K_M", "Q5_K", "Q6_K"])
def test_prompts_of_a_model_by_what_is_resident(mix):
    """layers as wide as the register form takes: the file's blocks alone, both copies, the repack alone"""
    from ntransformer_amd import engine as E
    toks = [int(t) for t in np.random.default_rng(3).integers(0, E.PRESETS["8b"]["vocab"], 16)]
    rows = []
    for level in (0, 1, 2):
        eng = E.Engine()
        eng.set_option("repack", level)
        eng.load_synthetic(E.synth_spec("8b", mix, seed=5, layers=3), 64)
        hd = []
        for n in (2, 16, 20):
            eng.forward(toks[:n], 0)
            hd.append(eng.forward(toks[:n], 0))
        rows.append(hd)
        eng.close()
    for a, b, c in zip(*rows):
        assert np.isfinite(a).all() and np.array_equal(b, c)
        assert np.abs(a - b).max() <= 1e-3 * np.abs(a).max()          # (the file's blocks alone: other sums, and another head)
