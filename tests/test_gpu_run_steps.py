"""DecodeModel::run around the step count from which it replays a captured step."""
import numpy as np
import pytest

from test_gpu_prefill import _fresh, dec  # noqa: F401 (dec: a fixture)

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("steps", [1, 2, 23, 24, 25, 40, 179, 180, 181])
def test_launched_and_replayed_steps_equal_single_steps(gpu, pkg, dec, steps):
    """Tokens, positions, logits and cache rows of run(steps) are those of `steps` calls of step(), twice in a row on one model."""
    host = pkg.host_api.host()
    host.init(0)
    cfg = dec.DecodeConfig(layers=2, hidden=256, n_q=4, n_kv=2, inter=512, vocab=1000, t_kv=200)      # replayed from 180 steps of two layers on
    weights = dec.make_model(cfg, 61)
    single, run = _fresh(pkg, host, cfg), _fresh(pkg, host, cfg)
    single.load(weights)
    run.load(weights)
    for first in (3, 11):
        single.reset(first, 2)
        for _ in range(steps):
            token = single.step()
        for use_graph in (True, False):
            run.reset(first, 2)
            assert run.run(steps, use_graph) > 0
            assert run.pos == single.pos == 2 + steps and run.token == token
            assert np.array_equal(run.logits(), single.logits())
            for layer in range(cfg.layers):
                for is_v in (False, True):
                    assert np.array_equal(run.kv(layer, is_v)[:, 2:2 + steps], single.kv(layer, is_v)[:, 2:2 + steps])
