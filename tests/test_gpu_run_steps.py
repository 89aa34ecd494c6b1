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
        for use_graph in (True, False, run.GRAPH_ALWAYS):
            run.reset(first, 2)
            assert run.run(steps, use_graph) > 0
            assert run.pos == single.pos == 2 + steps and run.token == token
            assert np.array_equal(run.logits(), single.logits())
            for layer in range(cfg.layers):
                for is_v in (False, True):
                    assert np.array_equal(run.kv(layer, is_v)[:, 2:2 + steps], single.kv(layer, is_v)[:, 2:2 + steps])


@pytest.mark.parametrize("steps", [3, 40])
def test_runs_on_the_callers_stream(gpu, pkg, dec, steps):
    """A caller whose launches go to a stream of its own that the null stream does not wait for: run() returns when its steps are done, launched or
    replayed, the time it returns is theirs, and the caller's stream is still the launch stream."""
    torch, dev, lib = gpu
    host = pkg.host_api.host()
    host.init(0)
    cfg = dec.DecodeConfig(layers=16, hidden=1024, n_q=8, n_kv=8, inter=4096, vocab=2000, t_kv=64)       # replayed from 23 steps of 16 layers on
    model = _fresh(pkg, host, cfg)
    stream = torch.cuda.Stream(device=dev)
    lib.set_sync(False)
    try:
        assert lib.set_stream(stream.cuda_stream) == 0
        model.reset(3, 2)
        model.run(steps, True)                                # kernels loaded
        for use_graph in (True, False, model.GRAPH_ALWAYS):
            model.reset(3, 2)
            torch.cuda.synchronize()
            begin, end = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
            begin.record(stream)
            ms = model.run(steps, use_graph)
            assert stream.query() and lib.get_stream() == stream.cuda_stream, use_graph
            end.record(stream)
            torch.cuda.synchronize()
            assert 0.015 * steps * cfg.layers < ms <= begin.elapsed_time(end), use_graph       # six dependent launches a layer
    finally:
        lib.set_stream(None)
        lib.set_sync(True)
