"""Token ids and the step state that travel with a launch."""
import ctypes

import numpy as np
import pytest

from gpu_util import from_dev, to_dev
from test_gpu_prefill import _fresh, dec  # noqa: F401 (dec: a fixture)

pytestmark = pytest.mark.gpu
ptr = lambda t: ctypes.c_void_p(t.data_ptr())


@pytest.mark.parametrize("n,D", [(1, 8), (3, 2056), (256, 64)])
def test_rows_of_host_ids(gpu, oracle, n, D):
    """The rows byte for byte, ids outside the table to its nearest row, nothing behind the last one; more ids than fit are refused."""
    torch, dev, lib = gpu
    rng = np.random.default_rng(n)
    rows = 50
    W = rng.integers(0, 1 << 16, size=(rows, D), dtype=np.uint16)
    ids = rng.integers(0, rows, size=n).astype(np.int32)
    ids[-1] = rows + 7
    if n > 1: ids[0] = -3
    wd, y = to_dev(torch, dev, W), torch.zeros(n * D + 8, dtype=torch.int16, device=dev)
    assert lib.c.hip_embed_ids_bf16(ids.ctypes.data_as(ctypes.c_void_p), n, ptr(wd), ptr(y), D, rows) == 0
    ids_then = ids.copy()
    ids[:] = 0                                      # the launch has its own copy
    torch.cuda.synchronize()
    got = from_dev(y, np.uint16)
    assert np.array_equal(got[:n * D].reshape(n, D), W[np.clip(ids_then, 0, rows - 1)]) and not got[n * D:].any()
    assert lib.c.hip_embed_ids_bf16(ids.ctypes.data_as(ctypes.c_void_p), 257, ptr(wd), ptr(y), D, rows) == -1
    assert lib.c.hip_embed_ids_bf16(ids.ctypes.data_as(ctypes.c_void_p), n, ptr(wd), ptr(y), D + 1, rows) == -1
    for w, out in ((wd.view(-1)[1:], y), (wd, y[1:]), (wd.view(-1)[4:], y)):            # off their 16 bytes
        assert lib.c.hip_embed_ids_bf16(ids.ctypes.data_as(ctypes.c_void_p), n, ptr(w), ptr(out), D, rows - 1) == -1


@pytest.mark.parametrize("D", [8, 2048, 4104])
def test_state_and_row_of_a_step(gpu, D):
    torch, dev, lib = gpu
    row = to_dev(torch, dev, np.arange(D, dtype=np.uint16))
    state, y = torch.full((3,), 9, dtype=torch.int32, device=dev), torch.zeros(D + 8, dtype=torch.int16, device=dev)
    assert lib.c.hip_decode_begin_bf16(ptr(state), 5, 77, ptr(row), ptr(y), D) == 0
    torch.cuda.synchronize()
    assert state.tolist() == [5, 77, 9] and torch.equal(y[:D], row) and not y[D:].any()
    assert lib.c.hip_decode_begin_bf16(ptr(state), 5, 77, ptr(row), ptr(y), D + 4) == -1
    for r, out in ((row[1:], y), (row, y[1:]), (row, y[4:])):                           # off their 16 bytes
        assert lib.c.hip_decode_begin_bf16(ptr(state), 5, 77, ptr(r), ptr(out), D) == -1


def test_state_of_a_reset_is_in_place_when_it_returns(gpu, pkg, dec):
    """reset on a stream with work in front of it, then the state read and a graph run asked for on another: the new token and position, and a run past
    the end of the cache refused."""
    torch, dev, lib = gpu
    host = pkg.host_api.host()
    host.init(0)
    cfg = dec.DecodeConfig(layers=2, hidden=256, n_q=4, n_kv=2, inter=512, vocab=1000, t_kv=64)
    model = _fresh(pkg, host, cfg)
    model.load(dec.make_model(cfg, 17))
    model.reset(1, 0)
    busy, other = (torch.cuda.Stream(device=dev) for _ in range(2))
    lib.set_sync(False)
    try:
        assert lib.set_stream(busy.cuda_stream) == 0
        with torch.cuda.stream(busy): torch.cuda._sleep(100_000_000)               # some 50 ms
        model.reset(7, 60)
        assert lib.set_stream(other.cuda_stream) == 0
        assert (model.token, model.pos) == (7, 60)
        assert lib_run(model, 5) == -2.0 and lib_run(model, 4) > 0
        assert model.pos == 64
        torch.cuda.synchronize()
    finally:
        lib.set_stream(None)
        lib.set_sync(True)


def test_a_graph_run_behind_a_prompt_on_another_stream_sees_its_position(gpu, pkg, dec):
    """A prompt's position is written by a launch: a graph run asked for on another stream waits for it before it looks whether its steps fit."""
    torch, dev, lib = gpu
    host = pkg.host_api.host()
    host.init(0)
    cfg = dec.DecodeConfig(layers=2, hidden=256, n_q=4, n_kv=2, inter=512, vocab=1000, t_kv=64)
    model = _fresh(pkg, host, cfg)
    model.load(dec.make_model(cfg, 17))
    model.prefill([1] * 60)                                     # its buffers are there
    model.reset(1, 0)
    busy, other = (torch.cuda.Stream(device=dev) for _ in range(2))
    prompt = np.arange(60, dtype=np.int32)
    lib.set_sync(False)
    try:
        assert lib.set_stream(busy.cuda_stream) == 0
        with torch.cuda.stream(busy): torch.cuda._sleep(100_000_000)
        assert model.lib.c.cccc_decode_prefill(model.handle, prompt.ctypes.data_as(ctypes.POINTER(ctypes.c_int)), 60, 0) == 0
        assert lib.set_stream(other.cuda_stream) == 0
        assert lib_run(model, 5) == -2.0 and lib_run(model, 4) > 0
        assert model.pos == 64
        torch.cuda.synchronize()
    finally:
        lib.set_stream(None)
        lib.set_sync(True)


def lib_run(model, n):
    return model.lib.c.cccc_decode_run(model.handle, n, 2)          # 2: with a graph whatever n is
