"""Attention of a few prompt tokens behind a long context: the keys split over workgroups (statistics, sums, combine)."""
import numpy as np
import pytest

from gpu_util import from_dev, to_dev
from test_gpu_prefill import dec, ptr, ulp_close  # noqa: F401 (dec: a fixture)

pytestmark = pytest.mark.gpu


def inputs(oracle, n_q, n_kv, T, pos0, t_kv):
    rng = np.random.default_rng(T + pos0)
    q = oracle.f32_to_bf16(rng.standard_normal((T, n_q, 128)).astype(np.float32))
    kc, vc = (oracle.f32_to_bf16(rng.standard_normal((n_kv, t_kv, 128)).astype(np.float32)) for _ in range(2))
    kc[:, pos0 + T:] = 0x7FC1
    vc[:, pos0 + T:] = 0xFFFF
    return q, kc, vc


# tiles x kv heads against blocks of 64 keys on 256 CUs: one head at the most ranges (32), ranges that end inside a token tile's last
# block, token tiles whose last range is empty, the fewest ranges (2) that pay, one to four query heads per kv head
@pytest.mark.parametrize("n_q,n_kv,T,pos0", [(1, 1, 2, 4100), (4, 1, 17, 1150), (8, 2, 33, 2046), (2, 2, 63, 1470), (8, 4, 16, 1263), (16, 8, 40, 1999), (4, 2, 30, 600), (32, 8, 200, 1850)])
def test_few_tokens_behind_a_long_context_follow_the_oracle(gpu, oracle, dec, n_q, n_kv, T, pos0):
    """The bounds of the attention in one piece (two BF16 steps, row error 4e-3): the same probabilities, sums in another order."""
    torch, dev, lib = gpu
    t_kv = pos0 + T + 40
    q, kc, vc = inputs(oracle, n_q, n_kv, T, pos0, t_kv)
    qd, kd, vd = to_dev(torch, dev, q), to_dev(torch, dev, kc), to_dev(torch, dev, vc)
    y = torch.zeros(T * n_q * 128 + 64, dtype=torch.int16, device=dev)
    assert lib.c.hip_attention_prefill_bf16(ptr(qd), ptr(kd), ptr(vd), ptr(y), n_q, n_kv, 128, t_kv, T, pos0) == 0
    out = from_dev(y, np.uint16)
    assert not out[T * n_q * 128:].any()
    got = out[:T * n_q * 128].reshape(T, n_q, 128)
    kf, vf = dec.f(kc), dec.f(vc)
    kf[:, pos0 + T:], vf[:, pos0 + T:] = 0.0, 0.0               # masked in the oracle too; NaN * 0 would poison its matrix products
    for t in sorted({0, 1, 15, 16, T // 2, T - 2, T - 1} & set(range(T))):
        want = dec.attention(dec.f(q[t]), kf, vf, pos0 + t, n_q, n_kv)
        assert np.isfinite(dec.f(got[t])).all(), t
        assert ulp_close(got[t], want, ulps=2.0, floor=2e-3 * np.abs(want).max()).all(), t
        assert np.linalg.norm(dec.f(got[t]) - want) <= 4e-3 * np.linalg.norm(want), t


@pytest.mark.parametrize("n_q,n_kv,T,pos0", [(1, 1, 1, 0), (8, 2, 20, 44), (4, 2, 33, 95), (2, 2, 17, 239), (8, 2, 130, 126), (4, 4, 16, 241), (4, 1, 20, 1500)])
def test_context_of_up_to_four_blocks_and_its_neighbours(gpu, oracle, dec, n_q, n_kv, T, pos0):
    """64, 128, 256 keys and one more or fewer, and a split context: the oracle's attention, and the same bits where the output is
    not aligned for wide stores."""
    torch, dev, lib = gpu
    t_kv = pos0 + T + 3
    q, kc, vc = inputs(oracle, n_q, n_kv, T, pos0, t_kv)
    qd, kd, vd = to_dev(torch, dev, q), to_dev(torch, dev, kc), to_dev(torch, dev, vc)
    y, z = (torch.zeros(T * n_q * 128 + 64, dtype=torch.int16, device=dev) for _ in range(2))
    for out in (y, z[1:]):
        assert lib.c.hip_attention_prefill_bf16(ptr(qd), ptr(kd), ptr(vd), ptr(out), n_q, n_kv, 128, t_kv, T, pos0) == 0
    torch.cuda.synchronize()
    assert torch.equal(y[:-1], z[1:]) and z[0] == 0 and not y[T * n_q * 128:].any()
    got = from_dev(y, np.uint16)[:T * n_q * 128].reshape(T, n_q, 128)
    kf, vf = dec.f(kc), dec.f(vc)
    kf[:, pos0 + T:], vf[:, pos0 + T:] = 0.0, 0.0
    for t in range(T):
        want = dec.attention(dec.f(q[t]), kf, vf, pos0 + t, n_q, n_kv)
        assert ulp_close(got[t], want, ulps=2.0, floor=2e-3 * np.abs(want).max()).all(), t
        assert np.linalg.norm(dec.f(got[t]) - want) <= 4e-3 * np.linalg.norm(want), t


def test_no_ranges_under_capture(gpu, oracle, dec):
    """A captured call runs in one piece, within the bounds of an eager one, whether or not the stream has scratch memory, and no graph holds
    memory of the library: replays keep their bits behind eager calls of other sizes and a grown GEMM workspace, and two graphs of one
    stream replay side by side on two streams."""
    torch, dev, lib = gpu
    n_q, n_kv, T, pos0, t_kv = 4, 1, 20, 1500, 1600
    sets = [[to_dev(torch, dev, a) for a in inputs(oracle, n_q, n_kv, T, pos0 + i, t_kv)] for i in (0, 1)]
    call = lambda i, y, T=T, pos0=pos0: lib.c.hip_attention_prefill_bf16(*(ptr(t) for t in sets[i]), ptr(y), n_q, n_kv, 128, t_kv, T, pos0)
    eager, other, *captured = (torch.zeros(T * n_q * 128, dtype=torch.int16, device=dev) for _ in range(5))
    lib.set_sync(False)
    try:
        graphs, streams = [], [torch.cuda.Stream(device=dev) for _ in range(2)]
        for stream, i, out, first in ((streams[0], 0, captured[0], True), (streams[0], 1, captured[1], True), (streams[1], 0, captured[2], False)):
            assert lib.set_stream(stream.cuda_stream) == 0
            if first:
                assert call(0, eager) == 0
                stream.synchronize()
            graphs.append(torch.cuda.CUDAGraph())
            with torch.cuda.graph(graphs[-1], stream=stream):
                assert call(i, out) == 0
        a, b = (dec.f(from_dev(t, np.uint16)) for t in (eager, captured[0]))      # not yet replayed
        assert not b.any()
        want = None
        for replay in range(3):
            for out in captured: out.zero_()
            torch.cuda.synchronize()
            for graph, stream in zip(graphs[:2], streams):
                with torch.cuda.stream(stream): graph.replay()
            torch.cuda.synchronize()
            graphs[2].replay()
            torch.cuda.synchronize()
            if want is None:
                want = [out.clone() for out in captured]
                b = dec.f(from_dev(want[0], np.uint16))
                assert np.linalg.norm(a - b) <= 4e-3 * np.linalg.norm(a)
                assert torch.equal(want[0], want[2]) and not torch.equal(want[0], want[1])
            assert all(torch.equal(w, out) for w, out in zip(want, captured)), replay
            assert lib.set_stream(streams[0].cuda_stream) == 0
            assert call(0, other, T=9, pos0=1200) == 0
            assert lib.workspace_reserve((1 << 24) << replay) == 0
            streams[0].synchronize()
            assert call(0, other) == 0
            streams[0].synchronize()
            assert torch.equal(other, eager)
            other.zero_()
        del graphs
    finally:
        lib.set_stream(None)
        lib.set_sync(True)
