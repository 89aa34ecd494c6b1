"""Attention of a prompt in one pass over the keys: the oracle's attention, whose probabilities are rounded behind the division."""
import numpy as np
import pytest

from gpu_util import from_dev, to_dev
from test_gpu_prefill import dec, ptr  # noqa: F401 (dec: a fixture)
from test_gpu_prefill_ranges import inputs

pytestmark = pytest.mark.gpu


# one and more tokens than a workgroup's tile (16 / 32 / 64 for 4 / 2 / 1 query heads per kv head), 63 to 65 keys and around 128, a context in
# ranges (the last of them empty for the first tile, or ending inside a block), heads of one XCD and of several
@pytest.mark.parametrize("n_q,n_kv,T,pos0", [(1, 1, 1, 0), (4, 1, 16, 0), (4, 1, 17, 47), (2, 1, 33, 31), (1, 1, 65, 0), (8, 2, 63, 65), (2, 2, 70, 57), (16, 8, 40, 88), (8, 4, 130, 500),
                                             (1, 1, 2, 4100), (4, 1, 17, 1150), (8, 2, 33, 2046), (2, 2, 127, 1470), (32, 8, 200, 1850), (4, 2, 300, 700)])
@pytest.mark.parametrize("keys", ["level", "rising", "falling"])
def test_follows_the_oracle_token_by_token(gpu, oracle, dec, n_q, n_kv, T, pos0, keys):
    """Either side rounds every probability to BF16 once, by at most 2^-9 of it (the oracle behind the division, the kernel before it), and the
    kernel its result: 2^-8 sum p |v| + 2^-9 |y|.  On top of that 2e-3 of the row's largest value, as in the tests of the two-pass form: a score
    next to a BF16 rounding boundary may fall either way.  The norm of a row's error: roundings of either sign, 3.6e-3 as of two 2^-9
    roundings of a probability and one of the result, 5.1e-3 at most where few keys carry a row; 8e-3 is allowed, a tenth of what the worst case of
    a long context allows.  rising: keys grow along the context, so that the running maximum moves again and again; falling: the first keys carry
    most of the weight, and a block or a range of them left out shows.  Rows past the prompt hold NaN and must not leak; the same bits where the output is off its 16 bytes."""
    torch, dev, lib = gpu
    t_kv = pos0 + T + 40
    q, kc, vc = inputs(oracle, n_q, n_kv, T, pos0, t_kv)
    if keys != "level":
        along = np.arange(pos0 + T, dtype=np.float32) / (pos0 + T)
        kf = dec.f(kc[:, :pos0 + T]) * (1.0 + 3.0 * along if keys == "rising" else 2.0 - along)[None, :, None]
        kc[:, :pos0 + T] = oracle.f32_to_bf16(kf.astype(np.float32))
    qd, kd, vd = to_dev(torch, dev, q), to_dev(torch, dev, kc), to_dev(torch, dev, vc)
    y, z = (torch.zeros(T * n_q * 128 + 64, dtype=torch.int16, device=dev) for _ in range(2))
    for out in (y, z[1:]):
        assert lib.c.hip_attention_prefill_fused_bf16(ptr(qd), ptr(kd), ptr(vd), ptr(out), n_q, n_kv, 128, t_kv, T, pos0) == 0
    torch.cuda.synchronize()
    assert torch.equal(y[:-1], z[1:]) and z[0] == 0 and not y[T * n_q * 128:].any()
    got = from_dev(y, np.uint16)[:T * n_q * 128].reshape(T, n_q, 128)
    kf, vf = dec.f(kc), dec.f(vc)
    kf[:, pos0 + T:], vf[:, pos0 + T:] = 0.0, 0.0               # masked in the oracle too; NaN * 0 would poison its matrix products
    for t in sorted({0, 1, 15, 16, 31, 32, 63, 64, T // 2, T - 2, T - 1} & set(range(T))):
        want = dec.attention(dec.f(q[t]), kf, vf, pos0 + t, n_q, n_kv)
        assert np.isfinite(dec.f(got[t])).all(), t
        bound = 2.0 ** -8 * dec.attention(dec.f(q[t]), kf, np.abs(vf), pos0 + t, n_q, n_kv) + 2.0 ** -9 * np.abs(want)
        assert (np.abs(dec.f(got[t]) - want) <= bound + 2e-3 * np.abs(want).max()).all(), t
        assert np.linalg.norm(dec.f(got[t]) - want) <= 8e-3 * np.linalg.norm(want), t


def test_a_buffer_for_each_form_and_one_piece_under_capture(gpu, oracle, dec):
    """The two-pass form's ranges first, then more ranges of the one-pass form in a larger buffer of its own, then a captured call, which uses none
    and is replayed beside eager calls.  Bad arguments are refused as by the two-pass form."""
    torch, dev, lib = gpu
    n_q, n_kv, T, pos0, t_kv = 32, 8, 256, 3000, 3300
    q, k, v = (to_dev(torch, dev, a) for a in inputs(oracle, n_q, n_kv, T, pos0, t_kv))
    exact, eager, graphed = (torch.zeros(T * n_q * 128, dtype=torch.int16, device=dev) for _ in range(3))
    args = lambda out, T=T, n_q=n_q: (ptr(q), ptr(k), ptr(v), ptr(out), n_q, n_kv, 128, t_kv, T, pos0)
    norm = lambda a, b: np.linalg.norm(dec.f(from_dev(a, np.uint16)) - dec.f(from_dev(b, np.uint16))) / np.linalg.norm(dec.f(from_dev(b, np.uint16)))
    stream = torch.cuda.Stream(device=dev)
    lib.set_sync(False)
    try:
        assert lib.set_stream(stream.cuda_stream) == 0
        assert lib.c.hip_attention_prefill_bf16(*args(exact)) == 0
        assert lib.c.hip_attention_prefill_fused_bf16(*args(eager)) == 0
        stream.synchronize()
        assert norm(eager, exact) <= 2.0 ** -7
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph, stream=stream):
            assert lib.c.hip_attention_prefill_fused_bf16(*args(graphed)) == 0
        first = None
        for _ in range(3):
            graphed.zero_()
            torch.cuda.synchronize()
            with torch.cuda.stream(stream): graph.replay()
            assert lib.c.hip_attention_prefill_fused_bf16(*args(eager)) == 0
            torch.cuda.synchronize()
            first = graphed.clone() if first is None else first
            assert torch.equal(graphed, first) and norm(graphed, eager) <= 2.0 ** -7
        for fn in (lib.c.hip_attention_prefill_bf16, lib.c.hip_attention_prefill_fused_bf16):
            assert fn(*args(eager, T=t_kv - pos0 + 1)) == -1 and fn(*args(eager, n_q=24)) == -1
            assert fn(ptr(q.view(-1)[1:]), ptr(k), ptr(v), ptr(eager), n_q, n_kv, 128, t_kv, T, pos0) == -1
    finally:
        lib.set_stream(None)
        lib.set_sync(True)


def test_memory_of_the_ranges(gpu, oracle):
    """On a stream of its own each form allocates what its header states, once: 33,280 bytes per CU for whole rows, 66,560 for one pass.  (4 MiB: the
    granularity of an allocation.)"""
    torch, dev, lib = gpu
    n_q, n_kv, T, pos0, t_kv = 32, 8, 64, 3000, 3100
    q, k, v = (to_dev(torch, dev, a) for a in inputs(oracle, n_q, n_kv, T, pos0, t_kv))
    y = torch.zeros(T * n_q * 128, dtype=torch.int16, device=dev)
    cus = torch.cuda.get_device_properties(dev).multi_processor_count
    forms = ((lib.c.hip_attention_prefill_bf16, 33280), (lib.c.hip_attention_prefill_fused_bf16, 66560))
    try:
        for stream in (torch.cuda.Stream(device=dev), torch.cuda.Stream(device=dev)):       # the first loads the kernels
            assert lib.set_stream(stream.cuda_stream) == 0
            used = []
            for form, per_cu in forms:
                free = torch.cuda.mem_get_info(dev)[0]
                for _ in range(2):
                    assert form(ptr(q), ptr(k), ptr(v), ptr(y), n_q, n_kv, 128, t_kv, T, pos0) == 0
                    stream.synchronize()
                used.append(free - torch.cuda.mem_get_info(dev)[0])
        for (_, per_cu), n in zip(forms, used): assert 0 < n <= per_cu * cus + (4 << 20), used
    finally:
        lib.set_stream(None)


# Values, keys and queries that are not finite: the two-pass form says which outputs they reach.  Tiles of 16, 32 and 64 tokens, in one piece and in ranges
@pytest.mark.parametrize("n_q,n_kv,T,pos0", [(4, 1, 40, 40), (2, 1, 40, 40), (1, 1, 70, 10), (2, 2, 130, 10), (32, 8, 40, 1500), (1, 1, 66, 2005), (2, 1, 53, 2021)])
@pytest.mark.parametrize("kind", ["later tokens", "last row", "no weight"])
def test_what_is_not_finite_reaches_the_same_outputs(gpu, oracle, n_q, n_kv, T, pos0, kind):
    """later tokens: infinite and NaN value rows of the prompt reach the tokens whose 16 see their block of 64 and no token before those.
    last row: infinite values in the last row that is written stay infinite in the last token.
    no weight: tokens whose scores are all minus infinity give 0."""
    torch, dev, lib = gpu
    t_kv = pos0 + T + 40
    q, kc, vc = inputs(oracle, n_q, n_kv, T, pos0, t_kv)
    if kind == "later tokens":
        vc[:, pos0 + T - 3, ::3] = 0x7F80
        vc[:, pos0 + T - 3, 1::3] = 0x7FC0
    if kind == "last row":
        vc[:, pos0 + T - 1, ::3] = 0x7F80
        vc[:, pos0 + T - 1, 1::3] = 0xFF80
    if kind == "no weight":
        q[5:] = 0x3F80
        kc[:, :pos0 + T] = 0xFF80
        q[:5] = 0
    qd, kd, vd = to_dev(torch, dev, q), to_dev(torch, dev, kc), to_dev(torch, dev, vc)
    one, two = (torch.zeros(T * n_q * 128, dtype=torch.int16, device=dev) for _ in range(2))
    for entry, y in ((lib.c.hip_attention_prefill_fused_bf16, one), (lib.c.hip_attention_prefill_bf16, two)):
        assert entry(ptr(qd), ptr(kd), ptr(vd), ptr(y), n_q, n_kv, 128, t_kv, T, pos0) == 0
    got, want = from_dev(one, np.uint16).reshape(T, -1), from_dev(two, np.uint16).reshape(T, -1)
    odd = lambda a: np.where((a & 0x7F80) != 0x7F80, 0, np.where(a & 0x7F, 1, a))              # 0, 1 for NaN, the bits of an infinity
    assert np.array_equal(odd(got), odd(want))
    if kind == "later tokens": assert odd(want)[-1].any() and not odd(want)[0].any()
    if kind == "last row": assert set(odd(want)[-1, :128].tolist()) == {0, 0x7F80, 0xFF80}
    if kind == "no weight": assert not want[5:].any() and not got[5:].any()
