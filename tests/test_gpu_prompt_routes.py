"""The prompt phase of the decode model: which attention a prompt takes, prompts on both sides of the launch that carries their ids, pieces."""
import numpy as np
import pytest

from gpu_util import from_dev, to_dev
from test_gpu_prefill import _fresh, dec, ptr  # noqa: F401 (dec: a fixture)
from test_gpu_prefill_ranges import inputs

pytestmark = pytest.mark.gpu


def state(model, n):
    return model.logits().copy(), [model.kv(li, is_v)[:, :n].copy() for li in range(2) for is_v in (False, True)]


def apart(dec, a, b):
    return max(np.linalg.norm(dec.f(x) - dec.f(y)) / np.linalg.norm(dec.f(y)) for x, y in zip([a[0], *a[1]], [b[0], *b[1]]))


def test_prompts_keep_the_references_rounding_points_unless_asked(gpu, pkg, dec):
    """A model whose decode steps use FP32 probabilities gives the prompt of one with exact attention, byte for byte; the one-pass attention is the
    caller's choice, within the distance of two rounding orders (2e-2 over two layers and the head; it must differ, or nothing was chosen)."""
    host = pkg.host_api.host()
    host.init(0)
    cfg = dec.DecodeConfig(layers=2, hidden=256, n_q=8, n_kv=2, inter=512, vocab=1000, t_kv=420)
    weights = dec.make_model(cfg, 31)
    prompt = [int(t) for t in np.random.default_rng(8).integers(0, cfg.vocab, size=400)]
    out = {}
    for name, exact, fused in (("exact", True, None), ("default", False, None), ("fused", False, True), ("fused and exact", True, True), ("off again", False, False)):
        model = _fresh(pkg, host, cfg)
        model.load(weights)
        model.set_exact_attention(exact)
        if name == "off again": model.set_fused_prompt_attention(True)
        if fused is not None: model.set_fused_prompt_attention(fused)
        out[name] = (model.prefill(prompt), state(model, 400))
    for name in ("default", "fused and exact", "off again"):
        assert out[name][0] == out["exact"][0] and np.array_equal(out[name][1][0], out["exact"][1][0]), name
        assert all(np.array_equal(a, b) for a, b in zip(out[name][1][1], out["exact"][1][1])), name
    assert 0 < apart(dec, out["fused"][1], out["exact"][1]) <= 2e-2


# 64-row tiles against the 16-token tiles that one query head per kv head takes while they are at most one per CU: (query heads, kv heads) of the call, heads
# per call on the other side.  257 to 1024 keys, which no call splits (129 to 256 tiles of 16 tokens, or more); tokens one past a tile, parts of a block
@pytest.mark.parametrize("n_q,n_kv,part", [(32, 8, 8), (16, 8, 8), (16, 16, 8)])
@pytest.mark.parametrize("T,pos0", [(257, 0), (260, 60), (273, 751), (300, 20), (320, 320)])
@pytest.mark.parametrize("odd", [False, True])
def test_tiles_of_64_rows_give_the_bits_of_16_token_tiles(gpu, oracle, n_q, n_kv, part, T, pos0, odd):
    """odd: infinities and NaN among the values, in the last row too, and a key whose scores are minus infinity: the same bits, so that no token sees
    another's block and no row is used twice."""
    torch, dev, lib = gpu
    t_kv = pos0 + T + 30
    q, kc, vc = inputs(oracle, n_q, n_kv, T, pos0, t_kv)
    if odd:
        vc[:, pos0 + T - 1, ::5] = 0x7F80
        vc[:, pos0 + T // 2, 3::11] = 0xFF80
        vc[:, pos0 + 70, 7] = 0x7FC0
        kc[:, pos0 + 33, 9] = 0xFF80
    def attention(q, k, v):
        y = torch.zeros(q.shape[0] * q.shape[1] * 128 + 8, dtype=torch.int16, device=dev)
        qd, kd, vd = (to_dev(torch, dev, np.ascontiguousarray(a)) for a in (q, k, v))
        assert lib.c.hip_attention_prefill_bf16(ptr(qd), ptr(kd), ptr(vd), ptr(y), q.shape[1], k.shape[0], 128, t_kv, T, pos0) == 0
        out = from_dev(y, np.uint16)
        assert not out[-8:].any()
        return out[:-8].reshape(q.shape)
    got = attention(q, kc, vc)
    of = np.arange(n_q) // (n_q // n_kv)                        # kv head of a query head
    want = np.concatenate([attention(q[:, h:h + part], kc[of[h:h + part]], vc[of[h:h + part]]) for h in range(0, n_q, part)], axis=1)
    nan = lambda a: (a & 0x7FFF) > 0x7F80
    assert np.array_equal(nan(got), nan(want)) and np.array_equal(got[~nan(got)], want[~nan(want)])
    assert nan(got).any() == odd


@pytest.mark.parametrize("T", [20, 60, 90])
def test_prompts_of_the_one_pass_attention_follow_the_oracle(gpu, pkg, dec, T):
    """Cache rows of every layer and the logits against the oracle fed token by token, and a step behind the prompt: the bounds of the exact form
    (2e-3 in the first layer, 1e-2) and half as much again for the other place of a rounding."""
    host = pkg.host_api.host()
    host.init(0)
    cfg = dec.DecodeConfig(layers=2, hidden=256, n_q=4, n_kv=2, inter=512, vocab=1000, t_kv=96)
    weights = dec.make_model(cfg, 53)
    model = _fresh(pkg, host, cfg)
    model.load(weights)
    model.set_fused_prompt_attention(True)
    prompt = [int(t) for t in np.random.default_rng(T).integers(0, cfg.vocab, size=T)]
    orc = dec.DecodeOracle(cfg, weights)
    for pos, tok in enumerate(prompt): want, want_next = orc.step(tok, pos)
    model.prefill(prompt)
    for li in range(cfg.layers):
        for is_v, want_c in ((False, orc.k[li]), (True, orc.v[li])):
            got_c = dec.f(model.kv(li, is_v)[:, :T])
            assert np.linalg.norm(got_c - want_c[:, :T]) <= (2e-3 if li == 0 else 1.5e-2) * np.linalg.norm(want_c[:, :T]), (li, is_v)
    for step in range(2):
        got = dec.f(model.logits())
        assert np.linalg.norm(got - want) <= 1.5e-2 * np.linalg.norm(want), step
        if step == 0:
            model.reset(want_next, T)
            model.step()
            want, _ = orc.step(want_next, T)


@pytest.mark.parametrize("fused", [False, True])
@pytest.mark.parametrize("T,pieces", [(256, 100), (257, 100), (257, 256), (2100, 256)])
def test_prompts_around_the_ids_of_a_launch_and_the_longest_piece(gpu, pkg, dec, fused, T, pieces):
    """256 ids travel with a launch, 257 are copied, 2100 tokens are a piece of 2048 and one of 52: what calls of `pieces` tokens leave, up to the
    sums of other GEMM tiles (1e-2 of the caches and the logits; for one pass other running maxima too, half as much again)."""
    host = pkg.host_api.host()
    host.init(0)
    cfg = dec.DecodeConfig(layers=2, hidden=256, n_q=4, n_kv=2, inter=512, vocab=1000, t_kv=2112)
    weights = dec.make_model(cfg, 37)
    prompt = [int(t) for t in np.random.default_rng(T).integers(0, cfg.vocab, size=T)]
    out = []
    for piece in (T, pieces):
        model = _fresh(pkg, host, cfg)
        model.load(weights)
        model.set_fused_prompt_attention(fused)
        for t0 in range(0, T, piece): token = model.prefill(prompt[t0:t0 + piece], pos0=t0)
        assert model.pos == T and model.token == token
        out.append(state(model, T))
    assert apart(dec, *out) <= (1.5e-2 if fused else 1e-2)
