"""Per-head norm, RoPE and cache append of a prompt, sixteen lanes per head: head counts that leave the last workgroup partly
empty and put q, k and v heads into one wave, pointers that lie on any element, and nothing written outside the rows.  The
oracle is the one-token kernel, token by token, which must leave the same bytes (it adds the squares in the same order)."""
import ctypes

import numpy as np
import pytest

from gpu_util import from_dev, to_dev
from test_gpu_prefill import dec  # noqa: F401 (a fixture)

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n_q,n_kv,T,pos0,off,normed", [(1, 1, 1, 0, 0, True), (5, 3, 9, 2, 0, True), (5, 3, 9, 2, 1, False), (4, 1, 17, 70, 3, True),
                                                        (32, 8, 2, 5, 0, True), (16, 8, 7, 0, 1, True)])
def test_rows_at_odd_head_counts_and_offsets(gpu, oracle, dec, n_q, n_kv, T, pos0, off, normed):  # noqa: F811
    torch, dev, lib = gpu
    rng = np.random.default_rng(n_q * 100 + T + off)
    t_kv = 96
    cos, sin = dec.rope_tables(dec.DecodeConfig(n_q=n_q, n_kv=n_kv, t_kv=t_kv))

    def at(a, skip):        # the array behind `skip` elements of the 16-byte aligned allocation, so that it starts on any element
        d = to_dev(torch, dev, np.concatenate([np.full(skip, 0x7FC1, np.uint16), a.reshape(-1)]))
        return d, ctypes.c_void_p(d.data_ptr() + 2 * skip)

    bf = lambda *shape: oracle.f32_to_bf16((2 * rng.standard_normal(shape)).astype(np.float32))
    q, k, v, qw, kw = bf(T, n_q, 128), bf(T, n_kv, 128), bf(T, n_kv, 128), bf(128), bf(128)
    base_k, base_v = bf(n_kv, t_kv, 128), bf(n_kv, t_kv, 128)
    keep, p = zip(*[at(a, s) for a, s in ((q, off), (k, off), (v, 2 * off), (qw, off), (kw, off), (cos, off), (sin, off),
                                          (np.zeros((T, n_q, 128), np.uint16), off), (base_k, off), (base_v, 2 * off))])
    w = p[3:5] if normed else (ctypes.c_void_p(0), ctypes.c_void_p(0))
    assert lib.c.hip_qk_norm_rope_kv_rows_bf16(p[0], p[1], p[2], *w, *p[5:], n_q, n_kv, 128, t_kv, T, pos0, ctypes.c_float(1e-6)) == 0
    kc, vc = to_dev(torch, dev, base_k), to_dev(torch, dev, base_v)
    q_ref = np.zeros((T, n_q, 128), np.uint16)
    tables = [to_dev(torch, dev, a) for a in (qw, kw, cos, sin)]
    tp = [ctypes.c_void_p(t.data_ptr()) for t in tables]
    w = tp[:2] if normed else (ctypes.c_void_p(0), ctypes.c_void_p(0))
    for t in range(T):
        one = [to_dev(torch, dev, a) for a in (q[t], k[t], v[t])]
        q1, pd = torch.zeros(n_q * 128, dtype=torch.int16, device=dev), torch.tensor([pos0 + t], dtype=torch.int32, device=dev)
        assert lib.c.hip_qk_norm_rope_kv_bf16(*[ctypes.c_void_p(a.data_ptr()) for a in one], *w, *tp[2:], ctypes.c_void_p(q1.data_ptr()), ctypes.c_void_p(kc.data_ptr()),
                                              ctypes.c_void_p(vc.data_ptr()), n_q, n_kv, 128, t_kv, ctypes.c_void_p(pd.data_ptr()), ctypes.c_float(1e-6)) == 0
        q_ref[t] = from_dev(q1, np.uint16).reshape(n_q, 128)
    for i, skip, want in ((7, off, q_ref), (8, off, from_dev(kc, np.uint16)), (9, 2 * off, from_dev(vc, np.uint16))):
        got = from_dev(keep[i], np.uint16)
        assert (got[:skip] == 0x7FC1).all()
        assert np.array_equal(got[skip:], want.reshape(-1))


@pytest.mark.parametrize("T,off", [(465, 0), (466, 0), (1303, 1), (1304, 1)])
def test_many_rows_leave_the_bytes_of_few(gpu, oracle, dec, T, off):  # noqa: F811
    """11 heads a token, one token short of the line from which sixteen lanes take a head and on it, aligned and not: the bytes of calls of at
    most 100 tokens, which give a wave to a head."""
    torch, dev, lib = gpu
    n_q, n_kv, t_kv, pos0 = 5, 3, T + 40, 33
    gen = torch.Generator(device=dev).manual_seed(T)
    make = lambda n: (2 * torch.randn(n + 16, device=dev, generator=gen)).to(torch.bfloat16).view(torch.int16)
    q, k, v, qw, kw = make(T * n_q * 128), make(T * n_kv * 128), make(T * n_kv * 128), make(128), make(128)
    cos, sin = make(t_kv * 64), make(t_kv * 64)
    results = []
    for piece in (T, 100):
        q_out, kc, vc = (torch.full((n + 16,), 0x7FC1, dtype=torch.int16, device=dev) for n in (T * n_q * 128, n_kv * t_kv * 128, n_kv * t_kv * 128))
        at = lambda t, element: ctypes.c_void_p(t.data_ptr() + 2 * element)
        for t in range(0, T, piece):
            assert lib.c.hip_qk_norm_rope_kv_rows_bf16(at(q, off + t * n_q * 128), at(k, off + t * n_kv * 128), at(v, 2 * off + t * n_kv * 128), at(qw, off), at(kw, off), at(cos, off), at(sin, off),
                                                       at(q_out, off + t * n_q * 128), at(kc, off), at(vc, 2 * off), n_q, n_kv, 128, t_kv, min(piece, T - t), pos0 + t, ctypes.c_float(1e-6)) == 0
        torch.cuda.synchronize()
        results.append((q_out, kc, vc))
    for a, b in zip(*results): assert torch.equal(a, b)
