"""Launch shapes of the fused FP4 linear: long rows on 4- and 8-wave workgroups, a pair with more groups than its grid has waves."""
import numpy as np
import pytest

from gpu_util import from_dev, to_dev
from test_gpu_decode import dec, ulp_close  # noqa: F401 (dec: a fixture)

pytestmark = pytest.mark.gpu


# two rows per wave (256 CUs): 8-wave workgroups for 2048 row groups of 12288 elements and more and for 6144 of any length beyond 8192, 4-wave ones one
# group beside that and for shorter rows; rows just past 8192 elements and with a ragged last k-step, odd rows; the pair: five workgroups per CU from
# 7680 rows on, up to 9216 and from 11520 on, four one row beside that, for longer rows and with fewer groups than workgroups
@pytest.mark.parametrize("block,K,n_out,pair", [(16, 12320, 4095, False), (32, 12288, 4097, False), (16, 12256, 4096, False), (16, 8224, 12287, False),
                                                (16, 288, 7680, True), (16, 256, 7679, True), (32, 256, 9216, True), (16, 256, 9217, True), (16, 320, 11520, True), (16, 5152, 7700, True),
                                                (16, 8224, 4093, False), (16, 8224, 4095, False), (32, 8256, 4097, False), (16, 10240, 8200, False),
                                                (16, 256, 5123, True), (32, 288, 5120, True), (16, 2048, 1021, True)])
def test_follows_the_oracle(gpu, pkg, oracle, dec, block, K, n_out, pair):
    from oracle import synth
    torch, dev, lib = gpu
    rng = np.random.default_rng(K + n_out)
    x, res = (oracle.f32_to_bf16(rng.standard_normal(n).astype(np.float32)) for n in (K, n_out))
    packed = [synth.weights_fp4(s, n_out, K, block) for s in ((1, 2) if pair else (1,))]
    W = [oracle.dequant_weight(nib, oracle.FP4, n_out, K, blk_sc=sc, block=block) for nib, sc in packed]
    nd, sd = [to_dev(torch, dev, nib) for nib, _ in packed], [to_dev(torch, dev, sc) for _, sc in packed]
    xd, rd = to_dev(torch, dev, x), to_dev(torch, dev, res)
    y = torch.zeros(n_out + 8, dtype=torch.int16, device=dev)
    d = pkg.capi.make_fused_linear(6, K, [w.data_ptr() for w in nd], [n_out] * len(nd), [y.data_ptr(), None][:len(nd)], xd.data_ptr(), pair=pair,
                                   residual=None if pair else rd.data_ptr(), blk_sc=[s.data_ptr() for s in sd], block_size=block)
    assert lib.quant_linear_fused(d) == 0 and lib.last_kernel() == "gemv_fused_fp4"
    out = from_dev(y, np.uint16)
    assert not out[n_out:].any()
    lin = [dec.linear(w, dec.f(x)) for w in W]
    if pair: assert ulp_close(out[:n_out], dec.silu_mul(*lin), ulps=3.0, floor=1e-4).all()
    else:
        want = dec.r(lin[0] + dec.f(res))
        tol = np.maximum(np.maximum(np.abs(lin[0]), np.abs(dec.f(res))), np.abs(want)) * 2.0 ** -7 + 1e-4       # a BF16 step of the linear or of the sum
        assert (np.abs(dec.f(out[:n_out]).astype(np.float64) - want) <= tol).all()
