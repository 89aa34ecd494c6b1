"""Where the absmax and FP4 block-scale kernels change from rounds of four pieces to single ones and to the tail, and FP4's ties."""
import numpy as np
import pytest

from gpu_util import from_dev, to_dev

pytestmark = pytest.mark.gpu

ROUND = 256 * 1024 * 4                  # floats in one piece of every lane: 256 workgroups of 1024 threads


@pytest.mark.parametrize("dtype", ["float", "half", "bf16"])
@pytest.mark.parametrize("n", [1, 5, 4099, ROUND, ROUND + 1, 3 * ROUND - 4, 4 * ROUND, 5 * ROUND + 7, 9 * ROUND + 4096])
def test_absmax_finds_a_single_maximum_anywhere(gpu, oracle, dtype, n):
    """The one largest magnitude at the first and last element, on both sides of every round and in the tail; exact."""
    torch, dev, lib = gpu
    real, code = {"float": (torch.float32, oracle.FLOAT), "half": (torch.float16, oracle.HALF), "bf16": (torch.bfloat16, oracle.BF16)}[dtype]
    per = ROUND if dtype == "float" else 2 * ROUND
    x = torch.rand(n, device=dev).to(real)
    result = torch.full((2,), -1.0, device=dev)
    places = {0, n - 1, n // 2, n & ~7, (n & ~7) - 1} | {r * per + d for r in range(10) for d in (-1, 0)}
    for at in sorted(p for p in places if 0 <= p < n):
        old = x[at].item()
        x[at] = -37.5
        torch.cuda.synchronize()
        assert lib.absmax(x.data_ptr(), code, n, result.data_ptr()) == 0
        assert result.tolist() == [37.5, -1.0], at
        x[at] = old
    x.fill_(float("nan"))
    torch.cuda.synchronize()
    assert lib.absmax(x.data_ptr(), code, n, result.data_ptr()) == 0 and result.tolist() == [0.0, -1.0]


@pytest.mark.parametrize("dtype", ["float", "half", "bf16"])
@pytest.mark.parametrize("n", [0, 1, 2, 9, 8 * 4096 - 1, 8 * 8192 + 9, ROUND + 5])
def test_absmax_of_pointers_off_their_16_bytes(gpu, oracle, dtype, n):
    """Every offset of whole elements: the maximum at the first and last element, on both sides of the first 16-byte boundary and of the last;
    larger values just outside, and a result of an earlier call, do not count.  One workgroup and several, an empty range."""
    torch, dev, lib = gpu
    real, code, per = {"float": (torch.float32, oracle.FLOAT, 4), "half": (torch.float16, oracle.HALF, 8), "bf16": (torch.bfloat16, oracle.BF16, 8)}[dtype]
    result = torch.full((2,), 99.0, device=dev)
    for off in range(per):
        x = torch.rand(n + 2 * per, device=dev).to(real)
        x[:off], x[off + n:] = -50.0, 50.0
        assert x.data_ptr() % 16 == 0
        places = {off, off + n - 1, off + n // 2} | {e + d for e in (per, 2 * per, (off + n) // per * per) for d in (-1, 0)}
        for at in sorted(p for p in places if off <= p < off + n) or [None]:
            if at is not None: old, x[at] = x[at].item(), -37.5
            torch.cuda.synchronize()
            assert lib.absmax(x[off:].data_ptr(), code, n, result.data_ptr()) == 0
            assert result.tolist() == [0.0 if at is None else 37.5, 99.0], (off, at)
            if at is not None: x[at] = old
            result[0] = 99.0


@pytest.mark.parametrize("block", [16, 32])
@pytest.mark.parametrize("n", [32, 4096 + 32, 4 * (1 << 20) - 32, 4 * (1 << 20) + 32, 16 * (1 << 20) + 32 * 77])
def test_fp4_codes_of_ties_and_their_neighbours(gpu, oracle, block, n):
    """Blocks whose largest value is 6 have factor 1, so the thresholds, the floats next to them, both zeros, infinities and NaN are encoded
    as they are; byte for byte with the oracle, up to pieces past a whole round of four."""
    torch, dev, lib = gpu
    rng = np.random.default_rng(n + block)
    ties = np.array([0.25, 0.75, 1.25, 1.75, 2.5, 3.5, 5.0, 1.0, 6.0], dtype=np.float32)
    values = np.concatenate([ties, np.nextafter(ties, np.float32(0)), np.nextafter(ties[:7], np.float32(9)), [0.0, 1e-38, 1e-45]]).astype(np.float32)
    values = np.concatenate([values, -values])
    x = values[rng.integers(0, values.size, size=n)]
    x[::block] = 6.0
    if n > block: x[block:2 * block] = (rng.standard_normal(block) * 0.02).astype(np.float32)
    x[3], x[n - 1] = np.nan, -np.nan
    if n > 4 * block: x[3 * block + 1], x[2 * block:3 * block] = np.inf, 0.0
    xd = to_dev(torch, dev, x)
    nib, sc = torch.zeros(n // 2 + 16, dtype=torch.uint8, device=dev), torch.zeros(n // block + 16, dtype=torch.uint8, device=dev)
    assert lib.float_to_fp4_blockscale(xd.data_ptr(), nib.data_ptr(), sc.data_ptr(), n, block) == 0
    want_nib, want_sc = oracle.quantize_fp4_blockscale_kernel(x, block)
    got_nib, got_sc = from_dev(nib, np.uint8), from_dev(sc, np.uint8)
    assert np.array_equal(got_nib[:n // 2], want_nib) and not got_nib[n // 2:].any()
    assert np.array_equal(got_sc[:n // block], want_sc) and not got_sc[n // block:].any()
