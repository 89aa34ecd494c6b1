"""Every compiled tile of the prompt GEMMs, unsplit and with the k range split, through the C-ABI: the planner is asked first, so
that a change of its tables cannot leave a kernel untested unseen."""
import ctypes

import numpy as np
import pytest

from gemm_plan_util import LINEAR, PAIR, SEGMENTS, plan
from gpu_util import MAX_REL, ROW_L2_REL, from_dev

pytestmark = pytest.mark.gpu

# weight layout, kind of launch, [(tokens, features, K, tokens / 16 and features / 64 of the tile, k ranges)] on 256 CUs: tokens and
# features one past a tile or well short of one, K from one or three k-tiles to an odd number of them; segments are the features and
# twice about a quarter of them
CASES = [
    ("tiled", LINEAR, [(17, 72, 192, 2, 1, 1), (17, 72, 1600, 2, 1, 3), (17, 16392, 640, 2, 2, 1), (17, 6152, 3136, 2, 2, 3), (65, 72, 192, 4, 1, 1), (65, 72, 2112, 4, 1, 2),
        (65, 136, 192, 4, 2, 1), (33, 5128, 3136, 4, 2, 4), (65, 8200, 192, 4, 3, 1), (129, 16392, 192, 4, 4, 1), (65, 5128, 6208, 4, 4, 5), (385, 9736, 192, 8, 3, 1),
        (65, 16392, 3136, 8, 4, 3)]),
    ("tiled", PAIR, [(17, 72, 192, 2, 2, 1), (17, 72, 1600, 2, 2, 3), (17, 8200, 8256, 2, 4, 3), (65, 72, 192, 4, 2, 1), (65, 72, 1600, 4, 2, 3), (129, 16392, 192, 4, 4, 1),
        (65, 2568, 6208, 4, 4, 5), (65, 16392, 192, 8, 4, 1), (65, 8200, 3136, 8, 4, 3)]),
    ("tiled", SEGMENTS, [(17, 72, 192, 2, 1, 1), (17, 72, 1600, 2, 1, 3), (17, 12296, 1088, 2, 2, 1), (17, 4104, 3136, 2, 2, 3), (65, 72, 192, 4, 1, 1), (65, 72, 1600, 4, 1, 3),
        (1030, 264, 192, 4, 2, 1), (257, 264, 4160, 4, 2, 6), (65, 12296, 192, 4, 4, 1), (129, 2056, 6208, 4, 4, 5), (1030, 9736, 192, 8, 4, 1), (65, 12296, 3136, 8, 4, 3)]),
    ("file", LINEAR, [(17, 72, 192, 2, 1, 1), (17, 72, 1600, 2, 1, 3), (17, 16392, 320, 2, 2, 1), (17, 5128, 3136, 2, 2, 5), (65, 72, 192, 4, 1, 1), (65, 72, 2112, 4, 1, 2),
        (65, 136, 192, 4, 2, 1), (33, 5128, 3136, 4, 2, 5), (65, 8200, 192, 4, 3, 1), (193, 12296, 192, 4, 4, 1), (193, 12296, 640, 8, 2, 1), (65, 5128, 4160, 8, 2, 4),
        (193, 16392, 192, 8, 3, 1), (257, 16392, 192, 8, 4, 1), (65, 16392, 3136, 8, 4, 3)]),
    ("file", PAIR, [(17, 72, 192, 2, 2, 1), (17, 72, 1088, 2, 2, 2), (17, 8200, 2112, 2, 4, 3), (65, 72, 192, 4, 2, 1), (65, 72, 1088, 4, 2, 2), (129, 16392, 192, 4, 4, 1),
        (33, 8200, 3136, 4, 4, 3), (2050, 72, 832, 8, 2, 1), (1030, 72, 2112, 8, 2, 3), (65, 16392, 192, 8, 4, 1), (65, 8200, 2112, 8, 4, 3)]),
    ("file", SEGMENTS, [(17, 72, 192, 2, 1, 1), (17, 72, 1600, 2, 1, 3), (17, 12296, 320, 2, 2, 1), (17, 4104, 4160, 2, 2, 4), (17, 12296, 2112, 2, 4, 3), (65, 72, 192, 4, 1, 1),
        (65, 72, 1600, 4, 1, 3), (1030, 264, 192, 4, 2, 1), (129, 1032, 3136, 4, 2, 5), (65, 12296, 192, 4, 4, 1), (33, 12296, 3136, 4, 4, 3), (2050, 264, 1088, 8, 2, 1),
        (700, 264, 4160, 8, 2, 5), (257, 16392, 192, 8, 4, 1), (65, 12296, 3136, 8, 4, 3)]),
    ("tiled_scaled", LINEAR, [(17, 72, 192, 2, 1, 1), (17, 72, 1600, 2, 1, 3), (17, 16392, 8256, 2, 4, 4), (65, 72, 192, 4, 1, 1), (65, 72, 2112, 4, 1, 2), (65, 136, 192, 4, 2, 1),
        (65, 2568, 3136, 4, 2, 3), (65, 8200, 192, 4, 3, 1), (129, 16392, 192, 4, 4, 1), (65, 16392, 4160, 4, 4, 3), (385, 9736, 192, 8, 3, 1), (65, 16392, 3136, 8, 4, 3)]),
    ("tiled_scaled", PAIR, [(17, 72, 192, 2, 2, 1), (17, 72, 1600, 2, 2, 3), (17, 8200, 4160, 2, 4, 3), (65, 72, 192, 4, 2, 1), (65, 72, 1600, 4, 2, 3), (129, 16392, 192, 4, 4, 1),
        (33, 8200, 3136, 4, 4, 3), (193, 9736, 192, 8, 4, 1), (65, 8200, 2112, 8, 4, 3)]),
    ("tiled_scaled", SEGMENTS, [(17, 72, 192, 2, 1, 1), (17, 72, 1600, 2, 1, 3), (17, 12296, 6208, 2, 4, 3), (65, 72, 192, 4, 1, 1), (65, 72, 1600, 4, 1, 3), (1030, 264, 192, 4, 2, 1),
        (385, 264, 2112, 4, 2, 4), (65, 16392, 192, 4, 4, 1), (33, 12296, 4160, 4, 4, 3), (1030, 9736, 192, 8, 4, 1), (65, 12296, 3136, 8, 4, 3)]),
    ("file_scaled", LINEAR, [(17, 72, 192, 2, 1, 1), (17, 72, 1600, 2, 1, 3), (17, 16392, 320, 2, 2, 1), (17, 5128, 3136, 2, 2, 5), (65, 72, 192, 4, 1, 1), (65, 72, 2112, 4, 1, 2),
        (65, 136, 192, 4, 2, 1), (33, 5128, 3136, 4, 2, 5), (65, 8200, 192, 4, 3, 1), (193, 12296, 192, 4, 4, 1), (65, 16392, 4160, 4, 4, 3), (193, 16392, 192, 8, 3, 1),
        (257, 16392, 192, 8, 4, 1), (700, 1032, 4160, 8, 4, 4)]),
    ("file_scaled", PAIR, [(17, 72, 192, 2, 2, 1), (17, 72, 1088, 2, 2, 2), (17, 8200, 2112, 2, 4, 3), (65, 72, 192, 4, 2, 1), (65, 72, 1088, 4, 2, 2), (129, 16392, 192, 4, 4, 1),
        (33, 8200, 2112, 4, 4, 3), (65, 16392, 192, 8, 4, 1), (65, 8200, 2112, 8, 4, 3)]),
    ("file_scaled", SEGMENTS, [(17, 72, 192, 2, 1, 1), (17, 72, 1600, 2, 1, 3), (17, 12296, 320, 2, 2, 1), (17, 4104, 4160, 2, 2, 4), (17, 12296, 2112, 2, 4, 3), (65, 72, 192, 4, 1, 1),
        (65, 72, 1600, 4, 1, 3), (1030, 264, 192, 4, 2, 1), (257, 264, 4160, 4, 2, 6), (65, 16392, 192, 4, 4, 1), (33, 12296, 3136, 4, 4, 3), (257, 16392, 192, 8, 4, 1),
        (65, 12296, 2112, 8, 4, 3)]),
    ("fp4", LINEAR, [(17, 72, 128, 2, 1, 1), (17, 72, 1152, 2, 1, 2), (17, 16392, 128, 2, 2, 1), (17, 12296, 2176, 2, 2, 4), (65, 72, 128, 4, 1, 1), (65, 72, 2176, 4, 1, 2),
        (2050, 520, 128, 4, 2, 1), (33, 8200, 4224, 4, 2, 6), (65, 16392, 128, 4, 3, 1), (385, 16392, 128, 4, 4, 1), (2050, 2056, 128, 8, 2, 1), (65, 16392, 3200, 8, 2, 3),
        (193, 16392, 384, 8, 3, 1)]),
    ("fp4", PAIR, [(17, 72, 128, 2, 2, 1), (17, 72, 1152, 2, 2, 2), (65, 72, 128, 4, 2, 1), (65, 72, 1152, 4, 2, 2), (129, 16392, 128, 4, 4, 1), (2050, 1032, 128, 8, 2, 1),
        (2050, 72, 1664, 8, 2, 3)]),
    ("fp4", SEGMENTS, [(17, 72, 128, 2, 1, 1), (17, 72, 1152, 2, 1, 2), (17, 12296, 128, 2, 2, 1), (17, 8200, 2176, 2, 2, 4), (65, 72, 128, 4, 1, 1), (65, 72, 1152, 4, 1, 2),
        (2050, 264, 128, 4, 2, 1), (1030, 264, 1664, 4, 2, 3), (193, 16392, 128, 4, 4, 1), (2050, 1544, 128, 8, 2, 1), (1030, 264, 6272, 8, 2, 7)]),
]


def widths_of(n_out):
    return [n_out] + [max(72, n_out // 4 // 8 * 8 + 8)] * 2


class Weight:
    """Random codes on the device (no NaN or infinity), their exact values in float64, and the registered tiled copy."""

    def __init__(self, gpu, oracle, layout, n_out, K, gen):
        self.torch, dev, self.lib = gpu
        torch = self.torch
        fp4, self.tiled = layout == "fp4", layout != "file" and layout != "file_scaled"
        self.type = oracle.FP4 if fp4 else oracle.E4M3 if "scaled" in layout else oracle.E5M2
        self.scale = 0.013 if "scaled" in layout else 1.0
        self.n_out, self.K, self.scales = n_out, K, None
        if fp4:
            self.codes = torch.randint(0, 256, (n_out, K // 2), dtype=torch.uint8, device=dev, generator=gen)
            self.scales = torch.randint(0x20, 0x40, (n_out, K // 16), dtype=torch.uint8, device=dev, generator=gen)
        else:
            codes = torch.randint(0, 256, (n_out, K), dtype=torch.uint8, device=dev, generator=gen)
            mask, one = (0x7C, 0x3C) if self.type == oracle.E5M2 else (0x7F, 0x38)
            self.codes = torch.where((codes & mask) == mask, torch.full_like(codes, one), codes)
        self.copy = torch.zeros(self.lib.tiled_size(self.type, n_out, K), dtype=torch.uint8, device=dev) if self.tiled else None
        if fp4: assert self.lib.weight_prepare_fp4(self.codes.data_ptr(), self.scales.data_ptr(), 16, n_out, K, self.copy.data_ptr()) == 0
        elif self.tiled: assert self.lib.weight_prepare(self.codes.data_ptr(), self.type, n_out, K, K, self.copy.data_ptr()) == 0

    def exact(self, oracle, half=False):
        torch = self.torch
        table = lambda bits: torch.from_numpy(oracle.bf16_to_f32(bits).astype(np.float64)).to(self.codes.device)
        every = np.arange(256, dtype=np.uint8)
        if self.scales is not None:
            nibbles = table(oracle.dequant_fp4_to_bf16(every[:16] | (every[:16] << 4), 32, 1.0)[::2])
            codes = self.codes.long()
            values = torch.stack([nibbles[codes & 15], nibbles[codes >> 4]], dim=2).view(self.n_out, self.K // 16, 16)
            return (values * table(oracle.dequant_fp8_to_bf16(every, oracle.E4M3, 1.0))[self.scales.long()][:, :, None]).view(self.n_out, self.K)
        if half:
            rc, bits = oracle.convert(every, self.type, oracle.HALF, 256, self.scale)
            assert rc == 0
            return torch.from_numpy(bits.view(np.float16).astype(np.float64)).to(self.codes.device)[self.codes.long()]
        return table(oracle.dequant_fp8_to_bf16(every, self.type, self.scale))[self.codes.long()]

    def release(self):
        if self.tiled: assert self.lib.weight_release(self.codes.data_ptr()) == 0


@pytest.mark.parametrize("layout,kind,shapes", CASES, ids=[f"{c[0]}-{('linear', 'pair', 'segments')[c[1]]}" for c in CASES])
def test_every_tile_against_the_exact_contraction(gpu, oracle, layout, kind, shapes):
    """The tolerance is that of the other linear tests (row L2 error 2e-3 and largest error 1e-2 of the exact contraction rounded
    to 16 bits; the SwiGLU product of two rounded linears 1e-2), nothing is written past the output; plain FP8 linears on HALF
    activations as well."""
    torch, dev, lib = gpu
    assert torch.cuda.get_device_properties(0).multi_processor_count == 256
    ptr = lambda t: ctypes.c_void_p(t.data_ptr())
    for tokens, n_out, K, mb, nb, splits in shapes:
        widths = {LINEAR: [n_out], PAIR: [n_out] * 2, SEGMENTS: widths_of(n_out)}[kind]
        chosen = plan(kind, tokens, widths if kind == SEGMENTS else n_out, K, fp4=layout == "fp4", row_major=layout.startswith("file"), scaled="scaled" in layout)
        assert chosen[:3] == (mb, nb, splits), (tokens, n_out, K)
        print(layout, kind, tokens, n_out, K, flush=True)
        gen = torch.Generator(device=dev).manual_seed(tokens + n_out + K)
        weights = [Weight(gpu, oracle, layout, n, K, gen) for n in widths]
        w0 = weights[0]
        x = (torch.randn(tokens, K, device=dev, generator=gen) * (0.05 if w0.type == oracle.E5M2 else 1.0)).to(torch.bfloat16)
        try:
            for half in (False, True):
                if half and (kind != LINEAR or layout == "fp4"): continue
                dtype = torch.float16 if half else torch.bfloat16
                xt = (x * 0.002).to(dtype) if half and w0.type == oracle.E5M2 else x.to(dtype)       # outputs within the range of HALF
                outs = [torch.zeros(tokens * n + 64, dtype=dtype, device=dev) for n in (widths[:1] if kind == PAIR else widths)]
                torch.cuda.synchronize()
                if kind == LINEAR:
                    rc = lib.linear(w0.codes.data_ptr(), w0.type, xt.data_ptr(), outs[0].data_ptr(), n_out, tokens, K, w0.scale,
                                    w0.scales.data_ptr() if layout == "fp4" else None, 16, act_type=oracle.HALF if half else oracle.BF16)
                elif kind == PAIR:
                    rc = lib.c.hip_quant_gemm_swiglu(n_out, tokens, K, ptr(w0.codes), ptr(weights[1].codes), w0.type, K, w0.scale, w0.scale, ptr(xt), K, ptr(outs[0]), n_out)
                else:
                    n = (ctypes.c_int * 3)(*widths)
                    rc = lib.c.hip_quant_gemm_segments(3, n, (ctypes.c_void_p * 3)(*(w.codes.data_ptr() for w in weights)), (ctypes.c_float * 3)(*[w0.scale] * 3),
                                                       (ctypes.c_void_p * 3)(*(o.data_ptr() for o in outs)), n, w0.type, tokens, K, K, ptr(xt), K)
                assert rc == 0
                torch.cuda.synchronize()
                exact = [(xt.double() @ w.exact(oracle, half).T).to(dtype).double() for w in weights]
                if kind == PAIR:
                    gate, up = exact
                    silu = (gate * torch.sigmoid(gate).to(dtype).double()).to(dtype).double()
                    exact = [(silu * up).to(dtype).double()]
                for out, want in zip(outs, exact):
                    assert not out[want.numel():].any()
                    diff = out[:want.numel()].view_as(want).double() - want
                    if kind == PAIR:
                        assert diff.norm() <= 1e-2 * want.norm(), (tokens, n_out, K)
                        continue
                    assert (diff.norm(dim=1) <= ROW_L2_REL * want.norm(dim=1)).all(), (tokens, n_out, K, half)
                    assert (diff.abs().amax(dim=1) <= MAX_REL * want.abs().amax(dim=1)).all(), (tokens, n_out, K, half)
        finally:
            for w in weights: w.release()


@pytest.mark.parametrize("layout,tokens,n_out,K,splits", [("fp4", 18, 72, 1024, 2), ("fp4", 65, 72, 2048, 2), ("fp4", 1030, 1032, 2048, 1), ("fp4", 800, 4096, 2048, 1),
                                                          ("fp4", 1030, 520, 3072, 3), ("fp4", 800, 2056, 3072, 3), ("file", 64, 3080, 1024, 1), ("file", 1030, 520, 3072, 3),
                                                          ("file", 800, 2056, 2048, 1), ("file", 800, 1032, 4096, 4), ("tiled", 640, 3080, 2048, 1), ("tiled", 257, 3080, 4096, 3),
                                                          ("tiled_scaled", 65, 3080, 3072, 3), ("file_scaled", 640, 520, 2048, 1)])
def test_residual_add_and_norm_behind_every_kind_of_plan(gpu, oracle, layout, tokens, n_out, K, splits):
    """hip_quant_gemm_add_rms_norm where the linear in front splits its k range (combine launch) and where it does not (row
    kernel): the bits of hip_quant_gemm, hip_add_bf16 and hip_rms_norm_fwd."""
    torch, dev, lib = gpu
    ptr = lambda t: ctypes.c_void_p(t.data_ptr())
    chosen = plan(LINEAR, tokens, n_out, K, fp4=layout == "fp4", row_major=layout.startswith("file"), scaled="scaled" in layout)
    assert chosen[2] == splits and chosen[4] > 1
    gen = torch.Generator(device=dev).manual_seed(tokens + n_out)
    w = Weight(gpu, oracle, layout, n_out, K, gen)
    x = (torch.randn(tokens, K, device=dev, generator=gen) * (0.05 if w.type == oracle.E5M2 else 1.0)).to(torch.bfloat16)
    res, norm = torch.randn(tokens, n_out, device=dev, generator=gen).to(torch.bfloat16), (1.0 + 0.1 * torch.randn(n_out, device=dev, generator=gen)).to(torch.bfloat16)
    try:
        o, s3, y3, s1, y1 = (torch.zeros(tokens * n_out + 64, dtype=torch.int16, device=dev) for _ in range(5))
        torch.cuda.synchronize()
        assert lib.linear(w.codes.data_ptr(), w.type, x.data_ptr(), o.data_ptr(), n_out, tokens, K, w.scale, w.scales.data_ptr() if layout == "fp4" else None, 16) == 0
        assert lib.c.hip_add_bf16(ptr(res), ptr(o), ptr(s3), tokens * n_out) == 0
        assert lib.c.hip_rms_norm_fwd(oracle.BF16, ptr(s3), ptr(y3), ptr(norm), None, tokens, n_out, ctypes.c_float(1e-6)) == 0
        assert lib.c.hip_quant_gemm_add_rms_norm(n_out, tokens, K, ptr(w.codes), w.type, K, w.scale, ptr(x), K, ptr(res), ptr(s1), ptr(norm), ptr(y1), ctypes.c_float(1e-6)) == 0
        assert np.array_equal(from_dev(s1, np.uint16), from_dev(s3, np.uint16)) and np.array_equal(from_dev(y1, np.uint16), from_dev(y3, np.uint16))
        assert s1[:tokens * n_out].any() and y1[:tokens * n_out].any()
    finally:
        w.release()
