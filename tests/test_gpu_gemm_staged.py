"""The prompt GEMM with waves that only load (gemm_staged.h): every tile, unsplit and with the k range split, through the C-ABI, for the
shapes whose plan it takes over."""
import ctypes
import subprocess
import tempfile
from pathlib import Path

import pytest

from gemm_plan_util import LINEAR, PAIR, SEGMENTS
from gpu_util import MAX_REL, ROW_L2_REL
from test_gpu_gemm_tiles import Weight, widths_of

SOURCE = r"""
#include "gemm_plan.h"
using namespace ccq;
extern "C" void plan(int kind, int row_major, int scaled, int tokens, int n_out, int K, int n_segments, const int* segments, int* out)
{
    LinearArgs a{};
    a.tokens = tokens;
    a.n_out = n_out;
    a.K = K;
    a.n_segments = n_segments;
    for (int s = 0; s < n_segments; s++) { a.seg_n_out[s] = segments[s]; }
    const GemmWeights w = { false, row_major != 0, scaled != 0 };
    const GemmPlan before = plan_gemm(a, (GemmKind)kind, w, 256, true), p = staged_plan(a, (GemmKind)kind, w, 256, before, true);
    out[0] = p.mb;
    out[1] = p.nb;
    out[2] = p.splits;
    out[3] = p.staged;
    out[4] = before.splits;
}
"""

_lib = None


def plan(layout, kind, tokens, widths, K):
    """(tokens / 16, features / 64, k ranges, staged?, k ranges of plan_gemm) of the launch the library makes on 256 CUs."""
    global _lib
    if _lib is None:
        csrc = Path(__file__).resolve().parent.parent / "cccc-lite_amd" / "csrc"
        with tempfile.TemporaryDirectory() as d:
            (Path(d) / "plan.cpp").write_text(SOURCE)
            subprocess.run(["g++", "-O1", "-std=c++17", "-Wall", "-Werror", "-shared", "-fPIC", "-I", str(csrc), "plan.cpp", "-o", "plan.so"], cwd=d, check=True)
            _lib = ctypes.CDLL(str(Path(d) / "plan.so"))
    segments = widths if kind == SEGMENTS else []
    out = (ctypes.c_int * 5)()
    _lib.plan(kind, layout.startswith("file"), "scaled" in layout, tokens, 0 if segments else widths[0], K, len(segments), (ctypes.c_int * 3)(*segments), out)
    return tuple(out)


# weight layout, kind of launch, [(tokens, features, K, tokens / 16 and features / 64 of the tile, k ranges)]: token counts one past a tile
# and short of one, features 8 past a tile, K an odd number of halves of a stage (the last stage half empty) or of whole stages
CASES = [
    ("file", LINEAR, [(17, 4104, 1600, 2, 1, 1), (17, 4104, 4160, 2, 1, 3), (17, 16392, 3136, 2, 2, 1), (65, 8200, 2112, 3, 2, 1),
        (65, 2056, 8256, 3, 2, 5), (65, 72, 1600, 4, 1, 1), (400, 72, 8256, 4, 1, 4), (49, 16392, 3136, 4, 2, 1), (209, 1032, 8256, 4, 2, 4),
        (65, 16392, 1088, 5, 2, 1), (65, 5128, 4160, 5, 2, 4), (100, 16392, 1088, 7, 2, 1), (100, 6152, 8256, 7, 2, 4)]),
    ("file", PAIR, [(5, 72, 1088, 2, 1, 1), (5, 72, 2112, 2, 1, 4), (5, 8200, 2112, 2, 2, 1), (33, 5128, 2112, 3, 2, 1), (33, 1032, 8256, 3, 2, 8),
        (65, 72, 1088, 4, 1, 1), (65, 72, 2112, 4, 1, 4), (257, 1544, 3136, 4, 2, 1), (100, 2056, 8256, 4, 2, 3), (65, 8200, 1088, 5, 2, 1),
        (65, 2568, 4160, 5, 2, 4), (100, 8200, 1600, 7, 2, 1), (100, 3080, 8256, 7, 2, 4)]),
    ("file", SEGMENTS, [(17, 776, 1600, 2, 1, 1), (5, 2056, 6208, 2, 1, 4), (5, 12296, 2112, 2, 2, 1), (65, 6152, 2112, 3, 2, 1),
        (129, 776, 8256, 3, 2, 5), (512, 136, 1600, 4, 1, 1), (400, 72, 8256, 4, 1, 4), (257, 2056, 3136, 4, 2, 1), (209, 776, 8256, 4, 2, 4),
        (65, 12296, 1088, 5, 2, 1), (65, 2568, 8256, 5, 2, 6), (100, 12296, 1600, 7, 2, 1), (100, 4104, 8256, 7, 2, 4)]),
    ("tiled", LINEAR, [(17, 4104, 1600, 2, 1, 1), (65, 8200, 2112, 3, 2, 1), (129, 2056, 6208, 3, 2, 3), (65, 72, 1600, 4, 1, 1),
        (400, 136, 8256, 4, 1, 4), (100, 10248, 3136, 4, 2, 1), (65, 16392, 1088, 5, 2, 1), (65, 5128, 6208, 5, 2, 4), (100, 16392, 1088, 7, 2, 1),
        (100, 6152, 8256, 7, 2, 4)]),
    ("tiled", PAIR, [(5, 72, 1088, 2, 1, 1), (5, 72, 2112, 2, 1, 4), (5, 8200, 8256, 2, 2, 1), (65, 4104, 2112, 3, 2, 1), (65, 1544, 8256, 3, 2, 4),
        (65, 72, 1088, 4, 1, 1), (65, 72, 2112, 4, 1, 4), (449, 1032, 3136, 4, 2, 1), (65, 8200, 1088, 5, 2, 1), (65, 2568, 4160, 5, 2, 4),
        (100, 8200, 1600, 7, 2, 1), (100, 3080, 8256, 7, 2, 4)]),
    ("tiled", SEGMENTS, [(17, 776, 1600, 2, 1, 1), (65, 6152, 2112, 3, 2, 1), (65, 2568, 6208, 3, 2, 3), (512, 136, 1600, 4, 1, 1),
        (400, 72, 8256, 4, 1, 4), (400, 1544, 3136, 4, 2, 1), (65, 12296, 1088, 5, 2, 1), (65, 2568, 8256, 5, 2, 6), (100, 12296, 1600, 7, 2, 1),
        (100, 4104, 8256, 7, 2, 4)]),
    ("file_scaled", LINEAR, [(17, 5128, 1600, 2, 1, 1), (17, 8200, 6208, 2, 1, 3), (17, 16392, 3136, 2, 2, 1), (17, 12296, 8256, 2, 2, 2),
        (33, 16392, 3136, 3, 2, 1), (81, 6152, 6208, 3, 2, 2), (65, 72, 1600, 4, 1, 1), (65, 2568, 3136, 4, 1, 2), (49, 16392, 3136, 4, 2, 1),
        (65, 16392, 1088, 5, 2, 1), (65, 5128, 4160, 5, 2, 4), (100, 16392, 1600, 7, 2, 1), (100, 8200, 3136, 7, 2, 3)]),
    ("file_scaled", PAIR, [(5, 72, 1088, 2, 1, 1), (5, 72, 2112, 2, 1, 4), (5, 8200, 1600, 2, 2, 1), (5, 3080, 8256, 2, 2, 4),
        (33, 8200, 2112, 3, 2, 1), (81, 3080, 6208, 3, 2, 2), (65, 72, 1088, 4, 1, 1), (65, 72, 2112, 4, 1, 4), (49, 8200, 3136, 4, 2, 1),
        (65, 8200, 1088, 5, 2, 1), (65, 2568, 4160, 5, 2, 5), (100, 8200, 1600, 7, 2, 1), (100, 4104, 3136, 7, 2, 3)]),
    ("file_scaled", SEGMENTS, [(5, 8200, 3136, 2, 1, 1), (17, 6152, 6208, 2, 1, 3), (5, 12296, 1600, 2, 2, 1), (5, 8200, 8256, 2, 2, 2),
        (33, 12296, 3136, 3, 2, 1), (33, 6152, 8256, 3, 2, 3), (337, 264, 1600, 4, 1, 1), (65, 1544, 6208, 4, 1, 3), (49, 12296, 3136, 4, 2, 1),
        (65, 12296, 1088, 5, 2, 1), (65, 4104, 4160, 5, 2, 4), (100, 12296, 1600, 7, 2, 1), (100, 6152, 3136, 7, 2, 3)]),
    ("tiled_scaled", LINEAR, [(33, 5128, 2112, 2, 1, 1), (65, 72, 1600, 4, 1, 1), (65, 16392, 1088, 5, 2, 1), (65, 5128, 4160, 5, 2, 4),
        (100, 16392, 1600, 7, 2, 1), (100, 6152, 8256, 7, 2, 4)]),
    ("tiled_scaled", PAIR, [(5, 72, 1088, 2, 1, 1), (5, 72, 2112, 2, 1, 4), (33, 8200, 3136, 3, 2, 1), (65, 72, 1088, 4, 1, 1),
        (65, 72, 2112, 4, 1, 4), (65, 8200, 1088, 5, 2, 1), (65, 2568, 4160, 5, 2, 5), (100, 8200, 1600, 7, 2, 1), (100, 3080, 8256, 7, 2, 4)]),
    ("tiled_scaled", SEGMENTS, [(5, 10248, 3136, 2, 1, 1), (81, 10248, 6208, 3, 2, 1), (337, 264, 1600, 4, 1, 1), (225, 2568, 8256, 4, 1, 2),
        (65, 12296, 1088, 5, 2, 1), (65, 4104, 4160, 5, 2, 4), (100, 12296, 1600, 7, 2, 1), (100, 4104, 8256, 7, 2, 4)]),
]


@pytest.mark.parametrize("layout", ["file", "tiled", "file_scaled", "tiled_scaled"])
@pytest.mark.parametrize("kind", [LINEAR, PAIR, SEGMENTS])
def test_short_sums_and_long_prompts_keep_the_register_fed_kernels(layout, kind):
    """The estimate of the staged kernel is fitted from K = 1024 on; above 512 tokens the larger tiles are level or ahead."""
    for tokens in (2, 17, 100, 512, 513, 2048):
        for n_out in (72, 4096, 16384):
            widths = widths_of(n_out)
            assert not plan(layout, kind, tokens, widths, 960)[3]
            assert tokens <= 512 or not plan(layout, kind, tokens, widths, 4096)[3]


@pytest.mark.parametrize("scaled", ["", "_scaled"])
@pytest.mark.parametrize("kind", [LINEAR, PAIR, SEGMENTS])
def test_the_layouts_of_a_weight_take_the_same_sums_where_they_did(scaled, kind):
    """With the same k ranges in the plans of the file layout and of the tiled copy, either both or none take the staged kernel, and
    then with the same k ranges: the copy of a weight gives the bits of its file layout."""
    staged = 0
    for tokens in (5, 17, 64, 100, 200, 301, 512):
        for n_out in (72, 328, 1032, 4096, 12288):
            for K in (1024, 2112, 4096, 12288):
                widths = widths_of(n_out) if kind == SEGMENTS else [n_out]
                file, copy = (plan(layout + scaled, kind, tokens, widths, K) for layout in ("file", "tiled"))
                if file[4] == copy[4]:
                    assert file[2:4] == copy[2:4], (tokens, n_out, K)
                    staged += file[3]
    assert staged > 0


@pytest.mark.gpu
@pytest.mark.parametrize("layout,kind,shapes", CASES, ids=[f"{c[0]}-{('linear', 'pair', 'segments')[c[1]]}" for c in CASES])
def test_every_staged_tile_against_the_exact_contraction(gpu, oracle, layout, kind, shapes):
    """Tolerances of the other tiles' test (row L2 error 2e-3 and largest error 1e-2 of the exact contraction rounded to 16 bits; the
    SwiGLU product of two rounded linears 1e-2); nothing is written past the output.  Linears also on HALF activations, and with
    alpha, beta and rows of odd length behind padded activations (no wide store)."""
    torch, dev, lib = gpu
    assert torch.cuda.get_device_properties(0).multi_processor_count == 256
    ptr = lambda t: ctypes.c_void_p(t.data_ptr())
    for tokens, n_out, K, mb, nb, splits in shapes:
        widths = {LINEAR: [n_out], PAIR: [n_out] * 2, SEGMENTS: widths_of(n_out)}[kind]
        assert plan(layout, kind, tokens, widths, K)[:4] == (mb, nb, splits, True), (tokens, n_out, K)
        print(layout, kind, tokens, n_out, K, flush=True)
        gen = torch.Generator(device=dev).manual_seed(tokens + n_out + K)
        weights = [Weight(gpu, oracle, layout, n, K, gen) for n in widths]
        w0 = weights[0]
        x = (torch.randn(tokens, K, device=dev, generator=gen) * (0.05 if w0.type == oracle.E5M2 else 1.0)).to(torch.bfloat16)
        ld = K + 8
        padded = torch.full((tokens, ld), float("nan"), dtype=torch.bfloat16, device=dev)
        padded[:, :K] = x
        old = torch.randn(tokens, n_out + 3, device=dev, generator=gen).to(torch.bfloat16)
        try:
            for form in ("plain", "half", "strided") if kind == LINEAR else ("plain",):
                half, strided = form == "half", form == "strided"
                dtype = torch.float16 if half else torch.bfloat16
                xt = (x * 0.002).to(dtype) if half and w0.type == oracle.E5M2 else x.to(dtype)       # outputs within the range of HALF
                outs = [torch.zeros(tokens * n + 64, dtype=dtype, device=dev) for n in (widths[:1] if kind == PAIR else widths)]
                if strided: outs = [torch.cat([old.view(-1), torch.zeros(64, dtype=dtype, device=dev)])]
                torch.cuda.synchronize()
                if strided:
                    rc = lib.c.hip_quant_gemm(1, 0, n_out, tokens, K, ctypes.c_float(0.5), ptr(w0.codes), w0.type, K, ctypes.c_float(w0.scale), ptr(padded), oracle.BF16, ld,
                                              ctypes.c_float(1.0), ctypes.c_float(-0.25), ptr(outs[0]), oracle.BF16, n_out + 3, ctypes.c_float(1.0), None, None, 16)
                elif kind == LINEAR:
                    rc = lib.linear(w0.codes.data_ptr(), w0.type, xt.data_ptr(), outs[0].data_ptr(), n_out, tokens, K, w0.scale, act_type=oracle.HALF if half else oracle.BF16)
                elif kind == PAIR:
                    rc = lib.c.hip_quant_gemm_swiglu(n_out, tokens, K, ptr(w0.codes), ptr(weights[1].codes), w0.type, K, ctypes.c_float(w0.scale), ctypes.c_float(w0.scale),
                                                     ptr(xt), K, ptr(outs[0]), n_out)
                else:
                    n = (ctypes.c_int * 3)(*widths)
                    rc = lib.c.hip_quant_gemm_segments(3, n, (ctypes.c_void_p * 3)(*(w.codes.data_ptr() for w in weights)), (ctypes.c_float * 3)(*[w0.scale] * 3),
                                                       (ctypes.c_void_p * 3)(*(o.data_ptr() for o in outs)), n, w0.type, tokens, K, K, ptr(xt), K)
                assert rc == 0
                torch.cuda.synchronize()
                exact = [xt.double() @ w.exact(oracle, half).T for w in weights]
                if strided:
                    got = outs[0][:tokens * (n_out + 3)].view(tokens, n_out + 3)
                    assert torch.equal(got[:, n_out:], old[:, n_out:])
                    outs = [torch.cat([got[:, :n_out].reshape(-1), outs[0][tokens * (n_out + 3):]])]
                    exact = [0.5 * exact[0] - 0.25 * old[:, :n_out].double()]
                exact = [e.to(dtype).double() for e in exact]
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
                    assert (diff.norm(dim=1) <= ROW_L2_REL * want.norm(dim=1)).all(), (tokens, n_out, K, form)
                    assert (diff.abs().amax(dim=1) <= MAX_REL * want.abs().amax(dim=1)).all(), (tokens, n_out, K, form)
        finally:
            for w in weights: w.release()


@pytest.mark.gpu
@pytest.mark.parametrize("layout", ["file", "tiled", "file_scaled", "tiled_scaled"])
@pytest.mark.parametrize("half", [False, True])
def test_infinities_at_the_end_of_a_row(gpu, oracle, layout, half):
    """K % 128 == 64, unsplit and split: an infinity among the last activations of a row gives the infinities of the exact contraction (NaN only
    where a weight is zero), one in the last whole stage likewise, and the other rows keep the tolerances of the test above."""
    torch, dev, lib = gpu
    dtype = torch.float16 if half else torch.bfloat16
    for tokens, n_out, K in ((65, 72, 1600), (65, 16392, 1088), (100, 6152, 8256), (65, 5128, 6208)):
        before = plan(layout, LINEAR, tokens, [n_out], K)
        assert before[3], (tokens, n_out, K)
        gen = torch.Generator(device=dev).manual_seed(tokens + n_out + K)
        weight = Weight(gpu, oracle, layout, n_out, K, gen)
        x = (torch.randn(tokens, K, device=dev, generator=gen) * (0.0001 if weight.type == oracle.E5M2 else 1.0)).to(dtype)
        for token, k, value in ((0, K - 1, float("inf")), (3, K - 8, -float("inf")), (17, K - 65, float("inf")), (40, K - 4, float("inf")), (64, 0, -float("inf"))): x[token, k] = value
        y = torch.zeros(tokens, n_out, dtype=dtype, device=dev)
        try:
            torch.cuda.synchronize()
            rc = lib.linear(weight.codes.data_ptr(), weight.type, x.data_ptr(), y.data_ptr(), n_out, tokens, K, weight.scale, act_type=oracle.HALF if half else oracle.BF16)
            assert rc == 0
            torch.cuda.synchronize()
            finite = torch.isfinite(x).all(dim=1)
            assert (~finite).sum() == 5
            w = weight.exact(oracle, half)
            want = torch.where(torch.isfinite(x), x, torch.zeros_like(x)).double() @ w.T
            for token in (~finite).nonzero().flatten().tolist():
                k = (~torch.isfinite(x[token])).nonzero().item()
                want[token] += x[token, k].double() * w[:, k]
            want = want.to(dtype).double()
            got = y.double()
            assert torch.equal(torch.isnan(got), torch.isnan(want)) and torch.equal(torch.isposinf(got), torch.isposinf(want)) and torch.equal(torch.isneginf(got), torch.isneginf(want)), (tokens, n_out, K)
            diff = (got - want)[finite]
            assert (diff.norm(dim=1) <= ROW_L2_REL * want[finite].norm(dim=1)).all(), (tokens, n_out, K)
        finally:
            weight.release()


def test_no_plan_of_one_k_range_is_split():
    """A launch whose k range plan_gemm leaves whole keeps it whole on the staged kernel."""
    for layout in ("file", "tiled", "file_scaled", "tiled_scaled"):
        for kind in (LINEAR, PAIR, SEGMENTS):
            for tokens in (17, 24, 48, 80, 112, 200, 301, 512):
                for n_out in (72, 1032, 2048, 6144, 12288, 16384):
                    for K in (1024, 2112, 4096, 8192, 12288):
                        p = plan(layout, kind, tokens, widths_of(n_out) if kind == SEGMENTS else [n_out], K)
                        assert p[4] > 1 or p[2] == 1, (layout, kind, tokens, n_out, K)


@pytest.mark.gpu
@pytest.mark.parametrize("layout", ["file", "tiled", "file_scaled", "tiled_scaled"])
def test_fused_launches_give_the_bits_of_the_separate_calls(gpu, oracle, layout):
    """Where neither splits k, a gate / up pair has the bits of its two linears and their product and a joint launch those of its linears,
    also where only one of the two is the staged kernel (several of the shapes below); K a whole number of stages and half a stage more."""
    torch, dev, lib = gpu
    ptr = lambda t: ctypes.c_void_p(t.data_ptr())
    compared = mixed = 0
    for tokens, n_out, K in ((17, 12288, 2048), (20, 4096, 1088), (32, 4096, 1024), (48, 3072, 1024), (88, 4096, 1088), (100, 8192, 2112), (128, 12288, 4096), (160, 8192, 1024), (200, 12288, 1024), (400, 2048, 1088), (512, 2048, 2112)):
        print(layout, tokens, n_out, K, flush=True)
        gen = torch.Generator(device=dev).manual_seed(tokens + n_out + K)
        x = (torch.randn(tokens, K, device=dev, generator=gen) * 0.05).to(torch.bfloat16)
        for kind, widths in ((PAIR, [n_out] * 2), (SEGMENTS, widths_of(n_out))):
            fused = plan(layout, kind, tokens, widths, K)
            alone = [plan(layout, LINEAR, tokens, [n], K) for n in widths]
            if fused[2] > 1 or all(p[2] > 1 for p in alone): continue
            weights = [Weight(gpu, oracle, layout, n, K, gen) for n in widths]
            w0 = weights[0]
            try:
                single = [torch.zeros(tokens, n, dtype=torch.bfloat16, device=dev) for n in widths]
                joint = [torch.zeros_like(s) for s in (single[:1] if kind == PAIR else single)]
                torch.cuda.synchronize()
                for w, s, n in zip(weights, single, widths): assert lib.linear(w.codes.data_ptr(), w.type, x.data_ptr(), s.data_ptr(), n, tokens, K, w.scale) == 0
                if kind == PAIR:
                    product = torch.zeros_like(single[0])
                    assert lib.c.hip_swiglu_bf16(ptr(single[0]), ptr(single[1]), ptr(product), ctypes.c_ulonglong(product.numel())) == 0
                    single = [product]
                    rc = lib.c.hip_quant_gemm_swiglu(n_out, tokens, K, ptr(w0.codes), ptr(weights[1].codes), w0.type, K, ctypes.c_float(w0.scale), ctypes.c_float(w0.scale),
                                                     ptr(x), K, ptr(joint[0]), n_out)
                else:
                    n = (ctypes.c_int * 3)(*widths)
                    rc = lib.c.hip_quant_gemm_segments(3, n, (ctypes.c_void_p * 3)(*(w.codes.data_ptr() for w in weights)), (ctypes.c_float * 3)(*[w0.scale] * 3),
                                                       (ctypes.c_void_p * 3)(*(o.data_ptr() for o in joint)), n, w0.type, tokens, K, K, ptr(x), K)
                assert rc == 0
                torch.cuda.synchronize()
                for s, j, p in zip(single, joint, alone):
                    if p[2] > 1: continue
                    compared += 1
                    mixed += p[3] != fused[3]
                    assert torch.equal(s.view(torch.int16), j.view(torch.int16)), (kind, tokens, n_out, K, fused, alone)
            finally:
                for w in weights: w.release()
    assert compared >= 12 and mixed >= 4
