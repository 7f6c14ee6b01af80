"""The fp32 assembly kernels on fp16 halves (opencnn_amd/csrc/gen_wino_f32_half_asm.py): CPU checks of the generator,
and on the GPU operands on both sides of the range that halves hold."""
import os
import re
import subprocess

import numpy as np
import pytest

from test_pieces import CLANG, CSRC, Replay, _run, split  # noqa: F401  (split: a fixture)

VARIANTS = [(kw, ragged, packed) for ragged, packed in ((False, False), (True, False), (True, True)) for kw in (2, 4)]


@pytest.fixture(scope="module")
def half(split):  # noqa: F811
    import importlib.util
    import sys

    sys.modules.setdefault("gen_wino_f32_split_asm", split)
    spec = importlib.util.spec_from_file_location("gen_wino_f32_half_asm", os.path.join(CSRC, "gen_wino_f32_half_asm.py"))
    mod = importlib.util.module_from_spec(spec)
    spec.loader.exec_module(mod)
    return mod


CLASSES = ["KernelHalf", "KernelQuads"]


@pytest.mark.parametrize("name", CLASSES)
@pytest.mark.parametrize("kw,ragged,packed", VARIANTS)
def test_kernel_text(half, name, kw, ragged, packed):
    k = getattr(half, name)(kw, ragged, packed)
    k.body()
    text = "\n".join(k.lines)
    assert k.vgpr_count <= 128 and k.sgpr_count <= 102
    # four chunks (first / last of a segment or not) on halves, their slow twins on pieces, two exact ones
    assert text.count("v_mfma_f32_32x32x16_f16") == text.count("v_mfma_f32_32x32x8_f16") == 4 * 8
    assert text.count("v_mfma_f32_32x32x16_bf16") == 4 * 24
    assert text.count("v_mfma_f32_32x32x2_f32") == 2 * 32
    assert all(int(n) <= 63 for n in re.findall(r"vmcnt\((\d+)\)", text))
    assert all(int(n) <= 15 for n in re.findall(r"lgkmcnt\((\d+)\)", text))
    labels = re.findall(r"^(\.L\w+):", text, re.M)
    assert len(labels) == len(set(labels))
    assert set(re.findall(r"s_c?branch\w* (\.L\w+)", text)) <= set(labels)
    # MFMA operands start on even registers; an operand is split two instructions before it is read
    lines = [l.strip() for l in k.lines]
    for i, line in enumerate(lines):
        if line.startswith("v_mfma_f32_32x32x") and "x2_f32" not in line:
            reads = [(int(a), int(b)) for a, b in re.findall(r"v\[(\d+):(\d+)\]", line)]
            assert all(a % 2 == 0 for a, _ in reads)
            for back in lines[i - 2:i]:
                m = re.match(r"v_(?!mfma|cmp)\w+ v(\d+),", back)
                assert not m or lines[i - 1] == "s_nop 1" or not any(a <= int(m.group(1)) <= b for a, b in reads), (back, line)


@pytest.mark.parametrize("name", CLASSES)
@pytest.mark.parametrize("kw,ragged,packed", VARIANTS)
def test_waits_of_a_whole_kernel_cover_its_loads(half, name, kw, ragged, packed):
    assert Replay(getattr(half, name)(kw, ragged, packed)).run() is None


@pytest.mark.parametrize("first,last", [(False, False), (True, False), (False, True), (True, True)])
@pytest.mark.parametrize("slow", [False, True])
@pytest.mark.parametrize("name,offsets", zip(CLASSES, (16, 4)))
def test_registers_that_live_through_a_chunk(half, name, offsets, first, last, slow):
    # what a segment sets up, or the output transform takes from it, no chunk writes: store offsets, patch offsets, addresses
    k = getattr(half, name)(4, True, True)
    (k.slow_chunk if slow else k.chunk)(first, last)
    live = {k.V[n] + i for n, count in (("Lane16", 1), ("Lane16Next", 1), ("EffP", 1), ("EffPrev", 1), ("Eff", 1), ("VOFF", offsets))
            for i in range(count)}
    for line in (l.strip() for l in k.lines):
        m = re.match(r"(v_(?!mfma|cmp|readf)\w+|ds_read\w+|buffer_load\w+) v\[?(\d+)(?::(\d+))?", line)
        if m:
            assert not live & set(range(int(m.group(2)), int(m.group(3) or m.group(2)) + 1)), line


@pytest.mark.skipif(not os.path.exists(CLANG), reason="ROCm LLVM assembler not installed")
def test_output_assembles_for_gfx950(tmp_path):
    src = tmp_path / "k.s"
    with open(src, "w") as f:
        subprocess.run(["python3", os.path.join(CSRC, "gen_wino_f32_half_asm.py")], check=True, stdout=f)
    subprocess.run([CLANG, "-x", "assembler", "-target", "amdgcn-amd-amdhsa", "-mcpu=gfx950", "-c", str(src),
                    "-o", str(tmp_path / "k.o")], check=True)


# ---------------------------------------------------------------- GPU
# (N, C, H, W, K): whole tiles with several segments a workgroup, pairs of filter blocks with tiles cut among workgroups, a
# ragged last chunk and filters that do not exist, packed columns, batches that break quads of images, a single group
SHAPES = [(64, 64, 40, 40, 64), (32, 256, 7, 7, 128), (33, 51, 9, 10, 300), (3, 100, 13, 11, 70), (20, 72, 15, 17, 200), (16, 136, 9, 9, 32)]
# every remainder of a quad of images, packed and not, small images whose last quad ends with the channel, and a row or column
# of tiles with a single input
BATCHES = [(n, 56, h, w, 64) for n, h, w in ((1, 5, 5), (2, 9, 4), (3, 1, 1), (4, 7, 7), (5, 2, 3), (6, 12, 11), (8, 6, 6), (12, 3, 8), (29, 5, 6),
                                              (30, 4, 5), (31, 3, 3), (35, 5, 3), (36, 4, 4))]


# packed columns that break quads of images, with the twelve units a compute unit from which such layers run on halves (the ones
# above run on pieces): one filter block, a pair of them with filters that do not exist
MANY_UNITS = [(33, 64, 56, 57, 64), (33, 56, 42, 41, 100)]


def _tensors(shape, seed):
    N, C, H, W, K = shape
    rng = np.random.default_rng(seed)
    return (np.maximum(rng.normal(size=(C, H, W, N)), 0).astype(np.float32),
            (rng.normal(size=(C, 3, 3, K)) * np.sqrt(2.0 / (9 * C))).astype(np.float32))


def _per_filter(ocn, oracle, torch, x, w, images=slice(None)):
    y, want = _run(ocn, torch, x, w).astype(np.float64)[..., images], oracle.direct_conv_f64(x, w).astype(np.float64)[..., images]
    y, want = y.reshape(y.shape[0], -1), want.reshape(want.shape[0], -1)
    return np.linalg.norm(y - want, axis=1) / np.linalg.norm(want, axis=1)


# fp32's bound at these sizes (tests/test_pieces.py): C roundings of 2^-24 and the transforms', below 1e-6; here per filter
BOUND = 2e-6


@pytest.mark.gpu
@pytest.mark.parametrize("ex,ew", [(0, 0), (-7, 0), (-9, 0), (-10, 0), (-11, 0), (-13, 0), (4, 0), (5, 0), (7, 0), (0, -10), (0, -12),
                                   (0, -13), (0, -15), (0, 3), (0, 5), (-12, 14), (8, -16)])
@pytest.mark.parametrize("shape", SHAPES)
def test_both_sides_of_the_ranges(ocn, oracle, torch_gpu, shape, ex, ew):
    # patches of 2^-10 ... 63.9 and transformed weights of 2^-17 ... 4: all units in range, some of them, none
    print(f"range {shape} 2^{ex} 2^{ew}", flush=True)
    x, w = _tensors(shape, 21)
    rel = _per_filter(ocn, oracle, torch_gpu, np.ldexp(x, ex), np.ldexp(w, ew))
    assert rel.max() <= BOUND, rel.max()


@pytest.mark.gpu
@pytest.mark.parametrize("shape", BATCHES)
def test_batches_and_quads(ocn, oracle, torch_gpu, shape):
    print(f"quads {shape}", flush=True)
    x, w = _tensors(shape, 28)
    x += 0.1 * np.random.default_rng(29).normal(size=x.shape).astype(np.float32)  # no pixel of zeros
    assert _per_filter(ocn, oracle, torch_gpu, x, w).max() <= BOUND


@pytest.mark.gpu
@pytest.mark.parametrize("shape", MANY_UNITS)
def test_broken_quads_of_images_with_many_units(ocn, oracle, torch_gpu, shape):
    # in range, out of range, and one image out of it
    for e, image in ((0, None), (-13, None), (0, shape[0] // 2)):
        print(f"odd {shape} 2^{e} {image}", flush=True)
        x, w = _tensors(shape, 31)
        x = np.ldexp(x, e)
        if image is not None:
            x[..., image] = np.ldexp(x[..., image], -25)
        assert _per_filter(ocn, oracle, torch_gpu, x, w).max() <= BOUND


@pytest.mark.gpu
@pytest.mark.parametrize("shape", SHAPES)
def test_single_operands_out_of_range(ocn, oracle, torch_gpu, shape):
    # One channel whose inputs and weights lie far apart, products like the others'; one image; one filter; a filter that sees
    # nothing but the small channel.  A unit out of range among others that are not, first, in the middle and last.
    N, C, H, W, K = shape
    for c in (0, C // 2, C - 1):
        for e in (-30, 30):
            print(f"one channel {shape} {c} {e}", flush=True)
            x, w = _tensors(shape, 22)
            x[c], w[c] = np.ldexp(x[c], e), np.ldexp(w[c], -e)
            assert _per_filter(ocn, oracle, torch_gpu, x, w).max() <= BOUND
        x, w = _tensors(shape, 23)
        x[c] = np.ldexp(x[c], -25)
        w[np.arange(C) != c, :, :, K // 3] = 0
        print(f"one filter of a small channel {shape} {c}", flush=True)
        assert _per_filter(ocn, oracle, torch_gpu, x, w).max() <= BOUND
    x, w = _tensors(shape, 24)
    x[..., N // 2] = np.ldexp(x[..., N // 2], -25)
    print(f"one image {shape}", flush=True)
    assert _per_filter(ocn, oracle, torch_gpu, x, w).max() <= BOUND
    assert _per_filter(ocn, oracle, torch_gpu, x, w, slice(N // 2, N // 2 + 1)).max() <= BOUND
    x, w = _tensors(shape, 30)
    w[..., K // 2] = 0  # stays in range
    w[::5, :, :, 1] = 0
    y_zero = _run(ocn, torch_gpu, x, w)
    assert not y_zero[K // 2].any()
    want = oracle.direct_conv_f64(x, w).astype(np.float64)
    assert np.linalg.norm(y_zero - want) <= BOUND * np.linalg.norm(want)
    for e in (-25, 25):
        x, w = _tensors(shape, 25)
        w[..., K // 2] = np.ldexp(w[..., K // 2], e)
        print(f"one filter {shape} {e}", flush=True)
        assert _per_filter(ocn, oracle, torch_gpu, x, w).max() <= BOUND


@pytest.mark.gpu
@pytest.mark.parametrize("shape", SHAPES)
def test_operands_that_pieces_of_either_scale_lose(ocn, oracle, torch_gpu, shape):
    # in one unit a channel of weights and a channel of inputs below what bf16 pieces hold without their scale, each with a
    # large partner: the poisoned tiles come from the fp32 MFMA
    C = shape[1]
    for c in (0, C // 8 * 8 - 8):
        print(f"small weights and small inputs in a unit {shape} {c}", flush=True)
        x, w = _tensors(shape, 26)
        x[c], w[c] = np.ldexp(x[c], -120), np.ldexp(w[c], 110)
        x[c + 1], w[c + 1] = np.ldexp(x[c + 1], 100), np.ldexp(w[c + 1], -113)
        assert _per_filter(ocn, oracle, torch_gpu, x, w).max() <= BOUND


@pytest.mark.gpu
@pytest.mark.parametrize("channels", [48, 49, 64, 512])
def test_errors_are_no_larger_than_on_pieces(ocn, oracle, torch_gpu, channels):
    # 48 channels still run on bf16 pieces (relative 2-norm error 1.9e-7 for 48, 5.4e-7 for 512 channels); the
    # bounds are the pieces' own errors at these sizes and data, 1.05 times for the spread between seeds
    x, w = _tensors((32, channels, 7, 7, 128), 27)
    want = oracle.direct_conv_f64(x, w).astype(np.float64)
    y = _run(ocn, torch_gpu, x, w).astype(np.float64)
    rel = np.linalg.norm(y - want) / np.linalg.norm(want)
    print(f"C={channels} rel {rel:.3e}", flush=True)
    assert rel <= 1.05 * {48: 2.0e-7, 49: 2.0e-7, 64: 2.1e-7, 512: 2.9e-7}[channels]


@pytest.mark.gpu
@pytest.mark.parametrize("shape", [(64, 64, 40, 40, 64), (32, 256, 7, 7, 128), (33, 56, 42, 41, 100), (1, 64, 14, 14, 64)])
def test_what_lds_held_before_does_not_matter(ocn, torch_gpu, shape):
    """A transpose in front of the layer leaves the compute units' LDS full of small integers, like the marks of units out of
    range: the layer's bits are the same after each of them."""
    torch = torch_gpu
    N, C, H, W, K = shape
    x, w = (torch.from_numpy(t).to("cuda:0") for t in _tensors(shape, 45))
    x += 0.5  # (every unit is in range)
    ws = torch.empty(ocn.workspace_bytes(C, K) // 4, device="cuda:0")
    ocn.filter_transform(w, ws, K, C, ocn.FILTER_CRSK, ocn.WW_MFMA)
    src = torch.empty(128 * 300000, dtype=torch.int32, device="cuda:0")
    dst = torch.empty_like(src)
    outputs = []
    for mark in [-1, *range(8), 0x7FA00000]:
        print(f"LDS of {mark} {shape}", flush=True)
        src.fill_(mark)
        y = torch.full((K * H * W * N,), float("nan"), device="cuda:0")
        ocn.nchw_to_chwn(src.view(torch.float32), dst.view(torch.float32), 128, 300000, 1, 1)
        ocn.conv_forward_desc(x, None, y, ws, N, C, H, W, K)
        torch.cuda.synchronize()
        assert bool((dst == mark).all())
        outputs.append(y)
    assert not torch.isnan(outputs[0]).any()
    assert [torch.equal(outputs[0], y) for y in outputs] == [True] * len(outputs)
