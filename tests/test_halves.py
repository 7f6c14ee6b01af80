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


def _simulate(items, regs, scalars):
    """The vector instructions of the range check on 64 lanes; returns vcc."""
    from test_pieces import Replay

    masks = {}
    for line in items:
        if line.startswith("s_nop"):
            continue
        op, rest = line.split(" ", 1)
        args = [a.strip() for a in rest.split(",")]

        def value(a):
            name = a.strip("|")
            x = regs[int(name[1:])] if name.startswith("v") else np.full(64, scalars[name] if name in scalars else int(name, 0) & 0xffffffff)
            return x & 0x7fffffff if a.startswith("|") else x
        if op.startswith("v_permlane"):
            a, b = (regs[int(x[1:])].reshape(-1, 32 if "lane32" in op else 16) for x in args)
            odd = a[1::2].copy()
            a[1::2], b[0::2] = b[0::2].copy(), odd
            continue  # (both are views of the registers)
        if op == "s_or_b64":
            masks["vcc"] = masks[args[1]] | masks[args[2]]
            continue
        src = [value(a).astype(np.uint32) for a in args[1:]]
        if op.startswith("v_cmp"):
            x, y = (z.view(np.float32) if op.endswith("f32") else z for z in src)
            masks[args[0]] = x > y if "_gt_" in op else x < y
            continue
        assert args[0] not in ("v0",) and Replay.vgprs(args[0])
        if op == "v_add_u32":
            out = src[0] + src[1]
        else:  # (magnitudes compare as integers do)
            out = (np.maximum if op.startswith("v_max") else np.minimum).reduce(src)
        regs[int(args[0][1:])] = out.astype(np.uint32)
    return masks["vcc"]


@pytest.mark.parametrize("name", CLASSES)
def test_patches_out_of_range(half, name):
    """The check that units carry against its definition: a patch is out of range if it has a magnitude above V_HIGH, or one of its
    four 3 x 3 windows (of an output each) has something in it but nothing of V_LOW or more."""
    k = getattr(half, name)(4, True, True)
    items = sum(k.magnitude_items("P"), []) + k.patch_range_items(1)[:3]
    low, high = np.float32(half.V_LOW), np.float32(half.V_HIGH)
    edges = np.array([0, -0.0, low, np.nextafter(low, np.float32(0)), 1e-45, high, np.nextafter(high, np.float32(100)), 1], np.float32)
    rng = np.random.default_rng(41)
    seen = set()
    for run in range(200):
        d = np.where(rng.random((64, 4, 4)) < rng.choice([0.3, 0.8, 0.97]), 0, rng.choice(edges, (64, 4, 4))).astype(np.float32)
        if run % 2:  # in range
            d = np.where(d > high, high, np.where(d < low, 0, d))
        d *= rng.choice([-1, 1], d.shape)
        m = np.abs(d)
        windows = np.array([m[:, i:i + 3, j:j + 3].max((1, 2)) for i in (0, 1) for j in (0, 1)])
        want = (m.max((1, 2)) > high) | ((windows > 0) & (windows < low)).any(0)
        regs = {i: np.zeros(64, np.uint32) for i in range(128)}
        raw = d.view(np.uint32)
        for r in range(4):
            for c in range(4):
                if name == "KernelHalf":  # a lane's own patch
                    regs[k.V["P"] + 4 * r + c] = raw[:, r, c].copy()
                else:  # lane 16 j + q: column j of the patches of columns 4 q + c
                    regs[k.V["P"] + 4 * r + c] = np.array([raw[4 * (l % 16) + c, r, l // 16] for l in range(64)])
        got = _simulate(items, regs, {k.sr("VHigh"): int(high.view(np.uint32))})
        if name == "KernelQuads":  # (each lane tells of another patch than its own)
            perm = np.array([4 * (l % 16) + (0, 2, 1, 3)[l // 16] for l in range(64)])
            assert np.array_equal(got, want[perm])
        else:
            assert np.array_equal(got, want)
        seen |= set(want)
    assert seen == {False, True}


def test_rows_and_columns_that_no_output_sees(half):
    """Behind the last output row or column of an odd size, a patch's last row / column repeats its first one."""
    k = half.KernelHalf(4, True, True)
    k.patch_offsets()
    moves = [re.match(r"\s*v_cndmask_b32 v(\d+), v(\d+), v(\d+), vcc", l) for l in k.lines]
    first = k.V["VOFF"]
    moves = [(int(m[1]) - first, int(m[3]) - first) for m in moves if m and m[1] == m[2] and 0 <= int(m[1]) - first < 16]
    assert moves == [(12 + c, c) for c in range(4)] + [(4 * r + 3, 4 * r) for r in range(4)]
    k = half.KernelQuads(4, True, True)
    k.patch_offsets()
    v = k.V["VOFF"]
    assert f"v_cndmask_b32 v{v + 3}, v{v + 3}, v{v}, vcc" in k.lines[-1]


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
@pytest.mark.parametrize("ex,ew", [(0, 0), (-7, 0), (-9, 0), (-10, 0), (-11, 0), (-12, 0), (-13, 0), (-14, 0), (2, 0), (3, 0), (4, 0), (5, 0), (7, 0), (0, -10), (0, -12),
                                   (0, -13), (0, -15), (0, 3), (0, 5), (-12, 14), (8, -16)])
@pytest.mark.parametrize("shape", SHAPES)
def test_both_sides_of_the_ranges(ocn, oracle, torch_gpu, shape, ex, ew):
    # windows of 2^-11 ... 63.9 and pairs of transformed weights of 2^-14 ... 4: all units in range, some of them, none
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
        assert "_packed_odd" in ocn.last_symbol()


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


# fp32 layers on either side of every line between the assembly kernels
SYMBOLS = [((32, 16, 14, 14, 64), "fp32:wino_f32_asm_kw2"), ((32, 17, 14, 14, 64), "pieces:wino_f32_asm_kw2_ragged"),
           ((32, 48, 7, 7, 128), "pieces:wino_f32_asm_kw4"), ((32, 49, 7, 7, 128), "halves:wino_f32_asm_kw4_ragged"),
           ((32, 56, 7, 7, 128), "halves:wino_f32_asm_kw4"), ((64, 64, 40, 40, 64), "halves:wino_f32_asm_kw2"),
           # whole quads of images; broken ones below and above twelve units a compute unit
           ((20, 72, 15, 17, 200), "halves:wino_f32_asm_kw4_packed"), ((16, 136, 9, 9, 32), "halves:wino_f32_asm_kw2_packed"),
           ((3, 100, 13, 11, 70), "pieces:wino_f32_asm_kw4_packed"), ((33, 128, 14, 14, 128), "pieces:wino_f32_asm_kw4_packed"),
           ((7, 64, 112, 112, 64), "pieces:wino_f32_asm_kw2_packed_cached"),
           ((33, 64, 56, 57, 64), "halves:wino_f32_asm_kw2_packed_odd_cached"),
           ((33, 56, 42, 41, 100), "halves:wino_f32_asm_kw4_packed_odd_cached"), ((17, 472, 28, 28, 64), "halves:wino_f32_asm_kw2_packed_odd"),
           ((17, 456, 28, 28, 64), "pieces:wino_f32_asm_kw2_packed"),
           # batches that are not packed need no whole quads
           ((33, 51, 9, 10, 300), "halves:wino_f32_asm_kw2_ragged"), ((1, 64, 14, 14, 64), "halves:wino_f32_asm_kw2_ragged_cached")]


@pytest.mark.gpu
@pytest.mark.parametrize("shape,symbol", SYMBOLS)
def test_which_kernel_runs(ocn, torch_gpu, shape, symbol):
    _run(ocn, torch_gpu, *_tensors(shape, 47))
    assert ocn.last_symbol() == symbol
    assert ocn.last_kernel() == symbol.split(":")[1].replace("_odd", "").replace("_cached", "")


@pytest.mark.gpu
@pytest.mark.parametrize("channels", [48, 49, 64, 512])
def test_errors_are_no_larger_than_on_pieces(ocn, oracle, torch_gpu, channels):
    # 48 channels still run on bf16 pieces (relative 2-norm error 1.9e-7 for 48, 5.4e-7 for 512 channels); the
    # bounds are the pieces' own errors at these sizes and data, 1.05 times for the spread between seeds
    x, w = _tensors((32, channels, 7, 7, 128), 27)
    want = oracle.direct_conv_f64(x, w).astype(np.float64)
    y = _run(ocn, torch_gpu, x, w).astype(np.float64)
    assert ocn.last_symbol().startswith("halves:" if channels > 48 else "pieces:")
    rel = np.linalg.norm(y - want) / np.linalg.norm(want)
    print(f"C={channels} rel {rel:.3e}", flush=True)
    assert rel <= 1.05 * {48: 2.0e-7, 49: 2.0e-7, 64: 2.1e-7, 512: 2.9e-7}[channels]


# quads of images, whole and ragged, tiles of one segment; packed columns; the kernels for broken quads
BRIGHT_SHAPES = [(32, 64, 8, 8, 64), (20, 72, 9, 11, 70), (33, 56, 42, 41, 100)]


@pytest.mark.gpu
@pytest.mark.parametrize("sparse", [False, True])
@pytest.mark.parametrize("e", [-9, -13, -20, -27, -40, -60])
@pytest.mark.parametrize("shape", BRIGHT_SHAPES)
def test_outputs_next_to_a_brighter_region(ocn, oracle, torch_gpu, shape, e, sparse):
    """Rows, columns and pixels of magnitude 1 on a background of 2^e: an output has fp32's accuracy relative to what its own
    3 x 3 window holds, also where its tile's patch holds something brighter.  One norm per output pixel."""
    N, C, H, W, K = shape
    rng = np.random.default_rng(43)
    base = rng.uniform(1, 2, size=(C, H, W, N)) * rng.choice([-1, 1], (C, H, W, N))
    if sparse:  # the background's windows hold one pixel or none
        base *= rng.random((C, H, W, N)) < 0.1
    w = _tensors(shape, 44)[1]
    for where in ((slice(1, 2), slice(None)), (slice(4, 5), slice(None)), (slice(None), slice(3, 4)), (slice(None), slice(6, 7)),
                  (slice(3, 4), slice(3, 4)), (slice(2, 3), slice(5, 6)), (slice(5, 8), slice(0, 2))):
        print(f"bright {shape} 2^{e} {sparse} {where}", flush=True)
        x = np.ldexp(base, e)
        x[(slice(None), *where)] = rng.normal(size=x[(slice(None), *where)].shape)
        x = x.astype(np.float32)
        y, want = _run(ocn, torch_gpu, x, w).astype(np.float64), oracle.direct_conv_f64(x, w).astype(np.float64)
        error, size = np.sqrt(((y - want) ** 2).sum((0, 3))), np.sqrt((want ** 2).sum((0, 3)))
        assert (error <= BOUND * size).all(), (error / size).max()


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


def _tight(shape, ex, ew, seed):
    """Inputs and weights of magnitudes 2^e ... 2^(e + 1): all windows on one side of a bound."""
    N, C, H, W, K = shape
    rng = np.random.default_rng(seed)
    draw = lambda e, *size: np.ldexp(rng.uniform(1, 2, size=size) * rng.choice([-1, 1], size), e).astype(np.float32)
    return draw(ex, C, H, W, N), draw(ew, C, 3, 3, K)


@pytest.mark.gpu
@pytest.mark.parametrize("channels", [51, 64, 128, 256])
@pytest.mark.parametrize("ex,ew", [(-9, -3), (-10, -3), (-11, -3), (-12, -3), (4, -3), (5, -3), (6, -3), (-1, -11), (-1, -12), (-1, -13), (-1, -14),
                                   (-1, -15), (-1, -16), (-1, -17), (-1, 0), (-1, 1), (-1, 2), (-11, -13), (-11, -14), (5, -14)])
def test_errors_at_the_edges_of_the_ranges(ocn, oracle, torch_gpu, channels, ex, ew):
    """Just inside and just outside each bound the worst filter errs hardly more than at a scale that no bound comes near
    (numbers scaled by powers of two err exactly alike in fp32): units that fall to pieces have 1.1 times the halves' error, and
    near a bound halves lose up to 2^-24 of a window's largest input or a pair's larger weight, next to roundings of 2^-22."""
    shape = (32, channels, 9, 10, 128)
    x, w = _tight(shape, 0, 0, 46)
    middle = _per_filter(ocn, oracle, torch_gpu, np.ldexp(x, -1), np.ldexp(w, -3)).max()
    edge = _per_filter(ocn, oracle, torch_gpu, np.ldexp(x, ex), np.ldexp(w, ew)).max()
    print(f"edge C={channels} 2^{ex} 2^{ew}: {edge:.3e}, in the middle {middle:.3e}", flush=True)
    assert edge <= 1.15 * middle
