"""The fp32 assembly kernels on bf16 pieces (opencnn_amd/csrc/gen_wino_f32_split_asm.py): CPU checks of the
generator, and on the GPU the operands that bf16 pieces cannot hold."""
import importlib.util
import os
import re
import subprocess
import sys

import numpy as np
import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CSRC = os.path.join(ROOT, "opencnn_amd", "csrc")
CLANG = "/opt/rocm/lib/llvm/bin/clang"
VARIANTS = [(False, False), (True, False), (True, True)]  # (ragged, packed)


@pytest.fixture(scope="module")
def split():
    def load(name):
        spec = importlib.util.spec_from_file_location(name, os.path.join(CSRC, name + ".py"))
        mod = importlib.util.module_from_spec(spec)
        sys.modules.setdefault(name, mod)
        spec.loader.exec_module(mod)
        return mod
    load("gen_wino_f32_asm")
    return load("gen_wino_f32_split_asm")


@pytest.mark.parametrize("ragged,packed", VARIANTS)
@pytest.mark.parametrize("kw", [2, 4])
def test_kernel_text(split, kw, ragged, packed):
    k = split.KernelSplit(kw, ragged, packed)
    k.body()
    text = "\n".join(k.lines)
    assert k.vgpr_count <= 128 and k.sgpr_count <= 100  # two waves per SIMD: 128 + 128 accumulators
    # four chunks (first / last of a segment or not) on pieces, two exact ones
    assert text.count("v_mfma_f32_32x32x16_bf16") == 4 * 24
    assert text.count("v_mfma_f32_32x32x2_f32") == 2 * 32
    # the counted waits rely on STORES stores per output transform: plain, published, merged, merged and
    # published, exact
    assert text.count("buffer_store_dword") == 5 * split.STORES
    assert len(re.findall(r"buffer_load_dword v\d+, [^\n]* sc0 sc1", text)) == 32  # a partial tile
    assert all(int(n) <= 63 for n in re.findall(r"vmcnt\((\d+)\)", text))
    assert all(int(n) <= 15 for n in re.findall(r"lgkmcnt\((\d+)\)", text))
    labels = re.findall(r"^(\.L\w+):", text, re.M)
    assert len(labels) == len(set(labels))
    for target in re.findall(r"s_c?branch\w* (\.L\w+)", text):
        assert target in labels
    # MFMA operands start on even registers; an operand is split two instructions before it is read
    lines = [l.strip() for l in k.lines]
    for i, line in enumerate(lines):
        if not line.startswith("v_mfma_f32_32x32x16"):
            continue
        reads = [(int(a), int(b)) for a, b in re.findall(r"v\[(\d+):(\d+)\]", line)]
        assert all(a % 2 == 0 for a, _ in reads)
        for back in lines[i - 2:i]:
            m = re.match(r"v_(?!mfma)\w+ v(\d+),", back)
            assert not m or back.startswith("s_nop") or lines[i - 1] == "s_nop 1" or \
                not any(a <= int(m.group(1)) <= b for a, b in reads), (back, line)
    # every wait for a flag is bounded, and the wave that gives up stores a 1 to the status word
    polls = re.findall(r"^(\.L\w+_poll_\d+):", text, re.M)
    assert len(polls) == 1
    loop = lines[lines.index(polls[0] + ":"):][:14]
    exits = [l.split()[-1] for l in loop if "s_cbranch" in l]
    assert len(exits) == 2 and "_got_" in exits[0] and "_giveup_" in exits[1]
    block = lines[lines.index(exits[1] + ":") + 1:][:5]
    one = f"v{k.V['One']}"
    assert block[0] == f"v_mov_b32 {one}, 1" and block[1] == "s_mov_b64 exec, 1"
    assert block[2].split()[2].rstrip(",") == one and f"s[{k.S['Status']}:{k.S['Status'] + 1}]" in block[2]
    assert block[4] == f"s_branch {exits[0]}"


@pytest.mark.skipif(not os.path.exists(CLANG), reason="ROCm LLVM assembler not installed")
def test_output_assembles_for_gfx950(tmp_path):
    src = tmp_path / "k.s"
    with open(src, "w") as f:
        subprocess.run(["python3", os.path.join(CSRC, "gen_wino_f32_split_asm.py")], check=True, stdout=f)
    subprocess.run([CLANG, "-x", "assembler", "-target", "amdgcn-amd-amdhsa", "-mcpu=gfx950", "-c", str(src),
                    "-o", str(tmp_path / "k.o")], check=True)


def test_waits_of_a_chunk_cover_its_loads(split):
    """The counted waits, replayed: at every wait for a load of a steady-state chunk, the loads that may still be
    in flight (the youngest vmcnt of them) do not include the ones the next split or transform reads."""
    k = split.KernelSplit(2)
    k.chunk(False, False)
    lines = [l.strip() for l in k.lines]
    one = [l for l in lines if l]
    stream = one + one  # the second copy is the chunk in its steady state
    inflight = []
    for i, line in enumerate(stream):
        m = re.match(r"buffer_load_dword(x4)? v\[?(\d+)", line)
        if m:
            first = int(m.group(2))
            inflight.append(set(range(first, first + (4 if m.group(1) else 1))))
        m = re.match(r"s_waitcnt vmcnt\((\d+)\)", line)
        if m:
            inflight = inflight[len(inflight) - min(int(m.group(1)), len(inflight)):]
        if i >= len(one) and line.startswith("v_") and not line.startswith("v_mfma"):
            regs = {int(r) for r in re.findall(r"\bv(\d+)\b", line)}
            busy = set().union(*inflight) if inflight else set()
            assert not regs & busy, (line, sorted(regs & busy))


class Replay:
    """The counted waits of a whole kernel, on every path through its text: a register that a load or an LDS read is
    still on its way to must not be read or written.  A state is (line, global accesses in flight, LDS accesses in
    flight, what is known of Kind); accesses of a kind return in order, so vmcnt(n) leaves the n youngest."""

    def __init__(self, kernel):
        kernel.body()
        self.kind = kernel.sr("Kind")
        self.lines = [l.split(";")[0].strip() for l in kernel.lines]
        self.labels = {l[:-1]: i for i, l in enumerate(self.lines) if l.endswith(":")}

    @staticmethod
    def vgprs(text):
        regs = set()
        for first, last in re.findall(r"\bv\[(\d+):(\d+)\]", text):
            regs.update(range(int(first), int(last) + 1))
        regs.update(int(r) for r in re.findall(r"\bv(\d+)\b", text))
        return frozenset(regs)

    def run(self):
        """(line number, line, registers) of the first access that comes too early, or None."""
        parsed = []
        for l in self.lines:
            op, _, rest = l.partition(" ")
            vm, lds = op.startswith(("buffer_", "global_")), op.startswith("ds_")
            load = "_load_" in op or op.startswith("ds_read")
            dst = self.vgprs(rest.split(",")[0]) if load else frozenset()
            n = {c: int(x) for c, x in re.findall(r"(vmcnt|lgkmcnt)\((\d+)\)", rest)} if op == "s_waitcnt" else {}
            smem = op.startswith(("s_load", "s_memrealtime"))
            parsed.append((op, rest, vm, lds or smem, dst, n, self.vgprs(rest)))
        seen, todo = set(), [(0, (), (), ())]
        while todo:
            at, vm, lds, known = state = todo.pop()
            if state in seen:
                continue
            seen.add(state)
            op, rest, is_vm, is_lds, dst, n, regs = parsed[at]
            if op == "s_endpgm":
                continue
            for q in vm + lds:
                if q & regs:
                    return at, self.lines[at], sorted(q & regs)
            if is_vm:
                vm += (dst,)
            elif is_lds:
                lds += (dst,)
            if "vmcnt" in n:
                vm = vm[max(0, len(vm) - n["vmcnt"]):]
            if "lgkmcnt" in n:
                lds = lds[max(0, len(lds) - n["lgkmcnt"]):]
            if op.startswith("s_or_b32") and rest.startswith(self.kind + ","):
                known = ()
            if op.startswith("s_cbranch"):
                taken, passed = (self.labels[rest], vm, lds, known), (at + 1, vm, lds, known)
                m = re.match(r"s_bitcmp1_b32 (\w+), (\d)", self.lines[at - 1])
                if m and m.group(1) == self.kind:
                    bit, on = int(m.group(2)), op == "s_cbranch_scc1"
                    for value in (dict(known)[bit],) if bit in dict(known) else (True, False):
                        target = taken if value == on else passed
                        todo.append(target[:3] + (tuple(sorted({**dict(known), bit: value}.items())),))
                else:
                    todo += [taken, passed]
            elif op == "s_branch":
                todo.append((self.labels[rest], vm, lds, known))
            else:
                todo.append((at + 1, vm, lds, known))
        return None


@pytest.mark.parametrize("ragged,packed", VARIANTS)
@pytest.mark.parametrize("kw", [2, 4])
def test_waits_of_a_whole_kernel_cover_its_loads(split, kw, ragged, packed):
    """Prologue, chunks of every place in a segment, output transforms with and without hand-overs, the exact pass."""
    assert Replay(split.KernelSplit(kw, ragged, packed)).run() is None


def test_replay_of_the_waits_finds_a_wait_that_is_missing(split):
    """Every counted wait taken out in turn: the replay has to object, except for two waits of each of the four chunks
    that others cover: that for the patch (its last loads are read behind the wait for U1, the others arrived with U0) and
    that for the last V reads (they precede the barrier, which waits for all)."""
    replay = Replay(split.KernelSplit(2))
    lines = replay.lines
    waits = [i for i, l in enumerate(lines) if re.match(r"s_waitcnt (vmcnt|lgkmcnt)\([1-9]\d*\)$", l)]
    assert len(waits) == 36
    missed = []
    for i in waits:
        good, lines[i] = lines[i], ""
        if replay.run() is None:
            missed.append(good)
        lines[i] = good
    assert len(missed) == 8 and set(missed) == {"s_waitcnt vmcnt(2)", "s_waitcnt vmcnt(34)", "s_waitcnt lgkmcnt(8)"}, missed


@pytest.mark.parametrize("symbol,peak", [
    ("halves:wino_f32_asm_kw2", 2500.0 / 3), ("halves:wino_f32_asm_kw4_packed_odd_cached", 2500.0 / 3),
    ("pieces:wino_f32_asm_kw4_packed", 2500.0 / 6), ("fp32:wino_f32_asm_kw2", 157.3), ("wino_f32_shallow", 157.3),
    ("wino_f32_fused", 157.3), ("wino_f32_fused_lds", 157.3), ("wino_bf16_asm_kw4", 2500.0), ("wino_f16_asm_kw4_ragged_cached", 2500.0),
    ("wino_h16_fused_lds", 2500.0)])
def test_bench_prices_a_layer_against_the_kernel_that_ran(symbol, peak):
    import bench

    assert bench.matrix_peak(symbol) == peak


# ---------------------------------------------------------------- GPU
# (N, C, H, W, K): three units with a ragged last one, an odd number of column groups, packed columns, tiles cut
# between two workgroups, tiles cut among several, two filter blocks with a pair that is not full, a single group
# of filters
SHAPES = [(32, 17, 6, 6, 64), (32, 24, 5, 5, 100), (5, 33, 9, 9, 40), (64, 64, 40, 40, 64), (32, 256, 7, 7, 128),
          (33, 40, 12, 13, 300), (16, 136, 9, 9, 32), (3, 20, 14, 11, 7)]


def _run(ocn, torch, x, w, family="_asm_", **settings):
    C, H, W, N = x.shape
    K = w.shape[3]
    dev = torch.device("cuda:0")
    guard = 1024
    raw = torch.full((K * H * W * N + 2 * guard,), float("nan"), device=dev)
    ws = torch.empty(ocn.workspace_bytes(C, K) // 4, device=dev)
    ocn.conv_forward_desc(torch.from_numpy(x).to(dev), torch.from_numpy(w).to(dev), raw[guard:-guard], ws, N, C, H, W, K,
                          **settings)
    torch.cuda.synchronize()
    assert family in ocn.last_kernel()
    assert torch.isnan(raw[:guard]).all() and torch.isnan(raw[-guard:]).all(), "wrote outside the output"
    return raw[guard:-guard].cpu().numpy().reshape(K, H, W, N)


def _tensors(shape, seed):
    N, C, H, W, K = shape
    rng = np.random.default_rng(seed)
    return (rng.normal(size=(C, H, W, N)).astype(np.float32),
            (rng.normal(size=(C, 3, 3, K)) * np.sqrt(2.0 / (9 * C))).astype(np.float32))


@pytest.mark.gpu
@pytest.mark.parametrize("shape", SHAPES)
def test_every_scale_of_the_operands(ocn, oracle, torch_gpu, shape):
    # Split times 2^16, pieces hold all of fp32 below 2^112; beyond (and where outputs come out huge) the tiles are
    # computed on the fp32 MFMA.  Relative to the fp64 direct convolution every scale has fp32's accuracy: C roundings of
    # 2^-24 and the transforms' (below 1e-6 at these sizes); 2^-132 leaves 2^-17 of a denormal's bits.
    x, w = _tensors(shape, 5)
    want = oracle.direct_conv_f64(x, w).astype(np.float64)
    for ex, ew in ((0, 0), (100, 0), (-100, 0), (0, -60), (-60, 40), (60, 60), (-115, 0), (0, -115), (-60, -60)):
        print(f"scale {shape} 2^{ex} 2^{ew}", flush=True)
        y = _run(ocn, torch_gpu, np.ldexp(x, ex), np.ldexp(w, ew)).astype(np.float64)
        y = np.ldexp(y, -(ex + ew))
        rel = np.linalg.norm(y - want) / np.linalg.norm(want)
        assert rel <= 2e-6, (ex, ew, rel)


@pytest.mark.gpu
@pytest.mark.parametrize("shape", SHAPES)
def test_operands_below_the_pieces(ocn, oracle, torch_gpu, shape):
    # Denormal inputs, which bf16 pieces hold only because they are scaled, in all channels, in the first or
    # second half of them only (the other half zero: with a tile cut between workgroups, one part says
    # nothing) or in one image; denormal filters; and zeros, which are exact as they are.
    x, w = _tensors(shape, 6)
    N, C, H, W, K = shape
    tiny = np.float32(1e-41)
    cases = {"inputs": (x * tiny, w), "filters": (x, w * tiny)}
    for name, part in (("first half", slice(0, C // 2)), ("second half", slice(C // 2, C))):
        z = np.zeros_like(x)
        z[part] = x[part] * tiny
        cases[name] = (z, w)
    z = x.copy()
    z[..., N // 2] *= tiny
    cases["one image"] = (z, w)
    for name, (xx, ww) in cases.items():
        print(f"below the pieces {shape} {name}", flush=True)
        y, direct = _run(ocn, torch_gpu, xx, ww), oracle.direct_conv_f64(xx, ww)
        if name == "one image":  # the others have fp32's errors at their own scale
            y, direct = y[..., N // 2], direct[..., N // 2]
        # multiples of 2^-149: every halving of a transform and every sum rounds to that grid, fewer than 16 * C
        # of them an output, most of them far less.  An output of a step or two may come out as zero.
        assert np.abs(y.astype(np.float64) - direct).max() <= 16 * C * 2.0 ** -149
        assert (y != 0).mean() >= 0.999 * (np.abs(direct) > 4 * 2.0 ** -149).mean() > 0.9
    zero = w.copy()
    zero[..., : K // 2] = 0
    y = _run(ocn, torch_gpu, x, zero)
    assert not y[: K // 2].any() and np.isfinite(y).all()
    assert not _run(ocn, torch_gpu, np.zeros_like(x), w).any()
    assert not _run(ocn, torch_gpu, x, np.zeros_like(w)).any()


# packed columns, pairs of filter blocks: batches up to ten that break quads of lanes, few channels and few tiles keep
# the fp32 MFMA; an edge of each
PACKED = [((2, 24, 27, 27, 250), False), ((1, 40, 42, 33, 100), False), ((10, 33, 31, 33, 100), False),
          ((2, 41, 27, 27, 250), True), ((4, 24, 27, 27, 250), True), ((11, 24, 31, 41, 100), True), ((2, 24, 27, 27, 60), True),
          ((7, 24, 40, 41, 250), True)]


@pytest.mark.gpu
@pytest.mark.parametrize("shape,pieces", [(s, True) for s in SHAPES] + [((32, 16, 6, 6, 64), False), ((33, 9, 9, 9, 300), False),
                                                                       ((128, 24, 28, 28, 32), False)] + PACKED)
def test_which_layers_run_on_pieces(ocn, torch_gpu, shape, pieces):
    # Both families of fp32 kernels go by the same names.  One channel, one pixel an image and the filters' centre alone:
    # an output is a single product.  The fp32 MFMA rounds it once; six products of pieces, added up, miss that in some
    # of the elements, by a step or two.
    N, C, H, W, K = shape
    rng = np.random.default_rng(13)
    x, w = np.zeros((C, H, W, N), np.float32), np.zeros((C, 3, 3, K), np.float32)
    x[C - 1, 2, 3], w[C - 1, 1, 1] = rng.normal(size=N), rng.normal(size=K)
    family = "_kw4_packed" if (shape, pieces) in PACKED and K > 64 else "_asm_" if pieces or K > 32 else "wino_f32_fused"
    y = _run(ocn, torch_gpu, x, w, family=family)
    once = w[C - 1, 1, 1][:, None] * x[C - 1, 2, 3][None]
    steps = np.abs(y[:, 2, 3] - once) / np.spacing(np.abs(once))
    assert steps.max() <= 2 and (steps != 0).any() == pieces, (steps.max(), (steps != 0).mean())


def _per_filter(y, want):
    """Relative 2-norm error of every filter's outputs."""
    y, want = (t.reshape(t.shape[0], -1) for t in (y, want))
    return np.linalg.norm(y - want, axis=1) / np.linalg.norm(want, axis=1)


@pytest.mark.gpu
@pytest.mark.parametrize("ex,ew", [(60, -120), (100, -130), (-120, 60), (-130, 100)])
@pytest.mark.parametrize("shape", SHAPES)
def test_small_operands_times_large_ones(ocn, oracle, torch_gpu, shape, ex, ew):
    # Operands of few bits above 2^-133, where bf16 ends, times such large ones that the outputs are ordinary.
    # Bound: fp32's error (2e-6, as above), and what the two halvings of the filter transform round off denormal weights: half
    # a step of 2^-149 each, against weights of the root mean square below.
    x, w = _tensors(shape, 8)
    x, w = np.ldexp(x, ex), np.ldexp(w, ew)
    print(f"small times large {shape} 2^{ex} 2^{ew}", flush=True)
    rel = _per_filter(_run(ocn, torch_gpu, x, w).astype(np.float64), oracle.direct_conv_f64(x, w).astype(np.float64))
    assert rel.max() <= 2e-6 + 2.0 ** -149 / np.sqrt(np.mean(w.astype(np.float64) ** 2)), rel.max()


@pytest.mark.gpu
@pytest.mark.parametrize("shape", SHAPES)
def test_one_small_filter_among_ordinary_ones(ocn, oracle, torch_gpu, shape):
    # The other filters' outputs say nothing about a filter of small weights: 2^-112 ... 2^-120 hold fp32's accuracy;
    # of 2^-136 a weight has 13 bits left, and so have its outputs (below 2^-128, in steps of 2^-149).
    for ew in (-112, -120, -136):
        x, w = _tensors(shape, 9)
        k = shape[4] // 2
        w[..., k] = np.ldexp(w[..., k], ew)
        print(f"one small filter {shape} 2^{ew}", flush=True)
        y, want = _run(ocn, torch_gpu, x, w).astype(np.float64), oracle.direct_conv_f64(x, w).astype(np.float64)
        rel = _per_filter(y, want)
        assert np.delete(rel, k).max() <= 2e-6
        if ew > -130:
            assert rel[k] <= 2e-6, (ew, rel[k])
        else:  # halvings of the filter transform and sums: fewer than 16 * C steps of the grid, weighted by inputs below 6
            assert np.abs(y[k] - want[k]).max() <= 6 * 16 * shape[1] * 2.0 ** -149 and rel[k] <= 0.1, rel[k]


@pytest.mark.gpu
@pytest.mark.parametrize("zero_filters", [False, True])
@pytest.mark.parametrize("N,C,H,K", [(32, 24, 5, 7), (32, 40, 9, 64), (32, 256, 7, 128)])
def test_small_inputs_in_one_channel(ocn, oracle, torch_gpu, N, C, H, K, zero_filters):
    # The only inputs that are not zero are denormals of one channel.  With 7 filters most waves store no output; or
    # the eight filters whose outputs the wave of the channel computes are zero.
    for c in (2, C - 1):
        x, w = _tensors((N, C, H, H, K), 10)
        z = np.zeros_like(x)
        z[c] = x[c] * np.float32(1e-41)
        zero = [k for k in range(K) if k % 32 // 4 == c % 8] if zero_filters else []
        w[..., zero] = 0
        print(f"one channel N={N} C={C} H={H} K={K} c={c} {zero_filters}", flush=True)
        y, want = _run(ocn, torch_gpu, z, w), oracle.direct_conv_f64(z, w)
        assert not y[zero].any()
        # one channel: halvings and sums of 16 products, fewer than 64 steps of 2^-149 an output
        assert np.abs(y.astype(np.float64) - want).max() <= 64 * 2.0 ** -149
        keep = [k for k in range(K) if k not in zero]
        assert (y[keep] != 0).mean() > 0.9 * (np.abs(want[keep]) > 2.0 ** -149).mean()


@pytest.mark.gpu
@pytest.mark.parametrize("ex,ew", [(92, 0), (95, 0), (109, -100), (113, -113), (-90, 110), (-100, 117), (47, 47)])
@pytest.mark.parametrize("shape", SHAPES)
def test_both_sides_of_the_largest_operands(ocn, oracle, torch_gpu, shape, ex, ew):
    # outputs on both sides of 2^94, inputs and weights on both sides of 2^112
    x, w = _tensors(shape, 11)
    print(f"largest operands {shape} 2^{ex} 2^{ew}", flush=True)
    want = np.ldexp(oracle.direct_conv_f64(x, w).astype(np.float64), ex + ew)
    rel = _per_filter(_run(ocn, torch_gpu, np.ldexp(x, ex), np.ldexp(w, ew)).astype(np.float64), want)
    assert rel.max() <= 2e-6, rel.max()


@pytest.mark.gpu
@pytest.mark.parametrize("sx,sw", [(1e-19, 1e-19), (1e-38, 1.0), (1.0, 1e-38), (1e-41, 1.0)])
@pytest.mark.parametrize("shape", SHAPES)
def test_denormal_operands_and_products_keep_their_bits(ocn, oracle, torch_gpu, shape, sx, sw):
    # fp32's error and, on the grid of denormals, half a step of 2^-149 for the output and for each halving of the
    # filter transform
    x, w = _tensors(shape, 12)
    x, w = (x * np.float64(sx)).astype(np.float32), (w * np.float64(sw)).astype(np.float32)
    print(f"denormals {shape} {sx} {sw}", flush=True)
    y, want = _run(ocn, torch_gpu, x, w).astype(np.float64), oracle.direct_conv_f64(x, w).astype(np.float64)
    assert np.abs(want).max() < 1e-36
    rms = lambda t: np.sqrt(np.mean(t.astype(np.float64) ** 2))
    rel = np.linalg.norm(y - want) / np.linalg.norm(want)
    assert rel <= 2e-6 + 2.0 ** -149 / rms(want) + 2.0 ** -149 / rms(w), rel
    # (an output nearer to zero than one element's error, C roundings of 2^-24 of the terms, may come out as zero)
    assert (y[np.abs(want) > shape[1] * 2.0 ** -24 * rms(want) + 2.0 ** -148] != 0).all()


@pytest.mark.gpu
@pytest.mark.parametrize("shape", SHAPES)
def test_non_finite_operands_stay_in_their_tiles(ocn, oracle, torch_gpu, shape):
    # An infinity in the last channel: the same non-finite elements as on the fp32 MFMA everywhere (the
    # restatement of the reference's arithmetic, or, since that takes square images only, the HIP kernels, which the
    # restatement checks on square ones), finite ones as accurate as ever.
    N, C, H, W, K = shape
    x, w = _tensors(shape, 7)
    x[C - 1, H // 2, 1, N - 1] = np.inf
    x[0, 0, 0, 0] = np.nan
    print(f"non-finite {shape}", flush=True)
    y, hip = _run(ocn, torch_gpu, x, w), _run(ocn, torch_gpu, x, w, family="wino_f32_", variant=ocn.KERNEL_HIP)
    for want in [hip] + ([oracle.winograd_f32(x, w)] if H == W else []):
        assert np.isnan(want).any() and np.array_equal(np.isnan(y), np.isnan(want))
        assert np.array_equal(np.isposinf(y), np.isposinf(want)) and np.array_equal(np.isneginf(y), np.isneginf(want))
        ok = np.isfinite(want)
        rel, _, _ = oracle.compare(np.where(ok, y, 0.0), np.where(ok, want, 0.0))
        assert rel <= 2e-6, rel
