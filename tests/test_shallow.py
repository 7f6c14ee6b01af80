"""Layers of few input channels: the kernel whose tiles are one unit each (conv_kernel_shallow.hpp)."""
import numpy as np
import pytest

SEED_X, SEED_W = 11, 12


def _run(ocn, torch, x, w, offset=0, variant=None):
    C, H, W, N = x.shape
    K = w.shape[3]
    dev = torch.device("cuda:0")
    guard = 1024 + offset
    raw = torch.full((K * H * W * N + guard + 1024,), float("nan"), device=dev)
    ws = torch.empty(ocn.workspace_bytes(C, K) // 4, device=dev)
    y = raw[guard:guard + K * H * W * N]
    try:
        if variant is not None:
            ocn.set_kernel_variant(variant)
        ocn.filter_transform(torch.from_numpy(w).to(dev), ws, K, C, ocn.FILTER_CRSK, ocn.WW_MFMA)
        ocn.conv_forward_pretransformed(torch.from_numpy(x).to(dev), ws, y, N, C, H, W, K)
        torch.cuda.synchronize()
        kernel = ocn.last_kernel()
    finally:
        ocn.set_kernel_variant(ocn.KERNEL_AUTO)
    assert torch.isnan(raw[:guard]).all() and torch.isnan(raw[guard + y.numel():]).all(), "wrote outside the output"
    return y.cpu().numpy().reshape(K, H, W, N), kernel


# (N, C, H, W, K, offset of the output in floats): one of everything, each channel count on both forms and with odd
# sizes, ragged filters on full and packed columns, one to five groups of filters, outputs off the 128-byte lines, more
# tiles than workgroups with a change of the filter block inside a range, 5 ... 8 channels on a single group
SHAPES = [(1, 1, 1, 1, 1, 0), (32, 1, 5, 6, 64, 0), (32, 2, 7, 7, 96, 0), (64, 3, 9, 8, 64, 0), (32, 4, 13, 12, 160, 0),
          (1, 3, 37, 41, 64, 0), (7, 3, 10, 11, 40, 0), (33, 1, 8, 9, 256, 0), (48, 4, 6, 5, 100, 0), (32, 3, 6, 6, 33, 0),
          (32, 3, 8, 8, 64, 1), (64, 4, 5, 5, 32, 17), (32, 3, 130, 70, 192, 0), (96, 2, 40, 40, 50, 0),
          (5, 4, 90, 111, 96, 0), (32, 5, 9, 9, 32, 0), (64, 8, 40, 41, 20, 0), (3, 7, 31, 33, 32, 0), (100, 6, 12, 13, 9, 0),
          (32, 8, 100, 90, 32, 0)]


@pytest.mark.gpu
@pytest.mark.parametrize("N,C,H,W,K,offset", SHAPES)
def test_equals_the_general_kernel(ocn, oracle, torch_gpu, N, C, H, W, K, offset):
    # the same products, summed in the same order, as the register kernel of the general path: equal to the bit
    print(f"shallow N={N} C={C} H={H} W={W} K={K} offset={offset}", flush=True)
    x, w = ocn.synth_input(N, C, H, W, seed=SEED_X), ocn.synth_filter(K, C, seed=SEED_W)
    y, kernel = _run(ocn, torch_gpu, x, w, offset)
    assert kernel == "wino_f32_shallow"
    general, kernel = _run(ocn, torch_gpu, x, w, offset, ocn.KERNEL_REGISTER)
    assert kernel == "wino_f32_fused"
    assert not np.isnan(y).any(), "an output element was never written"
    assert np.array_equal(y, general)
    # fp32 operands: a relative 1.2e-7 (2^-23) per rounding, some twenty of them on a path
    rel, _, _ = oracle.compare(y, oracle.direct_conv_f64(x, w))
    assert rel <= 20 * 2.0 ** -23


@pytest.mark.gpu
@pytest.mark.parametrize("N,C,K,shallow", [(32, 4, 64, True), (32, 5, 64, False), (32, 8, 32, True), (32, 9, 32, False),
                                           (5, 8, 33, False)])
def test_layers_it_takes(ocn, torch_gpu, N, C, K, shallow):
    x, w = ocn.synth_input(N, C, 8, 8, seed=SEED_X), ocn.synth_filter(K, C, seed=SEED_W)
    _, kernel = _run(ocn, torch_gpu, x, w)
    assert (kernel == "wino_f32_shallow") == shallow
    # a variant that is asked for is not overridden
    _, kernel = _run(ocn, torch_gpu, x, w, variant=ocn.KERNEL_HIP)
    assert kernel != "wino_f32_shallow"


@pytest.mark.gpu
@pytest.mark.parametrize("N,C,K", [(32, 3, 64), (5, 1, 40), (32, 8, 32)])
def test_values_that_are_not_finite_stay_in_their_windows(ocn, torch_gpu, N, C, K):
    # padded channels, dead columns and neighbours multiply zeros or nothing: an infinity reaches the outputs of the
    # tiles whose 4x4 patch holds it, of its own image, and nothing else
    H = W = 12
    x, w = ocn.synth_input(N, C, H, W, seed=SEED_X), ocn.synth_filter(K, C, seed=SEED_W)
    want, _ = _run(ocn, torch_gpu, x, w)
    x[C - 1, 5, 6, N // 2] = np.inf
    y, _ = _run(ocn, torch_gpu, x, w)
    touched = np.zeros(y.shape, bool)
    touched[:, 4:8, 4:8, N // 2] = True  # patch rows 2t-1 ... 2t+2 hold row 5 for t = 2, 3; columns 6 the same
    assert np.array_equal(y[~touched], want[~touched])
    assert not np.isfinite(y[:, 5, 6, N // 2]).any()


@pytest.mark.gpu
@pytest.mark.parametrize("N,H,W,shallow", [(32, 1831, 1832, True), (32, 1832, 1832, False), (33, 1803, 1804, True), (33, 1804, 1804, False)])
def test_store_offsets_at_their_limit(ocn, torch_gpu, N, H, W, shallow):
    # a lane's store offset spans five images: up to 2^31 bytes this kernel, beyond the general one, with every output written
    print(f"shallow limit N={N} H={H} W={W}", flush=True)
    torch = torch_gpu
    C, K = 1, 5
    assert (20 * N * H * W < 2 ** 31) == shallow
    gen = torch.Generator(device="cuda:0")
    gen.manual_seed(7)
    x = torch.rand(C * H * W * N, device="cuda:0", generator=gen)
    w = torch.rand(C * 9 * K, device="cuda:0", generator=gen)
    ws = torch.empty(ocn.workspace_bytes(C, K) // 4, device="cuda:0")
    y = torch.full((K * H * W * N,), float("nan"), device="cuda:0")
    ocn.conv_forward_desc(x, w, y, ws, N, C, H, W, K)
    torch.cuda.synchronize()
    kernel = ocn.last_kernel()
    general = torch.full_like(y, float("nan"))
    ocn.conv_forward_desc(x, w, general, ws, N, C, H, W, K, variant=ocn.KERNEL_REGISTER)
    torch.cuda.synchronize()
    assert not torch.isnan(general).any(), "an output element was never written"
    unwritten = int(torch.isnan(y).sum())
    assert unwritten == 0, unwritten
    assert torch.equal(y, general)
    assert (kernel == "wino_f32_shallow") == shallow
