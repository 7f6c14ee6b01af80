"""Assembly kernels with cached stores of final outputs: layers whose stores fill lines in pieces."""
import pytest

PACKED = {"kw2": (33, 45, 46, 64), "kw4": (33, 32, 33, 128)}
RAGGED = {"kw2": (31, 47, 46, 64), "kw4": (60, 25, 24, 128)}
# ((N, C, H, W, K), operands): outputs past 16 MB, packed and not, for one filter block and pairs, on the fp32 MFMA, on
# pieces, on halves (batches of whole quads of images, and with enough units others) and on 2-byte operands; small
# outputs of unpacked batches below 8; an output that only just passes 16 MB and one that does not
LAYERS = [((n, c, h, w, k), "F32") for form in (PACKED, RAGGED) for n, h, w, k in form.values() for c in (9, 17)]
LAYERS += [((36, 51, 43, 43, 64), "F32"), ((36, 51, 31, 31, 128), "F32"), ((33, 64, 56, 57, 64), "F32"), ((33, 56, 42, 41, 100), "F32"),
           ((31, 51, 47, 46, 64), "F32"), ((60, 51, 25, 24, 128), "F32")]
LAYERS += [((n, 20, h, w, k), p) for form in (PACKED, RAGGED) for n, h, w, k in form.values() for p in ("F16", "BF16")]
LAYERS += [((3, 64, 14, 14, 64), "F32"), ((1, 9, 7, 7, 128), "F32"), ((5, 20, 6, 6, 64), "F32"), ((3, 20, 9, 9, 64), "F16")]
LAYERS += [((12, 9, 74, 74, 64), "F32"), ((12, 9, 73, 74, 64), "F32")]
# stored past the caches: that last one, batches of whole half lines (one of halves, for pairs), packed batches that divide 32, and
# small outputs of batches of 8 or more
PAST_CACHES = [LAYERS[-1], ((48, 9, 40, 41, 64), "F32"), ((80, 64, 25, 26, 100), "F32"), ((8, 64, 93, 93, 64), "F32"), ((9, 64, 14, 14, 64), "F32"),
               ((48, 20, 40, 41, 64), "F16"), ((8, 20, 93, 93, 64), "BF16")]
LAYERS += PAST_CACHES[1:]
# fp32: some twenty roundings of 2^-23 on a path; fp16 / bf16: both operands of a product rounded, 2^-11 / 2^-8 each
BOUNDS = {"F32": 20 * 2.0 ** -23, "F16": 2 * 2.0 ** -11, "BF16": 2 * 2.0 ** -8}


def _exact(torch, x, w):
    C, H, W, N = x.shape
    padded = torch.zeros((C, H + 2, W + 2, N), dtype=torch.float64, device=x.device)
    padded[:, 1:-1, 1:-1] = x.double()
    y = torch.zeros((w.shape[3], H * W * N), dtype=torch.float64, device=x.device)
    for r in range(3):
        for s in range(3):
            y += w[:, r, s, :].double().t().contiguous() @ padded[:, r:r + H, s:s + W].reshape(C, -1)
    return y.view(w.shape[3], H, W, N)


@pytest.mark.gpu
@pytest.mark.parametrize("shape,operands", LAYERS)
def test_layers_with_cached_stores(ocn, torch_gpu, shape, operands):
    print(f"stores {shape} {operands}", flush=True)
    torch = torch_gpu
    N, C, H, W, K = shape
    gen = torch.Generator(device="cuda:0")
    gen.manual_seed(5)
    x = torch.randn((C, H, W, N), device="cuda:0", generator=gen)
    w = torch.randn((C, 3, 3, K), device="cuda:0", generator=gen)
    raw = torch.full((K * H * W * N + 2048,), float("nan"), device="cuda:0")
    ws = torch.empty(ocn.workspace_bytes(C, K) // 4, device="cuda:0")
    runs = []
    for _ in range(2):
        raw.fill_(float("nan"))
        ocn.conv_forward_desc(x, w, raw[1024:-1024], ws, N, C, H, W, K, precision=getattr(ocn, operands))
        torch.cuda.synchronize()
        assert "_asm_" in ocn.last_kernel()
        assert ocn.last_symbol().endswith("_cached") == ((shape, operands) not in PAST_CACHES), ocn.last_symbol()
        assert torch.isnan(raw[:1024]).all() and torch.isnan(raw[-1024:]).all(), "wrote outside the output"
        assert not torch.isnan(raw[1024:-1024]).any(), "an output element was never written"
        runs.append(raw.clone())
    assert torch.equal(runs[0][1024:-1024], runs[1][1024:-1024])
    want = _exact(torch, x, w)
    y = runs[0][1024:-1024].view(K, H, W, N).double()
    rel = float((y - want).norm() / want.norm())
    assert rel <= BOUNDS[operands], rel


@pytest.mark.gpu
@pytest.mark.parametrize("operands", ["F16", "BF16"])
@pytest.mark.parametrize("H,W,packed", [(1803, 1804, True), (1804, 1804, False)])
def test_packed_store_offsets_at_their_limit(ocn, torch_gpu, H, W, packed, operands):
    # on packed columns a lane's store offset spans five images: beyond 2^31 bytes the columns stay unpacked
    print(f"packed limit H={H} W={W} {operands}", flush=True)
    torch = torch_gpu
    N, C, K = 33, 1, 5
    assert (20 * N * H * W < 2 ** 31) == packed
    gen = torch.Generator(device="cuda:0")
    gen.manual_seed(8)
    x = torch.rand((C, H, W, N), device="cuda:0", generator=gen)
    w = torch.rand((C, 3, 3, K), device="cuda:0", generator=gen)
    ws = torch.empty(ocn.workspace_bytes(C, K) // 4, device="cuda:0")
    y = torch.full((K, H, W, N), float("nan"), device="cuda:0")
    ocn.conv_forward_desc(x, w, y, ws, N, C, H, W, K, precision=getattr(ocn, operands))
    torch.cuda.synchronize()
    unwritten = int(torch.isnan(y).sum())
    assert unwritten == 0, unwritten
    # the last rows of every filter, where the offsets are largest
    want = _exact(torch, x[:, -17:], w)[:, 1:]
    rel = (y[:, -16:].double() - want).flatten(1).norm(dim=1) / want.flatten(1).norm(dim=1)
    assert float(rel.max()) <= BOUNDS[operands], rel
    assert "_asm_" in ocn.last_kernel() and ocn.last_kernel().endswith("_packed") == packed
