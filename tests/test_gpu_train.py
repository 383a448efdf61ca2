"""The rest of the op namespace (sigmoid_mul, cross_entropy) and the backward of every
differentiable op, through the C-ABI, against torch.autograd on the CPU oracle in fp32.

fp32 cases use the reference's own test shapes and tolerances (tests/test_kernels.py:29-39,
69-79, 109-126, 166-179, 210-250). bf16 cases run at layer sizes; their gradients are
checked relative to the gradient's scale (bf16 rounds every output once: max error within
1.5% of the largest |reference|, mean error within 0.5% of the mean |reference|). Every
backward is also run twice and compared bit for bit (fixed-order reductions, no atomics).
"""
import pytest
import torch
import torch.nn.functional as F

from oracle import ops as O
from qwen3_5_vl_cuda_custom_amd import kernels as K
from tests.parity import assert_bf16_close, assert_close

pytestmark = pytest.mark.gpu
DEV = "cuda"


def rnd(*shape, seed=0, std=1.0, dtype=torch.float32):
    g = torch.Generator().manual_seed(seed)
    return (torch.randn(*shape, generator=g) * std).to(dtype)


def run_grads(fn, inputs, dy, device=DEV, dtype=None):
    """Gradients of sum(fn(*inputs) * dy) w.r.t. the float inputs (computed on `device`)."""
    with torch.enable_grad():
        # fresh leaves every call: .to() alone returns the caller's tensor when nothing changes
        xs = [t.detach().to(device=device, dtype=dtype or t.dtype).clone().requires_grad_(True)
              if t.is_floating_point() else t.to(device) for t in inputs]
        out = fn(*xs)
        out.backward(dy.to(device).to(out.dtype))
    return out.detach(), [x.grad for x in xs if x.is_floating_point()]


def ref_grads(fn, inputs, dy):
    return run_grads(fn, [t.float() if t.is_floating_point() else t for t in inputs], dy.float(), device="cpu")


def assert_grad_close(got, ref, what, max_rel=1.5e-2, mean_rel=5e-3):
    g, r = got.float().cpu(), ref.float().cpu()
    err = (g - r).abs()
    scale = float(r.abs().max())
    assert float(err.max()) <= max_rel * scale + 1e-12, f"{what}: max err {float(err.max()):.3e} vs scale {scale:.3e}"
    assert float(err.mean()) <= mean_rel * float(r.abs().mean()) + 1e-12, f"{what}: mean err {float(err.mean()):.3e}"


def twice_equal(fn):
    a, b = fn(), fn()
    for x, y in zip(a, b):
        assert torch.equal(x, y), "backward must be bitwise reproducible"


# ------------------------------------------------------------------ sigmoid_mul
def test_sigmoid_mul_reference_shapes_fp32():
    x, g = rnd(8, 128, seed=1), rnd(8, 128, seed=2)
    assert_close(K.sigmoid_mul(x.to(DEV), g.to(DEV)), O.sigmoid_mul(x, g), atol=1e-4, what="sigmoid_mul")
    x, g, dy = rnd(4, 64, seed=3), rnd(4, 64, seed=4), rnd(4, 64, seed=5)
    _, (gx, gg) = run_grads(K.sigmoid_mul, [x, g], dy)
    _, (rx, rg) = ref_grads(O.sigmoid_mul, [x, g], dy)
    assert_close(gx, rx, atol=1e-4, what="sigmoid_mul dx")
    assert_close(gg, rg, atol=1e-4, what="sigmoid_mul dgate")


def test_sigmoid_mul_bf16():
    x, g, dy = rnd(64, 1000, seed=6), rnd(64, 1000, seed=7, std=3.0), rnd(64, 1000, seed=8)
    xb, gb = x.bfloat16(), g.bfloat16()
    assert_bf16_close(K.sigmoid_mul(xb.to(DEV), gb.to(DEV)), O.sigmoid_mul(xb.float(), gb.float()), what="sm bf16")
    _, (gx, gg) = run_grads(K.sigmoid_mul, [xb, gb], dy.bfloat16())
    _, (rx, rg) = ref_grads(O.sigmoid_mul, [xb, gb], dy.bfloat16())
    assert_grad_close(gx, rx, "sigmoid_mul dx bf16")
    assert_grad_close(gg, rg, "sigmoid_mul dgate bf16")


# ------------------------------------------------------------------ cross_entropy
@pytest.mark.parametrize("ignore", [False, True])
def test_cross_entropy_reference_shapes_fp32(ignore):
    logits = rnd(16, 100, seed=10)
    tg = torch.randint(0, 100, (16,), generator=torch.Generator().manual_seed(11))
    if ignore:
        tg[[1, 5, 9]] = -100
    loss = K.cross_entropy(logits.to(DEV), tg.to(DEV))
    assert loss.dtype == torch.float32 and loss.dim() == 0
    assert_close(loss, O.cross_entropy(logits, tg), atol=1e-4, what="cross_entropy")
    assert_close(loss, F.cross_entropy(logits, tg), atol=1e-4, what="vs F.cross_entropy")
    with torch.enable_grad():
        lg = logits.to(DEV).requires_grad_(True)
        K.cross_entropy(lg, tg.to(DEV)).backward()
        lr = logits.clone().requires_grad_(True)
        O.cross_entropy(lr, tg).backward()
    assert_close(lg.grad, lr.grad, atol=1e-4, what="cross_entropy grad")


def test_cross_entropy_all_ignored_is_zero_and_grad_scale():
    logits = rnd(8, 50, seed=12).to(DEV)
    tg = torch.full((8,), -100, dtype=torch.int64, device=DEV)
    assert float(K.cross_entropy(logits, tg)) == 0.0
    # an upstream gradient of 3 scales the logits' gradient by 3 (read on the device)
    tg = torch.arange(8, device=DEV)
    with torch.enable_grad():
        a = logits.clone().requires_grad_(True)
        (3.0 * K.cross_entropy(a, tg)).backward()
        b = logits.clone().requires_grad_(True)
        K.cross_entropy(b, tg).backward()
    assert torch.allclose(a.grad, 3.0 * b.grad, rtol=1e-6, atol=0)


def test_cross_entropy_vocab_size_bf16():
    """4096 x 151,936 bf16 logits (the Qwen3-VL vocabulary): loss and sampled gradient rows."""
    N, V = 4096, 151936
    gd = torch.Generator(device=DEV).manual_seed(13)
    logits = (torch.randn(N, V, generator=gd, device=DEV) * 2.0).to(torch.bfloat16)
    tg = torch.randint(0, V, (N,), generator=gd, device=DEV)
    tg[::17] = -100
    with torch.enable_grad():
        lg = logits.clone().requires_grad_(True)
        loss = K.cross_entropy(lg, tg)
        loss.backward()
    lc, tc = logits.float().cpu(), tg.cpu()
    ref = O.cross_entropy(lc, tc)
    assert abs(float(loss) - float(ref)) <= 1e-4 * abs(float(ref)), (float(loss), float(ref))
    n_valid = int((tc != -100).sum())
    rows = [0, 1, 17, 1000, 4095]
    sm = torch.softmax(lc[rows], dim=-1)
    for j, r in enumerate(rows):
        want = torch.zeros(V) if int(tc[r]) == -100 else sm[j].clone()
        if int(tc[r]) != -100:
            want[int(tc[r])] -= 1.0
        assert_grad_close(lg.grad[r], want / n_valid, f"ce grad row {r}")
    twice_equal(lambda: (K.cross_entropy(logits, tg).reshape(1),))


# ------------------------------------------------------------------ norms, softmax, elementwise
def test_rmsnorm_backward_reference_shape_fp32():
    x, w, dy = rnd(4, 256, seed=20), rnd(256, seed=21), rnd(4, 256, seed=22)
    _, (gx, gw) = run_grads(lambda a, b: K.rmsnorm(a, b, 1e-6), [x, w], dy)
    _, (rx, rw) = ref_grads(lambda a, b: O.rmsnorm(a, b, 1e-6), [x, w], dy)
    assert_close(gx, rx, atol=1e-4, what="rmsnorm dx")
    assert_close(gw, rw, atol=1e-4, what="rmsnorm dw")


@pytest.mark.parametrize("rows,cols", [(512, 4096), (1000, 128), (33, 2048)])
def test_rmsnorm_backward_bf16(rows, cols):
    x, w, dy = rnd(rows, cols, seed=23).bfloat16(), (1 + 0.1 * rnd(cols, seed=24)).bfloat16(), rnd(rows, cols, seed=25)
    _, (gx, gw) = run_grads(lambda a, b: K.rmsnorm(a, b, 1e-6), [x, w], dy.bfloat16())
    _, (rx, rw) = ref_grads(lambda a, b: O.rmsnorm(a, b, 1e-6), [x, w], dy.bfloat16())
    assert_grad_close(gx, rx, "rmsnorm dx bf16")
    assert_grad_close(gw, rw, "rmsnorm dw bf16")
    twice_equal(lambda: run_grads(lambda a, b: K.rmsnorm(a, b, 1e-6), [x, w], dy.bfloat16())[1])


@pytest.mark.parametrize("rows,cols,dtype", [(4, 256, torch.float32), (3136, 1152, torch.bfloat16)])
def test_layernorm_backward(rows, cols, dtype):
    x, dy = rnd(rows, cols, seed=26, dtype=dtype), rnd(rows, cols, seed=29, dtype=dtype)
    w, b = (1 + 0.1 * rnd(cols, seed=27)).to(dtype), (0.1 * rnd(cols, seed=28)).to(dtype)
    _, (gx, gw, gb) = run_grads(lambda a, c, d: K.layernorm(a, c, d, 1e-6), [x, w, b], dy)
    _, (rx, rw, rb) = ref_grads(lambda a, c, d: O.layernorm(a, c, d, 1e-6), [x, w, b], dy)
    if dtype == torch.float32:
        for a, r, n in ((gx, rx, "dx"), (gw, rw, "dw"), (gb, rb, "db")):
            assert_close(a, r, atol=1e-4, what=f"layernorm {n}")
    else:
        for a, r, n in ((gx, rx, "dx"), (gw, rw, "dw"), (gb, rb, "db")):
            assert_grad_close(a, r, f"layernorm {n} bf16")


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("rows,cols", [(1, 8), (70, 128), (17, 136), (9, 520), (30, 1032), (5, 1152), (6, 2048),
                                       (3, 2056), (700, 4096), (2, 4104), (3, 8192), (2, 8200), (40, 127)])
def test_norm_backward_row_lengths(rows, cols, dtype):
    """Every instance of the norm backward (a row in 16 lanes, a wave, a block; rows it leaves to the scalar kernel)
    at both sides of its range, more rows than one pass of the grid, and both norms."""
    x, dy = rnd(rows, cols, seed=26, dtype=dtype), rnd(rows, cols, seed=29, dtype=dtype)
    w, b = (1 + 0.1 * rnd(cols, seed=27)).to(dtype), (0.1 * rnd(cols, seed=28)).to(dtype)
    got = list(run_grads(lambda a, c: K.rmsnorm(a, c, 1e-6), [x, w], dy)[1])
    got += run_grads(lambda a, c, d: K.layernorm(a, c, d, 1e-6), [x, w, b], dy)[1]
    ref = list(ref_grads(lambda a, c: O.rmsnorm(a, c, 1e-6), [x, w], dy)[1])
    ref += ref_grads(lambda a, c, d: O.layernorm(a, c, d, 1e-6), [x, w, b], dy)[1]
    for a, r, n in zip(got, ref, ("rms dx", "rms dw", "ln dx", "ln dw", "ln db")):
        if dtype == torch.float32:  # sums of up to 8200 (columns) or 700 (rows) fp32 terms of magnitude ~1
            assert_close(a, r, atol=1e-4, what=n)
        else:
            assert_grad_close(a, r, f"{n} bf16 {rows}x{cols}")


@pytest.mark.parametrize("N,V", [(3, 8), (5, 2048 * 4 + 24), (7, 1001), (2, 70000)])
def test_cross_entropy_rows_and_masked_logits_bf16(N, V):
    """Vector and scalar rows, a row shorter than a block, and logits masked with -inf (also a whole thread's share)."""
    x = rnd(N, V, seed=96, std=3.0).bfloat16()
    x[:, : V // 2] = float("-inf")
    tg = torch.full((N,), V - 1)
    if N > 2:
        tg[1] = -100
    with torch.enable_grad():
        a = x.to(DEV).requires_grad_(True)
        loss = K.cross_entropy(a, tg.to(DEV))
        loss.backward()
        r = x.double().requires_grad_(True)
        want = F.cross_entropy(r, tg)
        want.backward()
    assert abs(float(loss) - float(want)) <= 1e-5 * abs(float(want))
    assert torch.isfinite(a.grad).all()
    # one bf16 rounding of each value, and fp32 rounding of probabilities up to 1
    err = (a.grad.double().cpu() - r.grad).abs()
    assert bool((err <= 2.0 ** -8 * r.grad.abs() + 2.0 ** -20).all())


@pytest.mark.parametrize("V", [1, 3, 255, 257, 1023, 1025, 2049, 5003])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_cross_entropy_scalar_rows(V, dtype):
    """Rows that are no whole 16-byte pieces, around the 4 x 256 values of one pass: the loss and its gradient against
    float64 (the bounds of the test above; fp32 gradients 2^-20), masked values, and a NaN, which the loss keeps."""
    x = rnd(3, V, seed=97, std=2.0).to(dtype)
    x[0, V // 3:-1] = float("-inf")
    tg = torch.tensor([V - 1, V // 2, 0])
    with torch.enable_grad():
        a, r = x.to(DEV).requires_grad_(True), x.double().requires_grad_(True)
        loss, want = K.cross_entropy(a, tg.to(DEV)), F.cross_entropy(r, tg)
        loss.backward()
        want.backward()
    assert abs(float(loss) - float(want)) <= 1e-5 * max(1e-2, abs(float(want)))
    ulp = 2.0 ** -8 if dtype == torch.bfloat16 else 2.0 ** -20
    assert bool(((a.grad.double().cpu() - r.grad).abs() <= ulp * r.grad.abs() + 2.0 ** -20).all())
    x[1, V - 1] = float("nan")
    assert torch.isnan(K.cross_entropy(x.to(DEV), tg.to(DEV)))


@pytest.mark.parametrize("rows,cols,dtype", [(8, 256, torch.float32), (4096, 128, torch.bfloat16)])
def test_softmax_backward(rows, cols, dtype):
    x, dy = rnd(rows, cols, seed=30, dtype=dtype), rnd(rows, cols, seed=31, dtype=dtype)
    _, (gx,) = run_grads(K.softmax, [x], dy)
    _, (rx,) = ref_grads(O.softmax, [x], dy)
    if dtype == torch.float32:
        assert_close(gx, rx, atol=1e-5, what="softmax dx")
    else:
        assert_grad_close(gx, rx, "softmax dx bf16")


@pytest.mark.parametrize("n,dtype", [((8, 128), torch.float32), ((64, 12288), torch.bfloat16)])
def test_swiglu_and_gelu_backward(n, dtype):
    a, b, dy = rnd(*n, seed=32, dtype=dtype), rnd(*n, seed=33, dtype=dtype), rnd(*n, seed=34, dtype=dtype)
    _, (ga, gb) = run_grads(K.swiglu, [a, b], dy)
    _, (ra, rb) = ref_grads(O.swiglu, [a, b], dy)
    _, (gg,) = run_grads(K.gelu_tanh, [a], dy)
    _, (rg,) = ref_grads(O.gelu_tanh, [a], dy)
    _, (g1, g2) = run_grads(K.residual_add, [a, b], dy)
    if dtype == torch.float32:
        assert_close(ga, ra, atol=1e-4, what="swiglu dgate")
        assert_close(gb, rb, atol=1e-4, what="swiglu dup")
        assert_close(gg, rg, atol=1e-4, what="gelu dx")
    else:
        assert_grad_close(ga, ra, "swiglu dgate bf16")
        assert_grad_close(gb, rb, "swiglu dup bf16")
        assert_grad_close(gg, rg, "gelu dx bf16")
    assert torch.equal(g1, dy.to(DEV)) and torch.equal(g2, dy.to(DEV))


# ------------------------------------------------------------------ GEMMs
def test_matmul_backward_reference_shape_fp32():
    x, w, b, dy = rnd(8, 64, seed=40), rnd(32, 64, seed=41), rnd(32, seed=42), rnd(8, 32, seed=43)
    _, (gx, gw, gb) = run_grads(K.matmul, [x, w, b], dy)
    _, (rx, rw, rb) = ref_grads(O.linear, [x, w, b], dy)
    for a, r, n in ((gx, rx, "dx"), (gw, rw, "dw"), (gb, rb, "db")):
        assert_close(a, r, atol=1e-3, what=f"matmul {n}")


@pytest.mark.parametrize("shape", [(2, 256, 1024, 768), (1, 300, 520, 264), (1, 32, 4096, 4096)])
def test_matmul_backward_bf16(shape):
    B, S, K_, N = shape
    x, w = rnd(B, S, K_, seed=44).bfloat16(), rnd(N, K_, seed=45, std=0.02).bfloat16()
    b, dy = rnd(N, seed=46, std=0.02).bfloat16(), rnd(B, S, N, seed=47).bfloat16()
    _, (gx, gw, gb) = run_grads(K.matmul, [x, w, b], dy)
    _, (rx, rw, rb) = ref_grads(O.linear, [x, w, b], dy)
    for a, r, n in ((gx, rx, "dx"), (gw, rw, "dw"), (gb, rb, "db")):
        assert_grad_close(a, r, f"matmul {n} bf16 {shape}")
    twice_equal(lambda: run_grads(K.matmul, [x, w, b], dy)[1])


@pytest.mark.parametrize("M,N,K_", [(33, 72, 64), (63, 64, 136), (65, 200, 72), (127, 24, 40), (1023, 264, 520),
                                    (77, 61, 64)])
def test_matmul_backward_odd_rows_bf16(M, N, K_):
    """Token counts that are no multiple of 8 (the padded transposes), on both sides of the 64-row tiles, and an
    output width that is none (the scalar transpose and SIMT GEMM)."""
    x, w = rnd(M, K_, seed=44).bfloat16(), rnd(N, K_, seed=45, std=0.1).bfloat16()
    b, dy = rnd(N, seed=46, std=0.1).bfloat16(), rnd(M, N, seed=47).bfloat16()
    _, (gx, gw, gb) = run_grads(K.matmul, [x, w, b], dy)
    _, (rx, rw, rb) = ref_grads(O.linear, [x, w, b], dy)
    for a, r, n in ((gx, rx, "dx"), (gw, rw, "dw"), (gb, rb, "db")):
        assert_grad_close(a, r, f"matmul {n} bf16 {(M, N, K_)}")


@pytest.mark.parametrize("M,N,K_", [(1, 8, 8), (63, 136, 264), (64, 264, 136), (65, 520, 248), (129, 1032, 776),
                                    (300, 4096, 1160), (40, 8192, 512), (1000, 512, 2056), (33, 40, 16456),
                                    (1, 4304, 1152), (2, 8208, 40), (17, 4104, 520), (32, 3456, 264),
                                    (4104, 24, 520), (2056, 8, 264), (4097, 264, 136)])
def test_matmul_backward_untransposed_against_transposed(M, N, K_):
    """dX and dW on the operands as they are (tile edges in every dimension, the three tile shapes, splits over K with
    a shorter last split, also of products of at most 32 rows) against q3_matmul on transposed copies, which sums each element's products in fp32 too: the
    two may differ by one bf16 rounding of the element (2^-7) and the fp32 sums' order (2^-16 of the largest)."""
    x, w, dy = (rnd(M, K_, seed=44).bfloat16().to(DEV), rnd(N, K_, seed=45, std=0.1).bfloat16().to(DEV),
                rnd(M, N, seed=47).bfloat16().to(DEV))
    _, (gx, gw) = run_grads(K.matmul, [x, w], dy)
    pad = (-M) % 8
    zeros = lambda t: torch.cat([t, torch.zeros(pad, t.shape[1], dtype=t.dtype, device=t.device)])  # noqa: E731
    rx = K.matmul(dy, w.t().contiguous())
    rw = K.matmul(zeros(dy).t().contiguous(), zeros(x).t().contiguous())
    for a, b, n in ((gx, rx, "dx"), (gw, rw, "dw")):
        a, b = a.float(), b.float()
        over = float(((a - b).abs() - 2.0 ** -7 * b.abs() - 2.0 ** -16 * b.abs().max()).max())
        assert over <= 0, f"{n} {(M, N, K_)}: {over:.3e} over"


@pytest.mark.parametrize("M,N", [(1, 40), (256, 40), (257, 40), (64, 5000), (1024, 4096), (1025, 4096), (1088, 4104),
                                 (300, 77), (1300, 77)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
def test_bias_gradient_partial_rows(M, N, dtype):
    """Column sums on both sides of the rule for their second pass (few partial rows, many columns), whole 16-byte
    pieces and not: one rounding (2^-8 or 2^-24 of the sum) and the fp32 sums' error (M 2^-24 of the absolute sum)."""
    x, w, b, dy = (rnd(*s, seed=i).to(dtype) for i, s in enumerate([(M, 8), (N, 8), (N,), (M, N)]))
    gb = run_grads(K.matmul, [x, w, b], dy)[1][2].double().cpu()
    ref, mag = dy.double().sum(0), dy.double().abs().sum(0)
    ulp = 2.0 ** -8 if dtype == torch.bfloat16 else 2.0 ** -24
    assert bool(((gb - ref).abs() <= ulp * ref.abs() + M * 2.0 ** -24 * mag).all())


def test_matmul_backward_on_two_streams_shares_no_workspace():
    """Backward passes whose products split over K, in turn on two streams that are not ordered against each other:
    each gives the bits of a pass of its own (their partial planes lie in the call's memory)."""
    from qwen3_5_vl_cuda_custom_amd import _lib
    sets = [[t.bfloat16().to(DEV) for t in (rnd(33, 1160, seed=s), rnd(8208, 1160, seed=s + 1, std=0.1),
                                             rnd(33, 8208, seed=s + 2))] for s in (60, 70)]
    assert _lib.lib().q3_matmul_backward_workspace_bytes_for(*(t.data_ptr() for t in (sets[0][0], sets[0][1],
                                                                                      sets[0][2])),
                                                             33, 8208, 1160, _lib.Q3_BF16) >= 8 * 33 * 1160 * 4
    want = [run_grads(K.matmul, s[:2], s[2])[1] for s in sets]
    torch.cuda.synchronize()
    streams = [torch.cuda.Stream() for _ in sets]
    got = [[], []]
    for _ in range(8):
        for i, st in enumerate(streams):
            with torch.cuda.stream(st):
                got[i].append(run_grads(K.matmul, sets[i][:2], sets[i][2])[1])
    torch.cuda.synchronize()
    for g, w in zip(got, want):
        assert all(torch.equal(a, b) for run in g for a, b in zip(run, w))


@pytest.mark.parametrize("M,N,K_", [(1024, 4096, 12352), (512, 2048, 8256)])
def test_matmul_split_with_shorter_last_split(M, N, K_):
    """A K that no split count divides into whole 64-wide stages: the forward runs it unsplit (the backward's products
    split such a reduction: test_matmul_backward_untransposed_against_transposed). Outputs reach |11|, where half a
    bf16 step is 0.031: the bound is one rounding of each value (2^-8 of it) plus the fp32 sums' order (2^-16 of the
    largest), not the fixed 0.02 of unit-sized outputs."""
    x, w = rnd(M, K_, seed=44).bfloat16(), rnd(N, K_, seed=45, std=0.02).bfloat16()
    got, ref = K.matmul(x.to(DEV), w.to(DEV)).float().cpu(), O.linear(x.float(), w.float())
    over = float(((got - ref).abs() - 2.0 ** -8 * ref.abs() - 2.0 ** -16 * ref.abs().max()).max())
    assert over <= 0, f"split {M} {N} {K_}: {over:.3e} over"


@pytest.mark.parametrize("R,C", [(64, 64), (8, 200), (200, 8), (72, 136), (65, 64), (64, 65), (1, 7)])
def test_transpose_is_exact(R, C):
    """q3_transpose, whole 16-byte rows (the vector kernel) and not: bit-exact."""
    from qwen3_5_vl_cuda_custom_amd import _lib
    a = rnd(3, R, C, seed=95).bfloat16().to(DEV)
    b = torch.empty(3, C, R, dtype=a.dtype, device=DEV)
    _lib.call("q3_transpose", a.data_ptr(), b.data_ptr(), 3, R, C, _lib.dtype_code(a.dtype), _lib.stream())
    assert torch.equal(b, a.transpose(1, 2))


def test_matmul_residual_gradient_passes_through():
    x, w, r, dy = rnd(40, 64, seed=48), rnd(24, 64, seed=49), rnd(40, 24, seed=50), rnd(40, 24, seed=51)
    _, (gx, gw, gr) = run_grads(lambda a, c, d: K.matmul(a, c, residual=d), [x, w, r], dy)
    _, (rx, rw, rr) = ref_grads(lambda a, c, d: O.linear(a, c) + d, [x, w, r], dy)
    assert_close(gx, rx, atol=1e-3, what="dx")
    assert_close(gw, rw, atol=1e-3, what="dw")
    assert torch.equal(gr.cpu(), dy)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_batched_gemm_backward(dtype):
    x, w, dy = rnd(4, 40, 64, seed=52, dtype=dtype), rnd(4, 48, 64, seed=53, dtype=dtype), rnd(4, 40, 48, seed=54,
                                                                                              dtype=dtype)
    _, (gx, gw) = run_grads(K.cuda_batched_gemm, [x, w], dy)
    _, (rx, rw) = ref_grads(O.batched_gemm, [x, w], dy)
    if dtype == torch.float32:
        assert_close(gx, rx, atol=1e-3, what="bgemm dx")
        assert_close(gw, rw, atol=1e-3, what="bgemm dw")
    else:
        assert_grad_close(gx, rx, "bgemm dx bf16")
        assert_grad_close(gw, rw, "bgemm dw bf16")


# ------------------------------------------------------------------ attention
def _fa(groups, causal, scale):
    return lambda q, k, v: K.flash_attention(q, k, v, scale, causal, groups)


def _fa_ref(groups, causal, scale):
    return lambda q, k, v: O.flash_attention(q, k, v, scale, causal, groups)


@pytest.mark.parametrize("Hq,Hkv,causal", [(4, 4, True), (4, 4, False), (8, 2, True)])
def test_flash_attention_backward_reference_shapes_fp32(Hq, Hkv, causal):
    q, k, v = rnd(2, Hq, 16, 32, seed=60), rnd(2, Hkv, 16, 32, seed=61), rnd(2, Hkv, 16, 32, seed=62)
    dy = rnd(2, Hq, 16, 32, seed=63)
    s = 32 ** -0.5
    _, (gq, gk, gv) = run_grads(_fa(Hq // Hkv, causal, s), [q, k, v], dy)
    _, (rq, rk, rv) = ref_grads(_fa_ref(Hq // Hkv, causal, s), [q, k, v], dy)
    for a, r, n in ((gq, rq, "dq"), (gk, rk, "dk"), (gv, rv, "dv")):
        assert_close(a, r, atol=5e-3, what=f"flash {n}")


@pytest.mark.parametrize("Sq,Sk,D", [(1, 1, 8), (33, 17, 40), (17, 33, 32), (15, 31, 100), (47, 48, 72), (65, 64, 64)])
@pytest.mark.parametrize("causal", [True, False])
def test_flash_attention_backward_partial_tiles_fp32(Sq, Sk, D, causal):
    """Query and key counts around the SIMT kernels' 16-row tiles, every width of their lanes' share, against float64:
    fp32 sums of at most 65 terms of products of at most |6|, (65 + D) 2^-24 of the largest gradient and of dP."""
    q, k, v, dy = rnd(2, 4, Sq, D, seed=60), rnd(2, 2, Sk, D, seed=61), rnd(2, 2, Sk, D, seed=62), rnd(2, 4, Sq, D, seed=63)
    s = D ** -0.5
    _, got = run_grads(_fa(2, causal, s), [q, k, v], dy)
    with torch.enable_grad():
        xs = [t.double().requires_grad_(True) for t in (q, k, v)]
        a = xs[0] * s @ xs[1].repeat_interleave(2, 1).transpose(-1, -2)
        if causal:
            a = a.masked_fill(~torch.ones(Sq, Sk, dtype=torch.bool).tril(), float("-inf"))
        ref = torch.autograd.grad(a.softmax(-1) @ xs[2].repeat_interleave(2, 1), xs, dy.double())
    dp = float((dy @ v.repeat_interleave(2, 1).transpose(-1, -2)).abs().max())
    for a, r, n in zip(got, ref, ("dq", "dk", "dv")):
        tol = (65 + D) * 2.0 ** -24 * (4 * float(r.abs().max()) + dp)
        assert float((a.double().cpu() - r).abs().max()) <= tol, n


@pytest.mark.parametrize("B,Hq,Hkv,Sq,Sk,D,causal", [
    (1, 8, 2, 300, 300, 128, True),    # text GQA, ragged key tiles
    (2, 4, 4, 100, 100, 72, False),    # vision head dim, non-causal
    (1, 8, 1, 130, 130, 64, True),     # groups 8
    (1, 4, 2, 5, 77, 128, False),      # Sq != Sk
])
def test_flash_attention_backward_bf16(B, Hq, Hkv, Sq, Sk, D, causal):
    q, k, v = (rnd(B, Hq, Sq, D, seed=64).bfloat16(), rnd(B, Hkv, Sk, D, seed=65).bfloat16(),
               rnd(B, Hkv, Sk, D, seed=66).bfloat16())
    dy = rnd(B, Hq, Sq, D, seed=67).bfloat16()
    s = D ** -0.5
    _, (gq, gk, gv) = run_grads(_fa(Hq // Hkv, causal, s), [q, k, v], dy)
    _, (rq, rk, rv) = ref_grads(_fa_ref(Hq // Hkv, causal, s), [q, k, v], dy)
    for a, r, n in ((gq, rq, "dq"), (gk, rk, "dk"), (gv, rv, "dv")):
        assert_grad_close(a, r, f"flash {n} bf16 D={D}")
    twice_equal(lambda: run_grads(_fa(Hq // Hkv, causal, s), [q, k, v], dy)[1])


def _attention_backward_simt(q, k, v, dy, scale, causal):
    """(dq, dk, dv) of the SIMT kernels, which a workspace of one float per row selects."""
    from qwen3_5_vl_cuda_custom_amd import _lib
    from qwen3_5_vl_cuda_custom_amd.kernels.flash_attention import flash_attention_lse
    (B, Hq, Sq, D), (_, Hkv, Sk, _) = q.shape, k.shape
    qd, kd, vd, dyd = (t.to(DEV) for t in (q, k, v, dy))
    o, lse = flash_attention_lse(qd, kd, vd, scale, causal, Hq // Hkv)
    out = [torch.empty_like(t) for t in (qd, kd, vd)]
    nws = _lib.lib().q3_flash_attention_backward_workspace_bytes(B, Hq, Sq)
    ws = torch.empty(nws, dtype=torch.uint8, device=DEV)
    _lib.call("q3_flash_attention_backward", *(t.data_ptr() for t in (qd, kd, vd, o, lse, dyd, *out)), B, Hq, Hkv,
              Sq, Sk, D, scale, int(causal), _lib.dtype_code(q.dtype), ws.data_ptr(), nws, _lib.stream())
    return out


@pytest.mark.parametrize("B,Hq,Hkv,Sq,Sk,D,causal", [
    (1, 4, 1, 1, 1, 128, True), (2, 2, 2, 31, 33, 64, False), (1, 8, 2, 129, 129, 128, True),
    (1, 8, 2, 64, 200, 128, True), (1, 8, 2, 200, 64, 128, True), (1, 6, 2, 97, 127, 96, False),
    (2, 3, 3, 128, 128, 72, False), (1, 16, 1, 257, 257, 80, True), (3, 4, 4, 33, 96, 72, True),
    (1, 32, 8, 640, 640, 128, True),
])
def test_flash_attention_backward_mfma_against_simt(B, Hq, Hkv, Sq, Sk, D, causal):
    """The MFMA backward (tile, split and causal edges) against the fp32 oracle, and against the SIMT kernels (which
    a workspace of one float per row selects) on the same o and lse. Both keep P and dS in fp32 (the MFMA kernels as
    two bf16 terms, 2^-17 relative) and round once, so an element may differ by one bf16 rounding of its own value
    (2^-7 of it), the fp32 sums' error over terms up to the largest result (2^-14 of it), and, where dP - Dv cancels
    (one key: dS is 0 up to rounding), the fp32 rounding of dP and Dv (a few 2^-24 of the largest dP, here 2^-21)
    times the largest |scale * q| or |scale * k|."""
    q, k, v = (rnd(B, Hq, Sq, D, seed=64).bfloat16(), rnd(B, Hkv, Sk, D, seed=65).bfloat16(),
               rnd(B, Hkv, Sk, D, seed=66).bfloat16())
    dy = rnd(B, Hq, Sq, D, seed=67).bfloat16()
    s = D ** -0.5
    _, got = run_grads(_fa(Hq // Hkv, causal, s), [q, k, v], dy)
    _, ref = ref_grads(_fa_ref(Hq // Hkv, causal, s), [q, k, v], dy)
    simt = _attention_backward_simt(q, k, v, dy, s, causal)
    dp = (dy.float() @ v.float().repeat_interleave(Hq // Hkv, dim=1).transpose(-1, -2)).abs().max()
    noise = 2.0 ** -21 * float(dp * torch.maximum(q.abs().max(), k.abs().max())) * s
    for a, r, b, n in zip(got, ref, simt, ("dq", "dk", "dv")):
        x, y = a.float(), b.float()
        tol = 2.0 ** -7 * torch.maximum(x.abs(), y.abs()) + 2.0 ** -14 * y.abs().max() + noise
        over = float(((x - y).abs() - tol).max())
        assert over <= 0, f"{n} vs SIMT: {over:.3e} over"
        if float(r.abs().max()) > 1e-6:  # one key: P = 1, dS = 0 up to rounding
            assert_grad_close(a, r, f"flash {n} D={D}")


@pytest.mark.parametrize("D,where", [(64, (5, 7)), (72, (40, 70)), (128, (95, 127)), (128, (0, 0))])
def test_flash_attention_backward_keeps_infinities(D, where):
    """One infinite element of dO: the gradients of the matrix-core kernels are infinite, NaN and finite where the SIMT
    kernels' are, with the same signs, and the finite ones agree as without it (the bounds of the test above)."""
    q, k, v, dy = (rnd(1, 2, 96, D, seed=64 + i).bfloat16() for i in range(4))
    dy[0, 1][where] = float("inf")
    _, got = run_grads(_fa(1, False, D ** -0.5), [q, k, v], dy)
    simt = _attention_backward_simt(q, k, v, dy, D ** -0.5, False)
    assert any(bool(b.isinf().any()) for b in simt)
    noise = 2.0 ** -21 * 8 * D ** 0.5 * D ** -0.5
    for a, b, n in zip(got, simt, ("dq", "dk", "dv")):
        x, y = a.float(), b.float()
        assert torch.equal(x.isnan(), y.isnan()) and torch.equal(x.isinf(), y.isinf()), n
        assert torch.equal(x[x.isinf()], y[y.isinf()]), n
        x, y = x[x.isfinite()], y[y.isfinite()]
        tol = 2.0 ** -7 * torch.maximum(x.abs(), y.abs()) + 2.0 ** -14 * y.abs().max() + noise
        assert bool(((x - y).abs() <= tol).all()), n


@pytest.mark.parametrize("M,N,K_", [(1, 4, 4), (31, 33, 36), (33, 31, 132), (128, 256, 688), (130, 66, 260),
                                    (2050, 1030, 100), (65, 20, 30)])
def test_matmul_and_backward_fp32_tiles(M, N, K_):
    """fp32 GEMM, its gradients and the epilogue at the edges of the 32 x 32 and 64 x 64 tiles, of the K chunks and
    (the last: rows that are no whole pieces) on the SIMT kernel. fp32 products and sums: at most (K + 2) 2^-24 of
    the sum of absolute products."""
    x, w, b, r, dy = (rnd(*sh, seed=40 + i) for i, sh in enumerate([(M, K_), (N, K_), (N,), (M, N), (M, N)]))
    out, (gx, gw, gb, gr) = run_grads(lambda a, c, d, e: K.matmul(a, c, d, residual=e), [x, w, b, r], dy)
    xd, wd, dd = x.double(), w.double(), dy.double()
    for got, ref, mag, n in ((out, xd @ wd.t() + b.double() + r.double(), x.abs() @ w.abs().t() + b.abs() + r.abs(), K_),
                             (gx, dd @ wd, dy.abs() @ w.abs(), N), (gw, dd.t() @ xd, dy.abs().t() @ x.abs(), M)):
        over = float(((got.cpu().double() - ref).abs() - (n + 4) * 2.0 ** -24 * mag.double()).max())
        assert over <= 0, over


@pytest.mark.parametrize("B,Hq,Hkv,Sq,Sk,D,causal,dtype", [
    (1, 2, 1, 1, 1, 8, True, torch.float32), (2, 4, 2, 15, 33, 64, False, torch.float32),
    (1, 4, 2, 128, 128, 64, True, torch.float32), (1, 3, 3, 17, 70, 65, False, torch.float32),
    (1, 2, 2, 40, 40, 256, True, torch.float32), (2, 2, 1, 33, 31, 130, False, torch.float32),
    (1, 4, 1, 50, 50, 32, True, torch.bfloat16), (1, 2, 2, 20, 64, 7, False, torch.bfloat16),
])
def test_flash_attention_generic_forward(B, Hq, Hkv, Sq, Sk, D, causal, dtype):
    """The generic forward (fp32, other head dims) and its log-sum-exp at the edges of its 16-query and 32-key tiles."""
    from qwen3_5_vl_cuda_custom_amd.kernels.flash_attention import flash_attention_lse
    q, k, v = (rnd(B, h, s_, D, seed=60 + i, dtype=dtype) for i, (h, s_) in
               enumerate([(Hq, Sq), (Hkv, Sk), (Hkv, Sk)]))
    sc = D ** -0.5
    o, lse = flash_attention_lse(q.to(DEV), k.to(DEV), v.to(DEV), sc, causal, Hq // Hkv)
    ref = O.flash_attention(q.float(), k.float(), v.float(), sc, causal, Hq // Hkv)
    if dtype == torch.float32:
        assert_close(o, ref, atol=2e-5, what="o")  # sums of up to 70 fp32 terms of magnitude ~1
    else:
        assert_bf16_close(o, ref, what="o bf16")
    scores = (q.float() @ k.float().repeat_interleave(Hq // Hkv, dim=1).transpose(-1, -2)) * sc
    if causal:
        scores = scores.masked_fill(torch.ones(Sq, Sk).triu(1).bool(), float("-inf"))
    assert_close(lse, scores.logsumexp(-1), atol=2e-5, what="lse")


# ------------------------------------------------------------------ embedding, rotary, routing
@pytest.mark.parametrize("dtype,padding_idx", [(torch.float32, None), (torch.bfloat16, 3)])
def test_embedding_backward(dtype, padding_idx):
    w = rnd(100, 64, seed=70, dtype=dtype)
    ids = torch.randint(0, 100, (4, 16), generator=torch.Generator().manual_seed(71))
    ids[0, :4] = 3  # repeated ids (and the padding row) accumulate
    dy = rnd(4, 16, 64, seed=72, dtype=dtype)
    with torch.enable_grad():
        wd = w.detach().to(DEV).clone().requires_grad_(True)
        K.embedding(ids.to(DEV), wd, padding_idx).backward(dy.to(DEV))
        wr = w.detach().float().clone().requires_grad_(True)
        F.embedding(ids, wr, padding_idx=padding_idx).backward(dy.float())
    if dtype == torch.float32:
        assert_close(wd.grad, wr.grad, atol=1e-5, what="embedding dw")
    else:
        assert_grad_close(wd.grad, wr.grad, "embedding dw bf16")


def test_rope_and_mrope_backward():
    B, H, S, D = 2, 4, 50, 128
    x, dy = rnd(B, H, S, D, seed=73), rnd(B, H, S, D, seed=74)
    pos = torch.arange(S).view(1, 1, S).expand(3, B, S)
    cos3, sin3 = O.mrope_cos_sin(pos, D, 5e6)
    _, (gx,) = run_grads(lambda t: K.apply_mrope(t, cos3.to(DEV), sin3.to(DEV), [24, 20, 20]), [x], dy)
    _, (rx,) = ref_grads(lambda t: O.apply_mrope(t, cos3, sin3, [24, 20, 20]), [x], dy)
    assert_close(gx, rx, atol=1e-4, what="mrope dx")
    cos, sin = cos3[0, 0, :, :72], sin3[0, 0, :, :72]
    x2, dy2 = rnd(B, H, S, 72, seed=75), rnd(B, H, S, 72, seed=76)
    _, (gx,) = run_grads(lambda t: K.apply_rope(t, cos.to(DEV), sin.to(DEV)), [x2], dy2)
    _, (rx,) = ref_grads(lambda t: O.apply_rope(t, cos, sin), [x2], dy2)
    assert_close(gx, rx, atol=1e-4, what="rope dx")


@pytest.mark.parametrize("B,S,Hq,Hkv,D,dtype", [
    (1, 1, 1, 1, 64, torch.float32), (2, 5, 4, 2, 64, torch.bfloat16), (1, 300, 3, 1, 128, torch.bfloat16),
    (2, 600, 8, 2, 128, torch.float32), (1, 17, 5, 5, 256, torch.bfloat16),
])
@torch.enable_grad()
def test_qk_norm_rope_trains_like_the_single_ops_in_fp64(B, S, Hq, Hkv, D, dtype):
    """The fused q/k norm + rotation and its gradients at one token, fewer tokens than blocks and more, and rows
    that are no whole pass, on column views of one projection. Against fp64 with the same fp32 angles (sincosf: 2
    ulp, 2^-22, of rotated values up to max|y|): fp32 sums of up to D terms stay within (D + 8) 2^-24 of their
    magnitude, so 2^-15 of the largest value bounds them for D <= 256; the weight gradients add B S H terms; bf16
    adds one rounding, 2^-8 of the value."""
    from qwen3_5_vl_cuda_custom_amd.kernels.backward import QKNormRopeFunction
    sec, eps, H = (D // 2 - 2 * (D // 6), D // 6, D // 6), 1e-6, Hq + 2 * Hkv
    qkv = rnd(B, S, H, D, seed=80).to(dtype)
    w = [(1 + 0.1 * rnd(D, seed=81 + i)).to(dtype) for i in range(2)]
    dy = rnd(B, H, S, D, seed=83).to(dtype)
    pos = torch.randint(0, 5000, (3, B, S), generator=torch.Generator().manual_seed(84), dtype=torch.int32)
    inv = 1.0 / (5e6 ** (torch.arange(0, D, 2, dtype=torch.float32) / D))
    ins = [t.to(DEV).requires_grad_(True) for t in (qkv, *w)]
    out = torch.cat(QKNormRopeFunction.apply(ins[0][:, :, :Hq], ins[0][:, :, Hq:Hq + Hkv], ins[0][:, :, Hq + Hkv:],
                                             ins[1], ins[2], pos.to(DEV), inv.to(DEV), sec, eps), dim=1)
    got = torch.autograd.grad(out, ins, dy.to(DEV))
    x, wq, wk = (t.double().requires_grad_(True) for t in (qkv, *w))
    axis = torch.tensor([0] * sec[0] + [1] * sec[1] + [2] * sec[2])
    ang = (pos.float()[axis] * inv[:, None, None]).double().permute(1, 2, 0)[:, :, None]  # (B, S, 1, D / 2)

    def part(t, wt):
        n = t * torch.rsqrt(t.pow(2).mean(-1, keepdim=True) + eps) * wt
        a, b = n[..., :D // 2], n[..., D // 2:]
        return torch.cat([a * ang.cos() - b * ang.sin(), b * ang.cos() + a * ang.sin()], dim=-1).transpose(1, 2)

    ref_out = torch.cat([part(x[:, :, :Hq], wq), part(x[:, :, Hq:Hq + Hkv], wk), x[:, :, Hq + Hkv:].transpose(1, 2)], 1)
    ref = torch.autograd.grad(ref_out, (x, wq, wk), dy.double())
    rounding = 2.0 ** -8 if dtype == torch.bfloat16 else 0.0
    for a, r, n in ((out, ref_out, 1), (got[0], ref[0], 1), (got[1], ref[1], B * S * Hq), (got[2], ref[2], B * S * Hkv)):
        mag = r.abs().max() if n == 1 else n ** 0.5 * 16 + r.abs().max()
        over = float(((a.detach().cpu().double() - r.detach()).abs() - rounding * r.abs() - 2.0 ** -15 * mag).max())
        assert over <= 0, over


@pytest.mark.parametrize("B,H,Hkv,S,D,causal", [(1, 2, 2, 1, 72, False), (2, 4, 4, 130, 72, False),
                                                (1, 4, 1, 257, 128, True), (2, 4, 2, 64, 64, True)])
@torch.enable_grad()
def test_attention_gradients_on_token_major_storage(B, H, Hkv, S, D, causal):
    """The same kernels on (B, S, H, D) storage as on (B, H, S, D): the same bits, also for the vision block's
    rotation and attention on the fused projection against its single ops."""
    from qwen3_5_vl_cuda_custom_amd.kernels.backward import FlashAttentionFunction, RopeAttentionFunction
    q, k, v = (rnd(B, h, S, D, seed=85 + i).bfloat16().to(DEV).requires_grad_(True) for i, h in
               enumerate((H, Hkv, Hkv)))
    dy = rnd(B, S, H, D, seed=88).bfloat16().to(DEV).transpose(1, 2)
    outs = []
    for bshd in (False, True):
        o = FlashAttentionFunction.apply(q, k, v, D ** -0.5, causal, H // Hkv, bshd)
        outs.append((o.contiguous(), *torch.autograd.grad(o, (q, k, v), dy)))
    for a, b in zip(*outs):
        assert torch.equal(a, b)
    if causal:
        return
    qkv = rnd(B, S, 3, H, D, seed=89).bfloat16().to(DEV).requires_grad_(True)
    ang = rnd(S, D, seed=90).to(DEV)
    cos, sin = ang.cos(), ang.sin()
    o1 = RopeAttentionFunction.apply(qkv, cos, sin, D ** -0.5)
    qs, ks, vs = (qkv[:, :, i].transpose(1, 2) for i in range(3))
    o2 = K.flash_attention(K.apply_rope(qs, cos, sin), K.apply_rope(ks, cos, sin), vs, D ** -0.5, False,
                           1).transpose(1, 2)
    assert torch.equal(o1, o2)
    assert torch.equal(*(torch.autograd.grad(o, qkv, dy.transpose(1, 2))[0] for o in (o1, o2)))


@torch.enable_grad()
def test_text_attention_training_routes_agree():
    """Positions as floats, a hook on a norm and a frozen norm weight: every route gives the fused one's result up to
    the roundings between its single ops (three of 2^-8 of the largest). Which route each takes: the test below."""
    from qwen3_5_vl_cuda_custom_amd.modules import CudaFullAttention, TextMRoPE
    torch.manual_seed(0)
    att = CudaFullAttention(256, 4, 2, 64).to(DEV, torch.bfloat16)
    rope = TextMRoPE(64, 5e6, [12, 10, 10]).to(DEV)
    x = rnd(2, 70, 256, seed=91).bfloat16().to(DEV)
    pos = torch.arange(70, device=DEV).expand(3, 1, 70).contiguous()

    def run(p):
        xi = x.clone().requires_grad_(True)
        out, _ = att(xi, rope.bind(p))
        return out.detach(), torch.autograd.grad(out.float().pow(2).sum(), xi)[0]

    want, runs = run(pos), [run(pos.float()), run(pos.int())]
    seen = []
    h = att.q_norm.register_forward_hook(lambda *a: seen.append(1))
    runs.append(run(pos))
    h.remove()
    assert seen
    att.q_norm.weight.requires_grad_(False)
    runs.append(run(pos))
    for got in runs:
        for a, b in zip(got, want):
            assert float((a.float() - b.float()).abs().max()) <= 3 * 2.0 ** -8 * float(b.float().abs().max())


@torch.enable_grad()
@pytest.mark.parametrize("case", ["plain", "frozen weight", "float positions", "norm hook", "global hook",
                                  "global pre-hook", "replaced forward", "other rotary"])
def test_text_attention_training_fuses_only_plain_norms(case):
    """Norm and rotation train as one op only where nothing else is called with them and the positions are whole
    numbers; what the single ops would have called (hooks, a replaced forward, another rotary's angles, fractional
    positions) takes effect."""
    from torch.nn.modules import module as nn_module
    from qwen3_5_vl_cuda_custom_amd.modules import CudaFullAttention, CudaRMSNorm, TextMRoPE
    torch.manual_seed(0)
    att = CudaFullAttention(256, 4, 2, 64).to(DEV, torch.bfloat16)
    rope = TextMRoPE(64, 5e6, [12, 10, 10]).to(DEV)
    x = rnd(2, 70, 256, seed=91).bfloat16().to(DEV)
    pos, seen, handle = torch.arange(70, device=DEV).expand(3, 1, 70).contiguous(), [], None
    base = att(x, rope.bind(pos))[0].detach()
    hook = lambda m, *a: seen.append(1) if m is att.q_norm else None  # noqa: E731
    if case == "frozen weight":
        att.q_norm.weight.requires_grad_(False)
    elif case == "float positions":
        pos = pos + 0.5
    elif case == "norm hook":
        handle = att.q_norm.register_forward_hook(hook)
    elif case == "global hook":
        handle = nn_module.register_module_forward_hook(hook)
    elif case == "global pre-hook":
        handle = nn_module.register_module_forward_pre_hook(hook)
    elif case == "replaced forward":
        att.q_norm.forward = lambda t: seen.append(1) or CudaRMSNorm.forward(att.q_norm, t)
    elif case == "other rotary":
        class Halved(TextMRoPE):
            def compute_cos_sin(self, position_ids):
                return super().compute_cos_sin(position_ids.float() / 2)
        rope = Halved(64, 5e6, [12, 10, 10]).to(DEV)
    try:
        q, k, v = (torch.zeros(2, 70, h, 64, device=DEV, dtype=torch.bfloat16) for h in (4, 2, 2))
        fused = att._train_positions(rope.bind(pos), q, k, v) is not None
        assert fused == (case in ("plain", "frozen weight"))
        out = att(x, rope.bind(pos))[0].detach()
    finally:
        if handle is not None:
            handle.remove()
    assert bool(seen) == ("hook" in case or case == "replaced forward")
    q, k, v = (p(x).view(2, 70, -1, 64) for p in (att.q_proj, att.k_proj, att.v_proj))
    cos, sin = rope.compute_cos_sin(pos)
    q, k = (K.apply_mrope(K.rmsnorm(t, n.weight, n.eps).transpose(1, 2), cos, sin, [12, 10, 10])
            for t, n in ((q, att.q_norm), (k, att.k_norm)))
    ref = K.flash_attention(q, k, v.transpose(1, 2), scale=att.scale, is_causal=True, num_kv_groups=2)
    ref = att.o_proj(ref.transpose(1, 2).reshape(2, 70, 256)).detach().float()
    # the single ops' two roundings more than the fused one: three of 2^-8 of the largest
    assert float((out.float() - ref).abs().max()) <= 3 * 2.0 ** -8 * float(ref.abs().max())
    if case in ("float positions", "other rotary"):
        assert float((out.float() - base.float()).abs().max()) > 0


def test_topk_and_index_add_backward():
    x = rnd(64, 128, seed=77)
    gv = rnd(64, 8, seed=78)
    with torch.enable_grad():
        xd = x.to(DEV).requires_grad_(True)
        vals, idx = K.cuda_topk(xd, 8)
        vals.backward(gv.to(DEV))
    want = torch.zeros(64, 128).scatter_(-1, idx.cpu(), gv)
    assert torch.equal(xd.grad.cpu(), want)
    tgt, src = rnd(10, 16, seed=79), rnd(24, 16, seed=80)
    index = torch.randint(0, 10, (24,), generator=torch.Generator().manual_seed(81))
    dy = rnd(10, 16, seed=82)
    with torch.enable_grad():
        td, sd = tgt.to(DEV).requires_grad_(True), src.to(DEV).requires_grad_(True)
        out = K.cuda_index_add(td, sd, index.to(DEV))
        out.backward(dy.to(DEV))
    assert_close(out, tgt.index_add(0, index, src), atol=1e-5, what="index_add (autograd form)")
    assert torch.equal(td.grad.cpu(), dy) and torch.equal(sd.grad.cpu(), dy[index])
    assert torch.equal(td.detach().cpu(), tgt), "the autograd form leaves target unchanged"


def test_ops_without_backward_still_refuse_grad():
    x = rnd(8, 64, seed=83).to(DEV).requires_grad_(True)
    w = rnd(16, 64, seed=84).to(DEV)
    with torch.enable_grad(), pytest.raises(NotImplementedError):
        K.matmul_swiglu(x, w, w)


# ------------------------------------------------------------------ module-level training
def _module_grads(layer, fwd, x, dy):
    layer.requires_grad_(True)
    with torch.enable_grad():
        xd = x.detach().to(DEV).clone().requires_grad_(True)
        y = fwd(layer, xd)
        y.backward(dy.to(DEV).to(y.dtype))
    grads = {n: p.grad.float().cpu() for n, p in layer.named_parameters()}
    return y.detach().float().cpu(), xd.grad.float().cpu(), grads


def _oracle_grads(fn, p_dev, x, dy):
    p = {n: t.detach().float().cpu().requires_grad_(True) for n, t in p_dev.items()}
    with torch.enable_grad():
        xc = x.detach().float().cpu().clone().requires_grad_(True)
        y = fn(xc, p)
        y.backward(dy.float())
    return y.detach(), xc.grad, {n: t.grad for n, t in p.items()}


def _check_grads(got, ref, what, dtype):
    y, gx, gp = got
    ry, rgx, rgp = ref
    # bf16: a layer's backward rounds each of its ~20 intermediates to bf16, so its gradients carry
    # that accumulated rounding: max error within 5% of the largest |reference|, mean within 1.5%
    close = (lambda a, b, n: assert_close(a, b, atol=2e-3 * max(1.0, float(b.abs().max())), what=n)) \
        if dtype == torch.float32 else (lambda a, b, n: assert_grad_close(a, b, n, max_rel=5e-2, mean_rel=1.5e-2))
    close(y, ry, f"{what} output")
    close(gx, rgx, f"{what} d input")
    assert set(gp) == set(rgp)
    for n in gp:
        close(gp[n], rgp[n], f"{what} d {n}")


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_text_decoder_layer_trains_like_the_oracle(dtype):
    from oracle import layers as L
    from qwen3_5_vl_cuda_custom_amd import workloads as W
    cfg = W.C1
    layer = W.make_text_layer(cfg, dtype, DEV, seed=3)
    x, pos = W.text_inputs(cfg, 1, 128, dtype, DEV, seed=3)
    dy = rnd(1, 128, cfg.hidden, seed=90).to(dtype)
    bind = W.make_rope(cfg, DEV).bind(pos)
    got = _module_grads(layer, lambda m, t: m(t, bind)[0], x, dy)
    cos3, sin3 = O.mrope_cos_sin(pos.cpu(), cfg.head_dim, cfg.theta)
    kw = dict(num_heads=cfg.heads, num_kv_heads=cfg.kv_heads, head_dim=cfg.head_dim, eps=cfg.eps, cos_3d=cos3,
              sin_3d=sin3, mrope_section=list(cfg.mrope_section))
    ref = _oracle_grads(lambda t, p: L.text_decoder_layer(t, p, **kw)[0], dict(layer.named_parameters()), x, dy)
    _check_grads(got, ref, f"text layer {dtype}", dtype)


def test_moe_layer_trains_like_the_oracle():
    from oracle import layers as L
    from qwen3_5_vl_cuda_custom_amd.modules import CudaSparseMoE
    moe = CudaSparseMoE(hidden_size=128, moe_intermediate_size=48, num_experts=8, top_k=2).to(DEV)
    x, dy = rnd(1, 64, 128, seed=91), rnd(1, 64, 128, seed=92)
    got = _module_grads(moe, lambda m, t: m(t)[0], x, dy)
    ref = _oracle_grads(lambda t, p: L.sparse_moe(t, p, top_k=2)[0], dict(moe.named_parameters()), x, dy)
    _check_grads(got, ref, "moe layer", torch.float32)


@pytest.mark.parametrize("T,H,I,E,k", [(1, 64, 24, 4, 1), (64, 128, 48, 8, 2), (300, 264, 136, 16, 4),
                                       (600, 256, 128, 3, 2), (520, 512, 192, 128, 8)])
def test_moe_block_trains_in_bf16_like_the_oracle(T, H, I, E, k):
    """The grouped bf16 training path (experts with no rows, a few, and more than one 256-row tile) against the fp32
    oracle on the same routing: the block's ~6 bf16 intermediates each round once (the bounds of a layer)."""
    from oracle import layers as L
    from qwen3_5_vl_cuda_custom_amd.modules import CudaSparseMoE
    moe = CudaSparseMoE(hidden_size=H, moe_intermediate_size=I, num_experts=E, top_k=k).to(DEV).bfloat16()
    g = torch.Generator(device=DEV).manual_seed(9)
    with torch.no_grad():
        for p in moe.parameters():
            p.normal_(0, 0.1, generator=g)
    x, dy = rnd(1, T, H, seed=91).bfloat16(), rnd(1, T, H, seed=92).bfloat16()
    # the oracle routes on fp32 logits, the block on bf16 ones: keep the tokens whose k-th and next logit lie further
    # apart than the bf16 rounding of both (2^-8 of each)
    with torch.no_grad():
        ref = (x.float().view(T, H) @ moe.gate_weight.float().cpu().t()).sort(-1, descending=True).values
        same = (ref[:, k - 1] - ref[:, k] > 2.0 ** -7 * ref.abs().amax(-1)) if k < E else torch.ones(T, dtype=bool)
        same[0] = True
    x, dy = x[:, same], dy[:, same]
    got = _module_grads(moe, lambda m, t: m(t)[0], x, dy)
    ref = _oracle_grads(lambda t, p: L.sparse_moe(t, p, top_k=k)[0], dict(moe.named_parameters()), x, dy)
    _check_grads(got, ref, f"moe bf16 {(T, H, I, E, k)}", torch.bfloat16)
    moe.requires_grad_(False)
    fwd = moe(x.to(DEV))[0].float().cpu()  # the inference path on the same routing
    assert_grad_close(got[0], fwd, "train forward vs inference", max_rel=2e-2, mean_rel=5e-3)


def test_moe_training_gradients_are_reproducible_and_partial():
    """Twice the same bits, and the same bits with some gradients left out (a frozen weight, no input gradient)."""
    from qwen3_5_vl_cuda_custom_amd.kernels.moe_routing import moe_experts_train
    T, H, I, E, k = 200, 128, 64, 8, 2
    x, gu, dn = (rnd(*s, seed=i, std=0.1).bfloat16().to(DEV) for i, s in
                 enumerate([(T, H), (E, 2 * I, H), (E, H, I)]))
    idx = torch.stack([torch.randperm(E, generator=torch.Generator().manual_seed(t))[:k] for t in range(T)]).to(DEV)
    w, dy = torch.rand(T, k, device=DEV).bfloat16(), rnd(T, H, seed=5).bfloat16().to(DEV)

    def grads(which):
        ts = [t.clone().requires_grad_(i in which) for i, t in enumerate((x, gu, dn, w))]
        with torch.enable_grad():
            moe_experts_train(ts[0], ts[1], ts[2], idx, ts[3]).backward(dy)
        return [t.grad for t in ts]

    full = grads({0, 1, 2, 3})
    for which in ({0, 1, 2, 3}, {0}, {1}, {2}, {3}, {0, 3}):
        for i, (a, b) in enumerate(zip(grads(which), full)):
            assert torch.equal(a, b) if i in which else a is None


def test_moe_training_leaves_out_ids_that_are_no_experts():
    """Ids outside [0, E) (a NaN router row's top-k gives 0x7fffffff) are not dispatched: no output, no gradient and
    nothing read for them, whatever the state's memory held before (zeros here: an entry taken from it would name row
    0). Against the loop over the experts in fp32; a slot's product rounds its ~6 bf16 intermediates (a layer's bounds)."""
    from qwen3_5_vl_cuda_custom_amd import _lib
    from qwen3_5_vl_cuda_custom_amd.kernels.moe_routing import moe_experts_train
    T, H, I, E, k = 150, 128, 64, 6, 2
    x, gu, dn = (rnd(*s, seed=i, std=0.3).bfloat16() for i, s in enumerate([(T, H), (E, 2 * I, H), (E, H, I)]))
    idx = torch.stack([torch.randperm(E, generator=torch.Generator().manual_seed(t))[:k] for t in range(T)])
    idx[3] = 0x7fffffff
    idx[70, 1], idx[149, 0], idx[149, 1] = -1, E, 2
    w, dy = torch.rand(T, k, generator=torch.Generator().manual_seed(4)).bfloat16(), rnd(T, H, seed=5).bfloat16()

    def loop(x, gu, dn, w):
        out = torch.zeros(T, H)
        for e in range(E):
            t, s = (idx == e).nonzero(as_tuple=True)
            g, u = (x[t] @ gu[e].t()).chunk(2, dim=-1)
            out = out.index_add(0, t, (F.silu(g) * u @ dn[e].t()) * w[t, s, None])
        return out

    def block(x, gu, dn, w):
        before = torch.zeros(_lib.lib().q3_moe_train_state_bytes(T, H, I, E, k), dtype=torch.uint8, device=DEV)
        del before
        return moe_experts_train(x, gu, dn, idx.to(DEV), w)

    out, got = run_grads(block, (x, gu, dn, w), dy)
    ref_out, ref = ref_grads(loop, (x, gu, dn, w), dy)
    for a, b, n in zip((out, *got), (ref_out, *ref), ("out", "dx", "dgate_up", "ddown", "dw")):
        assert_grad_close(a, b, n, max_rel=5e-2, mean_rel=1.5e-2)
    assert not out[3].any() and not got[0][3].any()
    assert not got[3][3].any() and not got[3][70, 1] and not got[3][149, 0]


def test_moe_down_gradient_rounds_its_operand_once():
    """The weight gradient of down multiplies grad_out with w silu(g) u rounded to bf16 once. One token per expert, x a
    unit vector (g and u are entries of gate_up, exact) and a gradient of ones: each element is that operand itself,
    within half a bf16 step (8 significant bits: 2^-8 of it; expf's 2^-20 beside it). A rounding of silu(g) u before it would double that."""
    from qwen3_5_vl_cuda_custom_amd.kernels.moe_routing import moe_experts_train
    E, H, I = 16, 64, 128
    x = torch.zeros(E, H).bfloat16()
    x[:, 0] = 1
    gu, dn = rnd(E, 2 * I, H, seed=1).bfloat16(), rnd(E, H, I, seed=2).bfloat16()
    w = (torch.rand(E, 1, generator=torch.Generator().manual_seed(3)) + 0.1).bfloat16()
    idx = torch.arange(E, device=DEV).view(E, 1)
    _, got = run_grads(lambda *a: moe_experts_train(a[0], a[1], a[2], idx, a[3]), (x, gu, dn, w),
                       torch.ones(E, H).bfloat16())
    g, u = gu[:, :, 0].double().chunk(2, dim=1)
    ref = (F.silu(g) * u * w.double()).unsqueeze(1)
    assert bool(((got[2].cpu().double() - ref).abs() <= (2.0 ** -8 + 2.0 ** -20) * ref.abs()).all())


def test_moe_training_checks_its_operands():
    """What the inference entry refuses (routing on the host, other shapes, mixed types) is refused before a launch."""
    from qwen3_5_vl_cuda_custom_amd.kernels.moe_routing import moe_experts_train
    T, H, I, E, k = 6, 64, 32, 4, 2
    x, gu, dn, w = (torch.zeros(*s, device=DEV, dtype=torch.bfloat16) for s in ((T, H), (E, 2 * I, H), (E, H, I),
                                                                                 (T, k)))
    idx = torch.tensor([[0, 1]] * T, device=DEV)
    assert moe_experts_train(x, gu, dn, idx, w).shape == (T, H)
    for bad in ((x, gu, dn, idx.cpu(), w), (x, gu, dn, idx[:4], w[:4]), (x, gu, dn, idx[:4], w), (x, gu, dn, idx, w[:4]),
                (x, gu, dn, idx.float(), w), (x, gu, dn, idx[:, 0], w), (x, gu[:, :, :32], dn, idx, w),
                (x, gu, dn[:3], idx, w), (x[0], gu, dn, idx, w)):
        with pytest.raises(ValueError):
            moe_experts_train(*bad)
    with pytest.raises(RuntimeError):
        moe_experts_train(x, gu, dn, idx, w.cpu())
    with pytest.raises(TypeError):
        moe_experts_train(x, gu.float(), dn, idx, w)


def test_moe_training_records_what_it_declines(monkeypatch):
    """A bf16 call outside the grouped kernels is recorded, and in strict mode too left to the loop over the experts;
    fp32 and empty calls, which have no other path, are not recorded."""
    from qwen3_5_vl_cuda_custom_amd.kernels import _loader
    from qwen3_5_vl_cuda_custom_amd.kernels.moe_routing import moe_experts_train
    monkeypatch.setattr(_loader, "FALLBACK_LOG", [])
    monkeypatch.setenv("CUDA_QWEN3_VL_STRICT", "1")

    def call(T, H, I, dtype=torch.bfloat16, off=0):
        x, gu, dn, w = (torch.zeros(*s, device=DEV, dtype=dtype) for s in ((T * H + off,), (4, 2 * I, H), (4, H, I),
                                                                           (T, 2)))
        idx = torch.zeros(T, 2, dtype=torch.int32, device=DEV)
        idx[:, 1] = 1
        return moe_experts_train(x[off:].view(T, H), gu, dn, idx, w)

    assert call(6, 64, 32) is not None
    assert call(6, 64, 32, torch.float32) is None and call(0, 64, 32) is None
    assert _loader.FALLBACK_LOG == []
    assert call(6, 64, 20) is None and call(6, 64, 32, off=1) is None
    assert [(op, r.split(":")[0]) for op, r, _ in _loader.FALLBACK_LOG] == [("moe_experts_train",
                                                                             "experts_one_by_one")] * 2


def test_moe_block_trains_past_a_nan_token():
    """One token of NaN: its expert part is zero, the other tokens' outputs and the experts' weight gradients are those
    of the block without it (the same rows and tiles: equal up to the order of sums, one bf16 rounding)."""
    from qwen3_5_vl_cuda_custom_amd.modules import CudaSparseMoE
    torch.manual_seed(0)
    T, bad = 80, 7
    moe = CudaSparseMoE(hidden_size=128, moe_intermediate_size=64, num_experts=8, top_k=2).to(DEV).bfloat16()
    x, dy = rnd(1, T, 128, seed=91).bfloat16(), rnd(1, T, 128, seed=92).bfloat16()
    keep = torch.arange(T) != bad
    ref_y, _, ref = _module_grads(moe, lambda m, t: m(t)[0], x[:, keep], dy[:, keep])
    moe.zero_grad()
    x[0, bad] = float("nan")
    y, _, got = _module_grads(moe, lambda m, t: m(t)[0], x, dy)
    assert not y[0, bad].any()
    assert_grad_close(y[0, keep], ref_y[0], "other tokens' outputs", max_rel=2.0 ** -7, mean_rel=2.0 ** -8)
    for n in ("gate_up_proj", "down_proj"):
        assert_grad_close(got[n], ref[n], n, max_rel=2.0 ** -7, mean_rel=2.0 ** -8)


def test_vision_block_trains_like_the_oracle():
    from oracle import layers as L
    from qwen3_5_vl_cuda_custom_amd.modules import CudaVisionBlock
    from qwen3_5_vl_cuda_custom_amd import workloads as W
    blk = CudaVisionBlock(288, 4, 400).to(DEV)
    W.init_normal_(blk, seed=5, std=0.05, include_bias=True)
    cos, sin = L.vision_rope_tables([(1, 8, 8)], 72, 1e4, 2)
    x, dy = rnd(2, 64, 288, seed=93), rnd(2, 64, 288, seed=94)
    got = _module_grads(blk, lambda m, t: m(t, cos.to(DEV), sin.to(DEV)), x, dy)
    ref = _oracle_grads(lambda t, p: L.vision_block(t, p, num_heads=4, cos=cos, sin=sin, eps=1e-6),
                        dict(blk.named_parameters()), x, dy)
    _check_grads(got, ref, "vision block", torch.float32)
