"""Prefill GEMM (MFMA path) through the C ABI.  Gate: max |y - y_ref| / max |y_ref| <= 1e-2
(bf16 activations, bf16 or fp32 output, fp32 accumulate)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu
TOL = 1e-2


def rel_err(y, ref):
    return float(np.abs(y.astype(np.float64) - ref).max() / np.abs(ref).max())


@pytest.mark.parametrize("fmt", ["Q_G_4", "B32S4", "Q_G_3", "B32S8", "Q_G_8", "Q_8"])
@pytest.mark.parametrize("M,N,K", [(17, 48, 256), (64, 128, 512), (300, 200, 1024), (512, 33, 2304), (256, 384, 4096)])
def test_gemm_against_oracle(O, tfq, gpu, fmt, M, N, K):
    import torch
    print(f"gemm {fmt} M={M} N={N} K={K}", flush=True)
    w = O.rng_normal(42, N * K, 0.02)
    x = O.bf16_round(O.rng_normal(43, M * K, 1.0).reshape(M, K))
    pay = O.encode_tensor(fmt, w)
    ref = O.matmul(fmt, pay, N, K, x)
    W = tfq.Weight(fmt, N, K, pay)
    xt = torch.from_numpy(x).to(gpu).bfloat16()
    y = W.gemm(xt).cpu().numpy()
    assert y.shape == (M, N)
    assert rel_err(y, ref) <= TOL
    yb = W.gemm(xt, out_dtype=torch.bfloat16).float().cpu().numpy()
    assert rel_err(yb, ref) <= TOL
    # without scratch memory (no K split) the sums are the same up to the order of the fp32 additions
    y0 = W.gemm(xt, workspace=False).cpu().numpy()
    assert rel_err(y0, ref) <= TOL and rel_err(y, y0) <= 1e-5
    # the tile kernel and the 16-row GEMV path agree to the bf16 rounding of the decoded weights
    y16 = torch.cat([W.gemv(xt[i:i + 16]) for i in range(0, M, 16)]).cpu().numpy()
    assert rel_err(y, y16) <= 5e-3
    W.close()


def test_gemm_fp32_activations_take_the_exact_path(O, tfq, gpu):
    import torch
    M, N, K = 40, 64, 512
    w = O.rng_normal(42, N * K, 0.02)
    x = O.rng_normal(43, M * K, 1.0).reshape(M, K)
    pay = O.encode_tensor("Q_G_4", w)
    W = tfq.Weight("Q_G_4", N, K, pay)
    y = W.gemm(torch.from_numpy(x).to(gpu)).cpu().numpy()
    assert rel_err(y, O.matmul("Q_G_4", pay, N, K, x)) <= 1e-3
    W.close()


@pytest.mark.parametrize("fmt", ["B32S4", "Q_G_4", "Q_G_3", "B32S8", "Q_G_8"])
@pytest.mark.parametrize("N,K", [(14336, 4096), (4096, 14336)])
def test_config3_prefill_shapes(tfq, gpu, N, K, fmt):
    """M = 2048 tokens, bf16 activations N(0,1), block-32 weights from N(0, 0.02), bf16 output:
    against a dense fp32 torch matmul of the decoded matrix (for the companded 8-bit grid that also
    checks the line that stands for the grid in the matmul against the exact table of the decode)."""
    import torch
    M = 2048
    g = torch.Generator(device="cuda").manual_seed(3)
    w = torch.randn(N * K, device=gpu, generator=g) * 0.02
    print(f"prefill {fmt} M={M} N={N} K={K}", flush=True)
    W = tfq.Weight(fmt, N, K, tfq.encode(fmt, w))
    del w
    x = torch.randn(M, K, device=gpu, generator=g).bfloat16()
    y = W.gemm(x, out_dtype=torch.bfloat16)
    dense = W.decode()
    want = x.float() @ dense.T
    err = float((y.float() - want).abs().max() / want.abs().max())
    assert err <= TOL, err
    # linearity in x for power-of-two factors is exact
    y2 = W.gemm((x.float() * 2).bfloat16(), out_dtype=torch.float32)
    y1 = W.gemm(x, out_dtype=torch.float32)
    assert torch.equal(y2, 2 * y1)
    W.close()


@pytest.mark.parametrize("fmt", ["B32S4", "B32S8"])
def test_prefill_full_grid_is_repeatable(tfq, gpu, fmt):
    """On a full grid the step of the tile kernel runs in two barrier-separated phases with the two halves of a
    workgroup one phase apart, on LDS buffers that are reused every other step: forty launches of the gate shape
    give the same bits every time, and the rows of a tile do not depend on what the other rows hold (a call with
    half the tokens equals the first half of the whole call)."""
    import torch
    N, K, M = 14336, 4096, 2048
    g = torch.Generator(device="cuda").manual_seed(9)
    W = tfq.Weight(fmt, N, K, tfq.encode(fmt, torch.randn(N * K, device=gpu, generator=g) * 0.02))
    x = torch.randn(M, K, device=gpu, generator=g).bfloat16()
    ref = W.gemm(x, out_dtype=torch.float32).clone()
    for _ in range(40):
        assert torch.equal(W.gemm(x, out_dtype=torch.float32), ref)
    half = W.gemm(x[:M // 2], out_dtype=torch.float32)
    assert torch.equal(half, ref[:M // 2])
    W.close()


EXACT_FMTS = [("Q_G_4", "f32"), ("Q_G_3", "f32"), ("B32S4", "f32"), ("B32S8", "f32"), ("Q_G_8", "f32"), ("Q_8", "f32"),
              ("Q_G_2", "f32"), ("SB256A3", "f32"), ("SB256A2", "f32"), ("Q_4", "f32"), ("Q_G_6", "f32"), ("Q_4_K_H", "f32"),
              ("Q_G_2", "bf16"), ("SB256A3", "bf16"), ("SB256A2", "bf16"), ("Q_4", "bf16"), ("Q_G_6", "bf16")]


@pytest.mark.parametrize("fmt,dtype", EXACT_FMTS)
@pytest.mark.parametrize("M,N,K", [(17, 1, 256), (64, 128, 512), (65, 129, 768), (129, 250, 4352), (300, 48, 1024)])
def test_gemm_integer_operands(O, tfq, gpu, fmt, dtype, M, N, K):
    """The tile kernel with integer operands against the float64 product with the decoded matrix, at the edges of its
    tiles (64 / 128 rows of either side), of its K split and of the last block.  Derived bounds on the norm of the
    error: fp32 activations of the Tiled16 formats keep 16 bits (a part left out is below 2^-18 of a value, 4e-6),
    everything else is fp32 sums (1e-6); the companded grid is a line within 7.5e-5 of its levels."""
    import torch
    print(f"gemm {fmt} {dtype} M={M} N={N} K={K}", flush=True)
    w = O.rng_normal(42, N * K, 0.02)
    pay = O.encode_tensor(fmt, w)
    W = tfq.Weight(fmt, N, K, pay)
    x = torch.from_numpy(O.rng_normal(43, M * K, 1.0).reshape(M, K)).to(gpu)
    x = x.bfloat16() if dtype == "bf16" else x
    dense = torch.from_numpy(O.decode_tensor(fmt, pay, N * K).reshape(N, K)).to(gpu).double()
    want = x.double() @ dense.T
    bound = 1.5e-4 if fmt in ("Q_G_8", "Q_8") else 1e-6 if dtype == "bf16" or fmt in ("Q_4", "Q_G_6", "Q_4_K_H") else 1e-5
    for ws in (True, False):
        y = W.gemm(x, workspace=ws)
        assert float((y.double() - want).norm() / want.norm()) <= bound
    # a row does not depend on the other rows of its tile
    x2 = x.clone()
    x2[1:] = 0
    assert torch.equal(W.gemm(x2, workspace=False)[0], W.gemm(x, workspace=False)[0])
    yb = W.gemm(x, out_dtype=torch.bfloat16)
    assert torch.equal(yb, W.gemm(x).bfloat16())
    W.close()


@pytest.mark.parametrize("fmt", ["Q_G_4", "Q_G_3", "B32S4", "B32S8", "Q_G_8", "Q_8"])
@pytest.mark.parametrize("M,N,K", [(17, 8190, 4352), (33, 4100, 4352), (64, 4095, 4352), (65, 8200, 2304), (129, 3970, 2304)])
def test_gemm_few_bf16_rows_integer_operands(O, tfq, gpu, fmt, M, N, K):
    """bf16 rows of the 32-weight-group formats where their product is too small for the bf16 tile kernel, at the edges of
    the integer kernel's tiles (32, 64 and 128 rows; 128 and 256 weight rows), of its K split and of its last block, against
    the float64 product with the decoded matrix: exact operands and fp32 sums, 1e-6 on the norm as above (weights rounded to
    bf16 would be 1e-3 away)."""
    import torch
    print(f"gemm {fmt} bf16 M={M} N={N} K={K}", flush=True)
    pay = O.encode_tensor(fmt, O.rng_normal(42, N * K, 0.02))
    W = tfq.Weight(fmt, N, K, pay)
    x = torch.from_numpy(O.rng_normal(43, M * K, 1.0).reshape(M, K)).to(gpu).bfloat16()
    want = x.double() @ torch.from_numpy(O.decode_tensor(fmt, pay, N * K).reshape(N, K)).to(gpu).double().T
    y = W.gemm(x)
    assert float((y.double() - want).norm() / want.norm()) <= (1.5e-4 if fmt in ("Q_G_8", "Q_8") else 1e-6)
    assert torch.equal(W.gemm(x, out_dtype=torch.bfloat16), y.bfloat16())
    W.close()


@pytest.mark.parametrize("fmt,dtype,N,K,bound", [
    ("B32S4", "f32", 2000, 4096, 3.0e-6), ("Q_G_4", "f32", 2000, 4096, 3.0e-6), ("Q_G_3", "f32", 2000, 4096, 3.0e-6), ("SB256A3", "f32", 2000, 4096, 3.0e-6),
    ("Q_G_4", "bf16", 2000, 4096, 1.0e-6), ("Q_G_3", "bf16", 2000, 4096, 1.0e-6), ("Q_4", "f32", 1500, 14336, 1.3e-7), ("Q_G_6", "f32", 1500, 14336, 1.3e-7)])
@pytest.mark.parametrize("mean", [0.0, 1.0])
def test_gemm_integer_operands_error_with_a_mean(tfq, gpu, fmt, dtype, N, K, bound, mean):
    """Activations N(0, 1) and 1 + 0.1 N(0, 1), 9 to 333 rows, against the float64 product.  Two bf16 parts of an fp32 value
    leave out 2.5e-6 of it in the mean (uniform in the second part's half unit, 2^-17 of the value at most); a level times
    its scale is rounded once in the decoded matrix, which a mean of the activations adds up over a group, 32 of them against
    the 26 or so steps of the centred codes' sum: 9 times 2^-24, 0.5e-6 to 0.9e-6.  sqrt(2.5^2 + 0.9^2) = 2.7e-6, and 0.9e-6 without
    the parts, and a tenth for the fp32 sums.  Three parts leave nothing out: fp32 sums of 14336 terms in blocks, 1.3e-7."""
    import torch
    print(f"gemm mean {fmt} {dtype} N={N} K={K} mean={mean}", flush=True)
    g = torch.Generator(device="cuda").manual_seed(21)
    W = tfq.Weight(fmt, N, K, tfq.encode(fmt, torch.randn(N * K, device=gpu, generator=g) * 0.02))
    dense = W.decode().reshape(N, K).double()
    for M in (9, 16, 17, 64, 333):
        if dtype == "bf16" and M not in (17, 64):
            continue  # (other kernels' rows, whose rounding is their own)
        x = torch.randn(M, K, device=gpu, generator=g)
        x = x * 0.1 + mean if mean else x
        x = x.bfloat16() if dtype == "bf16" else x
        want = x.double() @ dense.T
        y = W.gemv(x) if M <= 16 else W.gemm(x, out_dtype=torch.float32)
        assert float((y.double() - want).norm() / want.norm()) <= bound, M
    W.close()


@pytest.mark.parametrize("fmt,dtype", [("Q_G_4", "f32"), ("B32S8", "bf16"), ("B32S4", "f32"), ("SB256A3", "f32"), ("SB256A2", "bf16"),
                                       ("Q_4", "f32"), ("Q_4", "bf16"), ("Q_G_6", "bf16"), ("Q_G_8", "f32")])
@pytest.mark.parametrize("M,N,K", [(40, 384, 2048), (300, 700, 1280), (257, 4100, 768)])
def test_gemm_integer_operands_any_scratch(tfq, gpu, fmt, dtype, M, N, K):
    """Every size of workspace is served, by other shapes and K splits as it shrinks: the product stays within the bounds
    above, and what lies behind the workspace and behind y stays as it was.  Where the activations' parts do not fit another
    kernel may serve: the decode kernels with their 16-bit activations (1e-5), or the bf16 tile kernel, whose weights are
    bf16 (2^-9 at most, 5e-3 as above)."""
    import ctypes as C
    import torch
    print(f"gemm {fmt} {dtype} M={M} N={N} K={K}", flush=True)
    g = torch.Generator(device="cuda").manual_seed(14)
    W = tfq.Weight(fmt, N, K, tfq.encode(fmt, torch.randn(N * K, device=gpu, generator=g) * 0.02))
    x = torch.randn(M, K, device=gpu, generator=g)
    x = x.bfloat16() if dtype == "bf16" else x
    want = x.double() @ W.decode().reshape(N, K).double().T
    bound = 1.5e-4 if fmt == "Q_G_8" else 1e-6 if dtype == "bf16" or fmt == "Q_4" else 1e-5
    lib, code = tfq.lib(), tfq.BF16 if dtype == "bf16" else tfq.F32
    need = int(lib.tfq_gemm_workspace_bytes(W.handle, code, M))
    for size in (need, need // 2 // 256 * 256, M * K * 7 // 256 * 256, M * K * 2 // 256 * 256, M * N * 8 // 256 * 256, 256):
        ws = torch.full((size + 4096,), 113, device=gpu, dtype=torch.uint8)
        y = torch.full((M * N + 1024,), 3.0, device=gpu)
        rc = lib.tfq_gemm_ws(W.handle, C.c_void_p(x.data_ptr()), code, M, C.c_void_p(y.data_ptr()), tfq.F32, C.c_void_p(ws.data_ptr()), size,
                             C.c_void_p(torch.cuda.current_stream().cuda_stream))
        assert rc == 0
        v = y[:M * N].reshape(M, N).double()
        other = 5e-3 if dtype == "bf16" and fmt == "B32S8" else max(bound, 1e-5)
        assert float((v - want).norm() / want.norm()) <= (bound if size == need else other), size
        assert bool((y[M * N:] == 3.0).all()) and bool((ws[size:] == 113).all()), size
    W.close()


@pytest.mark.parametrize("fmt,dtype", EXACT_FMTS + [(f, "bf16") for f in ("Q_G_4", "Q_G_3", "B32S4", "B32S8", "Q_G_8", "Q_8")])
@pytest.mark.parametrize("N,K", [(1, 256), (31, 896 + 128), (33, 1280), (200, 2816), (65, 4096), (96, 4352)])
def test_gemm_small_products_in_one_launch(tfq, gpu, rules, fmt, dtype, N, K):
    """Tiles of 32 x 32, K over the wavefronts of a workgroup: fewer half blocks than wavefronts, shares of different sizes, ragged
    tiles on either side.  With the workspace that is asked for the first three sizes are mostly one launch, the others K parts of
    such tiles; without it all that are served there are one launch.  Against the float64 product, the bounds of
    test_gemm_integer_operands_any_scratch (the bf16 rows' weights are not rounded either); a row's sums do not depend on
    the tile that it is in, nor on the rows beside it."""
    import torch
    g = torch.Generator(device="cuda").manual_seed(31)
    W = tfq.Weight(fmt, N, K, tfq.encode(fmt, torch.randn(N * K, device=gpu, generator=g) * 0.02))
    dense = W.decode().reshape(N, K).double()
    bound = 1.5e-4 if fmt in ("Q_G_8", "Q_8") else 1e-6 if dtype == "bf16" or fmt in ("Q_4", "Q_4_K_H", "Q_G_6") else 1e-5
    x = torch.randn(95, K, device=gpu, generator=g)
    x = x.bfloat16() if dtype == "bf16" else x
    want = x.double() @ dense.T
    for M in (17, 32, 33, 95):
        for workspace in (True, False):
            plan = rules.product(fmt, N, K, dtype == "f32", M, None if workspace else 0)
            if not workspace and (plan is None or plan.shape != rules.SOLO):
                continue  # (other kernels' rows)
            assert plan.shape == rules.SOLO and (workspace or plan.ksplit == 1)
            y = W.gemm(x[:M].contiguous(), out_dtype=torch.float32, workspace=workspace)
            assert float((y.double() - want[:M]).norm() / want[:M].norm()) <= bound, (fmt, dtype, N, K, M)
            assert torch.equal(W.gemm(x[:M].flip(0).contiguous(), out_dtype=torch.float32, workspace=workspace), y.flip(0))
    W.close()


@pytest.mark.parametrize("fmt", ["B32S4", "B32S8", "Q_G_4", "Q_G_8", "Q_8", "Q_G_3", "Q_G_2", "SB256A3", "SB256A2", "Q_4", "Q_G_6"])
@pytest.mark.parametrize("dtype", ["bf16", "f32"])
def test_gemm_small_products_longest_walk(tfq, gpu, rules, fmt, dtype):
    """Four steps of every wavefront over its LDS, each written by some lanes and read by others: the longest K in one part, which
    a call without scratch has, of ragged tiles.  Bounds as above; a row does not depend on those beside it, the whole tile's."""
    import torch
    N, K = 2017, 3072 if fmt in ("Q_4", "Q_G_6") and dtype == "f32" else 4096
    print(f"gemm longest walk {fmt} {dtype} N={N} K={K}", flush=True)
    g = torch.Generator(device="cuda").manual_seed(32)
    W = tfq.Weight(fmt, N, K, tfq.encode(fmt, torch.randn(N * K, device=gpu, generator=g) * 0.02))
    dense = W.decode().reshape(N, K).double()
    bound = 1.5e-4 if fmt in ("Q_G_8", "Q_8") else 1e-6 if dtype == "bf16" or fmt in ("Q_4", "Q_G_6") else 1e-5
    for M in (50, 95):
        plan = rules.product(fmt, N, K, dtype == "f32", M, scratch=0)
        assert (plan.shape, plan.ksplit) == (rules.SOLO, 1)
        x = torch.randn(M, K, device=gpu, generator=g)
        x = x.bfloat16() if dtype == "bf16" else x
        want = x.double() @ dense.T
        y = W.gemm(x, out_dtype=torch.float32, workspace=False)
        assert float((y.double() - want).norm() / want.norm()) <= bound, M
        assert torch.equal(W.gemm(x.flip(0).contiguous(), out_dtype=torch.float32, workspace=False), y.flip(0)), M
    W.close()


@pytest.mark.parametrize("fmt,dtype", [("B32S4", "bf16"), ("Q_G_4", "f32"), ("Q_G_8", "bf16"), ("SB256A3", "f32"), ("Q_4", "f32"), ("Q_G_6", "bf16")])
@pytest.mark.parametrize("N,K", [(96, 4608), (320, 6400), (65, 14336), (1, 15872)])
def test_gemm_small_products_in_k_parts(tfq, gpu, fmt, dtype, N, K):
    """Few tiles of a long K: eight parts of K over workgroups, of unequal length where the blocks do not divide.  Rows of a tile and of
    the next one, one to sixteen rows (gemv) and more.  The bounds of test_gemm_integer_operands_any_scratch."""
    import torch
    print(f"gemm k parts {fmt} {dtype} N={N} K={K}", flush=True)
    g = torch.Generator(device="cuda").manual_seed(33)
    W = tfq.Weight(fmt, N, K, tfq.encode(fmt, torch.randn(N * K, device=gpu, generator=g) * 0.02))
    dense = W.decode().reshape(N, K).double()
    bound = 1.5e-4 if fmt == "Q_G_8" else 1e-6 if dtype == "bf16" or fmt in ("Q_4", "Q_G_6") else 1e-5
    for M in (5, 16, 17, 32, 33, 70):
        x = torch.randn(M, K, device=gpu, generator=g)
        x = x.bfloat16() if dtype == "bf16" else x
        want = x.double() @ dense.T
        y = W.gemv(x) if M <= 16 else W.gemm(x, out_dtype=torch.float32)
        assert float((y.double() - want).norm() / want.norm()) <= bound, (M, float((y.double() - want).norm() / want.norm()))
    W.close()


@pytest.mark.parametrize("fmt,dtype,M,N,K,shape,parts", [
    ("Q_G_3", "f32", 241, 399, 2304, 4, 2), ("B32S8", "f32", 233, 294, 1792, 4, 3), ("SB256A3", "f32", 161, 53, 1536, 4, 6), ("Q_G_6", "f32", 18, 34, 1792, 4, 7),
    ("SB256A2", "f32", 208, 329, 2816, 3, 11), ("Q_G_4", "f32", 206, 228, 6912, 3, 14), ("B32S4", "f32", 228, 222, 8192, 3, 16), ("Q_4", "bf16", 241, 212, 7936, 3, 16),
    ("Q_G_8", "bf16", 232, 528, 7936, 2, 11), ("Q_G_6", "bf16", 231, 404, 7936, 2, 16)])
def test_gemm_k_parts_of_every_count(tfq, gpu, rules, fmt, dtype, M, N, K, shape, parts):
    """K parts in counts of two to sixteen: one batch of the loads of the launch that adds them, a whole and a ragged second one.
    (Bounds as above.)"""
    import torch
    plan = rules.product(fmt, N, K, dtype == "f32", M)
    assert (plan.shape, plan.ksplit) == (shape, parts)
    g = torch.Generator(device="cuda").manual_seed(34)
    W = tfq.Weight(fmt, N, K, tfq.encode(fmt, torch.randn(N * K, device=gpu, generator=g) * 0.02))
    bound = 1.5e-4 if fmt == "Q_G_8" else 1e-6 if dtype == "bf16" or fmt in ("Q_4", "Q_G_6") else 1e-5
    x = torch.randn(M, K, device=gpu, generator=g)
    x = x.bfloat16() if dtype == "bf16" else x
    want = x.double() @ W.decode().reshape(N, K).double().T
    y = W.gemm(x, out_dtype=torch.float32)
    assert float((y.double() - want).norm() / want.norm()) <= bound
    W.close()


@pytest.mark.parametrize("fmt", ["Q_4", "Q_G_6"])
def test_gemm_integer_operands_non_finite(O, tfq, gpu, fmt):
    """Infinite, not-a-number and huge activations give what the fp32 products of the 16-row path give."""
    import torch
    M, N, K = 20, 40, 512
    W = tfq.Weight(fmt, N, K, O.encode_tensor(fmt, O.rng_normal(42, N * K, 0.02)))
    x = torch.from_numpy(O.rng_normal(43, M * K, 1.0).reshape(M, K)).to(gpu)
    x[2, 7] = float("inf")
    x[3, 300] = -float("inf")
    x[4, 100] = float("nan")
    x[5] = 0
    x[5, 9] = 2.0 ** 120  # times an unscaled integer this overflows, times the weight it does not
    x[6] = 0
    x[6, 500] = 3.4e38    # its bf16 is infinite
    x[7] = float("inf")
    x[8] = float("nan")
    for xt in (x, x.bfloat16()):
        ref = torch.cat([W.gemv(xt[:16].contiguous()), W.gemv(xt[16:].contiguous())])
        y = W.gemm(xt)
        assert torch.equal(torch.isnan(W.gemm(xt, workspace=False)), torch.isnan(ref))
        assert torch.equal(torch.isnan(y), torch.isnan(ref)) and torch.equal(torch.isinf(y), torch.isinf(ref))
        assert torch.equal(y[torch.isinf(y)], ref[torch.isinf(ref)])
        f = torch.isfinite(ref)
        assert torch.allclose(y[f], ref[f], rtol=1e-4, atol=1e-5)
    W.close()


@pytest.mark.parametrize("fmt", ["Q_G_4", "Q_G_3", "B32S4", "B32S8", "Q_G_8", "Q_8"])
@pytest.mark.parametrize("M,N,K", [(64, 1000, 2048), (80, 16400, 512), (48, 4100, 4352)])
def test_gemm_infinite_bf16_activations(tfq, gpu, fmt, M, N, K):
    """An infinite bf16 activation gives the infinity (or, where the weight is zero, the NaN) of its fp32 product, whichever
    tile kernel serves the rows: with K in parts and whole."""
    import torch
    print(f"gemm inf {fmt} M={M} N={N} K={K}", flush=True)
    g = torch.Generator(device="cuda").manual_seed(31)
    W = tfq.Weight(fmt, N, K, tfq.encode(fmt, torch.randn(N * K, device=gpu, generator=g) * 0.02))
    x = torch.randn(M, K, device=gpu, generator=g).bfloat16()
    x[2, 7] = float("inf")
    x[3, 300] = -float("inf")
    x[35, 11] = x[35, K - 1] = float("inf")
    x[40, 100] = float("nan")
    want = x.double() @ W.decode().reshape(N, K).double().T
    for out in (torch.float32, torch.bfloat16):
        y = W.gemm(x, out_dtype=out).double()
        assert torch.equal(torch.isnan(y), torch.isnan(want)), (torch.isnan(y) != torch.isnan(want)).any(1).nonzero().flatten().tolist()
        assert torch.equal(torch.isposinf(y), torch.isposinf(want)) and torch.equal(torch.isneginf(y), torch.isneginf(want))
        f = torch.isfinite(want)
        assert float((y[f] - want[f]).norm() / want[f].norm()) <= TOL
    W.close()


@pytest.mark.parametrize("fmt,dtype", [f for f in EXACT_FMTS if f[0] not in ("Q_4", "Q_G_6", "Q_4_K_H")])
def test_gemm_tiled_operands_range(O, tfq, gpu, fmt, dtype):
    """Infinite, not-a-number, huge and tiny activations on the formats of the tiled layout: the same outputs are NaN as
    with the decode kernels, and what is finite there is finite and the same to fp32 rounding (an fp32 activation keeps
    16 bits).  A whole row of the largest power of two whose group sums the decode kernels hold: the tile kernel leaves
    more than a group's sum unscaled."""
    import torch
    M, N, K = 64, 40, 768
    top = {"B32S8": 111, "Q_G_8": 111, "Q_8": 111, "SB256A3": 113, "SB256A2": 114, "Q_G_2": 116}.get(fmt, 115)
    W = tfq.Weight(fmt, N, K, O.encode_tensor(fmt, O.rng_normal(42, N * K, 0.02)))
    x = torch.from_numpy(O.rng_normal(43, M * K, 1.0).reshape(M, K)).to(gpu)
    x[2, 7] = float("inf")
    x[3, 300] = -float("inf")
    x[4, 700] = float("nan")
    x[5] = 0
    x[5, 9] = 2.0 ** 120
    x[6] = 2.0 ** top
    x[7] = -(2.0 ** top)
    x[8] *= 2.0 ** (top - 3)
    x[9] *= 2.0 ** -100
    x = x.bfloat16() if dtype == "bf16" else x
    ref = torch.cat([W.gemv(x[m:m + 16].contiguous()) for m in range(0, M, 16)])
    for ws in (True, False):
        y = W.gemm(x, workspace=ws)
        assert torch.equal(torch.isnan(y), torch.isnan(ref)), (torch.isnan(y) != torch.isnan(ref)).any(1).nonzero().flatten().tolist()
        f = torch.isfinite(ref)
        assert f[6:10].all()
        assert torch.isfinite(y[f]).all(), (torch.isfinite(y) != f).any(1).nonzero().flatten().tolist()
        for m in range(M):
            if f[m].all():
                assert float((y[m].double() - ref[m].double()).norm() / ref[m].double().norm()) <= 1e-5, m
    W.close()


@pytest.mark.parametrize("fmt,dtype,M,N,K,workspace,slices", [
    ("Q_G_4", "f32", 17, 1024, 4096, False, True), ("Q_G_4", "f32", 200, 1024, 4096, False, False),
    ("B32S8", "f32", 33, 512, 14336, False, True), ("Q_G_3", "f32", 24, 512, 4096, False, True),
    ("SB256A3", "bf16", 40, 1024, 4096, False, True), ("Q_G_2", "f32", 32, 256, 14336, False, True),
    ("Q_G_6", "bf16", 17, 256, 4096, False, True), ("Q_4", "f32", 20, 14336, 1024, False, False),
    ("B32S4", "f32", 18, 28672, 4096, True, True), ("Q_G_4", "f32", 64, 28672, 4096, True, False)])
def test_gemm_rows_in_slices_or_tiles(tfq, gpu, fmt, dtype, M, N, K, workspace, slices):
    """Where a matrix makes few tiles and there is no scratch to split K, and for a few fp32 rows on a tall matrix, the
    rows go through the decode kernels 16 at a time, bit for bit; both ways are the product (float64, the decoded matrix)."""
    import torch
    g = torch.Generator(device="cuda").manual_seed(11)
    W = tfq.Weight(fmt, N, K, tfq.encode(fmt, torch.randn(N * K, device=gpu, generator=g) * 0.02))
    x = torch.randn(M, K, device=gpu, generator=g)
    x = x.bfloat16() if dtype == "bf16" else x
    y = W.gemm(x, workspace=workspace)
    rows = torch.cat([W.gemv(x[m:m + 16].contiguous()) for m in range(0, M, 16)])
    if K <= 4096:  # (a longer K is split by gemv's own workspace, which the slices of a call without one do not have)
        assert torch.equal(y, rows) == slices
    want = x.double() @ W.decode().reshape(N, K).double().T
    for v in (y, rows):
        assert float((v.double() - want).norm() / want.norm()) <= 1e-5  # 16 bits of an fp32 activation, as above
    W.close()


COLD_CAPTURE = """
import importlib, sys
import torch
tfq = importlib.import_module("transformers-fusion_amd")
tfq.init(0)
for fmt, dtype, M in (("Q_4", "bf16", 20), ("Q_G_6", "f32", 40), ("Q_4", "f32", 300), ("Q_G_4", "f32", 200), ("SB256A3", "f32", 300), ("SB256A3", "bf16", 40)):
    W = tfq.Weight(fmt, 1024, 1024, tfq.encode(fmt, torch.randn(1024 * 1024, device="cuda") * 0.02))
    x = torch.randn(M, 1024, device="cuda").to(torch.bfloat16 if dtype == "bf16" else torch.float32)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        y = W.gemm(x)
    for r in range(3):
        y.zero_()
        graph.replay()
        x2 = x + 0  # the program's own work between the replays
        torch.cuda.synchronize()
        assert torch.equal(y, W.gemm(x2)), (fmt, dtype, M, r)
print("captured")
"""


def test_first_call_inside_a_capture(gpu):
    """The first prefill call of a process may be one that is being captured, for each kernel of the integer tile route."""
    import os
    import subprocess
    import sys
    root = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
    r = subprocess.run([sys.executable, "-c", COLD_CAPTURE], cwd=root, capture_output=True, text=True, timeout=100)
    assert r.returncode == 0 and "captured" in r.stdout, r.stderr[-2000:]


@pytest.mark.parametrize("M,N", [(455, 4736), (455, 4735), (453, 4738), (455, 4737)])
def test_k_parts_of_the_bf16_tiles_are_added_whole(O, tfq, gpu, M, N):
    """The launch that adds the bf16 tile kernel's K parts takes four outputs a lane where the product has a multiple of four, one
    otherwise (also two and three over a multiple): every output of either type against the float64 product of the decoded weights.
    Bound: bf16 weights (2^-9 of a term) and a bf16 result (2^-9 of it); the workspace shows the parts."""
    import torch
    K = 2048
    w = torch.randn(N * K, generator=torch.Generator().manual_seed(N)).to(gpu) * 0.02
    pay = tfq.encode("Q_8", w)
    W = tfq.Weight("Q_8", N, K, pay)
    parts = int(tfq.lib().tfq_gemm_workspace_bytes(W.handle, 1, M)) / (4 * M * N)
    assert parts in (2.0, 4.0, 8.0), parts
    dense = tfq.decode("Q_8", pay, N * K).reshape(N, K).double()
    x = torch.randn(M, K, generator=torch.Generator().manual_seed(1)).to(gpu).bfloat16()
    want, terms = x.double() @ dense.T, (x.double().abs() @ dense.abs().T)
    for dt in (torch.float32, torch.bfloat16):
        y = W.gemm(x, out_dtype=dt).double()
        assert bool(((y - want).abs() <= terms * 2.0 ** -8 * 0.5 + (want.abs() * 2.0 ** -8 if dt == torch.bfloat16 else 0.0)).all()), dt
    W.close()


def test_k_parts_of_the_bf16_tiles_one_and_four_outputs_a_lane(O, tfq, gpu):
    """Four outputs a lane add the K parts in the order of one: a matrix and the same without its last row, whose products have a multiple
    of four outputs and one more than that, agree bit for bit where they share rows."""
    import torch
    K, N, M = 2048, 4736, 455
    w = torch.randn(N * K, generator=torch.Generator().manual_seed(3)).to(gpu) * 0.02
    x = torch.randn(M, K, generator=torch.Generator().manual_seed(4)).to(gpu).bfloat16()
    whole, less = (tfq.Weight("Q_8", n, K, tfq.encode("Q_8", w[:n * K])) for n in (N, N - 1))
    parts = [int(tfq.lib().tfq_gemm_workspace_bytes(W.handle, 1, M)) / (4 * M * n) for W, n in ((whole, N), (less, N - 1))]
    assert parts[0] == parts[1] in (2.0, 4.0, 8.0), parts
    for dt in (torch.float32, torch.bfloat16):
        assert torch.equal(whole.gemm(x, out_dtype=dt)[:, :N - 1], less.gemm(x, out_dtype=dt)), dt
    whole.close()
    less.close()
