"""One-pass decode GEMM for 1..64 rows (qe_matmul_w4_onepass_ex, wdec.hip) through the C-ABI vs the CPU oracle.

The kernel has the decode kernels' arithmetic: the exact products (u - 8) x summed in fp32 (as (128 + u) x and
-136 x on the matrix cores) and scaled once per 128-k group, i.e. the unrounded weights (u - 8) s: its fp32 output
is within 1e-4 * rms of the float64 product on those weights (the skinny kernel's gate), and inside the BASELINE
gate (2e-2 * rms) of the oracle's reference on the bf16 operand bf16_rn((u - 8) s). bf16 outputs are the RN of the
fp32 ones, GLU outputs silu(gate) up of the same sums. Rows of one call do not depend on each other (rows past m are
never stored), and the result does not depend on timing.
"""
import numpy as np
import pytest
import torch

import oracle
from qengine_amd import ops, synth
from test_gemv_gpu import (assert_gate, assert_glu_close, assert_rn_of, err_ratio, exact_w4, glu_act, matmul_f64,
                           oracle_ref, out_f32, setup_w4)

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,k", [(17408, 5120), (5120, 5120), (2048, 2048)])
@pytest.mark.parametrize("m", [1, 5, 32, 33, 64])
def test_onepass_vs_oracle(dev, n, k, m):
    """fp32 output within 1e-4 * rms of the float64 product on the unrounded weights and inside the BASELINE gate of
    the oracle's reference; the bf16 output is its RN bit for bit"""
    w, q, s = setup_w4(n, k, 1, seed=60 + m)
    xh = synth.x_host(m, k, seed=61 + m)
    x = synth.to_dev(xh)
    y = ops.matmul_w4_onepass(w, x)
    yb = ops.matmul_w4_onepass(w, x, out_bf16=True)
    torch.cuda.synchronize()
    assert y is not None and yb is not None
    r = err_ratio(y.cpu().numpy(), matmul_f64(xh, exact_w4(q, s, n, k, 1)))
    print(f"onepass n={n} k={k} m={m}: max|y - exact| / rms = {r:.2e}", flush=True)
    assert r <= 1e-4
    assert_gate(y.cpu().numpy(), oracle_ref(xh, q, s, n, k, 1), f"onepass n={n} k={k} m={m}")
    assert_rn_of(yb, y.cpu().numpy(), f"onepass m={m}")


@pytest.mark.parametrize("m", [7, 40])
def test_onepass_glu_and_bf16_scales(dev, m):
    """GLU matrices (the bf16 activation silu(gate) up, n / 2 columns) with fp16 scales, and plain bf16 scales"""
    n, k = 4096, 2048
    wg, qg, sg = setup_w4(n, k, 1, seed=70 + m, glu=True)
    xh = synth.x_host(m, k, seed=71 + m)
    x = synth.to_dev(xh)
    a = ops.matmul_w4_onepass(wg, x)
    wb, qb, sb = setup_w4(n, k, 0, seed=72 + m)
    yb = ops.matmul_w4_onepass(wb, x)
    torch.cuda.synchronize()
    act = glu_act(matmul_f64(xh, exact_w4(qg, sg, n, k, 1)))
    assert_glu_close(out_f32(a), act, 1e-4)
    assert err_ratio(yb.cpu().numpy(), matmul_f64(xh, exact_w4(qb, sb, n, k, 0))) <= 1e-4


def test_onepass_rows_independent_and_deterministic(dev):
    """a row's bits do not depend on the other rows of the call within a token-block count (m <= 32: one block of
    32; 33..64: two), and repeated calls are bit-identical"""
    n, k = 5120, 5120
    w, q, s = setup_w4(n, k, 1, seed=80)
    x = synth.to_dev(synth.x_host(64, k, seed=81))
    y64 = ops.matmul_w4_onepass(w, x).cpu().numpy().view(np.uint32)
    y40 = ops.matmul_w4_onepass(w, x[:40].contiguous()).cpu().numpy().view(np.uint32)
    y32 = ops.matmul_w4_onepass(w, x[:32].contiguous()).cpu().numpy().view(np.uint32)
    y3 = ops.matmul_w4_onepass(w, x[:3].contiguous()).cpu().numpy().view(np.uint32)
    y64b = ops.matmul_w4_onepass(w, x).cpu().numpy().view(np.uint32)
    assert np.array_equal(y64, y64b)
    assert np.array_equal(y40, y64[:40])
    assert np.array_equal(y3, y32[:3])


def test_onepass_shape_checks(dev):
    """shapes the kernel does not take are declined (returns None, nothing written): n % 64, an odd number of
    64-k steps per wave, x not 16-byte aligned"""
    w, _, _ = setup_w4(4096 + 16, 2048, 1, seed=90)
    x = synth.to_dev(synth.x_host(4, 2048, seed=91))
    assert ops.matmul_w4_onepass(w, x) is None
    w2, _, _ = setup_w4(1024, 1280, 1, seed=92)  # 20 steps: 5 per wave at m <= 32
    assert ops.matmul_w4_onepass(w2, synth.to_dev(synth.x_host(4, 1280, seed=93))) is None
    xb = torch.zeros(4 * 2048 + 1, dtype=torch.bfloat16, device=dev)[1:].view(4, 2048)
    w3, _, _ = setup_w4(1024, 2048, 1, seed=94)
    assert ops.matmul_w4_onepass(w3, xb) is None


@pytest.mark.parametrize("n,k", [(64, 128), (192, 384), (1024, 1280), (4160, 640)])
def test_onepass_33_rows_take_any_groups(dev, n, k):
    """33..64 rows: any whole number of 128-k groups is taken (up to 32 rows K % 512 == 0), other shapes are declined"""
    w, q, s = setup_w4(n, k, 1, seed=n)
    xh = synth.x_host(40, k, seed=k)
    x = synth.to_dev(xh)
    y = ops.matmul_w4_onepass(w, x)
    assert y is not None
    assert err_ratio(out_f32(y), matmul_f64(xh, exact_w4(q, s, n, k, 1))) <= 1e-4
    assert ops.matmul_w4_onepass(w, x[:32]) is None
    odd, _, _ = setup_w4(n + 16, k, 1, seed=n)
    assert ops.matmul_w4_onepass(odd, x) is None
    xb = torch.zeros(40 * k + 1, dtype=torch.bfloat16, device=dev)[1:].view(40, k)
    assert ops.matmul_w4_onepass(w, xb) is None


def test_onepass_tail_parts_deterministic_and_graph(dev):
    """N = 17408 has 272 slabs of 64 rows (33..48 rows take these too, two token blocks): the 16 past the last whole round of
    256 CUs run as K parts added by the last part to finish (a device-side count per tail slab, zero again after every call). Repeated calls, calls of
    other shapes in between, and a HIP graph captured on a stream that ran the kernel eagerly all give the same bits;
    a capture on a stream that never ran it within 1e-5 * rms (test_workspace_gpu.py: the same bits)"""
    n, k = 17408, 5120
    w, q, s = setup_w4(n, k, 1, seed=95)
    xh = synth.x_host(40, k, seed=96)
    x = synth.to_dev(xh)
    exact = matmul_f64(xh, exact_w4(q, s, n, k, 1))
    iv = torch.int32
    for m in (40, 8):
        xm = x[:m].contiguous()
        y1 = ops.matmul_w4_onepass(w, xm)
        w2, _, _ = setup_w4(4096, 2048, 1, seed=97)
        ops.matmul_w4_onepass(w2, synth.to_dev(synth.x_host(3, 2048, seed=98)))  # another shape in between
        y2 = ops.matmul_w4_onepass(w, xm)
        torch.cuda.synchronize()
        assert torch.equal(y1.view(iv), y2.view(iv)), m
        assert err_ratio(y1.cpu().numpy(), exact[:m]) <= 1e-4
        for warm in (True, False):
            cs = torch.cuda.Stream()
            cs.wait_stream(torch.cuda.current_stream())
            x_in = xm.clone()
            out = torch.empty(m, n, dtype=torch.float32, device=dev)
            if warm:
                with torch.cuda.stream(cs):
                    ops.matmul_w4_onepass(w, x_in, y=out)
            torch.cuda.synchronize()
            g = torch.cuda.CUDAGraph()
            with torch.cuda.graph(g, stream=cs):
                ops.matmul_w4_onepass(w, x_in, y=out)
            for r in range(3):
                xr = synth.to_dev(synth.x_host(m, k, seed=100 + r))
                want = ops.matmul_w4_onepass(w, xr)
                torch.cuda.synchronize()
                x_in.copy_(xr)
                g.replay()
                torch.cuda.synchronize()
                if warm:
                    assert torch.equal(out.view(iv), want.view(iv)), (m, r)
                else:
                    rr = err_ratio(out.cpu().numpy(), want.cpu().numpy())
                    assert rr <= 1e-5, (m, r, rr)


@pytest.mark.parametrize("n,k", [(64, 128), (192, 384), (4160, 640), (5120, 3712), (33024, 256), (4160, 3712),
                                 (32896, 896), (33088, 896)])
@pytest.mark.parametrize("m", [33, 48, 63, 64])
def test_decode_33_to_64_rows(dev, n, k, m):
    """the 33..64-row kernels through the row-count dispatch (skinny launches at 4160 x 640, 64-row slabs at 33024 x 256,
    else 128-row slabs) and alone: slabs with a ragged half (n % 128 = 64), K of fewer groups than K parts, uneven K
    parts, every slab split in K ranges (5120 and 4160 x 3712, the last ragged there), 256 whole slabs and 1 or 3 split
    ones (896, the last ragged at 33088); outputs at an odd offset and stride are the contiguous ones bit for bit; GLU"""
    w, q, s = setup_w4(n, k, 1, seed=n + m)
    xh = synth.x_host(m, k, seed=k + m)
    x = synth.to_dev(xh)
    y = ops.matmul_w4(w, x)
    assert err_ratio(out_f32(y), matmul_f64(xh, exact_w4(q, s, n, k, 1))) <= 1e-4
    big = torch.full((m, n + 7), float("nan"), dtype=torch.float32, device=dev)
    z = ops.matmul_w4(w, x, y=big[:, 1:1 + n])
    assert torch.equal(z.contiguous().view(torch.int32), y.view(torch.int32))
    assert torch.isnan(big[:, 0]).all() and torch.isnan(big[:, 1 + n:]).all()
    wg, qg, sg = setup_w4(n, k, 1, seed=n + m + 1, glu=True)
    a = ops.matmul_w4(wg, x)
    assert_glu_close(out_f32(a), glu_act(matmul_f64(xh, exact_w4(qg, sg, n, k, 1))), 1e-4)
    y1 = ops.matmul_w4_onepass(w, x)
    assert err_ratio(out_f32(y1), matmul_f64(xh, exact_w4(q, s, n, k, 1))) <= 1e-4
    assert torch.equal(ops.matmul_w4_onepass(w, x), y1)


@pytest.mark.parametrize("n,k", [(16384, 256), (9216, 512), (16384, 1024), (17408, 3072), (43008, 512), (49152, 512)])
@pytest.mark.parametrize("m", [33, 48, 64])
def test_decode_33_to_64_rows_small_slabs(dev, n, k, m):
    """33..64 rows where the 64-row slabs are the faster ones (one round of them, tail parts just past it up to 48 rows,
    short K) or the skinny launches are still taken (9216 x 512): the exact product, GLU, and outputs at an odd offset and stride"""
    w, q, s = setup_w4(n, k, 1, seed=n + m)
    xh = synth.x_host(m, k, seed=k + m)
    x = synth.to_dev(xh)
    y = ops.matmul_w4(w, x)
    assert err_ratio(out_f32(y), matmul_f64(xh, exact_w4(q, s, n, k, 1))) <= 1e-4
    big = torch.full((m, n + 7), float("nan"), dtype=torch.float32, device=dev)
    z = ops.matmul_w4(w, x, y=big[:, 1:1 + n])
    assert torch.equal(z.contiguous().view(torch.int32), y.view(torch.int32))
    assert torch.isnan(big[:, 0]).all() and torch.isnan(big[:, 1 + n:]).all()
    wg, qg, sg = setup_w4(n, k, 1, seed=n + m + 1, glu=True)
    a = ops.matmul_w4(wg, x)
    assert_glu_close(out_f32(a), glu_act(matmul_f64(xh, exact_w4(qg, sg, n, k, 1))), 1e-4)


@pytest.mark.parametrize("n,k", [(16384, 256), (16384, 1024)])
def test_decode_64_rows_one_pass_of_small_slabs(dev, n, k):
    """one round of 64-row slabs over a short K: the dispatch takes the one-pass kernel, which needs 0.4 to 0.7 of the
    time of the skinny launches that batch_invariant takes (MI355X: 5.1 against 13.3 us, 8.2 against 12.3 us). Best of
    5 replays of a graph of 20 calls each"""
    w, _, _ = setup_w4(n, k, 1, seed=7)
    x = synth.to_dev(synth.x_host(64, k, seed=8))
    y = torch.empty(64, n, dtype=torch.bfloat16, device=dev)

    def us():
        st = torch.cuda.Stream()
        st.wait_stream(torch.cuda.current_stream())
        with torch.cuda.stream(st):
            ops.matmul_w4(w, x, out_bf16=True, y=y)
        torch.cuda.synchronize()
        g = torch.cuda.CUDAGraph()
        with torch.cuda.graph(g, stream=st):
            for _ in range(20):
                ops.matmul_w4(w, x, out_bf16=True, y=y)
        best = float("inf")
        for _ in range(5):
            e0, e1 = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
            e0.record()
            g.replay()
            e1.record()
            torch.cuda.synchronize()
            best = min(best, e0.elapsed_time(e1) * 50)
        return best

    one = us()
    old = ops.set_config(batch_invariant=1)
    try:
        skinny = us()
    finally:
        ops.set_config(**old)
    print(f"{n} x {k}, m = 64: {one:.2f} us, skinny {skinny:.2f} us", flush=True)
    assert one < 0.85 * skinny
