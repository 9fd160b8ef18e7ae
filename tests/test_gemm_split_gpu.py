"""Prefill GEMM calls whose tiles do not fill the CUs, against the oracle (1e-4 * rms: the products are the oracle's, only
the order of the fp32 sums differs): what the cost model picks there (mostly 128 x 128 tiles in 9, 5 or 1 ranges at these
sizes), and each of the four tile shapes with 1, 3, 10 and 16 ranges for every weight format. K = 1152 and 2176 are 9
and 17 groups (ranges of unequal length), t crosses the 128- and 256-token tiles, n leaves ragged row tiles."""
import ctypes

import numpy as np
import pytest
import torch

import oracle
from qengine_amd import call, lib, ops, synth
from test_gemm_gpu import setup
from test_gemv_gpu import assert_glu_close, err_ratio, glu_act, matmul_f64, oracle_ref, oracle_ref_w8, out_f32
from test_q8_gpu import q8_host

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,k,t", [(272, 1152, 65), (2976, 2176, 75), (144, 2176, 128), (1040, 1152, 129),
                                   (528, 2176, 257), (4112, 1152, 300), (2048, 128, 200), (272, 1152, 1100)])
@pytest.mark.parametrize("glu", [False, True])
def test_underfilled_prefill(dev, n, k, t, glu):
    w, q, s = setup(n, k, 1, seed=n + t, glu=glu)
    xh = synth.x_host(t, k, seed=t)
    x = synth.to_dev(xh)
    rows = np.unique(np.r_[0, t // 2, 127 % t, 128 % t, t - 1, np.random.default_rng(t).integers(0, t, 8)])
    if glu:
        act = glu_act(oracle_ref(xh[rows], q, s, n, k, 1))
        y = ops.gemm_w4(w, x)
        assert_glu_close(out_f32(y)[rows], act, 1e-4)
        cols = n // 2
    else:
        ref = oracle_ref(xh, q, s, n, k, 1)
        y = ops.gemm_w4(w, x, out_bf16=True)
        y32 = ops.gemm_w4(w, x)
        assert err_ratio(out_f32(y32), ref) <= 1e-4
        assert torch.equal(y32.bfloat16().view(torch.int16), y.view(torch.int16))
        cols = n
    # rows of an odd stride at an odd offset (scalar stores, also of the split tiles' sums)
    big = torch.full((t, cols + 7), float("nan"), dtype=torch.bfloat16, device=dev)
    got = ops.gemm_w4(w, x, out_bf16=True, y=big[:, 1:1 + cols])
    assert torch.equal(got.contiguous().view(torch.int16), y.view(torch.int16))
    assert torch.isnan(big[:, 0]).all() and torch.isnan(big[:, 1 + cols:]).all()


@pytest.mark.parametrize("per_channel", [True, False])
def test_underfilled_prefill_w8(dev, per_channel):
    n, k, t = 272, 1152, 140
    q, s = synth.w8_host(n, k, seed=3, per_channel=per_channel)
    w = ops.tile_w8(synth.to_dev(q), synth.to_dev(s, torch.float16), per_channel)
    xh = synth.x_host(t, k, seed=4)
    y = ops.gemm_w8(w, synth.to_dev(xh))
    assert err_ratio(out_f32(y), oracle_ref_w8(xh, q, s, n, k, per_channel)) <= 1e-4


def test_capture_without_workspace_runs_unsplit(dev):
    """a split needs a workspace of its stream: a capture on a stream that has none runs the unsplit GEMM, and every
    replay gives the eager unsplit bits"""
    n, k, t = 272, 2176, 100
    w, q, s = setup(n, k, 1, seed=21)
    x = synth.to_dev(synth.x_host(t, k, seed=22))
    call("qe_gemm_set_sk_maxparts", 1)
    try:
        want = ops.gemm_w4(w, x)
    finally:
        call("qe_gemm_set_sk_maxparts", 0)
    eager = ops.gemm_w4(w, x)
    y = torch.empty_like(want)
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g, stream=torch.cuda.Stream()):
        ops.gemm_w4(w, x, y=y)
    for _ in range(3):
        y.zero_()
        g.replay()
        torch.cuda.synchronize()
        assert torch.equal(y.view(torch.int32), want.view(torch.int32))
    assert err_ratio(eager.cpu().numpy(), want.cpu().numpy()) <= 1e-5


def test_tune_file_with_two_tile_shapes(dev, tmp_path):
    """a tuning file that lists 256 x 256 and 256 x 128 tiles and splits 1, 2, 4 is still read; a choice outside that
    list makes it malformed"""
    lib().qe_gemm_tune_entries.restype = ctypes.c_int
    p = tmp_path / "tune.txt"
    head = "qengine_amd gemm tune v1 cfg=256x256,256x128 ks=1,2,4\ndevice 0000:00:00.0 256\n"
    call("qe_gemm_tune_clear")
    try:
        p.write_text(head + "0 2048 1024 512 0 1 2\n")
        call("qe_gemm_tune_file", ctypes.c_char_p(str(p).encode()))
        assert lib().qe_gemm_tune_entries() == 1
        call("qe_gemm_tune_clear")
        p.write_text(head + "0 2048 1024 512 0 2 2\n")
        call("qe_gemm_tune_file", ctypes.c_char_p(str(p).encode()))
        assert lib().qe_gemm_tune_entries() == 0
    finally:
        call("qe_gemm_tune_file", ctypes.c_char_p(b""))
        call("qe_gemm_tune_clear")


@pytest.fixture
def stored(tmp_path):
    """stored((fmt, n, k, bucket, glu, cfg, ks), ..): a tuning file of these choices for this device is loaded (fmt 0 W4,
    1 W8 group scales, 2 W8 per channel, 3 Q8)"""
    p = tmp_path / "tune.txt"

    def load(*entries):
        call("qe_gemm_tune_clear")
        call("qe_gemm_tune_file", ctypes.c_char_p(str(p).encode()))
        w, _, _ = setup(64, 128, 0, seed=1)
        y = torch.empty(70, 64, device="cuda")
        call("qe_gemm_w4_t", w.q, w.s, 64, 128, synth.to_dev(synth.x_host(70, 128, seed=1)), y, 70)  # writes the file
        head = p.read_text().splitlines()[:2]  # format and device
        p.write_text("\n".join(head + [" ".join(map(str, e)) for e in entries]) + "\n")
        call("qe_gemm_tune_clear")
        call("qe_gemm_tune_file", ctypes.c_char_p(str(p).encode()))
        lib().qe_gemm_tune_entries.restype = ctypes.c_int
        assert lib().qe_gemm_tune_entries() == len(entries)

    yield load
    call("qe_gemm_tune_file", ctypes.c_char_p(b""))
    call("qe_gemm_tune_clear")


def _us(f, calls=10):
    best = float("inf")
    f()
    for _ in range(5):
        e0, e1 = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
        e0.record()
        for _ in range(calls):
            f()
        e1.record()
        torch.cuda.synchronize()
        best = min(best, e0.elapsed_time(e1) * 1e3 / calls)
    return best


TILE = (1040, 2176, 270)  # 10 to 27 tiles: every one split
_FMT = {}


def _format(fmt):
    """(run(x), the oracle's product or GLU activation of the inputs, format number) of a weight format at TILE"""
    if fmt not in _FMT:
        n, k, t = TILE
        xh = synth.x_host(t, k, seed=41)
        glu = fmt.endswith("glu")
        if fmt.startswith("w4"):
            w, q, s = setup(n, k, 1, seed=42, glu=glu)
            run, ref, num = None, oracle_ref(xh, q, s, n, k, 1), 0
        elif fmt.startswith("q8"):
            q, s, _ = q8_host(n, k, 43)
            w = ops.repack_q8(synth.to_dev(q), synth.to_dev(s), glu=glu)
            if glu:
                q, s = oracle.glu_rows(q, s, n, k, bits=8)
            run, ref, num = ops.gemm_q8, matmul_f64(xh, oracle.bf16_to_f32(oracle.dequant_q8(q, s, n, k))), 3
        else:
            pc = fmt == "w8c"
            q, s = synth.w8_host(n, k, seed=44, per_channel=pc)
            w = ops.tile_w8(synth.to_dev(q), synth.to_dev(s, torch.float16), pc)
            run, ref, num = ops.gemm_w8, oracle_ref_w8(xh, q, s, n, k, pc), 2 if pc else 1
        _FMT[fmt] = w, run, glu_act(ref) if glu else ref, num, synth.to_dev(xh)
    return _FMT[fmt]


@pytest.mark.parametrize("ks", [1, 3, 10, 16])
@pytest.mark.parametrize("cfg", [0, 1, 2, 3])
@pytest.mark.parametrize("fmt", ["w4", "w4glu", "w8g", "w8c", "q8", "q8glu"])
def test_every_tile_shape_and_split(dev, stored, fmt, cfg, ks):
    """a given tile shape and split (INT4 by the hook, the others by a tuning file): the oracle's product, and where it is
    split other bits than unsplit"""
    n, k, t = TILE
    w, run, ref, num, x = _format(fmt)
    glu = fmt.endswith("glu")
    if run is None:
        y, applied = ops.gemm_w4_choice(w, x, cfg, ks)
        one, _ = ops.gemm_w4_choice(w, x, cfg, 1)
        assert applied == (ks > 1)
    else:
        stored((num, n, k, 512, int(glu), cfg, ks))
        y = run(w, x)
        stored((num, n, k, 512, int(glu), cfg, 1))
        one = run(w, x)
    if glu:
        assert_glu_close(out_f32(y), ref, 1e-3 if fmt == "q8glu" else 1e-4)
    else:
        assert err_ratio(out_f32(y), ref) <= 1e-4
    assert torch.equal(y, one) == (ks == 1)


@pytest.mark.parametrize("cfg", [1, 2, 3])
def test_whole_rounds_and_split_tiles(dev, cfg):
    """256 (128 x 128: 512) whole tiles and 33 to 49 of three ranges of 9 groups in one launch"""
    n, k, t = 4112, 1152, 2100
    w, q, s = setup(n, k, 1, seed=45)
    xh = synth.x_host(t, k, seed=46)
    y, applied = ops.gemm_w4_choice(w, synth.to_dev(xh), cfg, 3)
    assert applied
    rows = np.unique(np.r_[0, 127, 128, 255, 256, 1900, 1920, 2047, 2048, 2099, np.random.default_rng(1).integers(0, t, 30)])
    assert err_ratio(out_f32(y)[rows], oracle_ref(xh[rows], q, s, n, k, 1)) <= 1e-4


def test_stored_split_that_does_not_apply(dev, stored):
    """a stored choice serves every token count of its bucket. Where its split would take more than the workspace bound
    (80 tiles of 256 x 256 in 4 ranges), the call runs the untuned choice; where qe_gemm_set_sk_maxparts leaves no split,
    the best unsplit tiles, not the stored ones (5 blocks of 256 x 256 take about twice as long as 20 of 128 x 128)"""
    n, k, t = 5120, 4352, 1000
    w, _, _ = setup(n, k, 1, seed=31)
    x = synth.to_dev(synth.x_host(t, k, seed=32))
    assert not ops.gemm_w4_choice(w, x, cfg=0, ks=4)[1]
    want = ops.gemm_w4(w, x)
    assert not torch.equal(want, ops.gemm_w4_choice(w, x, cfg=0, ks=1)[0])  # (the untuned choice splits)
    stored((0, n, k, 1024, 0, 0, 4))
    assert torch.equal(ops.gemm_w4(w, x), want)

    n, k, t = 1280, 8192, 200
    w, _, _ = setup(n, k, 1, seed=33)
    x = synth.to_dev(synth.x_host(t, k, seed=34))
    big = _us(lambda: ops.gemm_w4_choice(w, x, cfg=0, ks=1))
    stored((0, n, k, 256, 0, 0, 12))
    call("qe_gemm_set_sk_maxparts", 1)
    try:
        us = _us(lambda: ops.gemm_w4(w, x))
    finally:
        call("qe_gemm_set_sk_maxparts", 0)
    print(f"1280 x 8192, t = 200 unsplit: 256 x 256 tiles {big:.1f} us, stored choice capped {us:.1f} us", flush=True)
    assert us < 0.8 * big


@pytest.mark.parametrize("n,k,t,G", [(272, 1152, 65, 64), (1040, 2176, 129, 32), (4112, 1152, 300, 128), (144, 128, 70, 64)])
@pytest.mark.parametrize("glu", [False, True])
def test_underfilled_w4a8(dev, n, k, t, G, glu):
    """W4A8 tiles split in uneven K ranges: the oracle's INT8 product to 1e-5 relative rms; rows stored through LDS
    (aligned) and one by one (an odd offset and stride) are the same bits"""
    w, q, s = setup(n, k, 1, seed=n + G, glu=glu)
    xh = synth.x_host(t, k, seed=t + 1)
    x = synth.to_dev(xh)
    xq, sx = oracle.x_to_i8(xh, G)
    ref = oracle.gemm_i8(xq, sx, oracle.unpack_w4(q, n, k), oracle.f16_to_f32(s).reshape(n, k // 128), G)
    y = ops.gemm_w4_i8(w, x, G=G, out_bf16=True)
    cols = n // 2 if glu else n
    if glu:
        assert_glu_close(out_f32(y), glu_act(ref), 1e-4)
    else:
        y32 = out_f32(ops.gemm_w4_i8(w, x, G=G)).astype(np.float64)
        assert np.sqrt(np.mean((y32 - ref) ** 2) / np.mean(ref ** 2)) < 1e-5
    big = torch.full((t, cols + 7), float("nan"), dtype=torch.bfloat16, device=dev)
    got = ops.gemm_w4_i8(w, x, G=G, out_bf16=True, y=big[:, 1:1 + cols])
    assert torch.equal(got.contiguous().view(torch.int16), y.view(torch.int16))
    assert torch.isnan(big[:, 0]).all() and torch.isnan(big[:, 1 + cols:]).all()


@pytest.mark.parametrize("n,t,out_bf16", [(272, 65, True), (272, 300, False), (528, 129, True)])
def test_w8a8_row_stores(dev, n, t, out_bf16):
    """W8A8 rows stored through LDS (16-byte aligned) and one by one (odd offset and stride): the same bits, and
    nothing outside the matrix"""
    k = 1024
    q, s = synth.w8_host(n, k, seed=n, per_channel=True)
    w = ops.tile_w8(synth.to_dev(q), synth.to_dev(s, torch.float16), True)
    x = synth.to_dev(synth.x_host(t, k, seed=t))
    dt, iv = (torch.bfloat16, torch.int16) if out_bf16 else (torch.float32, torch.int32)
    wide = torch.full((t + 1, n + 16), float("nan"), dtype=dt, device=dev)
    y = ops.gemm_w8a8(w, x, out_bf16=out_bf16, y=wide[:t, :n])
    odd = torch.full((t, n + 7), float("nan"), dtype=dt, device=dev)
    z = ops.gemm_w8a8(w, x, out_bf16=out_bf16, y=odd[:, 1:1 + n])
    assert torch.equal(y.contiguous().view(iv), z.contiguous().view(iv))
    assert torch.isnan(wide[t]).all() and torch.isnan(wide[:, n:]).all()
    assert torch.isnan(odd[:, 0]).all() and torch.isnan(odd[:, 1 + n:]).all()
