"""GPU parity of the prefill/verify GEMM (K3) through libhwk's C ABI against the oracle's
dequantize + blocked fp32 GEMM (the reference's shiftScale/Dequantize + sgemm.MulAdd).

Bar: max|Y - Y_oracle| <= 2e-3 * RMS(Y_oracle) in fp32; the fp16 output equal to RNE of the fp32
accumulator, bit for bit.
"""
import math
import os
import re

import numpy as np
import pytest
import torch

from hwnpu_amd import ops, synth

pytestmark = pytest.mark.gpu

TOL = 2e-3


def rms(a):
    return float(np.sqrt(np.mean(np.asarray(a, np.float64) ** 2)))


def check_close(got, want, tol=TOL):
    err = float(np.max(np.abs(np.asarray(got, np.float64) - np.asarray(want, np.float64))))
    assert err <= tol * rms(want), f"max|d|={err:.4g} rms={rms(want):.4g} ratio={err / rms(want):.3g}"


# K a multiple of 64: the paired form; (1, 128, 32), (130, 200, 96) and (500, 6000, 2080): the general form, the last
# in its 128 x 96 tile of two k groups with a ragged last step and partial edge tiles
@pytest.mark.parametrize("m,n,k", [(512, 6144, 2048), (5, 6144, 2048), (1, 128, 32), (130, 200, 96), (7, 1000, 4096),
                                   (256, 256, 6144), (300, 130, 2880), (500, 6000, 2080)])
def test_i8_gemm_parity(dev, orc, m, n, k):
    print(f"i8_gemm m={m} n={n} k={k}", flush=True)
    name = f"k3i8.{m}.{n}.{k}"
    x = synth.normal(m * k, name + ".x").view(m, k)
    q = synth.uniform_int(n * k, -127, 255, name + ".q", dtype=torch.int8).view(n, k)
    s = synth.uniform_real(n, 0.002, 0.02, name + ".s")
    wd = orc.i8_dequant(q.cpu().numpy(), s.cpu().numpy().view(np.uint16))
    want = orc.sgemm(x.cpu().numpy().astype(np.float32), wd, transb=True)
    y32 = ops.i8_gemm(x, q, s, "f32").cpu().numpy()
    check_close(y32, want)
    y16 = ops.i8_gemm(x, q, s, "f16").cpu().numpy()
    assert np.array_equal(y16.view(np.uint16), orc.f32_to_f16(y32))


# (1024, 2048, 6144) and (1024, 2048, 2048) are the prompt's down and o_proj shapes, (260, 1000, 4096)
# their tile with ragged rows and columns
@pytest.mark.parametrize("m,n,k", [(1024, 4096, 2048), (5, 2048, 6144), (1, 96, 64), (200, 12288, 2048), (33, 130, 32),
                                   (1024, 2048, 6144), (260, 1000, 4096), (1024, 2048, 2048)])
def test_mxfp4_gemm_parity(dev, orc, m, n, k):
    print(f"mxfp4_gemm m={m} n={n} k={k}", flush=True)
    name = f"k3mx.{m}.{n}.{k}"
    x = synth.normal(m * k, name + ".x").view(m, k)
    w, e = synth.mxfp4_normal(n, k, name + ".w", std=0.02)
    wd = orc.mxfp4_dequantize(w.cpu().numpy(), e.cpu().numpy())
    want = orc.sgemm(x.cpu().numpy().astype(np.float32), wd, transb=True)
    y32 = ops.mxfp4_gemm(x, w, e, "f32").cpu().numpy()
    check_close(y32, want)
    y16 = ops.mxfp4_gemm(x, w, e, "f16").cpu().numpy()
    assert np.array_equal(y16.view(np.uint16), orc.f32_to_f16(y32))
    # add mode
    y0 = synth.normal(m * n, name + ".y0", dtype=torch.float32).view(m, n)
    b0 = y0.cpu().numpy()
    ops.mxfp4_gemm(x, w, e, "add", y=y0)
    assert np.array_equal(y0.cpu().numpy(), (b0 + y32).astype(np.float32))


def test_mxfp4_gemm_uniform_codes(dev, orc):
    """The GEMV configuration's weights (every code, exponents -4..2) through the GEMM at m = 5."""
    m, n, k = 5, 8192, 2048
    x = synth.normal(m * k, "k3u.x").view(m, k)
    w, e = synth.mxfp4_uniform(n, k, "k3u.w")
    wd = orc.mxfp4_dequantize(w.cpu().numpy(), e.cpu().numpy())
    want = orc.sgemm(x.cpu().numpy().astype(np.float32), wd, transb=True)
    check_close(ops.mxfp4_gemm(x, w, e, "f32").cpu().numpy(), want)


def test_mxfp4_gemm_edge_exponents(dev, orc):
    """Block exponents outside [-23, 13], where a code times its scale is no fp16 value: rows whose
    scales reach 2^20 (6 * 2^20 overflows fp16) or fall to 2^-40, rows spanning 36 and 50 exponents,
    zero scales (e = 0) among normal ones. Each output column (one weight row) is checked against the
    oracle's fp32 Dequantize + sgemm relative to its own size."""
    m, n, k = 33, 96, 256
    rng = np.random.default_rng(11)
    x = synth.normal(m * k, "k3edge.x").view(m, k)
    w = rng.integers(0, 256, (n, k // 2), dtype=np.uint8)
    e = np.empty((n, k // 32), np.int64)
    nb = k // 32
    e[0:16] = rng.integers(127 + 10, 127 + 21, (16, nb))   # scales up to 2^20
    e[16:32] = rng.integers(127 - 40, 127 - 29, (16, nb))  # down to 2^-40
    e[32:48] = rng.integers(127 - 21, 127 + 16, (16, nb))  # a span of 36
    e[48:64] = rng.integers(127 - 4, 127 + 3, (16, nb))    # the usual range
    e[64:80] = rng.integers(127 - 4, 127 + 3, (16, nb))
    e[64:80, ::3] = 0                                       # zero scales among them
    e[80:96] = rng.integers(127 - 4, 127 + 3, (16, nb))
    e[80:96, 0] = 127 + 20                                  # a span of 50: the 2^-30 blocks lose
    e[80:96, 1] = 127 - 30                                  # bits below 2^-24 of the shifted scale
    e = e.astype(np.uint8)
    wd = orc.mxfp4_dequantize(w, e)
    want = orc.sgemm(x.cpu().numpy().astype(np.float32), wd, transb=True)
    got = ops.mxfp4_gemm(x, torch.from_numpy(w).cuda(), torch.from_numpy(e).cuda(), "f32").cpu().numpy()
    assert np.all(np.isfinite(got))
    for j in range(n):
        col_rms = rms(want[:, j])
        err = float(np.max(np.abs(got[:, j].astype(np.float64) - want[:, j])))
        assert err <= TOL * col_rms, f"column {j}: max|d|={err:.4g} rms={col_rms:.4g}"


@pytest.mark.parametrize("kind,m,n,k", [("mx", 1024, 3072, 2048), ("mx", 33, 96, 256), ("mx", 5, 512, 6144),
                                        ("i8", 200, 1536, 2048), ("i8", 7, 32, 96), ("i8", 512, 6144, 2048)])
def test_gemm_swiglu_output(dev, kind, m, n, k):
    """out_mode "swiglu" (the prompt's gate/up projection with its SwiGLU in the epilogue) equals the
    fp32 output followed by hwk_silu_mul over the column pairs (g, u) = (2c, 2c+1), bit for bit; both
    of those are pinned to the oracle on their own (the parity tests above, test_glue_gpu)."""
    print(f"gemm swiglu {kind} m={m} n={n} k={k}", flush=True)
    name = f"k3sw.{kind}.{m}.{n}.{k}"
    x = synth.normal(m * k, name + ".x").view(m, k)
    if kind == "mx":
        w, e = synth.mxfp4_normal(n, k, name + ".w", std=0.02)
        run = lambda mode: ops.mxfp4_gemm(x, w, e, mode)  # noqa: E731
    else:
        q = synth.uniform_int(n * k, -127, 255, name + ".q", dtype=torch.int8).view(n, k)
        s = synth.uniform_real(n, 0.002, 0.02, name + ".s")
        run = lambda mode: ops.i8_gemm(x, q, s, mode)  # noqa: E731
    y32 = run("f32")
    flat = y32.view(-1)
    want = ops.silu_mul(flat, flat[1:], "f16", stride=2, n=m * n // 2).view(m, n // 2)
    got = run("swiglu")
    assert got.shape == (m, n // 2) and got.dtype == torch.float16
    assert torch.equal(got.view(torch.int16), want.view(torch.int16))


def test_gemm_swiglu_rejects_ragged_n(dev):
    x = synth.normal(4 * 64, "k3swr.x").view(4, 64)
    w, e = synth.mxfp4_normal(24, 64, "k3swr.w", std=0.02)
    with pytest.raises(Exception, match="SwiGLU"):
        ops.mxfp4_gemm(x, w, e, "swiglu")


def _source(name):
    with open(os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "hwnpu_amd", "csrc", name)) as f:
        return f.read()


def paired_tile(mx, m, n, k):
    """The index of the tile that pick_pair takes, by its rule over the table in gemm_kernels.h."""
    body = _source("gemm_kernels.h").split("#define HWK_PAIR_" + ("MX" if mx else "I8") + "(F)")[1]
    body = re.match(r"(?:.*\\\n)*.*\n", body).group(0)
    best = []
    for i, t in enumerate(re.findall(r"F\(([\d, ]+)\)", body)):
        bm, bn, _, _, _, _, res, ps = map(int, t.split(","))
        most = -(-(-(-m // bm) * -(-n // bn)) // 256)
        best.append((most * ps * k + -(-most // res) * 3900000, i))
    return min(best)[1]


def general_tile(mx, m, n):
    """The tile that gemm.hip's pick_shape takes on 256 CUs, by its rule over kShapes."""
    body = _source("gemm.hip").split("kShapes[] = {")[1].split("};")[0]
    best = []
    for t in re.findall(r"\{([\d, ]+)\}", body):
        bm, bn, wm, wn, kg = map(int, t.split(","))
        tiles, eight = -(-m // bm) * -(-n // bn), wm * wn * kg == 8
        if (mx and kg != 1) or (eight and tiles > 256):
            continue
        cost = -(-tiles // 256) * bm * bn * (1 + 32 / bm + 32 / bn) * (0.75 if eight else 1)
        best.append((cost, len(best), (bm, bn, wm, wn, kg)))
    return min(best)[2]


def check_gemm(orc, mx, m, n, k, name, odd_scales=False):
    """A product against the oracle in fp32, its fp16 and added results against its fp32 ones bit for bit."""
    x = synth.normal(m * k, name + ".x").view(m, k)
    if mx:
        w, e = synth.mxfp4_normal(n, k, name + ".w", std=0.02)
        if odd_scales:
            room = torch.empty(e.numel() + 1, dtype=torch.uint8, device="cuda")
            room[1:] = e.view(-1)
            e = room[1:].view(e.shape)
            assert e.data_ptr() % 2 == 1
        wd = orc.mxfp4_dequantize(w.cpu().numpy(), e.cpu().numpy())
        run = lambda mode, y=None: ops.mxfp4_gemm(x, w, e, mode, y=y)  # noqa: E731
    else:
        q = synth.uniform_int(n * k, -127, 255, name + ".q", dtype=torch.int8).view(n, k)
        s = synth.uniform_real(n, 0.002, 0.02, name + ".s")
        wd = orc.i8_dequant(q.cpu().numpy(), s.cpu().numpy().view(np.uint16))
        run = lambda mode, y=None: ops.i8_gemm(x, q, s, mode, y=y)  # noqa: E731
    want = orc.sgemm(x.cpu().numpy().astype(np.float32), wd, transb=True)
    y32 = run("f32").cpu().numpy()
    check_close(y32, want)
    assert np.array_equal(run("f16").cpu().numpy().view(np.uint16), orc.f32_to_f16(y32))
    y0 = synth.normal(m * n, name + ".y0", dtype=torch.float32).view(m, n)
    b0 = y0.cpu().numpy()
    run("add", y0)
    assert np.array_equal(y0.cpu().numpy(), (b0 + y32).astype(np.float32))


# A case for each tile of the paired form (HWK_PAIR_MX, HWK_PAIR_I8, in the tables' order), with rows and columns left
# over: with one step of 64 values (fewer than its k groups and ring stages), with three (a ring's stages once), and
# with a number past the ring that its k groups do not divide.
PAIR_K = 832
PAIR_MX = [(898, 6152), (898, 4100), (450, 4100), (289, 4100), (198, 4100), (65, 6152), (37, 4100), (23, 4100), (9, 130)]
PAIR_I8 = [(390, 11044), (387, 6152), (450, 4100), (198, 4100), (65, 6152), (37, 4100), (23, 4100), (9, 130)]


@pytest.mark.parametrize("k", [64, 192, PAIR_K])
@pytest.mark.parametrize("mx,tile,m,n", [(True, i, m, n) for i, (m, n) in enumerate(PAIR_MX)] +
                         [(False, i, m, n) for i, (m, n) in enumerate(PAIR_I8)] + [(False, None, 898, 4100)])
def test_gemm_paired_tiles(dev, orc, mx, tile, m, n, k):
    print(f"gemm tiles mx={mx} tile={tile} {m}x{n}x{k}", flush=True)
    assert tile is None or paired_tile(mx, m, n, k) == tile
    check_gemm(orc, mx, m, n, k, f"k3pair.{mx}.{m}.{n}.{k}")


# A case for each tile of the general form (kShapes), K 32 past a multiple of 64: three steps of 128 values, the last
# of 96, and one of 96 alone; rows and columns left over.
GENERAL = [(True, (128, 64, 2, 4, 1), 33, 100), (True, (64, 128, 2, 2, 1), 146, 8200), (True, (128, 128, 2, 4, 1), 204, 8200),
           (True, (128, 96, 2, 2, 1), 523, 7212), (True, (128, 64, 2, 2, 1), 668, 5392), (True, (128, 128, 2, 2, 1), 668, 8876),
           (False, (128, 64, 2, 4, 1), 33, 100), (False, (64, 128, 2, 2, 1), 146, 8200), (False, (128, 96, 2, 2, 2), 204, 8200),
           (False, (128, 128, 2, 4, 1), 262, 8200), (False, (128, 96, 2, 2, 1), 523, 7212), (False, (128, 64, 2, 2, 1), 668, 5392),
           (False, (128, 128, 2, 2, 1), 668, 8876)]


@pytest.mark.parametrize("k", [96, 352])
@pytest.mark.parametrize("mx,tile,m,n", GENERAL)
def test_gemm_general_tiles(dev, orc, mx, tile, m, n, k):
    print(f"gemm general tiles mx={mx} tile={tile} {m}x{n}x{k}", flush=True)
    assert general_tile(mx, m, n) == tile
    check_gemm(orc, mx, m, n, k, f"k3gen.{mx}.{m}.{n}.{k}")


@pytest.mark.parametrize("m,n,k", [(37, 200, 128), (300, 130, 832)])
def test_mxfp4_gemm_odd_scale_address(dev, orc, m, n, k):
    """Scales that start at an odd address: the general form at a K that the paired one takes otherwise."""
    check_gemm(orc, True, m, n, k, f"k3odd.{m}.{n}.{k}", odd_scales=True)


@pytest.mark.parametrize("m,n,k", [(898, 6144, 64), (450, 4096, 192), (65, 6144, 192), (9, 128, PAIR_K)])
def test_mxfp4_gemm_shifted_tiles(dev, orc, m, n, k):
    """Rows whose exponents leave [-23, 13] in single tiles of a wide product (one k group and several): those
    tiles run again with their rows shifted, the others do not, and every column meets the oracle at its
    own size; the SwiGLU output equals that of the fp32 one."""
    rng = np.random.default_rng(m + n)
    x = synth.normal(m * k, f"k3shift.{m}.x").view(m, k)
    w = rng.integers(0, 256, (n, k // 2), dtype=np.uint8)
    e = rng.integers(127 - 9, 127 - 6, (n, k // 32))
    e[5] = 127 + 15 + np.arange(k // 32) % 4
    e[n // 2 + 3] = 127 - 30 - np.arange(k // 32) % 3
    e[n - 1, ::2] = 0
    e = e.astype(np.uint8)
    want = orc.sgemm(x.cpu().numpy().astype(np.float32), orc.mxfp4_dequantize(w, e), transb=True)
    wt, et = torch.from_numpy(w).cuda(), torch.from_numpy(e).cuda()
    y = ops.mxfp4_gemm(x, wt, et, "f32")
    got = y.cpu().numpy().astype(np.float64)
    col = np.sqrt(np.mean(want.astype(np.float64) ** 2, 0))
    assert np.all(np.max(np.abs(got - want), 0) <= TOL * col)
    flat = y.view(-1)
    want16 = ops.silu_mul(flat, flat[1:], "f16", stride=2, n=m * n // 2).view(m, n // 2)
    assert torch.equal(ops.mxfp4_gemm(x, wt, et, "swiglu").view(torch.int16), want16.view(torch.int16))


def test_mxfp4_gemm_zero_blocks_run_once(dev):
    """The encoder gives an all-zero block the scale byte 0, which needs no shift: a product over weights with such a
    block in every row gives the bits of the same weights with zero codes under an ordinary scale, in the same time
    (a tile that runs again takes about twice; the bound is halfway)."""
    m, n, k = 2048, 8192, 2048
    x = synth.normal(m * k, "k3zero.x").view(m, k)
    dense = synth.normal(n * k, "k3zero.w", std=0.02, dtype=torch.float32).view(n, k)
    dense[:, 64:96] = 0
    w, e = ops.mxfp4_encode(dense)
    assert int(e[:, 2].max()) == 0 and int(e[:, [0, 1, 3]].min()) > 104
    plain = e.clone()
    plain[:, 2] = 120
    y = [ops.mxfp4_gemm(x, w, s, "f32") for s in (e, plain)]
    assert torch.equal(y[0].view(torch.int32), y[1].view(torch.int32))
    best = [math.inf, math.inf]
    for _ in range(10):
        for i, s in enumerate((e, plain)):
            a, b = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
            a.record()
            for _ in range(5):
                ops.mxfp4_gemm(x, w, s, "f32", y=y[0])
            b.record()
            b.synchronize()
            best[i] = min(best[i], a.elapsed_time(b) * 200)
    print(f"zero blocks {best[0]:.1f} us, none {best[1]:.1f} us", flush=True)
    assert best[0] <= 1.5 * best[1]
