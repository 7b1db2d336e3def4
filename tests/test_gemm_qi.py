"""Prompt GEMM in the reference CPU path's arithmetic on the matrix cores (csrc/ext_gemm_qi.hip): Q8_K activation rows (engine-order RmsNorm + candle's
quantizer) x Q4_K / Q5_K / Q6_K weights through v_mfma_i32_32x32x32_i8 on exact integers (scale x quant as two int8 digits), combined in the decode engine's f32 order (ORD-U).
Every output row equals the decode engine's GEMV of that token (oracle/cpu_path_oracle.c orc_gemv_engine) BIT FOR BIT -- so does the GPU result against the
batch-1 decode kernel itself.  Also: v_mfma_f32_32x32x16_f16, which sums the mins (run sums x mins), is exact on integers below 2^24 (adversarial magnitudes)."""
import ctypes as C
import os
import re
import subprocess

import numpy as np
import pytest

from tests.abi_backends import GpuBackend, HostBackend

VP, CI = C.c_void_p, C.c_int


def run_gemm(O, be, tname, n, k, T, norm, glu=False, acc=False, seed=0, packed=None, x_override=None):
    t = getattr(O, tname)
    rng = np.random.default_rng(seed)
    if packed is None:
        packed = O.quantize(t, (rng.standard_normal((n, k)) * 0.05).astype(np.float32)).reshape(n, -1)
    nb = be.sym("mrs_gemm_qi_repack_bytes", [CI, C.c_longlong, C.c_longlong], C.c_size_t)(t, n, k)
    assert nb > 0
    src, wq = be.buf(np.ascontiguousarray(packed).reshape(-1)), be.buf(np.full(nb, 0xA5, np.uint8))
    assert be.sym("mrs_gemm_qi_repack", [VP, CI, C.c_longlong, C.c_longlong, VP, VP], CI)(src.ptr, t, n, k, wq.ptr, be.stream) == 0
    x = rng.standard_normal((T, k)).astype(np.float32)
    x2 = rng.standard_normal((T, k)).astype(np.float32) if glu else None
    if T > 2:
        x[1, : min(256, k)] = 0.0  # an all-zero activation block
    if x_override is not None:
        x = np.ascontiguousarray(x_override, dtype=np.float32)
    nw = (1.0 + 0.1 * rng.standard_normal(k)).astype(np.float32) if norm else None
    ab = be.sym("mrs_qi_act_bytes", [CI, CI], C.c_size_t)(T, k)
    act = be.buf(np.zeros(ab, np.uint8))
    xb = be.buf(x)
    x2b = be.buf(x2) if glu else None
    nwb = be.buf(nw) if norm else None
    tmp = be.buf(np.zeros((T, k), np.float32)) if glu else None
    rc = be.sym("mrs_qi_quantize_for", [CI, VP, VP, CI, VP, C.c_float, CI, CI, VP, VP, VP], CI)(t, xb.ptr, x2b.ptr if glu else None, k, nwb.ptr if norm else None, 1e-5, T, k, act.ptr,
                                                                                                   tmp.ptr if glu else None, be.stream)
    assert rc == 0, rc
    base = rng.standard_normal((T, n)).astype(np.float32) if acc else np.full((T, n), np.nan, np.float32)
    ob = be.buf(base.copy())
    rc = be.sym("mrs_gemm_qi", [VP, CI, CI, CI, VP, CI, VP, CI, CI, VP], CI)(wq.ptr, t, n, k, act.ptr, T, ob.ptr, n, 1 if acc else 0, be.stream)
    assert rc == 0, rc
    got = ob.numpy()
    # the split launch (one workgroup per run of superblocks + the reduce kernel): the same additions in the same order
    ws = be.buf(np.zeros(4 * T * n, np.float32))
    ob2 = be.buf(base.copy())
    rc = be.sym("mrs_gemm_qi_ws", [VP, CI, CI, CI, VP, CI, VP, CI, CI, VP, C.c_size_t, VP], CI)(wq.ptr, t, n, k, act.ptr, T, ob2.ptr, n, 1 if acc else 0, ws.ptr, 4 * T * n * 4, be.stream)
    assert rc == 0, rc
    assert np.array_equal(ob2.numpy(), got, equal_nan=True), "split launch differs from the single-pass launch"
    xin = O.fused_glu_engine(x, x2) if glu else x
    if norm:
        xin = O.rms_norm_engine(xin, nw, 1e-5)
    eng = np.concatenate([O.gemv_engine(t, packed, n, k, r) for r in xin], axis=0)
    want = base + eng if acc else eng
    assert np.array_equal(got, want), (tname, n, k, T, int((got != want).sum()), float(np.abs(got - want).max()))
    return packed, x, got


CASES = [("Q8_0", 40, 512, 5, 0), ("Q8_0", 66, 1280, 34, 1), ("Q8_0", 130, 1024, 133, 1), ("Q8_0", 32, 2816, 3, 0), ("Q5_K", 40, 512, 5, 0), ("Q5_K", 66, 1280, 34, 1), ("Q5_K", 32, 2816, 3, 0), ("Q4_K", 40, 512, 5, 0), ("Q4_K", 36, 1280, 4, 1), ("Q4_K", 130, 1024, 33, 1), ("Q4_K", 64, 4096, 7, 1), ("Q4_K", 33, 2816, 3, 0), ("Q6_K", 40, 512, 5, 0), ("Q6_K", 70, 1024, 130, 1),
         ("Q6_K", 32, 3584, 4, 0)]


@pytest.mark.parametrize("tname,n,k,T,norm", CASES)
def test_gemm_qi_host_emulation(oracle, tname, n, k, T, norm):
    run_gemm(oracle, HostBackend(), tname, n, k, T, norm, seed=n + k + T)


def test_gemm_qi_glu_and_accumulate_host_emulation(oracle):
    run_gemm(oracle, HostBackend(), "Q4_K", 48, 768, 6, 0, glu=True, seed=1)
    run_gemm(oracle, HostBackend(), "Q6_K", 36, 512, 9, 0, acc=True, seed=2)
    run_gemm(oracle, HostBackend(), "Q5_K", 40, 768, 6, 0, glu=True, acc=True, seed=3)
    run_gemm(oracle, HostBackend(), "Q8_0", 40, 768, 6, 0, glu=True, acc=True, seed=4)


def q5k_extreme_blocks(n, k):
    """block_q5_K bytes with every 6-bit scale 63 and every 5-bit value 31 (d = 1, dmin = 0): with activation rows whose Q8_K quants are all -128 / all 127 a superblock's
    integer sum is -64.0 M / +63.5 M -- the four f32 accumulators of the Q5_K branch each hold 16.0 M < 2^24, the largest they can be asked to"""
    blk = np.zeros(176, np.uint8)
    blk[0:2] = np.frombuffer(np.float16(1.0).tobytes(), np.uint8)
    blk[4:8] = 0xFF    # sc 0..3 = 63, top bits: the high bits of sc 4..7
    blk[8:12] = 0x00   # mn 0..3 = 0, high bits of mn 4..7 = 0
    blk[12:16] = 0x0F  # low nibbles of sc 4..7 = 15, of mn 4..7 = 0
    blk[16:176] = 0xFF  # qh, qs: every value 31
    out = np.tile(blk, (n, k // 256)).reshape(n, k // 256, 176)
    out[1::2, :, 16:176] = 0x00  # odd rows: every value 0 -- the kernel's signed operand sc (q - 16) = -1008 at its largest, isum = XA + XB + 16 S cancels to 0 exactly
    out[2::4, ::2, 16:48] = 0x00  # and rows mixing 15 / 31 by superblock
    return out.reshape(n, -1)


def run_q5k_extremes(O, be):
    n, k, T = 33, 1024, 4
    packed = q5k_extreme_blocks(n, k)
    x = np.ones((T, k), np.float32)          # all equal and positive: max = +x, iscale = -128 / x, every quant -128
    x[1] = -3.0                              # all equal and negative: every quant min(127, 128) = 127
    x[2, ::2] = -1.0                         # alternating signs: the first maximum is +1 -> quants -128 / +127
    x[3, :256] = 0.0
    run_gemm(O, be, "Q5_K", n, k, T, 0, seed=5, packed=packed, x_override=x)


def digit_extreme_blocks(tname, n, k):
    """Blocks at the ends of the weight operand's digits.  Q4_K: every scale and min 63, values 15 (sc q = 945, both digits 105), 0, or a mix;  Q6_K: scales -128 / 127 and values
    0 / 63 (sc (q - 32) = 4096, -3968, -4064, 3937: hi = 16 .. -16, lo = 0, -128, 32, 97)."""
    S = k // 256
    if tname == "Q4_K":
        out = np.full((n, S, 144), 0xFF, np.uint8)
        out[:, :, 0:4] = np.frombuffer(np.array([1.0, 0.5], np.float16).tobytes(), np.uint8)
        out[1::3, :, 16:] = 0x00
        out[2::3, :, 16:] = 0x0F  # low nibbles 15, high 0
    else:
        out = np.zeros((n, S, 210), np.uint8)
        out[:, :, 208:210] = np.frombuffer(np.float16(0.5).tobytes(), np.uint8)
        for i in range(4):
            out[i::4, :, :192] = 0xFF if i & 1 else 0x00
            out[i::4, :, 192:208] = 0x7F if i & 2 else 0x80
        out[3::5, :, 192:208:2] = 0x80
    return out.reshape(n, -1)


def run_digit_extremes(O, be, tname):
    n, k, T = 37, 1280, 4
    x = np.ones((T, k), np.float32)  # every quant -128
    x[1] = -3.0                      # every quant 127
    x[2, ::2] = -1.0                 # -128 / 127 in turn
    x[3, 256:512] = 0.0
    run_gemm(O, be, tname, n, k, T, 0, seed=6, packed=digit_extreme_blocks(tname, n, k), x_override=x)


@pytest.mark.parametrize("tname", ["Q4_K", "Q6_K"])
def test_gemm_qi_digit_extremes_host_emulation(oracle, tname):
    run_digit_extremes(oracle, HostBackend(), tname)


@pytest.mark.gpu
@pytest.mark.parametrize("tname", ["Q4_K", "Q6_K"])
def test_gemm_qi_digit_extremes_gpu(oracle, dev, tname):
    run_digit_extremes(oracle, GpuBackend(dev), tname)


def test_gemm_qi_q5k_extreme_magnitudes_host_emulation(oracle):
    run_q5k_extremes(oracle, HostBackend())


@pytest.mark.gpu
def test_gemm_qi_q5k_extreme_magnitudes_gpu(oracle, dev):
    run_q5k_extremes(oracle, GpuBackend(dev))


@pytest.mark.gpu
@pytest.mark.parametrize("tname,n,k,T,norm", CASES + [("Q4_K", 4096, 4096, 512, 1), ("Q5_K", 2048, 4096, 300, 1), ("Q5_K", 512, 14336, 129, 0), ("Q4_K", 1024, 14336, 300, 0), ("Q6_K", 1024, 4096, 512, 1), ("Q6_K", 512, 14336, 129, 0),
                                                     ("Q4_K", 28672, 4096, 64, 1), ("Q8_0", 4096, 4096, 512, 1), ("Q8_0", 1024, 14336, 300, 0)])
def test_gemm_qi_gpu(oracle, dev, tname, n, k, T, norm):
    run_gemm(oracle, GpuBackend(dev), tname, n, k, T, norm, seed=n + k + T)


@pytest.mark.gpu
def test_gemm_qi_glu_and_accumulate_gpu(oracle, dev):
    run_gemm(oracle, GpuBackend(dev), "Q4_K", 512, 14336, 70, 0, glu=True, seed=1)
    run_gemm(oracle, GpuBackend(dev), "Q6_K", 4096, 4096, 200, 0, acc=True, seed=2)
    run_gemm(oracle, GpuBackend(dev), "Q8_0", 512, 14336, 70, 0, glu=True, acc=True, seed=3)


@pytest.mark.gpu
def test_mfma_f16_accumulates_small_integers_exactly(dev):
    """The premise of the min terms, sum of mins (<= 63) x run sums (<= 2048) in one instruction: v_mfma_f32_32x32x16_f16 keeps integers below 2^24 exact.  The other magnitudes go
    further than any operand of the products (whose scale x quant are int8 digits), through chains of 16 instructions."""
    import torch
    from mistralrs_amd import _lib
    L = _lib.load("ext")
    L.mrs_mfma_f16_int_probe.argtypes = [VP, VP, VP, CI, VP]

    def run(A, B):
        ks = A.shape[0]
        lanes = np.arange(64)
        a_op = np.zeros((ks, 64, 8), np.float16); b_op = np.zeros((ks, 64, 8), np.float16)
        for j in range(8):
            a_op[:, :, j] = A[:, lanes % 32, 8 * (lanes // 32) + j]
            b_op[:, :, j] = B[:, lanes % 32, 8 * (lanes // 32) + j]
        ta, tb = torch.from_numpy(a_op).to(dev), torch.from_numpy(b_op).to(dev)
        out = torch.empty(64, 16, device=dev)
        assert L.mrs_mfma_f16_int_probe(ta.data_ptr(), tb.data_ptr(), out.data_ptr(), ks, torch.cuda.current_stream().cuda_stream) == 0
        o = out.cpu().numpy().astype(np.float64)
        got = np.zeros((32, 32))
        for l in range(64):
            for i in range(16):
                got[(i // 4) * 8 + (l // 32) * 4 + (i % 4), l % 32] = o[l, i]
        return got, np.einsum("srk,sck->rc", A.astype(np.int64), B.astype(np.int64))

    rng = np.random.default_rng(0)
    for amax, ks in ((504, 16), (480, 16), (256, 16), (2048, 1)):
        for _ in range(8):
            A = rng.integers(-amax, amax + 1, (ks, 32, 16)); B = rng.integers(-128, 128, (ks, 32, 16)) if amax != 2048 else rng.integers(0, 64, (ks, 32, 16))
            got, ref = run(A, B)
            assert np.array_equal(got, ref)
    got, ref = run(np.full((16, 32, 16), 504), np.full((16, 32, 16), -128))  # |sum| = 16.5 M, just below 2^24
    assert np.array_equal(got, ref) and ref[0, 0] == -16515072


# silu(g) * u rows: the largest row formed in registers and one past it, for both image formats
GLU_K = [("Q4_K", 14336), ("Q8_0", 14336), ("Q6_K", 14592)]


@pytest.mark.parametrize("tname,k", GLU_K)
def test_gemm_qi_glu_long_rows_host_emulation(oracle, tname, k):
    run_gemm(oracle, HostBackend(), tname, 32, k, 3, 0, glu=True, seed=5)


@pytest.mark.gpu
@pytest.mark.parametrize("tname,k", GLU_K)
def test_gemm_qi_glu_long_rows_gpu(oracle, dev, tname, k):
    run_gemm(oracle, GpuBackend(dev), tname, 64, k, 5, 0, glu=True, seed=5)


def run_multi(O, be, tname, ns, k, T, bounds=None, ws=False, acc=False, seed=0):
    """mrs_gemm_qi_multi: several tensors on the same operand rows; with `bounds` every tensor is a stack whose expert e takes the rows bounds[e] .. bounds[e + 1] - 1."""
    t = getattr(O, tname)
    rng = np.random.default_rng(seed)
    E = len(bounds) - 1 if bounds is not None else 1
    x = rng.standard_normal((T, k)).astype(np.float32)
    act = be.buf(np.zeros(be.sym("mrs_qi_act_bytes", [CI, CI], C.c_size_t)(T, k), np.uint8))
    xb = be.buf(x)
    assert be.sym("mrs_qi_quantize_for", [CI, VP, VP, CI, VP, C.c_float, CI, CI, VP, VP, VP], CI)(t, xb.ptr, None, k, None, 1e-5, T, k, act.ptr, None, be.stream) == 0
    keep, packed, base, outs = [act, xb], [], [], []
    for n in ns:
        p = O.quantize(t, (rng.standard_normal((E * n, k)) * 0.05).astype(np.float32)).reshape(E * n, -1)
        nb = be.sym("mrs_gemm_qi_repack_bytes", [CI, C.c_longlong, C.c_longlong], C.c_size_t)(t, E * n, k)
        src, wq = be.buf(np.ascontiguousarray(p).reshape(-1)), be.buf(np.full(nb, 0xA5, np.uint8))
        assert be.sym("mrs_gemm_qi_repack", [VP, CI, C.c_longlong, C.c_longlong, VP, VP], CI)(src.ptr, t, E * n, k, wq.ptr, be.stream) == 0
        b = rng.standard_normal((T, n)).astype(np.float32)
        o = be.buf(b.copy())
        keep += [src, wq]; packed.append(p); base.append(b); outs.append((wq, o))
    bb = be.buf(np.asarray(bounds, np.int32)) if bounds is not None else None
    w = be.buf(np.zeros(4 * T * sum(ns), np.float32)) if ws else None
    ptrs = lambda i: (VP * len(ns))(*[o[i].ptr for o in outs])  # noqa: E731
    ints = (CI * len(ns))(*ns)
    rc = be.sym("mrs_gemm_qi_multi", [CI, CI, VP, VP, CI, VP, CI, VP, VP, CI, VP, CI, CI, VP, C.c_size_t, VP], CI)(
        t, len(ns), ptrs(0), ints, k, act.ptr, T, ptrs(1), ints, int(acc), bb.ptr if bb else None, E, T, w.ptr if ws else None, 4 * T * sum(ns) * 4 if ws else 0, be.stream)
    assert rc == 0, rc
    for n, p, b, (_, o) in zip(ns, packed, base, outs):
        want = b.copy()
        for e in range(E):
            lo, hi = (bounds[e], bounds[e + 1]) if bounds is not None else (0, T)
            for r in range(lo, hi):
                want[r] = O.gemv_engine(t, p[e * n:(e + 1) * n], n, k, x[r])[0] + (b[r] if acc else 0)
        got = o.numpy()
        assert np.array_equal(got, want), (tname, n, int((got != want).sum()))


# segments of 1 .. 3 tensors with ragged row counts; one / two token tiles per wave with remainders; windows that are empty, one row, a tile and a tile + 1; runs of superblocks
# that are empty (5 superblocks: 2, 2, 1, 0) and whole launches cut by runs
MULTI = [("Q4_K", (40,), 512, 70, None, False, False), ("Q4_K", (130, 33, 64), 1280, 33, None, False, True), ("Q4_K", (128, 36), 1280, 65, None, True, True),
         ("Q4_K", (64, 32), 1024, 5, None, True, False), ("Q4_K", (32, 64), 512, 130, (0, 0, 64, 129, 130), False, False), ("Q4_K", (64,), 768, 40, (0, 33, 34, 34, 40), False, False),
         ("Q6_K", (40, 64), 512, 9, None, False, False), ("Q6_K", (64,), 512, 20, (0, 0, 1, 20), False, False), ("Q8_0", (40, 64), 512, 9, None, False, False),
         ("Q8_0", (64,), 512, 20, (0, 0, 1, 20), False, False), ("Q5_K", (64,), 512, 20, (0, 7, 7, 20), False, False),
         ("Q6_K", (130, 36), 1280, 65, None, True, True), ("Q5_K", (128, 36), 1280, 65, None, True, False), ("Q8_0", (132, 32), 1280, 65, None, True, True),
         ("Q6_K", (130,), 768, 33, None, False, True), ("Q5_K", (33,), 768, 70, None, False, True), ("Q8_0", (33,), 768, 33, None, False, False),
         ("Q6_K", (32, 64), 512, 130, (0, 0, 64, 129, 130), False, False), ("Q8_0", (64,), 512, 130, (0, 0, 64, 129, 130), False, False)]


@pytest.mark.parametrize("case", MULTI)
def test_gemm_qi_multi_host_emulation(oracle, case):
    run_multi(oracle, HostBackend(), *case, seed=3)


@pytest.mark.gpu
@pytest.mark.parametrize("case", MULTI + [("Q4_K", (1024, 256, 256), 4096, 200, None, True, True), ("Q4_K", (512,), 1024, 400, (0, 100, 100, 333, 400), False, False)])
def test_gemm_qi_multi_gpu(oracle, dev, case):
    run_multi(oracle, GpuBackend(dev), *case, seed=4)


# more than 32 workgroup columns of 128 rows: whole groups of columns and a remainder, a segment that begins inside a group, windows
WIDE = [("Q8_0", (4224,), 256, 66, None, False, False), ("Q4_K", (4000, 200), 256, 130, None, True, False), ("Q6_K", (2176, 2176), 256, 40, (0, 33, 40), False, False),
        ("Q8_0", (4100,), 1024, 40, None, True, True),
        # remainders of a tile, empty runs; windows of two token tiles per wave
        ("Q4_K", (4100, 160), 1280, 33, None, False, True), ("Q4_K", (4132,), 768, 65, None, True, False), ("Q4_K", (4224,), 512, 70, (0, 0, 64, 70), False, False),
        ("Q6_K", (4130,), 768, 33, None, False, False), ("Q6_K", (4100, 36), 1280, 40, None, True, True), ("Q5_K", (6400,), 256, 65, None, False, False),
        ("Q5_K", (6400,), 768, 98, None, True, False), ("Q5_K", (6400,), 256, 120, (0, 64, 120), False, False),
        ("Q8_0", (4224,), 256, 120, (0, 64, 120), False, False), ("Q8_0", (4224,), 256, 140, (0, 71, 140), False, False)]  # two tiles, one


@pytest.mark.parametrize("case", WIDE)
def test_gemm_qi_more_columns_than_a_group_host_emulation(oracle, case):
    run_multi(oracle, HostBackend(), *case, seed=8)


@pytest.mark.gpu
@pytest.mark.parametrize("case", WIDE + [("Q8_0", (14336, 14336), 512, 200, None, False, False), ("Q5_K", (8200,), 512, 300, None, False, False), ("Q5_K", (3200,), 2304, 200, None, True, True)])
def test_gemm_qi_more_columns_than_a_group_gpu(oracle, dev, case):
    run_multi(oracle, GpuBackend(dev), *case, seed=8)


# (type, rows, K, tokens, accumulate, workspace) -> token tiles of a wave, groups of waves, cut.  Every form of every type at sizes with remainders: rows that do not fill the last
# workgroup or panel, a partly filled last tile, runs of one superblock, unequal and empty ones (5 superblocks: 2, 2, 1, 0), odd ones of a pair
FORMS = [("Q4_K", (3500, 100), 1024, 9, False, True, (1, 1, 1)), ("Q4_K", (3500, 100), 1280, 9, False, False, (1, 4, 0)), ("Q4_K", (70,), 2304, 3, True, False, (1, 4, 0)),
         ("Q4_K", (200,), 4352, 40, False, True, (1, 2, 1)), ("Q4_K", (16516,), 256, 33, True, True, (2, 1, 0)), ("Q4_K", (4132,), 2048, 33, True, True, (2, 1, 1)),
         ("Q8_0", (5180,), 1280, 3, True, True, (1, 2, 1)), ("Q8_0", (70,), 1280, 3, True, False, (1, 4, 0)), ("Q8_0", (300,), 2816, 65, False, False, (1, 4, 0)),
         ("Q8_0", (16516,), 256, 40, False, True, (2, 1, 0)), ("Q6_K", (5900,), 1024, 1, True, True, (1, 1, 1)), ("Q6_K", (70,), 1280, 40, True, False, (1, 4, 0)),
         ("Q6_K", (200,), 4352, 3, True, True, (1, 2, 1)), ("Q6_K", (16516,), 256, 33, False, True, (2, 1, 0)), ("Q6_K", (4132,), 1024, 33, False, True, (2, 1, 1)),
         ("Q5_K", (200,), 4352, 33, False, True, (1, 2, 1)), ("Q5_K", (300,), 1280, 40, True, True, (1, 1, 1)), ("Q5_K", (16516,), 256, 33, True, True, (2, 1, 0)),
         ("Q5_K", (4132,), 1024, 33, True, True, (2, 1, 1))]
FORMS_GPU = [("Q4_K", (5400,), 1280, 34, True, True, (1, 4, 0)), ("Q4_K", (28672,), 4096, 32, True, True, (1, 4, 0)), ("Q4_K", (16516,), 2048, 33, True, True, (2, 2, 0)),
             ("Q4_K", (28672,), 2304, 64, False, True, (2, 2, 0)), ("Q4_K", (28672,), 4096, 130, False, True, (2, 1, 0)), ("Q4_K", (4096,), 14336, 128, True, True, (2, 1, 1)),
             ("Q8_0", (6850,), 1280, 65, False, True, (1, 4, 0)), ("Q8_0", (16516,), 1024, 33, False, True, (2, 2, 0)), ("Q8_0", (14336, 14336), 4096, 64, True, True, (2, 2, 0)),
             ("Q8_0", (16516,), 2048, 3, False, True, (1, 1, 1)), ("Q8_0", (5120,), 8192, 128, True, True, (1, 1, 1)), ("Q8_0", (16512,), 1024, 65, False, True, (1, 1, 0)),
             ("Q8_0", (9860,), 1024, 300, True, True, (2, 1, 0)), ("Q8_0", (12416,), 4096, 33, True, True, (2, 1, 1)), ("Q6_K", (8200,), 2304, 65, False, True, (1, 4, 0)),
             ("Q6_K", (28672,), 4096, 20, True, True, (1, 4, 0)), ("Q6_K", (16516,), 3072, 40, False, True, (2, 2, 0)), ("Q6_K", (4096,), 14336, 200, True, True, (2, 1, 1)),
             ("Q5_K", (28672,), 4096, 64, True, True, (2, 1, 0)), ("Q5_K", (6400,), 4096, 128, True, True, (2, 1, 1))]


def run_form(O, be, tname, ns, k, T, acc, ws, want):
    f = be.sym("mrs_gemm_qi_form", [CI, CI, VP, CI, CI, CI], CI)(getattr(O, tname), len(ns), (CI * len(ns))(*ns), k, T, int(ws))
    assert (f & 15, f >> 4 & 15, f >> 8) == want
    run_multi(O, be, tname, ns, k, T, None, ws=ws, acc=acc, seed=9)


@pytest.mark.parametrize("case", FORMS)
def test_gemm_qi_forms_host_emulation(oracle, case):
    run_form(oracle, HostBackend(), *case)


@pytest.mark.gpu
@pytest.mark.parametrize("case", FORMS + FORMS_GPU)
def test_gemm_qi_forms_gpu(oracle, dev, case):
    run_form(oracle, GpuBackend(dev), *case)


@pytest.mark.gpu
@pytest.mark.parametrize("tname,T", [("Q8_0", 2050), ("Q6_K", 4130), ("Q4_K", 4130)])
def test_long_rows_cut_by_runs_equal_the_whole_launch(oracle, dev, tname, T):
    """65 token tiles x 8 row tiles: one round of workgroups and part of a second; with a workspace the launch is cut by runs of superblocks, without it stays whole."""
    be, t, n, k = GpuBackend(dev), getattr(oracle, tname), 1024, 8192
    rng = np.random.default_rng(7)
    p = oracle.quantize(t, (rng.standard_normal((n, k)) * 0.05).astype(np.float32))
    src, wq = be.buf(np.ascontiguousarray(p).reshape(-1)), be.buf(np.zeros(be.sym("mrs_gemm_qi_repack_bytes", [CI, C.c_longlong, C.c_longlong], C.c_size_t)(t, n, k), np.uint8))
    assert be.sym("mrs_gemm_qi_repack", [VP, CI, C.c_longlong, C.c_longlong, VP, VP], CI)(src.ptr, t, n, k, wq.ptr, be.stream) == 0
    x, act = be.buf(rng.standard_normal((T, k)).astype(np.float32)), be.buf(np.zeros(be.sym("mrs_qi_act_bytes", [CI, CI], C.c_size_t)(T, k), np.uint8))
    assert be.sym("mrs_qi_quantize_for", [CI, VP, VP, CI, VP, C.c_float, CI, CI, VP, VP, VP], CI)(t, x.ptr, None, k, None, 1e-5, T, k, act.ptr, None, be.stream) == 0
    assert be.sym("mrs_gemm_qi_is_cut", [CI, CI, VP, CI, CI], CI)(t, 1, (CI * 1)(n), k, T) == 1
    ws, got = be.buf(np.zeros(4 * T * n, np.float32)), []
    for w in (ws, None):
        o = be.buf(np.zeros((T, n), np.float32))
        assert be.sym("mrs_gemm_qi_ws", [VP, CI, CI, CI, VP, CI, VP, CI, CI, VP, C.c_size_t, VP], CI)(
            wq.ptr, t, n, k, act.ptr, T, o.ptr, n, 0, w.ptr if w else None, 4 * T * n * 4 if w else 0, be.stream) == 0
        got.append(o.numpy())
    assert got[0].any() and np.array_equal(got[0], got[1])


def run_overflow(O, be, tname, T, n=36, k=1024):
    """A run of superblocks whose sum is +-inf: the runs behind it start from nothing (0 * inf would be NaN), whole and cut by runs, as in the decode engine's GEMV.
    Four runs; the first superblock overflows f32 in every other row (K-quants: activations of 1e37; Q8_0, whose scales are f16: an infinite weight scale in every row)."""
    t = getattr(O, tname)
    rng = np.random.default_rng(11)
    p = O.quantize(t, (rng.standard_normal((n, k)) * 40.0).astype(np.float32)).reshape(n, k // 256, -1)
    x = rng.standard_normal((T, k)).astype(np.float32)
    if tname == "Q8_0":
        p[:, 0, 0:2] = np.frombuffer(np.float16(np.inf).tobytes(), np.uint8)
    else:
        x[::2, :256] *= np.float32(1e37)
    if tname in ("Q4_K", "Q5_K"):
        p[:, 0, 2:4] = 0  # dmin: the difference of two infinities is NaN in any order
    p = p.reshape(n, -1)
    want = np.concatenate([O.gemv_engine(t, p, n, k, r) for r in x], axis=0)
    assert np.isnan(want).mean() < 1e-4 and np.isinf(want[::2]).mean() > 0.9 and (tname == "Q8_0" or np.isfinite(want[1::2]).all())
    for cut in (False, True):
        got = gemm_rows(O, be, t, p, n, k, x, cut)
        assert np.array_equal(got, want, equal_nan=True), (tname, cut, int(np.isnan(got).sum()))  # (NaN: an integer sum of 0 times the infinite scale)


def gemm_rows(O, be, t, p, n, k, x, cut, ws_off=0, ldo=None):
    """mrs_gemm_qi_ws on the rows x, with a workspace for the run sums (cut) or without; the first n columns of the output"""
    T, ldo = len(x), ldo or n
    src, wq = be.buf(np.ascontiguousarray(p).reshape(-1)), be.buf(np.zeros(be.sym("mrs_gemm_qi_repack_bytes", [CI, C.c_longlong, C.c_longlong], C.c_size_t)(t, n, k), np.uint8))
    assert be.sym("mrs_gemm_qi_repack", [VP, CI, C.c_longlong, C.c_longlong, VP, VP], CI)(src.ptr, t, n, k, wq.ptr, be.stream) == 0
    xb, act = be.buf(np.ascontiguousarray(x)), be.buf(np.zeros(be.sym("mrs_qi_act_bytes", [CI, CI], C.c_size_t)(T, k), np.uint8))
    assert be.sym("mrs_qi_quantize_for", [CI, VP, VP, CI, VP, C.c_float, CI, CI, VP, VP, VP], CI)(t, xb.ptr, None, k, None, 1e-5, T, k, act.ptr, None, be.stream) == 0
    ws, o = be.buf(np.zeros(4 * T * n + 8, np.float32)), be.buf(np.full((T, ldo), 7.0, np.float32))
    assert be.sym("mrs_gemm_qi_ws", [VP, CI, CI, CI, VP, CI, VP, CI, CI, VP, C.c_size_t, VP], CI)(wq.ptr, t, n, k, act.ptr, T, o.ptr, ldo, 0, ws.ptr + ws_off if cut else None,
                                                                                                 4 * T * n * 4 if cut else 0, be.stream) == 0
    got = o.numpy()
    assert (got[:, n:] == 7.0).all()
    return got[:, :n]


# rows of 1024 and 33 columns of 128 rows: Q6_K cut with two token tiles per wave; longer rows without a workspace: four groups of waves share the runs, an empty one among them (1280)
OVERFLOW = [("Q4_K", 5, 36, 1024), ("Q4_K", 33, 4132, 1024), ("Q5_K", 34, 36, 1024), ("Q6_K", 33, 36, 1024), ("Q6_K", 33, 4100, 1024), ("Q8_0", 5, 36, 1024), ("Q4_K", 33, 36, 2048),
            ("Q6_K", 33, 36, 1280), ("Q8_0", 34, 36, 1280)]


@pytest.mark.parametrize("tname,T,n,k", OVERFLOW)
def test_gemm_qi_infinite_run_host_emulation(oracle, tname, T, n, k):
    run_overflow(oracle, HostBackend(), tname, T, n, k)


@pytest.mark.gpu
@pytest.mark.parametrize("tname,T,n,k", OVERFLOW + [("Q5_K", 200, 3200, 1024), ("Q8_0", 33, 16516, 1024), ("Q4_K", 33, 16516, 2048), ("Q6_K", 33, 16516, 3072), ("Q4_K", 33, 4160, 2048)])
def test_gemm_qi_infinite_run_gpu(oracle, dev, tname, T, n, k):
    run_overflow(oracle, GpuBackend(dev), tname, T, n, k)


def multi_call(O, be, ns, k, T, bounds, experts, max_rows):
    """mrs_gemm_qi_multi on buffers of zeros that are large enough for the call: its return code"""
    t = O.Q4_K
    w = [be.buf(np.zeros(be.sym("mrs_gemm_qi_repack_bytes", [CI, C.c_longlong, C.c_longlong], C.c_size_t)(t, experts * (n + 31) // 32 * 32, k), np.uint8)) for n in ns]
    o = [be.buf(np.zeros((T, n), np.float32)) for n in ns]
    act, bb = be.buf(np.zeros(be.sym("mrs_qi_act_bytes", [CI, CI], C.c_size_t)(T, k), np.uint8)), be.buf(np.asarray(bounds, np.int32))
    ptrs = lambda bufs: (VP * len(ns))(*[b.ptr for b in bufs])  # noqa: E731
    return be.sym("mrs_gemm_qi_multi", [CI, CI, VP, VP, CI, VP, CI, VP, VP, CI, VP, CI, CI, VP, C.c_size_t, VP], CI)(
        t, len(ns), ptrs(w), (CI * len(ns))(*ns), k, act.ptr, T, ptrs(o), (CI * len(ns))(*ns), 0, bb.ptr, experts, max_rows, None, 0, be.stream)


def test_stacks_whose_experts_share_a_panel_are_refused_host_emulation(oracle):
    """The repack cuts a stack into panels of 32 rows: where an expert's rows are no multiple of 32, the next one begins inside a panel."""
    be = HostBackend()
    assert multi_call(oracle, be, (40,), 512, 20, (0, 7, 20), 2, 20) == -1
    assert multi_call(oracle, be, (64, 40), 512, 20, (0, 7, 20), 2, 20) == -1
    assert multi_call(oracle, be, (64, 32), 512, 20, (0, 7, 20), 2, 20) == 0
    assert multi_call(oracle, be, (40,), 512, 20, (0, 20), 1, 20) == 0  # one expert: nothing behind it


def run_win(O, be, tname, n, k, T, win, max_rows, seed=0):
    """mrs_gemm_qi_win: the window's rows are the decode engine's GEMV of those rows, the others stay as they are"""
    t = getattr(O, tname)
    rng = np.random.default_rng(seed)
    p = O.quantize(t, (rng.standard_normal((n, k)) * 0.05).astype(np.float32)).reshape(n, -1)
    x, base = rng.standard_normal((T, k)).astype(np.float32), rng.standard_normal((T, n)).astype(np.float32)
    src, wq = be.buf(np.ascontiguousarray(p).reshape(-1)), be.buf(np.zeros(be.sym("mrs_gemm_qi_repack_bytes", [CI, C.c_longlong, C.c_longlong], C.c_size_t)(t, n, k), np.uint8))
    assert be.sym("mrs_gemm_qi_repack", [VP, CI, C.c_longlong, C.c_longlong, VP, VP], CI)(src.ptr, t, n, k, wq.ptr, be.stream) == 0
    xb, act = be.buf(x), be.buf(np.zeros(be.sym("mrs_qi_act_bytes", [CI, CI], C.c_size_t)(T, k), np.uint8))
    assert be.sym("mrs_qi_quantize_for", [CI, VP, VP, CI, VP, C.c_float, CI, CI, VP, VP, VP], CI)(t, xb.ptr, None, k, None, 1e-5, T, k, act.ptr, None, be.stream) == 0
    wb, o = be.buf(np.asarray(win, np.int32)), be.buf(base.copy())
    fn = be.sym("mrs_gemm_qi_win", [VP, CI, CI, CI, VP, CI, VP, CI, VP, CI, CI, VP], CI)
    assert fn(wq.ptr, t, n, k, act.ptr, T, wb.ptr, max_rows, o.ptr, n, 0, be.stream) == 0
    want = base.copy()
    for r in range(*win):
        want[r] = O.gemv_engine(t, p, n, k, x[r])[0]
    assert np.array_equal(o.numpy(), want)
    assert fn(wq.ptr, t, n, k, act.ptr, T, wb.ptr, 0, o.ptr, n, 0, be.stream) == -1 and fn(wq.ptr, t, n, k, act.ptr, T, wb.ptr, T + 1, o.ptr, n, 0, be.stream) == -1


# windows of a wave's one tile and of more, an empty one, one that ends with the operand rows
WIN = [("Q4_K", 40, 512, 100, (33, 53), 20), ("Q4_K", 64, 512, 100, (10, 100), 90), ("Q6_K", 64, 512, 70, (69, 70), 1), ("Q5_K", 33, 512, 70, (5, 5), 7), ("Q8_0", 40, 512, 70, (1, 66), 65)]


@pytest.mark.parametrize("case", WIN)
def test_gemm_qi_window_host_emulation(oracle, case):
    run_win(oracle, HostBackend(), *case, seed=6)


@pytest.mark.gpu
@pytest.mark.parametrize("case", WIN)
def test_gemm_qi_window_gpu(oracle, dev, case):
    run_win(oracle, GpuBackend(dev), *case, seed=6)


def test_grid_of_a_window_follows_its_bound_host_emulation(oracle):
    """max_rows sizes the grid: tiles past it have no workgroup.  The window names 64 rows more than max_rows allows; with a grid over all operand rows they would be written."""
    be = HostBackend()
    t, n, k, T = oracle.Q4_K, 32, 256, 96
    wq, act, o = be.buf(np.zeros(be.sym("mrs_gemm_qi_repack_bytes", [CI, C.c_longlong, C.c_longlong], C.c_size_t)(t, n, k), np.uint8)), \
        be.buf(np.zeros(be.sym("mrs_qi_act_bytes", [CI, CI], C.c_size_t)(T, k), np.uint8)), be.buf(np.full((T, n), 7.0, np.float32))
    wb = be.buf(np.asarray((0, T), np.int32))
    assert be.sym("mrs_gemm_qi_win", [VP, CI, CI, CI, VP, CI, VP, CI, VP, CI, CI, VP], CI)(wq.ptr, t, n, k, act.ptr, T, wb.ptr, 32, o.ptr, n, 0, be.stream) == 0
    got = o.numpy()
    assert (got[:32] == 0).all() and (got[32:] == 7.0).all()


def run_bad_rows(O, be, tname, T, n=68, k=1024):
    """Activation rows with NaN and infinities share their tile's matrix instructions -- block scales included -- with rows that must not see them, whole and cut by runs."""
    t = getattr(O, tname)
    rng = np.random.default_rng(12)
    p = O.quantize(t, (rng.standard_normal((n, k)) * 0.05).astype(np.float32)).reshape(n, -1)
    x = rng.standard_normal((T, k)).astype(np.float32)
    bad = [0, 3, T - 2]
    x[0], x[3, 300], x[T - 2, 256:512] = np.nan, np.inf, -np.inf
    good = [r for r in range(T) if r not in bad]
    want = np.concatenate([O.gemv_engine(t, p, n, k, x[r]) for r in good], axis=0)
    for cut in (False, True):
        got = gemm_rows(O, be, t, p, n, k, x, cut)
        assert np.array_equal(got[good], want), (tname, cut)
        assert np.isnan(got[0]).all()  # the bad rows' own outputs stay bad
        assert not np.isfinite(got[[3, T - 2]]).any()


BAD_ROWS = [("Q4_K", 6, 68), ("Q4_K", 40, 68), ("Q4_K", 40, 4132), ("Q5_K", 40, 68), ("Q6_K", 6, 68), ("Q6_K", 66, 68), ("Q6_K", 40, 4100), ("Q8_0", 40, 68)]
BAD_ROWS = [c + (1024,) for c in BAD_ROWS] + [("Q4_K", 40, 68, 1280), ("Q6_K", 40, 68, 2048), ("Q8_0", 6, 68, 1280)]  # (without a workspace: four groups of waves)


@pytest.mark.parametrize("tname,T,n,k", BAD_ROWS)
def test_gemm_qi_rows_beside_nan_and_inf_host_emulation(oracle, tname, T, n, k):
    run_bad_rows(oracle, HostBackend(), tname, T, n, k)


@pytest.mark.gpu
@pytest.mark.parametrize("tname,T,n,k", BAD_ROWS + [("Q8_0", 40, 16516, 1024), ("Q4_K", 40, 16516, 2048), ("Q6_K", 40, 16516, 3072)])  # (two groups of two token tiles)
def test_gemm_qi_rows_beside_nan_and_inf_gpu(oracle, dev, tname, T, n, k):
    run_bad_rows(oracle, GpuBackend(dev), tname, T, n, k)


def same_bits(a, b):
    """equal as bits (signs of zeros included), or NaN on both sides"""
    return bool(((a.view(np.uint32) == b.view(np.uint32)) | (np.isnan(a) & np.isnan(b))).all())


def run_odd_scales(O, be, T, n, k):
    """Q8_0 weights whose block scales are negative, zero, subnormal, the largest f16, infinite or NaN, one kind per row: every output as the decode engine gives it, neighbours included.
    The last two rows have no other scale than zero: one with quants that make every product of the first token a negative zero, one with zeros."""
    t = O.Q8_0
    rng = np.random.default_rng(21)
    p = O.quantize(t, (rng.standard_normal((n, k)) * 0.05).astype(np.float32)).reshape(n, -1).copy()
    kinds = [-0.01, 0.0, -0.0, 5.96e-8, 65504.0, np.inf, -np.inf, np.nan]
    for r in range(1, n, 2):  # the rows between keep their scales
        kind = np.asarray(kinds[(r // 2) % len(kinds)], np.float16).tobytes()
        for b in {0, r % (k // 32), k // 32 - 1}:
            p[r, 34 * b: 34 * b + 2] = np.frombuffer(kind, np.uint8)
    x = rng.standard_normal((T, k)).astype(np.float32)
    blocks = p.reshape(n, k // 32, 34)
    blocks[-2:, :, :2] = 0
    blocks[-2, :, 2:] = (np.sign(x[0]) * -100).astype(np.int8).view(np.uint8).reshape(k // 32, 32)
    blocks[-1, :, 2:] = 0
    want = np.concatenate([O.gemv_engine(t, p, n, k, r) for r in x], axis=0)
    gap = k // 256 <= 3 * ((k // 256 + 3) // 4)  # an empty run adds + 0
    assert np.signbit(want[0, -2]) != gap and not want[:, -2:].any()
    for cut in (False, True):
        got = gemm_rows(O, be, t, p, n, k, x, cut)
        assert same_bits(got, want), cut
        assert np.isfinite(got[:, 0::2]).all() and np.isinf(want).any() and np.isnan(want).any()


# four runs, the last one empty; with a workspace cut, without it four groups of waves; more workgroups than CUs: two groups of two token tiles, no groups
ODD_SCALES = [(3, 36, 1280), (40, 36, 1280), (3, 36, 1024), (40, 36, 1024), (40, 4132, 1280), (40, 4132, 1024), (33, 16516, 1280), (40, 16516, 1024), (300, 9860, 1024), (65, 16516, 1024)]


@pytest.mark.parametrize("T,n,k", ODD_SCALES[:4])
def test_gemm_qi_q8_0_odd_scales_host_emulation(oracle, T, n, k):
    run_odd_scales(oracle, HostBackend(), T, n, k)


@pytest.mark.gpu
@pytest.mark.parametrize("T,n,k", ODD_SCALES)
def test_gemm_qi_q8_0_odd_scales_gpu(oracle, dev, T, n, k):
    run_odd_scales(oracle, GpuBackend(dev), T, n, k)


def test_rows_beyond_an_image_are_refused_host_emulation(oracle):
    """A row whose image does not fit LDS (from some 108000 values on) is refused with a norm and without, and nothing is written."""
    be = HostBackend()
    quantize = be.sym("mrs_qi_quantize_for", [CI, VP, VP, CI, VP, C.c_float, CI, CI, VP, VP, VP], CI)
    k = 131072
    x, act = be.buf(np.ones(k, np.float32)), be.buf(np.full(be.sym("mrs_qi_act_bytes", [CI, CI], C.c_size_t)(1, k), 0xA5, np.uint8))
    for t in (oracle.Q4_K, oracle.Q8_0):
        for norm in (None, x.ptr):
            assert quantize(t, x.ptr, None, k, norm, 1e-5, 1, k, act.ptr, None, be.stream) == -2
        assert quantize(t, x.ptr, x.ptr, k, None, 1e-5, 1, k, act.ptr, x.ptr, be.stream) == -2
    assert (act.numpy() == 0xA5).all()


def run_added_rows(O, be, tname, T, d, k):
    """h + a cut product by its run sums and the quantizer that adds them (mrs_gemm_qi_multi_planes, mrs_qi_quantize_added) == the accumulating product and the quantizer of h."""
    t = getattr(O, tname)
    rng = np.random.default_rng(31)
    p = O.quantize(t, (rng.standard_normal((d, k)) * 0.05).astype(np.float32)).reshape(d, -1)
    nb = be.sym("mrs_gemm_qi_repack_bytes", [CI, C.c_longlong, C.c_longlong], C.c_size_t)(t, d, k)
    src, wq = be.buf(np.ascontiguousarray(p).reshape(-1)), be.buf(np.zeros(nb, np.uint8))
    assert be.sym("mrs_gemm_qi_repack", [VP, CI, C.c_longlong, C.c_longlong, VP, VP], CI)(src.ptr, t, d, k, wq.ptr, be.stream) == 0
    x, h0, nw = (rng.standard_normal((T, k)).astype(np.float32), rng.standard_normal((T, d)).astype(np.float32), (1 + 0.1 * rng.standard_normal(d)).astype(np.float32))
    h0[T - 1, : min(256, d)] = 0.0
    quantize = be.sym("mrs_qi_quantize_for", [CI, VP, VP, CI, VP, C.c_float, CI, CI, VP, VP, VP], CI)
    nbytes = be.sym("mrs_qi_act_bytes", [CI, CI], C.c_size_t)
    xb, nwb, act, ws = be.buf(x), be.buf(nw), be.buf(np.zeros(nbytes(T, k), np.uint8)), be.buf(np.full(4 * T * d, np.nan, np.float32))
    assert quantize(t, xb.ptr, None, k, None, 0.0, T, k, act.ptr, None, be.stream) == 0
    a1, a2, h1, h2 = be.buf(np.zeros(nbytes(T, d), np.uint8)), be.buf(np.zeros(nbytes(T, d), np.uint8)), be.buf(h0.copy()), be.buf(h0.copy())
    assert be.sym("mrs_gemm_qi", [VP, CI, CI, CI, VP, CI, VP, CI, CI, VP], CI)(wq.ptr, t, d, k, act.ptr, T, h1.ptr, d, 1, be.stream) == 0
    assert quantize(t, h1.ptr, None, d, nwb.ptr, 1e-5, T, d, a1.ptr, None, be.stream) == 0
    w, n, o, ld = (VP * 1)(wq.ptr), (CI * 1)(d), (VP * 1)(h2.ptr), (CI * 1)(d)
    assert be.sym("mrs_gemm_qi_multi_planes", [CI, CI, VP, VP, CI, VP, CI, VP, VP, CI, VP, C.c_size_t, VP], CI)(t, 1, w, n, k, act.ptr, T, o, ld, 1, ws.ptr, 16 * T * d, be.stream) == 1
    assert np.array_equal(h2.numpy(), h0)
    assert be.sym("mrs_qi_quantize_added", [CI, VP, VP, VP, C.c_float, CI, CI, VP, VP], CI)(t, h2.ptr, ws.ptr, nwb.ptr, 1e-5, T, d, a2.ptr, be.stream) == 0
    assert np.array_equal(h1.numpy(), h2.numpy()) and np.array_equal(a1.numpy(), a2.numpy())


def run_planes_or_rows(O, be, tname, n, k, T, cut):
    """The return code of mrs_gemm_qi_multi_planes is what mrs_gemm_qi_is_cut says: 1 and four planes, `out` as it was, or 0 and the rows, the workspace as it was."""
    t = getattr(O, tname)
    rng = np.random.default_rng(37)
    p = O.quantize(t, (rng.standard_normal((n, k)) * 0.05).astype(np.float32)).reshape(n, -1)
    x = rng.standard_normal((T, k)).astype(np.float32)
    src, wq = be.buf(np.ascontiguousarray(p).reshape(-1)), be.buf(np.zeros(be.sym("mrs_gemm_qi_repack_bytes", [CI, C.c_longlong, C.c_longlong], C.c_size_t)(t, n, k), np.uint8))
    assert be.sym("mrs_gemm_qi_repack", [VP, CI, C.c_longlong, C.c_longlong, VP, VP], CI)(src.ptr, t, n, k, wq.ptr, be.stream) == 0
    xb, act = be.buf(x), be.buf(np.zeros(be.sym("mrs_qi_act_bytes", [CI, CI], C.c_size_t)(T, k), np.uint8))
    assert be.sym("mrs_qi_quantize_for", [CI, VP, VP, CI, VP, C.c_float, CI, CI, VP, VP, VP], CI)(t, xb.ptr, None, k, None, 0.0, T, k, act.ptr, None, be.stream) == 0
    ws, o, ns = be.buf(np.full((4, T, n), 3.0, np.float32)), be.buf(np.full((T, n), 7.0, np.float32)), (CI * 1)(n)
    got = be.sym("mrs_gemm_qi_multi_planes", [CI, CI, VP, VP, CI, VP, CI, VP, VP, CI, VP, C.c_size_t, VP], CI)(t, 1, (VP * 1)(wq.ptr), ns, k, act.ptr, T, (VP * 1)(o.ptr), ns, 0, ws.ptr,
                                                                                                             16 * T * n, be.stream)
    assert got == cut == be.sym("mrs_gemm_qi_is_cut", [CI, CI, VP, CI, CI], CI)(t, 1, ns, k, T)
    planes, rows = ws.numpy().reshape(4, T, n), o.numpy().reshape(T, n)
    assert (rows == 7.0).all() if cut else (planes == 3.0).all()
    out = ((planes[0] + planes[1]) + planes[2]) + planes[3] if cut else rows
    assert np.array_equal(out, np.concatenate([O.gemv_engine(t, p, n, k, r) for r in x], axis=0))


# either side of the lines from which a launch is whole
PLANES = [("Q4_K", 5760, 1280, 1, 1), ("Q4_K", 13568, 1280, 1, 0), ("Q4_K", 5760, 1280, 33, 0), ("Q4_K", 3968, 1280, 33, 1), ("Q8_0", 5760, 1024, 3, 1), ("Q8_0", 9984, 1024, 3, 0),
          ("Q8_0", 2816, 1024, 40, 1), ("Q8_0", 3328, 1024, 40, 0), ("Q6_K", 9216, 1024, 3, 1), ("Q6_K", 9344, 1024, 3, 0), ("Q6_K", 3840, 1024, 64, 0), ("Q5_K", 9216, 1024, 3, 1),
          ("Q5_K", 9344, 1024, 3, 0), ("Q4_K", 36, 768, 3, 0)]


@pytest.mark.parametrize("case", PLANES[3:4] + PLANES[7:8] + PLANES[-1:])
def test_planes_or_rows_host_emulation(oracle, case):
    run_planes_or_rows(oracle, HostBackend(), *case)


@pytest.mark.gpu
@pytest.mark.parametrize("case", PLANES)
def test_planes_or_rows_gpu(oracle, dev, case):
    run_planes_or_rows(oracle, GpuBackend(dev), *case)


ADDED = [("Q4_K", 1, 256, 1024), ("Q8_0", 5, 2304, 1280), ("Q6_K", 37, 768, 1024)]  # rows of one superblock, of more than the 2048 values of a thread's first piece


@pytest.mark.parametrize("tname,T,d,k", ADDED)
def test_added_rows_host_emulation(oracle, tname, T, d, k):
    run_added_rows(oracle, HostBackend(), tname, T, d, k)


@pytest.mark.gpu
@pytest.mark.parametrize("tname,T,d,k", ADDED + [("Q4_K", 37, 4096, 4096), ("Q4_K", 9, 14336, 4096)])
def test_added_rows_gpu(oracle, dev, tname, T, d, k):
    run_added_rows(oracle, GpuBackend(dev), tname, T, d, k)


def run_rope_cache(be, T, heads, kvh, pairs, neox, kv_dtype, planes):
    """mrs_prefill_rope_cache against the two products and their sum / difference in f32 (nothing contracted), K / V rounded to the page's type; rows whole and as four planes of run sums."""
    rng = np.random.default_rng(41)
    pages = 3 + (T + 5) // 32
    tables = [rng.standard_normal((T + 9, max(pairs, 1))).astype(np.float32) for _ in range(2)]
    pos = rng.permutation(T + 9)[:T].astype(np.uint32)
    order = rng.permutation(pages)
    slots = np.array([order[(i + 5) // 32] * 32 + (i + 5) % 32 for i in range(T)], np.int64)
    slots[T // 2] = -1  # a padding token
    raw = [rng.standard_normal((4 if planes else 1, T, n * 128)).astype(np.float32) for n in (heads, kvh, kvh)]
    q, k, v = (((r[0] + r[1]) + r[2]) + r[3] if planes else r[0] for r in raw)

    def rope(x):
        x = x.reshape(T, -1, 128).copy()
        a, b = (slice(0, 64), slice(64, 128)) if neox else (slice(0, 2 * pairs, 2), slice(1, 2 * pairs, 2))
        c, s = (t[pos][:, None, :pairs] for t in tables)
        xs, ys = x[..., a].copy(), x[..., b].copy()
        x[..., a], x[..., b] = xs * c - ys * s, ys * c + xs * s
        return x

    def bits(x):
        if kv_dtype == 0:
            return x.astype(np.float16).view(np.uint16)
        u = x.astype(np.float32).view(np.uint32).astype(np.uint64)
        return ((u + 0x7FFF + ((u >> 16) & 1)) >> 16).astype(np.uint16)

    kc, vc = np.full((pages, kvh, 16, 32, 8), 7, np.uint16), np.full((pages, kvh, 128, 32), 7, np.uint16)
    kb, vb, qb = be.buf(kc), be.buf(vc), be.buf(np.full((T, heads * 128), np.nan, np.float32) if planes else q.copy())
    ins = [be.buf(r) for r in raw]
    if not planes:
        ins[0] = qb  # in place
    cb, sb, pb, slb = (be.buf(z) for z in (tables[0], tables[1], pos, slots))
    fn = be.sym("mrs_prefill_rope_cache", [VP, C.c_size_t, CI] * 3 + [VP] * 7 + [CI] * 6 + [VP], CI)
    args = [z for b, n in zip(ins, (heads, kvh, kvh)) for z in (b.ptr, T * n * 128 if planes else 0, n * 128)]
    assert fn(*args, qb.ptr, kb.ptr, vb.ptr, slb.ptr, pb.ptr, cb.ptr, sb.ptr, T, heads, kvh, pairs, neox, kv_dtype, be.stream) == 0
    assert np.array_equal(qb.numpy().reshape(T, heads, 128), rope(q))
    want_k, want_v = kc.copy(), vc.copy()
    kr, vr = bits(rope(k)), bits(v.reshape(T, kvh, 128))
    for t, s in enumerate(slots):
        if s >= 0:
            want_k[s // 32, :, :, s % 32] = kr[t].reshape(kvh, 16, 8)
            want_v[s // 32, :, :, s % 32] = vr[t]
    assert np.array_equal(kb.numpy().reshape(kc.shape), want_k) and np.array_equal(vb.numpy().reshape(vc.shape), want_v)
    assert fn(*args, qb.ptr, kb.ptr, vb.ptr, slb.ptr, pb.ptr, cb.ptr, sb.ptr, T, heads, kvh, 65, 0, kv_dtype, be.stream) == -1


ROPE = [(1, 1, 1, 64, 0, 1, False), (8, 4, 2, 64, 1, 0, True), (37, 2, 1, 31, 0, 1, True), (45, 2, 2, 64, 1, 1, False), (9, 1, 1, 0, 0, 0, False)]


@pytest.mark.parametrize("case", ROPE)
def test_prefill_rope_cache_host_emulation(case):
    run_rope_cache(HostBackend(), *case)


@pytest.mark.gpu
@pytest.mark.parametrize("case", ROPE + [(1999, 32, 8, 64, 0, 1, False)])
def test_prefill_rope_cache_gpu(dev, case):
    run_rope_cache(GpuBackend(dev), *case)


def run_mixed(O, be, tname, ns, k, T, ws, keep=False, seed=0):
    """mrs_gemm_qi_mixed: tensors of Q6_K (all but the last `second` ones) and of another K-quant in one launch == every tensor's own launch, bit for bit."""
    t6, t2 = O.Q6_K, getattr(O, tname)
    types = [t6] + [t2] * (len(ns) - 1) if len(ns) < 3 or seed % 2 == 0 else [t6, t6, t2]
    rng = np.random.default_rng(seed)
    x = be.buf(rng.standard_normal((T, k)).astype(np.float32))
    act = be.buf(np.zeros(be.sym("mrs_qi_act_bytes", [CI, CI], C.c_size_t)(T, k), np.uint8))
    assert be.sym("mrs_qi_quantize_for", [CI, VP, VP, CI, VP, C.c_float, CI, CI, VP, VP, VP], CI)(t2, x.ptr, None, k, None, 1e-5, T, k, act.ptr, None, be.stream) == 0
    wq, want = [], []
    for i, (t, n) in enumerate(zip(types, ns)):
        packed = O.quantize(t, (rng.standard_normal((n, k)) * 0.05).astype(np.float32)).reshape(n, -1)
        src, w = be.buf(np.ascontiguousarray(packed).reshape(-1)), be.buf(np.zeros(be.sym("mrs_gemm_qi_repack_bytes", [CI, C.c_longlong, C.c_longlong], C.c_size_t)(t, n, k), np.uint8))
        assert be.sym("mrs_gemm_qi_repack", [VP, CI, C.c_longlong, C.c_longlong, VP, VP], CI)(src.ptr, t, n, k, w.ptr, be.stream) == 0
        o = be.buf(np.full((T, n), np.nan, np.float32))
        assert be.sym("mrs_gemm_qi", [VP, CI, CI, CI, VP, CI, VP, CI, CI, VP], CI)(w.ptr, t, n, k, act.ptr, T, o.ptr, n, 0, be.stream) == 0
        wq.append(w)
        want.append(o.numpy())
    outs = [be.buf(np.full((T, n + 3), 7.0, np.float32)) for n in ns]
    nt, n_all = len(ns), sum(ns)
    planes = be.buf(np.zeros(4 * T * n_all if ws else 1, np.float32))
    f = be.sym("mrs_gemm_qi_mixed", [VP, CI, VP, VP, CI, VP, CI, VP, VP, VP, C.c_size_t, CI, VP], CI)
    args = ((CI * nt)(*types), nt, (VP * nt)(*[w.ptr for w in wq]), (CI * nt)(*ns), k, act.ptr, T, (VP * nt)(*[o.ptr for o in outs]), (CI * nt)(*[n + 3 for n in ns]))
    rc = f(*args, planes.ptr if ws else None, 16 * T * n_all if ws else 0, int(keep), be.stream)
    assert rc == (be.sym("mrs_gemm_qi_is_cut", [CI, CI, VP, CI, CI], CI)(t2, nt, (CI * nt)(*ns), k, T) if keep and ws else 0)
    if rc == 1:
        p = planes.numpy().reshape(4, T, n_all)
        got = np.split(((p[0] + p[1]) + p[2]) + p[3], np.cumsum(ns)[:-1], axis=1)
    else:
        got = [o.numpy()[:, :n] for o, n in zip(outs, ns)]
        assert all((o.numpy()[:, n:] == 7.0).all() for o, n in zip(outs, ns))
    for g, w in zip(got, want):
        assert np.array_equal(g, w), (tname, ns, k, T, ws)
    bad = (CI * nt)(*types[::-1])
    assert f(bad, *args[1:], None, 0, 0, be.stream) == -1


# one token tile and two, cut and whole, groups of runs, columns that do not fill a workgroup, both orders of three tensors
MIXED = [("Q4_K", [40, 36], 512, 5, 0), ("Q4_K", [32, 132, 64], 1280, 34, 1), ("Q5_K", [64, 32, 160], 1024, 33, 1), ("Q4_K", [132, 8], 1024, 70, 0), ("Q5_K", [36, 128], 2816, 3, 1)]


@pytest.mark.parametrize("tname,ns,k,T,ws", MIXED)
def test_gemm_qi_mixed_host_emulation(oracle, tname, ns, k, T, ws):
    run_mixed(oracle, HostBackend(), tname, ns, k, T, ws, seed=T)
    run_mixed(oracle, HostBackend(), tname, ns, k, T, ws, keep=True, seed=T + 1)


MIXED_GPU = MIXED + [("Q4_K", [1024, 4096, 1024], 4096, T, 1) for T in (4, 37, 64, 130, 300, 700)] + [("Q4_K", [1024, 12288], 4096, 33, 0), ("Q5_K", [1024, 4096], 4096, 200, 1),
                                                                                                         ("Q4_K", [1024, 27648], 4096, 5, 0)]


@pytest.mark.gpu
@pytest.mark.parametrize("tname,ns,k,T,ws", MIXED_GPU)
def test_gemm_qi_mixed_gpu(oracle, dev, tname, ns, k, T, ws):
    run_mixed(oracle, GpuBackend(dev), tname, ns, k, T, ws, seed=T)
    run_mixed(oracle, GpuBackend(dev), tname, ns, k, T, ws, keep=True, seed=T + 1)


# two groups of waves that take a run's superblocks in turn: 17 superblocks = runs of 5, 5, 5 and 2, whose last step has no second term; one tile with a remainder and two; both orders of three
MIXED_PAIR = [("Q4_K", [36, 132], 4352, 3, 1), ("Q4_K", [64, 40, 132], 4352, 33, 1), ("Q5_K", [132, 64], 4352, 33, 1), ("Q5_K", [40, 64, 32], 4352, 3, 1)]
MIXED_PAIR_GPU = MIXED_PAIR + [("Q4_K", [512, 2048, 512], 4096, 5, 1), ("Q5_K", [512, 2048, 512], 4096, 5, 1)]


@pytest.mark.parametrize("tname,ns,k,T,ws", MIXED_PAIR)
def test_gemm_qi_mixed_pair_host_emulation(oracle, tname, ns, k, T, ws):
    run_mixed(oracle, HostBackend(), tname, ns, k, T, ws, seed=T)
    run_mixed(oracle, HostBackend(), tname, ns, k, T, ws, keep=True, seed=T + 1)


@pytest.mark.gpu
@pytest.mark.parametrize("tname,ns,k,T,ws", MIXED_PAIR_GPU)
def test_gemm_qi_mixed_pair_gpu(oracle, dev, tname, ns, k, T, ws):
    run_mixed(oracle, GpuBackend(dev), tname, ns, k, T, ws, seed=T)
    run_mixed(oracle, GpuBackend(dev), tname, ns, k, T, ws, keep=True, seed=T + 1)


def test_gemm_qi_mixed_forms(oracle):
    """Every form that a launch of two types can take is run above: a line that moves shows here where a case has lost its form."""
    form = HostBackend().sym("mrs_gemm_qi_form", [CI, CI, VP, CI, CI, CI], CI)
    want = [(1, 1, 0), (1, 1, 1), (1, 1, 1), (1, 1, 0), (1, 1, 1), (1, 1, 1), (2, 1, 1), (2, 1, 1), (1, 4, 0), (2, 2, 0), (2, 1, 0), (1, 4, 0), (2, 1, 1), (1, 4, 0)] + 6 * [(1, 2, 1)]
    got = []
    for tname, ns, k, T, ws in MIXED_GPU + MIXED_PAIR_GPU:
        f = form(getattr(oracle, tname), len(ns), (CI * len(ns))(*ns), k, T, ws)
        got.append((f & 15, f >> 4 & 15, f >> 8))
    assert got == want


# windows that end with 1, 32, 33 and 64 rows in their last workgroup of 64, an empty one, and enough workgroups (2048) for the kernel that takes a short end in one token tile
TAIL = [0, 65, 65, 161, 258, 322]


def test_gemm_qi_window_tails_host_emulation(oracle):
    run_multi(oracle, HostBackend(), "Q4_K", [26624], 256, TAIL[-1], bounds=TAIL, seed=9)


@pytest.mark.gpu
@pytest.mark.parametrize("tname,ns,k", [("Q4_K", [14336, 14336], 512), ("Q6_K", [26624], 256), ("Q5_K", [14336, 14336], 256)])
def test_gemm_qi_window_tails_gpu(oracle, dev, tname, ns, k):
    run_multi(oracle, GpuBackend(dev), tname, ns, k, TAIL[-1], bounds=TAIL, seed=9)


def run_norm_rows(O, be, tname, T, k):
    """The quantizer of rows with a norm == the engine's norm and the quantizer of rows without, byte for byte."""
    t = getattr(O, tname)
    rng = np.random.default_rng(k + T)
    x, nw = rng.standard_normal((T, k + 8)).astype(np.float32), (1 + 0.1 * rng.standard_normal(k)).astype(np.float32)
    x[T - 1, k - min(k, 256):] = 0.0  # the last superblock
    x[0, :k] *= np.float32(1e4)
    nbytes = be.sym("mrs_qi_act_bytes", [CI, CI], C.c_size_t)(T, k)
    xb, yb, nwb = be.buf(x), be.buf(O.rms_norm_engine(np.ascontiguousarray(x[:, :k]), nw, 1e-5)), be.buf(nw)
    got, want = be.buf(np.full(nbytes, 0xA5, np.uint8)), be.buf(np.full(nbytes, 0xA5, np.uint8))
    quantize = be.sym("mrs_qi_quantize_for", [CI, VP, VP, CI, VP, C.c_float, CI, CI, VP, VP, VP], CI)
    assert quantize(t, xb.ptr, None, k + 8, nwb.ptr, 1e-5, T, k, got.ptr, None, be.stream) == 0
    assert quantize(t, yb.ptr, None, k, None, 0.0, T, k, want.ptr, None, be.stream) == 0
    assert np.array_equal(got.numpy(), want.numpy())


# waves without a superblock, with one and with two, and the first row that is too long for two per wave; rows that are not next to each other
NORM_ROWS = [(tname, T, k) for tname in ("Q4_K", "Q8_0") for T, k in ((3, 256), (2, 1792), (1, 2048), (2, 2304), (5, 4096), (2, 4352))]


@pytest.mark.parametrize("tname,T,k", NORM_ROWS)
def test_norm_rows_host_emulation(oracle, tname, T, k):
    run_norm_rows(oracle, HostBackend(), tname, T, k)


@pytest.mark.gpu
@pytest.mark.parametrize("tname,T,k", NORM_ROWS + [("Q4_K", 1025, 4096), ("Q8_0", 700, 2560)])
def test_norm_rows_gpu(oracle, dev, tname, T, k):
    run_norm_rows(oracle, GpuBackend(dev), tname, T, k)


@pytest.mark.gpu
@pytest.mark.parametrize("tname,T,d", [("Q4_K", 2, 1792), ("Q8_0", 3, 2304), ("Q4_K", 2, 4352)])
def test_added_rows_of_every_length_gpu(oracle, dev, tname, T, d):
    run_added_rows(oracle, GpuBackend(dev), tname, T, d, 2048)


# either side of the lines of the K-quants' int8 products: three rounds of workgroups with one tile, Q5_K in two tiles, cut and whole, two tiles whole above the cut's line
LINES = [("Q4_K", (24448,), 4096, 5, False, True, (1, 1, 1)), ("Q4_K", (24576,), 4096, 5, False, True, (1, 4, 0)), ("Q5_K", (8320,), 3072, 40, True, True, (2, 1, 1)),
         ("Q5_K", (16512,), 2048, 100, False, True, (2, 1, 0)), ("Q6_K", (13952,), 8192, 130, True, True, (2, 1, 1)), ("Q6_K", (14080,), 8192, 130, True, True, (2, 1, 0))]


@pytest.mark.gpu
@pytest.mark.parametrize("case", LINES)
def test_gemm_qi_lines_gpu(oracle, dev, case):
    run_form(oracle, GpuBackend(dev), *case)


# the form on either side of a line, at sizes that the host emulation would multiply for minutes.  192 workgroups of Q4_K are three full rounds cut: whole one workgroup above it, at 192 itself
# where a row is shorter than 7168 values and the tile has more than two rows
FORM_LINES = [("Q4_K", 24576, 14336, 11, (1, 1, 1)), ("Q4_K", 24704, 14336, 11, (1, 4, 0)), ("Q4_K", 24576, 7168, 32, (1, 1, 1)), ("Q4_K", 24576, 6912, 32, (1, 4, 0)),
              ("Q4_K", 24576, 4096, 2, (1, 1, 1)), ("Q4_K", 24576, 4096, 3, (1, 4, 0)), ("Q4_K", 24704, 4096, 1, (1, 4, 0)),
              # two token tiles of Q5_K and Q6_K: cut up to K / 20 workgroups where these are few, up to K / 25 else
              ("Q6_K", 9600, 6144, 200, (2, 1, 1)), ("Q6_K", 9856, 6144, 200, (2, 1, 0)), ("Q5_K", 4608, 7168, 500, (2, 1, 1)), ("Q6_K", 12160, 9216, 220, (2, 1, 1)),
              ("Q6_K", 12416, 9216, 220, (2, 1, 0)), ("Q6_K", 13952, 11008, 200, (2, 1, 1)), ("Q6_K", 14208, 11008, 200, (2, 1, 0)), ("Q4_K", 9600, 6144, 200, (2, 1, 0)),
              # .. which does not bring two tiles where one is taken else, nor is it drawn for rows of up to 5120 values
              ("Q6_K", 19584, 6144, 81, (1, 1, 0)), ("Q5_K", 6784, 5632, 257, (1, 1, 0)), ("Q5_K", 21120, 4096, 47, (2, 1, 0)),
              # Q5_K in one tile: cut beside two that are not; 65 .. 96 tokens, short rows, more than two rounds, one whole and two cut; and the other sides
              ("Q5_K", 15360, 13824, 73, (1, 1, 1)), ("Q5_K", 9344, 11008, 132, (1, 1, 1)), ("Q5_K", 6016, 2560, 96, (1, 1, 1)), ("Q5_K", 6016, 2560, 64, (2, 1, 1)),
              ("Q5_K", 6144, 4096, 80, (2, 1, 1)), ("Q5_K", 16896, 9216, 90, (1, 1, 1)), ("Q5_K", 11776, 9216, 90, (2, 1, 1)), ("Q5_K", 18048, 7168, 96, (1, 1, 0)),
              ("Q5_K", 18432, 12288, 70, (2, 1, 1)), ("Q5_K", 18432, 14336, 64, (2, 1, 1)), ("Q5_K", 18432, 9216, 64, (2, 1, 1)),
              # one and two tiles of Q4_K that would take as long
              ("Q4_K", 29696, 11008, 79, (1, 1, 0)), ("Q4_K", 29696, 11008, 97, (2, 1, 0)), ("Q4_K", 28672, 4096, 96, (1, 1, 0)), ("Q4_K", 31104, 1024, 72, (2, 1, 0))]


@pytest.mark.parametrize("tname,n,k,T,want", FORM_LINES)
def test_gemm_qi_form_lines(oracle, tname, n, k, T, want):
    f = HostBackend().sym("mrs_gemm_qi_form", [CI, CI, VP, CI, CI, CI], CI)(getattr(oracle, tname), 1, (CI * 1)(n), k, T, 1)
    assert (f & 15, f >> 4 & 15, f >> 8) == want


def test_the_wait_of_a_superblock_covers_its_dma(tmp_path):
    """A superblock's rows are read from LDS behind a wait that leaves the requests behind its last DMA piece in flight, by their count.  Every way through the generated code to such a wait
    has to have made that many (one that the compiler drops, or moves in front of the DMA, would let a piece pass).  State: requests since the last DMA piece, at least; None: no piece in flight."""
    root = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
    csrc, hipcc, out = os.path.join(root, "mistral.rs_amd", "csrc"), os.environ.get("HIPCC", "/opt/rocm/bin/hipcc"), str(tmp_path / "qi.s")
    subprocess.run([hipcc, "--offload-arch=gfx950", "-O3", "-std=c++17", "-ffp-contract=off", "-w", "-I" + csrc, "-I" + os.path.join(root, "include"), "-Xclang", "-target-feature", "-Xclang",
                    "-packed-fp32-ops", "--cuda-device-only", "-S", os.path.join(csrc, "ext_gemm_qi.hip"), "-o", out], check=True)
    kernels = re.findall(r"^(_Z\w*gemm_qi_(?:wide|mixed|tail)_kernel\w*):(.*?)\.end_amdhsa_kernel", open(out).read(), re.M | re.S)
    assert len(kernels) >= 20
    for name, code in kernels:
        blocks, order = {"entry": []}, ["entry"]
        for line in code.splitlines():
            label = re.match(r"(\.LBB\w+):", line)
            if label:
                order.append(label.group(1))
                blocks[order[-1]] = []
            elif re.match(r"\s+[a-z]\w+", line):
                blocks[order[-1]].append(line.split())
                if line.split()[0].startswith("s_cbranch"):  # what follows is reached by falling through
                    order.append("%s+%d" % (order[-1], len(order)))
                    blocks[order[-1]] = []
        states, work, waits = {"entry": None}, ["entry"], {}

        def reach(block, state, states=states, work=work):
            if block not in states:
                states[block] = state
            elif state is None or (states[block] is not None and states[block] <= state):
                return
            else:
                states[block] = state
            work.append(block)
        while work:
            block = work.pop()
            d, waited, through = states[block], None, True
            for i, op in enumerate(blocks[block]):
                if op[0].startswith(("buffer_", "global_")):
                    d = 0 if op[-1] == "lds" else None if d is None else d + 1
                elif op[0] == "s_waitcnt" and any(o.startswith("vmcnt") for o in op):
                    n = int(re.search(r"vmcnt\((\d+)\)", " ".join(op)).group(1))
                    d = None if d is not None and n <= d else d
                    waited = n
                elif op[0] == "s_barrier":
                    if waited is not None:
                        waits[block, i] = (d, waited)
                    waited = None
                elif op[0].startswith(("s_cbranch", "s_branch")):
                    reach(op[1], d)
                    through = op[0] != "s_branch"
                elif op[0] == "s_endpgm":
                    through = False
            if through and order.index(block) + 1 < len(order):
                reach(order[order.index(block) + 1], d)
        # the kernels' own waits, by type and token tiles (a group of waves past its last superblock keeps the others' barriers behind a looser one of the compiler's: it reads nothing)
        form = [int(v) for v in re.findall(r"Li(\d+)E", name)]
        types, tiles = (form[:2], form[2:3]) if "mixed" in name else (form[:1], form[1:2] if "wide" in name else [1, 2])
        own = {5 if t == 8 else {(12, 2): 2, (12, 1): 3}.get((t, nt), 4 if nt == 2 else 6) for t in types for nt in tiles}
        seen = [(n, d) for d, n in waits.values() if n in own]
        assert {n for n, _ in seen} == own, (name, own, waits)
        assert all(d is None for _, d in seen), (name, waits)
