"""Batched decode on the matrix cores (csrc/ext_dec_mm.hip): mrs_dec_mm_proj / mrs_dec_mm_gate_up / mrs_dec_mm_qkv on the MFMA-order copy of the weights
(mrs_gemm_qi_repack) against the vector-ALU launches of the decode engine on the decode-layout copy (mrs_dec_proj_img / mrs_dec_gate_up_img / mrs_dec_qkv_img): the
SAME BITS for every column count 1..8 -- a token's result must not depend on which kernel produced it -- and, for the plain projection, bit equality with the
engine-order restatement of the oracle (oracle/cpu_path_oracle.c orc_gemv_engine).  Reference role: MMVQ's batch 1..8 from one pass over the weights
(mistralrs-quant/kernels/mmvq_gguf/mmvq_gguf.cu:724-792, gguf/fast_mmvq.rs:52).  Same bodies on the wave64 host emulation (CPU suite) and on the MI355X."""
import ctypes as C
import os
import re
import subprocess

import numpy as np
import pytest

from tests.abi_backends import GpuBackend, HostBackend
from tests.test_dec_engine import ACT_IMG, GLU_IMG, PROJ_IMG_, QKV_IMG, Mat, _act_image, _weights, repack

MM_PROJ = [C.c_void_p, C.c_int, C.c_int, C.c_int, C.c_void_p, C.c_void_p, C.c_int, C.c_int, C.c_float, C.c_int, C.c_void_p]
MM_GLU = [C.c_void_p, C.c_void_p, C.c_int, C.c_int, C.c_int, C.c_void_p, C.c_int, C.c_void_p, C.c_int, C.c_int, C.c_void_p]
MM_QKV = [C.c_void_p, C.c_int, C.c_int] * 3 + [C.c_int, C.c_void_p] + [C.c_void_p] * 7 + [C.c_int] * 6 + [C.c_void_p]


def qi_repack(be, t, packed, n, k):
    nbytes = be.sym("mrs_gemm_qi_repack_bytes", [C.c_int, C.c_longlong, C.c_longlong], C.c_size_t)(t, n, k)
    assert nbytes > 0
    src = be.buf(np.ascontiguousarray(packed).reshape(-1))
    dst = be.buf(np.zeros(nbytes, dtype=np.uint8))
    assert be.sym("mrs_gemm_qi_repack", [C.c_void_p, C.c_int, C.c_longlong, C.c_longlong, C.c_void_p, C.c_void_p], C.c_int)(src.ptr, t, n, k, dst.ptr, be.stream) == 0
    return dst


def check_mm_proj(O, be, tname, n, k, b, norm, mode=1):
    t = getattr(O, tname)
    packed = _weights(O, t, n, k, 61)
    keep, m = repack(be, O, t, packed, n, k)
    qi = qi_repack(be, t, packed, n, k)
    rng = np.random.default_rng(62)
    x = rng.standard_normal((b, k)).astype(np.float32)
    x[b - 1, :256] = 0.0  # an all-zero activation block
    nw = (1.0 + 0.1 * rng.standard_normal(k)).astype(np.float32)
    base = rng.standard_normal((b, n)).astype(np.float32)
    xb, nb = be.buf(x), (be.buf(nw) if norm else None)
    o1, o2 = be.buf(base.copy()), be.buf(base.copy())
    img = _act_image(be, t, xb, nb, k, b)
    assert be.sym("mrs_dec_mm_supported", [C.c_int, C.c_int, C.c_int], C.c_int)(t, k, b) == 1
    assert be.sym("mrs_dec_proj_img", PROJ_IMG_, C.c_int)(C.byref(m), n, img.ptr, o1.ptr, n, mode, 0.5, b, be.stream) == 0
    assert be.sym("mrs_dec_mm_proj", MM_PROJ, C.c_int)(qi.ptr, t, n, k, img.ptr, o2.ptr, n, mode, 0.5, b, be.stream) == 0
    a1, a2 = o1.numpy(), o2.numpy()
    assert np.array_equal(a1, a2), (tname, n, k, b, norm, float(np.abs(a1 - a2).max()))
    xe = O.rms_norm_engine(x, nw, 1e-5) if norm else x
    eng = np.concatenate([O.gemv_engine(t, packed, n, k, r) for r in xe], axis=0)
    if mode:
        eng = base * np.float32(0.5) + eng * np.float32(1.0)
    assert np.array_equal(a2, eng), (tname, n, k, b, norm, "engine-order oracle")


def check_mm_gate_up(O, be, tname, n, k, b):
    t = getattr(O, tname)
    pg, pu = _weights(O, t, n, k, 71), _weights(O, t, n, k, 72)
    kg, mg = repack(be, O, t, pg, n, k)
    ku, mu = repack(be, O, t, pu, n, k)
    qg, qu = qi_repack(be, t, pg, n, k), qi_repack(be, t, pu, n, k)
    rng = np.random.default_rng(73)
    x = rng.standard_normal((b, k)).astype(np.float32)
    nw = (1.0 + 0.1 * rng.standard_normal(k)).astype(np.float32)
    xb, nb = be.buf(x), be.buf(nw)
    o1, o2 = be.buf(np.zeros((b, n), np.float32)), be.buf(np.zeros((b, n), np.float32))
    img = _act_image(be, t, xb, nb, k, b)
    assert be.sym("mrs_dec_gate_up_img", GLU_IMG, C.c_int)(C.byref(mg), C.byref(mu), n, img.ptr, 0, o1.ptr, n, b, be.stream) == 0
    assert be.sym("mrs_dec_mm_gate_up", MM_GLU, C.c_int)(qg.ptr, qu.ptr, t, n, k, img.ptr, 0, o2.ptr, n, b, be.stream) == 0
    a1, a2 = o1.numpy(), o2.numpy()
    assert np.array_equal(a1, a2) and np.isfinite(a2).all() and np.count_nonzero(a2) > 0, (tname, n, k, b, float(np.abs(a1 - a2).max()))


def check_mm_qkv(O, be, tq, tv, heads, kvh, k, b, kvd=1):
    hd, bs = 128, 32
    nq, nkv = heads * hd, kvh * hd
    Tq, Tv = getattr(O, tq), getattr(O, tv)
    pq, pk, pv = _weights(O, Tq, nq, k, 81), _weights(O, Tq, nkv, k, 82), _weights(O, Tv, nkv, k, 83)
    kq, mq = repack(be, O, Tq, pq, nq, k)
    kk, mk = repack(be, O, Tq, pk, nkv, k)
    kv, mv = repack(be, O, Tv, pv, nkv, k)
    qq, qk, qv = qi_repack(be, Tq, pq, nq, k), qi_repack(be, Tq, pk, nkv, k), qi_repack(be, Tv, pv, nkv, k)
    rng = np.random.default_rng(84)
    x = rng.standard_normal((b, k)).astype(np.float32)
    nw = (1.0 + 0.05 * rng.standard_normal(k)).astype(np.float32)
    inv = 1.0 / (10000.0 ** (np.arange(0, hd, 2, dtype=np.float32) / hd))
    fr = np.arange(64, dtype=np.float32)[:, None] * inv[None, :]
    pos = np.array([5 + 7 * i for i in range(b)], dtype=np.int32)
    slots = np.array([(2 * i) * bs + int(pos[i]) % bs for i in range(b)], dtype=np.int64)
    if b > 1:
        slots[b - 1] = -1  # a padded sequence: nothing is written for it
    xb, nb, sb, pb, cb, snb = be.buf(x), be.buf(nw), be.buf(slots), be.buf(pos), be.buf(np.cos(fr).astype(np.float32)), be.buf(np.sin(fr).astype(np.float32))
    img = _act_image(be, Tq, xb, nb, k, b)
    res = []
    for mm in (False, True):
        kc, vc = be.buf(np.zeros((2 * b, kvh, hd // 8, bs, 8), dtype=np.uint16)), be.buf(np.zeros((2 * b, kvh, hd, bs), dtype=np.uint16))
        qb = be.buf(np.zeros((b, nq), dtype=np.float32))
        if mm:
            assert be.sym("mrs_dec_mm_qkv", MM_QKV, C.c_int)(qq.ptr, Tq, nq, qk.ptr, Tq, nkv, qv.ptr, Tv, nkv, k, img.ptr, qb.ptr, kc.ptr, vc.ptr, sb.ptr, pb.ptr, cb.ptr,
                                                              snb.ptr, hd, hd // 2, kvh, bs, kvd, b, be.stream) == 0
        else:
            assert be.sym("mrs_dec_qkv_img", QKV_IMG, C.c_int)(C.byref(mq), C.byref(mk), C.byref(mv), img.ptr, qb.ptr, kc.ptr, vc.ptr, sb.ptr, pb.ptr, cb.ptr, snb.ptr, hd,
                                                                hd // 2, kvh, bs, kvd, b, 0, be.stream) == 0
        res.append((qb.numpy(), kc.numpy(), vc.numpy()))
    for a1, a2 in zip(*res):
        assert np.array_equal(a1, a2)
    assert np.count_nonzero(res[1][0]) > 0 and np.count_nonzero(res[1][1]) > 0 and np.count_nonzero(res[1][2]) > 0


@pytest.mark.parametrize("tname,n,k,b,norm", [("Q4_K", 40, 1024, 3, True), ("Q6_K", 32, 512, 8, False), ("Q5_K", 33, 768, 5, True), ("Q8_0", 64, 512, 4, True),
                                              ("Q4_K", 32, 3584, 8, False), ("Q4_K", 16, 256, 1, False), ("Q6_K", 64, 1792, 2, False), ("Q4_K", 96, 2560, 8, True)])
def test_mm_proj_host_emulation(oracle, tname, n, k, b, norm):
    check_mm_proj(oracle, HostBackend(), tname, n, k, b, norm)  # (n = 33 / 40 / 16: a ragged last panel; k = 768: runs of one superblock, the fourth empty; k = 256: three empty runs)


# runs of superblocks taken two at a time (an odd run's last step has one: 1; 3; 4, 4, 4, 1), units of 16 rows (n = 48 ends inside a panel), columns that do not exist (b < 8)
@pytest.mark.parametrize("tname", ["Q4_K", "Q5_K", "Q6_K", "Q8_0"])
@pytest.mark.parametrize("n,k,b", [(48, 768, 1), (16, 2816, 6), (80, 3328, 8)])
def test_mm_odd_runs_and_half_panels_host_emulation(oracle, tname, n, k, b):
    check_mm_proj(oracle, HostBackend(), tname, n, k, b, True)


@pytest.mark.gpu
@pytest.mark.parametrize("tname", ["Q4_K", "Q5_K", "Q6_K", "Q8_0"])
@pytest.mark.parametrize("n,k,b", [(48, 768, 1), (16, 2816, 6), (80, 3328, 8), (4112, 1280, 2)])
def test_mm_odd_runs_and_half_panels_gpu(oracle, dev, tname, n, k, b):
    check_mm_proj(oracle, GpuBackend(dev), tname, n, k, b, True)


def test_mm_store_gate_up_qkv_host_emulation(oracle):
    be = HostBackend()
    check_mm_proj(oracle, be, "Q6_K", 96, 512, 2, True, mode=0)
    check_mm_gate_up(oracle, be, "Q4_K", 64, 512, 4)
    check_mm_gate_up(oracle, be, "Q8_0", 32, 512, 2)
    check_mm_qkv(oracle, be, "Q4_K", "Q6_K", 2, 1, 512, 3)
    check_mm_qkv(oracle, be, "Q5_K", "Q5_K", 2, 2, 256, 2, kvd=0)


def test_mm_entry_points_refuse_what_they_cannot_do_host_emulation(oracle):
    O, be = oracle, HostBackend()
    k, b, n = 512, 2, 32
    t = O.Q4_K
    packed = _weights(O, t, n, k, 3)
    qi = qi_repack(be, t, packed, n, k)
    x = be.buf(np.ones((b, k), np.float32))
    img = _act_image(be, t, x, None, k, b)
    out = be.buf(np.zeros((b, n), np.float32))
    sup = be.sym("mrs_dec_mm_supported", [C.c_int, C.c_int, C.c_int], C.c_int)
    assert sup(t, k, 8) == 1 and sup(t, k, 9) == 0 and sup(t, 300, 2) == 0 and sup(0, k, 2) == 0 and sup(t, 28672, 8) == 0 and sup(t, 28672, 4) == 1 and sup(t, 14336, 8) == 1
    fn = be.sym("mrs_dec_mm_proj", MM_PROJ, C.c_int)
    assert fn(qi.ptr, t, n, k, img.ptr, out.ptr, n, 0, 1.0, b, be.stream) == 0
    for bad in ((None, t, n, k, img.ptr, out.ptr, n, 0, 1.0, b), (qi.ptr, 0, n, k, img.ptr, out.ptr, n, 0, 1.0, b), (qi.ptr, t, n, 300, img.ptr, out.ptr, n, 0, 1.0, b),
                (qi.ptr, t, n, k, None, out.ptr, n, 0, 1.0, b), (qi.ptr, t, n, k, img.ptr, None, n, 0, 1.0, b), (qi.ptr, t, n, k, img.ptr, out.ptr, n, 0, 1.0, 9),
                (qi.ptr, t, n, k, img.ptr + 4, out.ptr, n, 0, 1.0, b)):
        assert fn(*bad, be.stream) == -1, bad
    # gate / up of different reduction formats share no activation image; q / k / v must agree on it too
    assert be.sym("mrs_dec_mm_qkv", MM_QKV, C.c_int)(qi.ptr, t, n, qi.ptr, t, n, qi.ptr, O.Q8_0, n, k, img.ptr, out.ptr, out.ptr, out.ptr, out.ptr, out.ptr, out.ptr, out.ptr,
                                                      128, 64, 1, 32, 1, b, be.stream) == -1


@pytest.mark.gpu
@pytest.mark.parametrize("tname,n,k,b,norm", [("Q4_K", 4096, 4096, 8, True), ("Q4_K", 4096, 14336, 8, False), ("Q6_K", 4096, 14336, 5, False), ("Q6_K", 32064, 4096, 8, True),
                                              ("Q5_K", 1000, 4096, 3, True), ("Q8_0", 1024, 4096, 8, True), ("Q4_K", 512, 28672, 4, False), ("Q4_K", 4096, 4096, 1, True)])
def test_mm_proj_gpu(oracle, dev, tname, n, k, b, norm):
    check_mm_proj(oracle, GpuBackend(dev), tname, n, k, b, norm)


@pytest.mark.gpu
def test_mm_store_gate_up_qkv_gpu(oracle, dev):
    be = GpuBackend(dev)
    check_mm_proj(oracle, be, "Q6_K", 8192, 4096, 8, True, mode=0)
    check_mm_gate_up(oracle, be, "Q4_K", 14336, 4096, 8)
    check_mm_gate_up(oracle, be, "Q8_0", 2048, 4096, 3)
    check_mm_gate_up(oracle, be, "Q6_K", 1024, 4096, 2)
    check_mm_qkv(oracle, be, "Q4_K", "Q6_K", 32, 8, 4096, 8)
    check_mm_qkv(oracle, be, "Q4_K", "Q4_K", 32, 8, 4096, 4, kvd=0)
    check_mm_qkv(oracle, be, "Q8_0", "Q8_0", 8, 2, 2048, 2)


def check_mm_experts(O, be, tname, tdown, ff, d, E, b, tk, ids):
    """mrs_dec_mm_gate_up_experts == mrs_dec_mm_gate_up of each token on its expert's slice; mrs_dec_mm_proj_experts == the engine-order oracle; mrs_moe_fold_routes == slot by slot."""
    VP, CI, CF = C.c_void_p, C.c_int, C.c_float
    t, td, R = getattr(O, tname), getattr(O, tdown), b * tk
    pg, pu, pd = _weights(O, t, E * ff, d, 71), _weights(O, t, E * ff, d, 72), _weights(O, td, E * d, ff, 73)
    qg, qu, qd = qi_repack(be, t, pg, E * ff, d), qi_repack(be, t, pu, E * ff, d), qi_repack(be, td, pd, E * d, ff)
    rng = np.random.default_rng(74)
    x, nw = rng.standard_normal((b, d)).astype(np.float32), (1.0 + 0.1 * rng.standard_normal(d)).astype(np.float32)
    xb, nb, idb = be.buf(x), be.buf(nw), be.buf(np.asarray(ids, np.int32).reshape(b, tk))
    isz = be.sym("mrs_dec_act_image_bytes", [CI, CI], C.c_size_t)
    rows_img = be.sym("mrs_dec_act_image_rows", [VP, CI, VP, CF, CI, CI, CI, VP, VP], CI)
    ok = be.sym("mrs_dec_mm_experts_supported", [CI] * 6, CI)
    assert ok(t, ff, d, E, b, tk) == 1 and ok(t, ff + 1, d, E, b, tk) == 0 and ok(t, ff, d, E, 9, tk) == 0
    img, act = be.buf(np.zeros(isz(d, b), np.uint8)), be.buf(np.full((R, ff), np.nan, np.float32))
    assert rows_img(xb.ptr, d, nb.ptr, 1e-5, d, t, b, img.ptr, be.stream) == 0
    assert be.sym("mrs_dec_mm_gate_up_experts", [VP, VP, CI, CI, CI, VP, CI, CI, CI, VP, CI, VP, CI, VP], CI)(qg.ptr, qu.ptr, t, ff, d, idb.ptr, E, b, tk, img.ptr, 0, act.ptr, ff,
                                                                                                             be.stream) == 0
    a = act.numpy()
    per = be.sym("mrs_gemm_qi_repack_bytes", [CI, C.c_longlong, C.c_longlong], C.c_size_t)(t, ff, d)
    glu = be.sym("mrs_dec_mm_gate_up", MM_GLU, CI)
    for r in range(R):
        one, e = be.buf(np.zeros((1, ff), np.float32)), ids[r]
        assert glu(qg.ptr + e * per, qu.ptr + e * per, t, ff, d, img.ptr + (r // tk) * isz(d, 1), 0, one.ptr, ff, 1, be.stream) == 0
        assert np.array_equal(a[r], one.numpy()[0]) and np.count_nonzero(a[r]) > 0, r
    img2, y = be.buf(np.zeros(isz(ff, R), np.uint8)), be.buf(np.full((R, d), np.nan, np.float32))
    assert rows_img(act.ptr, ff, None, 0.0, ff, td, R, img2.ptr, be.stream) == 0
    assert be.sym("mrs_dec_mm_proj_experts", [VP, CI, CI, CI, VP, CI, CI, CI, VP, VP, CI, VP], CI)(qd.ptr, td, d, ff, idb.ptr, E, b, tk, img2.ptr, y.ptr, d, be.stream) == 0
    yn = y.numpy()
    for r in range(R):
        assert np.array_equal(yn[r], O.gemv_engine(td, pd.reshape(E, d, -1)[ids[r]], d, ff, a[r])[0]), r
    h, w = rng.standard_normal((b, d)).astype(np.float32), rng.random((b, tk)).astype(np.float32)
    hb, wb = be.buf(h.copy()), be.buf(w)
    assert be.sym("mrs_moe_fold_routes", [VP, CF, VP, VP, CI, CI, CI, VP], CI)(hb.ptr, 0.5, y.ptr, wb.ptr, b, d, tk, be.stream) == 0
    want = h
    for s in range(tk):
        want = want * np.float32(0.5 if s == 0 else 1.0) + yn.reshape(b, tk, d)[:, s] * w[:, s:s + 1]
    assert np.array_equal(hb.numpy(), want)


# all tokens on one pair of experts (8 columns), every route on an expert of its own, experts without tokens, one token
EXPERTS = [("Q4_K", "Q6_K", 256, 256, 4, 8, 2, [1, 3] * 8), ("Q4_K", "Q4_K", 256, 512, 8, 4, 2, [0, 1, 2, 3, 4, 5, 7, 6]), ("Q5_K", "Q8_0", 256, 256, 3, 1, 1, [2]),
           ("Q8_0", "Q5_K", 256, 256, 5, 3, 3, [4, 0, 1, 0, 4, 3, 1, 4, 0]), ("Q6_K", "Q4_K", 512, 256, 6, 5, 2, [0, 1, 0, 2, 5, 0, 2, 1, 0, 5])]


@pytest.mark.parametrize("case", EXPERTS)
def test_mm_experts_host_emulation(oracle, case):
    check_mm_experts(oracle, HostBackend(), *case)


@pytest.mark.gpu
@pytest.mark.parametrize("case", [("Q4_K", "Q6_K", 14336, 1024, 8, 5, 2, [0, 1, 0, 2, 5, 0, 2, 1, 0, 5]), ("Q4_K", "Q4_K", 2048, 4096, 8, 8, 2, [7, 6] * 4 + [1, 2, 1, 0, 3, 7, 5, 4]),
                                  ("Q8_0", "Q5_K", 512, 768, 5, 3, 3, [4, 0, 1, 0, 4, 3, 1, 4, 0])])
def test_mm_experts_gpu(oracle, dev, case):
    check_mm_experts(oracle, GpuBackend(dev), *case)


def test_the_wait_for_the_image_leaves_exactly_the_weight_ring_in_flight(tmp_path):
    """The kernels wait for the image in front of the first barrier by a count of the requests behind it: the weight ring's, which alone are non-temporal.  A count above theirs (a
    request that the compiler drops) would let as many of the image's requests pass."""
    root = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
    csrc, hipcc, out = os.path.join(root, "mistral.rs_amd", "csrc"), os.environ.get("HIPCC", "/opt/rocm/bin/hipcc"), str(tmp_path / "mm.s")
    subprocess.run([hipcc, "--offload-arch=gfx950", "-O3", "-std=c++17", "-ffp-contract=off", "-w", "-I" + csrc, "-I" + os.path.join(root, "include"), "-Xclang", "-target-feature", "-Xclang",
                    "-packed-fp32-ops", "--cuda-device-only", "-S", os.path.join(csrc, "ext_dec_mm.hip"), "-o", out], check=True)
    kernels = re.findall(r"^(_Z\w*dec_mm\w*):(.*?)s_barrier", open(out).read(), re.M | re.S)
    assert len(kernels) >= 11
    for name, code in kernels:
        image, ring = code.rfind(" lds\n"), 0
        assert image > 0, name
        for line in code[image:].splitlines():
            ring += bool(re.match(r"\s+buffer_load.* nt\b", line))
            wait = re.match(r"\s+s_waitcnt vmcnt\((\d+)\)", line)
            if ring and wait:
                break
        assert wait and int(wait.group(1)) == ring, (name, line, ring)


def last_grid():
    """workgroups of the last launch of the host build"""
    return int((C.c_uint * 4).in_dll(HostBackend.lib(), "hiphost_last_launch")[0])


def test_mixes_with_q5_k_have_one_workgroup_per_cu_host_emulation(oracle):
    """Their kernels' registers admit no second one; 384 units (40 + 4 + 4 heads of 128 rows) are two for each of 192 workgroups, not a second round of 128."""
    be = HostBackend()
    check_mm_qkv(oracle, be, "Q5_K", "Q6_K", 40, 4, 256, 2)
    assert last_grid() == 192


@pytest.mark.gpu
def test_mixes_with_q5_k_gpu(oracle, dev):
    check_mm_qkv(oracle, GpuBackend(dev), "Q5_K", "Q6_K", 40, 4, 256, 8)
    check_mm_qkv(oracle, GpuBackend(dev), "Q4_K", "Q5_K", 32, 8, 4096, 3)


# 1001 panels, the last one of 20 rows: both units of one belong to a workgroup; 1000 and one on the last
@pytest.mark.parametrize("tname,grid", [("Q6_K", 251), ("Q4_K", 501)])
def test_mm_panels_stay_together_in_long_launches_host_emulation(oracle, tname, grid):
    check_mm_proj(oracle, HostBackend(), tname, 32020, 256, 2, False, mode=0)
    assert last_grid() == grid


@pytest.mark.gpu
@pytest.mark.parametrize("tname,n,k,b", [("Q4_K", 32020, 256, 8), ("Q5_K", 32020, 512, 3), ("Q6_K", 32052, 1024, 8), ("Q8_0", 49168, 768, 5)])
def test_mm_panels_stay_together_in_long_launches_gpu(oracle, dev, tname, n, k, b):
    check_mm_proj(oracle, GpuBackend(dev), tname, n, k, b, False, mode=0)


@pytest.mark.gpu
def test_mm_gate_up_of_long_launches_gpu(oracle, dev):
    check_mm_gate_up(oracle, GpuBackend(dev), "Q4_K", 32020, 512, 4)


def test_units_of_large_records_are_dealt_evenly_host_emulation(oracle):
    """Between one and two units per CU: 384 units of Q8_0 are two for each of 192 workgroups; 288 of them, and Q4_K's smaller records, a workgroup each."""
    be = HostBackend()
    for tname, heads, grid in (("Q8_0", 40, 192), ("Q8_0", 28, 288), ("Q4_K", 40, 384)):
        check_mm_qkv(oracle, be, tname, tname, heads, 4, 256, 2)
        assert last_grid() == grid, (tname, heads)
    check_mm_proj(oracle, be, "Q6_K", 10256, 256, 1, False)  # 642 units: three each
    assert last_grid() == 214


@pytest.mark.gpu
@pytest.mark.parametrize("tname,n,k,b", [("Q8_0", 8192, 4096, 8), ("Q6_K", 10256, 1280, 3), ("Q5_K", 16384, 1024, 5)])
def test_units_of_large_records_are_dealt_evenly_gpu(oracle, dev, tname, n, k, b):
    check_mm_proj(oracle, GpuBackend(dev), tname, n, k, b, False)
