"""Workspace of Llama::prefill (csrc/host/runtime.cpp): its size never falls as prompts grow, covers what the launches may use, and a smaller one is taken where only the parts
are missing that a call can do without (probabilities of the two-kernel attention, run sums of launches cut by runs) -- with the same bits."""
import ctypes as C

import numpy as np
import pytest

from mistralrs_amd.llama import LlamaConfig, _Cfg
from tests.abi_backends import HostBackend
from tests.test_dec_model import Q4KM, _mk

CI = C.c_int
CONFIGS = {"8b, 576": LlamaConfig.llama3_8b(max_context_len=576), "8b, 2048": LlamaConfig.llama3_8b(max_context_len=2048), "8b, 8192": LlamaConfig.llama3_8b(max_context_len=8192),
           "70b, 2304": LlamaConfig.llama3_70b(max_context_len=2304), "moe, 1024": LlamaConfig.mixtral_8x7b(max_context_len=1024),
           "small ffn": LlamaConfig(hidden_size=2048, intermediate_size=5632, num_layers=22, num_heads=32, num_kv_heads=4, vocab_size=32000, max_context_len=2048)}


def c_config(cfg):
    return _Cfg(cfg.hidden_size, cfg.intermediate_size, cfg.num_layers, cfg.num_heads, cfg.num_kv_heads, cfg.head_dim, cfg.vocab_size, cfg.head_dim, 1, cfg.rms_eps, cfg.block_size,
                cfg.max_blocks_per_seq, cfg.max_batch, cfg.max_context_len, 1, 1, 0, cfg.num_experts, cfg.num_experts_per_tok if cfg.num_experts else 0, 0, 0)


def sizes(cfg, lengths):
    f = HostBackend().sym("mrs_llama_prefill_workspace_bytes", [C.POINTER(_Cfg), CI], C.c_size_t)
    c = c_config(cfg)
    return [f(C.byref(c), t) for t in lengths]


@pytest.mark.parametrize("name", CONFIGS)
def test_workspace_of_a_longer_prompt_holds_a_shorter_one(name):
    cfg = CONFIGS[name]
    s = sizes(cfg, range(1, min(cfg.max_context_len, 2100) + 1))
    assert all(a <= b for a, b in zip(s, s[1:])), [t for t, (a, b) in enumerate(zip(s, s[1:]), 1) if a > b][:5]


def test_cut_launches_fit_the_bytes_reserved_for_them():
    """mrs_gemm_qi_cut_bytes(T, n, K) holds the run sums (4 T n_all floats) of every launch over n_all <= n rows of weights and up to T tokens that mrs_gemm_qi_multi would cut."""
    be = HostBackend()
    cut, room = be.sym("mrs_gemm_qi_is_cut", [CI, CI, C.c_void_p, CI, CI], CI), be.sym("mrs_gemm_qi_cut_bytes", [CI, CI, CI], C.c_size_t)
    seen = 0
    for k in (768, 1024, 4096, 8192, 14336):
        for ns in ((1024,), (4096,), (4096, 1024, 1024), (4096, 1024), (5632, 5632), (14336, 14336), (28672, 28672), (36,)):
            arr = (CI * len(ns))(*ns)
            for T in list(range(1, 140)) + [500, 512, 513, 600, 960, 961, 1024, 1728, 1999, 4032, 4096]:
                got = [cut(t, len(ns), arr, k, T) for t in (12, 13, 14, 8)]
                seen += sum(got)
                assert not any(got) or 16 * T * sum(ns) <= room(T, sum(ns), k), (k, ns, T, got)
                assert not any(got) or k >= 1024
    assert seen > 1000
    assert cut(12, 1, (CI * 1)(4096), 4096, 100) == 1 and cut(13, 2, (CI * 2)(12288, 12288), 4096, 32) == 1 and cut(13, 2, (CI * 2)(14336, 14336), 4096, 33) == 0
    assert cut(12, 1, (CI * 1)(1024), 8192, 700) == 1  # fewer rows are cut at longer prompts


def test_products_that_a_cut_slows_down_stay_whole():
    """Sizes (type, rows, K, tokens) on both sides of the line: whole where the four planes of run sums cost more than the shorter chain gives back, cut where they cost less."""
    cut = HostBackend().sym("mrs_gemm_qi_is_cut", [CI, CI, C.c_void_p, CI, CI], CI)
    whole = [(12, 8192, 2048, 400), (13, 2048, 2048, 2000), (14, 3072, 1024, 1000), (12, 28672, 4096, 128), (13, 28672, 4096, 100), (14, 14336, 4096, 256), (12, 28672, 8192, 128),
             (12, 8960, 1536, 300), (8, 8960, 1536, 160), (8, 3072, 1024, 512), (13, 65536, 8192, 20), (14, 65536, 8192, 32), (12, 4096, 14336, 1000)]
    parts = [(12, 2048, 2048, 100), (13, 4096, 4096, 200), (13, 24576, 4096, 32), (14, 8192, 8192, 300), (12, 4096, 14336, 700), (14, 4096, 14336, 1600), (8, 2048, 2048, 128),
             (8, 8192, 8192, 300), (12, 8192, 28672, 400)]
    # whole because a workgroup's groups of waves share the runs, and just below that line
    whole += [(12, 28672, 4096, 32), (12, 18816, 4096, 32), (8, 4096, 4096, 512), (14, 26624, 4096, 20), (12, 21632, 4096, 64), (12, 2048, 2048, 200), (8, 2048, 2048, 300)]
    parts += [(12, 18560, 4096, 32), (8, 26496, 4096, 1), (14, 26496, 4096, 20), (12, 8192, 4096, 64), (8, 8192, 4096, 33), (14, 8192, 4096, 33)]
    for case, want in [(c, 0) for c in whole] + [(c, 1) for c in parts]:
        t, n, k, T = case
        assert cut(t, 1, (CI * 1)(n), k, T) == want, case


@pytest.mark.gpu
@pytest.mark.parametrize("experts", [0, 4])
def test_prefill_takes_a_workspace_without_the_optional_parts(oracle, dev, request, experts):
    """The smallest workspace that prefill() takes, the one that mrs_llama_prefill_workspace_bytes names and one between: same logits, same pages, nothing written past any."""
    import torch
    types = Q4KM(oracle)
    T = 9 if request.config.getoption("--host-emulation") else 70
    _, _, m, _, _ = _mk(oracle, dev, types, "bf16", experts=experts)
    assert m.prefill_is_exact
    prompt = [(1000 + 37 * i) % m.cfg.vocab_size for i in range(T)]
    want = m.prefill(prompt, 0).clone()
    pages = [t.clone() for t in m.key_caches + m.value_caches]
    full = m._L.mrs_llama_prefill_workspace_bytes(C.byref(m._c), T)
    real = m._L

    class Sized:  # the library with another answer to how large the workspace has to be
        def __getattr__(self, name):
            return (lambda c, t: self.size) if name == "mrs_llama_prefill_workspace_bytes" else getattr(real, name)

    shim = Sized()
    guard = 1 << 16

    def run(size):
        for t in m.key_caches + m.value_caches:
            t.zero_()
        shim.size = size
        whole = torch.full((size + guard,), 0xA5, dtype=torch.uint8, device=m.device)
        m._prefill_ws, m._L = whole[:size], shim
        try:
            got = m.prefill(prompt, 0)
        finally:
            m._L = real
        assert (whole[size:] == 0xA5).all(), size
        assert torch.equal(got, want) and all(torch.equal(a.view(torch.int16), b.view(torch.int16)) for a, b in zip(pages, m.key_caches + m.value_caches)), size

    f = real.mrs_llama_prefill_min_workspace_bytes
    f.restype, f.argtypes = C.c_size_t, [C.c_void_p, CI]
    least = f(m._h, T)
    assert 0 < least < full
    with pytest.raises(ValueError, match="too small"):
        run(least - 1)
    for size in (least, (least + full) // 2, full):
        run(size)
