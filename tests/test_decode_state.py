"""Llama.set_state() and the host copy of the positions it leaves for replay()'s bounds, on the host build of the kernels (csrc/ext_decode.hip mrs_set_state); the GPU side is in
test_dec_model.py."""
import ctypes as C

import numpy as np
import pytest
import torch

from mistralrs_amd.llama import Llama, LlamaConfig
from tests.abi_backends import HostBackend


def host_state(max_batch=4, max_context_len=320):
    """A Llama object with the decode-state buffers only, on the host build of the kernels."""
    m = object.__new__(Llama)
    m.cfg = LlamaConfig(hidden_size=256, intermediate_size=256, num_layers=1, num_heads=2, num_kv_heads=1, vocab_size=512, max_batch=max_batch, max_context_len=max_context_len)
    m.device, m._L, m._stream = torch.device("cpu"), HostBackend.lib(), lambda: None
    m._L.mrs_set_state.argtypes = [C.c_void_p, C.c_void_p, C.c_int] + [C.c_void_p] * 5 + [C.c_int, C.c_int, C.c_void_p]
    m._L.mrs_last_error.restype = C.c_char_p
    m.input_ids, m.positions, m.context_lens = (torch.full((max_batch,), -7, dtype=torch.int32) for _ in range(3))
    m.slot_mapping = torch.full((max_batch,), -7, dtype=torch.int64)
    m.block_tables = torch.arange(max_batch * m.cfg.max_blocks_per_seq, dtype=torch.int32).view(max_batch, -1).flip(0).contiguous()
    m._state_pos, m._replays_left, m._need_embed = None, 3, False
    return m


def test_set_state_raises_when_its_launch_fails_host_emulation(oracle):
    """A state launch that did not happen must not leave a host copy of the positions for replay()'s bounds."""
    m = host_state()
    m.set_state([1, 2], [3, 4])
    assert m._state_pos.tolist() == [3, 4] and m.input_ids.tolist() == [1, 2, -7, -7]
    error = C.c_int.in_dll(m._L, "hiphost_next_error")
    error.value = 1
    try:
        with pytest.raises(RuntimeError):
            m.set_state([5, 6], [7, 8])
    finally:
        error.value = 0
    assert m._state_pos is None
