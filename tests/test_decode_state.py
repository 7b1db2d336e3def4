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


def test_set_state_takes_the_shapes_a_row_of_the_state_takes_host_emulation(oracle):
    """Token ids and positions broadcast to the b sequences like values assigned to a tensor's row: leading axes of length 1 and a single value for all are taken, a second axis
    is refused (its first b values are not the sequences')."""
    m = host_state()
    table = m.block_tables.numpy()

    def state(ids, pos):
        m.set_state(ids, pos)
        b = len(pos)
        assert m.positions[:b].tolist() == pos and m.context_lens[:b].tolist() == [p + 1 for p in pos]
        assert m.slot_mapping[:b].tolist() == [int(table[s, p // 32]) * 32 + p % 32 for s, p in enumerate(pos)]
        return m.input_ids[:b].tolist()

    assert state([1, 2, 3], [0, 31, 319]) == [1, 2, 3]
    assert state(np.array([4, 5], dtype=np.int64), [64, 65]) == [4, 5] and state(torch.tensor([6, 7]), [66, 67]) == [6, 7]
    for pos in (np.array([[8, 9]]), torch.tensor([[8, 9]]), [[8, 9]]):
        m.set_state([1, 2], pos)
        assert m.positions[:2].tolist() == [8, 9] and m._state_pos.tolist() == [8, 9]
    for pos in (5, [5], np.int64(5), [[5]]):
        m.set_state([1, 2], pos)
        assert m.positions[:2].tolist() == [5, 5]
    m.set_state([[9]], [3])
    assert int(m.input_ids[0]) == 9
    before = [t.clone() for t in (m.input_ids, m.positions)]
    for ids, pos in (([[1, 2], [3, 4]], [0, 1]), ([[1], [2]], [0, 1]), ([1, 2], [[0], [1]]), ([1, 2], [0, 1, 2]), ([1, 2, 3], [0, 1]), ([1] * 5, [0] * 5), ([1], [320]), ([1], [-1]), ([], [])):
        with pytest.raises(ValueError):
            m.set_state(ids, pos)
    assert all(torch.equal(a, b) for a, b in zip(before, (m.input_ids, m.positions)))


def test_set_state_slot_of_a_block_without_a_number_host_emulation(oracle):
    """Block tables are int32: an entry of -1 (no block) gives a negative slot, which the K / V writes drop, and no slot past the caches."""
    m = host_state()
    m.block_tables[1, 2] = -1
    m.set_state([1, 2, 3], [70, 70, 70])
    assert m.slot_mapping[:3].tolist() == [int(m.block_tables[0, 2]) * 32 + 6, -32 + 6, int(m.block_tables[2, 2]) * 32 + 6]
