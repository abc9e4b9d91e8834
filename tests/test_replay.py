"""Replay-buffer record handling on the CPU (hive_fnn/fnn_replay_buffer.py
counterpart): the opening-value merge."""
import numpy as np
import pytest
import torch

from hive_neuralnet_amd.orchestrator import FNNTrainingExample
from hive_neuralnet_amd.replay import build_forward_batch, compact_opening_value_examples


def _ex(turn, tag, value, w=1.0, use_v=True):
    s = np.zeros(3424, np.uint8)
    s[3412] = turn
    s[0] = tag
    return FNNTrainingExample(s, np.array([1.0], np.float32), value, True, use_v, w)


def test_opening_value_merge():
    a1, a2, a3 = _ex(1, 7, 1.0, 1.0), _ex(1, 7, -1.0, 3.0), _ex(1, 7, 1.0, 0.0)
    late = _ex(9, 7, 1.0)
    lone = _ex(2, 5, -1.0)
    novalue = _ex(0, 7, 1.0, use_v=False)
    out = compact_opening_value_examples([a1, late, a2, lone, novalue, a3], 4)
    # ungrouped first, in input order; then the groups in order of first occurrence: a repeated
    # position's members without value, then its merged value example; a lone position as is
    assert out[0] is late and out[1] is novalue and out[6] is lone
    members, merged = out[2:5], out[5]
    assert all(not m.use_for_value and m.use_for_policy for m in members)
    assert merged.use_for_value and not merged.use_for_policy and merged.value_weight == 4.0
    assert abs(merged.value_target - (1.0 * 1 - 1.0 * 3 + 1.0 * 0) / 4.0) < 1e-12
    assert len(out) == 7
    # weights summing to zero average over the count
    z = compact_opening_value_examples([_ex(0, 1, 1.0, 0.0), _ex(0, 1, -0.5, 0.0)], 4)
    assert z[-1].value_weight == 2.0 and z[-1].value_target == 0.0
    assert compact_opening_value_examples([a1, a2], 0) == [a1, a2]


class _Ext:
    """The two successor calls of build_forward_batch, recorded."""

    def __init__(self):
        self.calls = []

    def fnn_list_successor_features_batch(self, states, moves, num_legal, B):
        self.calls.append("list")
        n = num_legal[:B].to(torch.int64)
        return torch.ones((int(n.sum()), 122)), torch.repeat_interleave(torch.arange(B), n)

    def fnn_successor_features_batch(self, states, moves, a2r, idx, total):
        self.calls.append("rows")
        return torch.ones((total, 122))


@pytest.mark.parametrize("counts,B,route", [([2, 0, 3], 3, "list"), ([0, 0, 0], 3, "list"), ([2, 0, 3], 2, None),
                                            ([0, 0, 0], 2, ""), ([0, 0, 0], 5, ""), ([2, 0, 3], 5, None),
                                            ([[2], [0], [3]], 3, None), ([2, 0, 3], 0, None), ([0, 0, 0], 0, "")])
def test_forward_batch_counts(counts, B, route):
    """Cached action counts: one per root of the batch, or none at all; more or
    fewer of them than roots, or in another shape, are refused where any is
    positive."""
    ext, n = _Ext(), torch.tensor(counts)
    args = (ext, torch.zeros((3, 3424), dtype=torch.uint8), B, n, torch.zeros((3, 122)),
            torch.zeros((3, 256, 6), dtype=torch.uint8))
    if route is None:
        with pytest.raises(RuntimeError):
            build_forward_batch(*args)
        return
    _, succ, a2r, num = build_forward_batch(*args)
    assert ext.calls == [route] * bool(route) and succ.shape == (int(n.sum()), 122) and a2r.dtype == torch.int64
    assert a2r.tolist() == [i for i, k in enumerate(counts) for _ in range(k)] and torch.equal(num, n)
