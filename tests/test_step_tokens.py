"""A step's token, position and slot lists (ModelRunner): taken as they are, refused when they differ in length."""
import numpy as np
import pytest
import torch

from llmd_amd.engine.config import EngineConfig
from llmd_amd.engine.engine import LLMEngine


@pytest.fixture(scope="module")
def runner():
    return LLMEngine(EngineConfig.create("tiny-llama", device="cpu", block_size=16, num_gpu_blocks=16, max_num_batched_tokens=64,
                                         max_num_seqs=4, max_model_len=128, enforce_eager=True)).runner


def _plan(runner, **lists):
    w = runner.width
    pl = {"graph": False, "nd": 0, "ids": [5, 6, 7], "pos": [0, 1, 2], "slots": [3, 4, -1], "d_bt": np.zeros((0, w), np.int32),
          "d_len": np.zeros(0, np.int32), "p_ql": [3], "p_ctx": [3], "p_bt": np.zeros((1, w), np.int32)}
    pl.update(lists)
    return pl


def test_lists_arrive(runner):
    ids, meta = runner._eager_meta(_plan(runner, ids=[np.int64(5), 6, 1 << 40]))
    assert ids.tolist() == [5, 6, 1 << 40] and meta.positions.tolist() == [0, 1, 2] and meta.slot_mapping.tolist() == [3, 4, -1]
    assert ids.dtype == meta.positions.dtype == meta.slot_mapping.dtype == torch.long


@pytest.mark.parametrize("name", ["pos", "slots"])
@pytest.mark.parametrize("values", [[0], [0, 1], [0, 1, 2, 3], []])
def test_other_lengths_are_refused(runner, name, values):
    with pytest.raises(ValueError):
        runner._eager_meta(_plan(runner, **{name: values}))
