"""Captured decode steps of per-layer stacks against the same steps run launch by launch: batch sizes between the captured
ones, contexts on both sides of a cut into key ranges, steps with portions (never captured) in between, slots that change hands."""
import pytest
import torch

pytestmark = pytest.mark.gpu

STACKS = ["tiny-kakalorn", "tiny-koduzen", "tiny-kokatar", "mekusun", "tiny-negunex", "tiny-zumizen"]


def _serve(name, dtype, eager, tmp_path, lens=(300, 5, 61, 130, 2), new=(24, 12, 30, 9, 16), new_constants=False):
    from llmd_amd.engine.config import EngineConfig
    from llmd_amd.engine.engine import LLMEngine
    from llmd_amd.engine.request import SamplingParams

    kw = {}
    if name == "mekusun":  # no preset
        from llmd_amd.engine.config import ModelConfig
        from test_mekusun import MIXED, model_dir

        name, _ = model_dir(tmp_path, MIXED)
        kw = {"model_config": ModelConfig.from_hf(name), "load_format": "safetensors", "weights_path": name}
    cfg = EngineConfig.create(name, device="cuda", dtype=dtype, block_size=64, num_gpu_blocks=40, max_num_seqs=3, seed=3,
                              max_model_len=1000, max_num_batched_tokens=256, enforce_eager=eager, enable_prefix_caching=False,
                              **kw)
    eng = LLMEngine(cfg, capture_graphs=not eager)
    assert bool(eng.runner.graphs) == (not eager)
    if new_constants:
        eng.runner.model.finalize()
    seen, replays = [], [0]
    logits_of, replay = eng.runner.model.compute_logits, eng.runner._run_seq_graph

    def record(h):
        lg = logits_of(h)
        seen.append(lg.float().cpu())
        return lg

    def count(pl):
        replays[0] += 1
        return replay(pl)

    eng.runner.model.compute_logits, eng.runner._run_seq_graph = record, count
    g = torch.Generator().manual_seed(5)
    prompts = [torch.randint(0, cfg.model_config.vocab_size, (n,), generator=g).tolist() for n in lens]
    reqs = [eng.add_request(f"r{i}", p, SamplingParams(max_tokens=n, temperature=0.0, ignore_eos=True))
            for i, (p, n) in enumerate(zip(prompts, new))]
    while eng.has_unfinished():
        eng.step()
    return seen, [r.output_token_ids for r in reqs], replays[0]


@pytest.mark.parametrize("dtype", ["float32", "bfloat16"])
@pytest.mark.parametrize("name", STACKS)
def test_replayed_steps(name, dtype, tmp_path):
    want, toks, none = _serve(name, dtype, True, tmp_path)
    got, gtoks, replays = _serve(name, dtype, False, tmp_path)
    assert none == 0 and replays >= 30 and len(got) == len(want)
    tol = 1e-4 if dtype == "float32" else 3e-2
    for g, w in zip(got, want):
        assert g.shape == w.shape
        # a key range more or less changes the order of fp32 sums; in bf16 a rounded activation then moves by a place
        assert (g - w).norm() <= tol * w.norm()
        if not torch.equal(g.argmax(-1), w.argmax(-1)):
            assert dtype == "bfloat16"
            return  # other tokens from here on
    assert gtoks == toks


def test_new_constants_are_not_replayed(tmp_path):
    assert _serve("tiny-kakalorn", "float32", False, tmp_path, lens=(5,), new=(6,), new_constants=True)[2] == 0


def test_new_constants_are_reported(tmp_path, caplog):
    """Steps that leave their graphs because the constants are newer say so once; captured again, they are replayed."""
    import logging

    from llmd_amd.engine.config import EngineConfig
    from llmd_amd.engine.engine import LLMEngine
    from llmd_amd.engine.request import SamplingParams

    cfg = EngineConfig.create("tiny-koduzen", device="cuda", dtype="float32", block_size=64, num_gpu_blocks=8, max_num_seqs=1,
                              max_model_len=100, max_num_batched_tokens=64, enable_prefix_caching=False)
    eng = LLMEngine(cfg)
    replays, replay = [], eng.runner._run_seq_graph
    eng.runner._run_seq_graph = lambda pl: replays.append(1) or replay(pl)

    def serve(name):
        del replays[:]
        caplog.clear()
        with caplog.at_level(logging.WARNING):
            r = eng.add_request(name, [3, 1, 2], SamplingParams(max_tokens=6, temperature=0.0, ignore_eos=True))
            while eng.has_unfinished():
                eng.step()
        return r.output_token_ids, len(replays), sum("captured" in m.getMessage() for m in caplog.records)

    toks, n, said = serve("a")
    assert n == 5 and said == 0
    eng.runner.model.finalize()
    assert serve("b") == (toks, 0, 1) and serve("c") == (toks, 0, 0)
    eng.runner.capture_graphs()
    assert serve("d") == (toks, 5, 0)
