"""Recurrences sum in another order from a number of tokens of one request on: a step gives the same bits whether its shape was
captured, by whichever step of that shape, or runs eagerly."""
import numpy as np
import pytest
import torch

from gupitar_tiny import CONFIGS as GUPITAR, make_gupitar_folder
from mapedra_tiny import CONFIGS as MAPEDRA, make_mapedra_folder
from siditar_tiny import CONFIGS as SIDITAR, make_siditar_folder

# the design, its configuration, and portions just below and above a line that are padded to one shape
CASES = [(SIDITAR, "D", make_siditar_folder, 319, 325), (MAPEDRA, "A", make_mapedra_folder, 127, 133), (GUPITAR, "A", make_gupitar_folder, 31, 34)]


def model_on_host(config, dtype):
    from microllm_rocm_amd.config.registry import architecture_named
    from microllm_rocm_amd.parts.base import Runtime
    from microllm_rocm_amd.parts.model import Model
    return Model(architecture_named(config.architecture).build_spec(config), Runtime(dtype=dtype, device=torch.device("cpu")))


@pytest.mark.parametrize("configs,which,folder,below,above", CASES)
def test_the_shape_of_a_step_holds_the_side_of_every_line(configs, which, folder, below, above):
    from microllm_rocm_amd.engine.batch import FixedShape
    model = model_on_host(configs[which], torch.bfloat16)
    for requests in (1, 2, 32):
        passed = [sum(count >= line for line in model.portion_lines(requests)) for count in (below, above)]
        assert passed[0] + 1 == passed[1]
        shapes = [FixedShape(tokens=64, requests=requests, wanted=1, width=16, planned={}, lines_passed=count) for count in passed]
        assert shapes[0].key() != shapes[1].key()


@pytest.mark.gpu
@pytest.mark.parametrize("configs,which,folder,below,above", CASES)
def test_a_captured_shape_is_not_replayed_across_a_line(tmp_path, configs, which, folder, below, above):
    from microllm_rocm_amd.engine import Engine, StepEntry
    path = folder(tmp_path, which)
    vocab = configs[which].vocab
    rng = np.random.default_rng(3)
    tokens, beside = (rng.integers(0, vocab, size=count).tolist() for count in (above, 5))

    def step(engine, count):
        for name in ("long", "short"):
            engine.open(name)
        logits = engine.step([StepEntry("long", tokens[:count], [0, count - 1]), StepEntry("short", beside, [4])])
        kept = [logits.clone()]
        for name in ("long", "short"):      # the recurrences' states, float32
            kept += [values for _, _, values in engine.cache.save_slots([engine.cache.get(name).slot])]
        for name in ("long", "short"):
            engine.close(name)
        return kept

    def same(some, others):
        return len(some) == len(others) > 1 and all(torch.equal(one, other) for one, other in zip(some, others))

    options = dict(dtype="bfloat16", max_tokens=1024, max_requests=4)
    eager = [step(Engine.from_folder(path, **options), count) for count in (below, above)]
    for first, second in ((0, 1), (1, 0)):
        engine = Engine.from_folder(path, **options)
        for _ in range(3):
            assert same(step(engine, (below, above)[first]), eager[first])
        assert engine.mixed_graph_replays >= 1
        for _ in range(3):
            assert same(step(engine, (below, above)[second]), eager[second])


@pytest.mark.parametrize("heads,value_dim,requests,line", [(8, 64, 1, 320), (8, 128, 1, 352), (8, 128, 2, 352), (8, 128, 4, 320), (32, 128, 1, 320),
                                                           (4, 256, 1, 480), (2, 512, 1, 736), (2, 512, 4, 320)])
def test_where_a_decay_a_channel_runs_in_chunks(heads, value_dim, requests, line):
    """Narrow values and steps of many waves from 320 tokens of one request on, wide values of a few requests later."""
    from microllm_rocm_amd.parts.base import Runtime
    from microllm_rocm_amd.parts.registry import build_part
    from microllm_rocm_amd.parts.spec import PartSpec
    sizes = {"hidden_size": 64, "heads": heads, "key_dim": 64, "value_dim": value_dim, "decay_rank": 4, "tau": 16.0}
    part = lambda dtype: build_part("mixer", PartSpec("gated_linear_attention", sizes, {}), Runtime(dtype=dtype, device=torch.device("cpu")))
    assert part(torch.bfloat16).portion_line(requests) == line
    assert part(torch.float32).portion_line(requests) is None
