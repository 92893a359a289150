"""A hook, or a ``forward`` set on an instance, sees the calls it would see if no layer formed the next one's input."""
import pytest
import torch
import torch.nn as nn

from edgellm.engine import ragged_bench as rb
from edgellm.engine.ragged import RaggedEngine
from edgellm.models.hybrid import HybridLM
from edgellm.models.layers import Linear, plain_linear, unwatched

FAMILIES = {"nudadra": (rb.SIZES, rb.hybrid_config), "pagonex": (rb.PAGONEX_SIZES, rb.pagonex_config),
            "vetevik": (rb.VETEVIK_SIZES, rb.vetevik_config)}


DEVICES = ["cpu", pytest.param("cuda", marks=pytest.mark.gpu)]


def _model(family, device="cpu"):
    sizes, make = FAMILIES[family]
    model = HybridLM(make(dict(sizes["w1024"], layers=3, vocab=64)), torch.float32, "cpu")
    g = torch.Generator().manual_seed(0)
    for p in model.parameters():
        if p.dim() > 1:
            p.data.normal_(0, 0.02, generator=g)
    return model.to(device)


def _step(model):
    eng = RaggedEngine(model, 64, slots=1, page=16, use_graphs=False)
    return torch.cat([eng.step([(0, [5, 6, 7], [0, 1, 2])]), eng.step([(0, [8], [0])])])


def _norms(model):
    """The norms whose own call forms a sublayer's input (or the output projection's)."""
    own = [n for layer in model.layers for n in (getattr(layer, "norm1", None), getattr(layer, "norm2", None))
           if n is not None and type(n).__name__ in ("ScalarNorm", "GroupRMSNorm")]
    return own + [model.final_norm]


@pytest.mark.parametrize("family", FAMILIES)
def test_a_hook_for_all_modules_sees_every_norm(family):
    model, seen = _model(family), []
    ref = _step(model)
    h = nn.modules.module.register_module_forward_hook(lambda m, a, y: seen.append(m) and None)
    try:
        out = _step(model)
    finally:
        h.remove()
    for m in _norms(model):
        assert sum(s is m for s in seen) == 2, type(m)
    assert (out - ref).abs().max() <= 1e-5 * ref.abs().max()


@pytest.mark.parametrize("family", FAMILIES)
def test_a_forward_set_on_a_norm_runs(family):
    model = _model(family)
    for m in _norms(model):
        seen, real = [], m.forward
        m.forward = lambda *a, **k: seen.append(1) or real(*a, **k)
        _step(model)
        del m.forward
        assert len(seen) == 2, type(m)


@pytest.mark.parametrize("device", DEVICES)
def test_a_hook_on_a_parallel_mixer_alone_sees_the_stream(device):
    model, seen = _model("nudadra", device), []
    ref = _step(model)
    layer = model.layers[1]
    with torch.no_grad():
        h = layer.mix.register_forward_hook(lambda m, a, y: seen.append((a, y)) and None)
        out = _step(model)
        h.remove()
    assert len(seen) == 2
    for a, y in seen:                                        # stream, projected rows, step, state, feed-forward's output -> stream
        assert len(a) == 5 and y is a[0] and a[4].shape == a[0].shape
    assert (out - ref).abs().max() <= 1e-5 * ref.abs().max()


@pytest.mark.parametrize("device", DEVICES)
@pytest.mark.parametrize("half", ["left", "right"])
def test_a_hook_on_one_half_of_a_parallel_mixer_sees_its_own_arguments(device, half):
    model, seen = _model("nudadra", device), []
    ref = _step(model)
    h = getattr(model.layers[1].mix, half).register_forward_pre_hook(lambda m, a: seen.append(len(a)) and None)
    out = _step(model)
    h.remove()
    assert seen == [4, 4]                                    # projected rows, first column, step, state
    assert (out - ref).abs().max() <= 1e-5 * ref.abs().max()


@pytest.mark.parametrize("family", FAMILIES)
def test_a_hook_on_one_layer_sees_the_stream_alone(family):
    model, seen = _model(family), []
    h = model.layers[1].register_forward_hook(lambda m, a, y: seen.append((len(a), y is a[0])) and None)
    _step(model)
    h.remove()
    assert seen == [(3, True)] * 2                           # stream, step, state -> stream


def test_who_counts_as_watched():
    m = Linear(8, 8, False, torch.float32, "cpu")
    assert unwatched(m) and plain_linear(m)
    m.forward = lambda x: x
    assert not unwatched(m) and not plain_linear(m)
    del m.forward
    for register in (m.register_forward_hook, m.register_forward_pre_hook, nn.modules.module.register_module_forward_hook,
                     nn.modules.module.register_module_forward_pre_hook):
        h = register(lambda *a: None)
        assert not unwatched(m) and not plain_linear(m)
        h.remove()
    assert unwatched(m) and plain_linear(m)
