"""A model whose closes sum a mixture's parts still calls the mixture as a module where that shows: hooks on it and on the module around it, hooks on
all modules and a forward of the caller's run and see its rows, and what they return counts."""
import importlib

import pytest
import torch

pytestmark = pytest.mark.gpu

FAMILIES = {"lakatar": ("test_lakatar_gpu", ["RET_A", "WKV_A"]), "sokipel": ("test_sokipel_gpu", ["ATT_A", "DEL_A"]), "dinatar": ("test_dinatar_gpu", ["GLA_B", "HGRN_A"])}


@pytest.mark.parametrize("dtype", ["float32", "bfloat16"])
@pytest.mark.parametrize("family", FAMILIES)
def test_hooks(family, dtype, tmp_path):
    from nanovllm.layers.moe import SparseMoE
    name, layers = FAMILIES[family]
    T = importlib.import_module(name)
    case = T.Case(tmp_path, T.config([getattr(T, n) for n in layers], width=72, vocab=50), seed=3)
    tokens = T.tokens_of(case.cfg, 40, 5)
    rp = case.replay(dtype)
    try:
        def logits():
            return torch.tensor(rp.step([{"id": 0, "tokens": tokens, "want": list(range(len(tokens)))}], [0]))
        want = logits()
        mixtures = [m for m in rp.runner.model.modules() if isinstance(m, SparseMoE)]
        around = [m for m in rp.runner.model.modules() if isinstance(getattr(m, "moe", None), SparseMoE)]
        assert len(mixtures) == len(layers) and len(around) == (0 if family == "sokipel" else len(layers))
        seen = []

        def rows(out):
            return out["c32"] if isinstance(out, dict) else out

        def note(module, args, out):
            seen.append((module, rows(out).shape, rows(out).dtype))

        def halve(module, args, out):
            return {k: v * 0.5 for k, v in out.items()} if isinstance(out, dict) else out * 0.5
        for watched in (mixtures, around):
            handles = [m.register_forward_hook(note) for m in watched]
            assert torch.equal(logits(), want)               # (the rows and their close: the same bits as the parts in the close)
            assert seen == [(m, (len(tokens), 72), torch.float32) for m in watched]
            seen.clear()
            for h in handles:
                h.remove()
            handles = [m.register_forward_hook(halve) for m in watched[:1]]
            assert not watched or not torch.equal(logits(), want)
            for h in handles:
                h.remove()
            handles = [m.register_forward_pre_hook(lambda module, args: seen.append(module)) for m in watched]
            assert torch.equal(logits(), want) and seen == watched
            seen.clear()
            for h in handles:
                h.remove()
        handle = torch.nn.modules.module.register_module_forward_hook(lambda module, args, out: seen.append(module))
        assert torch.equal(logits(), want) and all(m in seen for m in mixtures + around)
        handle.remove()
        mixtures[0].forward = lambda x: SparseMoE.forward(mixtures[0], x) * 2
        assert not torch.equal(logits(), want)
        del mixtures[0].forward
        assert torch.equal(logits(), want)
    finally:
        rp.close()
