"""Decode attention over pieces: sequences cut by the step's own list, chains of pieces a workgroup, and the merge of a cut sequence in the same launch."""
import json
import os

import pytest
import torch

pytestmark = pytest.mark.gpu
CONFIGS = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "nano-vllm-v1_amd", "model_configs", "qwen3-tiny")


def _runner(tmp_path, hq, hkv, slots, pages, eager):
    from nanovllm.config import Config
    from nanovllm.engine.model_runner import ModelRunner
    with open(os.path.join(CONFIGS, "config.json")) as f:
        cfg = json.load(f)
    cfg.update(num_attention_heads=hq, num_key_value_heads=hkv)
    (tmp_path / "config.json").write_text(json.dumps(cfg))
    return ModelRunner(Config(str(tmp_path), max_num_batched_tokens=4096, max_num_seqs=slots, max_model_len=2048, num_kvcache_blocks=pages, chunked_prefill=True,
                              enforce_eager=eager), 0, [])


def _sequences(runner, lens, g):
    from nanovllm.engine.sequence import Sequence
    seqs, at = [], 0
    for n in lens:
        s = Sequence(torch.randint(0, 1024, (n,), generator=g).tolist())
        p = -(-n // 256)
        s.block_table, at = list(range(at, at + p)), at + p
        s.num_new_tokens = n - 1
        if n > 1:
            runner.run([s])
        s.num_cached_tokens, s.num_new_tokens = n - 1, 1
        seqs.append(s)
    return seqs


def _lens(kind, rows, g):
    if kind in ("long third", "long tenth"):                 # a third or a tenth of them cut in three
        return [2047 if i % (3 if kind == "long third" else 10) == 0 else 64 for i in range(rows)]
    if kind == "short":                                      # nothing is cut, a workgroup a piece
        return torch.randint(1, 130, (rows,), generator=g).tolist()
    if kind == "one long":                                   # one sequence cut in four: the most that the engine's contexts without a work list give
        return [2047] + [1 + i % 64 for i in range(rows - 1)]
    return [64 + (2047 - 64) * i // (rows - 1) for i in range(rows)]          # chains; ends on and around the edges of trips and pages


@pytest.mark.parametrize("hq,hkv,rows,kind", [(16, 8, 17, "spread"), (16, 8, 32, "one long"), (16, 8, 33, "spread"), (16, 8, 64, "spread"), (16, 8, 64, "one long"),
                                              (16, 8, 65, "spread"), (16, 8, 40, "short"), (8, 8, 20, "spread"), (32, 8, 33, "spread"), (40, 8, 20, "spread"),
                                              (40, 8, 33, "one long"), (64, 8, 33, "spread"), (16, 4, 66, "spread"),
                                              # (6 kv heads: 40 rows have places for another number of cuts than the captured step's 48; 82 have a list, its 96 have none)
                                              (12, 6, 40, "long third"), (12, 6, 82, "long tenth")])
def test_pieces_give_what_one_range_a_sequence_gives(tmp_path, hq, hkv, rows, kind):
    """A decode step over pieces against the same step with a workgroup a sequence, which other tests hold against the oracle.  Attention outputs are sums in
    another order in fp32, rounded to bf16: through two layers and the head, logits within a few of bf16's 2^-8; uncut ones (short) to the bit.
    The captured step, and the step with its sequences the other way round, give the pieces' own bits."""
    from nanovllm import _hip
    g = torch.Generator().manual_seed(rows + hq)
    lens = _lens(kind, rows, g)
    pages = sum(-(-n // 256) for n in lens)

    def switch(v):
        _hip.check(_hip.lib().nvh_set_switch(b"NVH_NO_DECODE_PIECES", v), "switch")

    got = {}
    for eager in (True, False):
        runner = _runner(tmp_path, hq, hkv, -(-rows // 16) * 16, pages, eager)
        try:
            seqs = _sequences(runner, lens, torch.Generator().manual_seed(rows))
            for replay in range(3 if not eager else 1):      # (arrival counters are put back by every step)
                out = runner.forward_logits(seqs)[0].clone()
                assert torch.equal(got.setdefault("pieces", out), out)
            assert torch.equal(runner.forward_logits(seqs[::-1])[0].flip(0), out)
            if eager:
                kv = runner.kv_cache[:, 0].clone()
                switch(1)
                one = runner.forward_logits(seqs)[0].clone()
                assert torch.equal(runner.kv_cache[:, 0], kv)                          # the first layer's new keys and values
            else:
                assert runner.graphs
        finally:
            switch(-1)
            runner.exit()
    assert torch.isfinite(got["pieces"]).all()
    if kind == "short":
        assert torch.equal(got["pieces"], one)
    a, b = got["pieces"].float(), one.float()
    assert (a - b).norm() <= 2.0 ** -7 * b.norm() and (a - b).abs().max() <= 2.0 ** -4 * b.abs().max()


@pytest.mark.parametrize("lq,lk", [(1, 700), (33, 600), (257, 513), (512, 512), (900, 1900), (1000, 1000)])
def test_prompt_attention_rows_do_not_depend_on_the_block(lq, lk, switches):
    """Query blocks of 32 and of 64 rows (taken where another step runs beside a mixed one): the same bits for every row."""
    from nanovllm import ops
    g = torch.Generator().manual_seed(lq + lk)
    q = torch.randn(lq, 16, 128, generator=g).bfloat16().cuda()
    pages = -(-lk // 256)
    kc, vc = (torch.randn(pages, 256, 8, 128, generator=g).bfloat16().cuda() for _ in range(2))
    table = torch.randperm(pages, generator=g).int()[None].cuda()
    cu = lambda n: torch.tensor([0, n], dtype=torch.int32).cuda()
    got = []
    for blocks in (-1, 0):
        switches("NVH_ATTN_RB1", blocks)
        got.append(ops.attn_varlen(q, kc, vc, cu(lq), cu(lk), lq, 128 ** -0.5, block_tables=table, max_seqlen_k=lk, num_splits=1))
    assert torch.isfinite(got[0]).all() and torch.equal(*got)
