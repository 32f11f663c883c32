"""Decode attention over pieces: sequences cut by the step's own list, chains of pieces a workgroup, and the merge of a cut sequence in the same launch."""
import json
import os

import pytest
import torch

from oracle import ref_ops as R

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
@pytest.mark.parametrize("splits", [1, 3])
def test_prompt_attention_rows_do_not_depend_on_the_block(lq, lk, splits, switches):
    """Query blocks of 32 rows (small grids) and of 64: the same bits for every row, in one key range and in several."""
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
        got.append(ops.attn_varlen(q, kc, vc, cu(lq), cu(lk), lq, 128 ** -0.5, block_tables=table, max_seqlen_k=lk, num_splits=splits))
    assert torch.isfinite(got[0]).all() and torch.equal(*got)


def test_mixed_steps_in_flight_give_the_bits_of_one_stream(tmp_path):
    """Three mixed steps in a row that read nothing back - decodes over pieces and portions of one prompt, each reading the keys of the one before, the last with
    its keys in ranges - with steps in flight and without: the same logits and caches."""
    from nanovllm.engine.sequence import Sequence
    rows, portions = 33, [(1500, 300), (1800, 270), (2070, 300)]
    g = torch.Generator().manual_seed(5)
    lens = torch.randint(1, 900, (rows,), generator=g).tolist()
    pages = [-(-(n + 3) // 256) for n in lens] + [10]
    runner = _runner(tmp_path, 16, 8, 48, sum(pages), True)
    runner.config.max_model_len = 4096
    tokens = [torch.randint(0, 1024, (n + 3,), generator=g).tolist() for n in lens + [2367]]
    tables, at = [], 0
    for p in pages:
        tables.append(list(range(at, at + p)))
        at += p
    cache = torch.randn(runner.kv_cache.shape, generator=g).bfloat16()
    events, forward = [], runner.native.forward

    def step(i):
        seqs = []
        for j, (tok, table) in enumerate(zip(tokens, tables)):
            cached, new = portions[i] if j == rows else (lens[j] - 1 + i, 1)
            s = Sequence(tok[:cached + new])
            s.block_table, s.num_cached_tokens, s.num_new_tokens = table[:-(-(cached + new) // 256)], cached, new
            seqs.append(s)
        return runner.forward_logits(seqs)[0].clone()

    got = []
    try:
        runner.native.forward = lambda *x, **k: (events.append((k["layer_events"], k["decode_prefix"])), forward(*x, **k))[1]
        for overlap in (False, True):
            runner.step_overlap, runner._last_step = overlap, None
            runner.kv_cache.copy_(cache)
            torch.cuda.synchronize()
            logits = [step(i) for i in range(3)]
            torch.cuda.synchronize()
            got.append(logits + [runner.kv_cache.clone()])
    finally:
        runner.exit()
    assert events == [((0, 0), rows)] * 3 + [((0, 1), rows), ((1, 2), rows), ((2, 1), rows)]
    assert all(torch.isfinite(x).all() and torch.equal(x, y) for x, y in zip(*got))


def _attention_runner(tmp_path, hq, hkv, slots, pages, max_len):
    """One layer whose logits are its attention's outputs: O projection and head are identities, the down projection is zero, and the embedding is small."""
    from nanovllm.config import Config
    from nanovllm.engine.model_runner import ModelRunner
    with open(os.path.join(CONFIGS, "config.json")) as f:
        cfg = json.load(f)
    cfg.update(num_attention_heads=hq, num_key_value_heads=hkv, num_hidden_layers=1, hidden_size=hq * 128, vocab_size=hq * 128, tie_word_embeddings=False,
               max_position_embeddings=max_len)
    (tmp_path / "config.json").write_text(json.dumps(cfg))
    runner = ModelRunner(Config(str(tmp_path), max_num_batched_tokens=1024, max_num_seqs=slots, max_model_len=max_len, num_kvcache_blocks=pages, chunked_prefill=True,
                                enforce_eager=True), 0, [])
    g = torch.Generator("cuda").manual_seed(hq)
    layer, h = runner.model.model.layers[0], hq * 128
    runner.model.model.embed_tokens.weight.data.normal_(generator=g).mul_(2.0 ** -8)
    layer.self_attn.qkv_proj.weight.data.normal_(generator=g).mul_(h ** -0.5)
    for eye in (layer.self_attn.o_proj.weight, runner.model.lm_head.weight):
        eye.data.copy_(torch.eye(h, device="cuda"))
    layer.mlp.down_proj.weight.data.zero_()
    for norm in (layer.input_layernorm, layer.post_attention_layernorm, layer.self_attn.q_norm, layer.self_attn.k_norm, runner.model.model.norm):
        norm.weight.data.fill_(1)
    runner.native.rebuild()
    runner.kv_cache.normal_(generator=g)
    return runner


def _attention_of(runner, seq, lost=None):
    """float64: what the logits of the sequence's last token should be, from the keys and values in the cache (lost: without those 64 keys)."""
    layer, eps = runner.model.model.layers[0], runner.model.model.norm.eps
    a = layer.self_attn
    n = seq.num_cached_tokens + seq.num_new_tokens
    e = runner.model.model.embed_tokens.weight.data[seq.token_ids[n - 1]][None]
    one = torch.ones(1, dtype=torch.bfloat16, device="cuda")
    q = R.linear(R.rms_norm(e, one, eps), a.qkv_proj.weight.data)[:, :a.q_size].view(1, a.num_heads, 128)
    cos, sin = a.rotary_emb.table2d()[n - 1].view(1, 1, 128).split(64, -1)
    q = R.rope_apply(R.rms_norm(q, one, eps), cos, sin)[0].double().view(a.num_kv_heads, -1, 128)
    k, v = (c[0][torch.tensor(seq.block_table, device="cuda")].flatten(0, 1)[:n].double().transpose(0, 1).contiguous() for c in runner.kv_cache)
    scores = (q @ k.transpose(1, 2).contiguous()) * 128 ** -0.5
    if lost is not None:
        scores[:, :, lost:lost + 64] = float("-inf")
    out = (scores.softmax(-1) @ v).view(-1) + e[0].double()
    return (out * (out.square().mean() + eps).rsqrt()).view(a.num_kv_heads, -1)


@pytest.mark.parametrize("hq,hkv,lens,new", [
    (16, 8, "spread 24", 0), (16, 8, "spread 64", 0), (8, 8, "spread 20", 0), (32, 8, "spread 33", 0), (40, 8, "spread 20", 0), (64, 8, "one long 33", 0), (16, 4, "spread 66", 0),
    # mixed steps: the list is the decoding sequences' alone, and 32 of them take more places than the step's 33 sequences would
    (16, 8, "spread 32", 300), (16, 8, "one long 32", 230), (16, 8, "spread 64", 64), (12, 6, "long third 42", 64), (32, 8, "spread 18", 1006),
    # contexts that the engine sends through a work list: eight pieces, and pieces of more trips than are counted one by one
    (16, 8, (16383,) + (64,) * 16, 0), (8, 8, (38400, 4161) + (1, 63, 65) * 6, 0), (40, 8, (9000,) + (700,) * 17, 100)])
def test_every_key_counts(tmp_path, hq, hkv, lens, new):
    """The attention itself, row by row and kv head by kv head, against float64 over the cache's own keys.  Roundings: the normed row's, the product's, the q norm's
    and the rotation's (2^-9 of q each: scores of unit variance move by 2^-8), attention output, sum and norm (2^-9 each): 2^-6 is twice their sum.
    Keys and values are noise, so one lost trip of 64 of n keys is sqrt(64 / n) of a row in the mean, and above twice that bound in every
    row and head up to 10000 keys (smallest seen: 0.053 at 9000, where the embedding takes a part and the noise's own weights another)."""
    from nanovllm.engine.sequence import Sequence
    if isinstance(lens, str):
        kind, rows = lens.rsplit(" ", 1)
        lens = _lens(kind, int(rows), torch.Generator().manual_seed(7))
    lens = list(lens) + ([new + 200] if new else [])
    pages = [-(-n // 256) for n in lens]
    runner = _attention_runner(tmp_path, hq, hkv, -(-len(lens) // 16) * 16, sum(pages), max(4096, -(-max(lens) // 256) * 256))
    runner.LONG_CONTEXT = 1 << 30                            # (no work list)
    try:
        g = torch.Generator().manual_seed(len(lens))
        table, seqs = torch.randperm(sum(pages), generator=g).tolist(), []
        for i, (n, p) in enumerate(zip(lens, pages)):
            s = Sequence(torch.randint(0, hq * 128, (n,), generator=g).tolist())
            s.block_table, table = table[:p], table[p:]
            s.num_new_tokens = new if new and i == len(lens) - 1 else 1
            s.num_cached_tokens = n - s.num_new_tokens
            seqs.append(s)
        got = runner.forward_logits(seqs)[0].double().view(len(lens), hkv, -1)
        for s, n, row in zip(seqs, lens, got):
            want = _attention_of(runner, s)
            assert ((row - want).norm(dim=-1) <= 2.0 ** -6 * want.norm(dim=-1)).all(), n
            if 128 <= n <= 10000:
                lost = _attention_of(runner, s, lost=64 * (n // 128))
                assert ((lost - want).norm(dim=-1) >= 2.0 ** -5 * want.norm(dim=-1)).all(), n
    finally:
        runner.exit()
