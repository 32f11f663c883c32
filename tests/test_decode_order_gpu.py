"""Decode attention whose sequences are dispatched longest first, and its two-trips-ahead loop at the edges of trips and pages."""
from pathlib import Path

import pytest
import torch

from oracle import ref_ops as R

pytestmark = pytest.mark.gpu

TINY = str(Path(__file__).resolve().parents[1] / "nano-vllm-v1_amd" / "model_configs" / "qwen3-tiny")


@pytest.mark.parametrize("hq,hkv", [(16, 8), (5, 1)])
@pytest.mark.parametrize("splits", [1, 3])
def test_trips_and_pages(hq, hkv, splits):
    """Contexts one short of, at and one past a trip (64 keys), two trips, a page (256 keys) and a range; bf16 inputs, tolerance as the decode
    attention's other tests: the result's own rounding (2^-9) and that of the 16-bit products' operands."""
    from nanovllm import ops
    lens = [1, 63, 64, 65, 127, 128, 129, 191, 192, 193, 255, 256, 257, 319, 320, 511, 512, 513, 577, 769]
    g = torch.Generator().manual_seed(11)
    pages = [-(-n // 256) for n in lens]
    perm = torch.randperm(sum(pages), generator=g).int()
    table = torch.full((len(lens), max(pages)), -1, dtype=torch.int32)
    at = 0
    for i, p in enumerate(pages):
        table[i, :p] = perm[at:at + p]
        at += p
    kc, vc = (torch.randn(sum(pages), 256, hkv, 128, generator=g).bfloat16() for _ in range(2))
    q = torch.randn(len(lens), hq, 128, generator=g).bfloat16()
    ctx = torch.tensor(lens, dtype=torch.int32)
    ref = R.attention_decode(q, kc, vc, ctx, table, 128 ** -0.5).float()
    got = ops.attn_decode(q.cuda(), kc.cuda(), vc.cuda(), ctx.cuda(), table.cuda(), 128 ** -0.5, num_splits=splits).float().cpu()
    assert (got - ref).abs().max() < 1.5e-2 + 2e-2 * ref.abs().max()


@pytest.mark.parametrize("count", [129, 150, 160, 257, 270])
@pytest.mark.parametrize("eager", [False, True])
def test_order_of_dispatch_changes_no_bit(count, eager):
    """A decode step of more workgroups than CUs (2 kv heads x 129 sequences and up; 150, 257, 270: with padded rows in the captured graph), the same
    sequences handed over in two orders: every sequence gets the same logits bit for bit.  Up to 256 of them are in a list of pieces, more in order of their
    lengths."""
    from nanovllm.config import Config
    from nanovllm.engine.model_runner import ModelRunner
    from nanovllm.engine.sequence import Sequence
    g = torch.Generator().manual_seed(count)
    lens = torch.randint(1, 520, (count,), generator=g).tolist()
    lens[0], lens[-1] = 1, 519
    pages = [-(-n // 256) for n in lens]
    runner = ModelRunner(Config(TINY, max_num_batched_tokens=1024, max_num_seqs=max(160, -(-count // 16) * 16), max_model_len=1024, num_kvcache_blocks=sum(pages), chunked_prefill=True,
                                enforce_eager=eager), 0, [])
    try:
        seqs, at = [], 0
        for n, p in zip(lens, pages):
            s = Sequence(torch.randint(0, 1024, (n,), generator=g).tolist())
            s.block_table, at = list(range(at, at + p)), at + p
            s.num_new_tokens = n - 1
            if n > 1:
                runner.run([s])
            s.num_cached_tokens, s.num_new_tokens = n - 1, 1
            seqs.append(s)
        one = runner.forward_logits(seqs)[0].clone()
        two = runner.forward_logits(seqs[::-1])[0].clone()
        assert torch.equal(one, two.flip(0))
        few = runner.forward_logits([seqs[0], seqs[-1], seqs[7]])[0].float()          # other tiles in the projections: equal to their rounding
        assert (few - one[[0, count - 1, 7]].float()).abs().max() < 5e-2
    finally:
        runner.exit()


@pytest.mark.parametrize("count", [129, 140, 257])
def test_order_in_a_mixed_step(count):
    """Decoding sequences in front of a portion of a prompt, enough for a list of pieces (up to 256) or the dispatch by length: handed over in two orders every
    sequence, the portion's last token too, gets the same logits bit for bit."""
    from nanovllm.config import Config
    from nanovllm.engine.model_runner import ModelRunner
    from nanovllm.engine.sequence import Sequence
    g = torch.Generator().manual_seed(count)
    lens = torch.randint(1, 520, (count,), generator=g).tolist() + [300]
    lens[0], lens[count - 1] = 1, 519
    pages = [-(-n // 256) for n in lens]
    runner = ModelRunner(Config(TINY, max_num_batched_tokens=1024, max_num_seqs=max(160, count + 1), max_model_len=1024, num_kvcache_blocks=sum(pages), chunked_prefill=True), 0, [])
    try:
        seqs, at = [], 0
        for i, (n, p) in enumerate(zip(lens, pages)):
            s = Sequence(torch.randint(0, 1024, (n,), generator=g).tolist())
            s.block_table, at = list(range(at, at + p)), at + p
            behind = n - 1 if i < count else 70              # (the portion: 230 tokens behind 70)
            s.num_new_tokens = behind
            if behind:
                runner.run([s])
            s.num_cached_tokens, s.num_new_tokens = behind, n - behind
            seqs.append(s)
        *running, prompt = seqs
        one = runner.forward_logits(running + [prompt])[0].clone()
        two = runner.forward_logits(running[::-1] + [prompt])[0].clone()
        assert torch.equal(one[:count], two[:count].flip(0)) and torch.equal(one[count], two[count])
    finally:
        runner.exit()
