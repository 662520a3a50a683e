"""GPU: linear draft attention over the working cache against the oracle.

Mirrors the reference's device test of batched draft attention
(tests/test_linear_attention_batch_npu.py:74-144): canonical slots in order
and permuted, NaN beyond every row's position, two consecutive draft steps,
output rows past the batch zero, working lengths advanced.  Every launch is
also checked against the oracle (diffspec/runtime.py:2024-2077): the working
caches bit for bit (the new key/value rows are copies), the output within
one bf16/fp16 rounding of the oracle's fp32 result, and within the
reference's own tolerance (rtol 0.03, atol 0.02) of its expectation.
"""

import pytest
import torch

from helpers import assert_attention_close, attention_terms, gen, randn
from oracle import diffspec_oracle as O

pytestmark = pytest.mark.gpu

REF_RTOL, REF_ATOL = 0.03, 0.02


def _same_bits(a, b):
    assert torch.equal(a.isnan(), b.isnan())
    assert torch.equal(torch.nan_to_num(a), torch.nan_to_num(b))


class Case:
    """Working caches with NaN past every slot's valid prefix, plus per-step inputs."""

    def __init__(self, seed, num_slots, hkv, hq, head_dim, budget, dtype=torch.bfloat16):
        self.g = gen(seed)
        self.shape = (num_slots, hkv, budget, head_dim)
        self.work_k = torch.full(self.shape, float("nan"), dtype=dtype)
        self.work_v = self.work_k.clone()
        self.lens = torch.zeros(num_slots, dtype=torch.int32)
        self.hkv, self.hq, self.head_dim, self.budget, self.dtype = hkv, hq, head_dim, budget, dtype

    def fill(self, slot, length):
        self.work_k[slot, :, :length] = randn((self.hkv, length, self.head_dim), self.dtype, self.g)
        self.work_v[slot, :, :length] = randn((self.hkv, length, self.head_dim), self.dtype, self.g)
        self.lens[slot] = length

    def inputs(self, tokens):
        q = randn((tokens, self.hq, self.head_dim), self.dtype, self.g)
        k = randn((tokens, self.hkv, self.head_dim), self.dtype, self.g)
        v = randn((tokens, self.hkv, self.head_dim), self.dtype, self.g)
        return q, k, v


class Device:
    def __init__(self, case, cuda, rows):
        from ds355 import attention

        self.k = case.work_k.to(cuda)
        self.v = case.work_v.to(cuda)
        self.lens = case.lens.to(cuda)
        self.ws = attention.new_attention_workspace(rows, case.hq, case.hkv, case.head_dim, case.budget, cuda)


def _step(case, dev, cuda, slots, positions, tokens, scale, device_positions=False):
    """One launch and the oracle on the same inputs; returns the GPU output."""
    from ds355 import attention

    q, k, v = case.inputs(tokens)
    if positions is None:
        host_pos = [int(case.lens[s]) for s in slots]
        pos_arg = None
    else:
        host_pos = list(positions)
        pos_arg = torch.tensor(host_pos, dtype=torch.int32, device=cuda) if device_positions else host_pos
    expected = torch.full_like(q, float("nan"))
    lens = case.lens.tolist()
    O.draft_linear_attention(q, k, v, scale, expected, case.work_k, case.work_v, lens, slots, host_pos)
    case.lens = torch.tensor(lens, dtype=torch.int32)
    out = torch.full_like(q, float("nan")).to(cuda)
    attention.draft_linear_attention(q.to(cuda), k.to(cuda), v.to(cuda), out, dev.k, dev.v, dev.lens, slots, pos_arg,
                                     scale=scale, workspace=dev.ws)
    torch.cuda.synchronize()
    actual = out.cpu()
    rows = len(slots)
    terms = attention_terms(q[:rows], case.work_k, case.work_v, slots, host_pos, scale)
    assert_attention_close(actual[:rows], expected[:rows], terms)
    assert actual[rows:].count_nonzero() == 0
    _same_bits(dev.k.cpu(), case.work_k)
    _same_bits(dev.v.cpu(), case.work_v)
    assert torch.equal(dev.lens.cpu(), case.lens)
    assert attention.attention_status(dev.ws) == 0
    return actual, q, k, v, host_pos


@pytest.mark.parametrize("slots", [[0], [0, 1, 2], [3, 0, 2]])
@pytest.mark.parametrize("heads,dim,query_heads", [(2, 128, 8), (4, 256, 4)])
def test_batched_linear_attention_matches_ragged_reference(cuda, slots, heads, dim, query_heads):
    """The reference's device test: budget 64, positions [3, 11, 6], two steps, 5 query rows."""
    case = Case(31, 4, heads, query_heads, dim, 64)
    positions = [3, 11, 6][: len(slots)]
    for s, p in zip(slots, positions):
        case.fill(s, p)
    keys_before = case.work_k.clone()
    values_before = case.work_v.clone()
    dev = Device(case, cuda, 5)
    for step in range(2):
        actual, q, new_k, new_v, _ = _step(case, dev, cuda, slots, [p + step for p in positions], 5, dim ** -0.5)
        for row, (slot, position) in enumerate(zip(slots, positions)):
            end = position + step + 1
            keys_before[slot, :, end - 1] = new_k[row]
            values_before[slot, :, end - 1] = new_v[row]
            k = keys_before[slot, :, :end].repeat_interleave(query_heads // heads, dim=0).float()
            v = values_before[slot, :, :end].repeat_interleave(query_heads // heads, dim=0).float()
            weights = torch.einsum("hd,hsd->hs", q[row].float(), k)
            expected = torch.einsum("hs,hsd->hd", (weights * dim ** -0.5).softmax(-1), v)
            torch.testing.assert_close(actual[row].float(), expected, rtol=REF_RTOL, atol=REF_ATOL)
            assert int(dev.lens[slot]) == end


def test_long_rows_span_merge_and_device_positions(cuda):
    """Budget 2048 with rows ending at span boundaries, permuted slots, then
    two steps that read positions from the slots' working lengths on the device."""
    from ds355 import attention

    case = Case(7, 12, 4, 32, 128, 2048)
    slots = [5, 0, 11, 3, 7, 1, 9, 2]
    lengths = [0, 1, 255, 256, 257, 1000, 1791, 2045]
    for s, n in zip(slots, lengths):
        case.fill(s, n)
    dev = Device(case, cuda, 10)
    _step(case, dev, cuda, slots, lengths, 10, 128 ** -0.5)
    for _ in range(2):
        _step(case, dev, cuda, slots, None, 10, 128 ** -0.5)
    assert attention.attention_epoch(dev.ws) == 3


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("hq,hkv,dim", [(8, 8, 64), (16, 2, 128), (64, 2, 128), (24, 2, 64), (8, 1, 256)])
def test_group_sizes_dtypes_and_head_dims(cuda, dtype, hq, hkv, dim):
    """G = 1, 8, 32 (two query blocks) and 12 (a partial block); head_dim 64/128/256; bf16 and fp16."""
    case = Case(hq * 100 + dim, 6, hkv, hq, dim, 1024, dtype)
    slots = [4, 1, 0]
    lengths = [700, 5, 1023 - 1]
    for s, n in zip(slots, lengths):
        case.fill(s, n)
    dev = Device(case, cuda, 3)
    _step(case, dev, cuda, slots, lengths, 3, dim ** -0.5, device_positions=True)
    _step(case, dev, cuda, slots, None, 3, dim ** -0.5)


def test_reused_workspace_across_shapes(cuda):
    """One workspace serves batches of different sizes and layouts one after another."""
    from ds355 import attention

    big = Case(3, 8, 4, 32, 128, 2048)
    for s in range(8):
        big.fill(s, 250 * s + 17)
    dev = Device(big, cuda, 8)
    _step(big, dev, cuda, list(range(8)), None, 8, 0.09)
    small = Case(4, 3, 2, 4, 64, 512)
    for s in range(3):
        small.fill(s, 100 * s + 300)
    dev_small = Device(small, cuda, 3)
    dev_small.ws = dev.ws  # larger than needed: counters and tags carry over
    _step(small, dev_small, cuda, [2, 0], None, 2, 0.2)
    _step(big, dev, cuda, [7, 3, 1], None, 4, 0.09)
    assert attention.attention_epoch(dev.ws) == 3


def test_out_of_range_position_zeroes_the_row_and_sets_status(cuda):
    """A device position past the budget cannot raise on the host: its row is
    zero, nothing else changes for it, the other rows are unaffected, and
    bit 0 of the status word is set."""
    from ds355 import attention

    case = Case(5, 3, 2, 8, 128, 256)
    for s in range(3):
        case.fill(s, 40 + s)
    dev = Device(case, cuda, 3)
    q, k, v = case.inputs(3)
    out = torch.full_like(q, float("nan")).to(cuda)
    pos = torch.tensor([40, 256, 42], dtype=torch.int32, device=cuda)
    attention.draft_linear_attention(q.to(cuda), k.to(cuda), v.to(cuda), out, dev.k, dev.v, dev.lens, [0, 1, 2], pos,
                                     scale=0.1, workspace=dev.ws)
    torch.cuda.synchronize()
    expected = torch.zeros_like(q)
    lens = case.lens.tolist()
    O.draft_linear_attention(q[[0, 2]], k[[0, 2]], v[[0, 2]], 0.1, expected[:2], case.work_k, case.work_v, lens,
                             [0, 2], [40, 42])
    actual = out.cpu()
    terms = attention_terms(q[[0, 2]], case.work_k, case.work_v, [0, 2], [40, 42], 0.1)
    assert_attention_close(actual[[0, 2]], expected[:2], terms)
    assert actual[1].count_nonzero() == 0
    assert dev.lens.cpu().tolist() == [41, 41, 43]
    _same_bits(dev.k.cpu(), case.work_k)
    assert attention.attention_status(dev.ws) & attention.STATUS_BAD_POSITION


def test_runtime_forward_attention_after_compact_prefill(cuda):
    """DiffSpecDraftCache: the rebuild arms the root step at each slot's history
    length; forward_attention then runs on the device state with no host reads."""
    from ds355 import runtime

    class Rotary:
        rotary_dim = 128
        is_neox_style = True

        def __init__(self):
            self.cos_sin_cache = O.rope_cos_sin_cache(128, 512, 1.0e6).to(torch.bfloat16)

    settings = runtime.DiffSpecSettings(chunk_size=16, token_budget=256, retrieval_interval=1, max_tree_nodes=4,
                                        max_tree_depth=4, tree_threshold=0.7, adaptive_profile=False)
    cache = runtime.DiffSpecDraftCache(settings, max_num_reqs=4, max_model_len=512, num_kv_heads=2, head_dim=128,
                                       target_num_layers=2, dtype=torch.bfloat16, device=cuda,
                                       rotary_embedding=Rotary())
    g = gen(21)
    cache.raw_key.copy_(randn(cache.raw_key.shape, torch.bfloat16, g))
    cache.raw_value.copy_(randn(cache.raw_value.shape, torch.bfloat16, g))
    cache.working_key.fill_(float("nan"))
    cache.working_value.fill_(float("nan"))
    cache.set_active_requests(["a", "b", "c"])
    cache.prepare_compact_prefill(None, 3, committed_seq_lens=[300, 40, 7])
    torch.cuda.synchronize()
    work_k, work_v = cache.working_key.cpu(), cache.working_value.cpu()
    lens = cache.working_lens.cpu().tolist()
    for step in range(3):
        if step:
            cache.prepare_draft_step()
        slots = list(cache._pending_request_indices)
        positions = [lens[s] for s in slots]
        q = randn((4, 8, 128), torch.bfloat16, g)
        k = randn((4, 2, 128), torch.bfloat16, g)
        v = randn((4, 2, 128), torch.bfloat16, g)
        expected = torch.empty_like(q)
        O.draft_linear_attention(q, k, v, 0.088, expected, work_k, work_v, lens, slots, positions)
        out = torch.full((4, 8 * 128), float("nan"), dtype=torch.bfloat16, device=cuda)
        cache.forward_attention(q.to(cuda), k.view(4, 256).to(cuda), v.to(cuda), 0.088, out)
        assert not cache.has_pending_attention()
        torch.cuda.synchronize()
        terms = torch.zeros((4, 8, 128))
        terms[: len(slots)] = attention_terms(q[: len(slots)], work_k, work_v, slots, positions, 0.088)
        assert_attention_close(out.view(4, 8, 128).cpu(), expected, terms)
        assert cache.working_lens.cpu().tolist() == lens
        _same_bits(cache.working_key.cpu(), work_k)
        _same_bits(cache.working_value.cpu(), work_v)


@pytest.mark.parametrize("seed", range(24))
def test_random_rows_positions_and_groups(cuda, seed):
    """Seeded random batches: rows on permuted spare slots at random positions (0 to the
    last cache row), GQA groups 1-32, head_dim 64/128/256, budgets 64-2048, bf16/fp16,
    output padding rows; one step with host positions, one reading the working lengths."""
    import random

    rnd = random.Random(500 + seed)
    hkv = rnd.choice([1, 2, 4, 8])
    group = rnd.choice([1, 2, 4, 8, 16, 32])
    dim = rnd.choice([64, 128, 256])
    budget = rnd.choice([64, 512, 2048])
    dtype = rnd.choice([torch.bfloat16, torch.float16])
    num_slots = rnd.randint(1, 24)
    rows = rnd.randint(1, num_slots)
    slots = rnd.sample(range(num_slots), rows)
    lengths = [rnd.choice([0, budget - 2, rnd.randint(0, budget - 2)]) for _ in range(rows)]
    print(f"seed {seed}: {rows} rows of {num_slots} slots, {hkv * group}/{hkv} heads x {dim}, budget {budget}, "
          f"{dtype}, lengths {lengths}", flush=True)
    case = Case(900 + seed, num_slots, hkv, hkv * group, dim, budget, dtype)
    for s, n in zip(slots, lengths):
        case.fill(s, n)
    tokens = rows + rnd.choice([0, 3])
    dev = Device(case, cuda, tokens)
    _step(case, dev, cuda, slots, lengths, tokens, dim ** -0.5)
    _step(case, dev, cuda, slots, None, tokens, dim ** -0.5)


@pytest.mark.parametrize("dim", [64, 128, 256])
@pytest.mark.parametrize("rows", [16, 400])
def test_rows_that_end_inside_a_tile(cuda, dim, rows):
    """Row ends at and beside the half tiles (8 tokens) that key loads take lines of, in the
    one-shot kernel and (many rows) the streamed one."""
    ends = [0, 1, 6, 7, 8, 9, 14, 15, 16, 17, 23, 24, 31, 32, 33, 63]
    positions = (ends * (rows // 16))[:rows]
    case = Case(17 + dim, rows, 4, 16, dim, 64)
    for s, p in enumerate(positions):
        case.fill(s, p)
    _step(case, Device(case, cuda, rows), cuda, list(range(rows)), positions, rows, dim ** -0.5, device_positions=True)


@pytest.mark.parametrize("rows,hq,hkv,dim,budget,dtype", [
    (20, 32, 4, 128, 2048, torch.bfloat16),  # 640 spans: just above one round of one-shot workgroups
    (33, 8, 8, 64, 2304, torch.float16),  # one query head per KV head
    (9, 64, 2, 256, 1100, torch.bfloat16),  # two query blocks, a last span that is not whole
    (48, 12, 2, 128, 1536, torch.float16),  # groups of 6
])
def test_streamed_batches(cuda, rows, hq, hkv, dim, budget, dtype):
    """Batches of more than one round of spans (attention_stream_kernel): rows that end at and
    beside step (128) and span (256) boundaries, empty and full rows, padding rows; one step
    with device positions, two that read the working lengths.  A slot out of range zeroes its
    row only."""
    from ds355 import attention

    case = Case(rows * 7 + dim, rows + 2, hkv, hq, dim, budget, dtype)
    edges = [0, 1, 31, 32, 127, 128, 129, 255, 256, 257, 383, 384, 1000, budget - 4, budget - 5]
    slots = [(5 * r + 3) % (rows + 2) if (rows + 2) % 5 else rows + 1 - r for r in range(rows)]
    lengths = [min(edges[r % len(edges)], budget - 4) for r in range(rows)]
    for s, n in zip(slots, lengths):
        case.fill(s, n)
    dev = Device(case, cuda, rows)
    _step(case, dev, cuda, slots, lengths, rows + 2, dim ** -0.5, device_positions=True)
    for _ in range(2):
        _step(case, dev, cuda, slots, None, rows + 2, dim ** -0.5)
    assert attention.attention_epoch(dev.ws) == 3
    # One row's slot is out of range: zeros for it, the others as before.
    q, k, v = case.inputs(rows)
    outs = []
    for bad in (None, rows // 2):
        k_dev, v_dev, lens = dev.k.clone(), dev.v.clone(), dev.lens.clone()
        out = torch.full_like(q, float("nan")).to(cuda)
        chosen = [-1 if r == bad else s for r, s in enumerate(slots)]
        attention.draft_linear_attention(q.to(cuda), k.to(cuda), v.to(cuda), out, k_dev, v_dev, lens, chosen, None,
                                         scale=dim ** -0.5, workspace=dev.ws)
        outs.append(out.cpu())
    keep = [r for r in range(rows) if r != rows // 2]
    whole, partly = outs
    assert partly[rows // 2].count_nonzero() == 0
    _same_bits(partly[keep], whole[keep])
    assert attention.attention_status(dev.ws) == attention.STATUS_BAD_POSITION


@pytest.mark.parametrize("rows,dim,budget", [(3, 128, 512), (20, 128, 2048)])
def test_expired_wait_keeps_the_working_lengths(cuda, rows, dim, budget):
    """A launch whose last workgroup stops waiting for the others (forced by the owner's header
    word) sets bit 1 and leaves the working lengths, in the one-shot and the streamed kernel; its
    outputs and cache rows are written, and the next launch on the workspace is an ordinary one."""
    from ds355 import attention

    case = Case(rows + dim, rows, 4, 32, dim, budget)
    for s in range(rows):
        case.fill(s, (97 * s + 40) % (budget - 2))
    dev = Device(case, cuda, rows)
    slots, positions = list(range(rows)), case.lens.tolist()
    q, k, v = case.inputs(rows)
    dev.ws[12:16].view(torch.int32).fill_(1)
    out = torch.full_like(q, float("nan")).to(cuda)
    attention.draft_linear_attention(q.to(cuda), k.to(cuda), v.to(cuda), out, dev.k, dev.v, dev.lens, slots, None,
                                     scale=0.1, workspace=dev.ws)
    torch.cuda.synchronize()
    assert attention.attention_status(dev.ws) == attention.STATUS_PARTIAL_TIMEOUT
    assert attention.attention_epoch(dev.ws) == 1
    assert torch.equal(dev.lens.cpu(), case.lens)
    expected = torch.zeros_like(q)
    O.draft_linear_attention(q, k, v, 0.1, expected, case.work_k, case.work_v, case.lens.tolist(), slots, positions)
    assert_attention_close(out.cpu(), expected, attention_terms(q, case.work_k, case.work_v, slots, positions, 0.1))
    _same_bits(dev.k.cpu(), case.work_k)
    _same_bits(dev.v.cpu(), case.work_v)
    dev.ws[8:16].view(torch.int32).zero_()
    _step(case, dev, cuda, slots, None, rows, 0.1)
    assert attention.attention_epoch(dev.ws) == 2


@pytest.mark.parametrize("rows,budget,inside", [
    (6, 512, [8, 14, 15, 16, 25, 30]),  # one-shot: the first tile pair of each wave's four
    (50, 2048, [8, 14, 15, 16, 25, 30, 31, 40, 47, 48, 60, 63])])  # streamed
@pytest.mark.parametrize("dim", [64, 128, 256])
def test_infinite_value_of_the_new_token(cuda, rows, budget, inside, dim):
    """An infinity in the new token's value stays that infinity in its output column, wherever the
    token lies within a wave's tiles: it is also loaded in place of rows past the position, with
    probability 0, and must not become NaN there.  bf16, whose probabilities split into two
    parts of one sign (fp16's lower part may be negative)."""
    from ds355 import attention

    case = Case(rows * dim, rows, 4, 16, dim, budget)
    positions = [64 * (5 * r % (budget // 64)) + inside[r % len(inside)] for r in range(rows)]
    for s, n in enumerate(positions):
        case.fill(s, n)
    q, k, v = case.inputs(rows)
    q.abs_()
    case.work_k[:, :, ::8].abs_()  # scores above 0 in every half tile; the new token's is 0,
    k.zero_()  # so both parts of its probability are above 0
    v[:, :, 5], v[:, :, dim - 3] = float("inf"), float("-inf")
    dev = Device(case, cuda, rows)
    out = torch.full_like(q, float("nan")).to(cuda)
    attention.draft_linear_attention(q.to(cuda), k.to(cuda), v.to(cuda), out, dev.k, dev.v, dev.lens,
                                     list(range(rows)), None, scale=dim ** -0.5, workspace=dev.ws)
    expected = torch.zeros_like(q)
    O.draft_linear_attention(q, k, v, dim ** -0.5, expected, case.work_k, case.work_v, case.lens.tolist(),
                             list(range(rows)), positions)
    actual = out.cpu()
    assert not expected.isnan().any() and (expected[:, :, 5] == float("inf")).all()
    for name in ("isnan", "isposinf", "isneginf"):
        differ = (getattr(torch, name)(actual) != getattr(torch, name)(expected)).nonzero().tolist()
        assert not differ, (name, differ[:4])


def _launched_streamed(ws, rows, hkv, group, dim, budget, tag):
    """Whether the launch of epoch `tag` was the streamed kernel: its workgroups, fewer than the
    batch's spans, are the ones that leave "seen" words."""
    spans = rows * hkv * ((group + 15) // 16) * (-(-budget // (256 if dim <= 128 else 128)))
    seen = ws[256 + 4 * 65536:][: 8 * spans].view(torch.int32)[1::2]
    return int((seen == tag).sum()) < spans


@pytest.mark.parametrize("rows,hq,hkv,dim,budget,dtype", [
    (24, 32, 4, 128, 2048, torch.bfloat16),  # one query block, units within and across ranges
    (57, 64, 8, 128, 4096, torch.float16),
    (48, 32, 8, 64, 2048, torch.bfloat16),
    (16, 64, 2, 256, 2048, torch.bfloat16),  # two query blocks
    (7, 16, 1, 256, 8192, torch.float16),  # fewer units than workgroups: units of many ranges
])
def test_a_row_has_the_same_bits_in_any_batch(cuda, rows, hq, hkv, dim, budget, dtype):
    """A row's output does not depend on the rows beside it, their order or count, nor on which
    kernel the batch's size selects: a streamed batch, its reverse, a part of it and every row
    alone (one-shot) give the same bits."""
    from ds355 import attention

    case = Case(rows + dim, rows, hkv, hq, dim, budget, dtype)
    edges = [0, 31, 127, 128, 255, 256, 511, 700, budget // 2, budget - 130, budget - 1]
    positions = [min(edges[(3 * r) % len(edges)] + r // len(edges), budget - 1) for r in range(rows)]
    case.work_k, case.work_v = (randn(case.shape, dtype, case.g) for _ in range(2))
    dev = Device(case, cuda, rows)
    q, k, v = (t.to(cuda) for t in case.inputs(rows))

    def run(order):
        at = torch.tensor(order, device=cuda)
        out = torch.empty((len(order), hq, dim), dtype=dtype, device=cuda)
        attention.draft_linear_attention(q[at], k[at], v[at], out, dev.k, dev.v, dev.lens, order,
                                         [positions[r] for r in order], scale=dim ** -0.5, workspace=dev.ws)
        torch.cuda.synchronize()
        streamed = _launched_streamed(dev.ws, len(order), hkv, hq // hkv, dim, budget,
                                      attention.attention_epoch(dev.ws))
        return out.cpu(), streamed

    whole, streamed = run(list(range(rows)))
    assert streamed
    backwards, streamed = run(list(range(rows))[::-1])
    assert streamed
    _same_bits(backwards.flip(0), whole)
    part, _ = run(list(range(1, rows, 2)))
    _same_bits(part, whole[1::2])
    for r in range(rows):
        alone, streamed = run([r])
        assert not streamed
        _same_bits(alone[0], whole[r])
    assert attention.attention_status(dev.ws) == 0


def test_streamed_and_one_shot_launches_share_a_workspace(cuda):
    """One workspace, launches of both kernels in turn (their "seen" words and partials lie
    elsewhere, the unit counters and the epoch are the same ones): each step has the oracle's
    outputs, caches and lengths, its own epoch and a clear status."""
    from ds355 import attention

    case = Case(77, 30, 4, 32, 128, 2048)
    for s in range(30):
        case.fill(s, [0, 40, 255, 256, 700, 1500, 2030][s % 7] + s // 7)
    dev = Device(case, cuda, 28)
    plan = [(range(28), True), ([3, 17, 4], False), (range(29, 4, -1), True), ([9], False), (range(0, 30, 2), False),
            (range(2, 30), True)]
    for n, (slots, expect) in enumerate(plan, 1):
        slots = list(slots)
        _step(case, dev, cuda, slots, None, len(slots) + 1, 0.09)
        assert attention.attention_epoch(dev.ws) == n
        assert _launched_streamed(dev.ws, len(slots), 4, 8, 128, 2048, n) == expect


@pytest.mark.parametrize("rows", [3, 50])
@pytest.mark.parametrize("dim,dtype", [(64, torch.float16), (128, torch.bfloat16), (256, torch.bfloat16)])
def test_strided_rows_and_heads(cuda, rows, dim, dtype):
    """Queries, keys and values that are parts of one packed buffer and an output with spare
    elements give the bits of contiguous ones, in the one-shot and the streamed kernel."""
    from ds355 import attention

    hq, hkv, budget = 16, 4, 2048
    case = Case(rows + dim, rows, hkv, hq, dim, budget, dtype)
    lengths = [(331 * r + 7) % (budget - 1) for r in range(rows)]
    for s, n in enumerate(lengths):
        case.fill(s, n)
    q, k, v = (t.to(cuda) for t in case.inputs(rows))
    packed = torch.full((rows, hq + 2 * hkv + 1, dim + 8), float("nan"), dtype=dtype, device=cuda)[..., :dim]
    packed[:, :hq], packed[:, hq: hq + hkv], packed[:, hq + hkv: hq + 2 * hkv] = q, k, v
    wide = torch.full((rows, hq + 3, dim + 16), float("nan"), dtype=dtype, device=cuda)
    results = []
    for args, out in (((q, k, v), torch.empty_like(q)),
                      ((packed[:, :hq], packed[:, hq: hq + hkv], packed[:, hq + hkv: hq + 2 * hkv]),
                       wide[:, 1: hq + 1, 8: dim + 8])):
        dev = Device(case, cuda, rows)
        attention.draft_linear_attention(*args, out, dev.k, dev.v, dev.lens, list(range(rows)), None,
                                         scale=dim ** -0.5, workspace=dev.ws)
        results.append((out.cpu(), dev.k.cpu(), dev.v.cpu(), dev.lens.cpu()))
        assert _launched_streamed(dev.ws, rows, hkv, hq // hkv, dim, budget, 1) == (rows == 50)
    for a, b in zip(*results):
        _same_bits(a, b)
    outside = wide.cpu()
    outside[:, 1: hq + 1, 8: dim + 8] = float("nan")
    assert outside.isnan().all()


def test_streamed_launch_replayed_from_a_graph(cuda):
    """A captured streamed launch, replayed with other inputs and the eager launch between the
    replays, gives the eager launch's bits every time."""
    from ds355 import attention

    rows, hq, hkv, dim, budget = 28, 32, 4, 128, 2048
    case = Case(5, rows, hkv, hq, dim, budget)
    for s in range(rows):
        case.fill(s, (211 * s + 250) % (budget - 6))
    slots = torch.tensor([(5 * r + 2) % rows for r in range(rows)], dtype=torch.int32, device=cuda)
    q, k, v = (t.to(cuda) for t in case.inputs(rows + 2))
    graphed, eager, warm = (Device(case, cuda, rows) for _ in range(3))

    def launch(dev):
        out = torch.full_like(q, float("nan"))
        attention.draft_linear_attention(q, k, v, out, dev.k, dev.v, dev.lens, slots, None, scale=dim ** -0.5,
                                         workspace=dev.ws)
        return out

    launch(warm)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        out = launch(graphed)
    for step in range(1, 5):
        for buffer, fresh in zip((q, k, v), case.inputs(rows + 2)):
            buffer.copy_(fresh)
        graph.replay()
        torch.cuda.synchronize()
        expected = launch(eager)
        _same_bits(out.cpu(), expected.cpu())
        for a, b in ((graphed.k, eager.k), (graphed.v, eager.v), (graphed.lens, eager.lens)):
            _same_bits(a.cpu(), b.cpu())
        assert attention.attention_epoch(graphed.ws) == step and attention.attention_status(graphed.ws) == 0
        assert _launched_streamed(graphed.ws, rows, hkv, hq // hkv, dim, budget, step)
