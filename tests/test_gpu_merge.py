"""Split-KV merge at the edges of its batches: splits per row around 8 (one
batch of a wavefront), 16 and 64 (one batch of each wavefront of a workgroup)
and an odd head count, eagerly and from a graph plan whose launch serves both
forms, against the oracle (tolerance of the attention tests: 16-bit partial
rows and outputs)."""
import pytest
import torch

import feattn
from feattn import workloads as W
from oracle import aten_attention as A

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", ["bf16", "f16"])
@pytest.mark.parametrize("rows", [1, 3])
def test_split_counts(dev, dtype, rows):
    # 5 kv heads: workgroups of one wavefront and shares of 64 tokens, so a
    # sequence alone is cut into ceil(tokens / 64) splits.
    hq = hkv = 5
    plan = feattn.Plan(hq, hkv, 128, 16, 2, 600, dtype == "bf16", 1200)
    graph_plan = feattn.Plan(hq, hkv, 128, 16, 2, 600, dtype == "bf16", 1200)
    for lens in ([64 * 130 + 7], [64 * 8], [64 * 8 + 1], [64 * 16 + 1], [64 * 64], [64 * 64 + 1], [70, 64 * 17]):
        b = W.make_batch(hq, hkv, starts=[n - rows for n in lens], qlens=[rows] * len(lens), seed=lens[0], pool=1200)
        q, kc, vc = W.make_tensors(b, seed=3, dtype=dtype)
        want, want_lse = A.run(b, q, kc, vc, True)
        q, kc, vc = q.to(dev), kc.to(dev), vc.to(dev)
        got = []
        for p, graph in ((plan, False), (graph_plan, True)):
            p.prepare(b.qo, b.kv, b.pages, b.last, b.batch, b.rows, graph=graph)
            forms = p.lists()
            assert forms.decode_items == sum(-(-n // 64) for n in lens) * hkv or len(lens) > 1
            assert forms.merge_rows == rows * len(lens) and forms.merge_wide == int(max(lens) > 8 * 64)
            out = torch.full_like(q, float("nan"))
            lse = torch.full((b.rows, hq), float("nan"), device=dev)
            p.run(q, kc, vc, out, causal=True, lse=lse)
            torch.cuda.synchronize()
            torch.testing.assert_close(out.float().cpu(), want.float(), atol=1e-2, rtol=1e-2)
            torch.testing.assert_close(lse.cpu(), want_lse, atol=1e-3, rtol=0)
            got.append((out, lse))
        assert torch.equal(got[0][0], got[1][0]) and torch.equal(got[0][1], got[1][1])
    plan.close()
    graph_plan.close()


@pytest.mark.parametrize("dtype", ["bf16", "f16"])
def test_infinite_values_stay_infinite(dev, dtype):
    """Infinite V entries in a row's first and last split, for split counts
    around and between the batches of both merge forms: every weight is
    positive, so the output is that infinity, exactly the elements of the
    oracle's that are; the others are within the tolerance."""
    hq = hkv = 5  # shares of 64 tokens: ceil(tokens / 64) splits
    plan = feattn.Plan(hq, hkv, 128, 16, 1, 300, dtype == "bf16", 600)
    graph_plan = feattn.Plan(hq, hkv, 128, 16, 1, 300, dtype == "bf16", 600)
    for splits in (2, 3, 4, 5, 7, 8, 9, 16, 17, 33, 65):
        n = 64 * splits - 5
        b = W.make_batch(hq, hkv, starts=[n - 1], qlens=[1], seed=splits, pool=600)
        q, kc, vc = W.make_tensors(b, seed=4, dtype=dtype)
        for tok, head, dim, sign in ((0, 0, 3, 1), (n - 1, 1, 17, 1), (n - 2, 4, 127, -1)):
            vc[b.tables[0][tok // 16], tok % 16, head, dim] = sign * float("inf")
        want, _ = A.run(b, q, kc, vc, True)
        inf = torch.isinf(want.float())
        assert int(inf.sum()) == 3 and not torch.isnan(want.float()).any()
        q, kc, vc = q.to(dev), kc.to(dev), vc.to(dev)
        for p, graph in ((plan, False), (graph_plan, True)):
            p.prepare(b.qo, b.kv, b.pages, b.last, b.batch, b.rows, graph=graph)
            out = torch.full_like(q, float("nan"))
            p.run(q, kc, vc, out, causal=True)
            torch.cuda.synchronize()
            out = out.float().cpu()
            assert torch.equal(out[inf], want.float()[inf]), splits
            torch.testing.assert_close(out[~inf], want.float()[~inf], atol=1e-2, rtol=1e-2)
    plan.close()
    graph_plan.close()


@pytest.mark.parametrize("hq,hkv,wide_lens,wide_rows,narrow_lens", [(32, 8, [9000, 5000] * 8, 4, [900] * 40),
                                                                    (5, 5, [1300] * 12, 16, [400, 70, 130] * 13)])
def test_graph_captured_on_one_short_sequence(dev, hq, hkv, wide_lens, wide_rows, narrow_lens):
    """A graph captured after a prepare of a single short sequence folds the
    splits of later, much larger batches: more rows and head pairs than the
    launch has workgroups for in the wide form (so workgroups take several),
    and the narrow one; every replay against the oracle and the bits of an
    eager plan."""
    blocks, batch, hpairs = 8000, 40, (hq + 1) // 2
    max_pages = 9000 // 16 + 3
    plan = feattn.Plan(hq, hkv, 128, 16, batch, max_pages, True, blocks)
    eager = feattn.Plan(hq, hkv, 128, 16, batch, max_pages, True, blocks)
    one = W.make_batch(hq, hkv, starts=[30], qlens=[1], seed=1, pool=blocks)
    plan.prepare(one.qo, one.kv, one.pages, one.last, one.batch, one.rows, graph=True)
    grid = plan.lists().merge_grid
    assert grid >= batch * hpairs  # one pass for every row of a batch of the plan's size
    assert grid < len(wide_lens) * wide_rows * hpairs  # several for these rows
    gen = torch.Generator().manual_seed(3)
    kc = torch.randn(blocks + 1, 16, hkv, 128, generator=gen).to(torch.bfloat16)
    vc = torch.randn(blocks + 1, 16, hkv, 128, generator=gen).to(torch.bfloat16)
    kd, vd = kc.to(dev), vc.to(dev)
    q = torch.zeros(16 * batch, hq, 128, dtype=torch.bfloat16, device=dev)
    out = torch.zeros_like(q)
    lse = torch.zeros(16 * batch, hq, device=dev)
    graph = torch.cuda.CUDAGraph()
    torch.cuda.synchronize()
    with torch.cuda.graph(graph):
        plan.run(q, kd, vd, out, causal=True, lse=lse)
    for wide, lens, rows in ((1, wide_lens, wide_rows), (0, narrow_lens, 1), (1, wide_lens, 1), (0, [40, 50], 1),
                             (1, wide_lens, wide_rows)):
        b = W.make_batch(hq, hkv, starts=[n - rows for n in lens], qlens=[rows] * len(lens), seed=len(lens),
                         pool=blocks)
        qb = torch.randn(b.rows, hq, 128, generator=gen).to(torch.bfloat16)
        q[:b.rows].copy_(qb)
        out.fill_(float("nan"))
        lse.fill_(float("nan"))
        plan.prepare(b.qo, b.kv, b.pages, b.last, b.batch, b.rows, graph=True)
        eager.prepare(b.qo, b.kv, b.pages, b.last, b.batch, b.rows)
        forms = plan.lists()
        assert forms.merge_wide == wide and (forms.merge_rows > 0 or lens == [40, 50])
        graph.replay()
        o2, l2 = torch.zeros_like(q[:b.rows]), torch.zeros_like(lse[:b.rows])
        eager.run(q, kd, vd, o2, causal=True, lse=l2)
        torch.cuda.synchronize()
        want, want_lse = A.run(b, qb, kc, vc, True)
        torch.testing.assert_close(o2.float().cpu(), want.float(), atol=1e-2, rtol=1e-2)
        torch.testing.assert_close(l2.cpu(), want_lse, atol=1e-3, rtol=0)
        assert torch.equal(out[:b.rows], o2) and torch.equal(lse[:b.rows], l2)
    plan.close()
    eager.close()
