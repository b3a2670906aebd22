"""Plans of small calls (planner.cpp: plan_short, plan_small_tiles): the item
lists over random batches, built with AddressSanitizer and UndefinedBehaviorSanitizer
(tests/cpp/short_check.cpp), and on the GPU the kernel's edges against the
oracle."""
import os
import shutil
import subprocess

import pytest
import torch

import feattn
from feattn import workloads as W
from oracle import aten_attention as A

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


@pytest.mark.skipif(shutil.which("g++") is None, reason="no host C++ compiler")
def test_short_items_cover_the_batch(tmp_path):
    exe = tmp_path / "short_check"
    subprocess.run(["g++", "-std=c++17", "-O1", "-g", "-fsanitize=address,undefined", "-fno-sanitize-recover=all",
                    "-I" + os.path.join(ROOT, "include"), "-I" + os.path.join(ROOT, "flashengine.cpp_amd", "csrc"),
                    os.path.join(ROOT, "tests", "cpp", "short_check.cpp"),
                    os.path.join(ROOT, "flashengine.cpp_amd", "csrc", "planner.cpp"), "-o", str(exe)],
                   check=True, timeout=300)
    r = subprocess.run([str(exe)], capture_output=True, text=True, timeout=300)
    assert r.returncode == 0, r.stdout + r.stderr


# Context lengths around one block, one block per wavefront, one round of
# loads (64 tokens per wavefront) and the longest uncut sequence of 8- and
# 4-wavefront workgroups (hkv 8 and 4), and cut ones.
LENS = {8: [1, 15, 16, 17, 127, 128, 129, 511, 512, 513, 640, 1023, 1024, 1025, 2100],
        4: [1, 16, 33, 63, 64, 65, 255, 256, 257, 500, 512, 513, 1300]}


@pytest.mark.gpu
@pytest.mark.parametrize("hq,hkv,rows,page", [(32, 8, 1, 16), (16, 8, 1, 64), (40, 8, 5, 16), (8, 8, 8, 32),
                                              (32, 8, 8, 16), (32, 4, 1, 16), (32, 4, 4, 32), (64, 4, 1, 16)])
@pytest.mark.parametrize("dtype,causal", [("bf16", True), ("f16", False)])
def test_short_kernel_edges(dev, hq, hkv, rows, page, dtype, causal):
    """All the lengths in one batch (cut into pieces and merged), then the
    uncut ones; eagerly and replayed from a graph captured on another batch.
    Everything a call may not read -- cache rows past a sequence's end and
    pages of no sequence -- is NaN.  The tolerance is the one of the other
    attention tests: 16-bit probabilities and outputs."""
    step = 64 * hkv
    plan = feattn.Plan(hq, hkv, 128, page, 16, 2200 // page + 2, dtype == "bf16", 12000 // page)
    graph_plan = feattn.Plan(hq, hkv, 128, page, 16, 2200 // page + 2, dtype == "bf16", 12000 // page)
    graph = None
    for lens in (LENS[hkv], [n for n in LENS[hkv] if n <= 2 * step], [2 * step]):
        lens = [max(n, rows) for n in lens]
        b = W.make_batch(hq, hkv, starts=[n - rows for n in lens], qlens=[rows] * len(lens), seed=len(lens),
                         page=page, pool=12000 // page)
        q, kc, vc = W.make_tensors(b, seed=7, dtype=dtype)
        want, want_lse = A.run(b, q, kc, vc, causal)
        used = torch.zeros((b.blocks + 1) * page, dtype=torch.bool)
        for s in range(b.batch):
            for t in range(b.lens[s]):
                used[b.tables[s][t // page] * page + t % page] = True
        used = used.view(b.blocks + 1, page)
        kc[~used] = float("nan")
        vc[~used] = float("nan")
        kd, vd, qd = kc.to(dev), vc.to(dev), q.to(dev)

        def run(p):
            out = torch.full_like(qd, float("nan"))
            lse = torch.full((b.rows, hq), float("nan"), device=dev)
            p.run(qd, kd, vd, out, causal=causal, lse=lse)
            return out, lse

        plan.prepare(b.qo, b.kv, b.pages, b.last, b.batch, b.rows)
        graph_plan.prepare(b.qo, b.kv, b.pages, b.last, b.batch, b.rows, graph=True)
        assert plan.lists(causal).short_units > 0 and graph_plan.lists(causal).short_units > 0
        got = [run(plan), run(graph_plan)]
        if graph is None:
            sq, sk, sv = qd.clone(), kd.clone(), vd.clone()
            so, sl = torch.full_like(sq, float("nan")), torch.full((b.rows, hq), float("nan"), device=dev)
            torch.cuda.synchronize()
            graph = torch.cuda.CUDAGraph()
            with torch.cuda.graph(graph):
                graph_plan.run(sq, sk, sv, so, causal=causal, lse=sl)
        sq[:b.rows].copy_(qd)
        sk.copy_(kd)
        sv.copy_(vd)
        graph.replay()
        got.append((so[:b.rows].clone(), sl[:b.rows].clone()))
        torch.cuda.synchronize()
        for out, lse in got:
            torch.testing.assert_close(out.float().cpu(), want.float(), atol=1e-2, rtol=1e-2)
            torch.testing.assert_close(lse.cpu(), want_lse, atol=1e-3, rtol=0)
            assert torch.equal(out, got[0][0]) and torch.equal(lse, got[0][1])
    plan.close()
    graph_plan.close()


@pytest.mark.gpu
@pytest.mark.parametrize("hq,hkv,rows,page", [(32, 8, 1, 16), (16, 8, 1, 64), (40, 8, 5, 16), (8, 8, 8, 32),
                                              (32, 8, 8, 16), (32, 4, 1, 16), (32, 4, 4, 32), (64, 4, 1, 16)])
@pytest.mark.parametrize("dtype,causal", [("bf16", True), ("f16", False)])
def test_share_kernel_edges(dev, hq, hkv, rows, page, dtype, causal):
    """The same lengths beside a chunk, which puts them on the decode shares
    (as long contexts are): the same edges of that kernel, eagerly and
    through a graph plan, which must give the same bits."""
    lens = [max(n, rows) for n in LENS[hkv]] + [70]
    b = W.make_batch(hq, hkv, starts=[n - rows for n in lens[:-1]] + [0], qlens=[rows] * (len(lens) - 1) + [70],
                     seed=len(lens), page=page, extra_pages=2)
    q, kc, vc = W.make_tensors(b, seed=8, dtype=dtype)
    want, want_lse = A.run(b, q, kc, vc, causal)
    used = torch.zeros((b.blocks + 1) * page, dtype=torch.bool)
    for s in range(b.batch):
        for t in range(b.lens[s]):
            used[b.tables[s][t // page] * page + t % page] = True
    used = used.view(b.blocks + 1, page)
    kc[~used] = float("nan")
    vc[~used] = float("nan")
    q, kc, vc = q.to(dev), kc.to(dev), vc.to(dev)
    got = []
    for graph in (False, True):
        plan = feattn.Plan(hq, hkv, 128, page, b.batch, b.max_pages(), dtype == "bf16", b.blocks)
        plan.prepare(b.qo, b.kv, b.pages, b.last, b.batch, b.rows, graph=graph)
        forms = plan.lists(causal)
        assert forms.short_units == 0 and forms.decode_items > 0 and forms.merge_rows > 0
        out = torch.full_like(q, float("nan"))
        lse = torch.full((b.rows, hq), float("nan"), device=dev)
        plan.run(q, kc, vc, out, causal=causal, lse=lse)
        torch.cuda.synchronize()
        plan.close()
        torch.testing.assert_close(out.float().cpu(), want.float(), atol=1e-2, rtol=1e-2)
        torch.testing.assert_close(lse.cpu(), want_lse, atol=1e-3, rtol=0)
        got.append((out, lse))
    assert torch.equal(got[0][0], got[1][0]) and torch.equal(got[0][1], got[1][1])


# (heads, cached tokens, new tokens, masks): the lists a plan reports, eagerly
# and for a graph.
FORMS = [
    (32, 8, [63] * 4, [1] * 4, dict(short_units=4 * 8, decode_items=0, merge_rows=0)),
    (32, 8, [700, 30], [1, 1], dict(short_units=3 * 8, merge_rows=1)),
    (32, 8, [3000] * 12, [1] * 12, dict(short_units=0, merge_rows=12, tile_items=0)),
    (5, 5, [300], [1], dict(short_units=0, decode_items=25, merge_rows=1, merge_wide=0)),
    (5, 5, [700], [1], dict(short_units=0, decode_items=55, merge_rows=1, merge_wide=1)),
    (16, 8, [0], [100], dict(short_units=0, tile_items=32, tile_rows=32, merge_rows=0)),
    (16, 8, [4000], [100], dict(tile_rows=64, merge_rows=100)),
    (32, 8, [60, 0], [1, 100], dict(short_units=0, tile_items=56, tile_rows=16)),
]


@pytest.mark.gpu
@pytest.mark.parametrize("hq,hkv,starts,qlens,want", FORMS)
@pytest.mark.parametrize("graph", [False, True])
def test_lists_report_the_prepared_form(dev, hq, hkv, starts, qlens, want, graph):
    b = W.make_batch(hq, hkv, starts=starts, qlens=qlens, seed=1)
    plan = feattn.Plan(hq, hkv, 128, 16, b.batch, b.max_pages(), True, b.blocks)
    with pytest.raises(RuntimeError, match="before prepare"):
        plan.lists()
    plan.prepare(b.qo, b.kv, b.pages, b.last, b.batch, b.rows, graph=graph)
    for causal in (True, False):
        got = plan.lists(causal)._asdict()
        assert {k: got[k] for k in want} == want
    plan.close()


@pytest.mark.gpu
@pytest.mark.parametrize("hq,hkv,starts,qlens", [
    (16, 8, [0], [17]), (16, 8, [0, 0, 0], [32, 33, 65]), (16, 8, [0], [777]), (32, 8, [0, 31], [15, 17]),
    (32, 8, [448, 0], [64, 512]), (32, 8, [449], [64]), (32, 4, [500, 100], [9, 40]), (40, 8, [300, 7], [12, 13]),
    (64, 1, [0, 90], [5, 70]), (32, 8, [100, 700, 0], [48, 1, 3]), (32, 8, [0], [1100]), (16, 8, [0], [912]),
    (16, 8, [0], [960]), (40, 8, [300] * 4, [180] * 4), (40, 8, [300] * 4, [194] * 4)])
@pytest.mark.parametrize("dtype,causal", [("bf16", True), ("f16", False)])
def test_small_tile_items(dev, hq, hkv, starts, qlens, dtype, causal):
    """Chunks at the edges of the 64-column items and of the rule that makes
    them, some beside decode rows, against the oracle (tolerance of the other
    attention tests); a graph plan gives the same bits."""
    b = W.make_batch(hq, hkv, starts=starts, qlens=qlens, seed=11, extra_pages=2)
    q, kc, vc = W.make_tensors(b, seed=5, dtype=dtype)
    want, want_lse = A.run(b, q, kc, vc, causal)
    q, kc, vc = q.to(dev), kc.to(dev), vc.to(dev)
    got = []
    for graph in (False, True):
        plan = feattn.Plan(hq, hkv, 128, 16, b.batch, b.max_pages(), dtype == "bf16", b.blocks)
        plan.prepare(b.qo, b.kv, b.pages, b.last, b.batch, b.rows, graph=graph)
        out = torch.full_like(q, float("nan"))
        lse = torch.full((b.rows, hq), float("nan"), device=dev)
        plan.run(q, kc, vc, out, causal=causal, lse=lse)
        torch.cuda.synchronize()
        plan.close()
        torch.testing.assert_close(out.float().cpu(), want.float(), atol=1e-2, rtol=1e-2)
        torch.testing.assert_close(lse.cpu(), want_lse, atol=1e-3, rtol=0)
        got.append((out, lse))
    assert torch.equal(got[0][0], got[1][0]) and torch.equal(got[0][1], got[1][1])


@pytest.mark.gpu
def test_graph_tile_policy_is_the_full_width_items(dev):
    """Short 16-row blocks of 8 heads per kv head are planned as half-width
    items, whose second block reads the K/V again; long ones are one item
    each.  A graph plan's cache policy is fixed by its first prepare, and that
    of the long ones whichever comes first; an eager plan follows each batch."""
    short = W.make_batch(32, 4, starts=[100, 60], qlens=[16, 16], seed=1, pool=2000)
    long = W.make_batch(32, 4, starts=[9000, 12000], qlens=[16, 16], seed=2, pool=2000)
    chunk = W.make_batch(32, 4, starts=[0, 30], qlens=[200, 16], seed=2, pool=2000)
    want = {id(short): (8, 0), id(long): (16, 1), id(chunk): (8, 0)}
    for first, policy in ((short, 1), (long, 1), (chunk, 0)):
        plan = feattn.Plan(32, 4, 128, 16, 2, 800, True, 2000)
        for b in (first, short, long, chunk):
            plan.prepare(b.qo, b.kv, b.pages, b.last, b.batch, b.rows, graph=True)
            for causal in (True, False):
                got = plan.lists(causal)
                assert (got.tile_rows, got.tile_stream) == (want[id(b)][0], policy)
        for b in (short, long, chunk):
            plan.prepare(b.qo, b.kv, b.pages, b.last, b.batch, b.rows)
            assert (plan.lists().tile_rows, plan.lists().tile_stream) == want[id(b)]
        plan.close()


@pytest.mark.gpu
@pytest.mark.parametrize("hq,hkv,seqs,hi", [(32, 8, 64, 64), (32, 4, 200, 64), (8, 8, 50, 60)])
@pytest.mark.parametrize("dtype", ["bf16", "f16"])
def test_graph_workgroups_take_several_short_units(dev, hq, hkv, seqs, hi, dtype):
    """More short-context units than a graph's launch has workgroups, so each
    takes a second one in the same LDS; captured on a single sequence, replayed
    on batches of this size, a smaller one and this again, against the oracle
    and the bits of an eager plan (one unit per workgroup)."""
    blocks = seqs * (hi // 16 + 1) + 2
    plan, eager = (feattn.Plan(hq, hkv, 128, 16, seqs, hi // 16 + 3, dtype == "bf16", blocks) for _ in range(2))
    one = W.make_batch(hq, hkv, starts=[20], qlens=[1], seed=1, pool=blocks)
    plan.prepare(one.qo, one.kv, one.pages, one.last, one.batch, one.rows, graph=True)
    q, kc, vc = W.make_tensors(W.make_batch(hq, hkv, starts=[hi - 1] * seqs, qlens=[1] * seqs, seed=2, pool=blocks),
                               seed=3, dtype=dtype)
    qd, kd, vd = q.to(dev), kc.to(dev), vc.to(dev)
    out, lse = torch.zeros_like(qd), torch.zeros(seqs, hq, device=dev)
    graph = torch.cuda.CUDAGraph()
    torch.cuda.synchronize()
    with torch.cuda.graph(graph):
        plan.run(qd, kd, vd, out, causal=True, lse=lse)
    cus = torch.cuda.get_device_properties(dev).multi_processor_count
    for i, n in enumerate((seqs, 3, seqs, seqs)):
        b = W.make_batch(hq, hkv, starts=[(37 * s + 5 * i) % hi for s in range(n)], qlens=[1] * n, seed=4 + i,
                         pool=blocks)
        plan.prepare(b.qo, b.kv, b.pages, b.last, b.batch, b.rows, graph=True)
        eager.prepare(b.qo, b.kv, b.pages, b.last, b.batch, b.rows)
        units = plan.lists().short_units
        assert units == n * hkv and (n == 3 or units > cus * 8 // hkv)  # the launch: 8 wavefronts per CU
        out.fill_(float("nan"))
        lse.fill_(float("nan"))
        graph.replay()
        o2, l2 = torch.zeros_like(qd[:n]), torch.zeros_like(lse[:n])
        eager.run(qd, kd, vd, o2, causal=True, lse=l2)
        torch.cuda.synchronize()
        want, want_lse = A.run(b, q[:n], kc, vc, True)
        torch.testing.assert_close(o2.float().cpu(), want.float(), atol=1e-2, rtol=1e-2)
        torch.testing.assert_close(l2.cpu(), want_lse, atol=1e-3, rtol=0)
        assert torch.equal(out[:n], o2) and torch.equal(lse[:n], l2)
    plan.close()
    eager.close()
