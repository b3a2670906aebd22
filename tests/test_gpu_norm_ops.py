"""GPU parity of the per-token operators (include/fe_ops.h) against
oracle/norm_ops.py: RMSNorm and the fused q/k RMSNorm + RoPE + paged append
bit-exact (and the fused call bit-identical to fe_norm + fe_rope + fe_store),
acceptance on the reference's matrix pattern (tests/gpu_ops_tests.cpp:55-79:
sentinels around the output, eager and HIP-graph replays), SiLU-gated product
within one rounding step of the 16-bit type."""

import numpy as np
import pytest
import torch

import feattn
from feattn import workloads as W
from oracle import norm_ops as N
from oracle import rope_store as R

pytestmark = pytest.mark.gpu


def u16(t):
    return t.detach().cpu().contiguous().view(torch.int16).numpy().view(np.uint16)


def dtype_of(bf16):
    return torch.bfloat16 if bf16 else torch.float16


@pytest.mark.parametrize("bf16", [True, False])
@pytest.mark.parametrize("width,residual", [(128, False), (128, True), (1000, False), (4096, True), (5120, False)])
def test_norm_bit_exact(dev, bf16, width, residual):
    dt = dtype_of(bf16)
    gen = torch.Generator().manual_seed(width + residual)
    rows = 37
    x = (torch.randn(rows, width, generator=gen) * 3).to(dt)
    r = torch.randn(rows, width, generator=gen).to(dt) if residual else None
    w = (1 + 0.1 * torch.randn(width, generator=gen)).to(dt)
    want, want_res = N.rms_norm(u16(x), u16(w), 1e-6, bf16, residual=u16(r) if residual else None)
    xd, wd = x.to(dev), w.to(dev)
    rd = r.to(dev) if residual else None
    out = torch.empty_like(xd)
    new_res = torch.empty_like(xd) if residual else None
    feattn.norm(xd, wd, out, rows, width, 1e-6, bf16, residual=rd, new_residual=new_res)
    torch.cuda.synchronize()
    assert np.array_equal(u16(out), want)
    if residual:
        assert np.array_equal(u16(new_res), want_res)
    # in place (output aliases x), as Net::forward's callers may do
    feattn.norm(xd, wd, xd, rows, width, 1e-6, bf16, residual=rd)
    torch.cuda.synchronize()
    assert np.array_equal(u16(xd), want)


@pytest.mark.parametrize("bf16", [True, False])
@pytest.mark.parametrize("width,offset", [(8, 0), (248, 0), (256, 0), (264, 0), (504, 0), (520, 0), (1024, 0),
                                          (1032, 0), (2048, 0), (3064, 0), (3840, 0), (4096, 0), (4104, 0), (5120, 0),
                                          (6144, 0), (8192, 0), (8200, 0), (1, 0), (257, 0), (1022, 0), (3001, 0),
                                          (6145, 0), (512, 1), (4096, 4)])
def test_norm_widths_and_alignments(dev, bf16, width, offset):
    """Bit-exact on both sides of every stripe, pair and register bound of the
    kernels, on widths that are no multiple of a load and on tensors that
    start `offset` elements past an aligned address; guard elements stay.  5
    rows take the block kernel, 515 (the same ones again and again) the
    wavefront-per-row kernel wherever it applies."""
    dt = dtype_of(bf16)
    gen = torch.Generator().manual_seed(3 * width + offset)
    rows, n, reps = 5, 5 * width, 103
    x = (torch.randn(rows, width, generator=gen) * 3).to(dt)
    r = torch.randn(rows, width, generator=gen).to(dt)
    w = (1 + 0.1 * torch.randn(width, generator=gen)).to(dt)

    def place(t):
        buf = torch.full((offset + t.numel() + 8,), 7.0, dtype=dt, device=dev)
        buf[offset:offset + t.numel()] = t.reshape(-1).to(dev)
        return buf, buf[offset:]

    for res in (None, r):
        want, want_res = N.rms_norm(u16(x), u16(w), 1e-6, bf16, residual=None if res is None else u16(res))
        (_, xd), (_, wd) = place(x), place(w)
        rd = None if res is None else place(res)[1]
        ob, out = place(torch.zeros(n))
        nb, new_res = place(torch.zeros(n))
        feattn.norm(xd, wd, out, rows, width, 1e-6, bf16, residual=rd, new_residual=new_res)
        torch.cuda.synchronize()
        assert np.array_equal(u16(out[:n]).reshape(rows, width), want)
        assert np.array_equal(u16(new_res[:n]).reshape(rows, width), want_res if res is not None else u16(x))
        for buf in (ob, nb):
            assert (buf[:offset] == 7.0).all() and (buf[offset + n:] == 7.0).all()
        many = rows * reps
        (_, xd) = place(x.repeat(reps, 1))
        rd = None if res is None else place(res.repeat(reps, 1))[1]
        ob, out = place(torch.zeros(n * reps))
        nb, new_res = place(torch.zeros(n * reps))
        feattn.norm(xd, wd, out, many, width, 1e-6, bf16, residual=rd, new_residual=None if res is None else new_res)
        torch.cuda.synchronize()
        got = u16(out[:n * reps]).reshape(reps, rows, width)
        assert np.array_equal(got, np.broadcast_to(want, got.shape))
        if res is not None:
            got = u16(new_res[:n * reps]).reshape(reps, rows, width)
            assert np.array_equal(got, np.broadcast_to(want_res, got.shape))
        for buf in (ob, nb):
            assert (buf[:offset] == 7.0).all() and (buf[offset + n * reps:] == 7.0).all()


@pytest.mark.parametrize("bf16", [True, False])
@pytest.mark.parametrize("rows,width", [(2051, 2048), (1031, 4096), (1031, 5120), (1031, 8192), (4099, 128 * 9)])
@pytest.mark.parametrize("residual", [True, False])
def test_norm_large_call_equals_small_calls(dev, bf16, rows, width, residual):
    """A call past the L2's size streams its tensors; every row's bits are
    those of the same rows in small calls (the last one, of an odd count).
    Then the large call in place, x and the residual overwritten."""
    rows = rows if residual else 2 * rows - 1
    assert rows * width * (8 if residual else 4) >= 32 << 20
    gen = torch.Generator(device=dev).manual_seed(5)
    x = (torch.randn(rows, width, generator=gen, device=dev) * 3).to(dtype_of(bf16))
    r = torch.randn(rows, width, generator=gen, device=dev).to(x.dtype) if residual else None
    w = (1 + 0.1 * torch.randn(width, generator=gen, device=dev)).to(x.dtype)
    out, part = torch.empty_like(x), torch.empty_like(x)
    new, part_new = (torch.empty_like(x), torch.empty_like(x)) if residual else (None, None)
    feattn.norm(x, w, out, rows, width, 1e-6, bf16, residual=r, new_residual=new)
    for i in range(0, rows, 300):
        n = min(300, rows - i)
        feattn.norm(x[i:], w, part[i:], n, width, 1e-6, bf16, residual=None if r is None else r[i:],
                    new_residual=None if new is None else part_new[i:])
    feattn.norm(x, w, x, rows, width, 1e-6, bf16, residual=r, new_residual=r)
    torch.cuda.synchronize()
    assert torch.equal(out.view(torch.int16), part.view(torch.int16))
    assert torch.equal(out.view(torch.int16), x.view(torch.int16))
    if residual:
        assert torch.equal(new.view(torch.int16), part_new.view(torch.int16))
        assert torch.equal(new.view(torch.int16), r.view(torch.int16))


@pytest.mark.parametrize("bf16", [True, False])
@pytest.mark.parametrize("width", [128, 4096, 5120, 8192])
def test_norm_in_place_many_rows(dev, bf16, width):
    """x and the residual overwritten by a call of more rows than the block
    kernel takes (and less than what streams): the oracle's bits."""
    gen = torch.Generator().manual_seed(width)
    rows, reps = 4, 130
    x = (torch.randn(rows, width, generator=gen) * 3).to(dtype_of(bf16))
    r = torch.randn(rows, width, generator=gen).to(x.dtype)
    w = (1 + 0.1 * torch.randn(width, generator=gen)).to(x.dtype)
    want, want_res = N.rms_norm(u16(x), u16(w), 1e-6, bf16, residual=u16(r))
    plain, _ = N.rms_norm(u16(x), u16(w), 1e-6, bf16, residual=None)
    xd, rd, yd = x.repeat(reps, 1).to(dev), r.repeat(reps, 1).to(dev), x.repeat(reps, 1).to(dev)
    feattn.norm(xd, w.to(dev), xd, rows * reps, width, 1e-6, bf16, residual=rd, new_residual=rd)
    feattn.norm(yd, w.to(dev), yd, rows * reps, width, 1e-6, bf16)
    torch.cuda.synchronize()
    for got, ref in ((xd, want), (rd, want_res), (yd, plain)):
        got = u16(got).reshape(reps, rows, width)
        assert np.array_equal(got, np.broadcast_to(ref, got.shape))


@pytest.mark.parametrize("bf16", [True, False])
@pytest.mark.parametrize("rows,width,residual", [(600, 9001, True), (1540, 9001, True), (1537, 9984, False),
                                                 (770, 12288, True), (769, 16384, False), (513, 16391, True),
                                                 (1030, 33 * 256, True)])
def test_norm_wide_rows(dev, bf16, rows, width, residual):
    """Rows of more stripes than the block kernel keeps, on both sides of the
    row counts where it keeps fewer; the same few rows again and again."""
    gen = torch.Generator().manual_seed(width)
    reps = -(-rows // 3)
    x = (torch.randn(3, width, generator=gen) * 3).to(dtype_of(bf16))
    r = torch.randn(3, width, generator=gen).to(x.dtype) if residual else None
    w = (1 + 0.1 * torch.randn(width, generator=gen)).to(x.dtype)
    want, want_res = N.rms_norm(u16(x), u16(w), 1e-6, bf16, residual=u16(r) if residual else None)
    xd = x.repeat(reps, 1)[:rows].to(dev)
    rd = r.repeat(reps, 1)[:rows].to(dev) if residual else None
    out, new = torch.empty_like(xd), torch.empty_like(xd) if residual else None
    feattn.norm(xd, w.to(dev), out, rows, width, 1e-6, bf16, residual=rd, new_residual=new)
    torch.cuda.synchronize()
    assert np.array_equal(u16(out), np.tile(want, (reps, 1))[:rows])
    if residual:
        assert np.array_equal(u16(new), np.tile(want_res, (reps, 1))[:rows])


def make_fused_case(bf16, rows, hq, hkv, row_stride, seed, cache_pages=64, max_pos=4096):
    dt = dtype_of(bf16)
    gen = torch.Generator().manual_seed(seed)
    buf = (torch.randn(rows * row_stride, generator=gen) * 2).to(dt)
    qw = (1 + 0.1 * torch.randn(128, generator=gen)).to(dt)
    kw = (1 + 0.1 * torch.randn(128, generator=gen)).to(dt)
    cache_slots = cache_pages * 16
    kc = torch.randn(cache_slots, hkv, 128, generator=gen).to(dt)
    vc = torch.randn(cache_slots, hkv, 128, generator=gen).to(dt)
    pos = torch.randint(0, max_pos, (rows,), generator=gen)
    pos[1] = -1
    pos[-1] = max_pos               # out of range: normalized, not rotated
    slots = torch.randperm(cache_slots, generator=gen)[:rows].clone()
    slots[2] = -1                   # padding row: no cache entry
    slots[3] = cache_slots          # out of range: skipped
    table = W.rope_table(max_pos, 1e6)
    return buf, qw, kw, kc, vc, pos, slots, table, cache_slots


@pytest.mark.parametrize("bf16", [True, False])
@pytest.mark.parametrize("rows,hq,hkv,extra", [(203, 32, 8, 0), (64, 16, 8, 0), (9, 40, 8, 64), (130, 32, 4, 0)])
def test_norm_rope_append_vs_oracle(dev, bf16, rows, hq, hkv, extra):
    row_stride = (hq + 2 * hkv) * 128 + extra
    buf, qw, kw, kc, vc, pos, slots, table, cs = make_fused_case(bf16, rows, hq, hkv, row_stride, rows + hq)
    wq, wkc, wvc = N.norm_rope_append(u16(buf), row_stride, u16(qw), u16(kw), 1e-6, u16(kc), u16(vc), pos.numpy(),
                                      slots.numpy(), table.numpy(), rows, hq, hkv, bf16, 4096, cs)
    q_out = torch.empty(rows, hq, 128, dtype=buf.dtype, device=dev)
    kcd, vcd = kc.to(dev), vc.to(dev)
    feattn.norm_rope_append(buf.to(dev), row_stride, qw.to(dev), kw.to(dev), 1e-6, q_out, kcd, vcd, pos.to(dev),
                            slots.to(dev), table.to(dev), rows, hq, hkv, bf16, 4096, cs)
    torch.cuda.synchronize()
    assert np.array_equal(u16(q_out), wq)
    assert np.array_equal(u16(kcd).reshape(cs, -1), wkc)      # untouched slots included
    assert np.array_equal(u16(vcd).reshape(cs, -1), wvc)


def test_norm_rope_append_special_values(dev):
    """bf16 projection rows holding NaNs (several payloads), infinities,
    the largest finite values and subnormals: every head, rotated or not,
    matches the oracle bit for bit (a NaN or infinity poisons its head's
    sum of squares; NaN results round to 0x7fc0)."""
    rows, hq, hkv = 47, 32, 8
    row_stride = (hq + 2 * hkv) * 128
    buf, qw, kw, kc, vc, pos, slots, table, cs = make_fused_case(True, rows, hq, hkv, row_stride, 11)
    specials = [0x7FC0, 0x7FC1, 0x7F81, 0xFFC0, 0x7FFF, 0x7F80, 0xFF80, 0x7F7F, 0xFF7F, 0x0001, 0x8001]
    flat = buf.view(torch.int16)
    gen = torch.Generator().manual_seed(12)
    for j, i in enumerate(torch.randperm(flat.numel(), generator=gen)[:6 * len(specials)].tolist()):
        flat[i] = np.int16(np.uint16(specials[j % len(specials)]))
    with np.errstate(all="ignore"):  # NaN and infinity arithmetic is the point here
        wq, wkc, wvc = N.norm_rope_append(u16(buf), row_stride, u16(qw), u16(kw), 1e-6, u16(kc), u16(vc),
                                          pos.numpy(), slots.numpy(), table.numpy(), rows, hq, hkv, True, 4096, cs)
    q_out = torch.empty(rows, hq, 128, dtype=buf.dtype, device=dev)
    kcd, vcd = kc.to(dev), vc.to(dev)
    feattn.norm_rope_append(buf.to(dev), row_stride, qw.to(dev), kw.to(dev), 1e-6, q_out, kcd, vcd, pos.to(dev),
                            slots.to(dev), table.to(dev), rows, hq, hkv, True, 4096, cs)
    torch.cuda.synchronize()
    assert (wq == 0x7FC0).any()  # the NaN path is exercised
    assert np.array_equal(u16(q_out), wq)
    assert np.array_equal(u16(kcd).reshape(cs, -1), wkc)
    assert np.array_equal(u16(vcd).reshape(cs, -1), wvc)


@pytest.mark.parametrize("bf16", [True, False])
def test_norm_rope_append_equals_unfused_sequence(dev, bf16):
    """Bit-identical to src/cuda_model.cpp:91-95 run as separate calls:
    norm(q), norm(k), rope(q, k), store(k, v)."""
    rows, hq, hkv = 150, 32, 8
    row_stride = (hq + 2 * hkv) * 128
    buf, qw, kw, kc, vc, pos, slots, table, cs = make_fused_case(bf16, rows, hq, hkv, row_stride, 7)
    b2 = buf.view(rows, hq + 2 * hkv, 128).to(dev)
    qwd, kwd, tabd, posd, slotsd = qw.to(dev), kw.to(dev), table.to(dev), pos.to(dev), slots.to(dev)
    q = torch.empty(rows, hq, 128, dtype=buf.dtype, device=dev)
    k = torch.empty(rows, hkv, 128, dtype=buf.dtype, device=dev)
    feattn.norm(b2[:, :hq].contiguous(), qwd, q, rows * hq, 128, 1e-6, bf16)
    feattn.norm(b2[:, hq:hq + hkv].contiguous(), kwd, k, rows * hkv, 128, 1e-6, bf16)
    feattn.rope(q, k, posd, tabd, rows, hq, hkv, 128, bf16, 4096)
    kc1, vc1 = kc.to(dev), vc.to(dev)
    feattn.store(k, b2[:, hq + hkv:].contiguous(), kc1, vc1, slotsd, rows, hkv * 128, bf16, cs)
    q2 = torch.empty_like(q)
    kc2, vc2 = kc.to(dev), vc.to(dev)
    feattn.norm_rope_append(buf.to(dev), row_stride, qwd, kwd, 1e-6, q2, kc2, vc2, posd, slotsd, tabd, rows, hq,
                            hkv, bf16, 4096, cs)
    torch.cuda.synchronize()
    assert torch.equal(q.view(torch.int16), q2.view(torch.int16))
    assert torch.equal(kc1.view(torch.int16), kc2.view(torch.int16))
    assert torch.equal(vc1.view(torch.int16), vc2.view(torch.int16))


@pytest.mark.parametrize("bf16", [True, False])
def test_draft_context_projection_layout(dev, bf16):
    """Net::project (src/cuda_model.cpp:102-107): per layer, k and v of a
    [rows][layers][2][hkv][128] projection; hq = 0, row stride over layers."""
    rows, layers, hkv = 48, 3, 8
    row_stride = layers * 2 * hkv * 128
    buf, _, kw, kc, vc, pos, slots, table, cs = make_fused_case(bf16, rows, 0, hkv, row_stride, 9)
    for lid in range(layers):
        off = lid * 2 * hkv * 128
        _, wkc, wvc = N.norm_rope_append(u16(buf)[off:], row_stride, None, u16(kw), 1e-6, u16(kc), u16(vc),
                                         pos.numpy(), slots.numpy(), table.numpy(), rows, 0, hkv, bf16, 4096, cs)
        kcd, vcd = kc.to(dev), vc.to(dev)
        feattn.norm_rope_append(buf.to(dev)[off:], row_stride, None, kw.to(dev), 1e-6, None, kcd, vcd, pos.to(dev),
                                slots.to(dev), table.to(dev), rows, 0, hkv, bf16, 4096, cs)
        torch.cuda.synchronize()
        assert np.array_equal(u16(kcd).reshape(cs, -1), wkc)
        assert np.array_equal(u16(vcd).reshape(cs, -1), wvc)


def test_accept_matrix_eager_and_graph(dev):
    """tests/gpu_ops_tests.cpp:55-79: draft = verify = 10 + j except
    verify[accepted] = 99 with accepted = (first + b) % (k + 1); 8 sentinel
    words on each side of the output stay untouched; the same launch replayed
    from a captured graph sees the new inputs."""
    checks = replays = 0
    for batch in (1, 2, 4, 8):
        for k in range(1, 16):
            draft = torch.zeros(batch, k, dtype=torch.int64, device=dev)
            verify = torch.zeros(batch, k + 1, dtype=torch.int64, device=dev)
            output = torch.full((batch * (k + 2) + 16,), -999, dtype=torch.int64, device=dev)
            run = lambda: feattn.accept(draft, verify, output[8:], batch, k)
            run()
            torch.cuda.synchronize()
            graph = torch.cuda.CUDAGraph()
            with torch.cuda.graph(graph):
                run()
            for first in range(k + 1):
                acc = [(first + b) % (k + 1) for b in range(batch)]
                d = np.tile(10 + np.arange(k), (batch, 1))
                v = np.tile(10 + np.arange(k + 1), (batch, 1))
                for b in range(batch):
                    v[b, acc[b]] = 99
                draft.copy_(torch.from_numpy(d))
                verify.copy_(torch.from_numpy(v))
                want = N.accept(d, v).reshape(-1)
                for captured in (False, True):
                    output.fill_(-999)
                    if captured:
                        graph.replay()
                        replays += 1
                    else:
                        run()
                    ids = output.cpu().numpy()
                    assert (ids[:8] == -999).all() and (ids[8 + batch * (k + 2):] == -999).all()
                    assert np.array_equal(ids[8:8 + batch * (k + 2)], want)
                    for b in range(batch):
                        row = ids[8 + b * (k + 2):8 + (b + 1) * (k + 2)]
                        assert row[k + 1] == acc[b] + 1 and row[acc[b]] == 99
                        assert row[:acc[b]].tolist() == list(range(10, 10 + acc[b]))
                        checks += 1
            del graph
    assert checks == 2 * sum(b * (k + 1) for b in (1, 2, 4, 8) for k in range(1, 16)) and replays > 0


@pytest.mark.parametrize("bf16", [True, False])
def test_silu_mul_within_one_step(dev, bf16):
    dt = dtype_of(bf16)
    gen = torch.Generator().manual_seed(4)
    rows, width = 77, 1536
    gu = (torch.randn(rows, 2 * width, generator=gen) * 4).to(dt)
    want = N.silu_mul(u16(gu), bf16)
    out = torch.empty(rows, width, dtype=dt, device=dev)
    feattn.silu_mul(gu.to(dev), out, rows, width, bf16)
    torch.cuda.synchronize()
    got = u16(out)
    a = R.to_f32(got, bf16).astype(np.float64)
    b = R.to_f32(want, bf16).astype(np.float64)
    step = np.maximum(np.abs(a), np.abs(b)) * (2.0 ** -7 if bf16 else 2.0 ** -10) + (0 if bf16 else 2.0 ** -24)
    assert (np.abs(a - b) <= step).all()
    assert np.mean(got == want) > 0.99


def silu_close(got, want, bf16):
    """One rounding step of the 16-bit type; NaN for NaN, infinities and every
    sign (of zeros and of results that underflow too) equal."""
    a, b = R.to_f32(got, bf16).astype(np.float64), R.to_f32(want, bf16).astype(np.float64)
    assert np.array_equal(np.isnan(a), np.isnan(b))
    if bf16:
        assert (got[np.isnan(a)] == 0x7FC0).all()
    inf = np.isinf(a) | np.isinf(b)
    assert np.array_equal(a[inf], b[inf])
    ok = ~(np.isnan(a) | inf)
    assert np.array_equal(np.signbit(a[~np.isnan(a)]), np.signbit(b[~np.isnan(b)]))
    # a result below 2^-126 has float32's own absolute spacing behind it
    step = np.maximum(np.abs(a), np.abs(b))[ok] * (2.0 ** -7 if bf16 else 2.0 ** -10) + (2.0 ** -133 if bf16
                                                                                        else 2.0 ** -24)
    assert (np.abs(a[ok] - b[ok]) <= step).all()


@pytest.mark.parametrize("bf16", [True, False])
@pytest.mark.parametrize("width,offset", [(65536, 0), (65536, 1), (8, 0), (24, 0), (1, 0), (1001, 0), (2056, 8)])
def test_silu_mul_all_gates(dev, bf16, width, offset):
    """Every 16-bit gate (NaNs, infinities, subnormals, both ends of the
    exponential) in rows of widths around the vector kernel's chunk, and on
    tensors `offset` elements past an aligned address."""
    dt = dtype_of(bf16)
    rows = max(1, 65536 // width)
    gen = torch.Generator().manual_seed(width + offset)
    x = torch.randperm(65536, generator=gen)[:rows * width].to(torch.int32).to(torch.int16).view(dt)
    if width == 1:
        x = torch.arange(65536, dtype=torch.int32).to(torch.int16).view(dt)
    up = torch.randn(rows, width, generator=gen).to(dt)
    gu = torch.cat([x.reshape(rows, width), up], 1)
    with np.errstate(all="ignore"):
        want = N.silu_mul(u16(gu), bf16)
    buf = torch.zeros(offset + gu.numel(), dtype=dt, device=dev)
    buf[offset:] = gu.reshape(-1).to(dev)
    ob = torch.full((offset + rows * width + 8,), 7.0, dtype=dt, device=dev)
    feattn.silu_mul(buf[offset:], ob[offset:], rows, width, bf16)
    torch.cuda.synchronize()
    silu_close(u16(ob[offset:offset + rows * width]).reshape(rows, width), want, bf16)
    assert (ob[:offset] == 7.0).all() and (ob[offset + rows * width:] == 7.0).all()


def test_silu_mul_large_call_equals_small_calls(dev):
    """A call past the L2's size streams its tensors: the bits of the same
    rows in small calls."""
    rows, width = 1031, 6144
    gen = torch.Generator(device=dev).manual_seed(9)
    gu = (torch.randn(rows, 2 * width, generator=gen, device=dev) * 4).bfloat16()
    out, part = (torch.empty(rows, width, device=dev, dtype=torch.bfloat16) for _ in range(2))
    feattn.silu_mul(gu, out, rows, width, True)
    for i in range(0, rows, 100):
        feattn.silu_mul(gu[i:], part[i:], min(100, rows - i), width, True)
    torch.cuda.synchronize()
    assert torch.equal(out.view(torch.int16), part.view(torch.int16))
