"""Edges of the standalone operations' kernels: remainders of their vector
loads, unaligned bases, the shortest and longest rows of each variant."""

from __future__ import annotations

import numpy as np
import pytest

torch = pytest.importorskip("torch")

from rtxllm_amd import formats as F  # noqa: E402
from rtxllm_amd import ops, packs  # noqa: E402
from rtxllm_amd._lib import lib  # noqa: E402

pytestmark = pytest.mark.gpu

P = ops.ptr


def at_offset(a: np.ndarray, floats: int) -> torch.Tensor:
    """a on the GPU, `floats` 4-byte words past a 16-byte boundary."""
    big = torch.zeros(a.size + 8, dtype=torch.float32, device="cuda:0")
    view = big[floats:floats + a.size]
    view.copy_(torch.from_numpy(np.ascontiguousarray(a.reshape(-1))))
    assert view.data_ptr() % 16 == 4 * floats % 16
    return view


def row_slice(pack: packs.Pack, first: int, rows: int) -> packs.Pack:
    """Rows [first, first + rows) of a row-major pack as a pack of its own."""
    nb = pack.cols // 256

    def part(a, width):
        return np.ascontiguousarray(a.reshape(-1)[first * nb * width:(first + rows) * nb * width])

    return packs.Pack(pack.fmt, rows, pack.cols, part(pack.payload, F.PAYLOAD_BYTES[pack.fmt]),
                      None if pack.meta is None else part(pack.meta, F.META_BYTES[pack.fmt]))


def matvec_batch_f32(w: ops.DevicePack, x: torch.Tensor) -> np.ndarray:
    """rtxllm_matvec_batch_f32 of x [batch][cols]."""
    batch = x.shape[0]
    need = int(lib().rtxllm_matvec_batch_workspace(w.fmt, w.rows, w.cols))
    ws = torch.empty(max(need, 16), dtype=torch.uint8, device="cuda:0")
    y = torch.empty((batch, w.rows), dtype=torch.float32, device="cuda:0")
    assert lib().rtxllm_matvec_batch_f32(w.fmt, P(w.payload), P(w.meta), P(x), P(y), w.rows, w.cols, batch, P(ws), need,
                                         ops.stream()) == 0
    return y.cpu().numpy()


@pytest.mark.parametrize("n", [1, 2, 3, 4, 5, 7, 4095, 4096, 8191, 8192, 8193, 32767, 32773, 128259])
@pytest.mark.parametrize("offset", [0, 1, 3])
def test_argmax_edges(orc, n, offset):
    """Lowest index among equal maxima wherever they lie (head, vectors, tail),
    NaN never wins, nothing above -FLT_MAX gives 0, -0 equals +0."""
    base = packs.normal_f32(n, n)
    rows = [base]
    for where in ((0,), (n - 1,), (n // 2, n - 1), (0, n // 3, n - 1)):
        r = base.copy()
        r[list(where)] = np.float32(99.0)
        rows.append(r)
    nan = base.copy()
    nan[: n - 1] = np.nan
    rows.append(nan)
    rows.append(np.full(n, np.nan, np.float32))
    rows.append(np.full(n, -np.finfo(np.float32).max, np.float32))
    inf = np.full(n, -np.inf, np.float32)
    inf[n // 2] = np.inf
    rows.append(inf)
    zero = np.full(n, -1.0, np.float32)
    zero[n // 2:] = np.float32(0.0)
    zero[n // 3] = np.float32(-0.0)
    rows.append(zero)
    x = np.stack(rows)
    idx = torch.full((len(rows),), -1, dtype=torch.int32, device="cuda:0")
    xd = at_offset(x, offset)
    assert lib().rtxllm_argmax(P(xd), n, len(rows), P(idx), ops.stream()) == 0
    got = idx.cpu().numpy()
    for r in range(len(rows)):
        assert int(got[r]) == orc.argmax(x[r]), r
    tok = torch.full((1,), 7, dtype=torch.int32, device="cuda:0")
    assert lib().rtxllm_launch_output_token_sample(xd.data_ptr() + 4 * n, P(tok), n, 50000, 11, ops.stream()) == 0
    assert int(tok.cpu()[0]) == (orc.argmax(x[1]) + 11) % 50000


@pytest.mark.parametrize("fmt", sorted(F.PAYLOAD_BYTES), ids=lambda f: F.NAMES[f])
@pytest.mark.parametrize("rows,cols", [(1, 256), (3, 256), (5, 768), (7, 2304), (33, 4096), (8192, 256),
                                       (8195, 256), (2731, 768)])
def test_dequant_edges_bit_exact(orc, fmt, rows, cols):
    """Block counts around the small outputs' one block a wave and the large ones'
    four (from 8193 blocks on), and an output buffer off its 16-byte alignment;
    nothing past the end is written."""
    pack = packs.make_pack(fmt, rows, cols, seed=900 + fmt)
    d = ops.DevicePack(pack)
    n = rows * cols
    big = torch.full((n + 9,), 7.0, dtype=torch.float32, device="cuda:0")
    src = {F.IQ2S_UNITS: (F.IQ2S, packs.iq2s_from_units), F.IQ3S_UNITS: (F.IQ3S, packs.iq3s_from_units),
           F.Q4K_RAW_PREDECODED: (F.Q4K_RAW, lambda raw: raw)}.get(fmt)  # its pairs are d sc and dmin m, rounded once
    ofmt, payload = (fmt, pack.payload) if src is None else (src[0], src[1](pack.payload))
    ref = orc.dequant(ofmt, payload, pack.meta, rows, cols).reshape(-1)
    for off in (0, 1):
        big.fill_(7.0)
        assert lib().rtxllm_dequant_f32(fmt, P(d.payload), P(d.meta), rows, cols, big.data_ptr() + 4 * off,
                                        ops.stream()) == 0
        got = big.cpu().numpy()
        assert np.array_equal(got[off:off + n].view(np.uint32), ref.view(np.uint32)), off
        assert np.all(got[:off] == 7.0) and np.all(got[off + n:] == 7.0)


@pytest.mark.parametrize("n,count", [(1, 2), (6, 3), (124, 3), (128, 3), (256, 3), (1024, 1), (1028, 130), (4096, 127), (4096, 128),
                                     (4100, 2), (16384, 2), (16388, 2)])
@pytest.mark.parametrize("offset", [0, 2])
def test_rmsnorm_edges(n, count, offset):
    """Each variant (vector lengths, few and many vectors) and the unaligned
    fallback, with and without weights, in place, against float64: the fp32 sum
    of squares (tree) and three roundings give at most 2e-6 relative."""
    x = packs.normal_f32(n, n * count).reshape(count, n) * np.float32(2.0)
    w = packs.normal_f32(n + 1, n, mean=1.0, std=0.1)
    x64 = x.astype(np.float64)
    norm = x64 / np.sqrt((x64 * x64).mean(1, keepdims=True) + 1e-6)
    wd = at_offset(w, offset)
    for weight, ref in ((wd, norm * w), (None, norm)):
        xd = at_offset(x, offset)
        out = at_offset(np.zeros_like(x), offset)
        for dst in (out, xd):  # xd last: in place
            assert lib().rtxllm_rmsnorm_w(P(xd), P(weight), n, count, 1e-6, P(dst), ops.stream()) == 0
            np.testing.assert_allclose(dst.cpu().numpy().reshape(count, n), ref, rtol=2e-6)


@pytest.mark.parametrize("heads,head_dim,count", [(1, 2, 1), (3, 6, 2), (5, 128, 63), (9, 128, 64), (2, 96, 70),
                                                  (33, 64, 65), (1, 2048, 64), (1, 2050, 2), (2, 2050, 65),
                                                  (33, 128, 48), (33, 64, 130), (9, 512, 64), (5, 1026, 128)])
def test_rope_edges(heads, head_dim, count):
    """A thread per pair, shared angles with one and with four pairs a thread, the
    remainders of each, and heads with more angles than a workgroup has threads,
    against float64 rotation of the fp32 angle."""
    theta = 10000.0
    vec = packs.normal_f32(head_dim, count * heads * head_dim).reshape(count, heads, head_dim // 2, 2)
    pos = (np.arange(count, dtype=np.uint32) * 37 + 5).astype(np.uint32)
    freq = np.power(theta, -2.0 * np.arange(head_dim // 2) / head_dim).astype(np.float32)
    angle = (pos.astype(np.float32)[:, None] * freq).astype(np.float64)[:, None]
    c, s = np.cos(angle), np.sin(angle)
    e, o = vec[..., 0].astype(np.float64), vec[..., 1].astype(np.float64)
    ref = np.stack([e * c - o * s, e * s + o * c], -1)
    vd, pd = ops.to_dev(vec), ops.to_dev(pos)
    assert lib().rtxllm_rope_theta(P(vd), heads, head_dim, theta, P(pd), count, ops.stream()) == 0
    # rounded cos, sin and two products: a few 2^-24 of |(e, o)|; a freq that
    # rounds the other way moves the angle by its last bit (2^-23 of the angle)
    tol = 4e-7 * np.abs(vec).max() + 1.3e-7 * float(angle.max()) * np.abs(vec).max() * 0.01
    np.testing.assert_allclose(vd.cpu().numpy(), ref, rtol=0, atol=tol)


@pytest.mark.parametrize("cols", [256, 768, 1024, 1280])
def test_embed_gather_edges(orc, cols):
    """Row widths around the four blocks a workgroup holds, unaligned output."""
    vocab = 50
    table = packs.synth_raw(F.Q5K, vocab, cols, seed=77)
    tokens = np.array([49, 0, 50, 7], np.uint32)
    td, kd = ops.to_dev(table), ops.to_dev(tokens)
    big = torch.full((len(tokens) * cols + 8,), 7.0, dtype=torch.float32, device="cuda:0")
    assert lib().rtxllm_embed_gather_q5k(P(td), vocab, cols, P(kd), len(tokens), big.data_ptr() + 4, ops.stream()) == 0
    got = big.cpu().numpy()
    assert got[0] == 7.0 and np.all(got[1 + len(tokens) * cols:] == 7.0)
    got = got[1:1 + len(tokens) * cols].reshape(len(tokens), cols)
    for i, t in enumerate(tokens):
        ref = np.empty(cols, np.float32)
        if t >= vocab:
            assert np.all(np.isnan(got[i]))
            continue
        orc.lib().orc_embed_q5k(orc.ptr(table), cols, int(t), orc.ptr(ref))
        assert np.array_equal(got[i].view(np.uint32), ref.view(np.uint32)), t


@pytest.mark.parametrize("n", [1, 3, 4, 5, 1023, 1024, 1027, 4099])
@pytest.mark.parametrize("offset", [0, 1])
def test_silu_mul_edges(orc, n, offset):
    """The vector kernel's remainders, the unaligned fallback, and in place."""
    g, u = packs.normal_f32(n, n) * np.float32(4.0), packs.normal_f32(n + 1, n)
    ref = np.empty(n, np.float32)
    orc.lib().orc_silu_mul(orc.ptr(g), orc.ptr(u), n, orc.ptr(ref))
    gd, ud = at_offset(g, offset), at_offset(u, 0)
    assert lib().rtxllm_silu_mul(P(gd), P(ud), n, P(gd), ops.stream()) == 0
    np.testing.assert_allclose(gd.cpu().numpy(), ref, rtol=2e-6, atol=1e-30)


@pytest.mark.parametrize("fmt", [F.Q4K_RAW, F.Q4K_SPLIT_NATIVE, F.Q5K, F.IQ2S, F.IQ3S], ids=lambda f: F.NAMES[f])
@pytest.mark.parametrize("cols", [512, 2048, 3072, 4096])
def test_batch_single_tile_equals_many_tiles(fmt, cols):
    """The single-tile kernels (few rows, every tile resident; by format and panels
    also the ring over one tile) and the ring over many tiles give a row the same
    bits, staged and self-staging; rows % 16 != 0 in both."""
    rows, few, batch = 70001 if cols == 512 else 16393, 71, 5
    pack = packs.make_pack(fmt, rows, cols, seed=40 + fmt)
    xd = ops.to_dev(packs.normal_f32(9, batch * cols).reshape(batch, cols))
    x16 = ops.stage_batch(xd)
    many = ops.matvec_batch(ops.DevicePack(pack), x16, batch).cpu().numpy()
    # the first rows (round 0 of the first workgroups), some of a middle round and
    # the last ones with the ragged tile
    for first in (0, rows // 2, rows - few):
        w = ops.DevicePack(row_slice(pack, first, few))
        for one in (ops.matvec_batch(w, x16, batch).cpu().numpy(), matvec_batch_f32(w, xd)):
            assert np.array_equal(many[:, first:first + few].view(np.uint32), one.view(np.uint32)), first


@pytest.mark.parametrize("heads,n_kv", [(1, 1), (6, 3), (4, 1), (16, 2)])
@pytest.mark.parametrize("count", [1, 3])
def test_attention_fp32_queries_unaligned(orc, heads, n_kv, count):
    """Each group size with the workgroup's own staging of q (few kv heads, a short
    last chunk, a single position), q off its 16-byte alignment, and a capacity
    that is no multiple of the 128-position chunk."""
    hd, page, cap = 128, 16, 304
    pps = cap // page
    npages = count * pps
    positions = np.array([303, 0, 129][:count], np.uint32)
    table = np.array([(5 * i + 3) % npages for i in range(npages)], np.int32)
    assert len(set(table.tolist())) == npages
    k = packs.normal_f16_bits(81, npages * n_kv * page * hd)
    v = packs.normal_f16_bits(82, npages * n_kv * page * hd)
    q = packs.normal_f32(83, count * heads * hd)
    qd, kd, vd = at_offset(q, 1), ops.to_dev(k), ops.to_dev(v)
    td, pd = ops.to_dev(table), ops.to_dev(positions)
    need = int(lib().rtxllm_attn_decode_workspace(heads, n_kv, cap, count))
    ws = torch.empty(need, dtype=torch.uint8, device="cuda:0")
    out = torch.empty(count * heads * hd, dtype=torch.float32, device="cuda:0")
    assert lib().rtxllm_attn_decode_gqa_f16(P(qd), P(kd), P(vd), P(td), pps, heads, n_kv, page, cap, P(pd), count,
                                            P(out), P(ws), need, ops.stream()) == 0
    got = out.cpu().numpy().reshape(count, heads, hd).astype(np.float64)
    kf = k.view(np.float16).reshape(npages, n_kv, page, hd).astype(np.float64)
    vf = v.view(np.float16).reshape(npages, n_kv, page, hd).astype(np.float64)
    for r in range(count):
        rows = table[r * pps:(r + 1) * pps]
        n = int(positions[r]) + 1
        for h in range(heads):
            g = h // (heads // n_kv)
            ks, vs = (t[rows, g].reshape(cap, hd)[:n] for t in (kf, vf))
            s = ks @ (q.reshape(count, heads, hd)[r, h].astype(np.float64) / np.sqrt(128.0))
            p = np.exp(s - s.max())
            ref = (p / p.sum()) @ vs
            # q enters as an fp16 hi / lo pair (~22 bits); scores up to ~40
            np.testing.assert_allclose(got[r, h], ref, rtol=0, atol=1e-5 * np.abs(ref).max())


@pytest.mark.parametrize("rows,cols", [(1, 3), (3, 5), (4, 1024), (7, 1025), (4096, 100), (4099, 4097),
                                       (16384, 1000), (16387, 17000)])
@pytest.mark.parametrize("offset", [0, 3])
def test_rmsnorm_feedback_edges(rows, cols, offset):
    """Remainders of the vector loads and of their steps, unaligned logits, fewer
    and more columns than rows, against float64: the fp32 sum (tree), rsqrtf and
    two roundings give at most 2e-6 relative."""
    x = packs.normal_f32(rows, rows) * np.float32(3.0)
    x64 = x.astype(np.float64)
    ref = (x64 / np.sqrt((x64 * x64).mean() + 1e-6))[np.arange(cols) % rows]
    act = torch.empty(cols, dtype=torch.float32, device="cuda:0")
    xd = at_offset(x, offset)
    assert lib().rtxllm_launch_rmsnorm_feedback(P(xd), P(act), rows, cols, 1e-6, ops.stream()) == 0
    np.testing.assert_allclose(act.cpu().numpy(), ref, rtol=2e-6)


@pytest.mark.parametrize("fmt", [F.Q4K_SPLIT_NATIVE, F.Q4K_SPLIT_COMPACT, F.Q5K, F.IQ2S, F.IQ3S, F.IQ2S_UNITS,
                                 F.IQ3S_UNITS], ids=lambda f: F.NAMES[f])
@pytest.mark.parametrize("rows,cols", [(1, 256), (1023, 512), (1030, 1024), (2049, 2048), (2055, 2304), (4097, 4096),
                                       (8195, 4352), (2048, 8192), (2051, 8448), (4099, 8192), (70001, 256),
                                       (3001, 1024), (5401, 768), (17001, 512), (2055, 4608), (9301, 4608)])
def test_matvec_shared_staging_equals_staged_input(fmt, rows, cols):
    """One, two, four or eight row groups a workgroup share the staging of an fp32 x, or none
    do (widths, row counts and formats on both sides of the rule): always the
    bits of rtxllm_stage_activation + rtxllm_matvec_xq, x aligned or not, and a
    NaN or infinite value poisons as there."""
    pack = packs.make_pack(fmt, rows, cols, seed=300 + fmt)
    w = ops.DevicePack(pack)
    x = packs.normal_f32(cols, cols)
    x[16:32] = 0.0
    x[40] *= np.float32(1e4)
    for bad in (None, np.nan, np.inf):
        if bad is not None:
            x[cols - 5] = bad
        ref = ops.matvec_xq(w, ops.stage(ops.to_dev(x))).cpu().numpy()
        for off in (0, 1):
            y = torch.empty(rows, dtype=torch.float32, device="cuda:0")
            xd = at_offset(x, off)
            assert lib().rtxllm_matvec(fmt, P(w.payload), P(w.meta), P(xd), P(y), rows, cols, ops.stream()) == 0
            assert np.array_equal(y.cpu().numpy().view(np.uint32), ref.view(np.uint32)), (bad, off)


@pytest.mark.parametrize("fmt", [F.Q4K_RAW, F.Q4K_SPLIT_NATIVE, F.Q5K, F.IQ2S, F.IQ3S], ids=lambda f: F.NAMES[f])
@pytest.mark.parametrize("rows", [1, 100, 6001, 16393])
@pytest.mark.parametrize("wide", [3584, 4096, 8192])
def test_batch_weights_through_lds_equal_field_loads(fmt, rows, wide):
    """Workgroups of seven or eight panels copy their weights through LDS (or, by the
    rule, do not), smaller ones read fields: with x zero but for a window of 2048
    columns the wide matrix gives the bits of those columns alone. The windows
    cover every panel of the workgroup and, at 8192 columns, both panel groups.
    Rows of one tile, several, more tiles than CUs (376: single tiles, two a CU)
    and many rounds, the last tile ragged. Self-staging gives the same bits."""
    batch, part_cols = 3, 2048
    pack = packs.make_pack(fmt, rows, wide, seed=60 + fmt)
    w = ops.DevicePack(pack)
    pb, mb, nb = F.PAYLOAD_BYTES[fmt], F.META_BYTES.get(fmt, 0), wide // 256

    def part(a, width, first):
        return np.ascontiguousarray(a.reshape(rows, nb, width)[:, first // 256:(first + part_cols) // 256]).reshape(-1)

    for first in sorted({*range(0, wide - part_cols + 1, part_cols), wide - part_cols}):
        narrow = packs.Pack(fmt, rows, part_cols, part(pack.payload, pb, first),
                            None if pack.meta is None else part(pack.meta, mb, first))
        xs = packs.normal_f32(5, batch * part_cols).reshape(batch, part_cols)
        x = np.zeros((batch, wide), np.float32)
        x[:, first:first + part_cols] = xs
        xd = ops.to_dev(x)
        ref = ops.matvec_batch(ops.DevicePack(narrow), ops.stage_batch(ops.to_dev(xs)), batch).cpu().numpy()
        assert np.array_equal(ops.matvec_batch(w, ops.stage_batch(xd), batch).cpu().numpy(), ref), first
        assert np.array_equal(matvec_batch_f32(w, xd), ref), first


@pytest.mark.parametrize("fmt", [F.IQ2S, F.IQ3S], ids=lambda f: F.NAMES[f])
@pytest.mark.parametrize("rows", [71, 16393])
def test_batch_weights_through_lds_two_byte_payload(fmt, rows):
    """An IQ payload 2 bytes past a 16-byte boundary, the least its entry points
    take, gives the bits of the aligned one, staged and self-staging."""
    cols, batch = 4096, 3
    w = ops.DevicePack(packs.make_pack(fmt, rows, cols, seed=90 + fmt))
    xd = ops.to_dev(packs.normal_f32(6, batch * cols).reshape(batch, cols))
    ref = ops.matvec_batch(w, ops.stage_batch(xd), batch).cpu().numpy()
    big = torch.zeros(w.payload.numel() + 16, dtype=torch.uint8, device="cuda:0")
    moved = big[2:2 + w.payload.numel()]
    moved.copy_(w.payload.reshape(-1))
    w.payload = moved
    assert w.payload.data_ptr() % 16 == 2
    assert np.array_equal(ops.matvec_batch(w, ops.stage_batch(xd), batch).cpu().numpy(), ref)
    assert np.array_equal(matvec_batch_f32(w, xd), ref)


@pytest.mark.parametrize("rows,batch", [(1, 1), (3, 1), (5, 3), (64, 8), (1023, 7)])
@pytest.mark.parametrize("cols", [4608, 5632, 10240])
def test_batch_panel_groups_are_added(orc, rows, batch, cols):
    """Three, eleven and four panel groups (fewer and more than the reduction
    reads at once), rows x batch with every remainder of four."""
    pack = packs.make_pack(F.Q4K_SPLIT_NATIVE, rows, cols, seed=70)
    xs = packs.normal_f32(rows, batch * cols).reshape(batch, cols)
    y = ops.matvec_batch(ops.DevicePack(pack), ops.stage_batch(ops.to_dev(xs)), batch).cpu().numpy()
    for s in range(batch):
        ref = orc.matvec_f32(F.Q4K_SPLIT_NATIVE, pack.payload, pack.meta, xs[s], rows, cols, 8)
        # the fp32 sequential oracle's own error at these widths
        assert float(np.max(np.abs(y[s] - ref))) <= 1e-4 * float(np.max(np.abs(ref)))
    # x zero outside a group's columns leaves that group's partial alone: the bits
    # of y are those partials added in group order
    panels = cols // 512
    width = 512 * max(d for d in range(1, 9) if panels % d == 0)
    total = np.zeros_like(y)
    for first in range(0, cols, width):
        xg = np.zeros_like(xs)
        xg[:, first:first + width] = xs[:, first:first + width]
        total += ops.matvec_batch(ops.DevicePack(pack), ops.stage_batch(ops.to_dev(xg)), batch).cpu().numpy()
    assert np.array_equal(y, total)
