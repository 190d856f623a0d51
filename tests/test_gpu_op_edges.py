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
@pytest.mark.parametrize("rows,cols", [(1, 256), (3, 256), (5, 768), (7, 2304), (33, 4096)])
def test_dequant_edges_bit_exact(orc, fmt, rows, cols):
    """Block counts around the kernel's 4 blocks a wave and 16 a workgroup, and an
    output buffer off its 16-byte alignment; nothing past the end is written."""
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
