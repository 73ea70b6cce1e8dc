"""The gradients of the bias tables from several gradients of one bias (tgt_graph_attn_bias_bwd_sum), against sums in 64 bits.

bfloat16 gradients of eight heads take the matrix cores in chunks of 120 positions: planes of one chunk and less, of odd and even size, ids
with and without a row of the products, padding, gradients that are no numbers."""
import ctypes

import pytest
import torch

from torchgt_amd import _lib

pytestmark = pytest.mark.gpu


def _reference(douts, sp, et, n_sp, n_e):
    """(spatial, edge, virtual) and the sums of magnitudes behind them"""
    res = []
    for d in (sum(d.double() for d in douts), sum(d.double().abs() for d in douts)):
        inner = d[:, :, 1:, 1:].permute(0, 2, 3, 1).reshape(-1, d.shape[1])
        tables = []
        for ids, n in ((sp, n_sp), (et, n_e)):
            t = torch.zeros(n, d.shape[1], dtype=torch.float64)
            for i in range(1, n):                      # (row by row: no number stays in the rows that look it up)
                t[i] = inner[ids.reshape(-1) == i].sum(0)
            tables.append(t)
        res.append((*tables, d[:, :, 0, :].sum((0, 2)) + d[:, :, 1:, 0].sum((0, 2))))
    return res


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("b,s,n_douts,heads,n_sp,n_e,odd_number", [
    (3, 9, 1, 8, 30, 12, None),       # a plane of 100: less than a chunk
    (3, 10, 2, 8, 30, 12, None),      # 121: one chunk and one position
    (2, 11, 1, 8, 6, 3, None),        # 144, tables of fewer ids than rows
    (5, 16, 3, 8, 40, 64, None),
    (1, 40, 4, 8, 512, 20, None),
    (7, 37, 2, 4, 30, 12, None),      # four heads
    (4, 33, 3, 8, 40, 64, "inf"),
    (4, 33, 1, 8, 40, 64, "nan"),
    (150, 31, 3, 8, 40, 64, None),    # several chunks a wave
])
def test_gradients_of_the_tables(cuda, b, s, n_douts, heads, n_sp, n_e, odd_number, dtype):
    g = torch.Generator().manual_seed(b * 1000 + s)
    sizes = torch.randint(2, s + 1, (b,), generator=g)
    sizes[0] = s
    valid = torch.arange(s)[None, :] < sizes[:, None]
    pairs = valid[:, :, None] & valid[:, None, :]
    sp = torch.where(torch.rand(b, s, s, generator=g) < 0.9, torch.randint(1, min(7, n_sp), (b, s, s), generator=g), torch.randint(1, n_sp, (b, s, s), generator=g)) * pairs
    et = torch.randint(0, n_e, (b, s, s), generator=g) * (torch.rand(b, s, s, generator=g) < 0.2) * pairs
    douts = [torch.randn(b, heads, s + 1, s + 1, generator=g).to(dtype) for _ in range(n_douts)]
    if odd_number:
        douts[-1][1, 2, 4, 5] = float(odd_number)
        sp[1, 3, 4], et[1, 3, 4] = 3, 2
    dev = [d.to(cuda) for d in douts]
    dsp, det = sp.to(cuda), et.to(cuda)
    L = _lib.lib()
    ws = torch.empty(L.tgt_graph_attn_bias_bwd_workspace_bytes(n_sp, n_e, heads), dtype=torch.uint8, device=cuda)
    out = [torch.full((n, heads), 7.0, dtype=dtype, device=cuda) for n in (n_sp, n_e, 1)]
    ptrs = (ctypes.c_void_p * 4)(*[d.data_ptr() for d in dev])
    _lib.check(L.tgt_graph_attn_bias_bwd_sum(ptrs, n_douts, dsp.data_ptr(), det.data_ptr(), 1, n_sp, n_e, b, s, heads, _lib.DTYPE_BF16 if dtype == torch.bfloat16 else _lib.DTYPE_F32,
                                             out[0].data_ptr(), out[1].data_ptr(), out[2].data_ptr(), ws.data_ptr(), ws.numel(), torch.cuda.current_stream().cuda_stream))
    want, size = _reference(douts, sp, et, n_sp, n_e)
    for name, o, w, m in zip(("spatial", "edge", "virtual"), out, want, size):
        o, w, m = o.double().cpu(), w.reshape(o.shape), m.reshape(o.shape)
        fine = torch.isfinite(w)
        assert torch.equal(torch.isfinite(o), fine), name
        assert torch.equal(torch.isnan(o), torch.isnan(w)), name
        # float sums: every partial sum within 2^-24 of itself, chains of a few hundred at the most; then the result's own rounding
        tol = 400 * 2.0 ** -24 * m + (2.0 ** -8 if dtype == torch.bfloat16 else 2.0 ** -23) * w.abs()
        assert bool(((o - w).abs() <= tol)[fine].all()), f"{name} {float(((o - w).abs() - tol)[fine].max())}"
