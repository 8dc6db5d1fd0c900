"""Parity of the packed-row rel-pos kernel (attn_relpos_rows.hip, f16 / bf16 grids of any width at hd 64 and
80) with the CPU oracle, on an MI355X, at the sizes where its tiling can go wrong."""
import numpy as np
import pytest
import torch

import sam_oracle as oracle
from parity import check, to_dev
from test_attn_relpos_gpu import hip, make_inputs, run_gpu  # noqa: F401

pytestmark = pytest.mark.gpu

# Every chunk count per row (1..8) with full, one-column and odd last chunks; grids of less than a tile and
# of one token; tiles that end inside a row and exactly on one; 128 and 129 tokens (the line between one
# wave group and two) and odd row counts, whose halves differ; heights up to 64; and bh that gives one group
# of 256 queries (300 heads of 9 x 17) and two.
GRIDS = [(1, 1, 2), (1, 7, 2), (3, 5, 2), (8, 8, 2), (16, 8, 2), (43, 3, 2), (64, 1, 2), (9, 9, 2), (13, 13, 2),
         (64, 16, 1), (5, 17, 2), (9, 17, 300), (16, 24, 2), (5, 25, 3), (10, 32, 2), (11, 33, 2), (24, 40, 1),
         (7, 41, 2), (8, 48, 2), (9, 49, 2), (37, 50, 2), (8, 56, 2), (5, 57, 2), (3, 63, 2)]


@pytest.mark.parametrize("dtype", ["f16", "bf16"])
@pytest.mark.parametrize("hd", [64, 80])
@pytest.mark.parametrize("h,w,bh", GRIDS)
def test_packed_rows_match_oracle(hip, h, w, bh, hd, dtype):  # noqa: F811
    print(f"packed rows {dtype} {h}x{w} bh={bh} hd={hd}", flush=True)
    arrays = make_inputs(h, w, bh, hd, 700 + 64 * h + w + hd, dtype, table_std=0.5)
    scale = hd ** -0.5
    got = run_gpu(hip, arrays, h, w, scale, dtype)
    heads = [0, bh - 1]
    q, kt, v, table = arrays
    want = oracle.attention_relpos(q[heads], kt[heads], v[heads], table, h, w, scale)
    check(got[heads], want, dtype, f"packed rows {h}x{w} hd={hd} {dtype}")


@pytest.mark.parametrize("h,w", [(9, 13), (11, 33)])
def test_packed_rows_keep_a_head_to_itself(hip, h, w):  # noqa: F811
    """kT is read in 16-byte pieces that pass the end of a row; NaN keys and values in one head must not
    reach its neighbours."""
    bh, hd = 3, 64
    q, kt, v, table = make_inputs(h, w, bh, hd, 5, "f16")
    clean = run_gpu(hip, [q, kt, v, table], h, w, hd ** -0.5, "f16")
    kt[1], v[1] = float("nan"), float("nan")
    got = run_gpu(hip, [q, kt, v, table], h, w, hd ** -0.5, "f16")
    assert (got[[0, 2]] == clean[[0, 2]]).all()
    assert torch.from_numpy(got[1]).isnan().all()


# Grids of 1 to 3 columns, where a chunk of 8 spans several rows and the loads of more than the last row's tile
# reach the head's end: one wave group (up to 128 tokens; 300 heads), and two.
NARROW = [(9, 1, 3), (12, 1, 3), (10, 2, 3), (9, 3, 3), (17, 3, 3), (49, 3, 3), (51, 3, 3), (51, 3, 300)]


@pytest.mark.parametrize("dtype", ["f16", "bf16"])
@pytest.mark.parametrize("hd", [64, 80])
@pytest.mark.parametrize("h,w,bh", NARROW)
def test_narrow_grids_read_nothing_past_a_head(hip, h, w, bh, hd, dtype):  # noqa: F811
    """NaN keys and values in one head, and past the last one, must not reach any other head."""
    print(f"narrow {dtype} {h}x{w} bh={bh} hd={hd}", flush=True)
    arrays = make_inputs(h, w, bh, hd, 40 + h + w + hd, dtype, table_std=0.5)
    q, kt, v, table = (to_dev(a, dtype) for a in arrays)

    def tailed(x):
        buf = torch.full((x.numel() + 4096,), float("nan"), device="cuda", dtype=x.dtype)
        buf[: x.numel()].copy_(x.reshape(-1))
        return buf[: x.numel()].view(x.shape)

    kt, v = tailed(kt), tailed(v)
    clean = hip.attention_relpos(q, kt, v, table, h, w, hd ** -0.5).float().cpu().numpy()
    heads = [0, bh - 1]
    want = oracle.attention_relpos(*(a[heads] for a in arrays[:3]), arrays[3], h, w, hd ** -0.5)
    check(clean[heads], want, dtype, f"narrow {h}x{w} hd={hd} {dtype}")
    kt[1], v[1] = float("nan"), float("nan")
    got = hip.attention_relpos(q, kt, v, table, h, w, hd ** -0.5).float().cpu().numpy()
    rest = [b for b in range(bh) if b != 1]
    assert (got[rest] == clean[rest]).all()
    assert torch.from_numpy(got[1]).isnan().all()


@pytest.mark.parametrize("dtype", ["f16", "bf16"])
@pytest.mark.parametrize("hd", [64, 80])
@pytest.mark.parametrize("h,w,rows", [(11, 33, (6, 8)), (11, 33, (0, 2)), (9, 13, (0, 4)), (51, 3, (26, 34))])
def test_tiles_of_infinite_keys(hip, h, w, rows, hd, dtype):  # noqa: F811
    """Infinite keys that fill the first tile of a wave group (the second's, the first's, a lone one's) give a
    query scores of -inf, weight 0, or of +inf, a NaN row, by the sign of its q."""
    bh, dim = 2, 5
    print(f"infinite keys {dtype} {h}x{w} rows {rows} hd={hd}", flush=True)
    q, kt, v, table = make_inputs(h, w, bh, hd, 8, dtype)
    keys = slice(rows[0] * w, rows[1] * w)
    kt[0, dim, keys] = np.inf
    got = run_gpu(hip, [q, kt, v, table], h, w, hd ** -0.5, dtype)
    masked = q[0, :, dim] < 0
    assert masked.any() and not masked.all()
    assert np.isnan(got[0][~masked]).all()
    kt[0, dim, keys] = 0
    i, j = np.divmod(np.arange(h * w), w)
    q64, t = q[0].astype(np.float64), table.astype(np.float64)
    bias = np.einsum("nd,nkd->nk", q64, t[i[:, None] - i[None] + h - 1] + t[2 * h - 1 + j[:, None] - j[None] + w - 1])
    logits = q64 @ kt[0].astype(np.float64) * hd ** -0.5 + bias
    logits[:, keys] = -np.inf
    p = np.exp(logits - logits.max(1, keepdims=True))
    want = (p / p.sum(1, keepdims=True)) @ v[0].astype(np.float64)
    check(got[0][masked], want[masked].astype(np.float32), dtype, f"infinite keys {h}x{w} hd={hd} {dtype}")


@pytest.mark.parametrize("dtype", ["f16", "bf16"])
@pytest.mark.parametrize("h,w,bh", [(10, 26, 140), (39, 32, 60), (40, 32, 60), (9, 60, 90)])
def test_even_widths_past_a_round(hip, h, w, bh, dtype):  # noqa: F811
    """Even widths of 25..32 and 57..64 at hd 64 past one round of workgroups, on both sides of the line between
    this kernel and the general one (39 rows are the last whose scratch lets two workgroups share a CU)."""
    print(f"even widths {dtype} {h}x{w} bh={bh}", flush=True)
    q, kt, v, table = make_inputs(h, w, bh, 64, 60 + h, dtype, table_std=0.5)
    got = run_gpu(hip, [q, kt, v, table], h, w, 0.125, dtype)
    heads = [0, bh // 2, bh - 1]
    want = oracle.attention_relpos(q[heads], kt[heads], v[heads], table, h, w, 0.125)
    check(got[heads], want, dtype, f"even widths {h}x{w} {dtype}")
