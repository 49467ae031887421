"""The 256 x 256 tile of the bfloat16 product (cq_dense.hip) at its edges, against float64 products of the rounded operands.

Bound: the products of bfloat16 operands are exact in f32; a sum of k of them in f32, k / 16 at a time, rounds k / 16 times (and within the matrix
instruction): below 2^-24 * sqrt(k / 16) * 4 = 4e-6 of the norm for k = 4160.
"""
import ctypes

import pytest
import torch

from candle_amd._lib import DenseArgs
from candle_amd import _lib

pytestmark = pytest.mark.gpu
BOUND = 4e-6


@pytest.mark.parametrize("x_bf16", [0, 1])
@pytest.mark.parametrize("m,n,k,pad", [(257, 20475, 1024, 0), (2300, 4610, 1088, 64), (2048, 5120, 4160, 0), (255, 40964, 1024, 128)])
@pytest.mark.parametrize("form", ["plain", "add", "swiglu", "bf16", "rows"])
def test_edges(m, n, k, pad, x_bf16, form):
    print(f"case {m} {n} {k} {pad} {x_bf16} {form}", flush=True)
    if form == "swiglu":
        n &= ~1
    g = torch.Generator(device="cuda").manual_seed(m + n + k)
    w = torch.randn((n, k + pad), generator=g, device="cuda").mul_(0.02).bfloat16()
    x = torch.randn((m, k + pad), generator=g, device="cuda")
    xd = x.bfloat16() if x_bf16 else x
    cols = n // 2 if form == "swiglu" else n
    y = torch.full((m + 2, cols + 3), 5.0, device="cuda", dtype=torch.bfloat16 if form == "bf16" else torch.float32)
    add = torch.randn((m, n), generator=g, device="cuda") if form == "add" else None
    perm = torch.randperm(m, generator=g, device="cuda").int() if form == "rows" else None
    a = DenseArgs(w_dev=w.data_ptr(), ldw=k + pad, x_dev=xd.data_ptr(), ldx=k + pad, x_bf16=x_bf16, dst_dev=y[1].data_ptr(), ldd=cols + 3, m=m, n=n, k=k, batch=1,
                  dst_bf16=int(form == "bf16"), act=2 if form == "swiglu" else 0, add_dev=add.data_ptr() if form == "add" else None, ld_add=n if form == "add" else 0,
                  dst_rows_dev=perm.data_ptr() if form == "rows" else None)
    L = _lib.mixer_lib()
    assert L.cq_dense_matmul_workspace_bytes(0, m, n, k) == 0
    _lib.check("cq_dense_product", L.cq_dense_product(0, ctypes.byref(a), None, 0, ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)))
    torch.cuda.synchronize()
    want = x[:, :k].bfloat16().double() @ w[:, :k].double().t()
    size = want.norm(dim=1, keepdim=True)
    if form == "add":
        want += add
    if form == "swiglu":
        want = torch.nn.functional.silu(want[:, 0::2]) * want[:, 1::2]
    got = y[1:m + 1, :cols].double()
    if form == "rows":
        got = got[perm.long()]
    err = (got - want).abs()
    if form == "bf16":
        err = (err - want.abs() * 2.0 ** -8).clamp(min=0)
    assert float((err.norm(dim=1, keepdim=True) / size).max()) <= BOUND * (4 if form == "swiglu" else 1)      # (silu and the gate: slopes up to 1.1, values to 4)
    assert (y[0] == 5).all() and (y[m + 1] == 5).all() and (y[:, cols:] == 5).all()


@pytest.mark.parametrize("k", [512, 768, 832, 896, 960])
@pytest.mark.parametrize("splits", [False, True])
def test_stages_on_their_way(k, splits):
    """The 128 x 128 tile of bfloat16 rows: up to 12 stages of k a workgroup with one of them on its way, beyond with three; all remainders of three."""
    m, n = (2000, 3201) if not splits else (700, 1157)
    k = k if not splits else 9 * k                         # 60 tiles: nine splits
    g = torch.Generator(device="cuda").manual_seed(k)
    w = torch.randn((n, k), generator=g, device="cuda").mul_(0.02).bfloat16()
    x = torch.randn((m, k), generator=g, device="cuda").bfloat16()
    y = torch.full((m + 2, n + 3), 5.0, device="cuda")
    L = _lib.mixer_lib()
    nb = L.cq_dense_matmul_workspace_bytes(0, m, n, k)
    assert (nb > 0) == splits
    ws = torch.empty(max(nb, 16), dtype=torch.uint8, device="cuda")
    a = DenseArgs(w_dev=w.data_ptr(), ldw=k, x_dev=x.data_ptr(), ldx=k, x_bf16=1, dst_dev=y[1].data_ptr(), ldd=n + 3, m=m, n=n, k=k, batch=1)
    _lib.check("cq_dense_product", L.cq_dense_product(0, ctypes.byref(a), ws.data_ptr(), nb, ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)))
    torch.cuda.synchronize()
    want = x.double() @ w.double().t()
    err = (y[1:m + 1, :n].double() - want).norm(dim=1) / want.norm(dim=1)
    assert float(err.max()) <= BOUND
    assert (y[0] == 5).all() and (y[m + 1] == 5).all() and (y[:, n:] == 5).all()


@pytest.mark.parametrize("m,n,k,pad", [(1100, 2500, 1024, 0), (1535, 2049, 1088, 64), (1500, 2817, 1024, 128), (1537, 2700, 4160, 0), (1290, 4485, 1024, 0), (1000, 5602, 1024, 0), (1500, 5633, 1088, 64)])
@pytest.mark.parametrize("form", ["plain", "add", "swiglu", "bf16", "rows"])
def test_ring_of_stages(m, n, k, pad, form):
    """One workgroup to a unit: 128 rows (180 and 204 tiles), 192 (one round), 128 in two rounds, 192 in two; stages of k even and odd."""
    print(f"case {m} {n} {k} {pad} {form}", flush=True)
    if form == "swiglu":
        n &= ~1
    g = torch.Generator(device="cuda").manual_seed(m + n + k)
    w = torch.randn((n, k + pad), generator=g, device="cuda").mul_(0.02).bfloat16()
    x = torch.randn((m, k + pad), generator=g, device="cuda").bfloat16()
    x[:, k:], w[:, k:] = float("nan"), float("nan")
    cols = n // 2 if form == "swiglu" else n
    y = torch.full((m + 2, cols + 3), 5.0, device="cuda", dtype=torch.bfloat16 if form == "bf16" else torch.float32)
    add = torch.randn((m, n), generator=g, device="cuda") if form == "add" else None
    perm = torch.randperm(m, generator=g, device="cuda").int() if form == "rows" else None
    scale = torch.rand(m, generator=g, device="cuda") + 0.5 if form == "swiglu" else None
    a = DenseArgs(w_dev=w.data_ptr(), ldw=k + pad, x_dev=x.data_ptr(), ldx=k + pad, x_bf16=1, dst_dev=y[1].data_ptr(), ldd=cols + 3, m=m, n=n, k=k, batch=1,
                  dst_bf16=int(form == "bf16"), act=2 if form == "swiglu" else 0, accumulate=int(form == "add"), add_dev=add.data_ptr() if form == "add" else None,
                  ld_add=n if form == "add" else 0, dst_rows_dev=perm.data_ptr() if form == "rows" else None, row_scale_dev=scale.data_ptr() if form == "swiglu" else None)
    L = _lib.mixer_lib()
    nb = L.cq_dense_matmul_workspace_bytes(0, m, n, k)
    ws = torch.empty(max(nb, 16), dtype=torch.uint8, device="cuda")
    _lib.check("cq_dense_product", L.cq_dense_product(0, ctypes.byref(a), ws.data_ptr(), nb, ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)))
    torch.cuda.synchronize()
    want = x[:, :k].double() @ w[:, :k].double().t()
    size = want.norm(dim=1, keepdim=True)
    if form == "add":
        want += add + 5.0
    if form == "swiglu":
        want = torch.nn.functional.silu(want[:, 0::2]) * want[:, 1::2] * scale[:, None]
    got = y[1:m + 1, :cols].double()
    if form == "rows":
        got = got[perm.long()]
    err = (got - want).abs()
    if form == "bf16":
        err = (err - want.abs() * 2.0 ** -8).clamp(min=0)
    if form == "add":
        err = (err - want.abs() * 2.0 ** -23).clamp(min=0)              # two more roundings
    assert float((err.norm(dim=1, keepdim=True) / size).max()) <= BOUND * (4 if form == "swiglu" else 1)
    assert (y[0] == 5).all() and (y[m + 1] == 5).all() and (y[:, cols:] == 5).all()


@pytest.mark.parametrize("m,n,k", [(2000, 2048, 1536), (1100, 2500, 1024), (1000, 1800, 2112), (1500, 2048, 7168), (1290, 4485, 1024), (1537, 2700, 4160), (1000, 5602, 1024),
                                   (1535, 4481, 512), (1500, 5633, 1088), (1200, 7168, 2048), (100, 49100, 1024)])
def test_ring_of_stages_keeps_bits(m, n, k):
    """Bit for bit what the same rows in f32 give, which go through the 128 x 128 tile (or the large one): a choice made from a product, like that of a token's
    experts, may not depend on the kernel.  One part of k, two to four, even and uneven; 128 rows and 192; a few rows of very many columns, where the large tile stays."""
    g = torch.Generator(device="cuda").manual_seed(m + n + k)
    w = torch.randn((n, k), generator=g, device="cuda").mul_(0.02).bfloat16()
    x = torch.randn((m, k), generator=g, device="cuda").bfloat16()
    L = _lib.mixer_lib()
    nb = L.cq_dense_matmul_workspace_bytes(0, m, n, k)
    ws = torch.empty(max(nb, 16), dtype=torch.uint8, device="cuda")
    got = []
    for rows in (x, x.float()):
        y = torch.randn((m, n), generator=torch.Generator(device="cuda").manual_seed(1), device="cuda")
        a = DenseArgs(w_dev=w.data_ptr(), ldw=k, x_dev=rows.data_ptr(), ldx=k, x_bf16=int(rows is x), dst_dev=y.data_ptr(), ldd=n, m=m, n=n, k=k, batch=1, accumulate=1)
        _lib.check("cq_dense_product", L.cq_dense_product(0, ctypes.byref(a), ws.data_ptr(), nb, ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)))
        got.append(y)
    assert torch.equal(*got)


@pytest.mark.parametrize("m,n,k", [(1500, 2048, 1024), (1290, 4485, 1024), (1000, 5602, 1024), (40, 516, 1024), (700, 517, 1024), (2300, 4610, 1088)])
@pytest.mark.parametrize("x_bf16", [0, 1])
def test_row_factors_of_sums(m, n, k, x_bf16):
    """The factor of a row is the product's alone: y + factor * (x w) + add, whichever kernel the call takes (ring of 128 and of 192 rows, small tiles in one part and
    in several, the large tile).  Three roundings more than the products alone."""
    g = torch.Generator(device="cuda").manual_seed(m + n + k)
    w = torch.randn((n, k), generator=g, device="cuda").mul_(0.02).bfloat16()
    x = torch.randn((m, k), generator=g, device="cuda").bfloat16()
    xd = x if x_bf16 else x.float()
    scale, add, y = torch.rand(m, generator=g, device="cuda") * 4 - 2, torch.randn((m, n), generator=g, device="cuda"), torch.randn((m, n), generator=g, device="cuda")
    product = x.double() @ w.double().t() * scale[:, None]
    want = y + product + add
    L = _lib.mixer_lib()
    nb = L.cq_dense_matmul_workspace_bytes(0, m, n, k)
    ws = torch.empty(max(nb, 16), dtype=torch.uint8, device="cuda")
    a = DenseArgs(w_dev=w.data_ptr(), ldw=k, x_dev=xd.data_ptr(), ldx=k, x_bf16=x_bf16, dst_dev=y.data_ptr(), ldd=n, m=m, n=n, k=k, batch=1, accumulate=1,
                  add_dev=add.data_ptr(), ld_add=n, row_scale_dev=scale.data_ptr())
    _lib.check("cq_dense_product", L.cq_dense_product(0, ctypes.byref(a), ws.data_ptr(), nb, ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)))
    size = product.norm(dim=1) + want.norm(dim=1)
    assert float(((y.double() - want).norm(dim=1) / size).max()) <= BOUND


@pytest.mark.parametrize("x_bf16", [0, 1])
@pytest.mark.parametrize("tiles,n,k", [(2, 1028, 8192), (3, 1028, 5120), (3, 4100, 5120), (6, 516, 5120), (7, 516, 5120)])
def test_last_row_tile_of_any_height(tiles, n, k, x_bf16):
    """128-row tiles, the last one with rows of one to four fragments: in the forms for each and in one form (7 row tiles), with one stage on its way and with three: the bits of the same
    rows with all tiles full, which come as near to float64 as the products of this file do; nothing behind the last row is written."""
    print(f"case {tiles} {n} {k} {x_bf16}", flush=True)
    L, full = _lib.mixer_lib(), 128 * tiles
    g = torch.Generator(device="cuda").manual_seed(tiles + n + k)
    w = torch.randn((n, k), generator=g, device="cuda").mul_(0.02).bfloat16()
    x = torch.randn((full, k), generator=g, device="cuda").bfloat16()
    xd = x if x_bf16 else x.float()
    nb = L.cq_dense_matmul_workspace_bytes(0, full, n, k)
    ws = torch.empty(nb, dtype=torch.uint8, device="cuda")

    def product(m):
        y = torch.full((m + 1, n), 5.0, device="cuda")
        a = DenseArgs(w_dev=w.data_ptr(), ldw=k, x_dev=xd.data_ptr(), ldx=k, x_bf16=x_bf16, dst_dev=y.data_ptr(), ldd=n, m=m, n=n, k=k, batch=1)
        assert L.cq_dense_matmul_workspace_bytes(0, m, n, k) == nb // full * m
        _lib.check("cq_dense_product", L.cq_dense_product(0, ctypes.byref(a), ws.data_ptr(), nb, ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)))
        assert bool((y[m] == 5).all())
        return y[:m]

    all_rows = product(full)
    want = x.double() @ w.double().t()
    assert float(((all_rows - want).norm(dim=1) / want.norm(dim=1)).max()) <= BOUND
    for last in (1, 15, 16, 17, 31, 32, 33, 63, 64, 65, 95, 96, 97, 127):
        m = full - 128 + last
        assert torch.equal(product(m), all_rows[:m]), last


@pytest.mark.parametrize("m,n,k,tile_rows", [(1100, 2506, 1024, 0), (1500, 5634, 1088, 0), (2000, 3202, 832, 0), (2000, 3266, 512, 0), (2300, 4612, 1088, 0), (300, 2506, 1024, 128), (130, 190, 512, 128),
                                             (130, 190, 512, 64), (70, 190, 512, 32)])
@pytest.mark.parametrize("form", ["bf16", "relu2", "swiglu", "sum"])
def test_results_on_and_off_16_bytes(m, n, k, tile_rows, form):
    """Results that lie on 16 bytes go out by whole rows, four lanes 64 bytes (bfloat16) or row by row with what they are added to asked for ahead (f32); elsewhere, and in the last
    columns, four at a time: the same bits.  Ring of 128 and of 192 rows, the 128 x 128 tile with three stages and with one, the large tile, tiles of a table with scattered rows and factors."""
    print(f"case {m} {n} {k} {tile_rows} {form}", flush=True)
    g = torch.Generator(device="cuda").manual_seed(m + n + k)
    groups = 3 if tile_rows else 1
    w = torch.randn((groups, n, k), generator=g, device="cuda").mul_(0.02).bfloat16()
    x = torch.randn((m, k), generator=g, device="cuda").bfloat16()
    scale, perm, cols = torch.rand(m, generator=g, device="cuda") + 0.5, torch.randperm(m, generator=g, device="cuda").int(), n // 2 if form == "swiglu" else n
    starts = [t for e in range(groups) for t in range(e * m // groups, (e + 1) * m // groups, tile_rows)] if tile_rows else []
    of = [next(e for e in range(groups) if t < (e + 1) * m // groups) for t in starts]
    tiles = torch.tensor([[e, t, min(tile_rows, (e + 1) * m // groups - t), 0] for e, t in zip(of, starts)], dtype=torch.int32, device="cuda")
    n_tiles = torch.tensor([len(starts)], dtype=torch.int32, device="cuda")
    L, got = _lib.mixer_lib(), []
    nb = L.cq_dense_matmul_workspace_bytes(0, m, n, k)
    ws = torch.empty(max(nb, 16), dtype=torch.uint8, device="cuda")
    for ld, first in (((cols + 7) // 8 * 8 + 8, 0), ((cols + 7) // 8 * 8 + 3, 1)):
        y = torch.full((m + 2, ld), 3.0, device="cuda", dtype=torch.float32 if form == "sum" else torch.bfloat16)
        add = torch.randn((m, n), generator=torch.Generator(device="cuda").manual_seed(1), device="cuda")
        add = torch.nn.functional.pad(add, (0, ld - n))
        a = DenseArgs(w_dev=w.data_ptr(), ldw=k, w_batch=n * k, x_dev=x.data_ptr(), ldx=k, x_bf16=1, dst_dev=y[1].data_ptr() + first * y.element_size(), ldd=ld, m=m, n=n, k=k, batch=1,
                      dst_bf16=int(form != "sum"), act={"relu2": 1, "swiglu": 2}.get(form, 0), row_scale_dev=scale.data_ptr(), dst_rows_dev=perm.data_ptr())
        if tile_rows:
            a.tiles_dev, a.n_tiles_dev, a.max_tiles, a.tile_rows = tiles.data_ptr(), n_tiles.data_ptr(), len(starts) + 2, tile_rows
        elif form == "sum":
            a.accumulate, a.add_dev, a.ld_add = 1, add.data_ptr(), ld
        _lib.check("cq_dense_product", L.cq_dense_product(0, ctypes.byref(a), ws.data_ptr(), nb, ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)))
        flat = y.flatten()[ld + first:]
        got.append(flat[:m * ld].view(m, ld)[:, :cols].clone())
        flat[:m * ld].view(m, ld)[:, :cols] = 3.0
        assert bool((y == 3).all())
    assert torch.equal(*got)
    rows = torch.cat([x[t:t + c].double() @ w[e].double().t() for e, t, c, _ in tiles.tolist()]) if tile_rows else x.double() @ w[0].double().t()
    size = rows.norm(dim=1, keepdim=True)
    if form == "swiglu":
        rows = torch.nn.functional.silu(rows[:, 0::2]) * rows[:, 1::2]
    if form == "relu2":
        rows, size = rows.clamp(min=0).square(), size * rows.abs().amax()      # (a square's slope: twice the value)
    rows = rows * scale[:, None]
    if form == "sum" and not tile_rows:
        rows = rows + 3.0 + add[perm.long(), :n]
    err = (got[0].double()[perm.long()] - rows).abs()
    err = (err - rows.abs() * (2.0 ** -22 if form == "sum" else 2.0 ** -8)).clamp(min=0)
    assert float((err.norm(dim=1, keepdim=True) / size).max()) <= BOUND * 4


@pytest.mark.parametrize("m,n,k", [(1000, 2048, 2048), (961, 2049, 1024), (260, 3500, 1088), (513, 2047, 2112), (850, 1024, 3584), (1024, 2500, 1024), (1153, 2178, 1088), (1536, 2048, 4160), (577, 4481, 1024)])
def test_ring_of_64_and_of_96_rows(m, n, k):
    """Last tiles of one row and of all but one, one part of k and up to ten: the bits of the 128 x 128 tile, and results of every kind."""
    test_ring_of_stages_keeps_bits(m, n, k)
    for form in ("add", "bf16", "rows"):
        test_ring_of_stages(m, n, k, 64, form)
    for form in ("bf16", "relu2", "sum"):
        test_results_on_and_off_16_bytes(m, n // 2 * 2, k, 0, form)


@pytest.mark.parametrize("form", ["plain", "add", "swiglu", "bf16", "rows"])
def test_ring_of_96_rows_or_of_128_of_silu_results(form):
    test_ring_of_stages(2000, 2046, 1088, 64, form)


@pytest.mark.parametrize("m,n,k", [(260, 3500, 2112), (850, 1024, 2560), (961, 1024, 4096)])
def test_ring_of_64_rows_in_three_parts_of_k_and_more(m, n, k):
    test_ring_of_64_and_of_96_rows(m, n, k)


@pytest.mark.parametrize("precision,x_bf16,m,n,k", [(0, 1, 1100, 2506, 1024), (0, 1, 2000, 2046, 1088), (0, 1, 1500, 5634, 1088), (0, 1, 961, 2050, 1024), (0, 1, 1000, 2046, 2048), (0, 1, 2000, 3202, 832), (0, 0, 2000, 3203, 512),
                                                    (0, 1, 2300, 4610, 1088), (0, 1, 50, 190, 512), (0, 0, 50, 189, 512), (0, 1, 20, 66, 256), (1, 0, 70, 190, 192), (1, 0, 70, 62, 192)])
@pytest.mark.parametrize("accumulate,addend", [(1, 0), (0, 1), (1, 1)])
def test_sums_off_16_bytes(precision, x_bf16, m, n, k, accumulate, addend):
    """Results added to what is there, to an addend and to both, off 16 bytes (what they are added to is asked for a row ahead, column by column) and on them: the same bits, in every kernel,
    and nothing beside them changes."""
    print(f"case {precision} {x_bf16} {m} {n} {k} {accumulate} {addend}", flush=True)
    g = torch.Generator(device="cuda").manual_seed(m + n + k)
    w = torch.randn((n, k), generator=g, device="cuda").mul_(0.02).bfloat16()
    x = torch.randn((m, k), generator=g, device="cuda")
    x = x.bfloat16() if x_bf16 else x
    there, more = (torch.randn((m, n), generator=g, device="cuda") for _ in range(2))
    L, got = _lib.mixer_lib(), []
    nb = L.cq_dense_matmul_workspace_bytes(precision, m, n, k)
    ws = torch.empty(max(nb, 16), dtype=torch.uint8, device="cuda")
    for ld, first in (((n + 3) // 4 * 4 + 4, 0), ((n + 3) // 4 * 4 + 5, 1)):
        y, add = (torch.nn.functional.pad(t, (0, ld - n, 1, 1), value=3.0).flatten().contiguous() for t in (there, more))
        y, add = (torch.cat([t.new_full((first,), 3.0), t]) for t in (y, add))
        a = DenseArgs(w_dev=w.data_ptr(), ldw=k, x_dev=x.data_ptr(), ldx=k, x_bf16=x_bf16, dst_dev=y.data_ptr() + 4 * (first + ld), ldd=ld, m=m, n=n, k=k, batch=1, accumulate=accumulate,
                      add_dev=add.data_ptr() + 4 * (first + ld) if addend else None, ld_add=ld if addend else 0)
        _lib.check("cq_dense_product", L.cq_dense_product(precision, ctypes.byref(a), ws.data_ptr(), nb, ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)))
        rows = y[first:].view(m + 2, ld)
        got.append(rows[1:m + 1, :n].clone())
        rows[1:m + 1, :n] = 3.0
        assert bool((y == 3.0).all())
    assert torch.equal(*got)
    want = (x if precision else x.bfloat16()).double() @ w.double().t()
    size = want.norm(dim=1, keepdim=True)
    want = want + accumulate * there + addend * more
    err = ((got[0] - want).abs() - want.abs() * 2.0 ** -22).clamp(min=0)       # (up to three roundings of the sums themselves)
    assert float((err.norm(dim=1, keepdim=True) / size).max()) <= BOUND
