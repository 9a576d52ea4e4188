"""Norms and embeddings with four or eight values a load, on both sides of what a thread and a workgroup hold, few rows and many, against the
plain torch functions."""
import pytest
import torch

from servelab_amd.kernels.values import PartialSums
from test_vekanex_kernels_gpu import DEV, close, tables

pytestmark = pytest.mark.gpu
# a bfloat16 result differs by one rounding at most (2^-8 of it), a float32 one by the order of its sums
BAR = {torch.float32: 4e-6, torch.bfloat16: 8e-3}


# one group of four, no whole wavefront, 1,024 groups and one more, the widest, one more, a width that is no multiple of four
@pytest.mark.parametrize("H", [4, 132, 4096, 4100, 8196, 16384, 16388, 1027])
@pytest.mark.parametrize("R", [3, 257])
@pytest.mark.parametrize("dtype", list(BAR))
def test_norms(H, R, dtype):
    hip, emu = tables(dtype)
    g = torch.Generator().manual_seed(H + R)
    stream, w, w2, bias = torch.randn(R, H, generator=g), *(1 + 0.3 * torch.randn(3, H, generator=g))
    y, y2 = (torch.randn(R, H, generator=g).to(dtype) for _ in range(2))
    rows = torch.tensor([R - 1, 0], dtype=torch.int32)
    dev = lambda t: None if t is None else t.to(DEV)

    def check(name, *args):
        a, b = stream.to(DEV), stream.clone()
        close(getattr(hip, name)(a, *(x.to(DEV) if isinstance(x, torch.Tensor) else x for x in args)), getattr(emu, name)(b, *args), BAR[dtype])
        close(a, b, BAR[torch.float32])

    for delta in (None, y):
        check("add_rmsnorm", delta, w, 1e-5)
        check("rows_add_rmsnorm", delta, rows, w, 1e-5)
    check("add_normed_rmsnorm", y, w2, 1e-5, w, 1e-6)
    check("add_postnorm", y, w, 1e-5, 0.5)
    for parts in (1, 2, 3, 4, 5, 8, 9):
        if parts * R * H > 2 ** 24:
            continue
        p = torch.randn(parts, R, H, generator=g)
        for add in (None, bias):
            a, b = stream.to(DEV), stream + p.sum(0) + (0 if add is None else add)
            got = hip.add_rmsnorm(a, PartialSums(dev(p), dev(add)), dev(w), 1e-5)
            close(a, b, BAR[torch.float32])
            close(got, emu.add_rmsnorm(b, None, w, 1e-5), BAR[dtype])
            a = stream.to(DEV)
            close(hip.rows_add_rmsnorm(a, PartialSums(dev(p), dev(add)), dev(rows), dev(w), 1e-5), emu.rows_add_rmsnorm(b, None, rows, w, 1e-5),
                  BAR[dtype])
            assert torch.equal(a.cpu(), stream)
    for deltas in (None, (y,), (y, y2)):
        for at, add in ((None, None), (None, bias), (rows, bias)):
            a, b = stream.to(DEV), stream.clone()
            got = hip.add_layernorm(a, deltas and tuple(map(dev, deltas)), dev(w), 1e-5, rows=dev(at), bias=dev(add))
            close(got, emu.add_layernorm(b, deltas, w, 1e-5, rows=at, bias=add), BAR[dtype])
            close(a, b, BAR[torch.float32])
    copies, mix, coef = torch.randn(R, 4, H, generator=g), torch.randn(4, 4, generator=g) / 2, torch.randn(2, 4, generator=g)
    if R * H < 2 ** 21:
        for outputs in ([], [(y, None, 0.0)], [(y, w2, 1e-5), (y2, w, 1e-5)]):
            for at in (None, rows):
                a, b = copies.to(DEV), copies.clone()
                got = hip.streams_norm(a, [(dev(t), dev(n), e) for t, n, e in outputs], dev(mix), dev(coef[0]), dev(coef[1]), dev(w),
                                       dev(bias), 1e-5, rows=dev(at)) if H <= 16384 else None
                if got is not None:
                    close(got, emu.streams_norm(b, outputs, mix, coef[0], coef[1], w, bias, 1e-5, rows=at), BAR[dtype])
                    close(a, b, BAR[torch.float32])


@pytest.mark.parametrize("H", [8, 520, 2048, 2056, 12])
@pytest.mark.parametrize("copies", [0, 1, 3])
@pytest.mark.parametrize("dtype", list(BAR))
def test_embeddings(H, copies, dtype):
    hip, emu = tables(dtype)
    g = torch.Generator().manual_seed(H)
    table, places = torch.randn(50, H, generator=g).to(dtype), torch.randn(9, H, generator=g).to(dtype)
    ids, at = torch.tensor([49, 0, 7], dtype=torch.int32), torch.tensor([8, 0, 3], dtype=torch.int32)
    for args, kw in (((), {}), ((at, places), {})):
        got = hip.embed(ids.to(DEV), table.to(DEV), 1.5, *(x.to(DEV) for x in args), copies=copies)
        close(got, emu.embed(ids, table, 1.5, *args, copies=copies), 1e-6)
