"""Routing with an expert a lane: 64 experts, one fewer and one more, as many choices as experts."""
import ctypes

import pytest
import torch

from servelab_amd.kernels import HipOps
from test_few_rows_experts_gpu import test_routes_and_their_tiles as routes_and_their_tiles
from test_few_rows_experts_gpu import test_routes_of_logits_that_are_not_numbers as routes_of_odd_logits

pytestmark = pytest.mark.gpu
FORMS = ["softmax", "over all", "sigmoid"]


@pytest.mark.parametrize("T,E,top", [(4, 64, 8), (3, 64, 11), (16, 63, 2), (11, 40, 3), (8, 65, 4), (1, 64, 64), (2, 3, 3)])
@pytest.mark.parametrize("form", FORMS)
def test_places_and_tiles(T, E, top, form):
    routes_and_their_tiles(T, E, top, form)


@pytest.mark.parametrize("T,E,top", [(4, 63, 8), (5, 64, 6), (16, 64, 2), (40, 64, 8)])
@pytest.mark.parametrize("form", FORMS)
def test_odd_logits(T, E, top, form):
    routes_of_odd_logits(T, E, top, form)


# no group of four channels behind the last whole workgroup, one, a width without groups; no choice beside a trip's eight, one, two trips; every form; few
# tokens, which take four channels a thread for some numbers of choices, and so many that they always do
@pytest.mark.parametrize("H", [4, 1024, 1028, 2052, 30])
@pytest.mark.parametrize("top", [1, 4, 5, 8, 9, 13, 17])
@pytest.mark.parametrize("many", [False, True])
def test_sums_over_the_choices(H, top, many):
    for dtype in (torch.float32, torch.bfloat16):
        ops, T, E = HipOps(dtype, "cuda:0"), -(-400000 // H) if many else 3, 5
        g = torch.Generator(device="cuda:0").manual_seed(H + top)
        new = lambda *s: torch.randn(*s, generator=g, device="cuda:0")
        y, base, x, gate = new(T * top, H), new(T, H).to(dtype), new(T, H).to(dtype), new(T, 2)
        place = torch.randperm(T * top, generator=g, device="cuda:0").int()
        shares, chosen = torch.rand(T, top, generator=g, device="cuda:0"), torch.randint(0, E + 2, (T, top), generator=g, device="cuda:0").int()
        lib, p = ops._lazy("routed"), lambda t: ctypes.c_void_p(t.data_ptr()) if t is not None else None
        for b, z, s, c in ((None, None, shares, None), (base, gate, shares, chosen), (base, None, None, None), (None, None, None, chosen)):
            out = torch.empty(T, H, dtype=dtype, device="cuda:0")
            ops._call(lib, "sl_routed_combine", p(y), p(place), p(s), T, top, p(b), p(z), 2, H, p(out), p(c), E, p(x) if c is not None else None)
            rows = y.double()[place.long()].view(T, top, H)
            if c is not None:
                rows = torch.where((c >= E)[..., None], x.double()[:, None], rows)
            if s is not None:
                rows = rows * s.double()[..., None]
            own = torch.zeros(T, H, dtype=torch.float64, device="cuda:0") if b is None else b.double() * (1 if z is None else z[:, :1].double().sigmoid())
            want, size = own + rows.sum(1), own.abs() + rows.abs().sum(1)
            # float sums of top + 1 terms, then a rounding to the activation type
            assert ((out.double() - want).abs() <= (top + 4) * 2.0 ** -23 * size + (2.0 ** -8 if dtype == torch.bfloat16 else 0) * want.abs()).all()
