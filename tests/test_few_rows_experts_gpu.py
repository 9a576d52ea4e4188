"""The grouped products where an expert has few rows, at the sizes where their split of K and their column blocks can
go wrong, against the plain torch form (tests/emulated_ops.py)."""
import pytest
import torch

from emulated_ops import EmulatedOps
from servelab_amd.kernels import HipOps
from servelab_amd.kernels.recurrent_ops import Routing

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


# (tokens, experts, top, ff, width): K of one step (seven of eight wavefronts without a share), of a number of steps that
# eight does not divide, the last column block of 32 half empty, 6 and 8 rows an expert and just beyond, every token at the
# same experts (tiles of 16 rows full, a second one with one row)
@pytest.mark.parametrize("T,E,top,ff,K", [(1, 4, 2, 16, 32), (3, 8, 3, 48, 352), (6, 2, 2, 48, 96), (8, 4, 4, 80, 288),
                                          (9, 4, 4, 80, 288), (17, 3, 1, 16, 64), (1, 64, 8, 1024, 2048)])
@pytest.mark.parametrize("form", ["gated", "plain", "weighed input"])
def test_few_rows_an_expert(T, E, top, ff, K, form):
    hip, emu = HipOps(torch.bfloat16, DEV), EmulatedOps(torch.bfloat16)
    g = torch.Generator().manual_seed(T + E)
    gated = form != "plain"
    x = torch.randn(T, K, generator=g).bfloat16()
    first = (torch.randn(E, (2 if gated else 1) * ff, K, generator=g) * K ** -0.5).bfloat16()
    down = (torch.randn(E, K, ff, generator=g) * ff ** -0.5).bfloat16()
    logits = torch.randn(T, E, generator=g)
    if T == 17:
        logits[:, 1] += 20.0
    r = hip.route_tokens(logits.to(DEV), E, top, sigmoid=form == "weighed input")
    assert r.tile_rows == 16
    options = dict(activation="silu" if gated else "relu2", gated=gated, weigh_input=form == "weighed input")
    want = emu.routed_experts(x, (r.chosen.cpu(), r.shares.cpu()), first, down, None, **options)
    for a, b in ((first.to(DEV), down.to(DEV)),
                 (hip.prepare_expert_matrices(first.to(DEV), gated=gated), hip.prepare_expert_matrices(down.to(DEV)))):
        got = hip.routed_experts(x.to(DEV), r, a, b, None, **options).float().cpu()
        # float sums in another order (2^-24 sqrt(K) of a sum) may round either way where the activation type is 2^-8
        # wide: at most three roundings (the activated row, its product, the result) of a value of this size
        bar = 3 * 2.0 ** -8 * want.float().abs().max().item()
        assert (got - want.float()).abs().max().item() <= bar


# tiles of 128 rows: one and two chunks of 64 values of k, more than the ring holds, a number of steps of 32 that is odd
# (the kernel beside it); column blocks of 128 (gated) and 256 with one tile of 16, and one more than whole; 12 rows an expert
# and less for most, a second tile of one row, every token at the same expert (the others without tiles)
@pytest.mark.parametrize("T,E,top,ff,K,one", [(12, 8, 8, 16, 64, False), (129, 8, 8, 144, 128, False), (300, 9, 1, 272, 320, True),
                                              (100, 16, 2, 96, 192, False), (70, 8, 2, 128, 96, False), (400, 4, 1, 64, 64, False)])
@pytest.mark.parametrize("form", ["gated", "plain", "weighed input"])
def test_tiles_of_128_rows(T, E, top, ff, K, one, form):
    hip, emu = HipOps(torch.bfloat16, DEV), EmulatedOps(torch.bfloat16)
    g = torch.Generator().manual_seed(T + E)
    gated = form != "plain"
    x = torch.randn(T, K, generator=g).bfloat16()
    first = (torch.randn(E, (2 if gated else 1) * ff, K, generator=g) * K ** -0.5).bfloat16()
    down = (torch.randn(E, K, ff, generator=g) * ff ** -0.5).bfloat16()
    logits = torch.randn(T, E, generator=g)
    if one:
        logits[:, 4] += 20.0
    r = hip.route_tokens(logits.to(DEV), E, top, sigmoid=form == "weighed input")
    assert r.tile_rows == 128
    options = dict(activation="silu" if gated else "relu2", gated=gated, weigh_input=form == "weighed input")
    want = emu.routed_experts(x, (r.chosen.cpu(), r.shares.cpu()), first, down, None, **options)
    for a, b in ((first.to(DEV), down.to(DEV)),
                 (hip.prepare_expert_matrices(first.to(DEV), gated=gated), hip.prepare_expert_matrices(down.to(DEV)))):
        got = hip.routed_experts(x.to(DEV), r, a, b, None, **options).float().cpu()
        # (as above)
        bar = 3 * 2.0 ** -8 * want.float().abs().max().item()
        assert (got - want.float()).abs().max().item() <= bar


def test_rows_a_tile_holds():
    hip = HipOps(torch.bfloat16, DEV)
    rows = lambda T, E, top: hip.route_tokens(torch.randn(T, E, device=DEV), E, top).tile_rows
    assert (rows(11, 8, 8), rows(12, 8, 8), rows(95, 4, 4), rows(96, 4, 4)) == (16, 128, 16, 128)
    assert HipOps(torch.float32, DEV).route_tokens(torch.randn(200, 8, device=DEV), 8, 8).tile_rows == 16


@pytest.mark.parametrize("T,E,top", [(4, 64, 8), (16, 300, 4), (17, 64, 8), (4, 5, 5)])
@pytest.mark.parametrize("form", ["softmax", "over all", "sigmoid"])
def test_routes_of_logits_that_are_not_numbers(T, E, top, form):
    """Every choice is an expert, NaN behind all numbers, and its row's shares say so; other rows are as without such a row."""
    hip = HipOps(torch.bfloat16, DEV)
    z = torch.randn(T, E, generator=torch.Generator().manual_seed(E))
    route = lambda z: hip.route_tokens(z.to(DEV), E, top, over_all=form == "over all", sigmoid=form == "sigmoid")
    before = route(z)
    z[1] = torch.nan
    z[2, top - 1:] = torch.nan                                        # one number too few
    z[3, E - 1] = torch.nan
    r = route(z)
    number = torch.where(z.isnan() | (z.isnan().any(-1, keepdim=True) if form == "over all" else False), -torch.inf, z)
    assert torch.equal(r.chosen.cpu().long(), torch.sort(-number, dim=-1, stable=True).indices[:, :top])
    odd = z.gather(1, r.chosen.cpu().long()).isnan()
    if form != "sigmoid":                                             # (a share takes in the chosen ones' sum, or that of all)
        odd = (z.isnan() if form == "over all" else odd).any(-1, keepdim=True).expand(T, top)
    assert torch.equal(r.shares.cpu().isnan(), odd)
    same = [t for t in range(T) if t not in (1, 2, 3)]
    assert torch.equal(r.chosen[same], before.chosen[same]) and torch.equal(r.shares[same], before.shares[same])
    flat, order = r.chosen.cpu().flatten().long(), r.order.cpu().long()
    assert torch.equal(order[r.place_of.cpu().long()], torch.arange(T * top)) and (flat[order].diff() >= 0).all()


# one workgroup for both up to 16 tokens and 1,024 experts, two kernels beyond; experts a wavefront adds up in one, two and
# more rounds, some without matrices, equal logits, logits of minus infinity
@pytest.mark.parametrize("T,E,top", [(1, 1, 1), (1, 64, 8), (16, 65, 8), (17, 65, 8), (5, 300, 64), (16, 1024, 3), (16, 1025, 3)])
@pytest.mark.parametrize("form", ["softmax", "over all", "sigmoid"])
def test_routes_and_their_tiles(T, E, top, form):
    hip = HipOps(torch.bfloat16, DEV)
    g = torch.Generator().manual_seed(T + E)
    z = torch.randn(T, E + 2, generator=g)[:, :E]
    if E > 1:
        z[0, E // 2] = z[0, 0] = 3.0
    if E > 2 * top:
        z[0, -top:] = -torch.inf
    real = max(1, E - 1)
    r = hip.route_tokens(z.to(DEV), E, top, over_all=form == "over all", with_matrices=real, sigmoid=form == "sigmoid")
    number = torch.softmax(z, -1) if form == "over all" else z
    order = torch.sort(-number, dim=-1, stable=True).indices[:, :top]
    assert torch.equal(r.chosen.cpu().long(), order)
    picked = number.gather(1, order).double()
    want = torch.sigmoid(picked) if form == "sigmoid" else (
        picked / (picked.sum(-1, keepdim=True) + 1e-20) if form == "over all" else torch.softmax(picked, -1))
    # exponentials and a sum of at most 64 float terms
    assert ((r.shares.cpu().double() - want).abs() <= 1e-5 * want + 1e-7).all()
    flat, order, place = r.chosen.cpu().flatten().long(), r.order.cpu().long(), r.place_of.cpu().long()
    assert torch.equal(order[place], torch.arange(T * top)) and (flat[order].diff() >= 0).all()
    tiles, first = [], 0
    for e in range(E):
        n = int((flat == e).sum())
        if e < real:
            tiles += [[e, first + i, min(r.tile_rows, n - i)] for i in range(0, n, r.tile_rows)]
        first += n
    got = r.tiles.cpu()
    assert got[:len(tiles)].tolist() == tiles and (got[len(tiles):] == 0).all()


@pytest.mark.parametrize("T,tile_rows", [(5, 16), (100, 128)])
def test_a_routing_put_together_by_a_caller(T, tile_rows):
    """Its tiles need not come from the router's buffer, nor the ones with rows first."""
    E, top, ff, K = 8, 2, 48, 64
    hip = HipOps(torch.bfloat16, DEV)
    g = torch.Generator().manual_seed(T)
    x = torch.randn(T, K, generator=g).bfloat16().to(DEV)
    first = hip.prepare_expert_matrices((torch.randn(E, 2 * ff, K, generator=g) * K ** -0.5).bfloat16().to(DEV), gated=True)
    down = hip.prepare_expert_matrices((torch.randn(E, K, ff, generator=g) * ff ** -0.5).bfloat16().to(DEV))
    r = hip.route_tokens(torch.randn(T, E, generator=g).to(DEV), E, top)
    assert r.tile_rows == tile_rows and r.tiles_in_use.item() == (r.tiles[:, 2] > 0).sum().item()
    own = Routing(r.chosen, r.shares, r.order, r.place_of, r.tiles.flip(0).contiguous(), tile_rows)
    assert torch.equal(hip.routed_experts(x, own, first, down), hip.routed_experts(x, r, first, down))


def test_tiles_asked_for_by_the_matrices():
    """Rows of an odd number of 32 values stay in tiles of 16 where the staged kernel cannot take them; either gives the same."""
    T, E, top, ff, K = 70, 8, 2, 1024, 96
    hip = HipOps(torch.bfloat16, DEV)
    g = torch.Generator().manual_seed(3)
    x = torch.randn(T, K, generator=g).bfloat16().to(DEV)
    first = hip.prepare_expert_matrices((torch.randn(E, 2 * ff, K, generator=g) * K ** -0.5).bfloat16().to(DEV), gated=True)
    down = hip.prepare_expert_matrices((torch.randn(E, K, ff, generator=g) * ff ** -0.5).bfloat16().to(DEV))
    logits = torch.randn(T, E, generator=g).to(DEV)
    rows = hip.expert_tile_rows(T * top, first)
    r, wide = (hip.route_tokens(logits, E, top, tile_rows=n) for n in (rows, None))
    assert (r.tile_rows, wide.tile_rows) == (16, 128)
    got, want = (hip.routed_experts(x, v, first, down).float() for v in (r, wide))
    # (as above)
    assert (got - want).abs().max() <= 3 * 2.0 ** -8 * want.abs().max()


@pytest.mark.parametrize("rows", [128, 256])
@pytest.mark.parametrize("gated,act", [(True, "silu"), (False, "relu2")])
def test_workgroups_that_walk_more_items_than_they_look_up(gated, act, rows):
    """Tiles of 128 and 256 rows: 104 row tiles (of 128) of 32 column blocks, of which a workgroup of 256 looks up twelve at a time; an
    expert without rows, one with a single row and one with half a tile among them."""
    hip = HipOps(torch.bfloat16, DEV)
    E, ff, K = 6, 4096 if gated else 8192, 64
    g = torch.Generator().manual_seed(3)
    counts = [6400, 0, 1, 64, 6399, 300] if rows == 128 else [12800, 0, 1, 128, 12799, 600]
    chosen = torch.repeat_interleave(torch.arange(E), torch.tensor(counts))[torch.randperm(sum(counts), generator=g)].view(-1, 1)
    T = chosen.shape[0]
    logits = torch.full((T, E), -30.0).scatter_(1, chosen, 5.0)
    x = torch.randn(T, K, generator=g).bfloat16()
    w1 = (torch.randn(E, 2 * ff if gated else ff, K, generator=g) * K ** -0.5).bfloat16()
    w2 = (torch.randn(E, K, ff, generator=g) * ff ** -0.5).bfloat16()
    first, second = hip.prepare_expert_matrices(w1.to(DEV), gated), hip.prepare_expert_matrices(w2.to(DEV))
    r = hip.route_tokens(logits.to(DEV), E, 1, tile_rows=rows)
    assert r.tiles_in_use.item() * (ff // 128 if gated else ff // 256) > 12 * hip._num_cus
    got = hip.routed_experts(x.to(DEV), r, first, second, activation=act, gated=gated).float().cpu()
    for e in range(E):
        at = (chosen[:, 0] == e).nonzero()[:, 0]
        z = x[at].double() @ w1[e].double().T
        h = torch.nn.functional.silu(z[:, :ff]) * z[:, ff:] if gated else z.clamp(min=0) ** 2
        want = h @ w2[e].double().T
        # what lies between the products and the result are rounded to bfloat16: 2^-9 of a value each, the first as often as it is added
        bar = 2.0 ** -8 * want.abs() + 2.0 ** -8 * (h.abs() @ w2[e].double().abs().T)
        assert ((got[at].double() - want).abs() <= bar).all(), e


@pytest.mark.parametrize("T,E,top,ff,K", [(400, 3, 2, 128, 64), (700, 2, 1, 272, 192), (257, 1, 1, 64, 128), (900, 3, 3, 96, 96)])
def test_tiles_of_256_rows_are_as_those_of_128(T, E, top, ff, K):
    """The same sums in the same order, gated and activated, with factors on the sums, row-major matrices and rows of an odd number of
    32 values (the kernel beside it) among them."""
    hip = HipOps(torch.bfloat16, DEV)
    torch.manual_seed(T)
    x, logits = torch.randn(T, K, device=DEV).bfloat16(), torch.randn(T, E, device=DEV)
    for gated, act in ((True, "silu"), (False, "relu2")):
        w1 = (torch.randn(E, 2 * ff if gated else ff, K, device=DEV) * K ** -0.5).bfloat16()
        w2 = (torch.randn(E, K, ff, device=DEV) * ff ** -0.5).bfloat16()
        for a, b in ((hip.prepare_expert_matrices(w1, gated), hip.prepare_expert_matrices(w2)), (w1, w2)):
            for weigh in (False, True):
                r = [hip.route_tokens(logits, E, top, tile_rows=rows) for rows in (128, 256)]
                narrow, wide = (hip.routed_experts(x, q, a, b, activation=act, gated=gated, weigh_input=weigh) for q in r)
                assert torch.equal(narrow, wide)


# three and six rows an expert, some hundred in row tiles of each height
@pytest.mark.parametrize("T,rows", [(3, 16), (7, 16), (40, 16), (400, 16), (400, 128), (400, 256)])
@pytest.mark.parametrize("tiled", [True, False])
def test_every_gate_of_an_expert_is_its_sigmoid_times_itself(T, rows, tiled):
    """Rows of x that pick a column of the gate matrix, which holds every bfloat16 from -200 to 200 of 2^-20 and more; the second product hands
    its input on."""
    hip = HipOps(torch.bfloat16, DEV)
    size = 512
    halves = torch.arange(-32768, 32768).to(torch.int16).view(torch.bfloat16)
    halves = halves[(halves.float().abs() <= 200) & (halves.float().abs() >= 2.0 ** -20)]
    strong = halves[(halves < -80) & (halves >= -130)]                 # (in every column, so that the first three hold them too)
    gate = torch.empty(size, size, dtype=torch.bfloat16)
    gate[:len(strong)] = strong[:, None]
    rest = size - len(strong)
    gate[len(strong):] = halves.repeat(-(-rest * size // len(halves)))[:rest * size].view(size, rest).T
    assert len(strong) > 90 and set(gate.view(torch.int16).flatten().tolist()) == set(halves.view(torch.int16).tolist())
    up = torch.zeros_like(gate) + 1.5
    x = torch.zeros(T, size, device=DEV).bfloat16()
    x[torch.arange(T), torch.arange(T)] = 1
    first, second = torch.cat([gate, up])[None].to(DEV), torch.eye(size, device=DEV).bfloat16()[None]
    if tiled:
        first, second = hip.prepare_expert_matrices(first, True), hip.prepare_expert_matrices(second)
    r = hip.route_tokens(torch.zeros(T, 1, device=DEV), 1, 1, tile_rows=rows)
    got = hip.routed_experts(x, r, first, second).double().cpu()
    z = gate.double().T[:T]
    want = 1.5 * z / (1 + torch.exp(-z))
    assert got.isfinite().all()
    # two roundings to bfloat16, of what lies between the products and of the result; zero where e^-z is no float any more
    assert ((got - want).abs() <= 2.0 ** -7 * want.abs() + 2.0 ** -120).all()
    assert (got[z < -88.7229] == 0).all()
