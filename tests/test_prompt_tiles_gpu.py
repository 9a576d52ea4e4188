"""Products of prompts on workgroups that walk their tiles (gemm_rounds.h), where a workgroup takes several tiles, where a tile is
one chunk of K, and the activation at values that are not ordinary numbers."""
import ctypes

import pytest
import torch

from servelab_amd.kernels import HipOps, KernelError

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


# 261 and 348 tiles on 256 CUs, a number of tiles that eight does not divide, tiles of one, two and three chunks
@pytest.mark.parametrize("M,N,K", [(700, 22064, 64), (700, 22064, 192), (600, 32800, 128)])
@pytest.mark.parametrize("rows", [128, 192, 256])
def test_workgroups_walk_several_tiles(M, N, K, rows):
    ops = HipOps(torch.bfloat16, DEV)
    assert -(-M // rows) * -(-N // 256) > ops._num_cus
    g = torch.Generator().manual_seed(K)
    x, w = torch.randn(M, K, generator=g).bfloat16(), (torch.randn(N, K, generator=g) * K ** -0.5).bfloat16()
    z = x.double() @ w.double().T
    ops.TILE_US = {rows: ops.TILE_US[rows]}
    parts = ops.linear_block(x.to(DEV), w.to(DEV), None, ks=1, partial=True, square=True).parts[0]
    # float sums of K terms: K 2^-24 of their absolute sum
    bar = K * 2.0 ** -24 * (x.double().abs() @ w.double().abs().T)
    assert ((parts.double().cpu() - z).abs() <= bar).all()
    half = ops.linear_block(x.to(DEV), w.to(DEV), None, square=True)
    assert torch.equal(half, parts.bfloat16())
    pair = z.view(M, N // 16, 2, 8)
    want = (torch.nn.functional.silu(pair[:, :, 0]) * pair[:, :, 1]).reshape(M, N // 2)
    got = ops.linear_gated_block(x.to(DEV), ops.prepare_weight(w.to(DEV)), None, rows, 1)
    # one rounding to bfloat16, and the sums' error in the gate (whose slope is 1.1 at most) and in its up product
    size = bar.max().item() * 2.2 * z.abs().max().item()
    assert ((got.double().cpu() - want).abs() <= 2.0 ** -8 * want.abs() + size).all()


def test_gates_that_are_not_ordinary_numbers():
    ops = HipOps(torch.bfloat16, DEV)
    inf, nan = float("inf"), float("nan")
    gates = torch.tensor([inf, -inf, nan, 0.0, -0.0, 1e38, -1e38, 1e-40, -80.0, -87.0, -100.0, 100.0, 20.0, -20.0, 1.0, -1.0])
    ups = torch.tensor([1.5, -2.0])
    N = 2 * len(gates) * 16
    bias = torch.empty(N // 16, 2, 8)
    bias[:, 0] = gates.repeat(2)[:, None]
    bias[:, 1] = ups.repeat_interleave(len(gates))[:, None]
    x, w = torch.zeros(8, 64, device=DEV).bfloat16(), torch.zeros(N, 64, device=DEV).bfloat16()
    got = ops.linear_gated_block(x, ops.prepare_weight(w), bias.view(-1).to(DEV), 256, 1).view(8, N // 16, 8)[3, :, 5].double().cpu()
    want = (torch.nn.functional.silu(gates).double()[None] * ups[:, None]).view(-1)
    assert torch.equal(got.isnan(), want.isnan())
    keep = ~want.isnan() & want.isfinite()
    # one rounding to bfloat16; results below the smallest normal float may be zero
    assert ((got - want).abs()[keep] <= 2.0 ** -8 * want.abs()[keep] + 2.0 ** -125).all()
    assert torch.equal(got[want.isinf()], want[want.isinf()])


def gates_to_sweep():
    """Every bfloat16 from -200 to 200 of 2^-20 and more, floats closely around where e^-z passes the largest float and its half, and
    between."""
    halves = torch.arange(-32768, 32768).to(torch.int16).view(torch.bfloat16).float()
    halves = halves[(halves.abs() <= 200) & (halves.abs() >= 2.0 ** -20)]
    near = [(torch.tensor(z).view(torch.int32) + torch.arange(-300, 300, dtype=torch.int32)).view(torch.float32)
            for z in (-88.7228394, -88.0296936, -87.3365479)]
    return torch.cat([halves, *near, torch.linspace(-131.0, -79.0, 4001), -torch.logspace(2.0, 38.5, 200)])


@pytest.mark.parametrize("rows", [128, 192, 256])
def test_every_gate_is_its_sigmoid_times_itself(rows):
    ops = HipOps(torch.bfloat16, DEV)
    gates = gates_to_sweep()
    gates = torch.cat([gates, gates.new_ones(-len(gates) % 8)])
    N = 2 * len(gates)
    bias = torch.full((N // 16, 2, 8), 1.5)
    bias[:, 0] = gates.view(-1, 8)
    x, w = torch.zeros(3, 64, device=DEV).bfloat16(), torch.zeros(N, 64, device=DEV).bfloat16()
    got = ops.linear_gated_block(x, ops.prepare_weight(w), bias.view(-1).to(DEV), rows, 1).double().cpu()
    z = gates.double()
    want = 1.5 * z / (1 + torch.exp(-z))
    assert got.isfinite().all()
    # one rounding to bfloat16; below -88.72, where e^-z is no float any more, the result is zero instead of 1.5 x 2.6e-37 at most
    assert ((got - want).abs() <= 2.0 ** -8 * want.abs() + 2.0 ** -120).all()
    below = z < -88.7229
    assert below.sum() > 1000 and (got[:, below] == 0).all()


def test_routes_by_estimated_rate():
    ops = HipOps(torch.bfloat16, DEV)
    tiles = ops._prompt_tiles
    # well filled rounds, in the height that takes less time; part-filled ones stay with the library
    assert [tiles(M, 37888, 3584) for M in (260, 400, 527, 1000, 2048, 2560)] == [None, 192, 192, 256, 256, 256]
    assert [tiles(M, 22016, 2048) for M in (400, 527, 640, 768)] == [256, 128, 128, 192]
    assert [tiles(M, 9216, 3584) for M in (527, 640, 900, 1536)] == [None, 128, 192, 256]
    assert tiles(255, 37888, 3584) is None and tiles(2561, 37888, 3584) is None and tiles(2048, 37888, 3600) is None
    assert tiles(2048, 4080, 3584) is None and tiles(2048, 37888, 8256) is None
    # either height gives the same sums
    x = torch.randn(527, 512, device=DEV).bfloat16()
    w = (torch.randn(22016, 512, device=DEV) * 0.05).bfloat16()
    weight = ops.prepare_weight(w)
    whole = ops.linear_gated_block(x, weight, None, 256, 1)
    assert torch.equal(ops.linear_gated_block(x, weight, None, 192, 1), whole) and torch.equal(ops.linear_gated_block(x, weight, None, 128, 1), whole)


# ragged rows of x and of W, both heights
@pytest.mark.parametrize("M,N,K,act", [(300, 4112, 128, "relu2"), (257, 1000, 192, "silu"), (385, 264, 64, "gelu_tanh"), (193, 520, 64, "relu")])
@pytest.mark.parametrize("rows", [128, 192, 256])
def test_activation_of_the_sums(M, N, K, act, rows):
    ops = HipOps(torch.bfloat16, DEV)
    g = torch.Generator().manual_seed(M)
    x, w = torch.randn(M, K, generator=g).bfloat16(), (torch.randn(N, K, generator=g) * K ** -0.5).bfloat16()
    b = torch.randn(N, generator=g)
    z = x.double() @ w.double().T + b.double()
    want = {"relu2": lambda t: t.clamp(min=0) ** 2, "relu": lambda t: t.clamp(min=0), "silu": torch.nn.functional.silu,
            "gelu_tanh": lambda t: torch.nn.functional.gelu(t, approximate="tanh")}[act](z)
    code = {"silu": 1, "relu": 2, "relu2": 3, "gelu_tanh": 4}[act]
    weight = ops.prepare_weight(w.to(DEV))
    got = ops.linear_activated_block(x.to(DEV), weight, b.to(DEV), rows, code)
    # one rounding to bfloat16; float sums of K terms: K 2^-24 of their absolute sum, times the activation's slope there
    size = K * 2.0 ** -24 * (x.double().abs() @ w.double().abs().T + b.double().abs())
    slope = 2 * z.abs() + size if act == "relu2" else 1.2
    assert ((got.double().cpu() - want).abs() <= 2.0 ** -8 * want.abs() + slope * size + 2.0 ** -20).all()


def test_activated_prompts_take_the_tiles():
    ops = HipOps(torch.bfloat16, DEV)
    w = (torch.randn(18944, 256, device=DEV) * 0.06).bfloat16()
    weight = ops.prepare_weight(w)
    x = torch.randn(1852, 256, device=DEV).bfloat16()
    ops.PROMPT_MIN_TFLOPS = 100.0                # (short rows: an estimated rate of 480 TFLOP/s)
    assert ops._prompt_tiles(1852, 18944, 256)
    got = ops.activated_linear(x, weight, "relu2")
    assert torch.equal(got, ops.linear_activated_block(x, weight, None, 256, 3))
    odd = torch.empty(x.numel() + 1, device=DEV, dtype=x.dtype)[1:].view(x.shape).copy_(x)
    plain = ops.activated_linear(odd, weight, "relu2")
    # (the library's product is rounded before the square as well)
    assert ((plain.float() - got.float()).abs() <= 2.0 ** -6 * got.float().abs() + 2.0 ** -12).all()


def test_tuned_shapes_whose_tiles_are_faster_still():
    ops = HipOps(torch.bfloat16, DEV)
    rate = lambda M, N, K: 2e-6 * M * N * K / ops._tiles_us(ops._tile_rows(M, N, K), M, N, K)
    shape, small = (2048, 37888, 3584), (1700, 8192, 1024)
    assert rate(*shape) > ops.PROMPT_TUNED_TFLOPS > rate(*small)
    assert ops._tiles_beat_tuned(*shape) and ops._tiles_beat_tuned(*small)                # (nothing was tuned)
    ops._tuned = {shape, small}
    assert ops._tiles_beat_tuned(*shape) and not ops._tiles_beat_tuned(*small)
    ops._tuned, ops._tuning = set(), True
    assert ops._tiles_beat_tuned(*shape) and not ops._tiles_beat_tuned(*small)


def test_products_that_the_wide_tiles_cannot_take():
    """Rows whose offsets pass 32 bits, and results that start 8 bytes past a multiple of 16: the tiles of 256 x 128 stand in."""
    ops = HipOps(torch.bfloat16, DEV)
    K = (1 << 22) + 64
    x, w = torch.randn(2, K, device=DEV).bfloat16(), torch.randn(8, K, device=DEV).bfloat16()
    got = ops.linear_block(x, w, None, ks=1, partial=True, square=True).parts[0].double()
    want, size = x.double() @ w.double().T, x.double().abs() @ w.double().abs().T
    # 131,074 additions in a row, each off by 2^-24 of the absolute sum at most: 2^-15.5 of it as a random walk, 2^-13 with room
    assert ((got - want).abs() <= 2.0 ** -13 * size).all()
    x, w = torch.randn(257, 128, device=DEV).bfloat16(), torch.randn(264, 128, device=DEV).bfloat16()
    y = torch.zeros(257 * 264 + 4, device=DEV).bfloat16()[4:].view(257, 264)
    assert y.data_ptr() % 16 == 8
    ops._call("gemm", "sl_gemm_block", *(ctypes.c_void_p(v.data_ptr()) for v in (x, w)), None, ctypes.c_void_p(y.data_ptr()),
              257, 264, 128, 0, 0, 0, 1, 256, None)
    assert torch.equal(y, ops.linear_block(x, w, None))
    with pytest.raises(KernelError, match="16 bytes"):
        ops._call("gemm", "sl_gemm_block", *(ctypes.c_void_p(v.data_ptr()) for v in (x, w)), None, ctypes.c_void_p(y.data_ptr()),
                  257, 264, 128, 0, 0, 3, 1, 256, None)
