"""Float32 products of three bfloat16 terms an operand: both widths of a workgroup at the edges of tiles, chunks and shares, values of
sizes from the least on, and operands that are not finite."""
import pytest
import torch

from servelab_amd.kernels import HipOps

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def draws(M, N, K, spread):
    """Values whose sizes are spread over 2^-spread .. 2^spread."""
    g = torch.Generator(device=DEV).manual_seed(M + N + K)
    x, w = torch.randn(M, K, generator=g, device=DEV), torch.randn(N, K, generator=g, device=DEV)
    two = lambda *s: torch.exp2((torch.rand(s, generator=g, device=DEV) * 2 - 1) * spread)
    return x * two(M, K), w * two(N, K)


# a row and a column past a tile of 128, past one of 256 (the wide form where many tiles fill the CUs), the rows of one chunk that float32 instructions
# take, rows below a segment of 512, a whole one, a chunk past a segment of 512, a last share of one chunk
@pytest.mark.parametrize("M,N,K", [(129, 129, 32), (129, 129, 480), (129, 129, 512), (70, 257, 544), (900, 8193, 608), (1025, 8191, 1056), (128, 256, 1536)])
@pytest.mark.parametrize("spread", [0, 12])
def test_sums_of_terms(M, N, K, spread):
    ops = HipOps(torch.float32, DEV)
    x, w = draws(M, N, K, spread)
    want, size = x.double() @ w.double().T, x.double().abs() @ w.double().abs().T
    for shares in {1, -(-K // 512)}:
        ops._f32_shares = lambda *_: shares
        got = ops.linear_f32_mfma(x, w, None).double()
        # six roundings of the running sum a chunk of 32, at most 16 chunks a sum, the sums' own, and 2^-26 of every product left out
        bar = (6 * min(K // 32, 16) + K // 512 + 2) * 2.0 ** -24 + 2.0 ** -26
        assert ((got - want).abs() <= bar * size).all()


# whole pairs of runs of eight chunks; one chunk more, and two; runs behind the last pair, of even and odd numbers of chunks; a share of its own for them
@pytest.mark.parametrize("K,shares", [(512, 1), (1024, 2), (544, 1), (576, 2), (608, 1), (672, 1), (768, 1), (768, 2), (896, 1), (1280, 1), (1280, 3)])
def test_sums_lie_on_neither_side(K, shares):
    """The matrix unit rounds sums down; that cancels only where as many chunks are summed with either sign."""
    ops = HipOps(torch.float32, DEV)
    ops._f32_shares = lambda *_: shares
    x, w = draws(1024, 2048, K, 0)
    want = x.double() @ w.double().T
    off, spread = ops.linear_f32_mfma(x, w, None).double() - want, want.square().mean().sqrt()
    # float32 instructions are 3.7e-7 to 4.1e-7 off here, and two terms an operand instead of three 4e-6
    assert off.norm() / want.norm() <= 3.2e-7
    # The mean over 2 M results, which share 3,072 rows: 3e-10 at whole pairs of runs (float32 instructions: 6e-10 at most).  A run of two chunks
    # more of one sign than of the other is 1.3e-9.
    assert abs(off.mean() / spread) <= 9e-10


@pytest.mark.parametrize("K,bar", [(64, 1.35e-7), (96, 1.5e-7), (128, 1.75e-7), (480, 3.0e-7)])
def test_short_rows(K, bar):
    """Three terms an operand from 64 values of k on: closer than float32 instructions, which are 1.44e-7, 1.77e-7, 2.03e-7 and 3.93e-7 off here."""
    ops = HipOps(torch.float32, DEV)
    x, w = draws(1024, 2048, K, 0)
    want = x.double() @ w.double().T
    off = ops.linear_f32_mfma(x, w, None).double() - want
    assert off.norm() / want.norm() <= bar
    assert abs(off.mean()) <= 0.012 * off.square().mean().sqrt()              # (an odd chunk: 1 % of it)


# sizes whose third term, second and first lie below the least bfloat16, subnormal floats, the least ones
@pytest.mark.parametrize("M,N,K", [(130, 300, 1056), (1024, 8192, 512)])
@pytest.mark.parametrize("e", [-112, -118, -126, -135, -142, -148])
def test_operands_of_the_least_sizes(M, N, K, e):
    ops = HipOps(torch.float32, DEV)
    x, w = draws(M, N, K, 0)
    small = lambda t: t * 2.0 ** -74 * 2.0 ** (e + 74)
    for a, b in ((small(x), w * 2.0 ** 40), (x * 2.0 ** 40, small(w))):
        want = a.double() @ b.double().T
        # no further off than at ordinary sizes: 2.4e-7 to 2.6e-7 there
        assert (ops.linear_f32_mfma(a, b, None).double() - want).norm() / want.norm() <= 3.2e-7


def test_both_widths_are_chosen():
    ops = HipOps(torch.float32, DEV)
    lib = ops._lib["gemm"]
    import ctypes
    lib.sl_gemm_f32_split_us.restype = ctypes.c_float
    assert ops._f32_shares(849, 1536, 8960) > 1
    # the estimate of one round of wide tiles on every CU lies below two of narrow ones, that of half as many tiles above one of them
    full, half = lib.sl_gemm_f32_split_us(1024, 8192, 1536, 1, 256), lib.sl_gemm_f32_split_us(512, 8192, 1536, 1, 256)
    assert full == 8 + 48 * 2.5 and abs(half - (6 + 48 * 1.48)) < 1e-3
    assert lib.sl_gemm_f32_split_us(512, 8192, 1536, 1, 0) == 0


@pytest.mark.parametrize("M,N,K,shares", [(130, 300, 1056, 1), (130, 300, 1056, 3), (1024, 8192, 512, 1)])
def test_operands_that_are_not_finite_or_hardly(M, N, K, shares):
    ops = HipOps(torch.float32, DEV)
    ops._f32_shares = lambda *_: shares
    x, w = draws(M, N, K, 0)
    w *= 2.0 ** -8
    clean = x.double() @ w.double().T
    x[5, 7], x[6, 8], x[70, 0] = float("inf"), float("-inf"), 3.4e38          # (the last is past the largest bfloat16)
    w[3, 9], w[200, 11] = float("nan"), float("inf")
    w[:, 7][4], w[9, 8] = 0.5, 0.0                                            # exact in one term; infinity times zero
    want = x.double() @ w.double().T
    got = ops.linear_f32_mfma(x, w, None)
    assert torch.equal(torch.isnan(got), torch.isnan(want)) and torch.equal(torch.isposinf(got), torch.isposinf(want))
    assert torch.equal(torch.isneginf(got), torch.isneginf(want))
    there = torch.isfinite(want)
    size = torch.where(torch.isfinite(x), x, 0).double().abs() @ torch.where(torch.isfinite(w), w, 0).double().abs().T
    assert ((got.double() - want).abs()[there] <= (K * 2.0 ** -24 * size)[there]).all() and there.sum() > 0.9 * clean.numel()


def test_results_that_are_not_finite_take_no_time_to_speak_of():
    """A NaN early in a prompt makes every product behind it end in NaN: one row, and all of them."""
    ops = HipOps(torch.float32, DEV)
    x, w = draws(849, 1536, 1536, 0)
    ops._f32_shares = lambda *_: 1
    clean = ops.linear_f32_mfma(x, w, None)

    def us():
        best = float("inf")
        for _ in range(5):
            a, b = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
            a.record()
            for _ in range(4):
                y = ops.linear_f32_mfma(x, w, None)
            b.record()
            torch.cuda.synchronize()
            best = min(best, a.elapsed_time(b) * 250)
        return best, y
    finite, _ = us()
    x[5, 7] = float("nan")
    one, y = us()
    assert torch.isnan(y[5]).all() and torch.equal(torch.cat([y[:5], y[6:]]), torch.cat([clean[:5], clean[6:]]))
    x[:, 7] = float("nan")
    all_rows, y = us()
    assert torch.isnan(y).all()
    # float32 instructions, at two and a half times the matrix units' time, behind the product; a lane a result took 8 and 90 times it
    assert one < 4 * finite and all_rows < 8 * finite, (finite, one, all_rows)
