"""The float32 table's products and prompt attention at the sizes where their forms can go wrong, against float64."""
import pytest
import torch

from servelab_amd.kernels import HipOps
from test_kernels_gpu import make_attention_case

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def relative(got, want):
    return float((got.double() - want).norm() / want.norm())


# two and four columns a workgroup (up to 2,048, up to 4,096 and more columns), rows of 1 to 8, columns that neither divides,
# K shorter than the workgroup's step of 1,024 values and not a multiple of it
@pytest.mark.parametrize("M", [1, 2, 3, 4, 5, 8])
@pytest.mark.parametrize("N,K", [(1, 4), (7, 1028), (2048, 252), (2051, 2052), (4097, 1536), (4099, 2048)])
def test_few_rows(M, N, K):
    ops = HipOps(torch.float32, DEV)
    g = torch.Generator().manual_seed(M + N)
    x, w, b = torch.randn(M, K, generator=g).to(DEV), torch.randn(N, K, generator=g).to(DEV), torch.randn(N, generator=g).to(DEV)
    got = ops.linear_rows(x, w, b, False)
    # 256 running sums of K / 256 products each, added in pairs: far below 2^-24 sqrt(K) of a result
    assert relative(got, x.double() @ w.double().T + b.double()) < 1e-6


# rows of 32 and of 128 a tile, one share and several, a last share with what no segment of 512 divides, odd columns
@pytest.mark.parametrize("M,N,K", [(17, 40, 528), (64, 256, 1552), (65, 130, 2048), (300, 133, 8960), (849, 1536, 1536), (70, 128, 496)])
def test_products_in_shares_of_k(M, N, K):
    ops = HipOps(torch.float32, DEV)
    g = torch.Generator().manual_seed(M + N)
    x, w, b = torch.randn(M, K, generator=g).to(DEV), torch.randn(N, K, generator=g).to(DEV), torch.randn(N, generator=g).to(DEV)
    want = x.double() @ w.double().T + b.double()
    errors = {}
    for shares in sorted({1, ops._f32_shares(M, N, K), -(-K // 512)}):
        ops._f32_shares = lambda *_: shares
        errors[shares] = relative(ops.linear_f32_mfma(x, w, b), want)
    # running sums of 512 products: 2^-24 sqrt(512) of a result; shares only shorten the chain of their sums
    assert max(errors.values()) < 1.4e-6 and all(e <= 1.05 * errors[1] for e in errors.values())


@pytest.mark.parametrize("nh,nkv,D", [(12, 2, 128), (14, 2, 64), (4, 4, 64), (8, 1, 128)])
@pytest.mark.parametrize("page,window", [(16, None), (32, 40), (64, 5)])
def test_prompt_attention_on_the_matrix_cores(nh, nkv, D, page, window):
    """Portions that start at zero and deep in their contexts, of one tile of 64 columns and several, ending inside a block of
    32 keys and at its end; single tokens behind them take the other kernels."""
    from emulated_ops import EmulatedOps
    ops, emu = HipOps(torch.float32, DEV), EmulatedOps(torch.float32)
    qkv, kc, vc, tables, batch = make_attention_case(torch.float32, nh, nkv, D, page, [(33, 33), (72, 2), (63, 32), (95, 90), (300, 40), (65, 1)])[:5]
    got = ops.paged_attention(qkv, nh, nkv, D, kc, vc, page, tables, batch, D ** -0.5, window)
    host = emu_batch(batch)
    want = emu.paged_attention(qkv.cpu(), nh, nkv, D, kc.cpu(), vc.cpu(), page, tables.cpu(), host, D ** -0.5, window)
    # float32 scores of 128 products and sums over at most 300 keys on both sides
    assert float((got.cpu() - want).abs().max()) <= 2e-6 * max(1.0, float(want.abs().max()))


@pytest.mark.parametrize("nh,nkv,D", [(12, 2, 128), (4, 4, 64)])
@pytest.mark.parametrize("window", [None, 9])
@pytest.mark.parametrize("value", [float("inf"), float("nan")])
def test_prompt_attention_beside_values_that_are_not_finite(nh, nkv, D, window, value):
    """One key's value at position 50 reaches the tokens that see it, in its kv head and channel, and no other result."""
    ops, page = HipOps(torch.float32, DEV), 16
    lens = [(72, 72), (40, 40)]
    qkv, kc, vc, tables, batch = make_attention_case(torch.float32, nh, nkv, D, page, lens)[:5]
    run = lambda: ops.paged_attention(qkv, nh, nkv, D, kc, vc, page, tables, batch, D ** -0.5, window).view(-1, nh, D)
    want = run()
    vc[int(tables[0, 50 // page]), 0, 3, 50 % page] = value
    got = run()
    reached = torch.zeros_like(want, dtype=torch.bool)
    reached[50:72 if window is None else 50 + window, :nh // nkv, 3] = True
    assert torch.equal(~torch.isfinite(got), reached)
    # the same products in another order of sums over at most 72 keys
    assert float((got - want)[~reached].abs().max()) <= 2e-6 * max(1.0, float(want.abs().max()))


def emu_batch(batch):
    import copy
    host = copy.copy(batch)
    for name, value in vars(batch).items():
        if torch.is_tensor(value):
            setattr(host, name, value.cpu())
    return host


def test_shares_cost_what_the_longest_one_takes():
    ops = HipOps(torch.float32, DEV)
    assert ops._f32_shares(512, 9728, 896) == 1                # two segments of 512 and 384 terms: as long as three rounds of 512
    assert ops._f32_shares(849, 1536, 8960) > 1 and ops._f32_shares(64, 256, 512) == 1


# rows that end a tile of 128 and pass it by one, odd columns, one chunk of 32, a chunk past a segment of 512, a last share of one chunk
@pytest.mark.parametrize("M,N,K", [(65, 1, 32), (128, 127, 544), (129, 130, 1056), (255, 129, 96), (1025, 1100, 64)])
def test_products_in_chunks_of_32(M, N, K):
    ops = HipOps(torch.float32, DEV)
    g = torch.Generator().manual_seed(M)
    x, w, b = torch.randn(M, K, generator=g), torch.randn(N, K, generator=g), torch.randn(N, generator=g)
    want, size = x.double() @ w.double().T + b.double(), x.double().abs() @ w.double().abs().T + b.double().abs()
    for shares in {1, -(-K // 512)}:
        ops._f32_shares = lambda *_: shares
        got = ops.linear_f32_mfma(x.to(DEV), w.to(DEV), b.to(DEV)).cpu()
        # running sums of up to 512 products: no further off than 512 roundings of 2^-24 of their absolute sum
        assert ((got.double() - want).abs() <= min(K, 512) * 2.0 ** -24 * size).all()


# two row tiles of 256 to 385 column tiles: whole rounds of two workgroups a CU, one tile more, at most one a CU and one more than that
@pytest.mark.parametrize("columns", [256, 257, 384, 385])
@pytest.mark.parametrize("K,shares", [(96, 1), (544, 1), (544, 2)])
def test_products_around_rounds_of_tiles(columns, K, shares):
    ops = HipOps(torch.float32, DEV)
    M, N = 129, columns * 128 // shares - 1
    g = torch.Generator().manual_seed(columns)
    x, w, b = torch.randn(M, K, generator=g).to(DEV), torch.randn(N, K, generator=g).to(DEV), torch.randn(N, generator=g).to(DEV)
    ops._f32_shares = lambda *_: shares
    got = ops.linear_f32_mfma(x, w, b).double()
    want, size = x.double() @ w.double().T + b.double(), x.double().abs() @ w.double().abs().T + b.double().abs()
    # running sums of up to 512 products: no further off than 512 roundings of 2^-24 of their absolute sum
    assert ((got - want).abs() <= min(K, 512) * 2.0 ** -24 * size).all()


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("nh,nkv,D", [(12, 2, 128), (14, 2, 64), (20, 2, 64), (2, 1, 128)])
@pytest.mark.parametrize("page,window", [(16, None), (32, 40), (64, 5)])
def test_single_tokens_in_blocks_of_16_keys(dtype, nh, nkv, D, page, window):
    """One key and one more or less than a block, a page and a share of several blocks; more heads than a wavefront takes; what lies
    behind a sequence's last key may be no number."""
    from emulated_ops import EmulatedOps
    ops, emu = HipOps(dtype, DEV), EmulatedOps(dtype)
    ops.use_mfma_attention = False
    lengths = [1, 16, 17] if nh == 20 else [1, 15, 1100, 65]
    qkv, kc, vc, tables, batch = make_attention_case(dtype, nh, nkv, D, page, [(n, 1) for n in lengths])[:5]
    ops.GENERAL_ATTENTION_WAVES = 1024                         # (as many wavefronts as have a SIMD to themselves)
    host = emu_batch(batch)
    want = emu.paged_attention(qkv.cpu(), nh, nkv, D, kc.cpu(), vc.cpu(), page, tables.cpu(), host, D ** -0.5, window)
    for i, n in enumerate(lengths):                            # the unused places of each last page
        last = int(tables[i, (n - 1) // page])
        kc[last, :, (n - 1) % page + 1:], vc[last, :, :, (n - 1) % page + 1:] = float("nan"), float("inf")
    got = ops.paged_attention(qkv, nh, nkv, D, kc, vc, page, tables, batch, D ** -0.5, window)
    # float32 scores of 128 products and sums over at most 1,100 keys; bfloat16: one rounding
    assert float((got.float().cpu() - want.float()).abs().max()) <= (3e-6 if dtype == torch.float32 else 2.0 ** -7) * max(1.0, float(want.abs().max()))


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("D,unseen", [(64, [(0, 16)]), (128, [(0, 48)]), (64, [(16, 32), (96, 112)])])
def test_single_tokens_with_blocks_of_keys_that_weigh_nothing(dtype, D, unseen):
    """Scores of minus infinity for whole blocks of 16 keys, the first of a share among them: they weigh nothing."""
    ops = HipOps(dtype, DEV)
    ops.use_mfma_attention, ops.GENERAL_ATTENTION_WAVES = False, 1024
    nh, nkv, n = 4, 2, 250
    qkv, kc, vc, tables, batch = make_attention_case(dtype, nh, nkv, D, 16, [(n, 1)])[:5]
    qkv[0, :nh * D:D] = 1.0
    keys, values = kc[tables[0].long()].transpose(1, 2).reshape(-1, nkv, D), vc[tables[0].long()].permute(0, 3, 1, 2).reshape(-1, nkv, D)
    for first, behind in unseen:
        for k in range(first, behind):
            kc[int(tables[0, k // 16]), :, k % 16, 0] = float("-inf")
            keys[k, :, 0] = float("-inf")
    got = ops.paged_attention(qkv, nh, nkv, D, kc, vc, 16, tables, batch, D ** -0.5, None).double().cpu()
    q = qkv[0, :nh * D].double().cpu().view(nkv, nh // nkv, D)
    scores = torch.einsum("ghd,kgd->ghk", q, keys[:n].double().cpu()) * D ** -0.5
    want = torch.einsum("ghk,kgd->ghd", scores.softmax(-1), values[:n].double().cpu()).reshape(1, nh * D)
    # float32 scores of 128 products and sums over at most 250 keys; bfloat16: one rounding
    assert float((got - want).abs().max()) <= (3e-6 if dtype == torch.float32 else 2.0 ** -7) * max(1.0, float(want.abs().max()))
