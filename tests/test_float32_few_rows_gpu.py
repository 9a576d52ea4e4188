"""float32 products of three to sixteen rows on the matrix units, at the edges of their forms, against sums in 64 bits."""
import pytest
import torch

from servelab_amd.kernels import HipOps

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


# rows of each form, the last of a block of four and the first of the next, and a second sixteen; columns that no wavefront's divide, each line of the choice of
# form and its other side; K shorter than a step of 64 and than the parts of K, not a multiple of it, long
@pytest.mark.parametrize("M", [3, 4, 5, 8, 9, 16, 19])
@pytest.mark.parametrize("N,K", [(1, 4), (6, 64), (1023, 3072), (1029, 3076), (2051, 3140), (2051, 8196), (4096, 196), (4099, 324), (16387, 260), (32771, 132), (32770, 2052)])
def test_sums(M, N, K):
    ops = HipOps(torch.float32, DEV)
    g = torch.Generator(device=DEV).manual_seed(M + N)
    x, w, b = (torch.randn(*s, generator=g, device=DEV) for s in ((M, K), (N, K), (N,)))
    bar = K * 2.0 ** -24 * (x.double().abs() @ w.double().abs().T)          # float sums of K products, rounded once a term at most
    want = x.double() @ w.double().T
    assert ((ops.linear_rows(x, w, None).double() - want).abs() <= bar).all()
    got = ops.linear_rows(x, w, b).double()
    assert ((got - want - b.double()).abs() <= bar + 2.0 ** -24 * got.abs()).all()


# the last columns in fours and the first beyond; few columns of short rows; up to four long rows as FMAs, and what lies around them
@pytest.mark.parametrize("M", [3, 4, 5])
@pytest.mark.parametrize("N,K", [(1024, 3076), (1025, 3076), (768, 68), (769, 1028), (768, 512), (768, 508), (1025, 6144), (1536, 6148), (1537, 6148), (1536, 6140)])
def test_sums_at_the_lines_of_few_columns(M, N, K):
    test_sums(M, N, K)


@pytest.mark.parametrize("M", [3, 7, 12])
def test_what_a_value_reaches(M):
    """NaN and infinities of a row of x or of W stay in that row and that column, also where a step passes the end of K."""
    ops = HipOps(torch.float32, DEV)
    N, K = 70, 100
    x, w = torch.ones(M, K, device=DEV), torch.ones(N, K, device=DEV)
    x[M - 1, 0] = float("inf")
    w[N - 1, 0] = float("nan")
    y = ops.linear_rows(x, w, None)
    assert (y[:M - 1, :N - 1] == K).all() and torch.isinf(y[M - 1, :N - 1]).all() and torch.isnan(y[:, N - 1]).all()
