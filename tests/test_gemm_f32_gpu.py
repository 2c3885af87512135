"""-m gpu: the layer lists' 32-bit products (csrc/kernels_gemm_f32.hip) one by one against 64 bits."""
import numpy as np
import pytest
import torch

from aha_amd._lib import check, lib

pytestmark = pytest.mark.gpu

# The weights are bf16 and an f32 activation is the sum of its three bf16 parts, so nothing is lost but in the f32 sums: 1 to 4e-7 of the results' spread.
# Without the third part every row is off by 0.6 to 1.4e-5 of it at K = 64 to 3072 (computed with the part left out, in 64 bits), without the second by 2.5 to 4.2e-3.
# In between:
BOUND = 1e-6


def product(gpu, A, W):
    """A (batch, M, K) f32, W (batch, N, K) bf16"""
    b, M, K = A.shape
    N = W.shape[1]
    Ad, Wd = A.to(gpu), W.to(gpu)
    C = torch.full((b * M * N + 8,), 7.0, device=gpu)
    check(lib().aha_hip_debug_gemm_f32(Ad.data_ptr(), Wd.data_ptr(), C.data_ptr(), M, N, K, b, torch.cuda.current_stream().cuda_stream))
    C = C.cpu()
    assert (C[b * M * N:] == 7.0).all()
    return C[:b * M * N].view(b, M, N)


def inputs(b, M, N, K, seed=3):
    g = torch.Generator().manual_seed(seed)
    return torch.randn(b, M, K, generator=g), (torch.randn(b, N, K, generator=g) * K ** -0.5).bfloat16()


# rows, columns, batch: every form that launch_gemm_f32 chooses between
FORMS = {
    "16 weight rows, 8 rows": (7, 324, 1), "16 weight rows, 16 rows": (16, 1000, 1), "16 weight rows, 32 rows": (27, 324, 1), "48 weight rows, 8 rows": (8, 24600, 1),
    "48 weight rows, 16 rows": (9, 24600, 1), "a batch of few rows": (2, 128, 5),
    "16 x 64, four chunks": (33, 324, 1), "32 x 64, four chunks": (150, 2624, 1), "32 x 64, two chunks": (300, 2624, 1), "32 x 64, two chunks, few rows": (20, 24600, 1),
    "64 x 64, one chunk": (500, 2624, 1), "a batch of tiles": (70, 192, 9), "no whole pieces": (37, 323, 1),
}


@pytest.mark.parametrize("form", FORMS)
@pytest.mark.parametrize("K", [64, 320, 1088])
def test_nothing_of_an_activation_is_lost(gpu, form, K):
    M, N, b = FORMS[form]
    A, W = inputs(b, M, N, K)
    want = A.double() @ W.double().transpose(1, 2)
    d = (product(gpu, A, W).double() - want) / want.std()
    assert float(d.pow(2).mean(-1).sqrt().max()) < BOUND and float(d.abs().max()) < 8 * BOUND


@pytest.mark.parametrize("M,N", [(5, 324), (40, 324), (300, 2624), (500, 2624)])
def test_a_deep_product(gpu, M, N):
    A, W = inputs(1, M, N, 3072)
    want = A.double() @ W.double().transpose(1, 2)
    d = (product(gpu, A, W).double() - want) / want.std()
    assert float(d.pow(2).mean(-1).sqrt().max()) < BOUND


@pytest.mark.parametrize("form", FORMS)
def test_activations_that_are_not_finite_or_at_the_ends_of_the_range(gpu, form):
    """An infinity's lower parts are inf - inf: the result is the infinity all the same, as one f32 product gives it, NaN only where that gives NaN, and no other row sees any
    of it.  The largest floats do not round up to an infinity on the way, and small ones keep their bits."""
    M, N, b = FORMS[form]
    A, W = inputs(b, M, N, 320, seed=4)
    inf = float("inf")
    W[:, 1, 17] = 0.0
    A[-1, 0, 17] = inf                    # an infinity, times zero in column 1
    if M > 1:
        A[-1, 1, 17], A[-1, 1, 200] = -inf, 3.0
    if M > 2:
        A[-1, 2, 5], A[-1, 2, 300] = inf, float("nan")
    if M > 4:
        A[-1, 3] = torch.where(torch.arange(320) == 40, 3.4028234e38, 0.0)
        A[-1, 4] *= 2.0 ** -100
    got = product(gpu, A, W)
    want = A.double() @ W.double().transpose(1, 2)
    rows = np.ones((b, M), dtype=bool)
    rows[-1, :min(M, 5)] = False
    assert float((got.double() - want)[torch.from_numpy(rows)].abs().max() / want[torch.from_numpy(rows)].std()) < 8 * BOUND
    for r in range(min(M, 3)):
        assert torch.equal(torch.isnan(got[-1, r]), torch.isnan(want[-1, r]))
        ok = ~torch.isnan(want[-1, r])
        assert torch.equal(got[-1, r][ok].double(), want[-1, r][ok])      # (every column: an infinity or NaN)
    for r in range(3, min(M, 5)):
        d = (got[-1, r].double() - want[-1, r]) / want[-1, r].std()
        assert torch.isfinite(got[-1, r]).all() and float(d.abs().max()) < 8 * BOUND
