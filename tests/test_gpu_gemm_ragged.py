"""mg_gemm_i8 on operands in place: any K and N, rows and bases of any alignment, products small enough for the 32 x 32
kernel and large enough for the 64 x 128 one (the boundary is 64 tiles of the latter), int32 and fp32 outputs alone and
together, all exact against integer arithmetic."""
import numpy as np
import pytest

from mignon_ai_amd import gemm_i8_device

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")


@pytest.mark.parametrize("M,K,N", [
    (1, 1, 1), (1, 15, 33), (2, 1446, 308), (31, 17, 32), (33, 64, 31), (64, 65, 64), (5, 1152, 4096), (1, 128, 2000),
    (899, 67, 93), (4096, 100, 1024), (4032, 63, 127), (4033, 64, 128), (4033, 63, 129), (8128, 65, 127), (32768, 63, 127), (32768, 64, 128), (32705, 129, 130), (4133, 384, 1027),
    (2100, 191, 2111)])
@pytest.mark.parametrize("shift", [0, 1])
def test_ragged_exact(M, K, N, shift):
    rng = np.random.default_rng(M + K + N)

    def dev(x):  # `shift` elements into a larger buffer: a base address of any alignment
        flat = torch.empty(x.size + 64, dtype=torch.from_numpy(x[:0].ravel()).dtype, device="cuda")
        flat[shift:shift + x.size] = torch.from_numpy(x.ravel()).cuda()
        return flat[shift:shift + x.size].view(x.shape)

    A, W = rng.integers(-128, 128, (M, K), np.int8), rng.integers(-128, 128, (N, K), np.int8)
    s = (1e-3 + rng.random(N)).astype(np.float32)
    dA, dW, ds = dev(A), dev(W), dev(s)
    want = (dA.double() @ dW.double().T).round().to(torch.int32)  # exact: |sums| < 2^53
    wantf = want.float() * ds
    for want_c, want_acc in ((True, False), (False, True), (True, True)):
        pad = torch.full((M * N + 64,), 7, dtype=torch.int32, device="cuda")
        cpad = pad.clone().view(torch.float32)
        acc = pad[shift:shift + M * N].view(M, N) if want_acc else None
        C = cpad[shift:shift + M * N].view(M, N) if want_c else None
        gemm_i8_device(dA, dW, ds, C, acc, torch.cuda.current_stream().cuda_stream)
        if want_acc:
            assert torch.equal(acc, want)
        if want_c:
            assert torch.equal(C.view(torch.int32), wantf.view(torch.int32))
        for t in (pad, cpad.view(torch.int32)):  # nothing around the outputs is written
            assert bool((t[:shift] == 7).all()) and bool((t[shift + M * N:] == 7).all())


@pytest.mark.parametrize("M", [64 * 64, 64 * 64 + 9])
@pytest.mark.parametrize("with_c", [False, True])
def test_only_the_accumulators_unaligned(M, with_c):
    """Whole tiles of aligned operands (64 of them, and a partial row of tiles) and the int32 output alone at an address of
    no 16 bytes, which the whole-tile kernel's 16-byte stores do not take."""
    K, N = 64, 128
    rng = np.random.default_rng(M)
    A, W = rng.integers(-128, 128, (M, K), np.int8), rng.integers(-128, 128, (N, K), np.int8)
    s = (1e-3 + rng.random(N)).astype(np.float32)
    dA, dW, ds = (torch.from_numpy(x).cuda() for x in (A, W, s))
    want = (dA.double() @ dW.double().T).round().to(torch.int32)
    pad = torch.full((M * N + 64,), 7, dtype=torch.int32, device="cuda")
    acc = pad[1:1 + M * N].view(M, N)
    C = torch.empty((M, N), device="cuda") if with_c else None
    gemm_i8_device(dA, dW, ds, C, acc, torch.cuda.current_stream().cuda_stream)
    assert torch.equal(acc, want)
    assert bool((pad[:1] == 7).all()) and bool((pad[1 + M * N:] == 7).all())
    if with_c:
        assert torch.equal(C.view(torch.int32), (want.float() * ds).view(torch.int32))


@pytest.mark.parametrize("M,K,N", [(32705, 128, 127), (4096, 64, 1000), (4033, 192, 129), (70000, 64, 4), (8129, 384, 255)])
def test_only_n_ragged(M, K, N):
    """Whole, aligned K steps and channels that are not: rows of W past the last are repeated, not stored."""
    test_ragged_exact(M, K, N, 0)
