"""Which kernel a size goes to, for the kernels that test_hyper_rows_gpu.py and test_few_rows_halves_gpu.py hold to 64 bits on both sides of
these lines."""
import pytest

from neuronx_distributed_llama3_2_amd import ops


@pytest.mark.parametrize("R,W,threads", [(1, 4, 256), (64, 1024, 256), (64, 1028, 512), (5, 2048, 512), (5, 2052, 1024), (64, 4096, 1024),
                                         (65, 2048, 0), (5, 4100, 0), (5, 1026, 0)])
def test_hyper_step(R, W, threads):
    f = ops.hybrid_ext().hyper_step_threads
    assert f(R, W, W + 4, W) == threads and f(R, W, W + 2, W) == f(R, W, W, W + 1) == 0


@pytest.mark.parametrize("N,K,halved", [(8, 64, True), (4096, 1936, True), (8192, 2048, True), (8208, 2048, False), (40, 2064, True), (3000, 4224, True),
                                        (32768, 2064, True), (32784, 2064, False), (40, 4232, False)])
def test_few_rows(N, K, halved):
    f = ops.ext().few_rows_halved
    assert f(17, N, K) == f(32, N, K) == halved and not f(16, N, K) and not f(33, N, K)
