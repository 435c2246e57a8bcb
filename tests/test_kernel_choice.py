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


# the line of three quarters of the CUs; rounds that are not filled; whole rounds of long reductions
@pytest.mark.parametrize("rows,weight_rows,K,glu,pays", [
    (768, 16384, 2048, True, True), (767, 16384, 2048, True, False), (4096, 16384, 4128, True, False), (4096, 16384, 2040, True, False),
    (1280, 16384, 2048, True, False), (1400, 16384, 2048, True, True), (1280, 16384, 2048, False, False), (1280, 16384, 1024, True, True), (640, 28672, 4096, True, False), (896, 22016, 4096, True, False),
    (896, 28672, 4096, True, True), (1536, 12288, 2048, False, True), (2304, 16384, 2048, True, True),
    (4096, 28672, 4096, True, False), (4096, 28672, 4096, False, True), (4096, 28672, 3072, True, True), (1024, 16384, 4096, True, True), (5120, 28672, 4096, True, True)])
def test_products_with_an_activation(rows, weight_rows, K, glu, pays):
    from neuronx_distributed_llama3_2_amd.ops import gemm

    assert gemm.act_pays(rows, weight_rows, K, glu) is pays


# blocks of 16 columns and chunks of 64 tokens: few blocks from 4 chunks on, up to 128 from 12, long keys from 2 up to 256; a gigabyte
@pytest.mark.parametrize("B,T,H,D,V,split", [(1, 193, 5, 128, 128, True), (1, 192, 5, 128, 128, False), (1, 704, 41, 64, 16, False), (1, 705, 41, 64, 16, True),
                                             (2, 512, 4, 128, 128, False), (1, 705, 16, 128, 128, True), (1, 4096, 129, 64, 16, False), (1, 65, 16, 256, 256, True),
                                             (1, 64, 16, 256, 256, False), (2, 4096, 9, 256, 256, False), (1, 1 << 16, 8, 128, 128, True), (1, 1 << 16, 16, 128, 128, False)])
def test_delta_rule_in_two_launches(B, T, H, D, V, split):
    assert (ops.hybrid_ext().delta_split_floats(B, T, H, D, V) > 0) is split
