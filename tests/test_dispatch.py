"""The rules on sizes that choose between kernels (csrc/dispatch.hpp), asked on
the CPU: every shape below was timed with both kernels on an MI355X, and the
rule takes the faster one (a tie may go either way)."""
import ctypes

import pytest

from gpu_util import dispatch_rules


@pytest.fixture(scope="module")
def rules():
    return dispatch_rules()


@pytest.mark.parametrize("vs_lds,rows,K,N,tall", [
    # against the LDS-resident GEMM: wide products of few rows stay there
    (1, 16, 1024, 32000, 0), (1, 64, 1024, 32000, 0), (1, 96, 1024, 32000, 0),
    (1, 128, 1024, 32000, 1), (1, 192, 1024, 32000, 1), (1, 288, 1024, 32000, 1),
    (1, 96, 512, 32000, 0), (1, 128, 512, 32000, 1), (1, 64, 256, 32768, 0),
    (1, 96, 128, 32768, 0), (1, 128, 128, 32768, 1), (1, 96, 1024, 24576, 0),
    (1, 128, 1024, 24576, 1), (1, 16, 1024, 200000, 0), (1, 512, 1024, 8192, 1),
    (1, 1024, 1024, 3072, 1), (1, 512, 1024, 3072, 0), (1, 8192, 1024, 8192, 1),
    # against the digit-plane GEMM
    (0, 64, 4096, 32000, 0), (0, 128, 4096, 32000, 1), (0, 192, 4096, 12288, 0),
    (0, 256, 4096, 12288, 1), (0, 288, 4096, 8192, 0), (0, 384, 4096, 8192, 1),
    (0, 4096, 4096, 1024, 1), (0, 64, 2048, 32768, 0), (0, 192, 2048, 12288, 0),
    (0, 256, 2048, 12288, 1), (0, 512, 2048, 6144, 1), (0, 32, 1024, 32000, 0),
    (0, 128, 1024, 32000, 1), (0, 32, 512, 32768, 0), (0, 64, 512, 32768, 1),
    (0, 64, 128, 32768, 1),
    # what the kernel does not take
    (1, 4096, 1024, 4104, 0), (0, 4096, 960, 4096, 0)])
def test_tall_gemm(rules, vs_lds, rows, K, N, tall):
    assert rules.gemm_tall_shape(rows, K, N, vs_lds) == tall


@pytest.mark.parametrize("B,S,H,D,q8,keys,prompt", [
    # long caches behind tiles of which much is empty, or fewer than the CUs
    (40, 40, 4, 16, 0, 16000, 0), (40, 40, 4, 16, 0, 4096, 0), (40, 20, 4, 16, 0, 8192, 0),
    (40, 40, 4, 16, 0, 512, 1), (40, 64, 4, 16, 0, 2048, 1), (20, 40, 8, 8, 0, 2048, 0),
    (20, 40, 8, 40, 0, 4096, 0), (20, 40, 8, 40, 0, 1024, 1), (20, 64, 8, 40, 0, 8192, 1),
    (20, 40, 8, 32, 0, 8192, 0), (20, 28, 8, 32, 0, 8192, 1), (20, 36, 8, 24, 0, 8192, 0),
    (5, 40, 32, 64, 1, 16000, 0), (5, 40, 32, 64, 1, 1024, 1), (5, 64, 32, 64, 1, 8192, 1),
    (10, 40, 16, 64, 0, 4000, 1), (10, 20, 16, 64, 0, 8000, 1), (128, 36, 8, 8, 0, 2048, 1),
    # prompts proper
    (4, 1000, 16, 64, 0, 1024, 1), (8, 300, 8, 32, 1, 4096, 1), (4, 1000, 16, 8, 0, 16384, 1),
    # too short, too few
    (64, 16, 16, 64, 0, 512, 0), (1, 100, 16, 64, 0, 512, 0), (1, 320, 16, 64, 0, 512, 1)])
def test_prompt_attention(rules, B, S, H, D, q8, keys, prompt):
    assert rules.attention_prompt_shape(B, S, H, D, q8, keys) == prompt


@pytest.mark.parametrize("rows,K,N,waves", [
    # a short K is split over 4 waves all the same
    (16, 252, 5626, 4), (256, 252, 352, 4), (64, 64, 2032, 4), (512, 128, 391, 4),
    (512, 252, 4096, 0), (1000, 60, 91, 0),
    # few rows: 32 x 32 tiles, which are counted as such
    (16, 4096, 5626, 8), (16, 2048, 5626, 8), (16, 1024, 8126, 8), (16, 1024, 12501, 4),
    (24, 4096, 3751, 8), (32, 2048, 31251, 4), (16, 1024, 62501, 4), (33, 1024, 62501, 0),
    (333, 772, 1544, 4), (64, 4096, 1024, 8), (512, 1024, 1024, 4), (2048, 1024, 4096, 0)])
def test_f32_gemm_tiles(rules, rows, K, N, waves):
    assert rules.gemm_f32_waves(rows, K, N) == waves


def test_f32_gemm_from_90000_outputs(rules):
    assert rules.gemm_f32_shape(16, 5625) and not rules.gemm_f32_shape(15, 60000)
    assert not rules.gemm_f32_shape(16, 5624) and rules.gemm_f32_shape(90000, 65536)


@pytest.mark.parametrize("n_out,n_red,along_sums,short", [
    (1 << 20, 2, 0, 1), (1 << 20, 1, 1, 1), (1 << 20, 32, 0, 1), (1 << 20, 64, 0, 1),
    (131072, 300, 0, 1), (8192, 32, 0, 1), (8192, 64, 0, 0), (16384, 1000, 0, 0),
    (1 << 20, 8, 1, 1), (1 << 20, 12, 1, 1), (1 << 20, 16, 1, 0), (262144, 17, 1, 1),
    (1 << 20, 24, 1, 1), (1 << 20, 32, 1, 0), (262144, 64, 1, 0),
    (100, 1024, 0, 0), (1024, 1024, 1, 0), (1, 1 << 20, 1, 0), (16, 4, 1, 1)])
def test_short_sums(rules, n_out, n_red, along_sums, short):
    f = rules.sum_short_shape
    f.argtypes = [ctypes.c_longlong, ctypes.c_longlong, ctypes.c_int]
    assert f(n_out, n_red, along_sums) == short


@pytest.mark.parametrize("M,K,N,short", [
    (1, 1, 1 << 20, 1), (1 << 20, 8, 1, 1), (1, 16, 100000, 1), (8, 4, 131072, 1),
    (32, 12, 1 << 20, 1), (1 << 20, 24, 32, 1), (8, 40, 1 << 20, 1), (3, 3, 70000, 1),
    (1, 16, 1000, 0), (8, 32, 131072, 0), (8, 64, 1 << 20, 0), (20000, 8, 8, 0),
    (64, 12, 1 << 20, 1), (64, 12, 262144, 0), (131072, 4, 1000, 1), (100, 12, 1 << 20, 1),
    (4096, 4, 16384, 0), (131072, 32, 1000, 0), (1024, 784, 1024, 0), (1024, 1024, 100, 0),
    (2048, 2048, 2048, 0), (2, 2, 2, 0)])
def test_short_products(rules, M, K, N, short):
    f = rules.matmul_short_shape
    f.argtypes = [ctypes.c_longlong] * 3
    assert f(M, N, K) == short
