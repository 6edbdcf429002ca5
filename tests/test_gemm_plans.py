"""CPU-only: which kernel the GPU tests' products take -- edge of an output tile, waves of a workgroup, splits of k (0: not looked
at) -- so that a change of the launcher's lines cannot leave a kernel without its test."""
import pytest

from __graft_entry__ import load_package

EIGHT, LARGE, SMALL, DIRECT = (128, 8), (128, 4), (64, 4), (32, 8)


@pytest.mark.parametrize("m,n,k,tA,tB,want", [
    # test_matrix_product_on_eight_waves
    (1000, 3460, 385, 0, 0, EIGHT), (1000, 3460, 388, 1, 0, EIGHT), (2040, 1793, 384, 1, 0, EIGHT), (128, 27300, 420, 0, 0, EIGHT),
    (1020, 6100, 900, 1, 0, EIGHT), (1018, 6101, 769, 0, 0, EIGHT), (1024, 15900, 387, 1, 0, EIGHT), (1021, 3300, 2050, 0, 0, EIGHT),
    # test_matrix_product_is_as_exact_as_fp32_sums: 128 x 128 tiles of operands of any length, in every order
    (3100, 3076, 516, 1, 0, EIGHT), (3101, 3077, 517, 1, 0, EIGHT), (3102, 3079, 515, 0, 0, EIGHT), (3100, 3076, 800, 0, 0, LARGE),
    (3076, 3100, 540, 0, 1, LARGE), (3077, 3101, 541, 0, 1, LARGE), (3101, 3077, 801, 1, 0, LARGE), (3102, 3079, 770, 0, 0, LARGE),
    # test_matrix_product_of_short_runs_and_full_generations
    (1024, 11900, 256, 1, 0, LARGE), (1024, 11900, 256, 0, 0, LARGE), (1012, 12001, 300, 1, 0, LARGE), (1936, 5999, 508, 0, 0, EIGHT),
    (1024, 11000, 252, 1, 0, SMALL), (1024, 5370, 768, 1, 0, EIGHT), (1020, 5110, 768, 0, 0, SMALL), (1024, 12700, 516, 0, 0, EIGHT),
    (1020, 9000, 800, 0, 0, LARGE), (1024, 5370, 900, 0, 0, EIGHT), (430, 21700, 640, 1, 0, LARGE), (432, 31350, 512, 0, 0, EIGHT),
    (300, 28900, 640, 1, 0, SMALL),
    # test_matrix_product_of_few_blocks
    (640, 1024, 40, 1, 0, DIRECT), (641, 1023, 41, 0, 0, SMALL),
])
def test_products(m, n, k, tA, tB, want):
    assert load_package().capi.probe_gemm_plan(m, n, k, 1, tA, not tB)[:2] == want


@pytest.mark.parametrize("P,D,N,problems,want,splits", [
    # test_wide_dense_gradient_on_eight_waves, test_weight_gradients_of_large_tiles_over_listed_slots
    (1024, 1024, 6200, 1, EIGHT, 8), (1000, 1022, 6401, 1, EIGHT, 8), (1300, 900, 6163, 1, EIGHT, 5), (1024, 1028, 6000, 1, EIGHT, 7),
    # test_weight_gradient_is_the_same_in_every_call, test_weight_gradients_of_wide_dense_layers
    (1024, 1028, 653, 1, SMALL, 2), (1024, 1028, 1200, 1, SMALL, 3), (512, 514, 2501, 1, SMALL, 9), (401, 603, 3001, 1, SMALL, 11),
    (37, 1, 2300, 1, SMALL, 9), (2048, 3072, 70, 1, SMALL, 1), (1026, 7, 1200, 1, DIRECT, 1), (128, 8192, 9000, 1, EIGHT, 8),
    # test_recurrent_weight_gradients_are_the_same_in_every_call: input and recurrent weights of 2 x 256 cells, of 2 x 520
    (512, 256, 4160, 8, EIGHT, 4), (256, 256, 4144, 8, SMALL, 0), (70, 520, 60, 8, DIRECT, 1),
])
def test_weight_gradients(P, D, N, problems, want, splits):
    plan = load_package().capi.probe_gemm_plan(P, D, N, problems, weight_gradient=True)
    assert plan[:2] == want and splits in (0, plan[2])
