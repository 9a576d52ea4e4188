"""The numbers that choose between kernels are one dataclass; a kernel table takes a changed set."""
from dataclasses import fields

import pytest

from servelab_amd.kernels.tuning import Tuning


def test_every_choice_lands_on_the_table_under_its_upper_case_name():
    class Table:
        pass
    t = Table()
    Tuning(few_wave_us=2.5, wide_min_m=33).apply(t)
    assert t.FEW_WAVE_US == 2.5 and t.WIDE_MIN_M == 33
    assert t.NARROW_ATTENTION_WORKGROUPS == Tuning().narrow_attention_workgroups
    assert {n for n in vars(t)} == {f.name.upper() for f in fields(Tuning)}


@pytest.mark.gpu
def test_a_kernel_table_with_other_choices_gives_the_same_numbers():
    """Choices move work between kernels, never the result beyond rounding: a decode attention
    split into few wavefronts or many, a product on the one-tile or the LDS-staged kernel."""
    import torch
    from servelab_amd.kernels import HipOps
    a = HipOps(torch.bfloat16, "cuda:0")
    b = HipOps(torch.bfloat16, "cuda:0", tuning=Tuning(few_wave_us=20.0, mid_min_elements=1 << 40,
                                                       mid_min_elements_many=1 << 40, resident_min_rounds=1 << 20))
    assert b.FEW_WAVE_US == 20.0 and a.FEW_WAVE_US == Tuning().few_wave_us
    assert b._decode_shares(32, 64, 128, 128) < a._decode_shares(32, 64, 128, 128)
    g = torch.Generator(device="cuda").manual_seed(0)
    x = torch.randn(40, 1024, device="cuda", generator=g).bfloat16()
    w = (torch.randn(12288, 1024, device="cuda", generator=g) * 0.03).bfloat16()
    wa, wb = a.prepare_weight(w), b.prepare_weight(w)
    assert a._takes_mid(40, 12288, 1024) and not b._takes_mid(40, 12288, 1024)
    ya, yb = a.linear(x, wa, None).float(), b.linear(x, wb, None).float()
    ref = x.float() @ w.float().T
    assert (ya - ref).abs().max() < 2 ** -6 * ref.abs().max()
    assert (yb - ref).abs().max() < 2 ** -6 * ref.abs().max()


def test_shapes_among_the_library_tuner_s_results():
    from servelab_amd.kernels.product_ops import tuned_shapes
    results = (("GemmAndBiasTunableOp_BFloat16_TN", "tn_16384_700_2048_ld_2048_2048_16384", "Gemm_Hipblaslt_1", 0.04),
               ("GemmTunableOp_BFloat16_TN", "tn_96_32_64_ld_64_64_96", "Default", 0.01),
               ("GemmTunableOp_BFloat16_NN", "nn_64_64_64_ld_64_64_64", "Gemm_Hipblaslt_2", 0.01),
               ("GemmTunableOp_float_TN", "tn_8_8_8_ld_8_8_8", "Gemm_Rocblas_3", 0.01))
    assert tuned_shapes(results) == {(700, 16384, 2048), (32, 96, 64)} and tuned_shapes(()) == set()


# (us measured, the library's product and its pass for the bias / the tiles, beside each)
@pytest.mark.parametrize("M,N,K,tiles", [
    (1000, 6160, 2048, True), (600, 10304, 2048, True), (1500, 4096, 2048, True),              # 44 / 37, 44 / 37, 37 / 36
    (1500, 7168, 3584, True), (1280, 10792, 3584, True), (2048, 14336, 4096, True),            # 85 / 73, 104 / 88, 218 / 198
    (1500, 10792, 3584, False), (2500, 7168, 3584, False), (1000, 5120, 5120, False),          # 123 / 133, 134 / 137, 62 / 66
    (1280, 14336, 4096, False), (2500, 14336, 4096, False), (768, 6160, 2048, False)])         # 148 / 153, 280 / 295, 35 / 37
def test_products_with_a_bias_take_tiles_where_these_are_faster(M, N, K, tiles):
    from test_qkv_shapes import Recorded
    assert Recorded()._bias_tiles(M, N, K) is tiles
