"""Convolutions over a packed filter: the kernel that a plan names, where a direct tile reads a filter that comes with the call."""
import pytest

import test_kernels_gpu as T
from plaidml_amd import hipkernels as hk
from test_kernels_gpu import (test_conv_bf16, test_conv_f32, test_conv_few_channel_patch_matrix, test_conv_few_channel_stride2,  # noqa: F401
                              test_conv_k_split_over_workgroups, test_conv_random_shapes_all_kinds, test_conv_register_filter,
                              test_conv_resident_filter, test_conv_resident_filter_general_tail)

pytestmark = pytest.mark.gpu


@pytest.fixture(autouse=True)
def filters_are_packed(monkeypatch):
    run = T.run_conv
    monkeypatch.setattr(T, 'run_conv', lambda *args, **named: run(*args, **dict(named, packed=True)))


# what the flag permits is plain fp32 where few results make that faster; a tile that is named keeps three bf16 products
@pytest.mark.parametrize('tile', ['64x64', '64x64ks'])
@pytest.mark.parametrize('M,N,K,ldb', [(1024, 1024, 1024, 1024), (100, 68, 72, 72), (64, 64, 36, 64), (200, 260, 132, 300), (130, 4, 8, 4),
                                       (96, 512, 2048, 516), (77, 66, 40, 66), (556, 38, 1264, 40)])
def test_split_products_of_a_named_tile(M, N, K, ldb, tile):
    flags = hk.FP32_AS_BF16X3 | hk.flag_tile(tile)
    for layout in (0, 1):
        assert '3 x f32' in text_of(M, N, K, K if layout else ldb, layout, flags)
    T.test_gemm_f32_right_hand_side_as_given(M, N, K, ldb, flags)


@pytest.mark.parametrize('flags', [0, hk.FP32_AS_BF16X3])
@pytest.mark.parametrize('M,N,K,ldb', [(2, 22, 3104, 22), (556, 38, 1264, 40), (36, 1896, 64, 1896)])
def test_layouts_agree_where_few_results_are_plain(M, N, K, ldb, flags):
    T.test_gemm_f32_right_hand_side_as_given(M, N, K, ldb, flags)


def test_ragged_split_product_of_a_named_tile(monkeypatch, capsys):
    monkeypatch.setitem(T.FORCED, 'flags', hk.flag_tile('64x64'))
    T.test_gemm_f32_as_three_bf16_products(257, 130, 68)
    assert '3 x f32' in capsys.readouterr().out


def text_of(m, n, k, ldb, layout, flags):
    d = hk.GemmDesc()
    d.in_dtype = d.out_dtype = d.c_dtype = hk.F32
    d.m, d.n, d.k, d.lda, d.ldb, d.ldc, d.b_layout, d.flags = m, n, k, k, ldb, n, layout, flags
    plan = hk.lib().pml_hip_gemm_dispatch(T.ctypes.byref(d))
    assert plan, hk.lib().pml_hip_last_error()
    text = hk.describe(plan)
    hk.lib().pml_hip_plan_free(plan)
    return text
