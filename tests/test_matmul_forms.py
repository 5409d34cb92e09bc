"""The batched matmul's choice of tiles (krh_matmul_form): the sizes of the GPU
tile tests reach every form, and the choice at measured sizes is the form that
was the fastest there (or within 3% of it)."""
import pytest

import krafla as K
from matmul_sizes import MATMUL_TILES, SWIGLU_TILES

S16, S32, T64, T128, RING64, RING128 = range(6)


def test_tile_sizes_reach_every_form():
    assert {K.hip.krh_matmul_form(*s, 0) for s in MATMUL_TILES} == {S16, S32, T64, T128, RING64, RING128}
    swiglu = [(14336, 4096, 300), (4864, 896, 511), (768, 288, 37), (96, 64, 5), (8192, 2048, 129)] + SWIGLU_TILES
    assert {K.hip.krh_matmul_form(*s, 1) for s in swiglu} == {T64, T128, RING64, RING128}
    assert K.hip.krh_matmul_form(0, 32, 1, 0) == -1


# prompts of a 15M model's widths and short ones of wide layers: the tiles for
# long reductions took up to 1.5 times as long there
@pytest.mark.parametrize("rows,cols,T,swiglu,forms", [
    (14336, 288, 700, 0, {RING128}), (14336, 288, 2047, 0, {RING128, T128}), (4096, 288, 700, 0, {RING64, T64}), (9024, 896, 200, 0, {T64}),
    (896, 288, 700, 0, {S32}), (896, 896, 700, 0, {S32}), (896, 896, 64, 0, {S16}), (4096, 14336, 37, 0, {S16}),
    (14336, 4096, 256, 0, {T64}), (14336, 4096, 511, 0, {T128}), (4864, 288, 2047, 1, {RING64, RING128}),
    (14336, 4096, 511, 1, {T128})])
def test_form_at_measured_sizes(rows, cols, T, swiglu, forms):
    assert K.hip.krh_matmul_form(rows, cols, T, swiglu) in forms
