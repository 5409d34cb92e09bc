"""The batched attention's choice of kernels (krh_attention_plan): the sizes of
the GPU form tests reach every form of every stage, and the choice at measured
shapes is the form that was the fastest there."""
import pytest

import krafla as K
from attn_sizes import BATCH_BLOCKS

TOKEN, BLOCK, ROWS = range(3)
KV = [K.ML_F32, K.ML_F16, K.ML_Q8_0]


def plan(kv, nh, nkv, hd, max_seq, window, ntok, last):
    p = K.hip.krh_attention_plan(kv, nh, nkv, hd, max_seq, window, ntok, last)
    assert p >= 0
    return p & 3, (p >> 2) & 3, p >> 4


@pytest.fixture(params=[0, 1 << 30, 512])
def choice(request):
    K.hip.krh_set_attn_rb_min(request.param)
    yield request.param
    K.hip.krh_set_attn_rb_min(512)


@pytest.mark.parametrize("kv", KV)
def test_form_tests_reach_every_form(kv, choice):
    """windowed and not; the token form for 1 to 16 heads a group (mix chunks of
    64 to 4 dims), the block form for the chunks it takes (16 and more)"""
    got = {}
    for nh, nkv, hd, pos0, T, w in BATCH_BLOCKS:
        if T > 1:
            sc, sm, mx = plan(kv, nh, nkv, hd, 512, w, T, pos0 + T - 1)
            group = nh // nkv
            chunk = 64 >> (group - 1).bit_length()
            got.setdefault(("scores", sc, w > 0), set()).add(hd)
            got.setdefault(("mix", mx), set()).add(chunk)
            got.setdefault(("softmax", sm), set()).add(w > 0)
    if choice == 0:
        assert got[("mix", ROWS)]
        if kv != K.ML_Q8_0:
            assert got[("scores", ROWS, True)] >= {48, 64, 80, 96, 128, 256} and got[("scores", ROWS, False)]
    elif choice == 1 << 30:
        assert got[("scores", BLOCK, True)] and got[("scores", BLOCK, False)]
        assert got[("mix", BLOCK)] >= {64, 32, 16} and got[("mix", TOKEN)] >= {8, 4}
    else:
        assert got[("scores", TOKEN, True)] and got[("scores", TOKEN, False)]
        assert got[("mix", TOKEN)] >= {64, 32, 16, 8, 4}
    assert got[("softmax", 1)] and got[("softmax", 2)]


def test_no_batch():
    for bad in [(4, 3, 64, 512, 0, 8, 7), (4, 2, 63, 512, 0, 8, 7), (4, 2, 64, 512, 0, 1, 0), (4, 2, 64, 512, 0, 8, 512),
                (4, 2, 64, 512, 0, 8, 6), (34, 2, 64, 512, 0, 8, 7)]:
        assert K.hip.krh_attention_plan(K.ML_F32, *bad) == -1


# few tokens over a window, and few over a long context: one token a workgroup
# (the token blocks took up to three times as long); longer prompts: blocks, rows
@pytest.mark.parametrize("nh,nkv,hd,pos0,T,window,mix", [
    (4, 1, 64, 2021, 101, 70, TOKEN), (2, 1, 256, 352, 51, 112, TOKEN), (32, 8, 64, 2000, 16, 1024, TOKEN),
    (32, 8, 64, 2000, 128, 1024, BLOCK), (6, 6, 48, 2000, 1024, 1024, BLOCK), (32, 8, 64, 2000, 2000, 0, ROWS),
    (8, 4, 256, 2048, 1021, 1024, ROWS), (32, 8, 128, 2000, 1024, 128, ROWS), (24, 8, 80, 2000, 1024, 0, BLOCK)])
def test_mix_at_measured_shapes(nh, nkv, hd, pos0, T, window, mix):
    assert plan(K.ML_F32, nh, nkv, hd, 4096, window, T, pos0 + T - 1)[2] == mix
