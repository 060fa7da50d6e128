"""Tile picks between whose ends another tile measured faster (us beside each): the dispatch is host code."""
import pytest

QKV, MLP = (2304, 768), (768, 3072)


@pytest.mark.parametrize("shape,int8,rows,cfg", [
    (QKV, 1, (641, 672), 35),     # 48x32 tiles 7.0, 128x64 8.2
    (MLP, 1, (641, 704), 36),     # two k groups 12.3, four 12.9
    (MLP, 1, (705, 768), 53),     # four 11.2, two 11.7
    (MLP, 1, (769, 832), 36),     # two 12.8, four 13.3
    (MLP, 1, (833, 896), 53),     # four 11.1, two 11.6
    (MLP, 1, (897, 960), 36),     # two 13.1, four 13.5
    (MLP, 1, (961, 1024), 53),    # four 11.5, two 11.8
])
def test_trunk_picks(L, shape, int8, rows, cfg):
    assert {L.gpt2_tune_gemm_pick_q(m, *shape, int8) for m in range(rows[0], rows[1] + 1)} == {cfg}
