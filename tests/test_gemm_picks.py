"""Tile picks where another tile measured slower (us beside each): the dispatch is host code."""
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


@pytest.mark.parametrize("n,k,int8,rows,cfg", [
    (50257, 768, 0, 192, 61), (50257, 768, 0, 448, 61),   # rows of C through LDS 35.0, directly 36.0; 69.3, 70.7
    (50257, 768, 0, 129, 46), (50257, 768, 1, 192, 46),   # directly 30.6, through LDS 32.0; 32.3, 34.0
    (50257, 192, 0, 512, 61),                             # 64 rows a tile 32.9, 192x128 tiles 35.9
    (24577, 768, 0, 700, 61),                             # 64 rows a tile 45.4, 192x128 tiles 57.0
    (16384, 768, 0, 700, 60),                             # 128x128 tiles 30.5, 192x128 34.9
    (36001, 768, 0, 256, 61),                             # 64 rows a tile 24.8, 128x128 tiles 29.1
    (49153, 768, 1, 192, 61),                             # through LDS 30.8, directly 32.6
])
def test_vocabulary_picks(L, n, k, int8, rows, cfg):
    assert L.gpt2_tune_gemm_pick_q(rows, n, k, int8) == cfg


@pytest.mark.parametrize("n,k,rows,cfg", [
    (768, 3072, (1345, 1984), 0), (768, 768, (1345, 1984), 0), (1500, 1024, (673, 960), 0),   # 26.3, 64x64 tiles 30.0; 9.1, 10.1; 10.9, 12.1
    (1001, 768, (961, 1024), 54), (2000, 2048, (449, 512), 54), (4096, 1024, (193, 256), 54),  # 6.1, one k group 8.0; 10.3, 16.3; 7.0, 9.4
    (4096, 640, (193, 256), 5),   # K not a multiple of 256
])
def test_int8_picks_about_one_tile_a_cu(L, n, k, rows, cfg):
    assert {L.gpt2_tune_gemm_pick_q(m, n, k, 1) for m in rows} == {cfg}
