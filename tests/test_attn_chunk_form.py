"""Which form a chunk's attention takes, and the matrix form's bits where it is taken."""

from __future__ import annotations

import pytest

from deepfold_amd import nf4
from test_prefill_glue import test_attn_chunk_on_the_matrix_cores as same_bits_as_the_decode_step


def form(n, n_q, n_kv, hd=128, waves=4, scale=128 ** -0.5, max_seq=4096):
    return nf4._load_ext().chr_dv2_attn_chunk_form(n, n_q, n_kv, hd, waves, scale, max_seq)


# chunks of few workgroups were up to 2.3 times slower on the matrix cores (8 on 8, 16 tokens behind 1000 rows: 18 us, 41)
@pytest.mark.parametrize("n_q,n_kv,last", [(8, 8, 320), (40, 40, 64), (28, 4, 91), (24, 8, 106), (32, 2, 80), (16, 8, 192),
                                           (32, 16, 96), (32, 8, 64), (16, 4, 128), (40, 8, 32), (10, 2, 128),
                                           (48, 8, 1), (16, 2, 1), (64, 8, 1)])
def test_chunks_of_few_workgroups_stay_on_the_vector_unit(n_q, n_kv, last):
    assert form(last, n_q, n_kv) == 0 and form(last + 1, n_q, n_kv) == 1


def test_what_the_matrix_form_is_not_made_for():
    assert form(64, 64, 8) == 1
    for other in (dict(hd=64), dict(waves=8), dict(scale=0.0), dict(scale=-1.0), dict(scale=float("nan")),
                  dict(max_seq=1 << 20)):
        assert form(64, 64, 8, **other) == 0, other
    assert form(64, 64, 0) == -3 and form(0, 64, 8) == -3 and form(64, 63, 8) == -3
    assert form(65535, 1 << 16, 1 << 13, max_seq=512) == 0  # more threads than a grid has


# as the cases of test_attn_chunk_on_the_matrix_cores, at sizes that take it
@pytest.mark.gpu
@pytest.mark.parametrize("n_q,n_kv,max_seq,first,n,odd", [
    (160, 160, 96, 40, 17, False),   # one query head a KV head: a tile and one query
    (6, 1, 130, 1, 64, False),       # six: a tile begins inside a token; rows end on and around whole tiles of 64
    (48, 8, 200, 0, 2, False),       # the first token sees nothing
    (8, 1, 200, 14, 4, False), (12, 2, 200, 63, 5, False), (40, 8, 320, 150, 33, False), (32, 8, 140, 60, 65, False),
    (96, 48, 64, 30, 33, False), (96, 32, 80, 40, 27, False), (68, 4, 120, 62, 38, False),
    (160, 160, 80, 40, 17, True), (6, 1, 150, 20, 40, True), (96, 48, 64, 20, 33, True), (8, 1, 70, 30, 9, True)])
def test_the_matrix_form_where_it_is_taken(n_q, n_kv, max_seq, first, n, odd):
    assert form(n, n_q, n_kv, max_seq=max_seq) == 1
    same_bits_as_the_decode_step(n_q, n_kv, max_seq, first, n, odd)
