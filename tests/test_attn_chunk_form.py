"""Which form a chunk's attention takes, and that every form has the decode step's bits where it is taken."""

from __future__ import annotations

import pytest

from deepfold_amd import nf4
from test_prefill_glue import test_attn_chunk_on_the_matrix_cores as same_bits_as_the_decode_step

NEVER = 2 ** 31 - 1


def matrix_from(n, n_q, n_kv, hd=128, waves=4, scale=128 ** -0.5, max_seq=4096):
    return nf4._load_ext().chr_dv2_attn_chunk_matrix_from(n, n_q, n_kv, hd, waves, scale, max_seq)


# chunks of few workgroups were up to 2.3 times slower on the matrix cores (8 on 8, 16 tokens behind 1000 rows: 18 us,
# 41), chunks of many up to 1.8 times on the vector unit (28 on 4, 90 tokens behind 1791 rows: 119 us, 68)
@pytest.mark.parametrize("n_q,n_kv,last,below", [
    (8, 8, 160, NEVER), (40, 40, 32, NEVER), (28, 4, 45, NEVER), (24, 8, 53, NEVER), (32, 2, 40, NEVER),
    (16, 8, 96, NEVER), (32, 16, 48, NEVER), (32, 8, 64, 350), (16, 4, 128, 350), (40, 8, 32, 1200), (10, 2, 128, 1200)])
def test_chunks_of_few_workgroups_stay_on_the_vector_unit(n_q, n_kv, last, below):
    assert matrix_from(last, n_q, n_kv) == below and matrix_from(last + 1, n_q, n_kv) == 0


def test_the_other_lines():
    assert matrix_from(32, 32, 8) == NEVER and matrix_from(33, 32, 8) == 350
    assert matrix_from(2, 40, 8) == matrix_from(2, 5, 1) == 650 and matrix_from(3, 40, 8) == 1200
    for n_q, n_kv in ((48, 8), (16, 2), (64, 8)):
        assert matrix_from(2, n_q, n_kv) == 0
    for n_q, n_kv in ((48, 8), (40, 8), (32, 8), (8, 8)):
        assert matrix_from(1, n_q, n_kv) == NEVER
    for other in (dict(hd=64), dict(waves=8), dict(scale=0.0), dict(scale=-1.0), dict(scale=float("nan")),
                  dict(max_seq=1 << 20)):
        assert matrix_from(64, 64, 8, **other) == NEVER, other
    assert matrix_from(64, 64, 0) == -3 and matrix_from(0, 64, 8) == -3 and matrix_from(64, 63, 8) == -3
    assert matrix_from(65535, 1 << 16, 1 << 13, max_seq=512) == NEVER  # more threads than a grid has


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
    assert matrix_from(n, n_q, n_kv, max_seq=max_seq) == 0
    same_bits_as_the_decode_step(n_q, n_kv, max_seq, first, n, odd)


# chunks whose form the device chooses, on both sides of its line: fewer tiles than workgroups, and a cache that ends
@pytest.mark.gpu
@pytest.mark.parametrize("n_q,n_kv,max_seq,first,n,odd", [
    (40, 8, 1300, 1199, 9, False), (40, 8, 1300, 1200, 9, False), (40, 8, 1300, 1200, 32, True), (5, 1, 1210, 1201, 12, False),
    (40, 8, 700, 649, 2, True), (40, 8, 700, 650, 2, True), (40, 8, 90, 0, 2, False), (40, 8, 90, 30, 32, True), (10, 2, 1400, 1203, 128, False),
    (32, 8, 420, 349, 40, False), (32, 8, 420, 350, 40, False), (16, 4, 500, 351, 128, True), (32, 8, 100, 0, 33, True)])
def test_the_form_the_device_chooses(n_q, n_kv, max_seq, first, n, odd):
    assert matrix_from(n, n_q, n_kv, max_seq=max_seq) == ((650 if n == 2 else 1200) if n_q == 5 * n_kv else 350)
    same_bits_as_the_decode_step(n_q, n_kv, max_seq, first, n, odd)
