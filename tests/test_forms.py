"""The rules that choose a kernel form, read through the library's form queries
(host arithmetic: they run without a GPU)."""
import pytest

from pulsar_amd import lib


@pytest.mark.parametrize("nh,nkv,hd,per_query,tiles", [
    (32, 8, 64, 64000, None), (8, 8, 64, 64000, None), (32, 32, 64, 64000, None), (32, 16, 128, 64000, None),
    (16, 4, 128, 66000, 90000), (32, 8, 128, 33000, 36000), (64, 8, 64, 12000, 12500), (64, 8, 128, 16000, 16500)])
def test_attention_one_query(nh, nkv, hd, per_query, tiles):
    """One query gives a matrix tile no second one to share its keys with: it takes tiles only
    where they measured faster (8 heads a kv head, or 4 of 128 over many keys)."""
    form = lib().pq_attn_decode_form
    for pos0 in (0, 255, 1500, per_query):
        assert form(nh, nkv, hd, pos0, 1, 0) == 0
    if tiles is not None:
        assert form(nh, nkv, hd, tiles, 1, 0) == 1
    assert form(nh, nkv, hd, 64000, 64, 0) == 1
    assert form(nh, nkv, hd, 0, 2, 0) == 0


def test_attention_form_refuses_what_the_call_refuses():
    form = lib().pq_attn_decode_form
    for bad in ((24, 8, 64, 0, 4, 0), (32, 8, 96, 0, 4, 0), (30, 8, 64, 0, 4, 0), (32, 0, 64, 0, 4, 0),
                (32, 8, 64, -1, 4, 0), (32, 8, 64, 0, 0, 0),
                (32, 8, 64, 0, 4, -1)):
        assert form(*bad) == -1


def test_gemm_forms_refuse_what_the_calls_refuse():
    L = lib()
    for bad in ((0, 2048, 4), (64, 2040, 4), (64, 2048, 0)):
        assert L.pq_q8_gemm_form(*bad) == -1 and L.pq_q8r_gemv_form(*bad) == -1
        assert L.pq_qlow_gemm_form(*bad, 4) == -1
    assert L.pq_q8r_gemv_form(8, 8992, 4) == -1                 # over 8 blocks a leaf
    assert L.pq_qlow_gemm_form(64, 2048, 4, 6) == -1 and L.pq_qlow_gemm_form(64, 16640, 4, 4) == -1


def test_gemm_even_split_over_xcds():
    """Whole row groups per XCD must not cost a round of workgroups that the chip as a whole does not need."""
    form = lib().pq_q8_gemm_form
    assert form(3104, 2048, 160) == 2 + 16 * 8 + 256    # 49 tiles x 5: 35 workgroups on one XCD's 32 CUs, 245 in all
    assert form(3104, 2048, 320) == 2 + 16 * 4 + 256    # 490 of 512, 70 of 64
    assert form(8200, 2048, 384) == 4 + 256             # 17 row groups x 12: 204 of 256, 36 of 32
    assert form(3104, 2048, 128) == 2 + 16 * 8          # 28 of 32 already
    assert form(33000, 2048, 256) == 4                  # three rounds either way
    assert form(16384, 2048, 256) == 4


def test_q8r_vector_form_beside_idle_tiles():
    """9 to 18 positions stay on the vector kernel where 16- or 32-wide tiles give the CUs an almost empty last
    round (6144 rows: 384 tiles, 10000: 625 16-wide ones, or 313 32-wide)."""
    form = lib().pq_q8r_gemv_form
    for N, K, T in ((6144, 2048, 9), (6144, 2048, 10), (10000, 2048, 9), (10000, 2048, 10), (10000, 2048, 17),
                    (20000, 1024, 9), (8200, 2048, 9)):
        assert form(N, K, T) == 0, (N, K, T)
    for N, K, T in ((2048, 2048, 9), (4096, 2048, 9), (6144, 2048, 14), (10000, 2048, 12), (16384, 2048, 9),
                    (65536, 2048, 9), (16384, 512, 9), (2048, 8192, 9), (2048, 7680, 6), (10000, 2048, 19)):
        assert form(N, K, T) in (16, 32), (N, K, T)
    for N in (1, 512, 6144, 65536):
        assert form(N, 2048, 8) == 0 and form(N, 7680, 5) == 0


def test_gemm_workspace_only_for_the_walking_form():
    """No other form of the Q8_0 GEMM splits K over workgroups through memory."""
    L = lib()
    for N in (1, 300, 3104, 8000, 16384, 40000):
        for K in (32, 2048, 8192):
            for T in (1, 32, 33, 97, 256):
                if L.pq_q8_gemm_form(N, K, T) % 16 != 1:
                    assert L.pq_q8_gemm_workspace_bytes(N, K, T) == 0
    assert L.pq_q8_gemm_form(2048, 8192, 32) == 1 and L.pq_q8_gemm_workspace_bytes(2048, 8192, 32) > 0
