"""Which form of a kernel a launch takes: the launchers' own rules, asked without a GPU (which stand for 256 CUs then)."""
import pytest


@pytest.fixture(scope="module")
def E():
    from aios_amd.runtime import native

    m = native.load(build_if_missing=False)
    if m is None:
        pytest.skip("native engine not built")
    return m


@pytest.mark.parametrize("H,Hkv,hd,start,T,groups", [
    # few tiles; workgroups for every CU at most
    (32, 8, 128, 0, 576, 1), (32, 8, 128, 0, 577, 2), (32, 8, 128, 0, 1024, 2), (32, 8, 128, 2000, 1024, 2),
    # a second round of workgroups: two groups only where it is much shorter than the first
    (32, 8, 128, 0, 1025, 1), (32, 8, 128, 0, 1500, 2), (32, 8, 128, 0, 1792, 2), (32, 8, 128, 0, 1793, 1), (32, 4, 64, 0, 2048, 1),
    (32, 8, 128, 0, 2049, 1), (64, 8, 128, 0, 1000, 1), (32, 8, 128, 2000, 1184, 1), (32, 4, 64, 2000, 2048, 1), (8, 2, 128, 2000, 4800, 2),
    (16, 8, 128, 0, 4096, 2), (16, 8, 128, 1000, 3008, 2), (16, 8, 128, 1000, 3520, 1),
    # in runs over the keys
    (8, 2, 64, 0, 2048, 1), (4, 2, 128, 0, 4096, 1), (32, 8, 128, 2000, 512, 2), (32, 8, 128, 6000, 300, 2), (4, 2, 64, 1300, 1950, 2),
    (4, 2, 64, 1300, 1951, 1), (2, 2, 128, 3000, 2049, 1), (16, 8, 128, 4000, 768, 1)])
def test_two_groups_of_waves_only_where_they_are_the_faster(E, H, Hkv, hd, start, T, groups):
    assert E.attn_prefill_form(H, Hkv, hd, start, T)[0] == groups


BF16, Q4_K, Q6_K = 30, 12, 14


@pytest.mark.parametrize("t,N,K,few,many", [  # slices for up to 16 rows, and for 17 to 32
    # as many as the registers ask for, or one more where that deals the tiles out more evenly
    (BF16, 2048, 8704, 4, 5), (Q6_K, 2048, 8704, 4, 4), (Q4_K, 2048, 8704, 4, 4), (Q4_K, 4096, 12288, 3, 3), (Q4_K, 4096, 14336, 4, 4),
    # bf16 of few tiles in two instead of one
    (BF16, 1536, 4096, 2, 2), (BF16, 1600, 4096, 1, 2), (BF16, 1088, 3136, 2, 2), (BF16, 1088, 2048, 1, 1),
    # ... in four instead of two
    (BF16, 1600, 5632, 4, 3), (BF16, 2048, 7168, 4, 4), (BF16, 2048, 7232, 2, 4), (BF16, 3072, 8192, 4, 0), (BF16, 2048, 8192, 2, 4),
    # Q6_K's long products of up to 16 rows: the ring's up to 10240 k
    (Q6_K, 3072, 10240, 0, 4), (Q6_K, 3072, 10496, 4, 4), (Q6_K, 3072, 14336, 4, 4), (Q6_K, 2944, 8448, 3, 3), (Q6_K, 3072, 8192, 2, 2)])
def test_slices_of_k_of_batched_decode(E, t, N, K, few, many):
    assert [E.gemm_wk_slices(t, N, K, M) for M in (2, 16, 17, 32)] == [few, few, many, many]


def test_slices_of_k_within_the_workspace(E):
    """the slice more only where its slabs and tickets fit; without room for those that the registers ask for the launch is another kernel's"""
    slab = 16 * 2048 * 4
    assert [E.gemm_wk_slices(Q6_K, 2048, 8704, 16, n * slab) for n in (4, 3, 2)] == [4, 3, 0]
    assert [E.gemm_wk_slices(Q6_K, 2048, 8704, 16, cnt_len=n) for n in (85, 64, 63)] == [4, 4, 0]
    assert [E.gemm_wk_slices(BF16, 2048, 7168, 16, n * slab) for n in (4, 3, 1)] == [4, 2, 0]
    assert [E.gemm_wk_slices(BF16, 1024, 4096, 16, n * slab // 2) for n in (2, 1, 0)] == [2, 1, 1]
