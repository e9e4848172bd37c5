"""Which form of the prefill attention a launch takes: host code, no GPU needed."""
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
