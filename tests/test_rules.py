"""Rules that choose between kernels, and what they ask of a step's workspace (no GPU: the library's host code alone)."""
import pytest

from gibbs_amd.ops.lib import library


@pytest.mark.parametrize("n,o", [(333, 1024), (700, 512), (1194, 1024)])
def test_float32_products_ask_for_a_workspace_where_their_kernel_uses_it(n, o):
    """Few tiles of a long inner size share their stretches through one.  Rows that are no whole 16 bytes take the plain kernel, which has
    no use for it."""
    assert library().gibbs_gemm_f32_workspace(n, o, 2052) > 0
    assert [library().gibbs_gemm_f32_workspace(n, o, 2052 + k) for k in (1, 2, 3)] == [0, 0, 0]


# us, measured without and with the stretches shared
@pytest.mark.parametrize("n,o,i,alone,shared", [
    (333, 1024, 4608, 71.3, 40.8), (1194, 1024, 2048, 56.4, 50.0), (333, 4096, 2048, 61.1, 58.9), (400, 4096, 2048, 61.5, 67.4),
    (1500, 1024, 2048, 58.0, 55.9), (1700, 1024, 2048, 59.0, 64.6), (1600, 1024, 2560, 69.2, 72.9), (1600, 1024, 3072, 82.2, 84.1),
    (1600, 1024, 4608, 119.1, 116.5), (800, 2048, 2048, 59.0, 63.2), (150, 3072, 2048, 36.1, 35.0), (65, 2048, 8192, 62.1, 61.1),
    (2048, 256, 4096, 64.9, 39.0)])
def test_float32_products_share_their_stretches_where_that_is_faster(n, o, i, alone, shared):
    assert (library().gibbs_gemm_f32_workspace(n, o, i) > 0) == (shared < alone)


# us, the general kernel in its slices and the one with 32 rows a wave in its own
@pytest.mark.parametrize("nh,nkv,hd,rows,reqs,keys,window,capped,general,wide", [
    (16, 8, 64, 45, 1, 45, 0, 0, 5.1, 4.7), (16, 16, 64, 79, 1, 79, 0, 0, 5.0, 6.6), (16, 4, 128, 45, 1, 45, 0, 0, 5.3, 7.0),
    (16, 4, 128, 128, 1, 228, 0, 0, 10.2, 12.2), (32, 8, 64, 128, 1, 828, 0, 0, 13.1, 13.7), (32, 8, 64, 64, 1, 512, 0, 0, 10.3, 11.3),
    (16, 4, 128, 64, 1, 764, 0, 0, 16.7, 17.6), (16, 8, 64, 80, 2, 622, 0, 0, 10.4, 10.9), (32, 8, 64, 256, 1, 768, 0, 0, 14.9, 15.2),
    (16, 8, 64, 256, 1, 2256, 0, 0, 16.7, 19.1), (16, 16, 64, 512, 64, 308, 0, 0, 21.9, 24.3), (16, 16, 128, 512, 1, 2012, 256, 0, 15.2, 19.0),
    (32, 8, 64, 512, 1, 2012, 1024, 0, 25.4, 28.0), (16, 8, 64, 512, 1, 512, 0, 1, 17.0, 22.8), (32, 8, 64, 512, 1, 512, 0, 1, 22.5, 23.2),
    (32, 8, 64, 512, 1, 512, 0, 0, 17.0, 11.5), (32, 8, 64, 16, 1, 4016, 0, 0, 15.2, 11.9), (32, 8, 128, 2, 1, 4002, 0, 0, 26.1, 14.6),
    (16, 4, 128, 1024, 1, 1024, 0, 0, 31.2, 27.2), (32, 8, 64, 2048, 1, 2048, 0, 0, 57.1, 35.3), (16, 8, 64, 2103, 3, 701, 0, 0, 25.5, 16.4),
    (16, 8, 64, 512, 64, 308, 0, 0, 26.5, 14.0), (32, 8, 64, 512, 1, 512, 1024, 0, 18.4, 14.8), (16, 8, 64, 2048, 1, 2048, 256, 0, 16.6, 13.5),
    (32, 8, 64, 2048, 1, 2048, 0, 1, 87.8, 81.0), (32, 8, 64, 200, 1, 8200, 0, 0, 48.4, 35.5),
    (32, 8, 64, 405, 3, 2005, 0, 0, 23.2, 25.3), (16, 8, 64, 2048, 1, 2048, 0, 1, 56.6, 64.0), (32, 8, 64, 256, 1, 2256, 0, 0, 22.9, 24.0),
    (32, 8, 64, 320, 16, 120, 0, 0, 10.1, 6.9), (16, 16, 128, 400, 1, 2400, 0, 0, 47.7, 29.8), (16, 16, 128, 256, 1, 2256, 0, 0, 24.0, 27.2)])
def test_prompt_attention_takes_the_kernel_that_is_not_slower_than_the_general_one(nh, nkv, hd, rows, reqs, keys, window, capped, general, wide):
    """The rule never takes the kernel with 32 rows a wave where that was measured slower; of the calls where it was faster it leaves the
    shortest to the general one."""
    from gibbs_amd.ops import prefill_rule
    heads = prefill_rule(rows, reqs, nh, nkv, hd, 16, keys, window, bool(capped))[1]
    assert heads != 0 if wide > general or rows == 45 else heads == 0


def test_prompt_attention_slices():
    """Slices of the kernel with 32 rows a wave, and the general kernel's own where the other does not take the heads, the pages or the call."""
    from gibbs_amd.ops import prefill_rule, prefill_splits
    lib = library()
    assert prefill_rule(2048, 1, 32, 8, 64, 16, 2048) == (1, 0)                # two workgroups a compute unit and more
    assert prefill_rule(1024, 1, 32, 8, 64, 16, 3024) == (1, 0)                # one, up to 3,000 keys a row
    assert prefill_rule(1024, 1, 32, 8, 64, 16, 9216) == (2, 0)
    assert prefill_rule(512, 1, 32, 8, 64, 16, 8192) == (4, 0)                 # 128 workgroups
    assert prefill_rule(200, 1, 32, 8, 64, 16, 4200) == (8, 0)                 # 56
    assert prefill_rule(16, 1, 32, 8, 64, 16, 4016) == (15, 0)                 # 8: slices of 256 keys
    assert prefill_rule(16, 1, 32, 8, 64, 16, 100000) == (16, 0)
    assert prefill_rule(2048, 1, 32, 8, 64, 16, 2048, 1024) == (1, 0)
    assert prefill_rule(2048, 1, 32, 8, 64, 16, 0)[0] == 1                     # no bound on the keys: the general kernel, whole
    for rows, reqs, nh, nkv, hd, page, keys, window, capped in ((64, 1, 32, 8, 64, 16, 512, 0, 0), (2048, 1, 32, 8, 64, 12, 4096, 0, 0),
                                                                (2048, 1, 32, 8, 64, 4, 4096, 0, 0), (2048, 1, 32, 8, 96, 16, 4096, 0, 0),
                                                                (512, 1, 32, 8, 64, 16, 2048, 0, 1), (300, 1, 16, 4, 128, 16, 900, 200, 0)):
        splits, heads = prefill_rule(rows, reqs, nh, nkv, hd, page, keys, window, bool(capped))
        assert splits == prefill_splits(lib.gibbs_rule_prefill_tiles(rows, reqs), nh, keys, window)
        assert heads == lib.gibbs_rule_prefill_heads(rows, reqs, nh, nkv, hd, keys, splits) > 0
