"""The first query of a workgroup's range is loaded before its window is planned, from the request that
holds the range's first plan tile. Ranges of one plan tile (some of them a request's switch tiles, which
hold no tokens), empty requests before, between and after, ranges that start inside a request and end in
the next, and fixed splits, in the three kernels that do so, against the oracle."""
import pytest
import torch

from tests.mla_cases import check_decode, make_case

pytestmark = pytest.mark.gpu

# (kv, rms, d_c, rope_w, heads, qrows, groups)
FAMILIES = {"ws": ("fp8", "log8", 512, 64, 24, 1, 1), "ws verify": ("fp8", "log8", 512, 64, 24, 4, 1),
            "wsb bf16": ("bf16", "bf16", 512, 64, 24, 1, 1), "wsb fp8": ("fp8", "log8", 768, 232, 24, 1, 1),
            "ro": ("fp8", "log8", 512, 64, 24, 4, 2), "ro 1 row": ("fp8", "log8", 512, 64, 24, 1, 2)}


@pytest.mark.parametrize("nwg", [1, 7, 16, 96])
@pytest.mark.parametrize("lens", [[0, 64, 0, 0, 9, 200, 0], [5, 1000, 63, 65, 64], [0, 0, 40], [777]], ids=str)
@pytest.mark.parametrize("family", sorted(FAMILIES))
def test_ranges(gpu, family, lens, nwg):
    import qmla
    kv, rms, d_c, rope_w, heads, qrows, groups = FAMILIES[family]
    c = make_case(batch=len(lens), heads=heads, d_c=d_c, rope_w=rope_w, page_size=16, lens=lens, kv=kv, rms_mode=rms,
                  seed=len(lens) + nwg, device=gpu, qrows=qrows, groups=groups, rms="spread")
    for splits in (0, 3) if nwg == 7 else (0,):
        o, lse = qmla.forward(c.q_nope, c.q_pe, c.cache, c.block_table, c.seq_lens, page_size=16, sm_scale=c.sm_scale,
                              fp8_rms=rms, k_scale=c.k_scale, qrows=qrows, groups=groups, num_splits=splits,
                              num_workgroups=nwg if splits == 0 else 0)
        torch.cuda.synchronize()
        assert not torch.isnan(o).any()
        check_decode(f"{family} {lens} nwg {nwg} splits {splits}", c, o, lse)
