"""Output rows on element boundaries only: the decode kernels write several columns per store, and a
caller's output may start anywhere and have any row and head stride. Final rows (one split, requests
that one workgroup finishes) of every warp-specialized family and type land exactly where the same call
with a dense output puts them, bit for bit, and nothing between the rows is touched."""
import pytest
import torch

from tests.mla_cases import check_decode, make_case

pytestmark = pytest.mark.gpu

# (kv, rms, d_c, heads, qrows, groups, rope_w)
FAMILIES = {
    "ws": ("fp8", "log8", 512, 24, 1, 1, 64),
    "ws_verify": ("fp8", "log8", 512, 24, 4, 1, 64),      # 3 head splits of 8 heads
    "gla": ("fp8", "log8", 512, 24, 3, 2, 64),            # rows that do not fill the last block
    "wsb_bf16": ("bf16", "bf16", 512, 23, 1, 1, 64),
    "wsb_r768": ("fp8", "log8", 768, 24, 1, 1, 232),
    "wsb_r256": ("fp8", "log8", 256, 12, 1, 1, 116),
}


@pytest.mark.parametrize("splits", [0, 1])
@pytest.mark.parametrize("dt", [torch.bfloat16, torch.float16, torch.float32], ids=["bf16", "f16", "f32"])
@pytest.mark.parametrize("family", sorted(FAMILIES))
def test_rows_on_element_boundaries(gpu, family, dt, splits):
    import qmla
    kv, rms, d_c, heads, qrows, groups, rope_w = FAMILIES[family]
    lens = [37, 0, 900, 5, 1500]
    c = make_case(batch=len(lens), heads=heads, d_c=d_c, rope_w=rope_w, page_size=64, lens=lens, kv=kv, rms_mode=rms,
                  seed=13, device=gpu, qrows=qrows, groups=groups, rms="spread")
    rows, dv = c.q_nope.shape[0], d_c // groups

    def run(o, lse):
        qmla.forward(c.q_nope, c.q_pe, c.cache, c.block_table, c.seq_lens, page_size=64, sm_scale=c.sm_scale,
                     fp8_rms=rms, k_scale=c.k_scale, qrows=qrows, groups=groups, num_splits=splits,
                     num_workgroups=5 if splits == 0 else 0, out=o, lse=lse)

    dense = torch.full((rows, heads, dv), float("nan"), dtype=dt, device=gpu)
    dlse = torch.empty(rows, heads, dtype=torch.float32, device=gpu)
    run(dense, dlse)
    sh = dv + 3                                            # odd strides, odd start
    sr = heads * sh + 5
    flat = torch.full((1 + rows * sr,), 7.0, dtype=dt, device=gpu)
    o = flat[1:].as_strided((rows, heads, dv), (sr, sh, 1))
    lse = torch.empty_like(dlse)
    run(o, lse)
    torch.cuda.synchronize()
    assert torch.equal(o, dense) and torch.equal(lse, dlse)
    o.fill_(7.0)
    assert bool((flat == 7.0).all()), "written between the rows"
    check_decode(f"{family} {dt} S={splits}", c, dense, dlse)
