"""A workgroup's start: its range of the concatenated requests, found from the lengths 256 at a time,
and page numbers by multiplication (x / page_size = x * mul >> sh). Request counts on both sides of the
64- and 256-request batches and page sizes of every kind, in each kernel family, against the oracle."""
import random

import pytest
import torch

from tests.mla_cases import check_decode, make_case

pytestmark = pytest.mark.gpu

# (kv, rms, d_c, rope_w, heads)
FAMILIES = {"ws": ("fp8", "log8", 512, 64, 24), "wsb": ("bf16", "bf16", 512, 64, 24), "cs": ("fp8", "log8", 1792, 232, 24),
            "partial": ("fp8", "e4m3", 512, 64, 24)}


def _run(gpu, family, lens, page, nwg):
    import qmla
    kv, rms, d_c, rope_w, heads = FAMILIES[family]
    c = make_case(batch=len(lens), heads=heads, d_c=d_c, rope_w=rope_w, page_size=page, lens=lens, kv=kv, rms_mode=rms,
                  seed=len(lens) + page, device=gpu, rms="spread")
    o = torch.full((len(lens), heads, d_c), float("nan"), dtype=torch.bfloat16, device=gpu)
    _, lse = qmla.forward(c.q_nope, c.q_pe, c.cache, c.block_table, c.seq_lens, page_size=page, sm_scale=c.sm_scale,
                          fp8_rms=rms, k_scale=c.k_scale, num_workgroups=nwg, out=o)
    torch.cuda.synchronize()
    assert not torch.isnan(o).any()
    check_decode(f"{family} n{len(lens)} page {page} nwg {nwg}", c, o, lse)


@pytest.mark.parametrize("n,nwg", [(63, 40), (64, 64), (65, 9), (256, 200), (257, 256), (321, 31)])
@pytest.mark.parametrize("family", ["ws", "wsb"])
def test_request_counts(gpu, family, n, nwg):
    rng = random.Random(n)
    _run(gpu, family, [rng.choice([0, 1, 5, 64, 65, 200]) for _ in range(n - 1)] + [130], 64, nwg)


@pytest.mark.parametrize("page", [1, 3, 16, 33, 96, 1000, 4096])
@pytest.mark.parametrize("family", sorted(FAMILIES))
def test_page_sizes(gpu, family, page):
    _run(gpu, family, [700, 0, 1, page, 33, 2 * page + 1 if page < 1000 else 1001], page, 11)
