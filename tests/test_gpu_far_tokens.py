"""Token and slot numbers around 2^31, where the writer and the gather change from a 32-bit
multiplication to a 64-bit division by the page size: block tables and caches just below and above that
line, in the kernels of one row and of several rows a wave."""
import pytest
import torch

from tests.mla_cases import make_case

pytestmark = pytest.mark.gpu

TOP = 2 ** 31


@pytest.mark.parametrize("n", [90, 4101])
@pytest.mark.parametrize("page,cols", [(4096, 600_000), (4095, 600_000), (4095, (TOP - 1) // 4095)], ids=str)
def test_gather(gpu, page, cols, n):
    """One sequence whose cached context ends near token 2^31: the same rows as through a table that holds
    only its last pages."""
    import qmla
    c = make_case(batch=1, heads=24, d_c=512, rope_w=64, page_size=page, lens=[4 * page], kv="fp8", rms_mode="log8",
                  seed=n, device=gpu, rms="spread")
    start = min(TOP - 1, page * cols) - n // 2
    if page * cols < TOP:
        start = page * cols - n                             # the last token of the largest table below 2^31
    first = min(start // page, cols - 3)                    # three pages hold the rows
    table = torch.full((1, cols), -1, dtype=torch.int32, device=gpu)
    table[0, first:first + 3] = c.block_table[0, :3].flip(0)
    out = []
    for bt, off in ((table, start), (table[:, first:first + 3].contiguous(), start - first * page)):
        dst = torch.full((n, c.row), 7.0, dtype=torch.bfloat16, device=gpu)
        qmla.gather_cache(src_cache=c.cache[:, :, 0, :], dst=dst, block_table=bt, num_tokens=n, kv_cache_dtype="fp8",
                          cu_seq_lens=torch.tensor([0, n], dtype=torch.int32, device=gpu),
                          token_to_seq=torch.zeros(n, dtype=torch.int32, device=gpu), scale=c.k_scale,
                          seq_starts=torch.tensor([off], dtype=torch.int32, device=gpu), mla_rms=(c.rms_offset, 24, "log8"))
        out.append(dst.view(torch.int16))
    assert torch.equal(out[0], out[1])
    assert bool((out[0][:, :c.rms_offset + 24].view(torch.bfloat16) != 7.0).any(1).all())


@pytest.mark.parametrize("kv,width", [("fp8", 16), ("bf16", 8)])
def test_write(gpu, kv, width):
    """A cache of just over 2^31 slots of 16 bytes (34 GB), rows at both sides of slot 2^31."""
    import qmla
    page, d_c = 4095, 8
    pages = TOP // page + 4
    cache = torch.empty(pages, page, width, dtype=torch.uint8 if kv == "fp8" else torch.bfloat16, device=gpu)
    for n in (7, 5001):
        kv_c = torch.randn(n, d_c, generator=torch.Generator(device="cuda").manual_seed(n), device=gpu).to(torch.bfloat16)
        slots = (TOP - 2 * n + 4 * torch.randperm(n, generator=torch.Generator().manual_seed(n))).cuda()
        qmla.cache_write(kv_c, torch.zeros(n, 8, dtype=torch.bfloat16, device=gpu), cache, slots, d_c=d_c, rope_w=0,
                         rms_heads=0, kv_fp8=kv == "fp8", rms="none", k_scale=torch.ones((), device=gpu))
        want = kv_c.float().to(torch.float8_e4m3fn).view(torch.uint8) if kv == "fp8" else kv_c
        assert int(slots.max()) > TOP > int(slots.min())
        assert torch.equal(cache.view(-1, width)[slots][:, :d_c], want)
    del cache
    torch.cuda.empty_cache()
