"""The writer and the gather deal several rows to a wave from a few thousand rows on. Row counts at and
around that line and around whole waves and workgroups, every deployed row and rms format, rows that go
nowhere: the same bytes as the same rows in calls too small for that path (which the oracle pins)."""
import pytest
import torch

from tests.mla_cases import make_case

pytestmark = pytest.mark.gpu

# (d_c, rope_w, heads): no whole 512-column block, one, one and a half with 232 / 116 rope columns (an rms
# tail at 4 mod 8), three
ROWS = [(256, 116, 12), (512, 64, 24), (768, 232, 24), (768, 116, 12), (1792, 232, 24), (512, 64, 64)]


@pytest.mark.parametrize("rms", ["log8", "bf16", "e4m3", "none"])
@pytest.mark.parametrize("d_c,rope,heads", ROWS)
def test_write(gpu, d_c, rope, heads, rms):
    import qmla
    g = torch.Generator(device="cuda").manual_seed(d_c + rope)
    width = -(-(d_c + rope + heads * {"bf16": 2, "none": 0}.get(rms, 1)) // 16) * 16
    for n in (2047, 2048, 2049, 2055, 4095, 4096, 4097, 4103, 5003):
        pages, page = n // 48 + 2, 48
        kv_c = (torch.randn(n + 1, d_c, generator=g, device=gpu) * 200).to(torch.bfloat16)
        pe_w = -(-(rope + heads) // 8) * 8
        k_pe = torch.exp(torch.randn(n + 1, pe_w, generator=g, device=gpu)).to(torch.bfloat16)
        slots = torch.randperm(pages * page - 1, generator=torch.Generator().manual_seed(n))[:n] + 1
        slots[n // 2] = pages * page + 3                    # past the cache: skipped
        slots[n // 3] = -1                                  # padding: slot 0
        slots = slots.cuda()
        ks = torch.tensor(0.37, device=gpu)
        got = torch.full((pages, page, width), 0xAB, dtype=torch.uint8, device=gpu)
        want = got.clone()
        kw = dict(rope_w=rope, rms_heads=heads, kv_fp8=True, rms=rms, k_scale=ks)
        qmla.cache_write(kv_c, k_pe, got, slots, **kw)
        for a in range(0, n, 1000):
            qmla.cache_write(kv_c[a:], k_pe[a:], want, slots[a:a + 1000], **kw)
        assert torch.equal(got, want), (n, torch.nonzero(got != want)[:4])


@pytest.mark.parametrize("d_c,rope,heads,rms", [(448, 128, 24, "log8"), (768, 264, 24, "e4m3"), (256, 512, 24, "bf16"),
                                                (504, 516, 63, "log8"), (1016, 512, 64, "log8")])
def test_write_two_chunk_passes(gpu, d_c, rope, heads, rms):
    """Rows of more than 64 chunks besides their whole 512-column blocks: two passes over the wave, from
    65536 rows on (d_c 1016 with rope 512 is the most a row can hold; 504 with 516 has a pre-tail)."""
    import qmla
    g = torch.Generator(device="cuda").manual_seed(d_c + rope)
    width = -(-(d_c + rope + heads * (2 if rms == "bf16" else 1)) // 16) * 16
    for n in (65535, 65537):
        kv_c = (torch.randn(n, d_c, generator=g, device=gpu) * 200).to(torch.bfloat16)
        k_pe = torch.exp(torch.randn(n, -(-(rope + heads) // 8) * 8, generator=g, device=gpu)).to(torch.bfloat16)
        slots = torch.randperm(n, generator=torch.Generator().manual_seed(n)).cuda()
        slots[n // 2] = 1 << 40                             # past the cache: skipped
        got = torch.full((n // 48 + 1, 48, width), 0xAB, dtype=torch.uint8, device=gpu)
        want = got.clone()
        kw = dict(rope_w=rope, rms_heads=heads, kv_fp8=True, rms=rms, k_scale=torch.tensor(0.37, device=gpu))
        qmla.cache_write(kv_c, k_pe, got, slots, **kw)
        for a in range(0, n, 1900):
            qmla.cache_write(kv_c[a:], k_pe[a:], want, slots[a:a + 1900], **kw)
        assert torch.equal(got, want), (n, torch.nonzero(got != want)[:4])


@pytest.mark.parametrize("kv", ["fp8", "bf16"])
@pytest.mark.parametrize("n", [70, 4097])
def test_write_without_rms_elements(gpu, kv, n):
    """Rows without rms elements: k_pe is exactly the rope wide and exactly n rows long, whatever rms_heads
    says (at both of the FP8 writer's row counts), and only latent and rope are written."""
    import qmla
    d_c, rope, heads = 512, 64, 24
    g = torch.Generator(device="cuda").manual_seed(n)
    kv_c = torch.randn(n, d_c, generator=g, device=gpu).to(torch.bfloat16)
    k_pe = torch.randn(n, rope, generator=g, device=gpu).to(torch.bfloat16)
    slots = torch.randperm(96 * 48, generator=torch.Generator().manual_seed(n))[:n].cuda()
    cache = torch.full((96, 48, 608), 7, dtype=torch.uint8 if kv == "fp8" else torch.bfloat16, device=gpu)
    qmla.cache_write(kv_c, k_pe, cache, slots, rope_w=rope, rms_heads=heads, kv_fp8=kv == "fp8", rms="none",
                     k_scale=torch.ones((), device=gpu))
    rows = cache.view(-1, 608)[slots]
    want = torch.cat([kv_c, k_pe], -1)
    if kv == "fp8":
        want = want.float().clamp(-448, 448).to(torch.float8_e4m3fn).view(torch.uint8)
    assert torch.equal(rows[:, :d_c + rope], want) and bool((rows[:, d_c + rope:] == 7).all())


def _check_gather(gpu, d_c, rope, heads, rms, n, step):
    import qmla
    lens = [1, n // 3, n - 1 - n // 3 - 7, 7]
    c = make_case(batch=4, heads=heads, d_c=d_c, rope_w=rope, page_size=48, lens=lens, kv="fp8",
                  rms_mode="bf16_bytes" if rms == "bf16" else rms, seed=n, device=gpu, rms="spread", amp=4.0)
    c.cache.view(torch.uint8).view(-1)[:2048] = torch.arange(2048, device=gpu).to(torch.uint8) & 0x8F   # small, -0
    table = c.block_table.clone()
    table[1, 5] = c.cache.shape[0] + 9                  # a page outside the cache: its rows are skipped
    t = torch.tensor(lens)
    cu = torch.cat([torch.zeros(1, dtype=torch.int64), t.cumsum(0)]).to(torch.int32).cuda()
    seq = torch.repeat_interleave(torch.arange(4, dtype=torch.int32), t).cuda()
    for dtype in (torch.bfloat16, torch.float16):
        got = torch.full((n + 2, c.row), 7.0, dtype=dtype, device=gpu)
        want = got.clone()

        def gather(dst, a, m):
            qmla.gather_cache(src_cache=c.cache[:, :, 0, :], dst=dst[a:a + m], block_table=table,
                              cu_seq_lens=cu - a, token_to_seq=seq[a:a + m], num_tokens=m, kv_cache_dtype="fp8",
                              scale=c.k_scale, mla_rms=(c.rms_offset, heads, rms))

        gather(got, 0, n)
        for a in range(0, n, step):
            gather(want, a, min(step, n - a))
        assert torch.equal(got.view(torch.int16), want.view(torch.int16)), (n, dtype)


@pytest.mark.parametrize("rms", ["log8", "bf16", "e4m3"])
@pytest.mark.parametrize("d_c,rope,heads", ROWS)
def test_gather(gpu, d_c, rope, heads, rms):
    for n in (4095, 4096, 4101) + ((16383, 16384, 16387) if rms == "log8" else ()):
        _check_gather(gpu, d_c, rope, heads, rms, n, 1000)


@pytest.mark.parametrize("d_c,rope,heads,n", [(768, 232, 24, 32769), (640, 64, 24, 32770), (448, 64, 64, 32771),
                                              (960, 64, 24, 150001), (1024, 116, 12, 150003)])
def test_gather_four_rows_a_wave(gpu, d_c, rope, heads, n):
    """Four rows a wave where the line lies higher: flat chunks that fill two rows' passes, no flat chunks
    at all, and rows of 1024 columns and more (with and without a tail at 4 mod 8)."""
    _check_gather(gpu, d_c, rope, heads, "log8", n, 4000)
