"""The balanced combine over its forms: chunks of a row split over 8, 4 or 2 waves or not at all, every
head width (one to four chunks, a last chunk partly filled), heads that do not fill a workgroup, and
requests of one to a few hundred segments, empty ones between them, on fp16 (fp8 caches) and fp32
partials. The outputs are held to the oracle, and to the same decode on one workgroup, which merges
nothing: both round P to at most 2^-9 of itself (an error of at most 2^-9 max|v| each) and the output
to bf16 (2^-9 of itself each), and the split one its partials to fp16 (2^-11 of a value <= max|v|)."""
import pytest
import torch

from tests.mla_cases import check_decode, make_case

pytestmark = pytest.mark.gpu

LENS = [2500, 0, 130, 64, 65, 700]


@pytest.mark.parametrize("kv,d_c,rope,heads,qrows,groups,batch,nwg", [
    ("fp8", 512, 64, 24, 1, 1, 1, 300),      # one request in 40 segments, 8 waves a chunk
    ("fp8", 512, 64, 24, 1, 1, 6, 64),       # 144 chunks: split 8
    ("bf16", 512, 64, 24, 1, 1, 20, 40),     # 480 chunks: split 4
    ("bf16", 512, 64, 24, 1, 1, 40, 256),    # 960 chunks: split 2
    ("fp8", 512, 64, 12, 1, 1, 120, 100),    # 1440 chunks, 12 heads: unsplit
    ("fp8", 512, 64, 23, 1, 1, 60, 64),      # 23 heads: the last workgroup's heads partly missing
    ("fp8", 768, 232, 24, 1, 1, 6, 64),      # 2 chunks, the second half filled: split 4
    ("fp8", 768, 232, 24, 1, 1, 50, 64),     # ... unsplit
    ("bf16", 1792, 64, 24, 1, 1, 3, 60),     # 4 chunks: split 2
    ("bf16", 1792, 64, 24, 1, 1, 12, 60),    # ... unsplit
    ("fp8", 512, 64, 24, 4, 2, 1, 256),      # 256 columns, 2 latent groups, verify rows: split 8
    ("fp8", 512, 64, 24, 4, 2, 24, 256),     # ... unsplit
])
def test_balanced_combine(gpu, kv, d_c, rope, heads, qrows, groups, batch, nwg):
    import qmla
    lens = [LENS[i % len(LENS)] for i in range(batch)]
    c = make_case(batch=batch, heads=heads, d_c=d_c, rope_w=rope, page_size=64, lens=lens, kv=kv,
                  rms_mode="log8" if kv == "fp8" else "bf16", seed=batch + d_c, device=gpu, qrows=qrows, groups=groups,
                  rms="spread")

    def run(n):
        return qmla.forward(c.q_nope, c.q_pe, c.cache, c.block_table, c.seq_lens, page_size=64, sm_scale=c.sm_scale,
                            k_scale=c.k_scale, qrows=qrows, groups=groups, num_workgroups=n)

    o, lse = run(nwg)
    o1, lse1 = run(1)
    torch.cuda.synchronize()
    vmax = 5.5                               # |N(0, 1)| of the cached latent, amplitude 1
    bound = 2 * (2 ** -9 * vmax + 2 ** -9 * o1.float().abs().max().item()) + 2 ** -11 * vmax
    diff = (o.float() - o1.float()).abs().max().item()
    live = torch.isfinite(lse1)
    assert torch.equal(torch.isfinite(lse), live)
    ldiff = (lse[live] - lse1[live]).abs().max().item()
    print(f"[combine {kv} {d_c} h{heads} b{batch} nwg{nwg}] split against one workgroup {diff:.2e} (bound {bound:.2e}), "
          f"lse {ldiff:.2e}", flush=True)
    assert diff <= bound and ldiff < 1e-4
    if batch <= 12:
        check_decode(f"combine {kv} {d_c} h{heads} b{batch} nwg{nwg}", c, o, lse)
