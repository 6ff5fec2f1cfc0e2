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
    ("fp8", 1792, 232, 24, 1, 1, 6, 64),     # split 2, requests of 2 to 40 segments: one wave up to 8
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


@pytest.mark.parametrize("rows", [5, 120])            # the segments of a row split over waves, and not
@pytest.mark.parametrize("kv", ["fp8", "bf16"])       # fp16 and fp32 partials
@pytest.mark.parametrize("dv", [100, 102, 258, 514, 770, 1026, 2046])
def test_combine_alone_at_other_widths(gpu, dv, kv, rows):
    """qmla_combine on partials written by hand, at widths no decode kernel is compiled for: whole lane
    vectors (100) and rows that end inside one, which are read element by element. Partials of finite,
    empty (-inf) and absent segments, against float64; a combine of 32-bit weights and sums rounds a
    result to bf16 (2^-9 of itself) after some 2^-22 of its largest partial."""
    from qmla import _lib
    from qmla.decode import _stream, build_params, workspace_bytes
    heads, page, nwg = 24, 64, 37
    g = torch.Generator().manual_seed(dv + rows)
    L = torch.randint(0, 3000, (rows,), generator=g)
    L[::4] = 0
    L[1] = 9000
    width = -(-(dv + 64) // 16) * 16
    fp8 = kv == "fp8"
    cache = torch.zeros(4, page, width, dtype=torch.uint8 if fp8 else torch.bfloat16, device=gpu)
    o = torch.full((rows, heads, dv), 9.0, dtype=torch.bfloat16, device=gpu)
    lse = torch.full((rows, heads), 9.0, device=gpu)
    scale = torch.tensor(0.37, device=gpu)
    args = dict(q_nope=torch.zeros(rows, heads, dv, dtype=torch.bfloat16, device=gpu), q_pe=None, kv_cache=cache,
                block_table=torch.zeros(rows, 150, dtype=torch.int32, device=gpu), seq_lens=L.int().to(gpu), out=o, lse=lse,
                d_c=dv, rope_w=0, rms_offset=-1, rms_mode=_lib.RMS_NONE, kv=_lib.KV_FP8 if fp8 else _lib.KV_BF16,
                page_size=page, sm_scale=1.0, k_scale=scale if fp8 else None, num_splits=0, num_workgroups=nwg)
    ws = torch.zeros(workspace_bytes(build_params(**args)), dtype=torch.uint8, device=gpu)
    p = build_params(workspace=ws, **args)
    assert _lib.lib().qmla_decode_supported(p) == _lib.ERR_NOKERNEL
    _lib.check("qmla_plan", _lib.lib().qmla_plan(p, _stream()))
    plan = ws[:4 * (rows + 3)].view(torch.int32).cpu().tolist()
    chunk, first = plan[0], plan[2:]
    # the partials of slot w + b, in the workspace's layout: plan, lse, outputs, each at a multiple of 256
    slots = nwg + rows
    up = lambda x: -(-x // 256) * 256
    lse_at = up(4 * (rows + 3))
    o_at = lse_at + up(4 * slots * heads)
    pl = torch.randn(slots, heads, generator=g) * 4
    pl[torch.rand(slots, heads, generator=g) < 0.2] = float("-inf")
    po = torch.randn(slots, heads, dv, generator=g)
    if fp8:
        po = po.half()
    ws[lse_at:lse_at + pl.numel() * 4] = pl.to(gpu).view(-1).view(torch.uint8)
    area = torch.zeros(slots, heads * dv * 4, dtype=torch.uint8)
    area[:, :heads * dv * po.element_size()] = po.reshape(slots, -1).view(torch.uint8)
    ws[o_at:o_at + area.numel()] = area.to(gpu).view(-1)
    _lib.check("qmla_combine", _lib.lib().qmla_combine(p, _stream()))
    torch.cuda.synchronize()
    o, lse = o.double().cpu(), lse.double().cpu()
    merged = 0
    for b in range(rows):
        c0, c1 = first[b], first[b + 1]
        w0, w1 = c0 // chunk, (c1 - 1) // chunk
        if c1 <= c0:
            assert not o[b].any() and bool((lse[b] == float("-inf")).all())
        elif w0 == w1:
            assert bool((o[b] == 9.0).all())          # finished by its one workgroup: not the combine's
        else:
            merged += 1
            l, v = pl[w0 + b:w1 + b + 1].double(), po[w0 + b:w1 + b + 1].double()
            want_l = torch.logsumexp(l, 0)
            w = torch.where(torch.isinf(l), 0.0, torch.exp(l - want_l.nan_to_num(neginf=0.0)))
            want = (w[:, :, None] * v).sum(0) * (scale.double().cpu() if fp8 else 1.0)
            live = torch.isfinite(want_l)
            assert torch.equal(torch.isfinite(lse[b]), live)
            assert bool(((lse[b] - want_l)[live].abs() < 1e-5 * want_l[live].abs().clamp(min=1)).all())
            assert bool(((o[b] - want).abs() <= 2.0 ** -8 * want.abs() + 1e-5).all()), (o[b] - want).abs().max()
    assert merged >= 3
