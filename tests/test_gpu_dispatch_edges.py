"""Sizes at the edges of the kernels' dispatch rules, against the oracle (bit for bit)."""

from __future__ import annotations

import pytest
import torch

from coffin_amd import _native, backend, synth
from coffin_amd.weights import QWeight, W4A8Weight
from tests import gpu_util as G

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("m,k", [(1, 8), (513, 64), (16385, 64), (31, 72), (8193, 128), (8192, 136), (4097, 256), (17, 264),
                                 (2049, 512), (2048, 520), (5, 1024), (3, 1032), (256, 520), (257, 1024)])
def test_quantiser_of_short_rows(orc, m, k):
    """Lane groups of 8 .. 64 per row, one or two rows each; rows that do not fill a workgroup."""
    x = synth.activations(m, k, synth.generator(m + k), outliers=True)
    q_ref, s_ref = orc.quant_act_i8(G.bits(x))
    q, s = G.quant(x.to(G.DEV))
    assert (q.cpu().numpy() == q_ref).all() and (s.cpu().numpy() == s_ref).all()


@pytest.mark.parametrize("m,k,skip", [(3, 1, 0), (2, 57, 0), (600, 100, 0), (5, 130, 0), (9000, 200, 1), (3, 504, 1), (300, 999, 0),
                                      (2, 1016, 0), (5, 1500, 0), (4, 3000, 3), (3, 9664, 0), (2, 16383, 0), (2, 32776, 0),
                                      (3, 33001, 0)])
def test_quantiser_of_rows_padded_to_whole_groups(orc, m, k, skip):
    """Every share of a row a lane can have, whole vectors and not, rows that start ``skip`` elements off a 16-byte boundary,
    and one whose scale is infinite: the rows that the entry leaves in its workspace, cleared past K."""
    g = synth.generator(m + k)
    x = synth.activations(m, k, g, outliers=True)
    x[m // 2, k // 2] = float("inf")
    q_ref, s_ref = orc.quant_act_i8(G.bits(x))
    xd = torch.empty(m * k + skip, dtype=torch.bfloat16, device=G.DEV)[skip:].view(m, k)
    xd.copy_(x)
    w = W4A8Weight.quantize(synth.dense_weight(16, k, g), group_size=128)
    w4, ws = G.w4_repack(w.packed.to(G.DEV), w.scale.to(G.DEV), k)
    lib = _native.load()
    kd = int(lib.cmi_w4_device_k(k, 128))
    nbytes = int(lib.cmi_linear_workspace_bytes(m, kd))
    work = torch.full((nbytes,), 0xA5, dtype=torch.uint8, device=G.DEV)
    y = torch.empty((m, 16), dtype=torch.bfloat16, device=G.DEV)
    _native.check(lib.cmi_linear_w4a8_bf16(G.ptr(w4), G.ptr(ws), G.ptr(xd), G.ptr(y), m, 16, k, 128, G.ptr(work), nbytes,
                                           G.stream()), "linear_w4a8_bf16")
    rows = work[:m * kd].view(torch.int8).view(m, kd).cpu()
    at = (m * kd + 255) // 256 * 256
    assert (rows[:, :k].numpy() == q_ref).all() and not rows[:, k:].any()
    assert (work[at:at + 4 * m].view(torch.float32).cpu().numpy() == s_ref).all()


@pytest.mark.parametrize("m,k", [(256, 8192), (257, 8192), (2, 8200), (257, 1032), (258, 16392), (3, 24584), (257, 32768), (2, 32776),
                                 (512, 2048), (513, 2048), (300, 2056), (3, 520), (7, 1544), (5, 2560), (9, 3072)])
def test_silu_mul_quant_at_the_edges_of_a_thread_s_share(orc, m, k):
    g = synth.generator(m + k)
    gate, up = (torch.randn((m, 2 * k), generator=g) * 3).to(torch.bfloat16).split(k, dim=1)
    gd, ud = (torch.cat([gate, up], dim=1).to(G.DEV)).split(k, dim=1)
    out = torch.empty((m, k), dtype=torch.bfloat16, device=G.DEV)
    q = torch.empty((m, k), dtype=torch.int8, device=G.DEV)
    s = torch.empty(m, dtype=torch.float32, device=G.DEV)
    lib = _native.load()
    rows = [0, 1, m - 1]
    o_ref, q_ref, s_ref = orc.silu_mul_quant(G.bits(gate[rows].contiguous()), G.bits(up[rows].contiguous()))
    for quantised in (True, False):
        out.zero_()
        _native.check(lib.cmi_silu_mul_quant(G.ptr(gd), G.ptr(ud), G.ptr(out), G.ptr(q if quantised else None),
                                             G.ptr(s if quantised else None), m, k, 2 * k, 2 * k, k, G.stream()), "silu")
        assert (G.bits(out[rows]) == o_ref).all()
    assert (q[rows].cpu().numpy() == q_ref).all() and (s[rows].cpu().numpy() == s_ref).all()


@pytest.mark.parametrize("m,n", [(256, 1024), (257, 512), (259, 520), (257, 1024), (2, 1032), (300, 8192), (3, 8200), (2, 16392),
                                 (257, 32768), (2, 32776), (1281, 1032), (1280, 1280), (2049, 1536), (1283, 1544), (4097, 1280),
                                 (4098, 1288), (3, 12288), (258, 8200), (1281, 2048), (1300, 2056)])
@pytest.mark.parametrize("with_add", [True, False])
def test_rms_norm_i8_at_the_edges_of_a_row_s_wavefronts(orc, m, n, with_add):
    g = synth.generator(m + n)
    x, add = synth.activations(m, n, g), synth.activations(m, n, g)
    gain = (1 + 0.1 * torch.randn(n, generator=g)).to(torch.bfloat16)
    xd, y = x.to(G.DEV), torch.empty((m, n), dtype=torch.bfloat16, device=G.DEV)
    q = torch.empty((m, n), dtype=torch.int8, device=G.DEV)
    s = torch.empty(m, dtype=torch.float32, device=G.DEV)
    ad, gd = add.to(G.DEV), gain.to(G.DEV)
    lib = _native.load()
    if with_add:
        rc = lib.cmi_add_rms_norm_i8(G.ptr(xd), G.ptr(ad), G.ptr(gd), G.ptr(y), G.ptr(q), G.ptr(s), m, n, n, n, n, 1e-6, G.stream())
    else:
        rc = lib.cmi_rms_norm_i8(G.ptr(xd), G.ptr(gd), G.ptr(y), G.ptr(q), G.ptr(s), m, n, n, n, 1e-6, G.stream())
    _native.check(rc, "rms_norm_i8")
    rows = [0, 1, m - 1]
    total = ((x.float() + add.float()).to(torch.bfloat16) if with_add else x)[rows].contiguous()
    y_ref, _ = orc.rms_norm(G.bits(total), G.bits(gain))
    q_ref, s_ref = orc.quant_act_i8(y_ref)
    assert (G.bits(xd[rows]) == G.bits(total)).all() and (G.bits(y[rows]) == y_ref).all()
    assert (q[rows].cpu().numpy() == q_ref).all() and (s[rows].cpu().numpy() == s_ref).all()


@pytest.mark.parametrize("gs", [128, 64, 256])
@pytest.mark.parametrize("tile", [64, 128, 192, 128192, 256, 320, 321, 6464])
@pytest.mark.parametrize("m,n,k", [(17, 33, 256), (129, 161, 256), (65, 97, 512), (130, 264, 768), (33, 129, 1024), (257, 40, 1280)])
def test_w4a8_tiles_at_their_edges(orc, tile, m, n, k, gs):
    """Every tile with a remainder in both directions, one to ten steps (fewer than it has stages, and whole chunks of
    four and not), odd and 16-byte rows of results."""
    g = synth.generator(m + n + k)
    w = synth.int4_weight(n, k, g, group_size=gs)
    x = synth.activations(m, k, g, outliers=True)
    xq, xs = orc.quant_act_i8(G.bits(x))
    _, y_ref = orc.linear_w4a8(xq, xs, w.packed.numpy(), w.scale.numpy(), k, gs)
    w4, ws = G.w4_repack(w.packed.to(G.DEV), w.scale.to(G.DEV), k, gs)
    G.set_option("gemm_tile", tile)
    _, y = G.w4a8(w4, ws, G.dev(xq), G.dev(xs), k, gemm=True, want_acc=False, gs=gs)
    assert (G.bits(y) == y_ref).all()


@pytest.mark.parametrize("gs", [128, 64, 256])
def test_w4a8_tiles_with_scales_near_the_end_of_the_range(orc, gs):
    """Scales whose sixteenth is not exact (below 2^-122, down to the last denormal), beside ordinary ones, zero and the
    largest: the tiles carry 16 times the sums and a sixteenth of the scale where they can."""
    g = synth.generator(gs)
    m, n, k = 70, 200, 1024
    w = synth.int4_weight(n, k, g, group_size=gs)
    exponent = torch.randint(-149, -118, w.scale.shape, generator=g)
    scale = torch.ldexp(1 + torch.rand(w.scale.shape, generator=g, dtype=torch.float64), exponent.double()).float()
    scale[:, ::3] = w.scale[:, ::3]                                # columns without a tiny scale
    scale[1, 3::5] = 0.0
    scale[0, 6::12] = 1e30
    x = (synth.activations(m, k, g).float() * 1e4).to(torch.bfloat16)
    xq, xs = orc.quant_act_i8(G.bits(x))
    _, y_ref = orc.linear_w4a8(xq, xs, w.packed.numpy(), scale.numpy(), k, gs)
    w4, ws = G.w4_repack(w.packed.to(G.DEV), scale.to(G.DEV), k, gs)
    assert (ws.cpu().view(torch.int32) == scale.t().contiguous().view(torch.int32)).all()
    for tile in (64, 128, 192, 128192, 256, 320, 321, 6464):
        G.set_option("gemm_tile", tile)
        _, y = G.w4a8(w4, ws, G.dev(xq), G.dev(xs), k, gemm=True, want_acc=False, gs=gs)
        assert (G.bits(y) == y_ref).all(), tile
    G.set_option("gemm_tile", 0)
    _, y = G.w4a8(w4, ws, G.dev(xq[:5]), G.dev(xs[:5]), k, gemm=False, want_acc=False, gs=gs)
    assert (G.bits(y) == y_ref[:5]).all()


@pytest.mark.parametrize("k", [128, 384, 640])
def test_w4a8_tiles_with_a_step_count_that_is_no_whole_chunk(orc, k):
    g = synth.generator(k)
    n, m = 200, 70
    w = synth.int4_weight(n, k, g)
    x = synth.activations(m, k, g)
    xq, xs = orc.quant_act_i8(G.bits(x))
    _, y_ref = orc.linear_w4a8(xq, xs, w.packed.numpy(), w.scale.numpy(), k, 128)
    w4, ws = G.w4_repack(w.packed.to(G.DEV), w.scale.to(G.DEV), k, 128)
    for tile in (64, 128, 192, 128192, 256, 320, 321, 6464):
        G.set_option("gemm_tile", tile)
        _, y = G.w4a8(w4, ws, G.dev(xq), G.dev(xs), k, gemm=True, want_acc=False)
        assert (G.bits(y) == y_ref).all(), tile


@pytest.mark.parametrize("m,n,k", [(1, 24, 128), (3, 40, 512), (17, 33, 640), (16, 64, 1024), (33, 65, 384), (47, 130, 1152), (49, 129, 2560), (97, 200, 3712),
                                   (65, 96, 4608)])
def test_w4a8_tiles_of_four_groups_a_step(orc, m, n, k):
    """One to many steps and one to four groups in the last, ragged in both directions, odd and 16-byte rows of results; then
    with scales below 2^-122 in some columns."""
    g = synth.generator(m + n + k)
    w = synth.int4_weight(n, k, g)
    x = synth.activations(m, k, g, outliers=True)
    xq, xs = orc.quant_act_i8(G.bits(x))
    tiny = w.scale.clone()
    tiny[:, ::3] = torch.ldexp(torch.ones(1), torch.tensor(-126)).item()
    tiny[k // 128 - 1, 1::3] = 2.0 ** -140
    tiny[0, 2::3] = 0.0
    for scale in (w.scale, tiny):
        _, y_ref = orc.linear_w4a8(xq, xs, w.packed.numpy(), scale.numpy(), k, 128)
        w4, ws = G.w4_repack(w.packed.to(G.DEV), scale.to(G.DEV), k)
        for code in (1664, 1665, 3232, 3233, 3264, 3265, 4864):
            G.set_option("w4_gemm_deep", code)
            _, y = G.w4a8(w4, ws, G.dev(xq), G.dev(xs), k, gemm=True, want_acc=False)
            assert (G.bits(y) == y_ref).all(), code
            if 3 <= m <= 16:
                _, y = G.w4a8(w4, ws, G.dev(xq), G.dev(xs), k, gemm=False, want_acc=False)
                assert (G.bits(y) == y_ref).all(), code
        G.set_option("w4_gemm_deep", 0)


@pytest.mark.parametrize("gs,m,n,k", [(64, 1, 24, 128), (64, 3, 40, 512), (64, 17, 33, 640), (64, 16, 64, 1024), (64, 33, 65, 384), (64, 49, 129, 2560),
                                      (64, 65, 96, 4608), (256, 1, 24, 256), (256, 5, 40, 512), (256, 17, 33, 768), (256, 16, 64, 1024),
                                      (256, 47, 130, 1280), (256, 97, 200, 3840)])
def test_w4a8_tiles_of_four_steps_of_other_groups(orc, gs, m, n, k):
    """Groups of 64 and 256: part of a stage to many, ragged in both directions; then with scales below 2^-122 in some columns."""
    g = synth.generator(gs + m + n + k)
    w = synth.int4_weight(n, k, g, group_size=gs)
    x = synth.activations(m, k, g, outliers=True)
    xq, xs = orc.quant_act_i8(G.bits(x))
    tiny = w.scale.clone()
    tiny[:, ::3] = 2.0 ** -126
    tiny[k // gs - 1, 1::3] = 2.0 ** -140
    tiny[0, 2::3] = 0.0
    for scale in (w.scale, tiny):
        _, y_ref = orc.linear_w4a8(xq, xs, w.packed.numpy(), scale.numpy(), k, gs)
        w4, ws = G.w4_repack(w.packed.to(G.DEV), scale.to(G.DEV), k, gs)
        for code in (0, 1664, 1665, 3232, 3233, 3264, 3265, 4864):
            G.set_option("w4_gemm_deep", code)
            for gemm in (True, False) if m <= 16 else (True,):
                _, y = G.w4a8(w4, ws, G.dev(xq), G.dev(xs), k, gemm=gemm, want_acc=False, gs=gs)
                assert (G.bits(y) == y_ref).all(), (code, gemm)
        G.set_option("w4_gemm_deep", 0)


@pytest.mark.parametrize("gs,k", [(64, 128), (64, 384), (64, 640), (64, 1024), (64, 2560), (64, 2688), (64, 4096), (64, 5120), (64, 5248), (64, 8192),
                                  (64, 8320), (64, 10240), (64, 12416), (64, 20480), (64, 20608), (256, 256), (256, 768), (256, 1024), (256, 2560),
                                  (256, 2816), (256, 5120), (256, 5376), (256, 10240), (256, 10496), (256, 20480), (256, 20736)])
def test_w4a8_rows_of_other_groups(orc, gs, k):
    """One row (quantised by the kernel or before it; every number of loads per wavefront, whole and not) and 2..16 rows (one
    line per wavefront to several passes, half lines)."""
    g = synth.generator(gs + k)
    n = 37
    w = synth.int4_weight(n, k, g, group_size=gs)
    x = synth.activations(16, k, g, outliers=True)
    xq, xs = orc.quant_act_i8(G.bits(x))
    sums_ref, y_ref = orc.linear_w4a8(xq, xs, w.packed.numpy(), w.scale.numpy(), k, gs, want_group_acc=True)
    w4, ws = G.w4_repack(w.packed.to(G.DEV), w.scale.to(G.DEV), k, gs)
    lib = _native.load()
    work = torch.empty(int(lib.cmi_linear_workspace_bytes(16, k)), dtype=torch.uint8, device=G.DEV)
    xd = x.to(G.DEV)
    for m in (1, 2, 5, 16):
        _, y = G.w4a8(w4, ws, G.dev(xq[:m]), G.dev(xs[:m]), k, gemm=False, want_acc=False, gs=gs)
        assert (G.bits(y) == y_ref[:m]).all(), m
        y = torch.empty((m, n), dtype=torch.bfloat16, device=G.DEV)
        _native.check(lib.cmi_linear_w4a8_bf16(G.ptr(w4), G.ptr(ws), G.ptr(xd), G.ptr(y), m, n, k, gs, G.ptr(work), work.numel(),
                                               G.stream()), "linear_w4a8_bf16")
        assert (G.bits(y) == y_ref[:m]).all(), m
    sums, y = G.w4a8(w4, ws, G.dev(xq[:1]), G.dev(xs[:1]), k, gemm=False, gs=gs)
    assert (sums.cpu().numpy() == sums_ref[:1]).all() and (G.bits(y) == y_ref[:1]).all()


@pytest.mark.parametrize("gs", [64, 256])
def test_one_row_of_other_groups_off_a_16_byte_boundary(orc, gs):
    g = synth.generator(gs)
    k, n = 2560, 24
    w = synth.int4_weight(n, k, g, group_size=gs)
    x = synth.activations(1, k, g)
    xq, xs = orc.quant_act_i8(G.bits(x))
    _, y_ref = orc.linear_w4a8(xq, xs, w.packed.numpy(), w.scale.numpy(), k, gs)
    w4, ws = G.w4_repack(w.packed.to(G.DEV), w.scale.to(G.DEV), k, gs)
    xd = torch.empty(k + 1, dtype=torch.bfloat16, device=G.DEV)[1:].view(1, k)
    xd.copy_(x)
    lib = _native.load()
    work = torch.empty(int(lib.cmi_linear_workspace_bytes(1, k)), dtype=torch.uint8, device=G.DEV)
    y = torch.empty((1, n), dtype=torch.bfloat16, device=G.DEV)
    _native.check(lib.cmi_linear_w4a8_bf16(G.ptr(w4), G.ptr(ws), G.ptr(xd), G.ptr(y), 1, n, k, gs, G.ptr(work), work.numel(),
                                           G.stream()), "linear_w4a8_bf16")
    assert (G.bits(y) == y_ref).all()


@pytest.mark.parametrize("m,n,k", [(16, 12288, 4096), (16, 32768, 5120), (5, 24238, 9728), (40, 2560, 9728), (70, 6144, 2560), (200, 2560, 9728)])
def test_w4a8_rows_through_the_chosen_tile(m, n, k):
    """Sizes where the choice is a tile of four groups a step: the results of the kernels without them."""
    if m <= 16:
        assert G.chosen_tile("_ZN3cmi20w4a8_rows_take_tilesEiiiPi", m, n, k)[0]
    else:
        assert G.chosen_tile("_ZN3cmi17gemm_w4a8_tile_usEiiiiPi", m, n, k, 128)[1] >= 8
    gen = torch.Generator(device=G.DEV).manual_seed(m + n + k)
    w4 = torch.randint(0, 256, (n, k // 2), dtype=torch.uint8, device=G.DEV, generator=gen)
    ws = torch.rand((n, k // 128), device=G.DEV, generator=gen) * 0.01 + 1e-4
    xq = torch.randint(-127, 128, (m, k), dtype=torch.int8, device=G.DEV, generator=gen)
    xs = torch.rand(m, device=G.DEV, generator=gen) + 0.5
    _, y = G.w4a8(w4, ws, xq, xs, k, gemm=m > 16, want_acc=False)
    G.set_option("w4_gemm_deep", 1)
    _, ref = G.w4a8(w4, ws, xq, xs, k, gemm=m > 16, want_acc=False)
    assert torch.equal(y.view(torch.int16), ref.view(torch.int16))


@pytest.mark.parametrize("n,k", [(65535, 2064), (65536, 1040), (65537, 3072), (70001, 4096), (65536, 1024), (65600, 4112), (65537, 1664), (65539, 2560), (300, 2560),
                                 (4096, 4096), (4097, 4096), (33, 9728)])
def test_weight_only_rows_keep_the_single_row_s_bits_at_the_edges_of_the_row_blocks(n, k):
    """Tall weights that are streamed or whose workgroups follow each other, and few outputs; last segments nearly empty, half full and
    full: integers of both signs, every row against the call with that row alone."""
    gen = torch.Generator(device=G.DEV).manual_seed(n + k)
    wq = torch.randint(-127, 128, (n, k), dtype=torch.int8, device=G.DEV, generator=gen)
    ws = torch.rand(n, device=G.DEV, generator=gen) * 0.01
    x = torch.randn((16, k), device=G.DEV, generator=gen).to(torch.bfloat16)
    lib = _native.load()

    def call(rows):
        y = torch.full((rows.shape[0], n), float("nan"), dtype=torch.bfloat16, device=G.DEV)
        _native.check(lib.cmi_gemv_w8a16(G.ptr(wq), G.ptr(ws), G.ptr(rows), G.ptr(y), rows.shape[0], n, k, G.stream()), "gemv")
        return y

    ref = torch.cat([call(x[r:r + 1].contiguous()) for r in range(16)])
    for m in (3, 4, 8, 9, 12, 13, 16):
        assert torch.equal(call(x[:m].contiguous()).view(torch.int16), ref[:m].view(torch.int16)), m


@pytest.mark.parametrize("m,n,k", [(17, 24, 128), (192, 256, 256), (193, 257, 384), (500, 300, 512), (385, 1000, 640), (576, 520, 2560),
                                   (31, 513, 4096)])
def test_192_row_tile_of_the_w8a8_gemm(orc, m, n, k):
    """Ragged in both directions, one to many K steps."""
    gen = synth.generator(m + n + k)
    q = synth.int8_weight(n, k, gen)
    x = synth.activations(m, k, gen, outliers=True)
    xq, xs = orc.quant_act_i8(G.bits(x))
    acc_ref, y_ref = orc.gemm_w8a8(xq, q.wq.numpy(), xs, q.scale.numpy())
    G.set_option("gemm_tile", 256192)  # (conftest resets it)
    acc, y = G.gemm_w8a8(G.dev(xq), q.wq.to(G.DEV), G.dev(xs), q.scale.to(G.DEV))
    assert (acc.cpu().numpy() == acc_ref).all() and (G.bits(y) == y_ref).all()


def _with_neighbours(a: torch.Tensor) -> torch.Tensor:
    """``a`` on the device, the bytes behind its last row 127."""
    home = torch.full((a.numel() + 512,), 127, dtype=a.dtype, device=G.DEV)
    home[:a.numel()] = a.reshape(-1).to(G.DEV)
    return home[:a.numel()].view(a.shape)


@pytest.mark.parametrize("m,n,k", [(3, 40, 144), (16, 33, 2064), (17, 8, 240), (31, 530, 1232), (70, 200, 9664), (100, 300, 10256), (129, 161, 208),
                                   (200, 520, 192), (260, 264, 1040), (300, 2560, 2496), (577, 650, 320), (200, 2560, 9664), (300, 2560, 9664)])
def test_w8a8_rows_that_end_inside_a_step(orc, m, n, k):
    """K of 16 .. 112 more than whole steps of 128: the library's choice (up to 16 rows, 17..256, beyond), then every tile (320 names
    the 256 x 256 one at such K), then with room to split K, which each of the three split tiles does at one size: 64 x 64, 128 x 64
    and 128 x 128.  Beyond a row's end lie other rows' values."""
    g = synth.generator(m + n + k)
    q = synth.int8_weight(n, k, g)
    x = synth.activations(m, k, g, outliers=True)
    xq, xs = orc.quant_act_i8(G.bits(x))
    acc_ref, y_ref = orc.gemm_w8a8(xq, q.wq.numpy(), xs, q.scale.numpy())
    xd, wd = _with_neighbours(torch.from_numpy(xq)), _with_neighbours(q.wq)
    xsd, wsd = G.dev(xs), q.scale.to(G.DEV)
    for tile in (0, 6464, 64, 128, 192, 128192, 256, 256192, 320, 321):
        G.set_option("gemm_tile", tile)
        acc, y = G.gemm_w8a8(xd, wd, xsd, wsd)
        assert (acc.cpu().numpy() == acc_ref).all() and (G.bits(y) == y_ref).all(), tile
    G.set_option("gemm_tile", 0)
    lib = _native.load()
    nbytes = int(lib.cmi_linear_w8a8_workspace_bytes(m, n, k))
    work = torch.full((nbytes,), 0xA5, dtype=torch.uint8, device=G.DEV)
    xb, y = x.to(G.DEV), torch.empty((m, n), dtype=torch.bfloat16, device=G.DEV)
    _native.check(lib.cmi_linear_w8a8_bf16(G.ptr(xb), G.ptr(wd), G.ptr(wsd), G.ptr(y), m, n, k, n, G.ptr(work), nbytes, G.stream()), "linear")
    assert (G.bits(y) == y_ref).all()
    partials = work[int(lib.cmi_linear_workspace_bytes(m, k)) + 1024:]         # behind the rows, their scales and the arrival counters
    assert bool((partials != 0xA5).any()) == ((m, n, k) in ((100, 300, 10256), (200, 2560, 9664), (300, 2560, 9664)))


@pytest.mark.parametrize("path", ["compiled", "adapters"])
@pytest.mark.parametrize("rows,k,n", [(64, 2560, 512), (65, 9728, 512), (100, 9728, 2560), (256, 4096, 512), (257, 9728, 2560), (500, 9728, 2560), (500, 2560, 6144),
                                      (1024, 2048, 256), (1025, 2048, 256)])
def test_w8a8_rows_are_handed_over_where_k_is_not_split(request, monkeypatch, rows, k, n, path):
    """Both sides of the rule at its edges: the bits of the call that quantises the bf16 rows."""
    request.addfinalizer(backend._drop_handed)                     # the adapters' rows are not for the compiled path
    g = synth.generator(rows + k)
    if path == "adapters":
        for name in backend._HOST_CALLS:
            monkeypatch.setattr(backend, "_host_" + name, lambda *args: None)
    used, real = [], backend._rows_quantised
    monkeypatch.setattr(backend, "_rows_quantised", lambda *args: (used.append(1), real(*args)))
    q = synth.int8_weight(n, k, g)
    w = QWeight(q.wq.to(G.DEV), q.scale.to(G.DEV))
    x = synth.activations(rows, k, g).to(G.DEV)
    gain = synth.activations(1, k, g)[0].to(G.DEV).contiguous()
    backend.linear_prefill(w, x)                                   # a quantising consumer has been seen
    before = _native.load_host().handed_uses()[1]
    h = backend.rms_norm(x, gain)
    y = backend.linear_prefill(w, h)
    taken = len(used) + _native.load_host().handed_uses()[1] - before
    assert taken == (0 if backend._splits_k(rows, n, k, x.device) else 1)
    assert torch.equal(y.view(torch.int16), backend.linear_prefill(w, h.clone()).view(torch.int16))


@pytest.mark.parametrize("m,n,k", [(5, 24, 128), (3, 40, 144), (16, 33, 1040), (17, 48, 1104), (33, 100, 2576), (64, 70, 2624), (63, 4808, 2624), (9, 4808, 2672),
                                   (50, 32784, 1296), (6, 32784, 1296), (49, 60, 5008), (17, 60, 5136), (64, 60, 10192), (16, 40, 10288), (20, 40, 10256),
                                   (40, 33, 13888), (64, 33, 13824), (65, 20, 20496), (1, 24, 2624)])
def test_matrix_pipe_rows_that_end_inside_a_line(m, n, k):
    """Every arrangement of the kernel, with what lies behind a row -- the next row, or NaN behind the last -- kept out of its sums;
    a row's bits are those of a call of sixteen."""
    g = synth.generator(m + n + k)
    q = synth.int8_weight(n, k, g)
    x = synth.activations(m, k, g, outliers=True)
    buf = torch.full((m * k + 256,), float("nan"), dtype=torch.bfloat16, device=G.DEV)
    xd = buf[:m * k].view(m, k)
    xd.copy_(x)
    wd, wsd = q.wq.to(G.DEV), q.scale.to(G.DEV)
    lib = _native.load()

    def call(rows):
        y = torch.full((rows.shape[0], n), float("nan"), dtype=torch.bfloat16, device=G.DEV)
        _native.check(lib.cmi_linear_w8a16_rows(G.ptr(wd), G.ptr(wsd), G.ptr(rows), G.ptr(y), rows.shape[0], n, k, G.stream()), "rows")
        return y

    y = call(xd)
    exact = (x.double() @ q.wq.double().t()) * q.scale.double()
    # fp32 sums of K exact products, then bf16: K eps of the sum of magnitudes, half a bf16 step of the result
    slack = (x.double().abs() @ q.wq.double().abs().t()) * q.scale.double() * (k * 2.0 ** -24)
    assert ((y.cpu().double() - exact).abs() <= slack + exact.abs() * 2.0 ** -8).all()
    if m < 16:
        more = synth.activations(16 - m, k, g).to(G.DEV)
        assert torch.equal(call(torch.cat([xd, more]))[:m].view(torch.int16), y.view(torch.int16))
    for lo in {*range(0, m - 15, 16), m - 16} if m > 16 else ():
        assert torch.equal(call(xd[lo:lo + 16].contiguous()).view(torch.int16), y[lo:lo + 16].view(torch.int16)), lo
    if k % 128 == 0 and m <= 64:
        ref = torch.empty_like(y)
        _native.check(lib.cmi_linear_w8a16(G.ptr(wd), G.ptr(wsd), G.ptr(xd), G.ptr(ref), m, n, k, 1, G.stream()), "mfma")
        assert torch.equal(ref.view(torch.int16), y.view(torch.int16))


@pytest.mark.parametrize("m,k", [(16, 5200), (63, 9664), (16, 13888), (40, 25536)])
def test_matrix_pipe_sums_of_rows_that_end_inside_a_line_are_as_exact_as_the_dot_product_s(m, k):
    """Rows whose products cancel to zero, so that a result is the error of its sum: in the root mean square no larger than the
    single-row order's (5 % for the sample: m x 2048 sums, and a ratio of 0.93 at 5200, 0.65 at 25536)."""
    n = 2048
    gen = torch.Generator(device=G.DEV).manual_seed(k)
    wq = (torch.randn((n, k), device=G.DEV, generator=gen) * 30).round().clamp(-127, 127).to(torch.int8)
    x = torch.randn((m, k), device=G.DEV, generator=gen).to(torch.bfloat16)
    order = torch.randperm(k, device=G.DEV, generator=gen)
    wq[:, order[k // 2:]], x[:, order[k // 2:]] = wq[:, order[:k // 2]], -x[:, order[:k // 2]]
    ws = torch.ones(n, device=G.DEV)
    magnitude = x.float().abs() @ wq.float().abs().t()
    lib = _native.load()
    rms = []
    for call in (lambda y: lib.cmi_linear_w8a16(G.ptr(wq), G.ptr(ws), G.ptr(x), G.ptr(y), m, n, k, 0, G.stream()),
                 lambda y: lib.cmi_linear_w8a16_rows(G.ptr(wq), G.ptr(ws), G.ptr(x), G.ptr(y), m, n, k, G.stream())):
        y = torch.empty((m, n), dtype=torch.bfloat16, device=G.DEV)
        _native.check(call(y), "w8a16")
        rms.append((y.double() / magnitude.double()).square().mean().sqrt().item() * 2.0 ** 24)
    assert rms[1] <= 1.05 * rms[0], rms


@pytest.mark.parametrize("m,k", [(9, 2640), (16, 5200), (40, 9664), (9, 13888), (40, 13888)])
def test_matrix_pipe_sums_of_rows_that_end_inside_a_line_that_are_infinite(m, k):
    """Infinite activations, and finite ones whose products or sums leave the range, with a NaN row beside them: the infinities,
    signs and NaN of the single-row order."""
    n = 48
    gen = torch.Generator(device=G.DEV).manual_seed(m + k)
    wq = torch.randint(1, 128, (n, k), dtype=torch.int8, device=G.DEV, generator=gen)
    wq[1::2] = -wq[1::2]
    x = torch.randn((m, k), device=G.DEV, generator=gen).to(torch.bfloat16)
    x[0, 5], x[1, k - 1], x[2, k // 2] = float("inf"), float("-inf"), 3e38
    x[3, 7::128] = 2e36                                            # a sum that overflows on the way
    x[4, 3], x[5, 3], x[5, k - 3] = float("nan"), float("inf"), float("-inf")
    wq[:, 7::128] = wq[:, 7:8]
    wq[:, 3], wq[:, k // 2] = wq[:, 5], wq[:, 5]
    wq[:, k - 3] = wq[:, 3]
    ws = torch.rand(n, device=G.DEV, generator=gen) * 0.01 + 1e-3
    lib = _native.load()
    dot, rows = (torch.empty((m, n), dtype=torch.bfloat16, device=G.DEV) for _ in range(2))
    _native.check(lib.cmi_linear_w8a16(G.ptr(wq), G.ptr(ws), G.ptr(x), G.ptr(dot), m, n, k, 0, G.stream()), "dot")
    _native.check(lib.cmi_linear_w8a16_rows(G.ptr(wq), G.ptr(ws), G.ptr(x), G.ptr(rows), m, n, k, G.stream()), "rows")
    assert dot[:2].isinf().all() and dot[4:6].isnan().all() and dot[6:].isfinite().all()
    for kind in (torch.isposinf, torch.isneginf, torch.isnan):
        assert torch.equal(kind(rows), kind(dot)), kind


@pytest.mark.parametrize("m,n,k,dot", [(5, 300, 12304, True), (8, 512, 16368, True), (9, 300, 12304, False), (8, 300, 9200, False), (6, 300, 8208, True),
                                       (6, 832, 9200, True), (7, 832, 9200, False), (5, 1024, 16368, True), (5, 1025, 16368, False),
                                       (5, 300, 8176, False), (5, 300, 16400, False), (5, 512, 20496, True), (6, 512, 20496, False)])
def test_few_outputs_of_long_rows_that_end_inside_a_line(m, n, k, dot):
    """Both sides of the rule at its edges.  The products cancel to zero, so that a result is what its sum rounded off and the bits say
    which kernel formed it; at most K eps of the sum of magnitudes."""
    gen = torch.Generator(device=G.DEV).manual_seed(m + n + k)
    wq = torch.randint(-127, 128, (n, k), dtype=torch.int8, device=G.DEV, generator=gen)
    ws = torch.ones(n, device=G.DEV)
    x = torch.randn((m, k), device=G.DEV, generator=gen).to(torch.bfloat16)
    order = torch.randperm(k, device=G.DEV, generator=gen)
    wq[:, order[k // 2:]], x[:, order[k // 2:]] = wq[:, order[:k // 2]], -x[:, order[:k // 2]]
    lib = _native.load()
    one, rows = (torch.empty((m, n), dtype=torch.bfloat16, device=G.DEV) for _ in range(2))
    _native.check(lib.cmi_linear_w8a16(G.ptr(wq), G.ptr(ws), G.ptr(x), G.ptr(one), m, n, k, 0, G.stream()), "dot")
    _native.check(lib.cmi_linear_w8a16_rows(G.ptr(wq), G.ptr(ws), G.ptr(x), G.ptr(rows), m, n, k, G.stream()), "rows")
    assert torch.equal(one.view(torch.int16), rows.view(torch.int16)) == dot
    assert (rows.double().abs() <= (x.double().abs() @ wq.double().abs().t()) * (k * 2.0 ** -24)).all()


@pytest.mark.parametrize("path", ["compiled", "adapters"])
def test_ragged_rows_take_the_matrix_pipe_where_the_call_site_may(monkeypatch, path):
    if path == "adapters":
        for name in backend._HOST_CALLS:
            monkeypatch.setattr(backend, "_host_" + name, lambda *args: None)
    g = synth.generator(3)
    k, n = 1344, 200
    q = synth.int8_weight(n, k, g)
    w = QWeight(q.wq.to(G.DEV), q.scale.to(G.DEV))
    lib = _native.load()
    for rows in (4, 5, 40):
        x = synth.activations(rows, k, g).to(G.DEV)
        dot, pipe = (torch.empty((rows, n), dtype=torch.bfloat16, device=G.DEV) for _ in range(2))
        _native.check(lib.cmi_linear_w8a16(G.ptr(w.wq), G.ptr(w.scale), G.ptr(x), G.ptr(dot), rows, n, k, 0, G.stream()), "dot")
        _native.check(lib.cmi_linear_w8a16_rows(G.ptr(w.wq), G.ptr(w.scale), G.ptr(x), G.ptr(pipe), rows, n, k, G.stream()), "rows")
        want = pipe if rows >= 5 else dot
        assert torch.equal(backend.linear_m_verify(w, x).view(torch.int16), want.view(torch.int16))
        assert torch.equal(backend.linear_prefill(w, x).view(torch.int16), want.view(torch.int16))
        assert torch.equal(backend.linear_m(w, x).view(torch.int16), dot.view(torch.int16))


#: Rows: (outputs, K), one for each kernel of gemv_w8a16_batch.hip (groups of four activation rows, row blocks a wavefront, segments a unit, sets of
#: wavefronts, windows, vectors carried to LDS) that the shapes at the test itself do not take.
_BATCH_KERNELS = {
    2: [(131, 2064), (131, 3088), (131, 4112), (131, 8208), (1027, 19984), (2051, 4112), (2051, 6160), (2051, 19984), (3075, 3088),
        (3075, 4112), (3075, 6160), (3075, 8208), (3075, 9232), (4099, 19472), (8195, 12288), (12001, 8720), (16387, 6160)],
    3: [(131, 3088), (2051, 8208), (2051, 16400), (3075, 11280), (6151, 16384), (12001, 8720)],
    4: [(131, 4112), (3075, 8208), (5121, 25600), (33001, 4096), (66001, 2048), (131075, 1024)],
    5: [(131, 16), (131, 1040), (131, 2064), (131, 3344), (131, 4112), (131, 6160), (1027, 2064), (1027, 3088), (1027, 4112),
        (1027, 6160), (2051, 6160), (2051, 9744), (3075, 16), (3075, 1040), (3075, 2064), (3075, 3088), (3075, 3344), (3075, 6160),
        (3075, 7184), (4099, 4112), (6151, 6160), (8195, 4112), (8195, 6160), (16387, 16), (16387, 2064), (16387, 3088)],
    6: [(2051, 4112), (2051, 8208)],
    8: [(131, 1040), (131, 2064), (3075, 2064), (3075, 4112), (8195, 5392)],
    9: [(131, 16), (131, 1040), (131, 3088), (131, 4112), (131, 4880), (1027, 1040), (2051, 2064), (2051, 4112), (3075, 3088),
        (4099, 1040), (4099, 2064), (4099, 3088), (4099, 4112), (6151, 3088), (9217, 16), (9217, 1040), (9217, 3088), (16385, 5136),
        (20001, 6160)],
    10: [(131, 3344)],
    12: [(131, 4112), (4099, 2064), (4099, 4112), (9217, 1552)],
    16: [(131, 528), (131, 1040), (701, 25600), (4099, 1552), (4099, 3088)],
}


@pytest.mark.parametrize("m,n,k", [(2, 1, 16), (3, 5, 1040), (4, 1023, 2560), (16, 1024, 2576), (4, 300, 9744), (8, 700, 9728),
                                   (7, 2047, 4096), (5, 2561, 4112), (2, 9000, 6416), (2, 1152, 16384), (2, 1153, 16384),
                                   (3, 200, 20496), (6, 500, 12304), (7, 2000, 33024), (4, 4096, 14336), (8, 3900, 9728), (6, 5000, 20496), (16, 300, 9728), (12, 5000, 6160), (9, 9300, 12304),
                                   (4, 5001, 2560), (8, 7000, 5136), (16, 8192, 1024), (2, 6000, 16), (13, 3333, 3072),
                                   (4, 32773, 4112), (5, 16385, 1040), (16, 9217, 2576), (15, 9301, 4096), (11, 4100, 5120),
                                   (3, 20000, 5136), (8, 8193, 6160), (16, 16400, 6160),
                                   (2, 8192, 1040), (2, 8193, 1040), (2, 16385, 1040), (2, 16385, 1152), (2, 16387, 2064), (2, 9001, 4096), (2, 8200, 1024),
                                   (2, 1025, 9744), (2, 1536, 12304), (2, 1537, 9744), (3, 1025, 1024), (4, 3072, 784)]
                         + [(m, n, k) for m, shapes in _BATCH_KERNELS.items() for n, k in shapes])
def test_batches_of_weight_only_rows_carry_the_single_row_bits(m, n, k):
    """Every kernel that 2..16 rows of cmi_gemv_w8a16 take, at odd counts of rows, outputs and chunks: few outputs by quarters of a row
    (units dealt to wavefronts, one block or two a wavefront), long rows in windows, many outputs streamed, sixteen rows in two halves
    (the second of one row, too), two rows that share a tree.
    Infinite and NaN activations stay in their rows; nothing is written past the outputs."""
    gen = torch.Generator(device=G.DEV).manual_seed(m + n + k)
    wq = torch.randint(-127, 128, (n, k), dtype=torch.int8, device=G.DEV, generator=gen)
    ws = torch.rand(n, device=G.DEV, generator=gen) * 0.01 + 1e-3
    x = torch.randn((m, k), device=G.DEV, generator=gen).to(torch.bfloat16)
    x[0, k - 1] = float("inf")
    x[m // 2, k // 2] = float("nan")
    lib = _native.load()
    y = torch.full((m * n + 64,), -77.0, dtype=torch.bfloat16, device=G.DEV)
    _native.check(lib.cmi_gemv_w8a16(G.ptr(wq), G.ptr(ws), G.ptr(x), G.ptr(y), m, n, k, G.stream()), "gemv")
    single = torch.cat([G.gemv_w8a16(wq, ws, x[r:r + 1].contiguous()) for r in range(m)])
    finite = [r for r in range(m) if r not in (0, m // 2)]
    got = y[:m * n].view(m, n)
    assert torch.equal(got[finite].view(torch.int16), single[finite].view(torch.int16)) and (y[m * n:] == -77.0).all()
    for kind in (torch.isposinf, torch.isneginf, torch.isnan):
        assert torch.equal(kind(got), kind(single)), kind
    if finite:
        xd, wd = x[finite[0]].double(), wq.double()
        exact = (wd @ xd) * ws.double()
        bound = exact.abs() * 2.0 ** -8 + (wd.abs() @ xd.abs()) * ws.double() * (k * 2.0 ** -24)
        assert ((got[finite[0]].double() - exact).abs() <= bound).all()


@pytest.mark.parametrize("n,k", [(20479, 1024), (20481, 1024), (131, 1040), (20301, 1040), (130001, 1040), (9103, 2304), (9041, 2320), (52429, 2560),
                                 (32769, 4096), (7, 16400), (1025, 20496)])
def test_one_weight_only_row_where_two_weight_rows_share_a_tree(n, k):
    """Both sides of the rules for one or two weight rows a wavefront and for a wavefront a whole row, odd outputs, several units: the bits of
    the batch kernels' rows, and the exact sum."""
    gen = torch.Generator(device=G.DEV).manual_seed(n + k)
    wq = torch.randint(-127, 128, (n, k), dtype=torch.int8, device=G.DEV, generator=gen)
    ws = torch.rand(n, device=G.DEV, generator=gen) * 0.01 + 1e-3
    x = torch.randn((1, k), device=G.DEV, generator=gen).to(torch.bfloat16)
    y = torch.full((n + 64,), -77.0, dtype=torch.bfloat16, device=G.DEV)
    _native.check(_native.load().cmi_gemv_w8a16(G.ptr(wq), G.ptr(ws), G.ptr(x), G.ptr(y), 1, n, k, G.stream()), "gemv")
    assert torch.equal(y[:n].view(torch.int16), G.gemv_w8a16(wq, ws, x.expand(4, k).contiguous())[3].view(torch.int16)) and (y[n:] == -77.0).all()
    xd, wd = x[0].double(), wq.double()
    exact = (wd @ xd) * ws.double()
    bound = exact.abs() * 2.0 ** -8 + (wd.abs() @ xd.abs()) * ws.double() * (k * 2.0 ** -24)
    assert ((y[:n].double() - exact).abs() <= bound).all()


@pytest.mark.parametrize("m,n,k", [(3, 655361, 256), (16, 145637, 1152), (9, 65543, 2560), (5, 62425, 2688), (4, 32768, 5120), (13, 33333, 5120)])
def test_rows_of_a_large_int4_weight_carry_the_small_weights_bits(m, n, k):
    """One line to the longest rows, odd counts of groups, rows and outputs, at the rule's edge: the bits of the kernels
    that the first and the last outputs take alone."""
    gen = torch.Generator(device=G.DEV).manual_seed(m + n + k)
    w4 = torch.randint(0, 256, (n, k // 2), dtype=torch.uint8, device=G.DEV, generator=gen)
    ws = torch.rand((n, k // 128), device=G.DEV, generator=gen) * 0.01 + 1e-3
    xq = torch.randint(-127, 128, (m, k), dtype=torch.int8, device=G.DEV, generator=gen)
    xs = torch.rand(m, device=G.DEV, generator=gen) + 0.1
    lib = _native.load()
    y = torch.full((m * n + 64,), -77.0, dtype=torch.bfloat16, device=G.DEV)
    _native.check(lib.cmi_gemv_w4a8(G.ptr(w4), G.ptr(ws), G.ptr(xq), G.ptr(xs), G.ptr(y), None, m, n, k, 128, G.stream()), "gemv_w4a8")
    got = y[:m * n].view(m, n)
    assert (y[m * n:] == -77.0).all()
    cut = n - 16 * 2048                                    # few enough outputs for the other kernels
    part = torch.empty((m, n - cut), dtype=torch.bfloat16, device=G.DEV)
    sums = torch.empty((m, k // 128, n - cut), dtype=torch.int32, device=G.DEV)
    _native.check(lib.cmi_gemv_w4a8(G.ptr(w4[cut:]), G.ptr(ws[cut:]), G.ptr(xq), G.ptr(xs), G.ptr(part), G.ptr(sums), m, n - cut, k, 128,
                                    G.stream()), "gemv_w4a8")
    assert torch.equal(got[:, cut:].contiguous().view(torch.int16), part.view(torch.int16))
    head = torch.empty((m, 4096), dtype=torch.bfloat16, device=G.DEV)
    _native.check(lib.cmi_gemv_w4a8(G.ptr(w4), G.ptr(ws), G.ptr(xq), G.ptr(xs), G.ptr(head), None, m, 4096, k, 128, G.stream()), "gemv_w4a8")
    assert torch.equal(got[:, :4096].contiguous().view(torch.int16), head.view(torch.int16))
