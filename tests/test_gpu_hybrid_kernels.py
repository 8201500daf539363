"""Kernels of the hybrid library one by one against plain PyTorch on the CPU."""
import ctypes

import pytest
import torch

from metaseq_amd import _capi
from metaseq_amd._capi import check, ptr
from metaseq_amd.hybrid_decoder import pack_tiles
from oracle import hybrid_oracle as O

pytestmark = pytest.mark.gpu
BF16, F32 = torch.bfloat16, torch.float32


def gen(seed):
    return torch.Generator().manual_seed(seed)


def pack_rows(x):
    """[M, K] bf16 -> the packed activation layout of at most 128 rows."""
    M, K = x.shape
    MB = (M + 15) // 16 if M <= 64 else 8
    full = torch.zeros(MB * 16, K, dtype=x.dtype)
    full[:M] = x
    return full.view(MB, 16, K // 32, 4, 8).permute(2, 0, 3, 1, 4).contiguous()


def unpack_rows(p, M, K):
    MB = (M + 15) // 16 if M <= 64 else 8
    return p.view(K // 32, MB, 4, 16, 8).permute(1, 3, 0, 2, 4).reshape(MB * 16, K)[:M]


def close(got, want, tol, what):
    err = float((got.double().cpu() - want.double()).abs().max() / want.double().abs().max())
    print(what, "%.2e" % err, flush=True)
    assert err <= tol, (what, err)


def glu(kind, g, u, limit):
    if kind == _capi.MSA_GLU_GELU:
        return O.gelu_tanh(g) * u
    g, u = g.clamp(max=limit), u.clamp(-limit, limit)
    return g * torch.sigmoid(1.702 * g) * (u + 1)


# rows x features x reduction: every kernel of the bf16 products (packed streaming up to 128 rows,
# 128 x 128 tiles, four-wave tiles of three widths, ragged bottoms)
SHAPES = [(1, 64, 128), (5, 208, 192), (17, 96, 256), (33, 4096, 512), (64, 272, 128),
          (100, 1040, 320), (128, 512, 1024), (129, 48, 128), (200, 272, 192), (300, 1600, 256),
          (700, 4112, 256), (1024, 8192, 128), (1100, 16384, 192)]


@pytest.mark.parametrize("M,N,K", SHAPES)
def test_linear_bf16(M, N, K):
    lib = _capi.load_hybrid()
    print("linear_bf16", M, N, K, flush=True)
    g = gen(M + N)
    x = torch.randn(M, K, generator=g).to(BF16)
    w = (torch.randn(N, K, generator=g) * K ** -0.5).to(BF16)
    ref = x.double() @ w.double().T
    wp = pack_tiles(w).cuda()
    packed = M <= 128
    xd = (pack_rows(x) if packed else x).cuda()
    flags = _capi.MSA_IN_PACKED if packed else 0
    for n32 in sorted({N, N - 16, N // 2 // 16 * 16, 0}):
        y = torch.zeros(M, n32, dtype=BF16, device="cuda")
        y32 = torch.zeros(M, N - n32, dtype=F32, device="cuda")
        check(lib.msa_linear_bf16(ptr(xd), ptr(wp), ptr(y), ptr(y32), M, N, K, n32, -1, 0.0, flags,
                                  _capi.stream_ptr()), lib)
        if n32:
            close(y, ref[:, :n32], 6e-3, "bf16 columns of n32=%d" % n32)
        if n32 < N:
            close(y32, ref[:, n32:], 1e-5, "fp32 columns of n32=%d" % n32)
    for kind, n32 in ((_capi.MSA_GLU_GELU, N // 32 * 32), (_capi.MSA_GLU_CLAMPED, N // 64 * 32)):
        if n32 == 0:
            continue
        out_packed = packed and (n32 // 2) % 32 == 0
        MB = (M + 15) // 16 if M <= 64 else 8
        y = torch.zeros((MB * 16 if out_packed else M) * (n32 // 2), dtype=BF16, device="cuda")
        y32 = torch.zeros(M, N - n32, dtype=F32, device="cuda")
        check(lib.msa_linear_bf16(ptr(xd), ptr(wp), ptr(y), ptr(y32), M, N, K, n32, kind, 0.7,
                                  flags | (_capi.MSA_OUT_PACKED if out_packed else 0),
                                  _capi.stream_ptr()), lib)
        got = unpack_rows(y.cpu(), M, n32 // 2) if out_packed else y.view(M, n32 // 2)
        close(got, glu(kind, ref[:, 0:n32:2], ref[:, 1:n32:2], 0.7), 6e-3, "glu %d" % kind)
        if n32 < N:
            close(y32, ref[:, n32:], 1e-5, "fp32 columns beside glu")
    for S in {1, lib.msa_linear_bf16_splits(M, N, K, int(packed))}:
        part = torch.zeros(S, M, N, dtype=F32, device="cuda")
        check(lib.msa_linear_partial_bf16(ptr(xd), ptr(wp), ptr(part), M, N, K, S, flags,
                                          _capi.stream_ptr()), lib)
        close(part.sum(0), ref, 1e-5, "partial sums, S=%d" % S)


@pytest.mark.parametrize("M,N,K", [
    # a wave per tile: vocabularies (13 and 14 tiles per workgroup) from one row on
    (1, 50272, 160), (17, 54000, 96), (33, 54000, 160), (64, 50272, 96), (65, 54000, 96), (128, 50272, 160),
    # (queues: one to three tiles of 33 to 64 rows, four of more; the last workgroup's tiles run out)
    (40, 3088, 160), (50, 8176, 96), (64, 12272, 224), (33, 12288, 96), (100, 16368, 160)])
def test_linear_bf16_of_a_wave_per_tile(M, N, K):
    test_linear_bf16(M, N, K)


# packed rows and 129 .. 256 row-major ones in queues: tiles to a workgroup and row blocks of either
@pytest.mark.parametrize("M,N,K", [(40, 16400, 320), (64, 28688, 192), (90, 24592, 576), (128, 20496, 320), (20, 32784, 192),
                                   (140, 6160, 576), (190, 10256, 320), (256, 8208, 1088)])
def test_linear_bf16_in_queues(M, N, K):
    test_linear_bf16(M, N, K)


# more tiles to a workgroup than queues take: the shared-activation kernel in one pass, K that ends inside a stage
@pytest.mark.parametrize("M,N,K", [(40, 49136, 192), (64, 40976, 320), (128, 36864, 320), (97, 40976, 192)])
def test_linear_bf16_beyond_queues(M, N, K):
    test_linear_bf16(M, N, K)


@pytest.mark.parametrize("M,K,most", [(1, 768, 1.0e-7), (33, 4096, 1.8e-7), (64, 9216, 2.5e-7), (100, 4096, 3.3e-7)])
def test_fp32_logits_of_a_vocabulary_are_no_single_chain_over_k(M, K, most):
    """The error of fp32 sums grows with the root of the additions behind each: K / 128 stages of four steps up to 64 rows,
    K / 64 steps beyond.  One chain of K / 32 steps has 1.6, 3.9, 6.1 and 3.9e-7 here."""
    lib, N = _capi.load_hybrid(), 50272
    g = torch.Generator("cuda").manual_seed(K)
    x = torch.randn(M, K, generator=g, device="cuda").to(BF16)
    w = (torch.randn(N, K, generator=g, device="cuda") * K ** -0.5).to(BF16)
    y = torch.empty(M, N, device="cuda")
    check(lib.msa_linear_partial_bf16(ptr(pack_rows(x.cpu()).cuda()), ptr(pack_tiles(w)), ptr(y), M, N, K, 1,
                                      _capi.MSA_IN_PACKED, _capi.stream_ptr()), lib)
    want = x.double() @ w.double().t()
    assert float((y.double() - want).norm() / want.norm()) <= most


@pytest.mark.parametrize("M,N,K,most", [(24, 5120, 20480, 1.26e-7), (32, 9216, 9216, 1.16e-7), (32, 2560, 10240, 1.06e-7)])
def test_fp32_sums_of_few_rows_are_no_longer_chains(M, N, K, most):
    """In the number of slices that is suggested; `most`: what the stream kernel's sums have (in twice the slices, or as many)."""
    lib = _capi.load_hybrid()
    g = torch.Generator("cuda").manual_seed(M + N)
    x = torch.randn(M, K, generator=g, device="cuda").to(BF16)
    w = (torch.randn(N, K, generator=g, device="cuda") * K ** -0.5).to(BF16)
    S = lib.msa_linear_bf16_splits(M, N, K, 1)
    part = torch.full((S, M, N), float("nan"), device="cuda")
    check(lib.msa_linear_partial_bf16(ptr(pack_rows(x.cpu()).cuda()), ptr(pack_tiles(w)), ptr(part), M, N, K, S,
                                      _capi.MSA_IN_PACKED, _capi.stream_ptr()), lib)
    got = part[0].clone()
    for s in range(1, S):
        got += part[s]
    want = x.double() @ w.double().t()
    assert float((got.double() - want).norm() / want.norm()) <= most


@pytest.mark.parametrize("M,N", [(4352, 16656), (600, 24576)])
def test_linear_partial_bf16_wide_panels(M, N):
    """More than 64 columns of tiles, taken in panels of 16; sums of one and two slices."""
    lib, K = _capi.load_hybrid(), 256
    g = torch.Generator("cuda").manual_seed(M)
    x = torch.randn(M, K, generator=g, device="cuda").to(BF16)
    w = (torch.randn(N, K, generator=g, device="cuda") * K ** -0.5).to(BF16)
    wp, ref = pack_tiles(w), x.float() @ w.float().t()
    for S in (1, 2):
        part = torch.full((S, M, N), float("nan"), device="cuda")
        check(lib.msa_linear_partial_bf16(ptr(x), ptr(wp), ptr(part), M, N, K, S, 0, _capi.stream_ptr()), lib)
        close(part.sum(0).cpu(), ref.cpu(), 1e-5, "partial sums, S=%d" % S)


@pytest.mark.parametrize("M,N,K", [(700, 4096, 2048), (2048, 4096, 8192), (1500, 4096, 16384)])
def test_linear_partial_bf16_in_two_slices(M, N, K):
    """Prompts whose tiles fill half of the chip or less: two slices are suggested, and sum to the product."""
    lib = _capi.load_hybrid()
    g = torch.Generator("cuda").manual_seed(M)
    x = torch.randn(M, K, generator=g, device="cuda").to(BF16)
    w = (torch.randn(N, K, generator=g, device="cuda") * K ** -0.5).to(BF16)
    assert lib.msa_linear_bf16_splits(M, N, K, 0) == 2 and lib.msa_linear_bf16_splits(M, N, K - 64, 0) == 1
    part = torch.full((2, M, N), float("nan"), device="cuda")
    check(lib.msa_linear_partial_bf16(ptr(x), ptr(pack_tiles(w)), ptr(part), M, N, K, 2, 0, _capi.stream_ptr()), lib)
    close(part.sum(0).cpu(), (x.float() @ w.float().t()).cpu(), 1e-5, "two slices")


@pytest.mark.parametrize("M,N", [(1500, 6032), (1500, 6912), (2305, 7168), (3000, 7680)])
def test_linear_bf16_pieces(M, N, K=256):
    """More than a round of tiles: sums of one and two slices, a gated activation with fp32 columns behind it."""
    lib = _capi.load_hybrid()
    print("rows", M, N, K, flush=True)
    g = torch.Generator("cuda").manual_seed(M)
    x = torch.randn(M, K, generator=g, device="cuda").to(BF16)
    w = (torch.randn(N, K, generator=g, device="cuda") * K ** -0.5).to(BF16)
    wp, ref = pack_tiles(w), (x.float() @ w.float().t()).cpu()
    for S in (1, 2):
        part = torch.full((S, M, N), float("nan"), device="cuda")
        check(lib.msa_linear_partial_bf16(ptr(x), ptr(wp), ptr(part), M, N, K, S, 0, _capi.stream_ptr()), lib)
        close(part.sum(0).cpu(), ref, 1e-5, "partial sums, S=%d" % S)
    n32 = N // 2 // 32 * 32
    y = torch.zeros(M, n32 // 2, dtype=BF16, device="cuda")
    y32 = torch.zeros(M, N - n32, device="cuda")
    check(lib.msa_linear_bf16(ptr(x), ptr(wp), ptr(y), ptr(y32), M, N, K, n32, _capi.MSA_GLU_CLAMPED, 0.7, 0,
                              _capi.stream_ptr()), lib)
    close(y.cpu(), glu(_capi.MSA_GLU_CLAMPED, ref[:, 0:n32:2], ref[:, 1:n32:2], 0.7), 6e-3, "glu")
    close(y32.cpu(), ref[:, n32:], 1e-5, "fp32 columns beside glu")


# the pieces that the last tiles are cut into as a whole product, as sums of one slice and of two (of eleven stages and more)
BF16_PIECES = [(3000, 5632, (4, 4, 4)), (2817, 6400, (4, 4, 1)), (3000, 7488, (2, 2, 1)), (3000, 6304, (4, 4, 2)),
               (1500, 6912, (1, 1, 2))]


@pytest.mark.parametrize("M,N,pieces", BF16_PIECES)
def test_linear_bf16_pieces_of_the_last_round(M, N, pieces):
    test_linear_bf16_pieces(M, N, 1408)


# (columns and rows of the taller tiles of the whole product)
BF16_EVEN = [(481, 8224, 128, 192), (577, 8224, 128, 224), (385, 8224, 128, 160), (898, 8224, 256, 160), (1345, 8224, 256, 224),
             (2465, 8224, 256, 192)]


@pytest.mark.parametrize("M,N,columns,rows", BF16_EVEN)
def test_linear_bf16_rows_cut_evenly_over_more_stages(M, N, columns, rows):
    test_linear_bf16_pieces(M, N, 1408)


@pytest.mark.parametrize("M,N", [(289, 6144), (387, 6144), (481, 8224), (577, 8224), (898, 8224), (1345, 8224), (2465, 8224)])
def test_linear_bf16_rows_cut_evenly(M, N):
    """Rows of tiles of 128 .. 256 rows in one launch, 128 and 256 columns wide, the last of them ragged."""
    test_linear_bf16_pieces(M, N)


@pytest.mark.parametrize("M,N,K", [(1, 16, 32), (70, 80, 96), (200, 144, 128)])
def test_linear_f32(M, N, K):
    lib = _capi.load_hybrid()
    g = gen(M)
    x, w = torch.randn(M, K, generator=g), torch.randn(N, K, generator=g) * K ** -0.5
    ref = x.double() @ w.double().T
    n32 = N // 32 * 32
    if n32 == N:
        n32 -= 32
    xd, wd = x.cuda(), w.cuda()
    for kind in (-1, 0, 1):
        cols = n32 if kind < 0 else n32 // 2
        y = torch.zeros(M, cols, device="cuda")
        y32 = torch.zeros(M, N - n32, device="cuda")
        check(lib.msa_linear_f32(ptr(xd), ptr(wd), ptr(y), ptr(y32), M, N, K, n32, kind, 0.6,
                                 _capi.stream_ptr()), lib)
        if cols:
            want = ref[:, :n32] if kind < 0 else glu(kind, ref[:, 0:n32:2], ref[:, 1:n32:2], 0.6)
            close(y, want, 2e-6, "glu %d" % kind)
        close(y32, ref[:, n32:], 2e-6, "tail")


# one fp32 kernel serves every shape: the smaller ones do
@pytest.mark.parametrize("M,N,K,dtype", [s + (BF16,) for s in SHAPES] + [
    s + (F32,) for s in SHAPES if s[0] * s[1] <= 1 << 21] + [
    # in queues of two to nine tiles to a workgroup (256 compute units), packed and, from 129 rows on, row-major
    s + (BF16,) for s in ((33, 4112, 128), (40, 8208, 192), (64, 20496, 192), (90, 32784, 128), (128, 24592, 192), (20, 20496, 320),
                          (200, 2064, 576), (140, 4112, 192), (256, 8208, 320))])
def test_linear_with_bias_activation_and_decays(M, N, K, dtype):
    """Every kernel behind msa_linear: a bias, relu^2, a second output, fp32 columns as they are and
    as decays (logits far out on both sides among them)."""
    lib = _capi.load_hybrid()
    print("linear", M, N, K, dtype, flush=True)
    g = gen(M + N + K)
    x = torch.randn(M, K, generator=g).to(dtype)
    w = (torch.randn(N, K, generator=g) * K ** -0.5).to(dtype)
    bias = torch.randn(N, generator=g)
    bias[-8:-4], bias[-4:] = -16.0, 30.0
    ref = x.double() @ w.double().T + bias.double()
    packed = M <= 128 and dtype == BF16
    xd = (pack_rows(x) if packed else x).cuda()
    wd = (pack_tiles(w) if dtype == BF16 else w).cuda()
    bd = bias.cuda()
    MB = (M + 15) // 16 if M <= 64 else 8
    tol = 6e-3 if dtype == BF16 else 2e-6
    for n2, n32, act, decays in ((N, N, 1, 0), (N // 64 * 32, N // 32 * 32, 0, 0),
                                 (0, N // 32 * 32 - 32, 0, 1), (16, N - 16, 1, 1), (N - 16, N - 16, 0, 1),
                                 (0, 0, 0, 1)):
        rate = torch.rand(N - n32, generator=g) * 3
        rd = rate.cuda()
        out2_packed = packed and (n32 - n2) % 32 == 0
        y = torch.zeros(M, n2, dtype=dtype, device="cuda")
        y2 = torch.zeros((MB * 16 if out2_packed else M) * (n32 - n2), dtype=dtype, device="cuda")
        y32 = torch.zeros(M, N - n32, device="cuda")
        a = _capi.LinearArgs()
        a.dtype, a.x, a.W, a.M, a.N, a.K = int(dtype == F32), ptr(xd), ptr(wd), M, N, K
        a.n32, a.n2, a.act, a.bias = n32, n2, act, ptr(bd)
        a.decay_rate = ptr(rd) if decays and n32 < N else None
        a.flags = (_capi.MSA_IN_PACKED if packed else 0) | (_capi.MSA_OUT2_PACKED if out2_packed else 0)
        a.y, a.y32 = ptr(y) if n2 else None, ptr(y32) if n32 < N else None
        if n2 < n32:
            a.y2 = ptr(y2)
        check(lib.msa_linear(ctypes.byref(a), _capi.stream_ptr()), lib)
        want = torch.relu(ref) ** 2 if act else ref
        what = "n2=%d n32=%d act=%d" % (n2, n32, act)
        if n2:
            close(y, want[:, :n2], tol, what)
        if n2 < n32:
            got = unpack_rows(y2.cpu(), M, n32 - n2) if out2_packed else y2.view(M, n32 - n2)
            close(got, want[:, n2:n32], tol, "second output, " + what)
        if n32 < N:
            z = ref[:, n32:]
            if decays:
                z = torch.exp(-rate.double() * torch.nn.functional.softplus(z))
            close(y32, z, 1e-5 if dtype == BF16 else 3e-6, "fp32 columns, " + what)
            if decays:   # next to 1 the distance from 1 counts
                slow = z > 0.999
                off = ((1 - y32.cpu().double()) - (1 - z)).abs()[slow]
                assert off.numel() == 0 or float(off.max()) < 3e-7, what


@pytest.mark.parametrize("M,N,K", [(385, 8208, 256), (577, 8208, 256), (1345, 8208, 128)])
def test_linear_with_bias_rows_cut_evenly(M, N, K):
    test_linear_with_bias_activation_and_decays(M, N, K, BF16)


@pytest.mark.parametrize("M,N,K", [(385, 8208, 704), (577, 8208, 704), (1345, 8208, 704)])
def test_linear_with_bias_rows_cut_evenly_over_more_stages(M, N, K):
    test_linear_with_bias_activation_and_decays(M, N, K, BF16)

@pytest.mark.parametrize("dtype", [BF16, F32], ids=["bf16", "f32"])
@pytest.mark.parametrize("M,D", [(1, 72), (5, 4096), (40, 1000), (130, 2100), (1100, 300),
                                 (1030, 5000), (3, 9000)])
def test_tail_of_two_sides_with_loop_terms(M, D, dtype):
    """Both sides' sums and norms, a bias, what a loop adds, the probe and the next norm."""
    lib = _capi.load_hybrid()
    g = gen(M + D)
    Dp, eps = (D + 63) // 64 * 64, 1e-3

    def wide(*shape):
        t = torch.zeros(*shape, Dp)
        t[..., :D] = torch.randn(*shape, D, generator=g)
        return t
    for S, S2, two, extra in ((1, 1, True, True), (3, 5, True, False), (2, 0, False, True)):
        x, part, part2 = wide(M), wide(S, M), wide(max(1, S2), M)
        bias, w, w2, add, step, nxt = wide(), wide(), wide(), wide(M), wide(), wide()
        b = part.double().sum(0) + (bias.double() if extra else 0)
        want = x.double()
        want = want + (O.rms(b[:, :D], eps, w[:D].double()) if two else b[:, :D]) \
            if Dp == D else want.clone()
        if Dp != D:
            want[:, :D] += O.rms(b[:, :D], eps, w[:D].double()) if two else b[:, :D]
        if two:
            want[:, :D] += O.rms(part2.double().sum(0)[:, :D], eps, w2[:D].double())
        probe = want.clone()
        if extra:
            want = want + add.double() + step.double()
        h = O.rms(want[:, :D], eps, nxt[:D].double())
        dev = [t.cuda() for t in (x, part, part2, bias, w, w2, add, step, nxt)]
        hd = torch.zeros(M, Dp, dtype=dtype, device="cuda")
        pd = torch.zeros(M, Dp, device="cuda")
        a = _capi.TailArgs()
        a.dtype, a.M, a.D, a.Dp, a.S, a.eps = int(dtype == F32), M, D, Dp, S, eps
        a.x, a.part, a.h, a.w_next, a.probe = ptr(dev[0]), ptr(dev[1]), ptr(hd), ptr(dev[8]), ptr(pd)
        if two:
            a.part2, a.S2, a.w_post, a.w_post2 = ptr(dev[2]), S2, ptr(dev[4]), ptr(dev[5])
        if extra:
            a.bias, a.add, a.step = ptr(dev[3]), ptr(dev[6]), ptr(dev[7])
        check(lib.msa_residual_rmsnorm_tail(ctypes.byref(a), _capi.stream_ptr()), lib)
        close(dev[0], want, 2e-6, "stream")
        close(pd, probe, 2e-6, "probe")
        close(hd[:, :D], h, 6e-3 if dtype == BF16 else 3e-6, "normed")


@pytest.mark.parametrize("dtype", [BF16, F32], ids=["bf16", "f32"])
@pytest.mark.parametrize("M,heads,vdim,off", [(1, 1, 5, 0), (17, 3, 40, 0), (5, 7, 64, 0), (33, 5, 100, 0),
                                              (40, 9, 128, 0), (3, 2, 200, 0), (9, 3, 256, 0), (5, 3, 300, 0),
                                              (2, 1, 512, 0), (17, 3, 40, 1), (6, 2, 300, 2)])
def test_delta_output(M, heads, vdim, off, dtype):
    """Norm and gate of every head's outputs, row-major and packed; gates that lie `off` elements off alignment."""
    lib = _capi.load_hybrid()
    g = gen(M + vdim)
    vp, eps = (vdim + 15) // 16 * 16, 1e-4
    o, w = torch.zeros(M, heads, vp), torch.zeros(vp)
    o[..., :vdim], w[:vdim] = torch.randn(M, heads, vdim, generator=g), torch.randn(vdim, generator=g)
    z = torch.randn(M, heads * vp + 8, generator=g).to(dtype)
    gate = z[:, off:off + heads * vp].double().view(M, heads, vp)
    od, wd, zd = o.cuda(), w.cuda(), z.cuda()
    for act, packed in ((0, False), (1, False), (0, True)):
        if packed and (dtype == F32 or heads * vp % 32 or M > 128):
            continue
        want = o.double() * torch.rsqrt((o.double() ** 2).sum(-1, keepdim=True) / vdim + eps) * w.double()
        want = (want * (torch.sigmoid(gate) if act else torch.nn.functional.silu(gate))).view(M, -1)
        mb = (M + 15) // 16 if packed else 0
        out = torch.full((mb * 16 if packed else M, heads * vp), 7.0, dtype=dtype, device="cuda")
        a = _capi.DeltaArgs()
        a.dtype, a.heads, a.vdim, a.vp, a.eps, a.gate_act = int(dtype == F32), heads, vdim, vp, eps, act
        a.o, a.w, a.gate, a.ld_gate = ptr(od), ptr(wd), ptr(zd[:, off:]), z.shape[1]
        a.out, a.ld_out, a.out_mb = ptr(out), heads * vp, mb
        check(lib.msa_delta_output(ctypes.byref(a), M, _capi.stream_ptr()), lib)
        got = unpack_rows(out.view(-1).cpu(), M, heads * vp) if packed else out
        close(got, want, 6e-3 if dtype == BF16 else 3e-6, "act %d packed %d" % (act, packed))


@pytest.mark.parametrize("D", [3000, 4096, 4104])
def test_tail_of_many_wide_rows(D):
    test_tail_of_two_sides_with_loop_terms(1030, D, BF16)


@pytest.mark.parametrize("M,D,top", [(1025, 4000, 3), (1025, 4096, 8), (1030, 8000, 5), (7, 4096, 5)])
def test_tail_of_routed_terms(M, D, top):
    """A gated sum and the routed terms, wherever their rows lie."""
    lib = _capi.load_hybrid()
    g = gen(M + top)
    Dp, eps = (D + 63) // 64 * 64, 1e-5
    x, part, pairs = (torch.zeros(n, Dp) for n in (M, M, M * top))
    for t in (x, part, pairs):
        t[:, :D] = torch.randn(len(t), D, generator=g)
    pairs = pairs.to(BF16)
    weight, gate = torch.rand(M, top, generator=g), torch.rand(M, generator=g)
    inverse = torch.randperm(M * top, generator=g).view(M, top)
    want = x.double() + part.double() * gate.double().view(M, 1)
    for k in range(top):
        want += weight[:, k:k + 1].double() * pairs[inverse[:, k]].double()
    dev = [t.cuda() for t in (x, part, pairs, weight, gate, inverse.int())]
    a = _capi.TailArgs()
    a.dtype, a.M, a.D, a.Dp, a.S, a.eps = 0, M, D, Dp, 1, eps
    a.x, a.part, a.pair_y, a.pair_w, a.gate, a.inverse = (ptr(t) for t in dev)
    a.top = top
    check(lib.msa_residual_rmsnorm_tail(ctypes.byref(a), _capi.stream_ptr()), lib)
    close(dev[0], want, 2e-6, "stream")


def _grouped(lib, dtype, heads, kv_heads, hd, vd, chunk, rot, segments, capacity, seed, fused=None):
    """One step of grouped attention over ``segments`` ((slot, first position, tokens)) through the
    three calls; returns its outputs and the caches with what they should be."""
    g = gen(seed)
    M = sum(n for _, _, n in segments)
    slots = 1 + max(s for s, _, _ in segments)
    rows = min(capacity, chunk) if chunk else capacity
    ld = (heads + kv_heads) * hd + kv_heads * vd + 16
    x = torch.randn(M, ld, generator=g).to(dtype)
    kc = torch.randn(slots, kv_heads, rows, hd, generator=g).to(dtype)
    vc = torch.randn(slots, kv_heads, rows, vd, generator=g).to(dtype)
    gate = torch.randn(M, heads + 3, generator=g)
    inv = 100.0 ** (-2.0 * torch.arange(rot // 2, dtype=torch.float64) / max(1, rot))
    scale = 1.5 * hd ** -0.5
    want, kw, vw = torch.zeros(M, heads, vd, dtype=torch.float64), kc.clone(), vc.clone()
    at = 0
    for slot, pos, n in segments:
        if pos >= 0:
            own = x[at:at + n].double()
            q = own[:, :heads * hd].view(n, heads, hd)
            k = own[:, heads * hd:(heads + kv_heads) * hd].view(n, kv_heads, hd)
            v = own[:, (heads + kv_heads) * hd:-16].view(n, kv_heads, vd)
            p = torch.arange(pos, pos + n)
            if rot:
                q, k = (O.rotate_half(t, p, 100.0, rot).to(dtype).double() for t in (q, k))
            c0 = pos // chunk * chunk if chunk else 0
            keys = torch.cat([kc[slot, :, :pos - c0].double().transpose(0, 1), k])
            vals = torch.cat([vc[slot, :, :pos - c0].double().transpose(0, 1), v])
            where = torch.arange(c0, pos + n)
            for h in range(heads):
                j = h // (heads // kv_heads)
                s = q[:, h] @ keys[:, j].T * scale
                first = p // chunk * chunk if chunk else torch.zeros_like(p)
                sees = (where <= p[:, None]) & (where >= first[:, None])
                s = s.masked_fill(~sees, float("-inf"))
                want[at:at + n, h] = torch.softmax(s, -1) @ vals[:, j] * torch.sigmoid(
                    gate[at:at + n, h:h + 1].double())
            last = (pos + n - 1) // chunk * chunk if chunk else 0
            for i in range(max(0, last - pos), n):
                kw[slot, :, pos + i - last] = k[i].to(dtype)
                vw[slot, :, pos + i - last] = v[i].to(dtype)
        at += n
    b, alive = _batch(segments, M)
    b.key_bound = max(max(p + n for _, p, n in segments), 1)
    xd, kd, vd_, gd, fd = x.cuda(), kc.cuda(), vc.cuda(), gate.cuda(), inv.cuda()
    out = torch.full((M, heads * vd), 7.0, dtype=dtype, device="cuda")
    a = _capi.GroupedArgs()
    a.dtype, a.heads, a.kv_heads, a.hd, a.vd = int(dtype == F32), heads, kv_heads, hd, vd
    a.chunk, a.rot_dims, a.rows, a.scale = chunk, rot, rows, scale
    a.inv_freq = ptr(fd) if rot else None
    es = x.element_size()
    a.q, a.k = xd.data_ptr(), xd.data_ptr() + heads * hd * es
    a.v, a.ld = a.k + kv_heads * hd * es, ld
    a.k_cache, a.v_cache, a.gate, a.ld_gate = ptr(kd), ptr(vd_), ptr(gd), heads + 3
    a.out, a.ldo = ptr(out), heads * vd
    a.fused = lib.msa_grouped_fuses(ctypes.byref(a), ctypes.byref(b)) if fused is None else fused
    part = torch.zeros(M * heads * 64 * (vd + 4), device="cuda")
    a.partial, s = ptr(part), _capi.stream_ptr()
    ref = (ctypes.byref(a), ctypes.byref(b))
    if not a.fused:
        check(lib.msa_grouped_rotate(*ref, s), lib)
    seg = 0
    counts = [n for _, _, n in segments]
    while seg < len(counts):
        end = seg + 1
        while end < len(counts) and (counts[end] == 1) == (counts[seg] == 1):
            end += 1
        a.splits = 1
        if counts[seg] == 1:
            a.splits = lib.msa_grouped_attention_splits(ctypes.byref(a), end - seg, b.key_bound)
        check(lib.msa_grouped_attention(*ref, seg, end, max(counts[seg:end]), s), lib)
        seg = end
    if not a.fused:
        check(lib.msa_grouped_append(*ref, s), lib)
    tol = 2e-5 if dtype == F32 else 1.5e-2
    on = torch.cat([torch.full((n,), p >= 0) for _, p, n in segments])
    close(out.view(M, heads, vd)[on.cuda()], want[on], tol, "outputs, splits=%d" % a.splits)
    # rotated keys in another order of operations: the last bit may differ
    close(kd, kw, 1e-6 if dtype == F32 else 8e-3, "keys kept")
    assert torch.equal(vd_.cpu(), vw), "values kept"


GROUPED = [(4, 2, 64, 64, 40), (8, 8, 128, 128, 128), (34, 2, 64, 128, 10), (3, 1, 192, 64, 0),
           (4, 1, 256, 256, 64), (2, 2, 128, 192, 126), (5, 5, 192, 256, 34), (16, 8, 256, 64, 2),
           (17, 1, 64, 192, 64), (3, 3, 80, 272, 16), (8, 8, 64, 256, 62), (2, 1, 128, 64, 0)]


@pytest.mark.parametrize("dtype", [BF16, F32], ids=["bf16", "f32"])
@pytest.mark.parametrize("heads,kv_heads,hd,vd,rot", GROUPED)
def test_grouped_attention(heads, kv_heads, hd, vd, rot, dtype):
    """Decode steps (fused and not, with and without splits), portions over several chunks, mixed
    batches with inactive segments, with and without chunks."""
    lib = _capi.load_hybrid()
    size = (heads, kv_heads, hd, vd)
    print("grouped", size, rot, flush=True)
    decode = [(2, 700, 1), (0, 0, 1), (1, -1, 1), (4, 255, 1), (3, 129, 1), (5, 511, 1)]
    mix = [(1, 250, 1), (0, 90, 70), (2, 5, 1), (3, -1, 1), (4, 0, 150), (5, 127, 2), (6, -1, 3),
           (7, 64, 64)]
    for chunk in (0, 100, 128, 1000):
        _grouped(lib, dtype, *size, chunk, rot, decode, 800, heads)
        _grouped(lib, dtype, *size, chunk, rot, decode, 800, heads, fused=0)
        _grouped(lib, dtype, *size, chunk, rot, mix, 300, heads + 1)
    _grouped(lib, dtype, *size, 7, rot, [(0, 3, 40), (1, 6, 1), (2, 0, 7), (3, 13, 2)], 300, hd)
    _grouped(lib, dtype, *size, 0, rot, [(0, 1500, 1)], 1600, hd)          # splits


@pytest.mark.parametrize("dtype", [BF16, F32], ids=["bf16", "f32"])
@pytest.mark.parametrize("M", [1, 16, 20, 64, 150])
def test_group_linear_dense(M, dtype):
    """Per-group columns (a head, a diagonal block), also with the groups' inputs shared."""
    lib = _capi.load_hybrid()
    for G, N, K, share in ((3, 48, 64, 0), (6, 160, 32, 3), (1, 272, 128, 0)):
        g = gen(M + G)
        xg = share or G
        x = torch.randn(M, xg * K, generator=g).to(dtype)
        w = (torch.randn(G, N, K, generator=g) * K ** -0.5).to(dtype)
        ref = torch.stack([x[:, (i % xg) * K:(i % xg + 1) * K].double() @ w[i].double().T
                           for i in range(G)], dim=1).view(M, G * N)
        wd = (pack_tiles(w.view(G * N, K)) if dtype == BF16 else w.view(G * N, K)).cuda()
        xd = x.cuda()
        for y_f32 in (0, 1):
            y = torch.zeros(M, G * N, dtype=F32 if y_f32 else dtype, device="cuda")
            a = _capi.GroupLinearArgs()
            a.dtype, a.glu = (0 if dtype == BF16 else 1), -1
            a.x, a.ldx, a.x_group, a.x_groups = ptr(xd), xg * K, K, share
            a.W, a.y, a.ldy, a.y_group, a.y_f32 = ptr(wd), ptr(y), G * N, N, y_f32
            a.N, a.K, a.groups, a.M = N, K, G, M
            check(lib.msa_group_linear(ctypes.byref(a), _capi.stream_ptr()), lib)
            tol = 2e-6 if dtype == F32 else (1e-5 if y_f32 else 6e-3)
            close(y, ref, tol, "groups %s" % ((G, N, K, share),))


# tiles of 256 rows and a last one of 128, 192 or 256: groups of no row, of one, at each edge and past a whole tile
@pytest.mark.parametrize("N,K", [(544, 704), (256, 128), (1056, 192)])
@pytest.mark.parametrize("kind", [-1, _capi.MSA_GLU_GELU, _capi.MSA_GLU_CLAMPED])
def test_group_linear_routed_tiles_as_high_as_the_rows(N, K, kind):
    lib = _capi.load_hybrid()
    print("routed", N, K, kind, flush=True)
    g, top = gen(N + kind), 2
    counts = [1, 128, 129, 0, 192, 193, 256, 257, 384, 385, 448, 449, 300, 100]
    E, P = len(counts), sum(counts)
    flat = torch.repeat_interleave(torch.arange(E), torch.tensor(counts))[torch.randperm(P, generator=g)]
    x = torch.randn((P + top - 1) // top, K, generator=g).to(BF16)
    w = (torch.randn(E, N, K, generator=g) * K ** -0.5).to(BF16)
    n_max = P // 256 + E
    ids = flat.int().cuda()
    perm, inv = (torch.full((P,), -1, dtype=torch.int32, device="cuda") for _ in range(2))
    end, n = torch.zeros(E, dtype=torch.int32, device="cuda"), torch.zeros(1, dtype=torch.int32, device="cuda")
    tg, tr = (torch.full((n_max,), -1, dtype=torch.int32, device="cuda") for _ in range(2))
    check(lib.msa_moe_plan(ptr(ids), P, E, 256, ptr(perm), ptr(inv), ptr(end), ptr(tg), ptr(tr), ptr(n), n_max,
                           _capi.stream_ptr()), lib)
    cols = N // 2 if kind >= 0 else N
    xd, wd = x.cuda(), pack_tiles(w.view(E * N, K)).cuda()
    y = torch.full((P + 1, cols), 7.0, dtype=BF16, device="cuda")
    a = _capi.GroupLinearArgs()
    a.dtype, a.glu, a.limit = 0, kind, 0.7
    a.x, a.ldx, a.W, a.y, a.ldy = ptr(xd), K, ptr(wd), ptr(y), cols
    a.N, a.K, a.groups, a.M = N, K, E, P
    a.perm, a.tile_group, a.tile_row, a.n_tiles, a.group_end = ptr(perm), ptr(tg), ptr(tr), ptr(n), ptr(end)
    a.rows_per_x, a.max_tiles, a.tile_rows = top, n_max, 256
    check(lib.msa_group_linear(ctypes.byref(a), _capi.stream_ptr()), lib)
    torch.cuda.synchronize()
    assert bool((y[P] == 7.0).all()), "wrote past the last row"
    first = 0
    order = torch.sort(flat, stable=True).indices
    for e, count in enumerate(counts):
        ref = x[order[first:first + count] // top].double() @ w[e].double().T
        if kind >= 0:
            ref = glu(kind, ref[:, 0::2], ref[:, 1::2], 0.7)
        if count:
            close(y[first:first + count], ref, 6e-3, "group of %d" % count)
        first += count


# groups whose mean is up to half a tile (their weights pass by the caches) and beyond, some of two tiles, in all heights of tiles;
# sums whose last stage of 16 or 8 steps is full, nearly empty or the only one
@pytest.mark.parametrize("rows", [16, 32, 64, 256])
@pytest.mark.parametrize("dense", [False, True])
@pytest.mark.parametrize("N,K", [(288, 704), (160, 128), (96, 1088)])
def test_group_linear_routed_tiles_read_once_or_often(rows, dense, N, K):
    lib = _capi.load_hybrid()
    print("routed", rows, dense, N, K, flush=True)
    g = gen(N + rows)
    counts = [0, 1, rows - 1, rows, rows + 1] + [2] * 9 + [rows] * (20 if dense else 0)
    E, P = len(counts), sum(counts)
    limit = 64 if rows == 256 else rows / 2
    assert (P > E * limit) == dense
    flat = torch.repeat_interleave(torch.arange(E), torch.tensor(counts))[torch.randperm(P, generator=g)]
    x = torch.randn(P, K, generator=g).to(BF16)
    w = (torch.randn(E, N, K, generator=g) * K ** -0.5).to(BF16)
    n_max = P // rows + E
    ids = flat.int().cuda()
    perm, inv = (torch.full((P,), -1, dtype=torch.int32, device="cuda") for _ in range(2))
    end, n = torch.zeros(E, dtype=torch.int32, device="cuda"), torch.zeros(1, dtype=torch.int32, device="cuda")
    tg, tr = (torch.full((n_max,), -1, dtype=torch.int32, device="cuda") for _ in range(2))
    check(lib.msa_moe_plan(ptr(ids), P, E, rows, ptr(perm), ptr(inv), ptr(end), ptr(tg), ptr(tr), ptr(n), n_max,
                           _capi.stream_ptr()), lib)
    xd, wd = x.cuda(), pack_tiles(w.view(E * N, K)).cuda()
    y = torch.full((P + 1, N), 7.0, dtype=BF16, device="cuda")
    a = _capi.GroupLinearArgs()
    a.dtype, a.glu = 0, -1
    a.x, a.ldx, a.W, a.y, a.ldy = ptr(xd), K, ptr(wd), ptr(y), N
    a.N, a.K, a.groups, a.M = N, K, E, P
    a.perm, a.tile_group, a.tile_row, a.n_tiles, a.group_end = ptr(perm), ptr(tg), ptr(tr), ptr(n), ptr(end)
    a.rows_per_x, a.max_tiles, a.tile_rows = 1, n_max, rows
    check(lib.msa_group_linear(ctypes.byref(a), _capi.stream_ptr()), lib)
    torch.cuda.synchronize()
    assert bool((y[P] == 7.0).all()), "wrote past the last row"
    order = torch.sort(flat, stable=True).indices
    ref = torch.stack([x[p].double() @ w[flat[p]].double().T for p in order.tolist()])
    close(y[:P], ref, 6e-3, "rows %d" % rows)


# experts of one tile of every height and of several, the first and the last among them, where each asks for its own
@pytest.mark.parametrize("rows,counts", [(16, [16, 0, 17, 1, 33, 15]), (32, [33, 32, 0, 64, 65, 1, 3, 31]), (64, [64, 65, 1, 128, 0, 129, 63]),
                                         (256, [130, 192, 0, 257, 406, 449, 193, 1, 128, 256, 129, 0, 3, 0, 0, 385] + [1] * 8)])
@pytest.mark.parametrize("kind", [-1, _capi.MSA_GLU_CLAMPED])
def test_group_linear_tiles_of_experts_of_one_and_several(rows, counts, kind):
    lib = _capi.load_hybrid()
    print("experts", rows, kind, flush=True)
    g, N, K = gen(rows + kind), 544, 576
    E, P = len(counts), sum(counts)
    assert rows < 256 or P <= E * 128
    flat = torch.repeat_interleave(torch.arange(E), torch.tensor(counts))[torch.randperm(P, generator=g)]
    x = torch.randn(P, K, generator=g).to(BF16)
    w = (torch.randn(E, N, K, generator=g) * K ** -0.5).to(BF16)
    n_max = P // rows + E
    ids = flat.int().cuda()
    perm, inv = (torch.full((P,), -1, dtype=torch.int32, device="cuda") for _ in range(2))
    end, n = torch.zeros(E, dtype=torch.int32, device="cuda"), torch.zeros(1, dtype=torch.int32, device="cuda")
    tg, tr = (torch.full((n_max,), -1, dtype=torch.int32, device="cuda") for _ in range(2))
    check(lib.msa_moe_plan(ptr(ids), P, E, rows, ptr(perm), ptr(inv), ptr(end), ptr(tg), ptr(tr), ptr(n), n_max,
                           _capi.stream_ptr()), lib)
    cols = N // 2 if kind >= 0 else N
    xd, wd = x.cuda(), pack_tiles(w.view(E * N, K)).cuda()
    y = torch.full((P + 1, cols), 7.0, dtype=BF16, device="cuda")
    a = _capi.GroupLinearArgs()
    a.dtype, a.glu, a.limit = 0, kind, 0.7
    a.x, a.ldx, a.W, a.y, a.ldy = ptr(xd), K, ptr(wd), ptr(y), cols
    a.N, a.K, a.groups, a.M = N, K, E, P
    a.perm, a.tile_group, a.tile_row, a.n_tiles, a.group_end = ptr(perm), ptr(tg), ptr(tr), ptr(n), ptr(end)
    a.rows_per_x, a.max_tiles, a.tile_rows = 1, n_max, rows
    check(lib.msa_group_linear(ctypes.byref(a), _capi.stream_ptr()), lib)
    torch.cuda.synchronize()
    assert bool((y[P] == 7.0).all()), "wrote past the last row"
    first, order = 0, torch.sort(flat, stable=True).indices
    for e, count in enumerate(counts):
        ref = x[order[first:first + count]].double() @ w[e].double().T
        if kind >= 0:
            ref = glu(kind, ref[:, 0::2], ref[:, 1::2], 0.7)
        if count:
            close(y[first:first + count], ref, 6e-3, "expert of %d" % count)
        first += count


@pytest.mark.parametrize("E,groups,keep,top", [(1, 1, 1, 1), (12, 1, 1, 5), (12, 4, 2, 3),
                                               (96, 8, 3, 10), (512, 16, 16, 8), (300, 100, 1, 3)])
def test_route_and_plan(E, groups, keep, top):
    lib = _capi.load_hybrid()
    M = 77
    z = torch.randn(M, E + 5, generator=gen(E)) * 2
    want_ids, want_w = O.route(z[:, :E].double(), dict(
        top=top, scale=1.7, groups=dict(count=groups, keep=keep)))
    zd = z.cuda()
    ids = torch.zeros(M, top, dtype=torch.int32, device="cuda")
    w = torch.zeros(M, top, device="cuda")
    sg = torch.zeros(M, device="cuda")
    check(lib.msa_moe_route(ptr(zd), E + 5, M, E, groups, keep, top, 1.7, ptr(ids), ptr(w), ptr(sg),
                            _capi.stream_ptr()), lib)
    assert torch.equal(ids.cpu().long(), want_ids)
    close(w, want_w, 1e-5, "weights")
    close(sg, torch.sigmoid(z[:, E].double()), 1e-6, "shared gate")
    P = M * top
    for rows in (16, 64):
        n_max = P // rows + min(E, P)
        perm, inv = (torch.full((P,), -1, dtype=torch.int32, device="cuda") for _ in range(2))
        end = torch.zeros(E, dtype=torch.int32, device="cuda")
        tg, tr = (torch.full((n_max,), -1, dtype=torch.int32, device="cuda") for _ in range(2))
        n = torch.zeros(1, dtype=torch.int32, device="cuda")
        check(lib.msa_moe_plan(ptr(ids), P, E, rows, ptr(perm), ptr(inv), ptr(end), ptr(tg), ptr(tr),
                               ptr(n), n_max, _capi.stream_ptr()), lib)
        flat = ids.cpu().view(-1).long()
        order = torch.sort(flat, stable=True).indices
        assert torch.equal(perm.cpu().long(), order)
        assert torch.equal(inv.cpu().long()[order], torch.arange(P))
        counts = torch.bincount(flat, minlength=E)
        assert torch.equal(end.cpu().long(), counts.cumsum(0))
        tiles = [(e, int(counts[:e].sum()) + r) for e in range(E)
                 for r in range(0, int(counts[e]), rows)]
        assert int(n) == len(tiles)
        assert list(zip(tg.cpu().tolist(), tr.cpu().tolist()))[:len(tiles)] == tiles


@pytest.mark.parametrize("P,E", [(1, 3), (64, 2), (1025, 512), (8192, 7), (8256, 64), (48304, 64)])
def test_plan_of_many_pairs(P, E):
    """Runs of pairs per wave of one load, of several and of a few left over; waves without any."""
    lib = _capi.load_hybrid()
    flat = torch.randint(0, E, (P,), generator=gen(P))
    rows, n_max = 256, P // 256 + min(E, P)
    ids = flat.int().cuda()
    perm, inv = (torch.full((P,), -1, dtype=torch.int32, device="cuda") for _ in range(2))
    end = torch.zeros(E, dtype=torch.int32, device="cuda")
    tg, tr = (torch.full((n_max,), -1, dtype=torch.int32, device="cuda") for _ in range(2))
    n = torch.zeros(1, dtype=torch.int32, device="cuda")
    check(lib.msa_moe_plan(ptr(ids), P, E, rows, ptr(perm), ptr(inv), ptr(end), ptr(tg), ptr(tr), ptr(n), n_max,
                           _capi.stream_ptr()), lib)
    order, counts = torch.sort(flat, stable=True).indices, torch.bincount(flat, minlength=E)
    assert torch.equal(perm.cpu().long(), order)
    assert torch.equal(inv.cpu().long()[order], torch.arange(P))
    assert torch.equal(end.cpu().long(), counts.cumsum(0))
    tiles = [(e, int(counts[:e].sum()) + r) for e in range(E) for r in range(0, int(counts[e]), rows)]
    assert list(zip(tg.cpu().tolist(), tr.cpu().tolist()))[:int(n)] == tiles


@pytest.mark.parametrize("hd", [32, 64, 96, 128, 192, 256])
@pytest.mark.parametrize("T,pos0", [(1, 0), (17, 3), (64, 64), (130, 0), (33, 400), (300, 100)])
def test_flash_attention(hd, T, pos0):
    lib = _capi.load_hybrid()
    heads, S = 3, T + pos0
    g = gen(hd + T)
    q = torch.randn(T, heads * hd, generator=g).to(BF16)
    kv = torch.randn(S, 2 * heads * hd, generator=g).to(BF16)
    scale = 1.5 * hd ** -0.5
    k, v = (t.double().view(S, heads, hd) for t in kv.split(heads * hd, dim=1))
    s = torch.einsum("thd,shd->hts", q.double().view(T, heads, hd), k) * scale
    mask = torch.arange(S).view(1, S) > pos0 + torch.arange(T).view(T, 1)
    p = torch.softmax(s.masked_fill(mask, float("-inf")), dim=-1)
    ref = torch.einsum("hts,shd->thd", p, v).reshape(T, heads * hd)
    out = torch.zeros(T, heads * hd, dtype=BF16, device="cuda")
    qd, kvd = q.cuda(), kv.cuda()
    check(lib.msa_flash_attention_bf16(ptr(qd), heads * hd, ptr(kvd), 2 * heads * hd, ptr(out),
                                       heads * hd, 0, 0, heads, hd, T, pos0, scale,
                                       _capi.stream_ptr()), lib)
    close(out, ref, 1e-2, "flash %d" % hd)


@pytest.mark.parametrize("hd,heads,segs", [
    (128, 9, [(130, 0), (1, 500), (128, 64), (17, 3), (300, 100)]), (64, 3, [(33, 0)]),
    (32, 8, [(17 + 3 * i, (5 * i) % 70) for i in range(32)])])
@pytest.mark.parametrize("packed", [False, True])
def test_flash_attention_of_several_segments(hd, heads, segs, packed):
    """The bits that each segment gives by itself, wherever its rows lie."""
    lib = _capi.load_hybrid()
    g = gen(hd)
    gap = 5                     # rows between the segments
    row0, kv0 = [], [0]
    for n, p in segs:
        row0.append(gap + (row0[-1] + segs[len(row0) - 1][0] if row0 else 0))
        kv0.append(kv0[-1] + n + p)
    M, D, scale = row0[-1] + segs[-1][0], heads * hd, 1.5 * hd ** -0.5
    mb = (M + 15) // 16 if packed else 0
    q = torch.randn(M, D, generator=g).to(BF16).cuda()
    kv = torch.randn(kv0[-1], 2 * D, generator=g).to(BF16).cuda()
    out, want = (torch.full((max(M, 16 * mb) * D,), 7.0, dtype=BF16, device="cuda") for _ in range(2))
    ints = lambda x: (ctypes.c_int32 * len(x))(*x)
    n, p = zip(*segs)
    check(lib.msa_flash_attention_segments_bf16(ptr(q), D, ptr(kv), 2 * D, ptr(out), D, mb, heads, hd, len(segs),
                                                ints(row0), ints(n), ints(p), scale, _capi.stream_ptr()), lib)
    for i, (n, p) in enumerate(segs):
        check(lib.msa_flash_attention_bf16(ptr(q[row0[i]:]), D, ptr(kv[kv0[i]:]), 2 * D, ptr(want), D, mb, row0[i],
                                           heads, hd, n, p, scale, _capi.stream_ptr()), lib)
    torch.cuda.synchronize()
    assert torch.equal(out, want) and bool((out != 7.0).any())
    one = ints([1] * 33)
    assert lib.msa_flash_attention_segments_bf16(ptr(q), D, ptr(kv), 2 * D, ptr(out), D, mb, heads, hd, 33, one, one,
                                                 one, scale, _capi.stream_ptr()) == -1


def test_flash_attention_of_more_than_1024_workgroups():
    """Head by head, where few workgroups take the longest query tiles of all heads first."""
    test_flash_attention_of_several_segments(64, 9, [(257 + 4 * i, 37 * i % 300) for i in range(32)], False)


@pytest.mark.parametrize("kv_heads,chunk", [(8, 0), (2, 0), (8, 100)])
def test_grouped_prompts_of_more_than_1024_workgroups(kv_heads, chunk):
    """Head by head, where few workgroups take the longest query tiles of all heads first: every segment holds the bits
    that it gets alone."""
    lib = _capi.load_hybrid()
    heads, hd, rows, g = 16, 64, 400, gen(kv_heads)
    segs = [(i, -1 if i == 7 else 3 * i % 50, 130 + 5 * i) for i in range(33)]
    M, D = sum(n for _, _, n in segs), (heads + 2 * kv_heads) * hd
    b, alive = _batch(segs, M)
    x = torch.randn(M, D, generator=g).to(BF16).cuda()
    kc, vc = (torch.randn(33, kv_heads, rows, hd, generator=g).to(BF16).cuda() for _ in range(2))
    out, want = (torch.full((M, heads * hd), 7.0, dtype=BF16, device="cuda") for _ in range(2))
    a = _capi.GroupedArgs()
    a.dtype, a.heads, a.kv_heads, a.hd, a.vd, a.chunk, a.rows, a.scale, a.splits = 0, heads, kv_heads, hd, hd, chunk, rows, 0.2, 1
    a.q, a.k, a.v, a.ld = ptr(x), ptr(x[:, heads * hd:]), ptr(x[:, (heads + kv_heads) * hd:]), D
    a.k_cache, a.v_cache, a.out, a.ldo = ptr(kc), ptr(vc), ptr(out), heads * hd
    to = ctypes.byref(a), ctypes.byref(b)
    assert heads * 3 * len(segs) > 1024
    check(lib.msa_grouped_attention(*to, 0, len(segs), max(n for _, _, n in segs), _capi.stream_ptr()), lib)
    a.out = ptr(want)
    for i, (_, _, n) in enumerate(segs):
        check(lib.msa_grouped_attention(*to, i, i + 1, n, _capi.stream_ptr()), lib)
    torch.cuda.synchronize()
    at = sum(n for _, _, n in segs[:7])
    assert torch.equal(out, want) and bool((out[:at] != 7.0).any(1).all()) and bool((out[at:at + segs[7][2]] == 7.0).all())
    del alive


# one and several segments of few workgroups (two groups of waves from 385 tokens on), an odd number of key tiles, cached
# keys in front, chunks; the plain sums in 64 bits
@pytest.mark.parametrize("heads,kv_heads,hd,chunk,segs", [
    (4, 2, 64, 0, [(0, 0, 385)]), (8, 8, 128, 0, [(0, 0, 449)]), (3, 1, 128, 0, [(1, 37, 600), (0, 0, 130)]),
    (2, 1, 64, 300, [(0, 50, 700)]), (4, 1, 128, 0, [(0, 0, 385), (1, -1, 20), (2, 5, 512)]), (2, 2, 192, 0, [(0, 0, 400)])])
def test_grouped_prompts_of_few_workgroups(heads, kv_heads, hd, chunk, segs, vd=None, groups=None):
    lib = _capi.load_hybrid()
    vd = vd or hd
    print("grouped", heads, kv_heads, hd, vd, chunk, segs, flush=True)
    rows, g, scale = 800, gen(hd), 0.15
    M, D = sum(n for _, _, n in segs), heads * hd + kv_heads * (hd + vd)
    b, alive = _batch(segs, M)
    x = torch.randn(M, D, generator=g).to(BF16)
    kc, vc = (torch.randn(len(segs), kv_heads, rows, n, generator=g).to(BF16) for n in (hd, vd))
    xd, kcd, vcd = x.cuda(), kc.cuda(), vc.cuda()
    out = torch.full((M, heads * vd), 7.0, dtype=BF16, device="cuda")
    a = _capi.GroupedArgs()
    a.dtype, a.heads, a.kv_heads, a.hd, a.vd, a.chunk, a.rows, a.scale, a.splits = 0, heads, kv_heads, hd, vd, chunk, rows, scale, 1
    a.q, a.k, a.v, a.ld = ptr(xd), ptr(xd[:, heads * hd:]), ptr(xd[:, (heads + kv_heads) * hd:]), D
    a.k_cache, a.v_cache, a.out, a.ldo = ptr(kcd), ptr(vcd), ptr(out), heads * vd
    if groups:
        assert lib.msa_grouped_attention_groups(ctypes.byref(a), ctypes.byref(b), 0, len(segs), b.max_count) == groups
    check(lib.msa_grouped_attention(ctypes.byref(a), ctypes.byref(b), 0, len(segs), max(n for _, _, n in segs),
                                    _capi.stream_ptr()), lib)
    torch.cuda.synchronize()
    first = 0
    for slot, pos, n in segs:
        mine, got = x[first:first + n].double(), out[first:first + n].double().cpu()
        first += n
        if pos < 0:
            assert bool((got == 7.0).all())
            continue
        start = pos // chunk * chunk if chunk else 0      # the cache holds the chunk that the first token is in
        q, k = mine[:, :(heads + kv_heads) * hd].view(n, -1, hd).split([heads, kv_heads], 1)
        v = mine[:, (heads + kv_heads) * hd:].view(n, -1, vd)
        k = torch.cat([kc[slot, :, :pos - start].double().transpose(0, 1), k]).repeat_interleave(heads // kv_heads, 1)
        v = torch.cat([vc[slot, :, :pos - start].double().transpose(0, 1), v]).repeat_interleave(heads // kv_heads, 1)
        at, key = torch.arange(pos, pos + n)[:, None], torch.arange(start, pos + n)[None]
        seen = (key <= at) & (key >= (at // chunk * chunk if chunk else 0))
        s = (torch.einsum("qhd,khd->hqk", q, k) * scale).masked_fill(~seen, float("-inf"))
        want = torch.einsum("hqk,khd->qhd", torch.softmax(s, -1), v).reshape(n, heads * vd)
        # probabilities rounded to bf16 (2^-9 each, of either sign) and one rounding of the result
        assert float((got - want).norm() / want.norm()) < 2.0 ** -8
    del alive


# values of another size than the keys; chunks that leave a tile of queries two, three and more key tiles, with both forms
@pytest.mark.parametrize("heads,kv_heads,hd,vd,chunk,segs,groups", [
    (4, 1, 64, 128, 0, [(0, 0, 500)], 2), (2, 2, 128, 64, 0, [(0, 20, 450)], 2), (2, 1, 192, 64, 0, [(0, 0, 385)], 2),
    (2, 1, 64, 192, 0, [(0, 0, 400), (1, 0, 90)], 2), (2, 2, 64, 64, 64, [(0, 0, 400)], 2), (4, 2, 64, 128, 48, [(0, 100, 400)], 2),
    (4, 2, 128, 128, 64, [(0, 30, 400)], 1), (4, 2, 128, 128, 64, [(0, 64, 400)], 2), (4, 2, 128, 128, 256, [(0, 200, 400)], 2), (64, 8, 128, 64, 64, [(0, 0, 640)], 1)])
def test_grouped_prompts_of_chunks_and_value_sizes(heads, kv_heads, hd, vd, chunk, segs, groups):
    test_grouped_prompts_of_few_workgroups(heads, kv_heads, hd, chunk, segs, vd, groups)


def test_gathered_latents():
    lib = _capi.load_hybrid()
    for rp, slots, counts in ((512, [3, 0, 2], [70, 1, 33]), (24, [1], [7]), (80, list(range(32)), [9] * 32)):
        c = torch.randn(32, 70, rp).to(BF16).cuda()
        out = torch.full((sum(counts) + 1, rp), 7.0, dtype=BF16, device="cuda")
        ints = lambda x: (ctypes.c_int32 * len(x))(*x)
        check(lib.msa_gather_latents_bf16(ptr(c), 70, rp, len(slots), ints(slots), ints(counts), ptr(out),
                                          _capi.stream_ptr()), lib)
        want = torch.cat([c[s, :n] for s, n in zip(slots, counts)])
        assert torch.equal(out[:-1], want) and bool((out[-1] == 7.0).all())
        assert lib.msa_gather_latents_bf16(ptr(c), 70, rp, 1, ints([0]), ints([71]), ptr(out), _capi.stream_ptr()) == -1


@pytest.mark.parametrize("dtype", [BF16, F32], ids=["bf16", "f32"])
@pytest.mark.parametrize("rp", [128, 192, 256, 384, 512, 640])
def test_latent_attention(rp, dtype):
    """Rows of several slots at their own positions, an inactive row, and one to eight splits."""
    lib = _capi.load_hybrid()
    heads, cap, slots = 19, 700, 3
    g = gen(rp)
    pos = [0, 31, 32, 127, 128, 129, 300, 640, 699, -1]
    slot = [i % slots for i in range(len(pos))]
    M = len(pos)
    c = torch.randn(slots, cap, rp, generator=g).to(dtype)
    q = torch.randn(M, heads, rp, generator=g).to(dtype)
    scale = 1.5 * rp ** -0.5
    ref = torch.zeros(M, heads, rp, dtype=torch.float64)
    for m in range(M):
        if pos[m] >= 0:
            rows = c[slot[m], :pos[m] + 1].double()
            ref[m] = torch.softmax(q[m].double() @ rows.T * scale, dim=-1) @ rows
    cd, qd = c.cuda(), q.cuda()
    ts = torch.tensor(slot, dtype=torch.int32, device="cuda")
    tp = torch.tensor(pos, dtype=torch.int32, device="cuda")
    for splits in (1, 2, 8):
        out = torch.full((M, heads, rp), 9.0, dtype=dtype, device="cuda")
        part = torch.zeros(M, heads, splits, rp + 4, device="cuda")
        check(lib.msa_latent_attention(0 if dtype == BF16 else 1, ptr(qd), ptr(cd), cap, heads, rp,
                                       scale, ptr(out), ptr(part), splits, ptr(ts), ptr(tp), M,
                                       _capi.stream_ptr()), lib)
        close(out, ref, 1e-2 if dtype == BF16 else 1e-5, "latent %d, %d splits" % (rp, splits))


def _batch(segments, M):
    """A msa_batch of (slot, first position, tokens) segments with its tensors."""
    start, slot, pos = [0], [], []
    tok = [[], [], []]
    for s, p, n in segments:
        start.append(start[-1] + n)
        slot.append(s)
        pos.append(p)
        tok[0] += [s] * n
        tok[1] += [p + i if p >= 0 else -1 for i in range(n)]
        tok[2] += range(n)
    dev = [torch.tensor(x, dtype=torch.int32, device="cuda") for x in tok + [start, slot, pos]]
    b = _capi.Batch()
    b.M, b.nseg, b.max_count = M, len(slot), max(n for _, _, n in segments)
    (b.tok_slot, b.tok_pos, b.tok_off, b.seg_start, b.seg_slot, b.seg_pos) = map(ptr, dev)
    host = [(ctypes.c_int32 * len(x))(*x) for x in (start, slot, pos)]
    b.host_start, b.host_slot, b.host_pos = host
    return b, (dev, host)


@pytest.mark.parametrize("heads,kv_heads,dim,dp,vp,counts", [
    (4, 2, 30, 32, 48, (5, 1, 40)), (3, 3, 128, 128, 64, (17, 16)), (2, 1, 250, 256, 32, (33,)),
    (32, 8, 64, 64, 64, (9, 2, 1, 30, 16, 17, 3, 4)),      # eight lanes per column
    (64, 64, 128, 128, 32, (7, 20, 1, 2, 1, 1, 1, 1)), (32, 16, 96, 96, 64, (5,) * 8),
    (6, 3, 90, 96, 80, (1, 1, 1)), (3, 1, 128, 128, 208, (1,) * 5)])
@pytest.mark.parametrize("channels", [False, True], ids=["head decays", "channel decays"])
@pytest.mark.parametrize("dtype", [BF16, F32], ids=["bf16", "f32"])
def test_delta_scan(heads, kv_heads, dim, dp, vp, counts, dtype, channels):
    """Several segments, one of them continuing its slot's state and (with three or more) one
    inactive; outputs and the states left behind.  Segments of one token each also through the
    one-launch step."""
    lib = _capi.load_hybrid()
    print("delta_scan", heads, kv_heads, dim, dp, vp, counts, channels, flush=True)
    g = gen(heads + dp)
    M, slots = sum(counts), len(counts) + 1
    C = 2 * kv_heads * dp + heads * vp
    qkv = torch.randn(M, C, generator=g)
    qkv[:, :2 * kv_heads * dp].view(M, 2 * kv_heads, dp)[:, :, dim:] = 0
    qkv = qkv.to(dtype)
    ba = torch.randn(M, 2 * heads + 3, generator=g)
    rate, dtb = torch.rand(heads, generator=g) * 0.3, torch.randn(heads, generator=g)
    decays = torch.rand(M, heads, dp, generator=g) ** 0.25
    state = torch.randn(slots, heads, vp, dp, generator=g)
    state[..., dim:] = 0
    segs = [(slots - 1 - i, 0 if i else 12, n) for i, n in enumerate(counts)]
    if len(counts) > 2:
        segs[1] = (segs[1][0], -1, segs[1][2])
    want, S = torch.zeros(M, heads, vp, dtype=torch.float64), state.double().clone()
    x = qkv.double()
    unit = lambda t: t / torch.sqrt((t * t).sum(-1, keepdim=True) + 1e-6)
    at = 0
    for slot, pos, n in segs:
        if pos >= 0:
            s = S[slot] if pos > 0 else torch.zeros_like(S[slot])       # [heads, vp, dp]
            for m in range(at, at + n):
                q = unit(x[m, :kv_heads * dp].view(kv_heads, dp)) * dim ** -0.5
                k = unit(x[m, kv_heads * dp:2 * kv_heads * dp].view(kv_heads, dp))
                q, k = (t.repeat_interleave(heads // kv_heads, 0) for t in (q, k))
                v = x[m, 2 * kv_heads * dp:].view(heads, vp)
                z = ba[m].double()
                beta = torch.sigmoid(z[:heads])
                decay = torch.exp(-rate.double() * torch.nn.functional.softplus(
                    z[heads:2 * heads] + dtb.double()))
                s = s * (decays[m].double().unsqueeze(1) if channels else decay.view(-1, 1, 1))
                u = beta.view(-1, 1) * (v - torch.einsum("hvd,hd->hv", s, k))
                s = s + u.unsqueeze(2) * k.unsqueeze(1)
                want[m] = torch.einsum("hvd,hd->hv", s, q)
            S[slot] = s
        at += n
    b, alive = _batch(segs, M)
    qd, bd, rd, td, sd, dd = (t.cuda() for t in (qkv, ba, rate, dtb, state, decays))
    o = torch.full((M, heads * vp), 7.0, device="cuda")
    a = _capi.DeltaArgs()
    a.dtype, a.heads, a.kv_heads, a.dim, a.dp, a.vp = int(dtype == F32), heads, kv_heads, dim, dp, vp
    a.qkv, a.ld, a.ba, a.ldba, a.state, a.o = ptr(qd), C, ptr(bd), 2 * heads + 3, ptr(sd), ptr(o)
    if channels:
        a.decay = ptr(dd)
    else:
        a.decay_rate, a.dt_bias = ptr(rd), ptr(td)
    if b.max_count == 1:
        step = state.cuda()
        out = torch.zeros(M, heads * vp, dtype=dtype, device="cuda")
        gate, w = torch.randn(M, heads * vp, generator=g).to(dtype), torch.randn(vp, generator=g)
        gd, wd = gate.cuda(), w.cuda()
        a.state, a.vdim, a.gate, a.ld_gate, a.w = ptr(step), vp, ptr(gd), heads * vp, ptr(wd)
        a.out, a.ld_out, a.eps = ptr(out), heads * vp, 1e-5
        for act, f in ((_capi.MSA_GATE_SILU, torch.nn.functional.silu),
                       (_capi.MSA_GATE_SIGMOID, torch.sigmoid)):
            step.copy_(state)
            a.gate_act = act
            check(lib.msa_delta_step(ctypes.byref(a), ctypes.byref(b), _capi.stream_ptr()), lib)
            normed = O.rms(want, 1e-5, w.double()) * f(gate.double()).view(M, heads, vp)
            on = [m for m in range(M) if segs[m][1] >= 0]
            close(out.view(M, heads, vp)[on], normed[on], 2e-5 if dtype == F32 else 6e-3, "step")
            close(step, S, 2e-5, "states of the step")
        a.state = ptr(sd)
    check(lib.msa_delta_scan(ctypes.byref(a), ctypes.byref(b), _capi.stream_ptr()), lib)
    close(o.view(M, heads, vp), want, 2e-5, "outputs")
    close(sd, S, 2e-5, "states")
    del alive


# segments around the chunks' edges (16 tokens) and the sizes from which they are taken: few segments (96 tokens),
# many (48), one column tile, four and eight, tiles of the state that do not fill the four waves
@pytest.mark.parametrize("channels", [False, True])
@pytest.mark.parametrize("heads,kv_heads,dim,dp,vp,counts", [
    (4, 2, 128, 128, 128, [100]), (4, 4, 120, 128, 16, [97, 112, 16, 1, 33]),
    (3, 1, 64, 64, 48, [96, 17, 200]), (2, 1, 90, 96, 32, [15, 111, 31]), (5, 5, 24, 32, 16, [129, 5, 64]),
    (32, 8, 128, 128, 128, [49, 3, 64, 17]), (33, 33, 64, 64, 64, [15, 50, 1, 32]),
    (64, 32, 32, 32, 128, [48, 16])])
@pytest.mark.parametrize("dtype", [BF16, F32])
def test_delta_chunks(heads, kv_heads, dim, dp, vp, counts, dtype, channels):
    """Sixteen tokens at a time against the recurrence in float64, beside the token-by-token scan of the same
    fp32 precision: channels that forget at once or never, a segment that continues its slot's state, an
    inactive one."""
    lib = _capi.load_hybrid()
    print("delta_chunks", heads, kv_heads, dim, dp, vp, counts, channels, flush=True)
    g = gen(heads + dp)
    M, slots = sum(counts), len(counts) + 1
    C = 2 * kv_heads * dp + heads * vp
    qkv = torch.randn(M, C, generator=g)
    qkv[:, :2 * kv_heads * dp].view(M, 2 * kv_heads, dp)[:, :, dim:] = 0
    qkv = qkv.to(dtype)
    ba = torch.randn(M, 2 * heads, generator=g)
    rate, dtb = torch.rand(heads, generator=g) * 0.3, torch.randn(heads, generator=g)
    decays = torch.rand(M, heads, dp, generator=g) ** 0.25
    decays[:, :, 5::13], decays[:, :, 3::11] = 0.0, 1.0
    decays[:, :, ::7] **= 40
    state = torch.randn(slots, heads, vp, dp, generator=g)
    state[..., dim:] = 0
    segs = [(slots - 1 - i, 0 if i else 12, n) for i, n in enumerate(counts)]
    if len(counts) > 2:
        segs[1] = (segs[1][0], -1, segs[1][2])
    want, S, x, at = torch.zeros(M, heads, vp, dtype=torch.float64), state.double().clone(), qkv.double(), 0
    unit = lambda t: t / torch.sqrt((t * t).sum(-1, keepdim=True) + 1e-6)
    q = (unit(x[:, :kv_heads * dp].view(M, kv_heads, dp)) * dim ** -0.5).repeat_interleave(heads // kv_heads, 1)
    k = unit(x[:, kv_heads * dp:2 * kv_heads * dp].view(M, kv_heads, dp)).repeat_interleave(heads // kv_heads, 1)
    v, z = x[:, 2 * kv_heads * dp:].view(M, heads, vp), ba.double()
    beta = torch.sigmoid(z[:, :heads])
    one = torch.exp(-rate.double() * torch.nn.functional.softplus(z[:, heads:] + dtb.double()))
    decay = decays.double() if channels else one.unsqueeze(2).expand(M, heads, dp)
    for slot, pos, n in segs:
        if pos >= 0:
            s = S[slot] if pos > 0 else torch.zeros_like(S[slot])       # [heads, vp, dp]
            for m in range(at, at + n):
                s = s * decay[m].unsqueeze(1)
                u = beta[m].unsqueeze(1) * (v[m] - (s * k[m].unsqueeze(1)).sum(-1))
                s = s + u.unsqueeze(2) * k[m].unsqueeze(1)
                want[m] = (s * q[m].unsqueeze(1)).sum(-1)
            S[slot] = s
        at += n
    want = want.view(M, -1)
    b, alive = _batch(segs, M)
    qd, bd, rd, td, dd = (t.cuda() for t in (qkv, ba, rate, dtb, decays))
    rel = lambda got, ref: float((got.double().cpu() - ref).norm() / ref.norm())
    errors = []
    for chunked in (False, True):
        sd, o = state.cuda(), torch.full((M, heads * vp), 7.0, device="cuda")
        a = _capi.DeltaArgs()
        a.dtype, a.heads, a.kv_heads, a.dim, a.dp, a.vp = int(dtype == F32), heads, kv_heads, dim, dp, vp
        a.qkv, a.ld, a.ba, a.ldba, a.state, a.o = ptr(qd), C, ptr(bd), 2 * heads, ptr(sd), ptr(o)
        if channels:
            a.decay = ptr(dd)
        else:
            a.decay_rate, a.dt_bias = ptr(rd), ptr(td)
        need = lib.msa_delta_scratch_floats(ctypes.byref(a), ctypes.byref(b))
        assert need > 0
        to = ctypes.byref(a), ctypes.byref(b)
        if chunked:
            scratch = torch.full((need,), float("nan"), device="cuda")
            assert lib.msa_delta_scan_chunks(*to, ptr(scratch), need - 1, _capi.stream_ptr()) == -2
            check(lib.msa_delta_scan_chunks(*to, ptr(scratch), need, _capi.stream_ptr()), lib)
        else:
            check(lib.msa_delta_scan(*to, _capi.stream_ptr()), lib)
        errors.append((rel(o, want), rel(sd, S)))
    print(errors, flush=True)
    # fp32 throughout, some 2 dp + 32 roundings behind every output, of random sign; the scan shows 1 to 3e-7
    for scan, chunks in zip(*errors):
        assert chunks <= max(1.5 * scan, 4 * 2.0 ** -24), errors
    del alive


@pytest.mark.parametrize("channels", [False, True])
@pytest.mark.parametrize("heads", [2, 64])
def test_delta_chunks_keep_a_nan_from_earlier_tokens(heads, channels):
    """A value that is not finite spoils its own column from its token on, a key that is not its head."""
    lib = _capi.load_hybrid()
    g, M, dp, vp, bad = gen(3), 128, 32, 128, 37
    C = 2 * heads * dp + heads * vp
    qkv = torch.randn(M, C, generator=g).to(BF16)
    qkv[bad, 2 * heads * dp + 5] = float("inf")              # value column 5 of head 0
    qkv[bad, heads * dp + dp + 3] = float("nan")             # a key of head 1
    ba, decays = torch.randn(M, 2 * heads, generator=g), torch.rand(M, heads, dp, generator=g)
    b, alive = _batch([(0, 0, M)], M)
    out = []
    for chunked in (False, True):
        qd, bd, dd = qkv.cuda(), ba.cuda(), decays.cuda()
        sd, o = torch.zeros(1, heads, vp, dp, device="cuda"), torch.zeros(M, heads * vp, device="cuda")
        rd = torch.ones(heads, device="cuda")
        a = _capi.DeltaArgs()
        a.dtype, a.heads, a.kv_heads, a.dim, a.dp, a.vp = 0, heads, heads, dp, dp, vp
        a.qkv, a.ld, a.ba, a.ldba, a.state, a.o = ptr(qd), C, ptr(bd), 2 * heads, ptr(sd), ptr(o)
        if channels:
            a.decay = ptr(dd)
        else:
            a.decay_rate, a.dt_bias = ptr(rd), ptr(rd)
        to = ctypes.byref(a), ctypes.byref(b)
        if chunked:
            scratch = torch.empty(lib.msa_delta_scratch_floats(*to), device="cuda")
            check(lib.msa_delta_scan_chunks(*to, ptr(scratch), scratch.numel(), _capi.stream_ptr()), lib)
        else:
            check(lib.msa_delta_scan(*to, _capi.stream_ptr()), lib)
        out.append((torch.isfinite(o).cpu(), o.cpu()))
    (fine, scan), (kept, chunks) = out
    assert not fine[bad, 5] and not fine[bad, vp] and bool(fine[:bad].all())
    assert torch.equal(fine, kept)
    assert float((scan - chunks)[fine].abs().max()) <= 2e-6 * float(scan[fine].abs().max())
    del alive

def _scan_and_chunks(qkv, ba, decays, state, heads, dp, vp, channels, segments=None):
    """Outputs and state of the scan and of the chunks over the same inputs."""
    lib = _capi.load_hybrid()
    M, C = qkv.shape
    b, alive = _batch(segments or [(0, 12, M)], M)
    out = []
    for chunked in (False, True):
        qd, bd, dd, sd = qkv.cuda(), ba.cuda(), decays.cuda(), state.cuda()
        o, rd = torch.zeros(M, heads * vp, device="cuda"), torch.ones(heads, device="cuda")
        a = _capi.DeltaArgs()
        a.dtype, a.heads, a.kv_heads, a.dim, a.dp, a.vp = int(qkv.dtype == F32), heads, heads, dp, dp, vp
        a.qkv, a.ld, a.ba, a.ldba, a.state, a.o = ptr(qd), C, ptr(bd), ba.shape[1], ptr(sd), ptr(o)
        if channels:
            a.decay = ptr(dd)
        else:
            a.decay_rate, a.dt_bias = ptr(rd), ptr(rd)
        to = ctypes.byref(a), ctypes.byref(b)
        if chunked:
            scratch = torch.empty(lib.msa_delta_scratch_floats(*to), device="cuda")
            check(lib.msa_delta_scan_chunks(*to, ptr(scratch), scratch.numel(), _capi.stream_ptr()), lib)
        else:
            check(lib.msa_delta_scan(*to, _capi.stream_ptr()), lib)
        out.append((o.cpu(), sd.cpu()))
    del alive
    return out


@pytest.mark.parametrize("channels", [False, True])
@pytest.mark.parametrize("heads", [3, 64])
@pytest.mark.parametrize("bad", [37, 111])
def test_delta_chunks_keep_a_nan_of_the_gates_from_earlier_tokens(bad, heads, channels):
    """A beta that is NaN (head 0), or a decay (head 1), spoils its head from its token on and nothing else."""
    g, M, dp, vp = gen(4), 112, 32, 128
    qkv = torch.randn(M, 2 * heads * dp + heads * vp, generator=g).to(BF16)
    ba, decays = torch.randn(M, 2 * heads, generator=g), torch.rand(M, heads, dp, generator=g)
    ba[bad, 0] = ba[bad, heads + 1] = decays[bad, 1] = float("nan")
    (scan, s_scan), (chunks, s_chunks) = _scan_and_chunks(qkv, ba, decays, torch.randn(1, heads, vp, dp, generator=g),
                                                          heads, dp, vp, channels)
    fine = torch.isfinite(scan)
    assert bool(fine[:bad].all()) and not bool(fine[bad:, :2 * vp].any()) and bool(fine[:, 2 * vp:].all())
    assert torch.equal(torch.isfinite(chunks), fine)
    assert torch.equal(torch.isfinite(s_chunks), torch.isfinite(s_scan))
    assert float((scan - chunks)[fine].abs().max()) <= 2e-6 * float(scan[fine].abs().max())


@pytest.mark.parametrize("channels", [False, True])
@pytest.mark.parametrize("heads", [3, 64])
def test_delta_segments_without_tokens(heads, channels):
    """In front, between and behind others: they change nothing, but one that begins its sequence leaves a state of
    zeros."""
    g, M, dp, vp = gen(6), 160, 32, 128
    qkv = torch.randn(M, 2 * heads * dp + heads * vp, generator=g).to(BF16)
    ba, decays = torch.randn(M, 2 * heads, generator=g), torch.rand(M, heads, dp, generator=g)
    state = torch.randn(6, heads, vp, dp, generator=g)
    run = lambda segs: _scan_and_chunks(qkv, ba, decays, state, heads, dp, vp, channels, segs)
    plain = run([(1, 12, 48), (4, 0, 112)])
    gaps = run([(0, 7, 0), (1, 12, 48), (2, 0, 0), (4, 0, 112), (3, 5, 0), (5, 0, 0)])
    for (o, s), (o2, s2) in zip(plain, gaps):
        assert torch.equal(o, o2)
        s[2] = s[5] = 0.0
        assert torch.equal(s, s2)


@pytest.mark.parametrize("channels", [False, True])
@pytest.mark.parametrize("heads", [3, 64])
@pytest.mark.parametrize("M", [112, 121])
def test_delta_chunks_of_huge_and_tiny_keys(M, heads, channels):
    """Keys and queries far from unit length, values and a state of up to 1e25: products of the raw vectors would
    overflow where the scan, which divides by the norms first, stays finite.  Vectors whose squared norm itself
    overflows count as zeros in both.  Seven and eight chunks; the last tokens are huge ones."""
    g, dp, vp = gen(5), 64, 128
    qk = torch.randn(M, 2 * heads, dp, generator=g)
    qk *= 10.0 ** torch.randint(-3, 19, (M, 2 * heads, 1), generator=g)
    qk[-1], qk[40] = 1e18 * torch.sign(qk[-1]), 3e25 * torch.sign(qk[40])
    v = torch.randn(M, heads * vp, generator=g) * 10.0 ** torch.randint(0, 26, (1, heads * vp), generator=g)
    qkv = torch.cat([qk.view(M, -1), v], dim=1)
    ba, decays = torch.randn(M, 2 * heads, generator=g), torch.rand(M, heads, dp, generator=g) ** 0.25
    state = torch.randn(1, heads, vp, dp, generator=g) * 10.0 ** torch.randint(0, 26, (vp, 1), generator=g)
    unit = lambda t: t / torch.sqrt((t * t).sum(-1, keepdim=True) + 1e-6)
    for x in (qkv, qkv.to(BF16)):
        d = x.double()
        q, k = (unit(t.view(M, heads, dp)) for t in (d[:, :heads * dp], d[:, heads * dp:2 * heads * dp]))
        q, k, v = q * dp ** -0.5, k.clone(), d[:, 2 * heads * dp:].view(M, heads, vp)
        q[40] = k[40] = 0.0
        beta = torch.sigmoid(ba[:, :heads].double())
        one = torch.exp(-torch.nn.functional.softplus(ba[:, heads:].double() + 1.0))
        s, want = state[0].double(), []
        size, most = s.norm(dim=-1), torch.zeros(heads, vp, dtype=torch.float64)  # of what is summed, per column
        for m in range(M):
            g = decays[m].double().unsqueeze(1) if channels else one[m].view(-1, 1, 1)
            s = s * g
            add = beta[m].unsqueeze(1) * (v[m] - (s * k[m].unsqueeze(1)).sum(-1))
            s = s + add.unsqueeze(2) * k[m].unsqueeze(1)
            want.append((s * q[m].unsqueeze(1)).sum(-1))
            size = torch.maximum(torch.maximum(size * g.amax(-1), add.abs()), s.norm(dim=-1))
            most = torch.maximum(most, size * dp ** -0.5)
        want = torch.stack(want)
        for o, end in _scan_and_chunks(x, ba, decays, state, heads, dp, vp, channels):
            assert bool(torch.isfinite(o).all()) and bool(torch.isfinite(end).all()) and not bool(o[40].any())
            off = float(((o.view(M, heads, vp).double() - want).abs().amax(0) / most).max())
            end_off = float(((end[0].double() - s).norm(dim=-1) / size).max())
            print(off, end_off, flush=True)
            # sums of dp + 32 terms of random sign, rounded each: 10 * 2^-24 of what is summed, and three times that
            # for the worst of thousands
            assert off <= 30 * 2.0 ** -24 and end_off <= 30 * 2.0 ** -24, (off, end_off)


@pytest.mark.parametrize("heads,kv_heads,dim,dp,vp,counts", [
    # a last group of one to three column tiles, in batches that fill the chip; one tile of many heads
    (16, 4, 24, 32, 80, [50, 3, 64, 17, 48, 1, 30, 50]), (64, 1, 64, 64, 144, [49, 48]), (43, 43, 90, 96, 112, [33, 20, 48]),
    (128, 2, 128, 128, 176, [49]), (64, 2, 120, 128, 16, [50, 48])])
def test_delta_chunks_of_any_number_of_column_tiles(heads, kv_heads, dim, dp, vp, counts):
    for channels in (False, True):
        test_delta_chunks(heads, kv_heads, dim, dp, vp, counts, BF16, channels)


@pytest.mark.parametrize("heads,vp,segs", [
    (31, 16, [(0, 12, 1700), (2, -1, 90), (3, 5, 1400), (1, 0, 10)]), (61, 48, [(1, 0, 1), (0, 3, 1601)])])
def test_delta_operands_kept_for_a_portion_of_the_chunks(heads, vp, segs):
    """More chunks than the scratch holds: segments that end before, in and behind a portion, a state carried across
    their borders."""
    g, dp, M = gen(9), 128, sum(n for _, _, n in segs)
    a, b = _capi.DeltaArgs(), _capi.Batch()
    a.heads, a.dp, a.vp, a.decay, b.M, b.nseg, b.max_count = heads, dp, vp, 4096, M, len(segs), max(n for _, _, n in segs)
    need = _capi.load_hybrid().msa_delta_scratch_floats(ctypes.byref(a), ctypes.byref(b))
    assert need <= 40 << 20 and need < (M // 16 + len(segs)) * heads * 6880
    qkv = torch.randn(M, 2 * heads * dp + heads * vp, generator=g).to(BF16)
    ba, decays = torch.randn(M, heads, generator=g), torch.rand(M, heads, dp, generator=g) ** 0.125
    state = torch.randn(4, heads, vp, dp, generator=g)
    (o, s), (o2, s2) = _scan_and_chunks(qkv, ba, decays, state, heads, dp, vp, True, segs)
    # both sum in fp32 what 2 dp + 32 products add, of random sign: some 3e-7 each
    assert float((o - o2).norm() / o.norm()) <= 1e-6 and float((s - s2).norm() / s.norm()) <= 1e-6


@pytest.mark.parametrize("channels", [False, True])
def test_delta_segments_without_tokens_beside_a_last_group_of_columns(channels):
    g, M, heads, dp, vp = gen(6), 160, 43, 32, 80
    qkv = torch.randn(M, 2 * heads * dp + heads * vp, generator=g).to(BF16)
    ba, decays = torch.randn(M, 2 * heads, generator=g), torch.rand(M, heads, dp, generator=g)
    state = torch.randn(6, heads, vp, dp, generator=g)
    out = _scan_and_chunks(qkv, ba, decays, state, heads, dp, vp, channels,
                           [(0, 7, 0), (1, 12, 48), (3, -1, 12), (2, 0, 0), (4, 0, 100)])
    (o, s), (o2, s2) = out
    assert torch.equal(s[[0, 2, 3, 5]], s2[[0, 2, 3, 5]]) and not bool(s2[2].any())
    assert torch.equal(s2[0], state[0]) and not bool(o2[48:60].any())
    assert float((o - o2).norm() / o.norm()) <= 1e-6 and float((s - s2).norm() / s.norm()) <= 1e-6


def test_selection_over_fp32_logits():
    """The fp32 forms of selection, scoring and sampling agree with plain PyTorch, at row strides
    and vocabulary sizes that are no multiple of 8."""
    lib = _capi.load()
    for V, ld in ((101, 112), (1000, 1000), (50001, 50016)):
        z = torch.randn(5, ld, generator=gen(V)).cuda() * 3
        lp = torch.log_softmax(z[:, :V].double(), dim=-1)
        tok = torch.zeros(5, dtype=torch.long, device="cuda")
        score = torch.zeros(5, device="cuda")
        ban = (ctypes.c_int32 * 1)(1)
        none = (ctypes.c_int32 * 1)()
        check(lib.msa_greedy_select_f32(ptr(z), ld, 5, V, 1.0, ban, 1, none, 0, None, None, 0, 2,
                                        ptr(tok), 1, ptr(score), 1, None, _capi.stream_ptr()))
        masked = lp.clone()
        masked[:, 1] = float("-inf")
        assert torch.equal(tok, masked.argmax(dim=-1))
        close(score, masked.max(dim=-1).values.cpu(), 1e-5, "score")
        target = torch.randint(0, V, (5,), generator=gen(1)).cuda()
        got = torch.zeros(5, device="cuda")
        check(lib.msa_target_logprob_f32(ptr(z), ld, 5, V, 1.0, ptr(target), ptr(got),
                                         _capi.stream_ptr()))
        close(got, lp.gather(1, target.view(-1, 1)).view(-1).cpu(), 1e-5, "target")
        rows = torch.zeros(5, V, device="cuda")
        check(lib.msa_log_softmax_f32(ptr(z), 0, ld, 1, 5, V, 1.0, ptr(rows), 0, V,
                                      _capi.stream_ptr()))
        close(rows, lp.cpu(), 1e-5, "log-softmax")
        noise = torch.empty(5, V, device="cuda").exponential_()
        check(lib.msa_sample_topp_f32(ptr(z), ld, 5, V, 1.0, None, ban, 1, none, 0, None, None, 0, 2,
                                      None, 0.999999, ptr(noise), None, None, 0.0, 0.0, 0.0, 0.0,
                                      None, None, 0, ptr(tok), 1, ptr(score), 1, _capi.stream_ptr()))
        p = torch.softmax(z[:, :V].double(), dim=-1)
        p[:, 1] = 0
        assert torch.equal(tok, (p / noise.double()).argmax(dim=-1))
