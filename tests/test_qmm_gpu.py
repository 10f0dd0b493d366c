"""GPU parity of the MFMA prefill product (logan_hip_affine_qmm) against the
oracle's restatement of the reference QMM (backend_metal.mm:1480-1560:
bf16-rounded dequantised weights, f32 accumulation).

Bars: f32 output within max|y-ŷ|/max|ŷ| <= 1e-5 of the oracle (the weights
are identical bf16 values; only the f32 summation order differs); bf16 output
equal to RNE of the f32 output; rows and columns past a tile edge untouched.
"""
import numpy as np
import pytest

import oracle
from logan_amd.synth import bf16_to_f32, make_affine, make_x

from _util import normwise_rel

pytestmark = pytest.mark.gpu


def to_dev(a, torch, dtype=None):
    t = torch.from_numpy(np.ascontiguousarray(a))
    if dtype is not None:
        t = t.view(dtype)
    return t.cuda()


def dev_matrix(torch, w, sc, bi, O, I, bits, gs, fp16=False):
    from logan_amd.device import AffineMatrix

    return AffineMatrix(to_dev(w, torch), to_dev(sc.view(np.int16), torch),
                        to_dev(bi.view(np.int16), torch), O, I, bits, gs, fp16)


def qmm_route(mats, M):
    """(form, tile rows, k ranges) that the library gives these matrices."""
    import ctypes as C
    from logan_amd import _lib as L

    arr = (L.Affine * len(mats))(*[m.c() for m in mats])
    r = (C.c_int * 3)()
    assert L.lib().logan_hip_affine_qmm_route(arr, len(mats), M, mats[0].I, r) == 1
    return tuple(r)


CASES = [
    # (M, O, I, bits, gs, fp16): tile edges in M and O, every width, group sizes
    (1, 64, 64, 4, 64, False),
    (7, 100, 128, 4, 32, False),
    (64, 64, 256, 5, 64, False),
    (130, 200, 256, 6, 128, True),
    (96, 72, 192, 8, 64, False),
    (64, 512, 2048, 4, 64, False),   # config-5 attention projection shape, one tile of M
    (33, 192, 1024, 5, 32, True),
    (65, 130, 512, 8, 128, False),
    (200, 96, 320, 5, 64, False),    # M > 64, partial tiles in M and N
    (300, 257, 128, 4, 32, True),
]


@pytest.mark.parametrize("M,O,I,bits,gs,fp16", CASES,
                         ids=lambda v: str(v))
def test_qmm_matches_oracle(gpu, M, O, I, bits, gs, fp16):
    import torch
    from logan_amd.device import affine_qmm

    rng = np.random.default_rng(M * 1000 + O + bits)
    w, sc, bi = make_affine(rng, O, I, bits, gs, fp16)
    xb = make_x(rng, M, I).reshape(M, I)
    m = dev_matrix(torch, w, sc, bi, O, I, bits, gs, fp16)
    x = to_dev(xb.view(np.int16), torch).view(torch.bfloat16)
    y = affine_qmm(m, x, out_dtype=torch.float32).cpu().numpy()
    ref = oracle.affine_qmm_bf16(bf16_to_f32(xb).reshape(M, I), w, sc, bi, O, I, bits, gs, fp16)
    assert normwise_rel(y, ref) <= 1e-5
    yb = affine_qmm(m, x, out_dtype=torch.bfloat16)
    assert torch.equal(yb, torch.from_numpy(y).cuda().to(torch.bfloat16))


def test_qmm_prefill_chunk(gpu):
    """M = 512 (the config-5 prefill chunk) through one 2048 x 2048 4-bit
    projection, against the oracle on a sample of output columns."""
    import torch
    from logan_amd.device import affine_qmm

    rng = np.random.default_rng(55)
    M, O, I, bits, gs = 512, 2048, 2048, 4, 64
    w, sc, bi = make_affine(rng, O, I, bits, gs)
    xb = make_x(rng, M, I).reshape(M, I)
    m = dev_matrix(torch, w, sc, bi, O, I, bits, gs)
    x = to_dev(xb.view(np.int16), torch).view(torch.bfloat16)
    y = affine_qmm(m, x, out_dtype=torch.float32).cpu().numpy()
    cols = np.arange(0, O, 61)
    ws = w.reshape(O, -1)[cols]
    ng = I // gs
    scs = sc.reshape(O, ng)[cols].reshape(-1)
    bis = bi.reshape(O, ng)[cols].reshape(-1)
    ref = oracle.affine_qmm_bf16(bf16_to_f32(xb).reshape(M, I), ws, scs, bis, len(cols), I, bits, gs)
    assert normwise_rel(y[:, cols], ref) <= 1e-5


@pytest.mark.parametrize("bits,gs,fp16", [(4, 64, False), (5, 64, True), (8, 128, False)])
def test_qmm_large_tiles_ragged(gpu, bits, gs, fp16):
    """50 column tiles of the tile kernel, partial tiles in both M and N,
    against the oracle on a sample of output columns (every column of the
    last, partial tile included)."""
    import torch
    from logan_amd.device import affine_qmm

    rng = np.random.default_rng(bits * 3 + gs)
    M, O, I = 500, 6337, 256
    w, sc, bi = make_affine(rng, O, I, bits, gs, fp16)
    xb = make_x(rng, M, I).reshape(M, I)
    m = dev_matrix(torch, w, sc, bi, O, I, bits, gs, fp16)
    x = to_dev(xb.view(np.int16), torch).view(torch.bfloat16)
    y = affine_qmm(m, x, out_dtype=torch.float32).cpu().numpy()
    cols = np.concatenate([np.arange(0, O, 53), np.arange(O - 65, O)])
    ng = I // gs
    ws = w.reshape(O, -1)[cols]
    scs = sc.reshape(O, ng)[cols].reshape(-1)
    bis = bi.reshape(O, ng)[cols].reshape(-1)
    ref = oracle.affine_qmm_bf16(bf16_to_f32(xb).reshape(M, I), ws, scs, bis, len(cols), I, bits, gs,
                                 fp16)
    assert normwise_rel(y[:, cols], ref) <= 1e-5
    yb = affine_qmm(m, x, out_dtype=torch.bfloat16)
    assert torch.equal(yb, torch.from_numpy(y).cuda().to(torch.bfloat16))


def test_qmm_leaves_outside_untouched(gpu):
    """A y with a wider stride: columns beyond O keep their contents."""
    import torch
    from logan_amd.device import AffineMatrix
    from logan_amd import _lib as L
    import ctypes as C

    rng = np.random.default_rng(9)
    M, O, I, bits, gs = 40, 70, 128, 4, 64
    w, sc, bi = make_affine(rng, O, I, bits, gs)
    m = dev_matrix(torch, w, sc, bi, O, I, bits, gs)
    x = to_dev(make_x(rng, M, I).reshape(M, I).view(np.int16), torch).view(torch.bfloat16)
    y = torch.full((M, 80), 7.0, dtype=torch.float32, device="cuda")
    a = m.c()
    rc = L.lib().logan_hip_affine_qmm(C.byref(a), x.data_ptr(), M, I, y.data_ptr(), 80,
                                      L.LOGAN_HIP_F32, None)
    torch.cuda.synchronize()
    assert rc == 1
    assert torch.all(y[:, O:] == 7.0)


@pytest.mark.parametrize("O,I", [(64, 2048), (512, 2048), (2048, 4096), (8192, 2048)],
                         ids=["ba", "k_v", "o_out", "q"])
def test_qmm_config5_prefill_projections(gpu, O, I):
    """The config-5 projections at the prefill chunk M = 512: grids with few
    tiles split K (ordered f32 partials and a reduction launch). Sampled
    output columns against the oracle; two calls give identical bits."""
    import torch
    from logan_amd.device import affine_qmm

    print(f"qmm config5 O={O} I={I}", flush=True)
    rng = np.random.default_rng(O + I)
    M, bits, gs = 512, 4, 64
    w, sc, bi = make_affine(rng, O, I, bits, gs)
    xb = make_x(rng, M, I).reshape(M, I)
    m = dev_matrix(torch, w, sc, bi, O, I, bits, gs)
    x = to_dev(xb.view(np.int16), torch).view(torch.bfloat16)
    y = affine_qmm(m, x, out_dtype=torch.float32)
    y2 = affine_qmm(m, x, out_dtype=torch.float32)
    assert torch.equal(y, y2)
    yb = affine_qmm(m, x, out_dtype=torch.bfloat16)
    assert torch.equal(yb, y.to(torch.bfloat16))
    y = y.cpu().numpy()
    cols = np.unique(np.concatenate([np.arange(0, O, max(1, O // 24)), [O - 1]]))
    ng = I // gs
    ws = w.reshape(O, -1)[cols]
    scs = sc.reshape(O, ng)[cols].reshape(-1)
    bis = bi.reshape(O, ng)[cols].reshape(-1)
    ref = oracle.affine_qmm_bf16(bf16_to_f32(xb).reshape(M, I), ws, scs, bis, len(cols), I, bits, gs)
    assert normwise_rel(y[:, cols], ref) <= 1e-5


MULTI_CASES = [
    # (M, [O_i], I, bits, gs, fp16)
    (512, [8192, 512, 512], 2048, 4, 64, False),   # config-5 q / k / v in one grid
    (512, [12288, 64], 2048, 4, 64, False),        # config-5 qkvz / ba
    (300, [100, 257, 64], 192, 5, 64, True),       # ragged tiles, 5-bit runs at bit 16
    (256, [130, 72], 512, 6, 128, False),
    (384, [200, 96, 40, 33], 256, 8, 32, False),
    (270, [96, 64], 192, 4, 96, False),            # group size 96
    (64, [128, 96], 256, 4, 64, False),            # few rows, in one grid too
]


KSLAB_CASES = [
    # grids with few tiles and a long K: several k ranges
    (300, [2048], 1024, 5, 32, True),
    (270, [200, 130], 2048, 6, 128, False),        # ragged N and M
    (511, [1000], 3072, 8, 64, False),
    (256, [64, 96, 40], 1024, 4, 64, True),
    (257, [520, 33], 2048, 4, 32, False),          # one row in the last M tile
]

MULTI_CASES += KSLAB_CASES


@pytest.mark.parametrize("M,Os,I,bits,gs,fp16", MULTI_CASES, ids=lambda v: str(v))
def test_qmm_multi_matches_oracle(gpu, M, Os, I, bits, gs, fp16):
    """Matrices that share x in one product launch (logan_hip_affine_qmm_multi):
    every output against the oracle (sampled columns of the wide ones, every
    column of each last tile), the bf16 outputs equal to RNE of the f32 ones,
    and repeated calls identical."""
    import torch
    from logan_amd.device import affine_qmm_multi

    print(f"qmm multi M={M} Os={Os} I={I} bits={bits} gs={gs}", flush=True)
    rng = np.random.default_rng(M + sum(Os) + bits)
    mats, devs = [], []
    for O in Os:
        w, sc, bi = make_affine(rng, O, I, bits, gs, fp16)
        mats.append((w, sc, bi))
        devs.append(dev_matrix(torch, w, sc, bi, O, I, bits, gs, fp16))
    xb = make_x(rng, M, I).reshape(M, I)
    x = to_dev(xb.view(np.int16), torch).view(torch.bfloat16)
    ys = affine_qmm_multi(devs, x, out_dtype=torch.float32)
    ys2 = affine_qmm_multi(devs, x, out_dtype=torch.float32)
    ybs = affine_qmm_multi(devs, x, out_dtype=torch.bfloat16)
    xf = bf16_to_f32(xb).reshape(M, I)
    ng = I // gs
    for (w, sc, bi), O, y, y2, yb in zip(mats, Os, ys, ys2, ybs):
        assert torch.equal(y, y2)
        assert torch.equal(yb, y.to(torch.bfloat16))
        cols = np.unique(np.concatenate([np.arange(0, O, max(1, O // 40)),
                                         np.arange(max(0, O - 130), O)]))
        ws = w.reshape(O, -1)[cols]
        scs = sc.reshape(O, ng)[cols].reshape(-1)
        bis = bi.reshape(O, ng)[cols].reshape(-1)
        ref = oracle.affine_qmm_bf16(xf, ws, scs, bis, len(cols), I, bits, gs, fp16)
        assert normwise_rel(y.cpu().numpy()[:, cols], ref) <= 1e-5, O


def test_split_qmm_on_three_overlapping_streams(gpu):
    """Split-K products pass their partial sums through 2 library-owned
    slots. Three streams, each issuing four split products back to back
    with no synchronisation between the streams, so more calls are in flight
    than there are slots: every output equals the single-stream result
    bitwise (the kernels are deterministic), and one per stream matches the
    oracle."""
    import torch
    from logan_amd.device import affine_gemv, affine_qmm

    M, O, I, bits, gs = 64, 512, 4096, 4, 64  # 8 tiles: the grid splits K
    mats, xs, hosts = [], [], []
    for s in range(3):
        rng = np.random.default_rng(900 + s)
        w, sc, bi = make_affine(rng, O, I, bits, gs)
        xb = make_x(rng, M, I).reshape(M, I)
        mats.append(dev_matrix(torch, w, sc, bi, O, I, bits, gs))
        xs.append(to_dev(xb.view(np.int16), torch).view(torch.bfloat16))
        hosts.append((w, sc, bi, xb))
    serial = [affine_qmm(mats[s], xs[s], out_dtype=torch.float32) for s in range(3)]
    serial_g = [affine_gemv(mats[s], xs[s][:8], out_dtype=torch.float32) for s in range(3)]
    torch.cuda.synchronize()
    streams = [torch.cuda.Stream() for _ in range(3)]
    outs = [[torch.full((M, O), float("nan"), device="cuda") for _ in range(4)] for _ in range(3)]
    outs_g = [[torch.full((8, O), float("nan"), device="cuda") for _ in range(4)] for _ in range(3)]
    torch.cuda.synchronize()
    for r in range(4):
        for s in range(3):
            with torch.cuda.stream(streams[s]):
                affine_qmm(mats[s], xs[s], out=outs[s][r], stream=streams[s])
                affine_gemv(mats[s], xs[s][:8], out=outs_g[s][r], stream=streams[s])
    torch.cuda.synchronize()
    for s in range(3):
        for r in range(4):
            assert torch.equal(outs[s][r], serial[s]), (s, r)
            assert torch.equal(outs_g[s][r], serial_g[s]), (s, r)
        w, sc, bi, xb = hosts[s]
        cols = np.arange(0, O, 37)
        ng = I // gs
        ref = oracle.affine_qmm_bf16(bf16_to_f32(xb).reshape(M, I), w.reshape(O, -1)[cols],
                                     sc.reshape(O, ng)[cols].reshape(-1),
                                     bi.reshape(O, ng)[cols].reshape(-1), len(cols), I, bits, gs)
        assert normwise_rel(serial[s].cpu().numpy()[:, cols], ref) <= 1e-5


def test_split_tile_products_on_overlapping_streams(gpu):
    """The two kernels with K split lay their partial sums out differently in
    the same 2 slots: tile products of one and of several matrices and a 64 x
    64 one, back to back on each of three streams with no synchronisation
    between them. Every output equals the single-stream result bitwise; the
    serial results against the oracle on a sample of columns."""
    import torch
    from logan_amd.device import affine_qmm, affine_qmm_multi

    # (M, Os, I, bits), all split: one matrix, several, and the 64 x 64 kernel
    jobs = [(512, (512,), 2048, 4), (270, (200, 130), 2048, 6), (64, (512,), 4096, 4)]
    sets, serial = [], []
    for s in range(3):
        rng = np.random.default_rng(950 + s)
        row = []
        for M, Os, I, bits in jobs:
            mats = [make_affine(rng, O, I, bits, 64) for O in Os]
            dev = [dev_matrix(torch, *m, O, I, bits, 64) for m, O in zip(mats, Os)]
            xb = make_x(rng, M, I).reshape(M, I)
            x = to_dev(xb.view(np.int16), torch).view(torch.bfloat16)
            form, _, split = qmm_route(dev, M)
            assert (form == 1 and split > 1) if M > 64 else form == 0
            row.append((dev, x, mats, xb))
        sets.append(row)
        serial.append([affine_qmm_multi(dev, x, out_dtype=torch.float32) if len(dev) > 1
                       else [affine_qmm(dev[0], x, out_dtype=torch.float32)] for dev, x, _, _ in row])
    torch.cuda.synchronize()
    streams = [torch.cuda.Stream() for _ in range(3)]
    outs = [[[[torch.full_like(y, float("nan")) for y in ys] for ys in serial[s]] for _ in range(4)]
            for s in range(3)]
    torch.cuda.synchronize()
    for r in range(4):
        for s in range(3):
            with torch.cuda.stream(streams[s]):
                for i in range(3):
                    dev, x, _, _ = sets[s][(i + s) % 3]
                    ys = outs[s][r][(i + s) % 3]
                    if len(dev) > 1:
                        affine_qmm_multi(dev, x, outs=ys, stream=streams[s])
                    else:
                        affine_qmm(dev[0], x, out=ys[0], stream=streams[s])
    torch.cuda.synchronize()
    for s in range(3):
        for r in range(4):
            for ys, want in zip(outs[s][r], serial[s]):
                assert all(torch.equal(a, b) for a, b in zip(ys, want)), (s, r)
        for (M, Os, I, bits), (_, _, mats, xb), ys in zip(jobs, sets[s], serial[s]):
            for (w, sc, bi), O, y in zip(mats, Os, ys):
                cols = np.arange(0, O, 37)
                ng = I // 64
                ref = oracle.affine_qmm_bf16(bf16_to_f32(xb).reshape(M, I), w.reshape(O, -1)[cols],
                                             sc.reshape(O, ng)[cols].reshape(-1),
                                             bi.reshape(O, ng)[cols].reshape(-1), len(cols), I, bits, 64)
                assert normwise_rel(y.cpu().numpy()[:, cols], ref) <= 1e-5


TILE_CASES = [
    # (M, O, I, bits, gs, fp16): rows at the edges of the tiles; 1, 2, 3, 5, 9,
    # 45 steps of 64 codes (pipelines that never fill, chunks of scale words that
    # end early); rows of an odd number of groups, which start inside a dword;
    # group sizes 32 to 192
    (31, 130, 64, 8, 64, False),
    (33, 257, 128, 4, 32, True),
    (65, 96, 192, 6, 64, False),
    (128, 384, 320, 5, 64, True),
    (129, 200, 576, 8, 192, False),
    (191, 132, 2880, 4, 64, False),
    (193, 128, 384, 6, 96, True),
    (256, 130, 448, 5, 32, False),
    (257, 70, 832, 4, 64, True),
    (513, 260, 1088, 8, 64, False),
    # an odd total of groups: the last word is copied alone
    (40, 33, 192, 4, 64, False),
    (140, 161, 320, 8, 64, True),
    # few column tiles: row tiles and k ranges in turn over the chip
    (300, 64, 2048, 8, 128, False),
]


@pytest.mark.parametrize("M,O,I,bits,gs,fp16", TILE_CASES, ids=lambda v: str(v))
def test_qmm_tile_edges(gpu, M, O, I, bits, gs, fp16):
    """Shapes where tiles, pipelines and scale rows end unevenly: alone (most
    are small enough for the 64 x 64 kernel) and as the second of two matrices,
    which the tile kernel always takes. Every column of both against the
    oracle, and the two calls against each other (f32 sums in another order)."""
    import torch
    from logan_amd.device import affine_qmm, affine_qmm_multi

    rng = np.random.default_rng(M * 7 + O + bits)
    w, sc, bi = make_affine(rng, O, I, bits, gs, fp16)
    xb = make_x(rng, M, I).reshape(M, I)
    x = to_dev(xb.view(np.int16), torch).view(torch.bfloat16)
    xf = bf16_to_f32(xb).reshape(M, I)
    ref = oracle.affine_qmm_bf16(xf, w, sc, bi, O, I, bits, gs, fp16)
    m = dev_matrix(torch, w, sc, bi, O, I, bits, gs, fp16)
    y = affine_qmm(m, x, out_dtype=torch.float32)
    assert normwise_rel(y.cpu().numpy(), ref) <= 1e-5
    O2 = 37
    w2, sc2, bi2 = make_affine(rng, O2, I, bits, gs, fp16)
    mats = [dev_matrix(torch, w2, sc2, bi2, O2, I, bits, gs, fp16), m]
    assert qmm_route(mats, M)[0] == 1
    assert qmm_route([m], M)[0] == (0 if M * O <= 65536 else 1)
    y2, yt = affine_qmm_multi(mats, x, out_dtype=torch.float32)
    assert normwise_rel(yt.cpu().numpy(), ref) <= 1e-5
    ref2 = oracle.affine_qmm_bf16(xf, w2, sc2, bi2, O2, I, bits, gs, fp16)
    assert normwise_rel(y2.cpu().numpy(), ref2) <= 1e-5
    assert normwise_rel(yt.cpu().numpy(), y.cpu().numpy()) <= 1e-5


def shifted(torch, t, nbytes):
    """A copy of t that starts nbytes past an aligned address and ends with its buffer."""
    flat = t.contiguous().view(torch.uint8).reshape(-1)
    buf = torch.empty(nbytes + flat.numel(), dtype=torch.uint8, device=t.device)
    buf[nbytes:].copy_(flat)
    return buf[nbytes:].view(t.dtype).view(t.shape)


ALIGN_CASES = [
    # (M, O, I, bits, gs, fp16): odd and even numbers of groups per row (and in
    # all), every group form, one and several k ranges, chunks of scale words
    # that end early
    (65, 1033, 192, 4, 64, False),
    (130, 2880, 2880, 8, 64, False),
    (300, 4096, 1152, 6, 192, True),
    (700, 4090, 448, 5, 64, True),
    (2000, 4090, 320, 8, 64, True),
    (1999, 4100, 256, 8, 32, False),
    (1500, 4090, 1088, 4, 32, True),
    (520, 4001, 2880, 5, 96, False),
    (270, 515, 2048, 6, 32, False),
]


@pytest.mark.parametrize("M,O,I,bits,gs,fp16", ALIGN_CASES, ids=lambda v: str(v))
def test_qmm_operand_alignment(gpu, M, O, I, bits, gs, fp16):
    """Weights off 16 bytes and sidecars on the second half of a dword, each
    alone and together: the tile kernel, with the bits of the aligned call
    where the tiles are the same, else (and for it) within 1e-5 of the oracle on
    a sample of columns."""
    import torch
    from logan_amd.device import AffineMatrix, affine_qmm

    print(f"qmm align M={M} O={O} I={I} bits={bits} gs={gs}", flush=True)
    rng = np.random.default_rng(M + O + bits)
    w, sc, bi = make_affine(rng, O, I, bits, gs, fp16)
    xb = make_x(rng, M, I).reshape(M, I)
    x = to_dev(xb.view(np.int16), torch).view(torch.bfloat16)
    m = dev_matrix(torch, w, sc, bi, O, I, bits, gs, fp16)
    y = affine_qmm(m, x, out_dtype=torch.float32)
    cols = np.unique(np.concatenate([np.arange(0, O, max(1, O // 24)), np.arange(O - 5, O)]))
    ng = I // gs
    ref = oracle.affine_qmm_bf16(bf16_to_f32(xb).reshape(M, I), w.reshape(O, -1)[cols],
                                 sc.reshape(O, ng)[cols].reshape(-1), bi.reshape(O, ng)[cols].reshape(-1),
                                 len(cols), I, bits, gs, fp16)
    assert normwise_rel(y.cpu().numpy()[:, cols], ref) <= 1e-5
    for ow, os_, ob in ((4, 0, 0), (12, 2, 2), (0, 2, 2), (0, 2, 0), (8, 0, 2)):
        ms = AffineMatrix(shifted(torch, m.weights, ow), shifted(torch, m.scales, os_),
                          shifted(torch, m.biases, ob), O, I, bits, gs, fp16)
        want = 1 if bits == 5 and os_ == ob == 0 else 2
        assert qmm_route([ms], M)[0] == want
        ys = affine_qmm(ms, x, out_dtype=torch.float32)
        if qmm_route([ms], M)[1:] == qmm_route([m], M)[1:]:
            assert torch.equal(ys, y), (ow, os_, ob)
        assert normwise_rel(ys.cpu().numpy()[:, cols], ref) <= 1e-5, (ow, os_, ob)


# Sizes that give each tile height its one k range: (rows, M) with 32 column
# tiles, M short of whole tiles
TILE_ROWS = [(32, 250), (64, 500), (128, 1000), (192, 1500), (256, 2000)]
TILE_OS = (3901, 77)  # ragged column tiles, odd totals of groups where a row has an odd number
# (I, gs, fp16, bytes off alignment of weights, scales, biases): 1 to 17 steps of
# 64 codes (pipelines that never fill, chunks of scale words that end early),
# every group form and aux type; then the dword form
TILE_KINDS = [(64, 64, False, None), (128, 64, True, None), (192, 64, False, None), (576, 64, True, None),
              (1088, 64, False, None), (128, 32, True, None), (320, 32, False, None), (1088, 32, True, None),
              (192, 96, True, None), (576, 192, False, None),
              (576, 64, True, (4, 2, 2)), (1088, 64, False, (8, 2, 0)), (320, 32, True, (4, 0, 2)),
              (576, 192, False, (12, 2, 2)), (1088, 32, False, (4, 2, 2))]


def tile_rows(rows, bits, gs, off):
    """256 rows of 8-bit dwords exist for groups of 64 only."""
    return 128 if rows == 256 and bits == 8 and gs != 64 and off else rows


def weights64(torch, m):
    """bf16(code * scale + bias) of a device matrix, in float64."""
    at = torch.arange(m.I, device="cuda") * m.bits
    w = m.weights.reshape(m.O, -1).int()
    lo = at // 8
    c = ((w[:, lo] | (w[:, torch.clamp(lo + 1, max=w.shape[1] - 1)] << 8)) >> (at % 8).int()) & ((1 << m.bits) - 1)
    t = torch.float16 if m.aux_fp16 else torch.bfloat16
    s, b = (p.reshape(m.O, -1).view(t).double().repeat_interleave(m.group_size, 1) for p in (m.scales, m.biases))
    return (c.double() * s + b).float().to(torch.bfloat16).double()


@pytest.mark.parametrize("bits", [4, 5, 6, 8])
@pytest.mark.parametrize("rows,M", TILE_ROWS)
def test_qmm_tile_forms(gpu, rows, M, bits):
    """Every form of the tile kernel: two matrices in one grid against float64
    (sums of at most 1088 products in f32, another order: 1e-5 of the largest),
    bf16 outputs the RNE of the f32 ones; one matrix into rows of an odd stride
    (element stores), nothing past its columns; and a part of it on the 64 x 64
    kernel."""
    import ctypes as C

    import torch
    from logan_amd import _lib as L
    from logan_amd.device import AffineMatrix, affine_qmm, affine_qmm_multi

    for I, gs, fp16, off in TILE_KINDS:
        print(f"qmm tile rows={rows} M={M} bits={bits} I={I} gs={gs} off={off}", flush=True)
        rng = np.random.default_rng(rows + bits * I + gs)
        mats = []
        for O in TILE_OS:
            m = dev_matrix(torch, *make_affine(rng, O, I, bits, gs, fp16), O, I, bits, gs, fp16)
            if off:
                m = AffineMatrix(shifted(torch, m.weights, off[0]), shifted(torch, m.scales, off[1]),
                                 shifted(torch, m.biases, off[2]), O, I, bits, gs, fp16)
            mats.append(m)
        x = to_dev(make_x(rng, M, I).reshape(M, I).view(np.int16), torch).view(torch.bfloat16)
        want = (2 if off else 1, tile_rows(rows, bits, gs, off), 1)
        assert qmm_route(mats, M) == want
        ys = affine_qmm_multi(mats, x, out_dtype=torch.float32)
        ybs = affine_qmm_multi(mats, x, out_dtype=torch.bfloat16)
        for m, y, yb in zip(mats, ys, ybs):
            ref = x.double() @ weights64(torch, m).T.contiguous()
            assert float((y.double() - ref).abs().max() / ref.abs().max()) <= 1e-5, m.O
            assert torch.equal(yb, y.to(torch.bfloat16))
        m, y = mats[0], ys[0]
        assert qmm_route([m], M) == want
        for dt, yd in ((torch.float32, L.LOGAN_HIP_F32), (torch.bfloat16, L.LOGAN_HIP_BF16)):
            wide = torch.full((M, m.O + 2), 7.0, dtype=dt, device="cuda")
            a = m.c()
            rc = L.lib().logan_hip_affine_qmm(C.byref(a), x.data_ptr(), M, I, wide.data_ptr(), m.O + 2, yd, None)
            torch.cuda.synchronize()
            assert rc == 1
            assert torch.equal(wide[:, :m.O], y.to(dt)) and torch.all(wide[:, m.O:] == 7.0)
        n = 1000
        part = AffineMatrix(m.weights[:n], m.scales.reshape(m.O, -1)[:n], m.biases.reshape(m.O, -1)[:n], n, I, bits,
                            gs, fp16)
        assert qmm_route([part], 64)[0] == 0
        y64 = affine_qmm(part, x[:64], out_dtype=torch.float32)
        assert float((y64 - y[:64, :n]).abs().max() / y64.abs().max()) <= 1e-5


def test_tile_products_in_a_graph(gpu):
    """Tile products (one k range and several, one matrix and several, the
    dword form) captured in one graph: every replay, with eager products and
    synchronisations between, gives the eager bits."""
    import torch
    from logan_amd.device import AffineMatrix, affine_qmm, affine_qmm_multi

    jobs = []
    for M, Os, I, bits, off in [(512, (512,), 2048, 4, 0), (270, (200, 130), 2048, 6, 0), (100, (4096,), 1024, 8, 2),
                                (300, (12352,), 512, 4, 0), (200, (1000,), 2880, 8, 2)]:
        rng = np.random.default_rng(M + I)
        mats = [dev_matrix(torch, *make_affine(rng, O, I, bits, 64), O, I, bits, 64) for O in Os]
        if off:
            mats = [AffineMatrix(m.weights, shifted(torch, m.scales, off), shifted(torch, m.biases, off), m.O, I, bits,
                                 64, False) for m in mats]
        x = to_dev(make_x(rng, M, I).reshape(M, I).view(np.int16), torch).view(torch.bfloat16)
        assert qmm_route(mats, M)[0] == (2 if off else 1)
        jobs.append((mats, x, [torch.empty((M, O), device="cuda") for O in Os]))
    splits = [qmm_route(mats, x.shape[0])[2] for mats, x, _ in jobs]
    assert min(splits) == 1 and max(splits) > 1

    def step():
        for mats, x, ys in jobs:
            if len(mats) > 1:
                affine_qmm_multi(mats, x, outs=ys)
            else:
                affine_qmm(mats[0], x, out=ys[0])

    step()
    torch.cuda.synchronize()
    want = [[y.clone() for y in ys] for _, _, ys in jobs]
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        step()
    for _ in range(4):
        for _, _, ys in jobs:
            for y in ys:
                y.fill_(float("nan"))
        graph.replay()
        torch.cuda.synchronize()
        for (_, _, ys), ws in zip(jobs, want):
            assert all(torch.equal(y, w) for y, w in zip(ys, ws))
        step()
        torch.cuda.synchronize()
